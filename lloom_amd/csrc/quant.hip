// quant.hip -- quantize (activations and weights) and dequantize kernels.
//
// All of these are bit-exact restatements of lloom-tensor's from_float /
// to_float (lloom-tensor/src/quantized/k_quants.rs) on gfx950: the same f32
// operations in the same order, contraction off, IEEE division, Rust's
// half-away rounding and saturating casts.  Work is spread one block per
// wave (Q8_K), per 8 lanes (Q8_0), or one sub-block per lane for the
// iterative weight fitters, which run their sequential loops unchanged.
#include "kq_common.hpp"
#include "kq_quant.hpp"
#include "kernels.hpp"

#pragma clang fp contract(off)

namespace lloom {

// ------------------------------------------------- activation quantizers --

// Q8_K: one 256-element block per wave, written in the GGUF block layout
// (f32 d, i8 qs[256], i16 bsums[16]).  nblocks = elems / 256.
__global__ __launch_bounds__(256) void k_quantize_q8k(const float* __restrict__ x,
                                                      uint8_t* __restrict__ out, int64_t nblocks) {
    int lane = threadIdx.x & 63;
    int64_t blk = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (blk >= nblocks) return;
    float4 v = *(const float4*)(x + blk * 256 + 4 * lane);
    float d;
    int bs;
    uint32_t q = q8k_block_wave(v, &d, &bs);
    uint8_t* b = out + blk * Q8K_BYTES;
    *(uint32_t*)(b + Q8K_QS + 4 * lane) = q;
    if ((lane & 3) == 0) *(int16_t*)(b + Q8K_BS + 2 * (lane >> 2)) = (int16_t)bs;
    if (lane == 0) *(float*)b = d;
}

// Q8_K into the split layout read by the MFMA kernels: d [k/256][mp] (m
// padded to mp = a multiple of 16) and qs [m][k] with each 256-byte
// superblock permuted so that element 32j + 8g + b (sub-block j, lane group
// g, byte b) sits at 64g + 8j + b: an MFMA lane group's 8 bytes of every
// sub-block are then one contiguous 64-byte run.  One block per wave; the
// values are those of k_quantize_q8k.  With bsp, also the 32-element sums
// of every sub-block j as an MFMA operand: bsp [k/256][mp][16] bytes, byte j
// = sum & 63 and byte 8 + j = sum >> 6 (sum = 64 hi + lo, both int8).
// With `tiled`, qs is instead [mp/16][k/256][4][64][16] bytes: 16-row
// groups, and in each superblock the 64-byte run of lane group g of row r
// (the permuted offsets 64g .. 64g+63) split into four 16-byte pieces i,
// piece i at [i][16g + r % 16]: the MFMA lane 16g + r % 16 then loads its
// operand piece i of a row group's superblock from 1 KB of contiguous bytes.
template <bool X16>
__global__ __launch_bounds__(256) void k_quantize_split_q8k(const float* __restrict__ x, int8_t* __restrict__ qs,
                                                            float* __restrict__ dt, int8_t* __restrict__ bsp, int m,
                                                            int k, int mp, int tiled) {
    const int nsb = k >> 8;
    const int sb = blockIdx.y * 4 + (threadIdx.x >> 6), mi = blockIdx.x;
    if (sb >= nsb) return;
    q8k_split_block<X16>(x, qs, dt, bsp, k, mp, tiled, mi, sb, threadIdx.x & 63);
}

static int64_t pad16(int64_t m) { return (m + 15) & ~(int64_t)15; }

size_t split_q8k_bytes(int64_t k, int64_t m) {
    size_t qb = ((size_t)pad16(m) * k + 255) & ~(size_t)255;  // the tiled layout's padded rows
    return qb + (size_t)(k / 256) * pad16(m) * (sizeof(float) + 16);
}

void split_q8k_ptrs(void* base, int64_t k, int64_t m, int8_t** qs, float** d, int8_t** bsp) {
    size_t qb = ((size_t)pad16(m) * k + 255) & ~(size_t)255;
    *qs = (int8_t*)base;
    *d = (float*)((uint8_t*)base + qb);
    if (bsp) *bsp = (int8_t*)((uint8_t*)base + qb + (size_t)(k / 256) * pad16(m) * sizeof(float));
}

hipError_t launch_quantize_split_q8k(const float* x, int64_t m, int64_t k, int8_t* qs, float* d, hipStream_t s,
                                     int8_t* bsp, bool tiled, bool x16) {
    const int64_t nsb = k / 256;
    hipLaunchKernelGGL(x16 ? k_quantize_split_q8k<true> : k_quantize_split_q8k<false>,
                       dim3((unsigned)m, (unsigned)((nsb + 3) / 4)), dim3(256), 0, s, x, qs, d, bsp, (int)m, (int)k, (int)pad16(m), tiled ? 1 : 0);
    return hipGetLastError();
}

// Q8_0: one 32-element block per 8 lanes (f16 d, i8 qs[32]); the 34-byte
// blocks are 2-byte aligned, so bytes are stored as halves.
__global__ __launch_bounds__(256) void k_quantize_q8_0(const float* __restrict__ x,
                                                       uint8_t* __restrict__ out, int64_t nblocks) {
    int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
    int64_t blk = t >> 3;
    int sub = (int)(t & 7);
    bool ok = blk < nblocks;
    float4 v = ok ? *(const float4*)(x + blk * 32 + 4 * sub) : make_float4(0, 0, 0, 0);
    uint16_t d16;
    uint32_t q = q8_0_block_8lanes(v, &d16);
    if (!ok) return;
    uint8_t* b = out + blk * Q8_0_BYTES;
    uint16_t* h = (uint16_t*)(b + 2 + 4 * sub);
    h[0] = (uint16_t)(q & 0xffffu);
    h[1] = (uint16_t)(q >> 16);
    if (sub == 0) *(uint16_t*)b = d16;
}

// ------------------------------------------------------ Q4_K from_float --
// One lane fits one 32-element sub-block (the reference's sums are
// sequential), 8 lanes a superblock, 8 superblocks a wave.  Bound by VALU
// issue: about 13 instructions an element and fitting round, five rounds at
// most.  So every loop is unrolled and the 32 values and 32 levels stay in
// registers (with run-time indexes they lived in scratch memory: [8192, 2048]
// 500 us), the wave's 8 KB of x come in as whole lines and reach their lanes
// through LDS, and levels are floats (integers to 15: every product, sum of
// squares and compare is exact).

// n / d, correctly rounded, for r = 1 / d correctly rounded, and 2^-24 <= |d|:
// n r corrected by its residual (exact in an fma) is within one ulp, and a
// second correction of such a quotient rounds correctly (P. Markstein,
// "Computation of elementary functions on the IBM RISC System/6000
// processor", 1990, theorem on division).  Quotients past 64, infinities and
// NaN come back uncorrected: the callers clamp them to 15 or 0.
__device__ __forceinline__ float div_by(float n, float d, float r) {
    const float q = n * r;
    float c = __builtin_fmaf(__builtin_fmaf(-q, d, n), r, q);
    c = __builtin_fmaf(__builtin_fmaf(-c, d, n), r, c);
    return __builtin_fabsf(q) < 64.0f ? c : q;
}

// clampi(nearest_int(v), 0, 15) as a float: below zero the clamp decides, so
// the half is added with no sign; a NaN gives 0, as the saturating cast does.
__device__ __forceinline__ float level15(float v) {
    return __builtin_truncf(__builtin_amdgcn_fmed3f(v + 0x1.fffffep-2f, 0.0f, 15.0f));
}

// utils.rs:227-290 make_qkx1_quants(15, 5, x) -> (scale, -min).
__device__ __forceinline__ void make_qkx1_quants_dev(const float (&x)[32], float* out_scale, float* out_min) {
    // min_by(total_cmp) keeps the first minimum, max_by the last maximum.
    auto key = [](float f) -> int {
        int b = __builtin_bit_cast(int, f);
        return b ^ (int)(((unsigned)(b >> 31)) >> 1);
    };
    // equal keys are equal bits, so the extreme keys name the values
    int kmn = key(x[0]), kmx = kmn;
#pragma unroll
    for (int i = 1; i < 32; i++) {
        kmn = min(kmn, key(x[i]));
        kmx = max(kmx, key(x[i]));
    }
    const float mn = __builtin_bit_cast(float, key(__builtin_bit_cast(float, kmn)));
    const float mx = __builtin_bit_cast(float, key(__builtin_bit_cast(float, kmx)));
    if (mx == mn) {
        *out_scale = 0.0f;
        *out_min = 0.0f;
        return;
    }
    float min = __builtin_fminf(mn, 0.0f);
    float iscale = 15.0f / (mx - min);
    float scale = 1.0f / iscale;
    float l[32];
#pragma unroll
    for (int i = 0; i < 32; i++) l[i] = 0.0f;
    for (int it = 0; it < 5; it++) {
        float sumlx = 0.0f, suml2 = 0.0f;
        bool did_change = false;
#pragma unroll
        for (int i = 0; i < 32; i++) {
            const float xm = x[i] - min, li = level15(iscale * xm);
            did_change |= li != l[i];
            l[i] = li;
            sumlx += xm * li;
            suml2 = __builtin_fmaf(li, li, suml2);
        }
        scale = sumlx / suml2;
        float sum = -0.0f;
#pragma unroll
        for (int i = 0; i < 32; i++) sum += x[i] - scale * l[i];
        min = sum * 0.03125f;
        if (min > 0.0f) min = 0.0f;
        iscale = 1.0f / scale;
        if (!did_change) break;
    }
    *out_scale = scale;
    *out_min = -min;
}

__device__ __forceinline__ void scale_min_k4(int j, const uint8_t* q, int* d, int* m) {
    if (j < 4) {
        *d = q[j] & 63;
        *m = q[j + 4] & 63;
    } else {
        *d = (q[j + 4] & 0xF) | ((q[j - 4] >> 6) << 4);
        *m = (q[j + 4] >> 4) | ((q[j] >> 6) << 4);
    }
}

// max over the 8 lanes of a superblock
__device__ __forceinline__ float max8(float v) {
    v = __builtin_fmaxf(v, dpp<DPP_XOR1>(v));
    v = __builtin_fmaxf(v, dpp<DPP_XOR2>(v));
    return __builtin_fmaxf(v, dpp<DPP_HALF_MIRROR>(v));
}

struct __attribute__((packed, aligned(4))) Quad {
    uint32_t v[4];
};

constexpr int Q4Q_WAVES = 4, Q4Q_PITCH = 36;  // floats from lane to lane in LDS

// BlockQ4K::from_float (k_quants.rs:1622-1680).  8 lanes per superblock,
// lane j fits sub-block j; a wave covers 8 superblocks.
__global__ __launch_bounds__(64 * Q4Q_WAVES) void k_quantize_q4k(const float* __restrict__ x,
                                                                 uint8_t* __restrict__ out, int64_t nblocks) {
    __shared__ __align__(16) float buf[Q4Q_WAVES][64 * Q4Q_PITCH];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, j = lane & 7;
    const int64_t blk0 = ((int64_t)blockIdx.x * Q4Q_WAVES + wave) * 8, blk = blk0 + (lane >> 3);
    if (blk0 >= nblocks) return;  // the whole wave
    // 8 KB as eight coalesced loads; float f of the wave's 2048 belongs to
    // lane f / 32 (past the end the last superblock repeats)
    float* lb = buf[wave];
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const int64_t src = min(blk0 + i, nblocks - 1) * 256 + 4 * lane;
        *(float4*)(lb + (8 * i + (lane >> 3)) * Q4Q_PITCH + 4 * (lane & 7)) = *(const float4*)(x + src);
    }
    // a wave's LDS operations complete in order; this keeps the compiler from
    // moving the reads above the writes
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    float xs[32];
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const float4 v = *(const float4*)(lb + lane * Q4Q_PITCH + 4 * i);
        xs[4 * i] = v.x;
        xs[4 * i + 1] = v.y;
        xs[4 * i + 2] = v.z;
        xs[4 * i + 3] = v.w;
    }
    float sc, mn;
    make_qkx1_quants_dev(xs, &sc, &mn);
    const float max_scale = max8(__builtin_fmaxf(sc, 0.0f)), max_min = max8(__builtin_fmaxf(mn, 0.0f));
    const float inv_scale = max_scale > 0.0f ? 63.0f / max_scale : 0.0f;
    const float inv_min = max_min > 0.0f ? 63.0f / max_min : 0.0f;
    const int a = nearest_int(inv_scale * sc), c = nearest_int(inv_min * mn);
    const uint32_t ls = (uint32_t)(a < 63 ? a : 63) & 0xffu, lm = (uint32_t)(c < 63 ? c : 63) & 0xffu;
    // the 12 scale bytes, as three dwords, from the eight lanes' pairs
    uint32_t pk[3] = {0, 0, 0};
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const uint32_t v = (uint32_t)__shfl((int)(ls | lm << 8), (lane & ~7) + i, 64), s = v & 0xffu, m = v >> 8;
        if (i < 4) {
            pk[0] |= s << (8 * i);
            pk[1] |= m << (8 * i);
        } else {
            pk[2] |= ((s & 0xF) | ((m & 0xF) << 4)) << (8 * (i - 4));
            pk[0] |= (((s >> 4) << 6) & 0xffu) << (8 * (i - 4));
            pk[1] |= (((m >> 4) << 6) & 0xffu) << (8 * (i - 4));
        }
    }
    const uint16_t dh = f32_to_f16(max_scale / 63.0f), mh = f32_to_f16(max_min / 63.0f);
    const uint32_t b0 = byte_of(pk[0], j & 3), b1 = byte_of(pk[1], j & 3), b2 = byte_of(pk[2], j & 3);
    const int s6 = (int)(j < 4 ? b0 & 63 : (b2 & 0xF) | ((b0 >> 6) << 4));
    const int m6 = (int)(j < 4 ? b1 & 63 : (b2 >> 4) | ((b1 >> 6) << 4));
    const float d = f16_to_f32(dh) * (float)s6, dm = f16_to_f32(mh) * (float)m6;
    uint32_t q[8];  // this lane's 32 levels, a byte each
#pragma unroll
    for (int i = 0; i < 8; i++) q[i] = 0;
    if (d != 0.0f) {
        const float r = 1.0f / d;
#pragma unroll
        for (int i = 0; i < 32; i++) q[i >> 2] |= (uint32_t)level15(div_by(xs[i] + dm, d, r)) << (8 * (i & 3));
    }
    // sub-blocks 2c and 2c + 1 share the 32 bytes qs[32c ..]: the even lane
    // stores the first 16, the odd lane the rest
    uint32_t w[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const uint32_t theirs = (uint32_t)dppi<DPP_XOR1>((int)((j & 1) ? q[i] : q[4 + i]));
        w[i] = (j & 1) ? theirs | (q[4 + i] << 4) : q[i] | (theirs << 4);
    }
    if (blk >= nblocks) return;
    uint8_t* b = out + blk * Q4K_BYTES;
    *(Quad*)(b + 16 + 16 * j) = Quad{{w[0], w[1], w[2], w[3]}};
    if (j == 0) *(Quad*)b = Quad{{(uint32_t)dh | ((uint32_t)mh << 16), pk[0], pk[1], pk[2]}};
}

// ------------------------------------------------------ Q6_K from_float --
// utils.rs:62-225 make_qx_quants(n = 16, nmax, x, ls, rmse_type, qw = null).
__device__ float make_qx_quants_dev(int nmax, const float* x, int8_t* ls, int rmse_type) {
    const int n = 16;
    float max = 0.0f, amax = 0.0f;
    for (int i = 0; i < n; i++) {
        float ax = __builtin_fabsf(x[i]);
        if (ax > amax) {
            amax = ax;
            max = x[i];
        }
    }
    if (amax == 0.0f) {
        for (int i = 0; i < n; i++) ls[i] = 0;
        return 0.0f;
    }
    float iscale = -(float)nmax / max;
    if (rmse_type == 0) {
        for (int i = 0; i < n; i++) {
            int l = nearest_int(iscale * x[i]);
            ls[i] = (int8_t)(nmax + clampi(l, -nmax, nmax - 1));
        }
        return 1.0f / iscale;
    }
    const bool wt = (rmse_type % 2) == 1;
    float sumlx = 0.0f, suml2 = 0.0f;
    for (int i = 0; i < n; i++) {
        float xv = x[i];
        int l = clampi(nearest_int(iscale * xv), -nmax, nmax - 1);
        ls[i] = (int8_t)(l + nmax);
        float w = wt ? xv * xv : 1.0f;
        float lf = (float)l;
        sumlx += w * xv * lf;
        suml2 += w * lf * lf;
    }
    float scale = sumlx / suml2;
    float best = scale * sumlx;
    for (int itry = 0; itry < 3; itry++) {
        float is2 = 1.0f / scale;
        float slx = 0.0f, sl2 = 0.0f;
        bool changed = false;
        for (int i = 0; i < n; i++) {
            float xv = x[i];
            int l = clampi(nearest_int(is2 * xv), -nmax, nmax - 1);
            if (l + nmax != (int)ls[i]) changed = true;
            float w = wt ? xv * xv : 1.0f;
            float lf = (float)l;
            slx += w * xv * lf;
            sl2 += w * lf * lf;
        }
        if (!changed || sl2 == 0.0f || slx * slx <= best * sl2) break;
        for (int i = 0; i < n; i++) {
            int l = nearest_int(is2 * x[i]);
            ls[i] = (int8_t)(nmax + clampi(l, -nmax, nmax - 1));
        }
        sumlx = slx;
        suml2 = sl2;
        scale = sumlx / suml2;
        best = scale * sumlx;
    }
    for (int itry = 0; itry < 5; itry++) {
        int n_changed = 0;
        for (int i = 0; i < n; i++) {
            float xv = x[i];
            float w = wt ? xv * xv : 1.0f;
            int l = (int)ls[i] - nmax;
            float slx = sumlx - w * xv * (float)l;
            if (slx > 0.0f) {
                float sl2 = suml2 - w * (float)l * (float)l;
                int new_l = clampi(nearest_int(xv * sl2 / slx), -nmax, nmax - 1);
                if (new_l != l) {
                    slx += w * xv * (float)new_l;
                    sl2 += w * (float)new_l * (float)new_l;
                    if (sl2 > 0.0f && slx * slx * suml2 > sumlx * sumlx * sl2) {
                        ls[i] = (int8_t)(nmax + new_l);
                        sumlx = slx;
                        suml2 = sl2;
                        scale = sumlx / suml2;
                        best = scale * sumlx;
                        n_changed++;
                    }
                }
            }
        }
        if (n_changed == 0) break;
    }
    if (rmse_type < 3) return scale;
    for (int is = -4; is < 4; is++) {
        if (is == 0) continue;
        iscale = -((float)nmax + 0.1f * (float)is) / max;
        float slx = 0.0f, sl2 = 0.0f;
        for (int i = 0; i < n; i++) {
            float xv = x[i];
            int l = clampi(nearest_int(iscale * xv), -nmax, nmax - 1);
            float w = wt ? xv * xv : 1.0f;
            float lf = (float)l;
            slx += w * xv * lf;
            sl2 += w * lf * lf;
        }
        if (sl2 > 0.0f && slx * slx > best * sl2) {
            for (int i = 0; i < n; i++) {
                int l = nearest_int(iscale * x[i]);
                ls[i] = (int8_t)(nmax + clampi(l, -nmax, nmax - 1));
            }
            scale = slx / sl2;
            best = scale * slx;
        }
    }
    return scale;
}

// BlockQ6K::from_float (k_quants.rs:2174-2244).  16 lanes per superblock,
// lane ib fits 16-element group ib; a 64-thread group covers 4 superblocks.
__global__ __launch_bounds__(64) void k_quantize_q6k(const float* __restrict__ x,
                                                     uint8_t* __restrict__ out, int64_t nblocks) {
    __shared__ int8_t lbuf[4][256];
    int t = threadIdx.x;
    int g = t >> 4, ib = t & 15;
    int64_t blk = (int64_t)blockIdx.x * 4 + g;
    bool ok = blk < nblocks;
    const float* xb = x + (ok ? blk : 0) * 256 + 16 * ib;
    float xs[16];
    for (int i = 0; i < 16; i++) xs[i] = ok ? xb[i] : 0.0f;
    int8_t l[16];
    float scale = make_qx_quants_dev(32, xs, l, 1);
    // max_abs_scale over ib ascending, strict '>' : the first maximum wins
    float a = __builtin_fabsf(scale);
    if (a != a) a = -1.0f;
    float best_a = a, best_s = scale;
    int best_i = ib;
    for (int o = 1; o < 16; o <<= 1) {
        float oa = __shfl_xor(best_a, o, 64);
        float os = __shfl_xor(best_s, o, 64);
        int oi = __shfl_xor(best_i, o, 64);
        if (oa > best_a || (oa == best_a && oi < best_i)) {
            best_a = oa;
            best_s = os;
            best_i = oi;
        }
    }
    float max_scale = best_a > 0.0f ? best_s : 0.0f;
    float iscale = -128.0f / max_scale;
    uint16_t dh = f32_to_f16(1.0f / iscale);
    int sv = nearest_int(iscale * scale);
    int8_t ysc = (int8_t)(sv < 127 ? sv : 127);
    float d = f16_to_f32(dh) * (float)ysc;
    if (d != 0.0f) {
        for (int i = 0; i < 16; i++) {
            int ll = clampi(nearest_int(xs[i] / d), -32, 31);
            l[i] = (int8_t)(ll + 32);
        }
    }
    for (int i = 0; i < 16; i++) lbuf[g][16 * ib + i] = l[i];
    // scales: every lane of the group needs the 16 i8 scales for the store
    __syncthreads();
    if (!ok) return;
    uint8_t* b = out + blk * Q6K_BYTES;
    // lane ib packs ql/qh for li in [2*ib, 2*ib+2) of each 128-half
    for (int h = 0; h < 2; h++) {
        const int8_t* L = lbuf[g] + 128 * h;
        for (int li = 2 * ib; li < 2 * ib + 2; li++) {
            uint8_t q1 = L[li] & 0xF, q2 = L[li + 32] & 0xF, q3 = L[li + 64] & 0xF,
                    q4 = L[li + 96] & 0xF;
            b[64 * h + li] = (uint8_t)(q1 | (q3 << 4));
            b[64 * h + li + 32] = (uint8_t)(q2 | (q4 << 4));
            b[Q6K_QH + 32 * h + li] = (uint8_t)((L[li] >> 4) | ((L[li + 32] >> 4) << 2) |
                                                ((L[li + 64] >> 4) << 4) | ((L[li + 96] >> 4) << 6));
        }
    }
    b[Q6K_SC + ib] = (uint8_t)ysc;
    if (ib == 0) {
        b[Q6K_D] = (uint8_t)(dh & 0xff);
        b[Q6K_D + 1] = (uint8_t)(dh >> 8);
    }
}

// ---------------------------------------------------------- dequantize --

// Four outputs from element i (a multiple of 4) as one store: a wave writes 1
// KB (f32) of whole lines, and each lane reads its four quants at once.
// [8192, 2048] to f32 / f16, us, against one element a lane or four separate
// stores: Q8_0 13.7 / 10.9 (24.7 / 23.3), Q4_K 16.9 / 14.4 (19.5 / 21.5), Q6_K
// 13.5 / 11.1 (13.7 / 13.4).  y has its type's alignment; f16 takes the wide store where it is
// 8-byte aligned.
struct __attribute__((packed, aligned(4))) Out4 {
    float v[4];
};
__device__ __forceinline__ void store_out4(float* y, int64_t i, float a, float b, float c, float d) {
    *(Out4*)(y + i) = Out4{{a, b, c, d}};
}
__device__ __forceinline__ void store_out4(uint16_t* y, int64_t i, float a, float b, float c, float d) {
    const uint16_t h[4] = {f32_to_f16(a), f32_to_f16(b), f32_to_f16(c), f32_to_f16(d)};
    if (((uintptr_t)y & 7) == 0) {  // uniform
        *(uint2*)(y + i) = make_uint2(h[0] | (uint32_t)h[1] << 16, h[2] | (uint32_t)h[3] << 16);
    } else {
        for (int e = 0; e < 4; e++) y[i + e] = h[e];
    }
}
// Four bytes at a 2-byte-aligned address.
__device__ __forceinline__ uint32_t load4_a2(const uint8_t* p) {
    return *(const uint16_t*)p | (uint32_t)*(const uint16_t*)(p + 2) << 16;
}

// Row gather of the dequantizers (QTensor::embedding, mod.rs:1101-1137; the
// CPU arm's QuantizedType::embedding, :812-838): output block ob belongs to
// output row ob / rb and reads block ob % rb of weight row ids[row].  With
// ids null the map is the identity (dequantize).  An id >= rows stores a
// zero row and raises the flags.
struct RowMap {
    const uint32_t* ids;
    int64_t rb, rows;
    IdFlags flags;
};

// The source block of output block ob, or -1 for a bad id.
__device__ __forceinline__ int64_t src_block(int64_t ob, const RowMap& rm) {
    if (!rm.ids) return ob;
    const int64_t r = ob / rm.rb;
    const uint32_t id = rm.ids[r];
    if ((int64_t)id >= rm.rows) {
        if (ob % rm.rb == 0) {
            *rm.flags.sticky = 1;
            if (rm.flags.call) *rm.flags.call = 1;
        }
        return -1;
    }
    return (int64_t)id * rm.rb + (ob - r * rm.rb);
}

// BlockQ8_0::to_float (k_quants.rs:720-736): y = q * f32(d).
template <typename OutT>
__global__ __launch_bounds__(256) void k_dequant_q8_0(const uint8_t* __restrict__ w, OutT* __restrict__ y,
                                                      int64_t elems, RowMap rm) {
    const int64_t i = 4 * ((int64_t)blockIdx.x * 256 + threadIdx.x);
    if (i >= elems) return;
    const int64_t sb = src_block(i >> 5, rm);
    if (sb < 0) {
        store_out4(y, i, 0.0f, 0.0f, 0.0f, 0.0f);
        return;
    }
    const uint8_t* b = w + sb * Q8_0_BYTES;
    const float d = f16_to_f32(*(const uint16_t*)b);
    const uint32_t q = load4_a2(b + 2 + (i & 31));
    store_out4(y, i, (float)(int8_t)byte_of(q, 0) * d, (float)(int8_t)byte_of(q, 1) * d,
               (float)(int8_t)byte_of(q, 2) * d, (float)(int8_t)byte_of(q, 3) * d);
}

// BlockQ8K::to_float (k_quants.rs:2440-2451): y = d * q.
template <typename OutT>
__global__ __launch_bounds__(256) void k_dequant_q8k(const uint8_t* __restrict__ w, OutT* __restrict__ y,
                                                     int64_t elems, RowMap rm) {
    const int64_t i = 4 * ((int64_t)blockIdx.x * 256 + threadIdx.x);
    if (i >= elems) return;
    const int64_t sb = src_block(i >> 8, rm);
    if (sb < 0) {
        store_out4(y, i, 0.0f, 0.0f, 0.0f, 0.0f);
        return;
    }
    const uint8_t* b = w + sb * Q8K_BYTES;
    const float d = *(const float*)b;
    const uint32_t q = *(const uint32_t*)(b + Q8K_QS + (i & 255));
    store_out4(y, i, d * (float)(int8_t)byte_of(q, 0), d * (float)(int8_t)byte_of(q, 1),
               d * (float)(int8_t)byte_of(q, 2), d * (float)(int8_t)byte_of(q, 3));
}

// BlockQ4K::to_float (k_quants.rs:1747-1774): per 64-chunk c, low nibbles
// y = d*sc(2c)*q - dmin*m(2c), high nibbles with sub-block 2c+1.
// One superblock a wave, lane t elements 4t .. 4t + 3 (sub-block t / 8).
template <typename OutT>
__global__ __launch_bounds__(256) void k_dequant_q4k(const uint8_t* __restrict__ w, OutT* __restrict__ y,
                                                     int64_t nblocks, RowMap rm) {
    const int64_t blk = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (blk >= nblocks) return;
    const int t = threadIdx.x & 63;
    const int64_t sb = src_block(blk, rm), i = blk * 256 + 4 * t;
    if (sb < 0) {
        store_out4(y, i, 0.0f, 0.0f, 0.0f, 0.0f);
        return;
    }
    const uint8_t* b = w + sb * Q4K_BYTES;
    const uint32_t dm = *(const uint32_t*)b;
    const int j = t >> 3;
    int s, m;
    scale_min_k4(j, b + 4, &s, &m);
    const float d1 = f16_to_f32(dm & 0xffffu) * (float)s, mm = f16_to_f32(dm >> 16) * (float)m;
    const uint32_t q = (*(const uint32_t*)(b + 16 + 32 * (j >> 1) + 4 * (t & 7)) >> (4 * (j & 1))) & 0x0F0F0F0Fu;
    store_out4(y, i, d1 * (float)byte_of(q, 0) - mm, d1 * (float)byte_of(q, 1) - mm, d1 * (float)byte_of(q, 2) - mm,
               d1 * (float)byte_of(q, 3) - mm);
}

// BlockQ6K::to_float (k_quants.rs:2327-2358): y = d * sc[is] * q, with
// q = (4 low bits | 2 high bits) - 32.  One superblock a wave, lane t elements
// 4t .. 4t + 3: 128 (t / 32) + 32 r + l with run r = (t / 8) % 4.
template <typename OutT>
__global__ __launch_bounds__(256) void k_dequant_q6k(const uint8_t* __restrict__ w, OutT* __restrict__ y,
                                                     int64_t nblocks, RowMap rm) {
    const int64_t blk = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (blk >= nblocks) return;
    const int t = threadIdx.x & 63;
    const int64_t sb = src_block(blk, rm), i = blk * 256 + 4 * t;
    if (sb < 0) {
        store_out4(y, i, 0.0f, 0.0f, 0.0f, 0.0f);
        return;
    }
    const uint8_t* b = w + sb * Q6K_BYTES;
    const int h = t >> 5, r = (t >> 3) & 3, l = 4 * (t & 7);
    const uint32_t lo = (load4_a2(b + 64 * h + 32 * (r & 1) + l) >> (4 * (r >> 1))) & 0x0F0F0F0Fu;
    const uint32_t q = lo | ((load4_a2(b + Q6K_QH + 32 * h + l) >> (2 * r)) & 0x03030303u) << 4;
    const float d = f16_to_f32(*(const uint16_t*)(b + Q6K_D)) * (float)(int8_t)b[Q6K_SC + 8 * h + 2 * r + (l >> 4)];
    store_out4(y, i, d * (float)((int)byte_of(q, 0) - 32), d * (float)((int)byte_of(q, 1) - 32),
               d * (float)((int)byte_of(q, 2) - 32), d * (float)((int)byte_of(q, 3) - 32));
}

// ------------------------------------------------------------- launches --

static inline unsigned grid_of(int64_t work, int64_t per) { return (unsigned)((work + per - 1) / per); }

hipError_t launch_quantize_act(int vt, const float* x, void* out, int64_t elems, hipStream_t s) {
    if (vt == T_Q8K) {
        int64_t nb = elems / 256;
        hipLaunchKernelGGL(k_quantize_q8k, dim3(grid_of(nb, 4)), dim3(256), 0, s, x, (uint8_t*)out, nb);
    } else {
        int64_t nb = elems / 32;
        hipLaunchKernelGGL(k_quantize_q8_0, dim3(grid_of(nb * 8, 256)), dim3(256), 0, s, x, (uint8_t*)out,
                           nb);
    }
    return hipGetLastError();
}

hipError_t launch_quantize_weights(int type, const float* x, void* out, int64_t elems, hipStream_t s) {
    switch (type) {
        case T_Q8_0:
        case T_Q8K: return launch_quantize_act(type, x, out, elems, s);
        case T_Q4K: {
            int64_t nb = elems / 256;
            hipLaunchKernelGGL(k_quantize_q4k, dim3(grid_of(nb, 8 * Q4Q_WAVES)), dim3(64 * Q4Q_WAVES), 0, s, x, (uint8_t*)out,
                               nb);
            return hipGetLastError();
        }
        case T_Q6K: {
            int64_t nb = elems / 256;
            hipLaunchKernelGGL(k_quantize_q6k, dim3(grid_of(nb, 4)), dim3(64), 0, s, x, (uint8_t*)out, nb);
            return hipGetLastError();
        }
    }
    return hipErrorInvalidValue;
}

template <typename OutT>
static hipError_t dequant_t(int type, const void* w, OutT* y, int64_t elems, const RowMap& rm, hipStream_t s) {
    const uint8_t* b = (const uint8_t*)w;
    switch (type) {
        case T_Q8_0:
            hipLaunchKernelGGL(k_dequant_q8_0<OutT>, dim3(grid_of(elems, 1024)), dim3(256), 0, s, b, y, elems, rm);
            break;
        case T_Q8K:
            hipLaunchKernelGGL(k_dequant_q8k<OutT>, dim3(grid_of(elems, 1024)), dim3(256), 0, s, b, y, elems, rm);
            break;
        case T_Q4K:
            hipLaunchKernelGGL(k_dequant_q4k<OutT>, dim3(grid_of(elems / 256, 4)), dim3(256), 0, s, b, y,
                               elems / 256, rm);
            break;
        case T_Q6K:
            hipLaunchKernelGGL(k_dequant_q6k<OutT>, dim3(grid_of(elems / 256, 4)), dim3(256), 0, s, b, y,
                               elems / 256, rm);
            break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_dequantize(int type, const void* w, void* y, int out_dtype, int64_t elems, hipStream_t s) {
    const RowMap rm{nullptr, 1, 0, {nullptr, nullptr}};
    if (out_dtype == T_F16) return dequant_t<uint16_t>(type, w, (uint16_t*)y, elems, rm, s);
    return dequant_t<float>(type, w, (float*)y, elems, rm, s);
}

hipError_t launch_embedding(int type, const void* w, int64_t rows, int64_t hidden, const uint32_t* ids, int64_t n_ids,
                            void* y, int out_dtype, IdFlags flags, hipStream_t s) {
    const RowMap rm{ids, hidden / block_elems(type), rows, flags};
    const int64_t elems = n_ids * hidden;
    if (out_dtype == T_F16) return dequant_t<uint16_t>(type, w, (uint16_t*)y, elems, rm, s);
    return dequant_t<float>(type, w, (float*)y, elems, rm, s);
}

// ---------------------------------------------------------------- cast --
// Tensor::to_dtype between F32 and F16 (the cast the CPU arm's callers make
// around a quantized matmul: matmul_t_f16 converts its f16 lhs to f32 first
// and its f32 sums to f16 last, k_quants.rs:2802-2835; indexed_moe_forward_as
// casts x to act first, mod.rs:1567-1571).  f16 -> f32 is exact, f32 -> f16
// round-to-nearest-even (half::f16::from_f32).  Four elements a lane.
__global__ __launch_bounds__(256) void k_cast_f32_f16(const float* __restrict__ x, uint16_t* __restrict__ y,
                                                      int64_t count) {
    const int64_t i = 4 * ((int64_t)blockIdx.x * 256 + threadIdx.x);
    if (i + 4 <= count) {
        const float4 v = *(const float4*)(x + i);
        uint2 o;
        o.x = (uint32_t)f32_to_f16(v.x) | ((uint32_t)f32_to_f16(v.y) << 16);
        o.y = (uint32_t)f32_to_f16(v.z) | ((uint32_t)f32_to_f16(v.w) << 16);
        *(uint2*)(y + i) = o;
    } else {
        for (int64_t j = i; j < count; j++) y[j] = f32_to_f16(x[j]);
    }
}

__global__ __launch_bounds__(256) void k_cast_f16_f32(const uint16_t* __restrict__ x, float* __restrict__ y,
                                                      int64_t count) {
    const int64_t i = 4 * ((int64_t)blockIdx.x * 256 + threadIdx.x);
    if (i + 4 <= count) {
        const uint2 v = *(const uint2*)(x + i);
        *(float4*)(y + i) = make_float4(f16_to_f32(v.x & 0xffffu), f16_to_f32(v.x >> 16), f16_to_f32(v.y & 0xffffu),
                                        f16_to_f32(v.y >> 16));
    } else {
        for (int64_t j = i; j < count; j++) y[j] = f16_to_f32(x[j]);
    }
}

hipError_t launch_cast(int src_t, const void* src, int dst_t, void* dst, int64_t count, hipStream_t s) {
    if (count <= 0) return hipSuccess;
    const unsigned grid = (unsigned)((count + 1023) / 1024);
    if (src_t == T_F32 && dst_t == T_F16)
        hipLaunchKernelGGL(k_cast_f32_f16, dim3(grid), dim3(256), 0, s, (const float*)src, (uint16_t*)dst, count);
    else if (src_t == T_F16 && dst_t == T_F32)
        hipLaunchKernelGGL(k_cast_f16_f32, dim3(grid), dim3(256), 0, s, (const uint16_t*)src, (float*)dst, count);
    else
        return hipErrorInvalidValue;
    return hipGetLastError();
}

}  // namespace lloom
