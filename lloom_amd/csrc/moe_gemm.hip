// moe_gemm.hip -- routed experts with several planes an expert (prefill):
// QTensor::indexed_moe_forward* as a grouped GEMM on v_mfma_f32_32x32x16_f16.
//
// The contract is the CPU arm's (matmul_t_indexed, lloom-tensor/src/quantized
// /mod.rs:766-810): f32 activations, exactly dequantized weights, f32 sums.
// Two launches a call:
//  1. k_moe_gemm_prep: one workgroup an expert collects the (b, t) planes
//     routed to it and cuts them into tiles of up to 64; the others convert the
//     activation rows, each once: x' = x * 2^s (one power of two a row, max
//     |x'| in [2^13, 2^14): exact) as fp16 hi + lo / 2^13, in the order the
//     GEMM's operands want, and (Q4_K) the 32-element sums of x' likewise.
//  2. k_moe_gemm: one workgroup per (tile of planes, block of weight rows).
//     Weights go from HBM to registers and are unpacked there, once per 64
//     planes, into exact fp16 integers; activations stream through LDS.
//
// The arithmetic per superblock of 256, the products of hi and of lo in sums of
// their own (acc = acc_hi + acc_lo / 2^13):
//   Q4_K  acc = sum (sc q) x'     (sc q <= 945: exact in fp16)
//         out += d acc - dmin sum_j m_j X_j   (X_j: the sub-blocks' sums)
//         Tiles of 32 planes take q - 8 for q and 8 d sc_j - dmin m_j for
//         -dmin m_j (as an fp16 pair): their sums are of the result's own size
//         and round less than those of the unsigned q, which nearly cancel.
//   Q6_K  acc = sum (sc (q - 32)) x'; |sc (q - 32)| <= 4096 takes 12 bits,
//         one more than fp16 has, so the weight is an fp16 pair hi + lo too
//         (exact) and lo meets the activations' hi: a third MFMA
//         out += d acc
// Every product is exact in f32 and only the sums round.  What an element of x
// loses to its two halves is at most 2^-23 of it, or 2^-50 of its row's largest
// element where that is more; Q6_K's fourth product, lo lo, is at most 2^-22 of
// the whole one (and zero for the weights below 2048).  Error against 64 bits
// (2-norm, standard normal x into k = 1280 .. 2048 and products of two normals
// into k = 512 and 768; k_moe_lds and k_moe_mfma before / this):
//   Q4_K  tiles of 32: SwiGLU 3.4e-7 (from 8 planes an expert 5.5e-7) / 2.0e-7,
//         one weight 2.3e-7 (3.9e-7) / 1.3e-7; tiles of 64: 5.6e-7 / 4.8e-7 and
//         3.9e-7 / 3.3e-7
//   Q6_K  one weight 2.4e-7 / 1.4e-7
// With hi and lo in one sum and lo unscaled it was 5.7e-7, 4.0e-7 and 1.7e-7,
// and an element lost up to 2^-39 of its row's largest.
#include "kernels.hpp"
#include "kq_common.hpp"
#include "kq_gemm.hpp"
#include "kq_mfma.hpp"

namespace lloom {

#pragma clang fp contract(off)

typedef _Float16 gh8 __attribute__((ext_vector_type(8)));
typedef _Float16 gh2 __attribute__((ext_vector_type(2)));
typedef float gf16 __attribute__((ext_vector_type(16)));

// x' = hi + lo / MG_LO.  |x'| < 2^14 leaves |x' - hi| <= 4, so lo stays below
// 2^15, and it is a normal number wherever hi is one.
constexpr float MG_LO = 8192.0f;
constexpr float MG_SUM = 32.0f;  // the sums of 32 x' are stored / 32: below 2^14 too
constexpr int MG_WAVES = 4;   // waves of a GEMM workgroup
constexpr int MG_COLS = MG_WAVES * 32;  // weight rows of a workgroup (SwiGLU: half of each weight)

// ---------------------------------------------------------- the workspace --
// int hdr[16] ([1] tiles), then at 256-byte steps:
// int4 tiles[] (expert, first place in sorted, planes), int sorted[planes],
// float inv[rows] (2^-s), fp16 sums[rows][K/256][2][hi, lo][4] (sub-block 4h +
// i at [h][..][i], / 32), and x' [rows][K/256][1 KB].
static size_t up256(size_t b) { return (b + 255) & ~(size_t)255; }

// Planes of a tile, at most: 64, and 32 up to 16 planes an expert, where the
// smaller LDS and register budget keeps three workgroups a CU instead of two
// (Q6_K SwiGLU: two).  [128, 768, 2048], T tokens top-8, us with tiles of 32 /
// 64: Q4_K T = 64 45.8 / 47.2, 256 45.5 / 51.0, 512 65.4 / 63.3; its SwiGLU
// launch 256 77 / 77, 512 114 / 102; Q6_K 64 66 / 71, 256 69 / 74, 512 104 /
// 90.  Q4_K rows past 32768 elements, which f32 dots served before, stay with
// the tiles of 32 and their smaller error.
static int mg_tile_rows(int type, int64_t E, int64_t planes, int64_t k) {
    return planes > 16 * (E < planes ? E : planes) && !(type == T_Q4K && k > 32768) ? 64 : 32;
}

struct MgLayout {
    size_t tiles, sorted, inv, sums, xq, total;
    int64_t max_tiles;
};
static MgLayout mg_layout(int64_t E, int64_t planes, int64_t rows, int64_t k) {
    MgLayout l;
    l.max_tiles = planes / 32 + (E < planes ? E : planes);
    l.tiles = 256;
    l.sorted = l.tiles + up256((size_t)l.max_tiles * 16);
    l.inv = l.sorted + up256((size_t)planes * 4);
    l.sums = l.inv + up256((size_t)rows * 4);
    l.xq = l.sums + up256((size_t)rows * (k / 256) * 32);
    l.total = l.xq + up256((size_t)rows * k * 4);
    return l;
}

size_t moe_gemm_workspace_bytes(int64_t E, int64_t planes, int64_t rows, int64_t k) {
    return mg_layout(E, planes, rows, k).total;
}

// Where this route is taken.  It can be: rows of whole superblocks, 32-bit
// byte offsets into x' and into one expert's weights.  It is the faster one:
// its time hardly depends on the planes while each active expert has one tile
// (11 us at k = 256, 25 at 2048, then the weight stream), and k_moe_lds's
// grows with planes * n * k.  Measured against k_moe_lds with random routing
// and the weights in HBM, us for one weight, SwiGLU in brackets, [E, n, k]:
//   Q4_K, planes an expert: [128, 768, 2048] 3.5 45 (77) / 53 (97); [64, 1280,
//     2048] 3.5 43 (64) / 47 (83); and planes * n: [32, 2048, 768] 229 K 20 (28)
//     / 18 (30), 262 K 20 (28) / 21 (35); [32, 768, 2048] 98 K 23 (31) / 21 (35),
//     123 K 23 (32) / 29 (43)
//   Q6_K [128, 768, 2048] 3 82 (146) / 74 (194), 4 81 (147) / 84 (233); [32,
//     2048, 768] 4 28 (44) / 31 (71); [32, 768, 2048] 147 K 42 (57) / 42 (84);
//     [8, 768, 2048] 8 planes an expert 34 (34) / 31 (41), 12 34 (34) / 41 (55)
// Over E 8 .. 256, n 512 .. 2048, k 256 .. 4096 the rule is at most 1.11 (Q4_K)
// and 1.19 (Q6_K, [8, 768, 4096] with 12 planes an expert) of the better one.
// With 8 planes an expert Q4_K comes here at any size (11 / 13 us at [8, 256,
// 256], 21 / 53 at [8, 768, 2048] against k_moe_mfma).
bool moe_gemm_fits(int type, int64_t E, int64_t planes, int64_t rows, int64_t n, int64_t k) {
    if ((type != T_Q4K && type != T_Q6K) || k % 256) return false;
    if (rows * k * 4 >= ((int64_t)1 << 32) || n * (k / 256) * block_bytes(type) >= ((int64_t)1 << 31)) return false;
    const int64_t experts = E < planes ? E : planes, size = planes * n;
    if (type == T_Q4K) return planes >= 8 * experts || (2 * planes >= 7 * experts && size >= 131072);
    return (planes >= 12 * experts && size >= 65536) || (planes >= 4 * experts && size >= 196608);
}

// ------------------------------------------------------------------- prep --

// Workgroups that route, at most: each reads all ids, so past a CU's worth of
// them more would only repeat that ([4096, 64, 256], 128 K planes: 365 us with one
// an expert, 130 with these, 291 with k_moe_route and k_moe_mfma).
constexpr int MG_ROUTERS = 256, MG_PER_MAX = (MOE_MAX_EXPERTS + MG_ROUTERS - 1) / MG_ROUTERS;

// Workgroup r of R collects the planes of `per` experts.  It counts every
// expert's planes, so it knows by itself where its planes and tiles go and the
// workgroups need nothing of each other (one workgroup for all experts took
// 17 us at 4096 planes, this 4).  The order inside an expert follows the LDS
// atomics; every plane's dot is computed on its own, so no result depends on
// it.
__device__ void mg_route(const uint32_t* __restrict__ ids, int planes, int r, int per, int E, int* hdr, int4* tiles,
                         int* sorted, IdFlags flags, float* y, float* y2, int n, int tile_rows) {
    __shared__ int s_cnt[MOE_MAX_EXPERTS], s_at[MG_PER_MAX];
    __shared__ int s_first, s_tile, s_tiles;
    const int tid = threadIdx.x, lane = tid & 63, R = (E + per - 1) / per;
    const int e0 = r * per, e1 = min(e0 + per, E);
    for (int i = tid; i < E; i += 1024) s_cnt[i] = 0;
    if (tid == 0) s_first = s_tile = s_tiles = 0;
    __syncthreads();
    int bad = 0;
    for (int p0 = tid; p0 < planes; p0 += 8 * 1024) {
        uint32_t id[8];
#pragma unroll
        for (int i = 0; i < 8; i++) id[i] = p0 + i * 1024 < planes ? ids[p0 + i * 1024] : 0u;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            if (p0 + i * 1024 >= planes) continue;
            if (id[i] < (uint32_t)E) atomicAdd(&s_cnt[id[i]], 1);
            else bad = 1;
        }
    }
    bad = __syncthreads_or(bad);
    if (bad) {
        // out-of-range ids: zero outputs, and the flags.  Runs of 64 planes are
        // dealt to the workgroups' waves, which store a plane together (one
        // lane a plane, in one workgroup, took 1.8 ms for 4096 planes of 768
        // outputs, the call this way 45 us)
        for (int64_t p = 64 * (r + R * (tid >> 6)); p < planes; p += 64 * 16 * R) {
            const bool out = p + lane < planes && ids[p + lane] >= (uint32_t)E;
            for (uint64_t m = __ballot(out); m; m &= m - 1) {
                const int64_t at = (p + __builtin_ctzll(m)) * n;
                for (int j = lane; j < n; j += 64) {
                    y[at + j] = 0.0f;
                    if (y2) y2[at + j] = 0.0f;
                }
            }
        }
    }
    int first = 0, tile = 0, all = 0;  // planes and tiles of smaller experts, tiles of all
    for (int i = tid; i < E; i += 1024) {
        const int c = s_cnt[i], t = (c + tile_rows - 1) / tile_rows;
        first += i < e0 ? c : 0;
        tile += i < e0 ? t : 0;
        all += t;
    }
#pragma unroll
    for (int o = 32; o; o >>= 1) {
        first += __shfl_xor(first, o, 64);
        tile += __shfl_xor(tile, o, 64);
        all += __shfl_xor(all, o, 64);
    }
    if (lane == 0 && all) {
        atomicAdd(&s_first, first);
        atomicAdd(&s_tile, tile);
        atomicAdd(&s_tiles, all);
    }
    __syncthreads();
    if (tid == 0 && r == 0) {
        report_ids(flags, bad);
        hdr[1] = s_tiles;
    }
    first = s_first;
    tile = s_tile;
    const int none = first;
    for (int e = e0; e < e1; e++) {
        // the planes over as few tiles as hold them, each a multiple of 32
        const int c = s_cnt[e], k = (c + tile_rows - 1) / tile_rows;
        if (c) {
            const int rows = ((c + k - 1) / k + 31) & ~31;
            for (int i = tid; i < k; i += 1024) tiles[tile + i] = make_int4(e, first + i * rows, min(rows, c - i * rows), 0);
        }
        if (tid == 0) s_at[e - e0] = first;
        first += c;
        tile += k;
    }
    if (first == none) return;  // uniform
    __syncthreads();
    for (int p0 = tid; p0 < planes; p0 += 8 * 1024) {
        uint32_t id[8];
#pragma unroll
        for (int i = 0; i < 8; i++) id[i] = p0 + i * 1024 < planes ? ids[p0 + i * 1024] : ~0u;
#pragma unroll
        for (int i = 0; i < 8; i++)
            if (id[i] - e0 < (uint32_t)(e1 - e0)) sorted[atomicAdd(&s_at[id[i] - e0], 1)] = p0 + i * 1024;
    }
}

// Place of the 8-element group G (elements 8G .. 8G + 7) of a superblock in
// the GEMM's operand order: lane half h of MFMA step t (16 of them) takes
//   Q4_K  qs bytes 64h + 8 (t / 2) .., the low (t even) or high nibbles
//   Q6_K  ql bytes 64h + 8 (t / 2) .., likewise
// so a lane's weights of a superblock are 64 contiguous bytes (Q6_K: and 32
// of qh), and eight steps hold half of them.
template <int TYPE>
__device__ __forceinline__ void mg_place(int G, int& t, int& h) {
    h = G >> 4;
    const int q = (G >> 2) & 3;  // the 32-element run in the half
    // Q4_K: runs 2i, 2i + 1 are the nibbles of qs bytes 32i ..; Q6_K: runs q,
    // q + 2 those of ql bytes 32q ..
    const int chunk = TYPE == T_Q4K ? q >> 1 : q & 1, nib = TYPE == T_Q4K ? q & 1 : q >> 1;
    t = 2 * (4 * chunk + (G & 3)) + nib;
}

// x' of a superblock: [half t / 8][hi, lo][(t / 4) & 1][t & 3][h][8] fp16, so a
// GEMM stage (eight steps) takes whole 128-byte lines of a row.
__device__ __forceinline__ int mg_xq_off(int t, int h) {
    return (t >> 3) * 512 + ((t >> 2) & 1) * 128 + ((t & 3) * 2 + h) * 16;
}

// The first ceil(E / per) workgroups route; the others convert 16 rows each, one
// a wave.
template <int TYPE>
__global__ __launch_bounds__(1024) void k_moe_gemm_prep(const float* __restrict__ X, int rows, int K,
                                                        uint8_t* __restrict__ xq, _Float16* __restrict__ sums,
                                                        float* __restrict__ inv, const uint32_t* __restrict__ ids,
                                                        int planes, int per, int E, int* hdr, int4* tiles, int* sorted,
                                                        IdFlags flags, float* y, float* y2, int n, int tile_rows) {
    const int routers = (E + per - 1) / per;
    if ((int)blockIdx.x < routers) {
        mg_route(ids, planes, blockIdx.x, per, E, hdr, tiles, sorted, flags, y, y2, n, tile_rows);
        return;
    }
    const int lane = threadIdx.x & 63, row = (blockIdx.x - routers) * 16 + (threadIdx.x >> 6);
    if (row >= rows) return;
    const int k8 = K >> 3;
    const float* x = X + (int64_t)row * K;
    float mx = 0.0f;
    for (int i = lane; i < k8; i += 64) {
        const float4 a = *(const float4*)(x + 8 * i), b = *(const float4*)(x + 8 * i + 4);
        mx = fmaxf(mx, fmaxf(fmaxf(fmaxf(fabsf(a.x), fabsf(a.y)), fmaxf(fabsf(a.z), fabsf(a.w))),
                             fmaxf(fmaxf(fabsf(b.x), fabsf(b.y)), fmaxf(fabsf(b.z), fabsf(b.w)))));
    }
    mx = wave_max(mx);
    const bool fin = mx > 0.0f && mx <= 3.4028234e38f;
    int ex = 0;
    if (fin) (void)frexpf(mx, &ex);
    // max |x'| in [2^13, 2^14); 2^s and 2^-s stay normal numbers (a row of
    // subnormals comes out smaller, its last bit 2^-23: still exact)
    const int sh = fin ? max(-126, min(126, 14 - ex)) : 0;
    const float sc = ldexpf(1.0f, sh);
    if (lane == 0) inv[row] = ldexpf(1.0f, -sh);
    uint8_t* q = xq + (size_t)row * K * 4;
    _Float16* sm = sums + (size_t)row * (K >> 8) * 16;
    for (int i = lane; i < k8; i += 64) {
        const float4 a = *(const float4*)(x + 8 * i), b = *(const float4*)(x + 8 * i + 4);
        const float v[8] = {a.x * sc, a.y * sc, a.z * sc, a.w * sc, b.x * sc, b.y * sc, b.z * sc, b.w * sc};
        gh8 hi, lo;
        float sum = 0.0f;
#pragma unroll
        for (int u = 0; u < 8; u++) {
            // Q4_K's unpacking gives a dword's bytes in the order 0, 2, 1, 3
            const int at = TYPE == T_Q4K && (u & 3) % 3 ? u ^ 3 : u;
            const _Float16 h = (_Float16)v[u];
            hi[at] = h;
            lo[at] = (_Float16)((v[u] - (float)h) * MG_LO);
            sum += v[u];
        }
        const int sb = i >> 5, G = i & 31;
        int s, g;
        mg_place<TYPE>(G, s, g);
        uint8_t* d = q + sb * 1024 + mg_xq_off(s, g);
        *(gh8*)d = hi;
        *(gh8*)(d + 256) = lo;
        if constexpr (TYPE == T_Q4K) {
            // the four groups of a 32-element sub-block are a quad of lanes
            sum += dpp<DPP_XOR1>(sum);
            sum += dpp<DPP_XOR2>(sum);
            if ((G & 3) == 0) {
                const float s32 = sum * (1.0f / MG_SUM);
                const _Float16 h = (_Float16)s32;
                _Float16* sj = sm + sb * 16 + (G >> 4) * 8 + ((G >> 2) & 3);
                sj[0] = h;
                sj[4] = (_Float16)((s32 - (float)h) * MG_LO);
            }
        }
    }
}

// ------------------------------------------------------------------- GEMM --

// A lane's weights of one superblock of its row: half h of the quants.
template <int TYPE>
struct MgW;
template <>
struct MgW<T_Q4K> {
    uint4 hdr, q[4];
    static constexpr int LOADS = 5;
};
template <>
struct MgW<T_Q6K> {
    uint4 q[4], h[2];
    uint2 sc;
    uint32_t d;
    static constexpr int LOADS = 10;  // at least: 68, 36, 12 and 2 bytes by at most 16
};

template <int TYPE>
__device__ __forceinline__ void mg_load(const uint8_t* __restrict__ b, int h, MgW<TYPE>& w) {
    if constexpr (TYPE == T_Q4K) {
        w.hdr = *(const uint4*)b;
#pragma unroll
        for (int i = 0; i < 4; i++) w.q[i] = *(const uint4*)(b + 16 + 64 * h + 16 * i);
    } else {
        load32_a2(b + 64 * h, w.q[0], w.q[1]);
        load32_a2(b + 64 * h + 32, w.q[2], w.q[3]);
        load32_a2(b + Q6K_QH + 32 * h, w.h[0], w.h[1]);
        w.sc = load8_a2(b + Q6K_SC + 8 * h);
        w.d = *(const uint16_t*)(b + Q6K_D);
    }
}

__device__ __forceinline__ gh2 as_h2(uint32_t v) { return __builtin_bit_cast(gh2, v); }
__device__ __forceinline__ gh2 both(_Float16 v) { return gh2{v, v}; }
__device__ __forceinline__ uint32_t dword_of(const uint4& v, int i) { return i == 0 ? v.x : i == 1 ? v.y : i == 2 ? v.z : v.w; }
// two bytes (0..63) as fp16
__device__ __forceinline__ gh2 bytes_h2(uint32_t w) {
    return as_h2(__builtin_amdgcn_perm(0x64646464u, w, 0x04010400u)) + both((_Float16)-1024.0f);
}

// Scales (mins) of sub-blocks 4h .. 4h + 3, a byte each: 0-3 are the low six
// bits of hdr.y (hdr.z), 4-7 the low (high) nibbles of hdr.w under its top bits.
__device__ __forceinline__ uint32_t q4k_scales4(const uint4& hdr, int h) {
    const uint32_t lo = hdr.y & 0x3F3F3F3Fu, hi = (hdr.w & 0x0F0F0F0Fu) | ((hdr.y >> 2) & 0x30303030u);
    return h ? hi : lo;
}
__device__ __forceinline__ uint32_t q4k_mins4(const uint4& hdr, int h) {
    const uint32_t lo = hdr.z & 0x3F3F3F3Fu, hi = ((hdr.w >> 4) & 0x0F0F0F0Fu) | ((hdr.z >> 2) & 0x30303030u);
    return h ? hi : lo;
}

// The scales of a lane's half superblock.
template <int TYPE>
struct MgS;
template <>
struct MgS<T_Q4K> {
    gh2 s[2], o[2];  // [32-byte chunk]{low, high nibbles}: scale and offset
};
template <>
struct MgS<T_Q6K> {
    gh2 s[2][2];  // [32-byte chunk][low, high nibbles]{bytes 0-15, 16-31}
};

template <int TYPE, bool MID>
__device__ __forceinline__ void mg_scales(const MgW<TYPE>& w, int h, MgS<TYPE>& c) {
    if constexpr (TYPE == T_Q4K) {
        // MID: (64 + q) sc - 72 sc = (q - 8) sc.  Else (1024 + q) sc - 1024 sc,
        // and for a high nibble left in place (1024 + 16 q) (sc / 16) - 64 sc:
        // both q sc.  All of it exact.
        const uint32_t v = q4k_scales4(w.hdr, h);
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const gh2 p = bytes_h2(v >> (16 * i));
            c.s[i] = MID ? p : p * gh2{(_Float16)1.0f, (_Float16)0.0625f};
            c.o[i] = MID ? p * both((_Float16)-72.0f) : p * gh2{(_Float16)-1024.0f, (_Float16)-64.0f};
        }
    } else {
        // element 128h + 32q + l has scale sc[8h + 2q + l / 16]
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const uint32_t v = i ? w.sc.y : w.sc.x;  // runs 2i, 2i + 1: high nibbles of chunks 0, 1 for i = 1
#pragma unroll
            for (int j = 0; j < 2; j++)
                c.s[j][i] = gh2{(_Float16)(int)(int8_t)byte_of(v, 2 * j), (_Float16)(int)(int8_t)byte_of(v, 2 * j + 1)};
        }
    }
}

// (v & mask) | base: two nibbles of v under the exponent of 1024 or, four bits
// higher, of 64.  With both constants in registers it is one instruction; left
// alone the compiler takes two (and, or), each with a literal.
constexpr uint32_t MG_1024 = 0x64006400u, MG_64 = 0x54005400u;
__device__ __forceinline__ gh2 and_or(uint32_t v, uint32_t mask, uint32_t base) {
    uint32_t r;
    asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(r) : "v"(v), "s"(mask), "v"(base));
    return as_h2(r);
}

// The B operand(s) of step t (compile-time): eight weights of the lane.
template <int TYPE, bool MID>
__device__ __forceinline__ void mg_unpack(const MgW<TYPE>& w, const MgS<TYPE>& c, int t, uint32_t base, gh8& bh, gh8& bl) {
    const int nib = t & 1, g = t >> 1, chunk = g >> 2;  // byte group g of 8: bytes 8g .. 8g + 7 of the lane's 64
    uint32_t r[4], l[4];
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const uint32_t v = dword_of(w.q[g >> 1], 2 * (g & 1) + i);
        if constexpr (TYPE == T_Q4K) {
            const gh2 sc = both(c.s[chunk][nib]), of = both(c.o[chunk][nib]);
            const uint32_t mask = MID || nib ? 0x00F000F0u : 0x000F000Fu;
            const gh2 e = and_or(MID && !nib ? v << 4 : v, mask, base), o = and_or(MID && !nib ? v >> 4 : v >> 8, mask, base);
            r[2 * i] = __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(e, sc, of));
            r[2 * i + 1] = __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(o, sc, of));
        } else {
            // the two high bits of run q = chunk + 2 nib are bits 2q of qh byte 8 (g % 4) ..
            const uint32_t hb = dword_of(w.h[(g & 3) >> 1], 2 * (g & 1) + i);
            const int sh = 2 * chunk + 4 * nib;  // to bits 4, 5
            const uint32_t hi2 = (sh <= 4 ? hb << (4 - sh) : hb >> (sh - 4)) & 0x30303030u;
            const uint32_t q = ((nib ? v >> 4 : v) & 0x0F0F0F0Fu) | hi2;
            const gh2 k = both((_Float16)-1056.0f);  // -(1024 + 32)
            const gh2 sc = both(c.s[chunk][nib][(g & 3) >> 1]);
#pragma unroll
            for (int j = 0; j < 2; j++) {
                const gh2 x = as_h2(__builtin_amdgcn_perm(0x64646464u, q, j ? 0x04030402u : 0x04010400u)) + k;
                const gh2 hi = x * sc;
                r[2 * i + j] = __builtin_bit_cast(uint32_t, hi);
                l[2 * i + j] = __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(x, sc, -hi));
            }
        }
    }
    bh = __builtin_bit_cast(gh8, make_uint4(r[0], r[1], r[2], r[3]));
    if constexpr (TYPE == T_Q6K) bl = __builtin_bit_cast(gh8, make_uint4(l[0], l[1], l[2], l[3]));
}

// The B operands that meet the sums of x' (MFMA k 8h + i: the hi of sub-block
// 4h + i for i < 4, then the lo), and their scale: d, cs and ch (with MID, cl
// too) such that the superblock adds d acc + cs (sums . (ch + cl)).
template <bool MID>
__device__ __forceinline__ void mg_mins(const uint4& hdr, int h, float& d, float& cs, gh8& ch, gh8& cl) {
    d = f16_to_f32(hdr.x & 0xffffu);
    const float dmin = f16_to_f32(hdr.x >> 16);
    const gh2 il = both((_Float16)(1.0f / MG_LO));
    const uint32_t mv = q4k_mins4(hdr, h);
    if constexpr (!MID) {
        cs = -MG_SUM * dmin;
        const gh2 m0 = bytes_h2(mv), m1 = bytes_h2(mv >> 16), l0 = m0 * il, l1 = m1 * il;
        ch = gh8{m0[0], m0[1], m1[0], m1[1], l0[0], l0[1], l1[0], l1[1]};
    } else {
        // c = 8 d sc - dmin m, rounded once, times a power of two that brings
        // the larger of 8 d and dmin into [2^7, 2^8): |c| < 2^15
        const float d8 = 8.0f * d;
        const int ex = 8 - __builtin_amdgcn_frexp_expf(fmaxf(fabsf(d8), fabsf(dmin)));
        const float ds = ldexpf(d8, ex), ms = ldexpf(dmin, ex);
        cs = ldexpf(MG_SUM, -ex);
        const uint32_t sv = q4k_scales4(hdr, h);
        gh2 hi[2], lo[2];
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const float a = __builtin_fmaf(ds, (float)byte_of(sv, 2 * i), -(ms * (float)byte_of(mv, 2 * i)));
            const float b = __builtin_fmaf(ds, (float)byte_of(sv, 2 * i + 1), -(ms * (float)byte_of(mv, 2 * i + 1)));
            hi[i] = gh2{(_Float16)a, (_Float16)b};
            lo[i] = gh2{(_Float16)(a - (float)hi[i][0]), (_Float16)(b - (float)hi[i][1])};
        }
        const gh2 h0 = hi[0] * il, h1 = hi[1] * il, l0 = lo[0] * il, l1 = lo[1] * il;
        ch = gh8{hi[0][0], hi[0][1], hi[1][0], hi[1][1], h0[0], h0[1], h1[0], h1[1]};
        cl = gh8{lo[0][0], lo[0][1], lo[1][0], lo[1][1], l0[0], l0[1], l1[0], l1[1]};
    }
}

// LDS of a workgroup: two stages of half a superblock, two of the sums
constexpr int mg_stage(int rows) { return rows * 512; }
constexpr int mg_lds(int rows) { return 2 * mg_stage(rows) + 2 * rows * 32; }

template <int N>
__device__ __forceinline__ void mg_wait_barrier() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

// Keep a superblock's weights in registers at this point.
__device__ __forceinline__ void mg_keep(uint4& v) { asm volatile("" : "+v"(v.x), "+v"(v.y), "+v"(v.z), "+v"(v.w)); }
__device__ __forceinline__ void mg_keep(MgW<T_Q4K>& w) {
    mg_keep(w.hdr);
#pragma unroll
    for (int i = 0; i < 4; i++) mg_keep(w.q[i]);
}
__device__ __forceinline__ void mg_keep(MgW<T_Q6K>& w) {
#pragma unroll
    for (int i = 0; i < 4; i++) mg_keep(w.q[i]);
    mg_keep(w.h[0]);
    mg_keep(w.h[1]);
    asm volatile("" : "+v"(w.sc.x), "+v"(w.sc.y), "+v"(w.d));
}

// The order of half a step's instructions: its LDS reads, then half of the
// next step's unpacking spread between its n MFMAs.
template <int TYPE, int MT>
__device__ __forceinline__ void mg_sched(int n) {
    constexpr int V = TYPE == T_Q6K ? 32 : 12;  // about the VALU instructions of a step's unpacking
    constexpr int M = (TYPE == T_Q6K ? 3 : 2) * MT;
    __builtin_amdgcn_sched_group_barrier(0x100, MT, 0);
#pragma unroll
    for (int i = 0; i < n; i++) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, (V + M - 1) / M, 0);
    }
}

struct MgArgs {
    const uint8_t* w[2];
    float* y[2];
    const uint8_t* xq;
    const uint8_t* sums;
    int n, K, rowdiv;  // activation row of plane p: p / rowdiv
};

// A 16-byte LDS read serves a wave in four passes of 16 lanes, the first two
// lanes {0-3, 12-15, 20-27} and the rest of 0-31: with row r's piece p at
// place p ^ key(r) of its 128-byte line, the 16 rows of a pass read 16
// different pieces of the 256 bytes of the banks.
__device__ __forceinline__ int mg_key(int r) { return (r >> 1) & 7; }

// A tile of np <= 32 MT planes against the workgroup's weight rows.  MFMA
// operands (32x32x16): lane l holds plane (weight row) l % 32, elements 8 (l /
// 32) .. of the step; the result's lane l holds weight row l % 32, planes 8 (i
// / 4) + 4 (l / 32) + i % 4.
//
// LDS holds two stages of half a superblock (eight MFMA steps): the rows' x'
// in octets of 8 rows, an octet's 128-byte line (hi or lo, four steps) as one
// 1 KB DMA: row r's 16-byte piece u at place u ^ mg_key(r) of its line.
// While a stage is computed, the next one's DMAs and (Q4_K) the next
// superblock's weight loads are in flight; a stage starts with one counted wait
// and one barrier.  Q6_K's weights are 2-byte aligned and realigned where they
// are loaded, which waits for them (and for the DMAs) there.  Rows past np hold
// whatever LDS held: their sums are not stored.
template <int TYPE, int ROWS, int MT, bool GLU, bool MID>
__device__ __forceinline__ void mg_tile(const MgArgs& A, int np, int col0, const uint8_t* W0, const uint8_t* W1, float* Y,
                                        uint8_t* smem, const int* s_plane, const int* s_row, const float* s_inv) {
    constexpr int STAGE = mg_stage(ROWS);
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int h = lane >> 5, c32 = lane & 31;
    const int nsb = A.K >> 8;

    // this lane's weight row: SwiGLU takes 16 of the gate (lanes c32 < 16) and
    // the same 16 of the up weight
    const int wrow = GLU ? col0 + wave * 16 + (c32 & 15) : col0 + wave * 32 + c32;
    const uint8_t* wp = (GLU && c32 >= 16 ? W1 : W0) + (size_t)min(wrow, A.n - 1) * ((uint32_t)nsb * block_bytes(TYPE));
    auto load_w = [&](int sb, MgW<TYPE>& w) { mg_load<TYPE>(wp + (size_t)sb * block_bytes(TYPE), h, w); };

    // x' DMAs: wave w moves line w (hi or lo, step quad) of every octet
    const int octets = (np + 7) >> 3;
    uint32_t xoff[4 * MT];
#pragma unroll
    for (int o = 0; o < 4 * MT; o++) {
        const int r = 8 * o + (lane >> 3);
        xoff[o] = (uint32_t)s_row[min(r, np - 1)] * (uint32_t)A.K * 4u + (uint32_t)(((lane & 7) ^ mg_key(r & 31)) * 16);
    }
    const uint32_t soff = (uint32_t)s_row[min(32 * (wave & 1) + (lane >> 1), np - 1)] * (uint32_t)nsb * 32u + (lane & 1) * 16;
    const uint32_t lds0 = lds_addr(smem);
    auto issue = [&](int sb, int half) {
        const uint8_t* base = A.xq + (size_t)sb * 1024 + half * 512 + wave * 128;
        const uint32_t to = lds0 + half * STAGE + wave * 1024;
#pragma unroll
        for (int o = 0; o < 4 * MT; o++)
            if (o < octets) dma16s(base, xoff[o], to + o * 4096);  // uniform
    };
    auto issue_sums = [&](int sb) {
        if constexpr (TYPE == T_Q4K)
            if (wave < MT)
                dma16s(A.sums + (size_t)sb * 32, soff, lds0 + 2 * STAGE + (sb & 1) * (ROWS * 32) + wave * 1024);
    };
    static_assert(MG_WAVES == 4, "a wave a line");

    // the operand reads of a stage: row 32 T + c32, piece 2 (t % 4) + h
    const uint32_t a0 = (uint32_t)((c32 >> 3) * 4096 + (c32 & 7) * 128 + ((h ^ mg_key(c32)) * 16));
    const uint8_t* ap[4] = {smem + a0, smem + (a0 ^ 32u), smem + (a0 ^ 64u), smem + (a0 ^ 96u)};

    gf16 out[MT], acc[MT], acl[MT];
    const gf16 z = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int T = 0; T < MT; T++) out[T] = z;

    // A step's MFMAs take the activations' lo, then their hi; its hi is read
    // while lo's MFMAs run, the next step's lo while hi's run, and the next
    // step's weights are unpacked between them.
    gh8 ah[MT], al[MT], bh[2], bl[2];
    MgW<TYPE> w, nxt;
    MgS<TYPE> sc;
    uint32_t base = MID ? MG_64 : MG_1024;
    asm("" : "+v"(base));
    auto read_a = [&](int t, int lo, gh8(&a)[MT]) {
        const uint8_t* p = ap[t & 3] + (t >> 3) * STAGE + lo * 2048 + ((t >> 2) & 1) * 1024;
#pragma unroll
        for (int T = 0; T < MT; T++) a[T] = *(const gh8*)(p + T * 16384);
    };
    auto take_w = [&]() {
        // the loaded weights become the current ones here, before the next
        // loads and DMAs go out: the wait the compiler puts in front of their
        // use then finds nothing younger in flight
        w = nxt;
        mg_keep(w);
        mg_scales<TYPE, MID>(w, h, sc);
    };
    load_w(0, nxt);
    issue(0, 0);
    issue_sums(0);
    mg_wait_barrier<0>();
    take_w();
    issue(0, 1);
    load_w(min(1, nsb - 1), nxt);
    read_a(0, 1, al);
    mg_unpack<TYPE, MID>(w, sc, 0, base, bh[0], bl[0]);
    for (int sb = 0; sb < nsb; sb++) {
        float d, cs;
        gh8 am[MT], ch, cl;
        const bool last = sb + 1 == nsb;
#pragma unroll
        for (int t = 0; t < 16; t++) {
            const int cur = t & 1;
            read_a(t, 0, ah);
#pragma unroll
            for (int T = 0; T < MT; T++)
                acl[T] = __builtin_amdgcn_mfma_f32_32x32x16_f16(al[T], bh[cur], t ? acl[T] : z, 0, 0, 0);
            if (t < 15) {
                mg_unpack<TYPE, MID>(w, sc, t + 1, base, bh[cur ^ 1], bl[cur ^ 1]);
                mg_sched<TYPE, MT>(MT);
            }
            if (t == 7) {
                // the half's last reads are done: the other half has landed
                // (its DMAs are older than the weight loads), and this one's
                // place is free
                mg_wait_barrier<MgW<TYPE>::LOADS>();
                if (!last) {
                    issue(sb + 1, 0);
                    issue_sums(sb + 1);
                }
            }
            if (t < 15) {
                read_a(t + 1, 1, al);
            } else {
                // the epilogue's operands, before w moves on
                if constexpr (TYPE == T_Q4K) {
                    mg_mins<MID>(w.hdr, h, d, cs, ch, cl);
                    const uint8_t* sp = smem + 2 * STAGE + (sb & 1) * (ROWS * 32) + c32 * 32 + h * 16;
#pragma unroll
                    for (int T = 0; T < MT; T++) am[T] = *(const gh8*)(sp + T * 1024);
                } else {
                    d = f16_to_f32(w.d);
                }
                if (!last) {  // uniform
                    mg_wait_barrier<0>();
                    take_w();
                    issue(sb + 1, 1);
                    load_w(min(sb + 2, nsb - 1), nxt);
                    read_a(0, 1, al);
                    mg_unpack<TYPE, MID>(w, sc, 0, base, bh[0], bl[0]);
                }
            }
            if constexpr (TYPE == T_Q6K) {
#pragma unroll
                for (int T = 0; T < MT; T++)
                    acc[T] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah[T], bl[cur], t ? acc[T] : z, 0, 0, 0);
            }
#pragma unroll
            for (int T = 0; T < MT; T++)
                acc[T] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah[T], bh[cur], TYPE == T_Q6K || t ? acc[T] : z, 0, 0, 0);
            if (t != 15) mg_sched<TYPE, MT>((TYPE == T_Q6K ? 2 : 1) * MT);
        }
        // the superblock's scale, and (Q4_K) what the sums of x' contribute
#pragma unroll
        for (int T = 0; T < MT; T++) {
            if constexpr (TYPE == T_Q4K) {
                gf16 mt = z;
                if constexpr (MID) mt = __builtin_amdgcn_mfma_f32_32x32x16_f16(am[T], cl, mt, 0, 0, 0);
                mt = __builtin_amdgcn_mfma_f32_32x32x16_f16(am[T], ch, mt, 0, 0, 0);
#pragma unroll
                for (int i = 0; i < 16; i++) out[T][i] = __builtin_fmaf(cs, mt[i], out[T][i]);
            }
#pragma unroll
            for (int i = 0; i < 16; i++)
                out[T][i] = __builtin_fmaf(d, __builtin_fmaf(acl[T][i], 1.0f / MG_LO, acc[T][i]), out[T][i]);
        }
    }
#pragma unroll
    for (int T = 0; T < MT; T++) {
        if constexpr (GLU) {
            // lanes c32 < 16 hold the gate's sums, the others the up weight's
            // of the same rows: exchanged between the two 16-lane rows, the
            // first row has both of plane i, the second of plane i + 1
#pragma unroll
            for (int i = 0; i < 16; i += 2) {
                const auto r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(unsigned, (float)out[T][i]),
                                                                __builtin_bit_cast(unsigned, (float)out[T][i + 1]), false, false);
                const unsigned r0 = r[0], r1 = r[1];
                const int q = 32 * T + 8 * (i >> 2) + 4 * h + (i & 3) + (c32 >> 4);
                if (q < np && wrow < A.n) {
                    const float a = __builtin_bit_cast(float, r0) * s_inv[q], b = __builtin_bit_cast(float, r1) * s_inv[q];
                    Y[(int64_t)s_plane[q] * A.n + wrow] = a / (1.0f + expf(-a)) * b;
                }
            }
        } else {
#pragma unroll
            for (int i = 0; i < 16; i++) {
                const int q = 32 * T + 8 * (i >> 2) + 4 * h + (i & 3);
                if (q < np && wrow < A.n) Y[(int64_t)s_plane[q] * A.n + wrow] = out[T][i] * s_inv[q];
            }
        }
    }
}

// What bounds it: [128, 768, 2048] Q4_K, 2000 tokens top-8, the SwiGLU launch
// (two weights, 201 GFLOP of hi and lo products) takes 267 us with its prep
// (0.75 PFLOP/s; 262 with hi and lo in one sum).  The matrix cores are busy 44 %
// of the cycles, the VALU 39, both 14, neither 31: two waves a SIMD, whose
// barriers (two a superblock) and L2 round trips the other one covers in part.
// Q6_K, one weight of [128, 2048, 768]: 226 us with its prep, 35, 34, 15 and 46:
// its loads are waited for in place.  At 64 tokens the Q4_K call is the weight
// stream (113 MB in 46 us, 2.5 TB/s).  Tried on earlier forms of this kernel:
// 16x16x32 MFMAs (SwiGLU launch 301 against 273 then: twice the issue slots
// left less room for the unpacking); eight waves sharing one x' tile, half the
// L2 stream (313 against 290: one workgroup a CU leaves nothing to run at its
// barriers and its ends); the rows of x' interleaved by half superblock instead
// of whole (the same).
// A workgroup takes item (tile of planes, weight block): items are dealt to
// the XCDs in contiguous runs (workgroup b runs on XCD b % 8), so the blocks
// of one tile, which read the same activations, and the tiles of one expert,
// which read the same weights, meet in one XCD's L2.
template <int TYPE, int ROWS, bool GLU>
__global__ __launch_bounds__(64 * MG_WAVES, ROWS == 64 || (GLU && TYPE == T_Q6K) ? 2 : 3) void k_moe_gemm(
    MgArgs A, const int* __restrict__ hdr, const int4* __restrict__ tiles, const int* __restrict__ sorted,
    const float* __restrict__ inv, int nblk, int pair) {
    constexpr bool MID = TYPE == T_Q4K && ROWS == 32;
    extern __shared__ __align__(16) uint8_t smem[];
    __shared__ int s_plane[ROWS], s_row[ROWS];
    __shared__ float s_inv[ROWS];
    const int per_tile = nblk << pair, total = hdr[1] * per_tile;
    const int per = (total + 7) >> 3, at = (int)(blockIdx.x >> 3), item = (int)(blockIdx.x & 7) * per + at;
    if (at >= per || item >= total) return;  // uniform
    const int tile = item / per_tile, in = item - tile * per_tile;
    const int second = pair ? in / nblk : 0, blk = in - second * nblk;
    const int4 tl = tiles[tile];
    const int e = tl.x, np = tl.z;
    if ((int)threadIdx.x < ROWS) {
        const int p = sorted[tl.y + min((int)threadIdx.x, np - 1)];
        s_plane[threadIdx.x] = p;
        s_row[threadIdx.x] = p / A.rowdiv;
        s_inv[threadIdx.x] = inv[p / A.rowdiv];
    }
    __syncthreads();
    const size_t ebytes = (size_t)e * A.n * (A.K >> 8) * block_bytes(TYPE);
    const uint8_t* W0 = A.w[second] + ebytes;
    const uint8_t* W1 = GLU ? A.w[1] + ebytes : W0;
    float* Y = A.y[second];
    const int col0 = blk * (GLU ? MG_COLS / 2 : MG_COLS);
    if constexpr (ROWS == 64) {
        if (np > 32) {  // uniform
            mg_tile<TYPE, ROWS, 2, GLU, MID>(A, np, col0, W0, W1, Y, smem, s_plane, s_row, s_inv);
            return;
        }
    }
    mg_tile<TYPE, ROWS, 1, GLU, MID>(A, np, col0, W0, W1, Y, smem, s_plane, s_row, s_inv);
}

template <int TYPE>
static hipError_t moe_gemm_type(const MoeGemmCall& c, hipStream_t s) {
    const int64_t planes = c.batch * c.topk, rows = c.in_dim1 == 1 ? c.batch : planes;
    const MgLayout l = mg_layout(c.E, planes, rows, c.k);
    const int tile_rows = mg_tile_rows(TYPE, c.E, planes, c.k);
    const int per = (int)((c.E + MG_ROUTERS - 1) / MG_ROUTERS);
    uint8_t* ws = (uint8_t*)c.ws;
    int* hdr = (int*)ws;
    int4* tiles = (int4*)(ws + l.tiles);
    int* sorted = (int*)(ws + l.sorted);
    float* inv = (float*)(ws + l.inv);
    uint8_t* sums = ws + l.sums;
    uint8_t* xq = ws + l.xq;
    hipLaunchKernelGGL(k_moe_gemm_prep<TYPE>, dim3((unsigned)((c.E + per - 1) / per + (rows + 15) / 16)), dim3(1024), 0, s,
                       c.x, (int)rows, (int)c.k, xq, (_Float16*)sums, inv, c.ids, (int)planes, per, (int)c.E, hdr, tiles,
                       sorted, c.flags, c.y, c.mode == MOE_PAIR ? c.y2 : nullptr, (int)c.n, tile_rows);
    if (hipError_t e = hipGetLastError()) return e;
    const bool glu = c.mode == MOE_GLU;
    const int pair = c.mode == MOE_PAIR ? 1 : 0;
    const int cols = glu ? MG_COLS / 2 : MG_COLS;
    const int nblk = (int)((c.n + cols - 1) / cols);
    const int64_t items = ((planes / tile_rows + (c.E < planes ? c.E : planes)) * nblk) << pair;
    const MgArgs a{{(const uint8_t*)c.w, (const uint8_t*)c.w2}, {c.y, c.y2}, xq, sums, (int)c.n, (int)c.k,
                   c.in_dim1 == 1 ? (int)c.topk : 1};
    const dim3 grid((unsigned)((items + 7) / 8 * 8));
    auto gemm = [&](auto kern, int rows_) -> hipError_t {
        if (hipError_t e = set_lds_limit((const void*)kern, mg_lds(rows_))) return e;
        hipLaunchKernelGGL(kern, grid, dim3(64 * MG_WAVES), mg_lds(rows_), s, a, hdr, tiles, sorted, inv, nblk, pair);
        return hipGetLastError();
    };
    if (tile_rows == 64) return glu ? gemm(k_moe_gemm<TYPE, 64, true>, 64) : gemm(k_moe_gemm<TYPE, 64, false>, 64);
    return glu ? gemm(k_moe_gemm<TYPE, 32, true>, 32) : gemm(k_moe_gemm<TYPE, 32, false>, 32);
}

hipError_t launch_moe_gemm(const MoeGemmCall& c, hipStream_t s) {
    return c.type == T_Q4K ? moe_gemm_type<T_Q4K>(c, s) : c.type == T_Q6K ? moe_gemm_type<T_Q6K>(c, s)
                                                                         : hipErrorInvalidValue;
}

}  // namespace lloom
