// Dense EXL3 kernels for gfx950: trellis dequant (raw and Hadamard-folded) and
// the small-row GEMV/GEMM y = had_out(had_in(x) . Wq) * svh.  Templates only;
// exl3_dense_inst.hip instantiates them once per bit width.
#pragma once

#include <stdlib.h>
#include <algorithm>

#include "exl3_gemv.hpp"
#include "exl3_capi_util.hpp"

namespace exl3 {

// ---------------------------------------------------------------- dequant (raw)

// One lane per tile; writes the 16x16 fp16 block in row-major [K][N], or with
// NK in row-major [N][K] (the transposed operand, which hipBLASLt's fp16 GEMM
// reads faster).  With NK neighbouring lanes take tiles neighbouring along k,
// so each of a lane's 16 n-rows lands next to its neighbours' in memory.
template <int BITS, int CB, bool NK = false>
__global__ __launch_bounds__(64) void dequant_raw_kernel(const int16_t* __restrict__ trellis,
                                                         int k16, int n16, uint16_t* __restrict__ out) {
    const int tile = blockIdx.x * 64 + threadIdx.x;
    if (tile >= k16 * n16) return;
    int kt, nt;
    if constexpr (NK) {
        nt = tile / k16;
        kt = tile - nt * k16;
    } else {
        kt = tile / n16;
        nt = tile - kt * n16;
    }
    TileRegs<BITS> t;
    load_tile<BITS>(t, reinterpret_cast<const u32x4_t*>(trellis) + ((size_t)kt * n16 + nt) * tile_vecs<BITS>());
    const uint32_t* W = t.words();
    if constexpr (NK) {
        const size_t K = (size_t)k16 * 16;
        static_for<16>([&](auto NI) {
            constexpr int n = decltype(NI)::value;
            u32x4_t col[2];
            static_for<8>([&](auto PI) {
                constexpr int p = decltype(PI)::value;
                const uint32_t lo = decode_half<BITS, CB, tile_t(2 * p, n)>(W);
                const uint32_t hi = decode_half<BITS, CB, tile_t(2 * p + 1, n)>(W);
                col[p >> 2][p & 3] = lo | (hi << 16);
            });
            u32x4_t* o = reinterpret_cast<u32x4_t*>(out + (size_t)(nt * 16 + n) * K + kt * 16);
            o[0] = col[0];
            o[1] = col[1];
        });
    } else {
        const size_t N = (size_t)n16 * 16;
        static_for<16>([&](auto KI) {
            constexpr int k = decltype(KI)::value;
            u32x4_t row[2];
            static_for<8>([&](auto PI) {
                constexpr int p = decltype(PI)::value;
                const uint32_t lo = decode_half<BITS, CB, tile_t(k, 2 * p)>(W);
                const uint32_t hi = decode_half<BITS, CB, tile_t(k, 2 * p + 1)>(W);
                row[p >> 2][p & 3] = lo | (hi << 16);
            });
            u32x4_t* o = reinterpret_cast<u32x4_t*>(out + (size_t)(kt * 16 + k) * N + nt * 16);
            o[0] = row[0];
            o[1] = row[1];
        });
    }
}

// 8 consecutive halves at any 2-byte alignment, as one 16-byte load where the
// target allows it.
__device__ __forceinline__ u32x4_t load_half8(const uint16_t* p) {
    typedef u32x4_t __attribute__((aligned(2))) u32x4_u;
    return *(gptr_t<u32x4_u>)p;
}

// ---------------------------------------------------------------- dequant (Hadamard folded)

// W = diag(suh) H Wq H diag(svh) / 128 in the operation order of dequant_cpu
// (recipe-lna/lna2/bindings.cpp:80-99): row transforms (* 1/sqrt(128)), then
// column transforms, value = ((v*norm)*su)*sv.  One workgroup of eight waves
// per 128x128 block:
//   1. rows: a lane owns one tile of the block and wave w its tile rows 2w and
//      2w + 1.  A tile row's 16 values are decoded into registers, transformed
//      by butterflies h = 1..8 in registers and h = 16, 32, 64 with the lanes of
//      the same tile row (lane ^ 1, 2, 8: one DPP move each), normalised, and
//      written to LDS as fp32.
//   2. columns: wave w owns columns 16w..16w+15, the lanes of 16-lane row q the
//      rows 32q..32q+31 of them: butterflies h = 1..16 in registers; for h = 32
//      and 64 two registers swap 16- and 32-lane rows, which brings both
//      operands of two butterflies into one lane; then norm, su, sv, fp16.
// The butterfly stages run in the order h = 1, 2, ..., 64 of the reference's
// scalar loop and every butterfly is a single fp32 add or subtract of the same
// two operands, so the result is bitwise the loop's.
//
// Bound by its ~30 VALU instructions per weight, so by waves in flight: the fp32
// block is 64 KB of LDS, two workgroups a CU, and eight waves each make four a
// SIMD.  Against four waves a workgroup, with the last column stage through the
// LDS permute and whole tiles decoded by 16-bit multiplies: 4096x4096 at 3 bits
// 28.2 -> 19.1 us ([n][k]), 25.0 -> 19.5 ([k][n]); 4096x12288 at 6 bits 70.1 ->
// 51.6 and 62.2 -> 52.2.
//
// LDS position of block element (r, c), fp32, unpadded: 16-byte chunks are
// XOR-swizzled by the tile column (c >> 4) & 7, so the lanes of a tile row
// writing the same chunk of their own tiles fall on distinct banks, and by r >> 5,
// so the four 16-lane rows reading 16 columns of rows 32 apart do.
__device__ __forceinline__ int hb_pos(int r, int c) {
    return r * 128 + ((((c >> 2) ^ ((c >> 4) & 7) ^ (((r >> 5) & 3) << 2)) << 2) | (c & 3));
}

// The value of lane ^ 8 of a 16-lane row (rotation by half a row).
__device__ __forceinline__ float dpp_ror8(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0x128, 0xF, 0xF, false));
}

// Phase 1 for tile rows K0, K0 + 1 of this lane's tile (kt, nt).  s1, s2, s4:
// -1 in the lanes whose nt has that bit, else 1.
template <int BITS, int CB, int K0>
__device__ __forceinline__ void had_rows(const uint32_t* W, int kt, int nt, float s1, float s2, float s4, float* mat) {
    static_for<2>([&](auto KI) {
        constexpr int k = K0 + decltype(KI)::value;
        float v[16];
        static_for<16>([&](auto NI) {
            constexpr int n = decltype(NI)::value;
            const uint32_t x = decode_pair<BITS, CB, tile_t(k, n)>(W);
            const _Float16 lo = __builtin_bit_cast(_Float16, (uint16_t)x);
            if constexpr (CB == CB_MUL1) v[n] = (float)lo;
            else v[n] = (float)(_Float16)(lo + __builtin_bit_cast(_Float16, (uint16_t)(x >> 16)));
        });
#pragma unroll
        for (int h = 1; h < 16; h <<= 1)
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const int i = (j / h) * 2 * h + (j % h);
                const float a = v[i], b = v[i + h];
                v[i] = a + b;
                v[i + h] = a - b;
            }
#pragma unroll
        for (int n = 0; n < 16; ++n) v[n] = bfly(v[n], dpp_xor<1>(v[n]), s1);
#pragma unroll
        for (int n = 0; n < 16; ++n) v[n] = bfly(v[n], dpp_xor<2>(v[n]), s2);
#pragma unroll
        for (int n = 0; n < 16; ++n) v[n] = bfly(v[n], dpp_ror8(v[n]), s4);
        const int r = 16 * kt + k;
#pragma unroll
        for (int q = 0; q < 4; ++q)
            *reinterpret_cast<float4_t*>(mat + hb_pos(r, 16 * nt + 4 * q)) =
                float4_t{v[4 * q] * HAD_NORM, v[4 * q + 1] * HAD_NORM, v[4 * q + 2] * HAD_NORM,
                         v[4 * q + 3] * HAD_NORM};
    });
}

// Butterfly across 16-lane rows 2i, 2i + 1 (ROWS 16) or 32-lane halves (ROWS 32)
// of two registers: after the swap a lane of an even row (lower half) holds both
// operands of a's butterfly, one of an odd row (upper half) those of b's.  a
// becomes their sum, b the lower minus the upper.
template <int ROWS>
__device__ __forceinline__ void swap_bfly(float& a, float& b) {
    unsigned lo, hi;
    if constexpr (ROWS == 16) {
        const auto t = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(unsigned, a), __builtin_bit_cast(unsigned, b),
                                                        false, false);
        lo = t[0];
        hi = t[1];
    } else {
        const auto t = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, a), __builtin_bit_cast(unsigned, b),
                                                        false, false);
        lo = t[0];
        hi = t[1];
    }
    const float x = __builtin_bit_cast(float, lo), y = __builtin_bit_cast(float, hi);
    a = x + y;
    b = x - y;
}

template <int BITS, int CB, bool NK = false>
__global__ __launch_bounds__(512, 4) void dequant_had_kernel(const int16_t* __restrict__ trellis, int k16,
                                                             int n16, const uint16_t* __restrict__ suh,
                                                             const uint16_t* __restrict__ svh,
                                                             uint16_t* __restrict__ out) {
    __shared__ __align__(16) float mat[128 * 128];
    const int lane = threadIdx.x & (WAVE - 1), wave = threadIdx.x / WAVE;
    const int nbc = n16 / 8;
    const int br = blockIdx.x / nbc, bc = blockIdx.x - br * nbc;
    const size_t N = (size_t)n16 * 16;
    {
        const int nt = (lane & 3) | ((lane >> 1) & 4), kt = ((lane >> 2) & 1) | ((lane >> 3) & 6);
        const float s1 = (nt & 1) ? -1.f : 1.f, s2 = (nt & 2) ? -1.f : 1.f, s4 = (nt & 4) ? -1.f : 1.f;
        TileRegs<BITS> t;
        load_tile<BITS>(t, reinterpret_cast<const u32x4_t*>(trellis) +
                               ((size_t)(8 * br + kt) * n16 + 8 * bc + nt) * tile_vecs<BITS>());
        const uint32_t* W = t.words();
        switch (wave) {
            case 0: had_rows<BITS, CB, 0>(W, kt, nt, s1, s2, s4, mat); break;
            case 1: had_rows<BITS, CB, 2>(W, kt, nt, s1, s2, s4, mat); break;
            case 2: had_rows<BITS, CB, 4>(W, kt, nt, s1, s2, s4, mat); break;
            case 3: had_rows<BITS, CB, 6>(W, kt, nt, s1, s2, s4, mat); break;
            case 4: had_rows<BITS, CB, 8>(W, kt, nt, s1, s2, s4, mat); break;
            case 5: had_rows<BITS, CB, 10>(W, kt, nt, s1, s2, s4, mat); break;
            case 6: had_rows<BITS, CB, 12>(W, kt, nt, s1, s2, s4, mat); break;
            default: had_rows<BITS, CB, 14>(W, kt, nt, s1, s2, s4, mat); break;
        }
    }
    const int c = 16 * wave + (lane & 15), q = lane >> 4;
    // after the swaps this lane's rows are k0 + 32 i + j, i < 4, j < 8
    const int k0 = 16 * (q & 1) + 8 * (q >> 1);
    u32x4_t su4[4];                                // requested before the barrier
#pragma unroll
    for (int i = 0; i < 4; ++i) su4[i] = load_half8(suh + 128 * br + k0 + 32 * i);
    const float sv = f16_bits_to_f32(svh[128 * bc + c]);
    __syncthreads();
    float v[32];
#pragma unroll
    for (int j = 0; j < 32; ++j) v[j] = mat[hb_pos(32 * q + j, c)];
    if constexpr (!NK) __syncthreads();            // mat is free: it becomes the fp16 output tile
#pragma unroll
    for (int h = 1; h < 32; h <<= 1)
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            const int i = (j / h) * 2 * h + (j % h);
            const float a = v[i], b = v[i + h];
            v[i] = a + b;
            v[i + h] = a - b;
        }
    // h = 32: v[j], j < 16, becomes row 64 (q >> 1) + 16 (q & 1) + j, v[j + 16] the row 32 below
#pragma unroll
    for (int j = 0; j < 16; ++j) swap_bfly<16>(v[j], v[j + 16]);
    // h = 64: of the first 16, v[j], j < 8, becomes row k0 + j and v[j + 8] row 64 + k0 + j; the second 32 below
#pragma unroll
    for (int j = 0; j < 8; ++j) swap_bfly<32>(v[j], v[j + 8]);
#pragma unroll
    for (int j = 16; j < 24; ++j) swap_bfly<32>(v[j], v[j + 8]);
    uint16_t* o16 = reinterpret_cast<uint16_t*>(mat);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        // rows k0 + 32 i ..: i = 0, 1, 2, 3 in v[0..7], v[16..23], v[8..15], v[24..31]
        const int b = 16 * (i & 1) + 8 * (i >> 1);
        u32x4_t o;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            float x = v[b + j] * HAD_NORM;
            x = x * f16_bits_to_f32((uint16_t)(su4[i][j >> 1] >> (16 * (j & 1))));
            x = x * sv;
            const uint32_t h = f32_to_f16_bits(x);
            if constexpr (NK) o[j >> 1] = (j & 1) ? (o[j >> 1] | (h << 16)) : h;
            else o16[(k0 + 32 * i + j) * 128 + c] = (uint16_t)h;
        }
        if constexpr (NK)
            *reinterpret_cast<u32x4_t*>(out + (size_t)(128 * bc + c) * ((size_t)k16 * 16) + 128 * br + k0 + 32 * i) = o;
    }
    if constexpr (NK) return;
    __syncthreads();
    // 128 rows x 256 bytes, 16 bytes per lane and pass
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int id = i * 512 + (int)threadIdx.x, row = id >> 4, seg = id & 15;
        *reinterpret_cast<u32x4_t*>(out + (size_t)(128 * br + row) * N + 128 * bc + 8 * seg) =
            *reinterpret_cast<const u32x4_t*>(o16 + row * 128 + 8 * seg);
    }
}

// ---------------------------------------------------------------- row Hadamard (had_r_128)

// y[r][128b + i] = (H128 v / sqrt(128))[i] * scale * post[128b + i] for every
// 128-block b of every row r, v = x[r][128b ..]; with a pre scale v is
// half(half(x) * pre), the rounding of the GEMV path's input rotation.  Butterflies
// in fp32, h = 1, 2, ..., 64.  One wave per (row, two blocks): lanes 0-31 and
// 32-63 hold one block each, 4 consecutive elements per lane; a block past the
// row (odd block count) is computed from block 2p and not stored.
__device__ __forceinline__ void load4_kind(const void* p, int kind, size_t i, float (&v)[4], bool to_half) {
    if (kind == OUT_F32) {
        const float4_t f = *reinterpret_cast<const float4_t*>(reinterpret_cast<const float*>(p) + i);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = to_half ? f16_bits_to_f32(f32_to_f16_bits(f[e])) : f[e];
    } else {
        const uint2 u = *reinterpret_cast<const uint2*>(reinterpret_cast<const uint16_t*>(p) + i);
        const uint16_t h[4] = {(uint16_t)(u.x & 0xffffu), (uint16_t)(u.x >> 16), (uint16_t)(u.y & 0xffffu),
                               (uint16_t)(u.y >> 16)};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            if (kind == OUT_F16) v[e] = f16_bits_to_f32(h[e]);
            else v[e] = to_half ? f16_bits_to_f32(f32_to_f16_bits(bf16_to_f32(h[e]))) : bf16_to_f32(h[e]);
        }
    }
}

template <int DUMMY = 0>
__global__ __launch_bounds__(64) void had_rows_kernel(const void* x, int x_kind, void* y, int y_kind, int cols,
                                                      const uint16_t* pre, const uint16_t* post, float scale) {
    const int nb = cols / 128, npair = (nb + 1) / 2;
    const int r = blockIdx.x / npair, pb = blockIdx.x - r * npair;
    const int lane = threadIdx.x;
    int b = 2 * pb + (lane >> 5);
    const bool keep = b < nb;
    if (!keep) b = 2 * pb;
    const int c0 = 128 * b + 4 * (lane & 31);
    const size_t i0 = (size_t)r * cols + c0;
    float v[4];
    load4_kind(x, x_kind, i0, v, pre != nullptr);
    if (pre) {
        const uint2 u = *reinterpret_cast<const uint2*>(pre + c0);
        const uint16_t s[4] = {(uint16_t)(u.x & 0xffffu), (uint16_t)(u.x >> 16), (uint16_t)(u.y & 0xffffu),
                               (uint16_t)(u.y >> 16)};
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = f16_bits_to_f32(f32_to_f16_bits(v[e] * f16_bits_to_f32(s[e])));
    }
    fwht128_x4(v);
    float sv[4] = {1.f, 1.f, 1.f, 1.f};
    if (post) {
        const uint2 u = *reinterpret_cast<const uint2*>(post + c0);
        sv[0] = f16_bits_to_f32((uint16_t)(u.x & 0xffffu)); sv[1] = f16_bits_to_f32((uint16_t)(u.x >> 16));
        sv[2] = f16_bits_to_f32((uint16_t)(u.y & 0xffffu)); sv[3] = f16_bits_to_f32((uint16_t)(u.y >> 16));
    }
    if (!keep) return;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        float o = v[e] * HAD_NORM;
        if (scale != 1.0f) o = o * scale;
        if (post) o = o * sv[e];
        store_out(y, i0 + e, y_kind, o);
    }
}

// ---------------------------------------------------------------- dense GEMV
//
// y = had_in(x) . Wq for rows 0..R-1 (R <= 32), split over workgroups by
// 128-column block (one output Hadamard block) and k-chunk.  A workgroup is
// 2 x nkg waves (nkg = 2, 4 or 8; gemv_plan_hb): column half cg (64 columns, 4 n-tiles) and
// k-group kg, which takes the chunk's 64-row steps kg, kg + nkg, ...  The
// k-groups' sums meet in LDS, so a k-chunk of 512 rows leaves one partial
// vector, and a call whose chunk is all of K is finished in the same launch.
//
// Quarter tiles.  Four lanes share an n-tile: lane c of a 16-lane row holds
// columns n = 4j + p (p = c & 3) of n-tile c >> 2.  By the tile permutation
// (tile_t) column n + p's windows sit 32 p elements after column n's for
// n & 7 = 0 or 4, so the lane reads its tile rotated by p blocks of BITS words
// and decodes columns 0, 4, 8 and 12 at their compile-time positions (the
// stream is circular): 2 (BITS + 1) of the tile's 8 BITS words.  A step is
// then 64 weights and 16 MFMAs per lane instead of 256 and 64, so a matrix of
// a few million weights spreads over every SIMD with one short step per wave,
// and each tile word is requested once instead of by every column group.
// A few-row call is latency-bound: what this split shortens is the chain of
// first load, rotation, decode and sum, and the partials that the finish reads
// (one per 512 k-rows).  At 4096x4096, 6 bits, 1 row: input there at 1.2 us,
// rotated 1.9, weights 2.45 (at memory rate), decoded and multiplied 4.7, sums
// stored 5.5, plus two launches.  Against 256-column items of 128 k-rows on four
// waves that each decode a quarter of every whole tile (us per call in a graph,
// before / now): 4096x4096 6-bit 1 row 10.4 / 9.5, 16 rows 13.3 / 11.0;
// 4096x1536 3-bit 16 rows 11.2 / 8.7; 4096x12288 4-bit 1 row 17.6 / 13.8;
// 8192x8192 3-bit 16 rows 25.7 / 20.6; 2048x2048 2-bit 1 row 7.6 / 5.9.
//
// The rotated input is kept in LDS with every half doubled, so an MFMA's A
// operand is one 16-byte read.

constexpr int GEMV_COLS = 128;      // columns per workgroup: one Hadamard block
constexpr int GEMV_NCG = 2;         // column halves per workgroup
constexpr int GEMV_MAX_NKG = 8;     // k-groups per workgroup
constexpr int GEMV_MAX_ROWS = 32;   // rows per call: one or two 16-row MFMA blocks share each decode
constexpr int GEMV_LDS = 160 << 10;  // bytes a CU has
constexpr int GEMV_RED_LD = 130;    // row stride (floats) of the k-groups' sums in LDS

struct GemvPlan {
    int nsteps;         // 64-row steps per k-chunk (even; the last chunk may hold fewer)
    int n_kc;           // k-chunks
    int n_hb;           // 128-column blocks
    int nkg;            // k-groups per workgroup
    bool xcd = false;   // items and finish keyed by column block (xcd_split)
};

inline int64_t gemv_block_rows(int64_t m) { return m > MAX_ROWS ? GEMV_MAX_ROWS : MAX_ROWS; }

// EXL3_GEMV_STEPS overrides the plan's steps per k-chunk (an even number; read
// once per process: the sizes callers reserve for depend on it).
inline int gemv_steps_override() {
    static const int steps = [] {
        const char* v = getenv("EXL3_GEMV_STEPS");
        const int x = v && *v ? atoi(v) : 0;
        return x >= 2 && x % 2 == 0 ? x : 0;
    }();
    return steps;
}

// Rows of the A tile in LDS, odd so that the units of neighbouring k-slices
// fall on different banks.
__host__ __device__ constexpr int gemv_a_rows(int R) { return R | 1; }

inline int gemv_lds_bytes(int64_t R, int nsteps, int nkg) {
    const int64_t a = (int64_t)nsteps * 256 * gemv_a_rows((int)R);
    const int64_t red = (int64_t)nkg * (R < MAX_ROWS ? R : MAX_ROWS) * GEMV_RED_LD * 4;
    return (int)(a > red ? a : red);
}

inline GemvPlan gemv_plan_hb(int64_t rows, int64_t k, int64_t total_hb, int cus) {
    const int env_steps = gemv_steps_override();
    GemvPlan p;
    p.n_hb = (int)total_hb;
    const int S = std::max((int)(k / STEP_K), 2);      // even
    const int64_t r = rows < GEMV_MAX_ROWS ? rows : GEMV_MAX_ROWS;
    const int cap = r > MAX_ROWS ? 16 : 32;            // LDS: at most 136 KB of A
    // Chunk length by the time it is expected to take (us): rounds of
    // workgroups a CU holds at once (16 waves), each a start of 2.7; the steps'
    // decode at 0.43 per wave-step and SIMD, and their input's rotation; for a
    // split K the finish launch, its loads and the partials' round trip.
    // Against the best of 2-32 steps at 1, 4, 16 and 32 rows on nine shapes
    // (512x256 to 8192x8192) the choice is within 4%.
    int nsteps = 2;
    double best = 1e30;
    for (int ns = 2; ns <= cap && ns <= S; ns += 2) {
        const int64_t n_kc = (S + ns - 1) / ns, wgs = total_hb * n_kc, per_cu = (wgs + cus - 1) / cus;
        const int resident = ns >= 8 ? 1 : ns >= 4 ? 2 : 4;
        double t = 2.7 * (double)((per_cu + resident - 1) / resident);
        t += (double)(per_cu * ns) * (0.215 * (r > MAX_ROWS ? 1.3 : 1.0) + 0.0094 * (double)r);
        if (n_kc > 1) t += 2.0 + 0.03 * (double)n_kc + 2e-6 * (double)(n_kc * r * total_hb * GEMV_COLS);
        if (t < best) {
            best = t;
            nsteps = ns;
        }
    }
    p.nsteps = nsteps;
    p.nkg = nsteps >= 8 ? GEMV_MAX_NKG : nsteps >= 4 ? 4 : 2;
    // Eight k-groups make a workgroup that fills a CU, whose start, exchange and
    // finish nothing covers: where a launch is several such workgroups a CU, two
    // or four k-groups leave room for others to decode meanwhile.  Expected time
    // (us) by k-groups and, where K is split anyway, chunk length: a launch's
    // start, rounds of the workgroups a CU holds (by waves and by LDS), each a
    // start and its longest chain of steps, less the more there are to cover it,
    // and the steps' decode and rotation.  Only chunks of 8 steps and more: below
    // that the first choice holds four waves a SIMD already.  One round is left as
    // it is unless the gain is clear.  On 63 shapes (512x256 to 4096x129280, 1-32
    // rows, 2-6 bits) at most 2% slower than the first choice with eight k-groups,
    // which one-wave items of whole tiles had beaten by up to 15% there; us, those
    // items / eight k-groups / this rule: 512x129280 2-bit 1 row 14.8 / 17.4 / 12.4;
    // 4096x65536 2-bit 1 row 37.9 / 42.1 / 37.9; 4096x129280 6-bit 1 row 100 / 103 /
    // 85; 8192x65536 6-bit 4 rows 105 / 113 / 96; 4096x12288 2-bit 4 rows 14.3 /
    // 14.6 / 12.5.
    if (nsteps >= 8) {
        auto time = [&](int ns, int nkg) {
            constexpr double covered[5] = {1.0, 1.0, 0.86, 0.79, 0.74};
            const int64_t n_kc = (S + ns - 1) / ns, per_cu = (total_hb * n_kc + cus - 1) / cus;
            const int resident = std::max(std::min(GEMV_MAX_NKG / nkg, GEMV_LDS / gemv_lds_bytes(r, ns, nkg)), 1);
            double t = 2.4 + std::max((double)per_cu / resident, 1.0) * (1.44 + 0.4 * ns / nkg) * covered[resident];
            t += (double)(per_cu * ns) * (0.205 * (r > MAX_ROWS ? 1.55 : 1.0) + 0.014 * (double)r);
            if (n_kc > 1) t += 2.06 + 0.0267 * (double)n_kc + 4.6e-7 * (double)(n_kc * r * total_hb * GEMV_COLS);
            return t;
        };
        const bool whole = nsteps >= S;
        const bool rounds = total_hb * ((S + nsteps - 1) / nsteps) > cus;
        double least = time(nsteps, GEMV_MAX_NKG) * (rounds ? 1.0 : 0.9);
        for (int ns = whole ? S : 8; ns <= (whole ? S : std::min(cap, S - 1)); ns += 8)
            for (int nkg = 2; nkg <= GEMV_MAX_NKG; nkg *= 2) {
                const double t = time(ns, nkg);
                if (t < least) {
                    least = t;
                    p.nsteps = ns;
                    p.nkg = nkg;
                }
            }
    }
    if (env_steps && env_steps <= cap) {
        p.nsteps = env_steps < S ? env_steps : S;
        p.nkg = p.nsteps >= 8 ? GEMV_MAX_NKG : p.nsteps >= 4 ? 4 : 2;
    }
    p.n_kc = (S + p.nsteps - 1) / p.nsteps;
    return p;
}

// The items of a column block and that block's finish run on one XCD
// (xcd_split) when the column blocks (of a matrix, or of all members of a fan)
// are a multiple of 8.  EXL3_XCD_ORDER=0 turns it off (read at every call, so
// one process can compare both orders).
inline bool xcd_order_allowed() {
    const char* v = getenv("EXL3_XCD_ORDER");
    return !(v && *v && atoi(v) == 0);
}

inline GemvPlan gemv_plan(int64_t rows, int64_t k, int64_t n, int cus) {
    GemvPlan p = gemv_plan_hb(rows, k, std::max<int64_t>(n / GEMV_COLS, 1), cus);
    p.xcd = xcd_order_allowed() && p.n_hb % N_XCD == 0;
    return p;
}

// Split-K partials of a matrix: [128-column block][row][k-chunk][128] fp32, so
// the finish of one (column block, row) reads its k-chunks from one
// contiguous range (strided reads of the same offset in every k-chunk all
// fell on a few memory channels).
inline int64_t gemv_partial_bytes(int64_t rows, int64_t n_hb, int64_t n_kc) {
    return n_kc > 1 ? n_hb * (rows < GEMV_MAX_ROWS ? rows : GEMV_MAX_ROWS) * n_kc * GEMV_COLS * 4 : 0;
}
__device__ __forceinline__ size_t gemv_partial_off(int hb, int row, int kc, int R, int n_kc) {
    return ((size_t)(hb * R + row) * n_kc + kc) * GEMV_COLS;
}

// The words of a lane's quarter tile: rotated blocks 0 and 4 and the word
// before each (the windows of columns 0, 4, 8 and 12 reach at most 16 - BITS
// bits back).  The other words are never written or read, so they take no
// registers.
template <int BITS>
struct QuarterTile {
    uint32_t w[8 * BITS];
};

template <int N>
__device__ __forceinline__ void load_words_g(uint32_t* dst, gptr_t<uint32_t> src) {
    typedef u32x4_t __attribute__((aligned(4))) u32x4_u;
    typedef uint32_t u32x2_u __attribute__((ext_vector_type(2), aligned(4)));
    if constexpr (N >= 4) {
        const u32x4_t v = *(gptr_t<u32x4_u>)src;
        dst[0] = v[0]; dst[1] = v[1]; dst[2] = v[2]; dst[3] = v[3];
        if constexpr (N > 4) load_words_g<N - 4>(dst + 4, src + 4);
    } else if constexpr (N >= 2) {
        const u32x2_u v = *(gptr_t<u32x2_u>)src;
        dst[0] = v[0]; dst[1] = v[1];
        if constexpr (N > 2) dst[2] = src[2];
    } else {
        dst[0] = src[0];
    }
}

// `t`: the lane's tile (8 BITS words), p: its rotation in blocks of BITS words.
template <int BITS>
__device__ __forceinline__ void load_quarter(QuarterTile<BITS>& d, gptr_t<uint32_t> t, int p) {
    load_words_g<BITS>(d.w, t + p * BITS);
    d.w[8 * BITS - 1] = t[p ? p * BITS - 1 : 8 * BITS - 1];
    load_words_g<BITS + 1>(d.w + 4 * BITS - 1, t + (p + 4) * BITS - 1);
}

// decode_pair on a quarter tile: every word it can read has been loaded.
template <int BITS>
constexpr bool quarter_holds(int w) {
    return w < BITS || (w >= 4 * BITS - 1 && w < 5 * BITS) || w == 8 * BITS - 1;
}
template <int BITS, int T>
constexpr bool quarter_window() {          // the words of element T's window
    using S = WinSel<BITS, T>;
    return quarter_holds<BITS>(S::I1) && (S::O >= 16 || quarter_holds<BITS>((S::I1 + 8 * BITS - 1) % (8 * BITS)));
}
template <int BITS, int CB, int T>
__device__ __forceinline__ uint32_t decode_quarter(const QuarterTile<BITS>& t) {
    static_assert(quarter_window<BITS, T>() && quarter_window<BITS, WinSel<BITS, T>::SRC_T>() &&
                      quarter_holds<BITS>(null_word<BITS, T>()),
                  "a word that load_quarter leaves out");
    return decode_pair<BITS, CB, T>(t.w);
}

// The lane's MFMA columns in decode order: columns n and n + 8, whose eight
// windows at one k-group are consecutive in the stream, back to back.
__host__ __device__ constexpr int quarter_col(int j) { return 4 * (j >> 1) + 8 * (j & 1); }

// Output rotation, svh and store of two consecutive columns per lane of one
// row's 128-column block.
__device__ __forceinline__ void gemv_finish(float v0, float v1, const uint16_t* __restrict__ svh,
                                            void* __restrict__ out, int out_kind, int N, int row, int col) {
    const float w0 = f16_bits_to_f32(svh[col]), w1 = f16_bits_to_f32(svh[col + 1]);
    fwht128_x2(v0, v1);
    store_out(out, (size_t)row * N + col, out_kind, v0 * HAD_NORM * w0);
    store_out(out, (size_t)row * N + col + 1, out_kind, v1 * HAD_NORM * w1);
}

// One item: 128-column block hb, k-chunk kc.  smem: gemv_lds_bytes.
template <int BITS, int CB, int RB>
__device__ __forceinline__ void gemv_item(const uint16_t* __restrict__ x, const int16_t* __restrict__ trellis,
                                          const uint16_t* __restrict__ suh, const uint16_t* __restrict__ svh,
                                          void* __restrict__ out, int out_kind, int R, int K, int N, int nsteps,
                                          int n_kc, int hb, int kc, float* __restrict__ partials, char* smem) {
    const int lane = threadIdx.x & (WAVE - 1);
    const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / WAVE));
    const int nw = (int)blockDim.x / WAVE, nkg = nw / GEMV_NCG;
    const int cg = w & (GEMV_NCG - 1), kg = w / GEMV_NCG;
    const int g = lane >> 4, c = lane & 15;
    const int s0 = kc * nsteps, ns = min(nsteps, K / STEP_K - s0);     // this chunk's steps, even
    const int Rp = gemv_a_rows(R);

    // Input rotation jobs: (row, 128-block), one per 16 lanes.  The first
    // pass's inputs are requested before the weights, so waiting for them
    // (loads complete in issue order) does not wait for the tile.
    const int nblk = ns / 2, jobs = R * nblk;
    u32x4_t xv, sv;
    int row, blk;
    auto rot_load = [&](int j0) {
        const int id = min(j0 + g, jobs - 1);
        row = id / nblk;
        blk = id - row * nblk;
        const int col = s0 * STEP_K + 128 * blk + 8 * c;
        xv = load_half8(x + (size_t)row * K + col);
        sv = load_half8(suh + col);
    };
    if (4 * w < jobs) rot_load(4 * w);

    // the lane's quarter tile of step s
    const int p = c & 3, n16 = N / 16;
    gptr_t<uint32_t> tp = as_global(reinterpret_cast<const uint32_t*>(trellis)) +
                          ((size_t)(4 * (s0 + kg) + g) * n16 + 8 * hb + 4 * cg + (c >> 2)) * (8 * BITS);
    const size_t tstep = (size_t)4 * nkg * n16 * (8 * BITS);
    QuarterTile<BITS> t0, t1;
    if (kg < ns) load_quarter<BITS>(t0, tp, p);

    for (int j0 = 4 * w; j0 < jobs; j0 += 4 * nw) {
        if (j0 != 4 * w) rot_load(j0);
        float v[8];
        scaled8(xv, sv, 0, v);
        const u32x4_t h = rotated8(v);
        if (j0 + g < jobs) {
            // halves 8c .. 8c + 7 of the block: k-slice c >> 1, its lower or upper 8 rows;
            // k-group r takes rows 2r, 2r + 1 of both (unit [slice][r][row], 16 bytes)
            uint2* d = reinterpret_cast<uint2*>(smem) + (size_t)((8 * blk + (c >> 1)) * 4 * Rp + row) * 2 + (c & 1);
#pragma unroll
            for (int r = 0; r < 4; ++r)
                d[(size_t)r * Rp * 2] = make_uint2(__builtin_amdgcn_perm(h[r], h[r], 0x01000100u),
                                                   __builtin_amdgcn_perm(h[r], h[r], 0x03020302u));
        }
    }
    __syncthreads();

    float4_t acc[RB][4];
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[rb][j] = float4_t{0.f, 0.f, 0.f, 0.f};
    // A rows >= R repeat row R-1 (a valid row, no branch): their outputs are never stored
    const half8_t* ap[RB];
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
        ap[rb] = reinterpret_cast<const half8_t*>(smem) + g * 4 * Rp + min(16 * rb + c, R - 1);

    auto step_mma = [&](const QuarterTile<BITS>& t, int s) {
        half8_t A[RB][4];
#pragma unroll
        for (int rb = 0; rb < RB; ++rb)
#pragma unroll
            for (int r = 0; r < 4; ++r) A[rb][r] = ap[rb][(16 * s + r) * Rp];
        static_for<4>([&](auto JI) {
            constexpr int j = decltype(JI)::value, n = quarter_col(j);
            static_for<4>([&](auto RI) {
                constexpr int r = decltype(RI)::value;
                constexpr int T0 = 32 * (n & 7) + 8 * r + 4 * (n >> 3);
                u32x4_t b;
                b[0] = decode_quarter<BITS, CB, T0 + 0>(t);
                b[1] = decode_quarter<BITS, CB, T0 + 1>(t);
                b[2] = decode_quarter<BITS, CB, T0 + 2>(t);
                b[3] = decode_quarter<BITS, CB, T0 + 3>(t);
#pragma unroll
                for (int rb = 0; rb < RB; ++rb)
                    acc[rb][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A[rb][r], __builtin_bit_cast(half8_t, b),
                                                                        acc[rb][j], 0, 0, 0);
            });
        });
    };
    for (int s = kg; s < ns; s += 2 * nkg) {
        if (s + nkg < ns) load_quarter<BITS>(t1, tp + tstep, p);
        step_mma(t0, s);
        if (s + nkg < ns) {
            tp += 2 * tstep;
            if (s + 2 * nkg < ns) load_quarter<BITS>(t0, tp, p);
            step_mma(t1, s + nkg);
        }
    }

    // Sum over the k-groups in LDS, one 16-row block at a time, then the
    // finish (whole K) or the chunk's partial vector.
    float* red = reinterpret_cast<float*>(smem);
    const int hcol = 128 * hb + 2 * lane;
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
        const int rows = min(R - 16 * rb, 16);
        __syncthreads();                               // A (or the previous block's sums) no longer read
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int m = 4 * g + i;
            if (m < rows) {
                float* d = red + (size_t)(kg * min(R, 16) + m) * GEMV_RED_LD + 64 * cg + 16 * (c >> 2) + p;
#pragma unroll
                for (int j = 0; j < 4; ++j) d[quarter_col(j)] = acc[rb][j][i];
            }
        }
        __syncthreads();
        for (int m = w; m < rows; m += nw) {
            float v0 = 0.f, v1 = 0.f;
#pragma unroll
            for (int q = 0; q < GEMV_MAX_NKG; ++q)
                if (q < nkg) {
                    const float2 t = *reinterpret_cast<const float2*>(red + (size_t)(q * min(R, 16) + m) * GEMV_RED_LD + 2 * lane);
                    v0 += t.x;
                    v1 += t.y;
                }
            if (n_kc > 1)
                *reinterpret_cast<float2*>(partials + gemv_partial_off(hb, 16 * rb + m, kc, R, n_kc) + 2 * lane) =
                    make_float2(v0, v1);
            else
                gemv_finish(v0, v1, svh, out, out_kind, N, 16 * rb + m, hcol);
        }
    }
}

template <int BITS, int CB, int RB>
__global__ __launch_bounds__(WAVE * GEMV_NCG * GEMV_MAX_NKG) void gemv_kernel(
    const uint16_t* __restrict__ x, const int16_t* __restrict__ trellis, const uint16_t* __restrict__ suh,
    const uint16_t* __restrict__ svh, void* __restrict__ out, int out_kind, int R, int K, int N, int nsteps, int n_kc,
    int xcd, float* __restrict__ partials) {
    extern __shared__ __align__(16) char gemv_smem[];
    int hb, kc;
    xcd_split(blockIdx.x, n_kc, xcd, hb, kc);          // group: column block
    gemv_item<BITS, CB, RB>(x, trellis, suh, svh, out, out_kind, R, K, N, nsteps, n_kc, hb, kc, partials, gemv_smem);
}

// Split-K finish of (128-column block hb, row m): the partials of chunks
// 0..n_kc-1 summed in chunk order, output Hadamard, svh, store; two columns
// per lane, up to RED_BATCH loads in flight.  Plain loads: a previous launch
// wrote the partials.
constexpr int RED_BATCH = 16;

template <int BATCH>
__device__ __forceinline__ void gemv_reduce_block(const float* __restrict__ partials, const uint16_t* __restrict__ svh,
                                                  void* __restrict__ out, int out_kind, int R, int N, int n_kc,
                                                  int hb, int m) {
    const int lane = threadIdx.x & (WAVE - 1);
    const float* p = partials + gemv_partial_off(hb, m, 0, R, n_kc) + 2 * lane;
    float v0 = 0.f, v1 = 0.f;
    for (int k0 = 0; k0 < n_kc; k0 += BATCH) {
        float2 t[BATCH];
#pragma unroll
        for (int j = 0; j < BATCH; ++j)
            if (k0 + j < n_kc) t[j] = *reinterpret_cast<const float2*>(p + (size_t)(k0 + j) * GEMV_COLS);
#pragma unroll
        for (int j = 0; j < BATCH; ++j)
            if (k0 + j < n_kc) {
                v0 = v0 + t[j].x;
                v1 = v1 + t[j].y;
            }
    }
    gemv_finish(v0, v1, svh, out, out_kind, N, m, 128 * hb + 2 * lane);
}

// Split-K finish, one wave per (128-column block, row).  Runs after
// gemv_kernel on the same stream.
template <int BATCH>
__global__ __launch_bounds__(64) void gemv_reduce_kernel(const float* __restrict__ partials,
                                                         const uint16_t* __restrict__ svh, void* __restrict__ out,
                                                         int out_kind, int R, int N, int n_kc, int xcd) {
    int hb, m;
    xcd_split(blockIdx.x, R, xcd, hb, m);              // group: the block whose partials were written on this XCD
    gemv_reduce_block<BATCH>(partials, svh, out, out_kind, R, N, n_kc, hb, m);
}

// ---------------------------------------------------------------- dense GEMM (33 to a few hundred rows)
//
// y = xh . Wq for rows in tiles of 16 RB (RB <= 5) rows, as the GEMV above but
// with the rotation in a launch of its own (its cost per column block would
// grow with the rows): gemm_rotate_kernel writes had_in(x) with every half
// doubled, in units of 16 bytes [step][k-slice][k-group][row], so the A
// operand of an MFMA is one coalesced 16-byte load per lane (from L2: the
// rotated input is 4 K bytes a row).  Each decoded operand feeds RB row
// blocks.  A workgroup is GEMM_NKG k-groups of a (64-column half of a
// 128-column block, k-chunk, row tile); their sums meet in LDS and leave one
// partial tile in the accumulators' own layout, which gemm_finish_kernel sums
// over the k-chunks, rotates and stores.  A chunk of the k-groups' length keeps
// the partials short: they are written, flushed at the launch's end and read
// again, and cost more than the decode (72 rows of 4096x4096 at 4 bits, of
// 11.5 us: first loads 1.4, decode and MFMAs 4.5, exchange and store 1.5, the
// rest launch and flush).
//
// What it replaces above 32 rows is the reconstructed weight in memory and a
// library GEMM between two row-Hadamard launches.  Us per call, before / with
// this kernel (fp16 in, bf16 out): 4096x4096 at 4 bits, 33 rows 29.7 / 15.4, 72
// rows 32.8 / 18.2, 128 rows 38.1 / 21.2, 256 rows 37.6 / 31.2; 4096x12288 at 6
// bits, 72 rows 65.3 / 33, 256 rows 87 / 76; 1536x4096 at 3 bits, 256 rows 28.1 /
// 19.1.  From 384 rows the reconstructed weight is read often enough to win
// (4096x4096 at 6 bits 42 / 49).

constexpr int GEMM_NKG = 8;
constexpr int GEMM_MAX_RB = 5;      // LDS of the k-groups' exchange: 28 KB per row block

// Rows of one GEMM launch (exl3_gemm runs more rows in slabs of this many).
constexpr int GEMM_MAX_ROWS = 256;

// Rows that take this path: above 32 all, 17-32 where a column block's own
// rotation of the rows, repeated by every one of them, costs more than two more
// launches.  That work goes with the rows and the weights, and a short K or few
// columns leave the GEMM's launches idle.  The bound's worst choices over 116
// matrices of 128-16384 x 1024-65536 at 17-32 rows are within 14% of the better
// kernel, the mean within 0.2%.  Us, GEMV / GEMM: 4096x4096 6-bit 24 rows 13.3 /
// 14.0, 32 rows 14.4 / 14.2; 4096x12288 3-bit 17 rows 20.9 / 19.9, 32 rows 26.8 /
// 19.7; 16384x6144 6-bit 32 rows 52.0 / 32.0; but 256x8192 6-bit 24 rows 7.6 / 9.8
// and 1024x32768 6-bit 20 rows 14.3 / 17.5.
// The rotated input's byte offsets are 32-bit.
inline bool gemm_takes(int64_t m, int64_t k, int64_t n) {
    if (k > (1 << 20) || m <= MAX_ROWS) return false;
    if (m > GEMV_MAX_ROWS) return true;
    return k >= 768 && n > 2048 && (m - 10) * k * n >= (k > 1024 || n <= 16384 ? 250000000 : 900000000);
}

struct GemmPlan {
    int rb;             // 16-row blocks per row tile
    int n_rt;           // row tiles
    int nsteps, n_kc;   // 64-row steps per k-chunk (the last may hold fewer), k-chunks
    int n_hb;           // 128-column blocks
    int64_t xd_bytes, partial_bytes;
};

inline GemmPlan gemm_plan(int64_t R, int64_t k, int64_t n, int cus) {
    GemmPlan p;
    p.n_hb = std::max((int)(n / GEMV_COLS), 1);
    const int S = std::max((int)(k / STEP_K), 1);
    const int rt0 = (int)((R + 16 * GEMM_MAX_RB - 1) / (16 * GEMM_MAX_RB));
    // Row tiles and k-chunks: whole rounds of one workgroup per CU, each a start
    // (us) and a step's decode and MFMAs per step of a wave (two waves a SIMD),
    // plus the partials' way to memory and back.  On 4096x4096, 4096x12288,
    // 1536x4096, 8192x8192 and 2048x512 at 33-512 rows the k-chunks this picks are
    // within 3% of the best of 1, 2, 3, 4, 6 and 8.  One row tile more than the
    // rows need pays where it fills a round that the fewer, taller ones leave
    // part empty (us, without / with it: 2048x9216 5-bit 81 rows 27.5 / 22.6;
    // 4096x12288 5-bit 208 rows 82 / 75, where the reconstruct path takes 78); a
    // gain of less than 5% by this model measured between 0.95x and 1.06x, so it is
    // not taken.
    // Everything here depends on the rows' 16-row blocks only, which
    // exl3_gemm_scratch_bytes relies on.
    const int blocks = (int)((R + 15) / 16);
    double best = 1e30;
    for (int n_rt = rt0; n_rt <= rt0 + 1; ++n_rt) {
        const int rb = std::max((blocks + n_rt - 1) / n_rt, 2);
        const double ts = 0.75 + 0.13 * rb;
        for (int kc = 1; kc <= 32 && kc <= S; ++kc) {
            const int ns = (S + kc - 1) / kc, n_kc = (S + ns - 1) / ns;
            if (n_kc != kc) continue;
            const int64_t wgs = (int64_t)p.n_hb * GEMV_NCG * n_rt * n_kc;
            const double rounds = (double)((wgs + cus - 1) / cus);
            double t = rounds * (1.5 + ts * ((ns + GEMM_NKG - 1) / GEMM_NKG)) +
                       2e-6 * n_kc * (16.0 * blocks) * (double)n;
            if (n_rt > rt0) t /= 0.95;
            if (t < best) {
                best = t;
                p.n_rt = n_rt;
                p.rb = rb;
                p.nsteps = ns;
                p.n_kc = n_kc;
            }
        }
    }
    const int64_t Rp = (int64_t)p.n_rt * 16 * p.rb;
    p.xd_bytes = Rp * k * 4;
    p.partial_bytes = (int64_t)p.n_hb * p.n_kc * Rp * GEMV_COLS * 4;
    return p;
}

inline int64_t gemv_scratch_bytes(const GemvPlan& p, int64_t rows) {
    return align_up(gemv_partial_bytes(rows, p.n_hb, p.n_kc), 256) + 256;
}

// Scratch of exactly this call.
inline int64_t dense_scratch_bytes(int64_t rows, int64_t k, int64_t n, int cus) {
    if (!gemm_takes(rows, k, n)) {
        const int64_t b = gemv_scratch_bytes(gemv_plan(rows, k, n, cus), rows);
        return rows > GEMV_MAX_ROWS && rows % GEMV_MAX_ROWS
                   ? std::max(b, dense_scratch_bytes(rows % GEMV_MAX_ROWS, k, n, cus))    // the last block
                   : b;
    }
    const GemmPlan g = gemm_plan(rows < GEMM_MAX_ROWS ? rows : GEMM_MAX_ROWS, k, n, cus);
    int64_t b = align_up(g.xd_bytes, 256) + g.partial_bytes;
    if (rows > GEMM_MAX_ROWS && rows % GEMM_MAX_ROWS)
        b = std::max(b, dense_scratch_bytes(rows % GEMM_MAX_ROWS, k, n, cus));      // the last slab
    return b;
}

// 8 consecutive values of kind KIND (an OutKind) as fp16 bits, at the type's own
// alignment; bf16 and fp32 values are rounded to nearest even.
template <int KIND>
__device__ __forceinline__ u32x4_t load_as_half8(const void* x, size_t i) {
    if constexpr (KIND == OUT_F16) {
        return load_half8(reinterpret_cast<const uint16_t*>(x) + i);
    } else {
        float f[8];
        if constexpr (KIND == OUT_BF16) {
            const u32x4_t b = load_half8(reinterpret_cast<const uint16_t*>(x) + i);
#pragma unroll
            for (int e = 0; e < 8; ++e) f[e] = bf16_to_f32((uint16_t)(b[e >> 1] >> (16 * (e & 1))));
        } else {
            typedef float4_t __attribute__((aligned(4))) float4_u;
            const float4_t lo = *(gptr_t<float4_u>)(reinterpret_cast<const float*>(x) + i);
            const float4_t hi = *(gptr_t<float4_u>)(reinterpret_cast<const float*>(x) + i + 4);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                f[e] = lo[e];
                f[e + 4] = hi[e];
            }
        }
        u32x4_t o;
#pragma unroll
        for (int e = 0; e < 4; ++e)
            o[e] = (uint32_t)f32_to_f16_bits(f[2 * e]) | ((uint32_t)f32_to_f16_bits(f[2 * e + 1]) << 16);
        return o;
    }
}

// KIND: x's type.  A cast in front of it is one more launch and the input's way
// to memory and back (us a call with bf16 rows, with the cast / without:
// 256x512 3-bit 33 rows 13.3 / 10.5, 4096x4096 6-bit 33 rows 19.0 / 16.1, 256
// rows 34.9 / 32.7).
template <int KIND>
__global__ __launch_bounds__(256) void gemm_rotate_kernel(const void* __restrict__ x,
                                                          const uint16_t* __restrict__ suh, int R, int K, int Rp,
                                                          u32x4_t* __restrict__ xd) {
    // one wave: four rows of one 128-block
    const int lane = threadIdx.x & (WAVE - 1), c = lane & 15;
    const int nblk = K / 128;
    const int id = (int)blockIdx.x * 4 + (int)(threadIdx.x / WAVE);
    const int rg = id / nblk, blk = id - rg * nblk;
    const int row = 4 * rg + (lane >> 4);
    if (4 * rg >= R) return;
    const int rr = min(row, R - 1);
    const int col = 128 * blk + 8 * c;
    const u32x4_t xv = load_as_half8<KIND>(x, (size_t)rr * K + col), sv = load_half8(suh + col);
    float v[8];
    scaled8(xv, sv, 0, v);
    const u32x4_t h = rotated8(v);
    if (row >= R) return;
    uint2* d = reinterpret_cast<uint2*>(xd) + ((size_t)(8 * blk + (c >> 1)) * 4 * Rp + row) * 2 + (c & 1);
#pragma unroll
    for (int r = 0; r < 4; ++r)
        d[(size_t)r * Rp * 2] = make_uint2(__builtin_amdgcn_perm(h[r], h[r], 0x01000100u),
                                           __builtin_amdgcn_perm(h[r], h[r], 0x03020302u));
}

// Partial tiles: [128-column block][k-chunk][16-row block][column j][half][lane] of four rows each, the
// accumulators' own layout: lane l's unit j is rows 4 (l >> 4) .. + 3 of column
// 64 half + 16 ((l & 15) >> 2) + (l & 3) + quarter_col(j).
__device__ __forceinline__ size_t gemm_partial_unit(int hb, int kc, int n_kc, int rb, int n_rb, int j, int cg) {
    return ((((size_t)hb * n_kc + kc) * n_rb + rb) * 4 + j) * GEMV_NCG + cg;
}

template <int BITS, int CB, int RB>
__global__ __launch_bounds__(WAVE * GEMM_NKG) void gemm_kernel(
    const u32x4_t* __restrict__ xd, const int16_t* __restrict__ trellis, int Rp, int K, int N, int nsteps, int n_kc,
    int n_rt, int xcd, float4_t* __restrict__ partials) {
    // the other k-groups' sums of each accumulator unit (rb, j): [unit][source][lane]
    extern __shared__ __align__(16) char gemm_smem[];
    float4_t* red = reinterpret_cast<float4_t*>(gemm_smem);
    int hb, jj;
    xcd_split(blockIdx.x, GEMV_NCG * n_kc * n_rt, xcd, hb, jj);
    const int cg = jj & (GEMV_NCG - 1), jr = jj / GEMV_NCG;
    const int kc = jr / n_rt, rt = jr - kc * n_rt;
    const int lane = threadIdx.x & (WAVE - 1);
    const int kg = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / WAVE));
    const int g = lane >> 4, c = lane & 15, p = c & 3, n16 = N / 16;
    const int s0 = kc * nsteps, ns = min(nsteps, K / STEP_K - s0);
    const int row0 = rt * 16 * RB;

    gptr_t<uint32_t> tp = as_global(reinterpret_cast<const uint32_t*>(trellis)) +
                          ((size_t)(4 * (s0 + kg) + g) * n16 + 8 * hb + 4 * cg + (c >> 2)) * (8 * BITS);
    const size_t tstep = (size_t)4 * GEMM_NKG * n16 * (8 * BITS);
    // A unit ((s * 4 + g) * 4 + r) * Rp + row, through a buffer resource of the
    // rotated input's size: past the wave's last step the offset lies beyond
    // it, so the prefetch reads nothing and the loop needs no branch around it
    const uint32_t abytes = (uint32_t)((size_t)K / STEP_K * 16 * Rp * 16);
    const __amdgpu_buffer_rsrc_t ar = __builtin_amdgcn_make_buffer_rsrc(const_cast<u32x4_t*>(xd), (short)0, (int)abytes, 0x00020000);
    uint32_t av = (uint32_t)((((s0 + kg) * 16 + 4 * g) * Rp + row0 + c) * 16);
    const uint32_t astep = (uint32_t)(16 * GEMM_NKG * Rp * 16);

    float4_t acc[RB][4];
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
        for (int q = 0; q < 4; ++q) acc[rb][q] = float4_t{0.f, 0.f, 0.f, 0.f};

    QuarterTile<BITS> t0, t1;
    half8_t A[4][RB];
    auto load_a = [&](int r) {
        const uint32_t v = av + (uint32_t)(r * Rp * 16);
#pragma unroll
        for (int rb = 0; rb < RB; ++rb)
            A[r][rb] = __builtin_bit_cast(half8_t, __builtin_amdgcn_raw_buffer_load_b128(ar, v + 256 * rb, 0, 0));
    };
    // One step; the next step's A is requested k-group by k-group as this step's is used up.
    auto step = [&](const QuarterTile<BITS>& t, bool more) {
        av = more ? av + astep : 0x80000000u;
        static_for<4>([&](auto RI) {
            constexpr int r = decltype(RI)::value;
            static_for<4>([&](auto JI) {
                constexpr int q = decltype(JI)::value, n = quarter_col(q);
                constexpr int T0 = 32 * (n & 7) + 8 * r + 4 * (n >> 3);
                u32x4_t b;
                b[0] = decode_quarter<BITS, CB, T0 + 0>(t);
                b[1] = decode_quarter<BITS, CB, T0 + 1>(t);
                b[2] = decode_quarter<BITS, CB, T0 + 2>(t);
                b[3] = decode_quarter<BITS, CB, T0 + 3>(t);
#pragma unroll
                for (int rb = 0; rb < RB; ++rb)
                    acc[rb][q] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A[r][rb], __builtin_bit_cast(half8_t, b),
                                                                        acc[rb][q], 0, 0, 0);
            });
            __builtin_amdgcn_sched_barrier(0);         // the loads stay behind the MFMAs that read their registers
            load_a(r);
        });
    };
    if (kg < ns) {
        load_quarter<BITS>(t0, tp, p);
#pragma unroll
        for (int r = 0; r < 4; ++r) load_a(r);
        for (int s = kg; s < ns; s += GEMM_NKG) {
            const bool more = s + GEMM_NKG < ns;
            tp += more ? tstep : 0;                    // past the end the last tile again
            load_quarter<BITS>(t1, tp, p);
            step(t0, more);
            t0 = t1;
        }
    }

    // Unit (rb, j) is finished by k-group j + 4 (rb & 1); the others hand it their sums.
    static_for<4>([&](auto JI) {
        constexpr int j = decltype(JI)::value;
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) {
            const int own = j + 4 * (rb & 1);
            if (kg != own)
                red[((rb * 4 + j) * (GEMM_NKG - 1) + (kg < own ? kg : kg - 1)) * WAVE + lane] = acc[rb][j];
        }
    });
    __syncthreads();
    static_for<4>([&](auto JI) {
        constexpr int j = decltype(JI)::value;
        if ((kg & 3) == j) {
#pragma unroll
            for (int rb = 0; rb < RB; ++rb) {
                if ((rb & 1) != kg / 4) continue;
                const float4_t* s = red + (rb * 4 + j) * (GEMM_NKG - 1) * WAVE + lane;
                float4_t v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int k = 0; k < GEMM_NKG; ++k)             // k-group order
                    v += k == kg ? acc[rb][j] : s[(k < kg ? k : k - 1) * WAVE];
                partials[gemm_partial_unit(hb, kc, n_kc, rt * RB + rb, n_rt * RB, j, cg) * WAVE + lane] = v;
            }
        }
    });
}

// Two consecutive outputs at any 2-byte alignment.
__device__ __forceinline__ void store_out2(void* out, size_t idx, int kind, float a, float b) {
    if (kind == OUT_F32) {
        reinterpret_cast<float*>(out)[idx] = a;
        reinterpret_cast<float*>(out)[idx + 1] = b;
    } else {
        typedef uint32_t __attribute__((aligned(2))) u32_u;
        const uint32_t lo = kind == OUT_F16 ? f32_to_f16_bits(a) : f32_to_bf16_rne(a);
        const uint32_t hi = kind == OUT_F16 ? f32_to_f16_bits(b) : f32_to_bf16_rne(b);
        *reinterpret_cast<u32_u*>(reinterpret_cast<uint16_t*>(out) + idx) = lo | (hi << 16);
    }
}

// Finish of (128-column block, 16-row block): the k-chunks' partial tiles
// summed in chunk order, output Hadamard, svh, store.  Wave cg holds columns
// 64 cg .. 64 cg + 63 in the accumulators' layout: stages h = 1, 2, 16, 32 run
// between lanes (DPP), 4 and 8 in registers, 64 when the rows are read back
// from LDS in storing order.
template <int DUMMY = 0>
__global__ __launch_bounds__(2 * WAVE) void gemm_finish_kernel(const float4_t* __restrict__ partials,
                                                               const uint16_t* __restrict__ svh,
                                                               void* __restrict__ out, int out_kind, int R, int N,
                                                               int n_kc, int n_rb, int xcd) {
    __shared__ float buf[MAX_ROWS * GEMV_RED_LD];
    int hb, rb;
    xcd_split(blockIdx.x, (R + 15) / 16, xcd, hb, rb);
    const int lane = threadIdx.x & (WAVE - 1), cg = threadIdx.x / WAVE;
    const int g = lane >> 4, c = lane & 15, p = c & 3;
    float4_t v[4];
    {
        const float4_t* s = partials + gemm_partial_unit(hb, 0, n_kc, rb, n_rb, 0, cg) * WAVE + lane;
        const size_t kstride = (size_t)n_rb * 4 * GEMV_NCG * WAVE;
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = float4_t{0.f, 0.f, 0.f, 0.f};
        constexpr int BATCH = 4;
        for (int k0 = 0; k0 < n_kc; k0 += BATCH) {
            float4_t t[BATCH][4];
#pragma unroll
            for (int k = 0; k < BATCH; ++k)
                if (k0 + k < n_kc)
#pragma unroll
                    for (int j = 0; j < 4; ++j) t[k][j] = s[(k0 + k) * kstride + j * GEMV_NCG * WAVE];
#pragma unroll
            for (int k = 0; k < BATCH; ++k)
                if (k0 + k < n_kc)
#pragma unroll
                    for (int j = 0; j < 4; ++j) v[j] += t[k][j];
        }
    }
    const float s1 = (c & 1) ? -1.f : 1.f, s2 = (c & 2) ? -1.f : 1.f;
    const float s4 = (c & 4) ? -1.f : 1.f, s8 = (c & 8) ? -1.f : 1.f;
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) v[j][i] = bfly(v[j][i], dpp_xor<1>(v[j][i]), s1);
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) v[j][i] = bfly(v[j][i], dpp_xor<2>(v[j][i]), s2);
    // units 0..3 are columns p + 0, 8, 4, 12: h = 4 pairs (0, 2), (1, 3), h = 8 pairs (0, 1), (2, 3)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const float4_t a = v[j], b = v[j + 2];
        v[j] = a + b;
        v[j + 2] = a - b;
    }
#pragma unroll
    for (int j = 0; j < 4; j += 2) {
        const float4_t a = v[j], b = v[j + 1];
        v[j] = a + b;
        v[j + 1] = a - b;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) v[j][i] = bfly(v[j][i], dpp_xor<4>(v[j][i]), s4);
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) v[j][i] = bfly(v[j][i], dpp_xor<8>(v[j][i]), s8);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        float* d = buf + (4 * g + i) * GEMV_RED_LD + 64 * cg + 16 * (c >> 2) + p;
#pragma unroll
        for (int j = 0; j < 4; ++j) d[quarter_col(j)] = v[j][i];
    }
    __syncthreads();
    // a half-wave per row: lane l of it columns 2l, 2l + 1 and 64 + 2l, 65 + 2l
    const int l = lane & 31, col = 128 * hb + 2 * l;
    float w[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) w[q] = f16_bits_to_f32(svh[col + (q & 1) + 64 * (q >> 1)]);
#pragma unroll
    for (int m0 = 0; m0 < MAX_ROWS; m0 += 4) {
        const int m = m0 + 2 * cg + (lane >> 5), row = 16 * rb + m;
        if (row < R) {
            const float2 a = *reinterpret_cast<const float2*>(buf + m * GEMV_RED_LD + 2 * l);
            const float2 b = *reinterpret_cast<const float2*>(buf + m * GEMV_RED_LD + 64 + 2 * l);
            store_out2(out, (size_t)row * N + col, out_kind, (a.x + b.x) * HAD_NORM * w[0], (a.y + b.y) * HAD_NORM * w[1]);
            store_out2(out, (size_t)row * N + col + 64, out_kind, (a.x - b.x) * HAD_NORM * w[2],
                       (a.y - b.y) * HAD_NORM * w[3]);
        }
    }
}

// ---------------------------------------------------------------- same-input fan
//
// Several matrices that read the same input x (same K, each with its own
// suh/svh, N, bit width and output): one launch of partial sums over all of
// them per bit width present, then one split-K finish launch over all of them.
// A matrix's items and sums are those of exl3_gemm at the fan's k-chunking.
// Reference counterpart: exl3_mgemm with a broadcast A (bszm_in == 1),
// recipe-lna/vllm_exl3_exl3.py.lna:546-613.

constexpr int MAX_FAN = 8;

struct FanParams {
    const uint16_t* x;
    int R, K, nsteps, n_kc, nkg, count, out_kind;
    const int16_t* trellis[MAX_FAN];
    const uint16_t* suh[MAX_FAN];
    const uint16_t* svh[MAX_FAN];
    void* out[MAX_FAN];
    float* partials[MAX_FAN];
    int N[MAX_FAN];
    int bits[MAX_FAN];
    int xcd;                    // items and finish keyed by the fan's column block (xcd_split)
    int hb0[MAX_FAN + 1];       // 128-column blocks: member j owns [hb0[j], hb0[j+1])
};

__device__ __forceinline__ int fan_member(const FanParams& P, int hb) {
    int j = 0;
    while (j + 1 < P.count && hb >= P.hb0[j + 1]) ++j;
    return j;
}

// Items of the members with bit width BITS; the other members' items return
// at once (one launch per width present).
template <int BITS, int CB, int RB>
__global__ __launch_bounds__(WAVE * GEMV_NCG * GEMV_MAX_NKG) void gemv_fan_kernel(FanParams P) {
    extern __shared__ __align__(16) char gemv_smem[];
    // the members' column blocks in order are the fan's column blocks
    int hb, kc;
    xcd_split(blockIdx.x, P.n_kc, P.xcd, hb, kc);
    const int j = fan_member(P, hb);
    if (P.bits[j] != BITS) return;
    gemv_item<BITS, CB, RB>(P.x, P.trellis[j], P.suh[j], P.svh[j], P.out[j], P.out_kind, P.R, P.K, P.N[j], P.nsteps,
                            P.n_kc, hb - P.hb0[j], kc, P.partials[j], gemv_smem);
}

template <int BATCH>
__global__ __launch_bounds__(64) void gemv_fan_reduce_kernel(FanParams P) {
    int hb, m;
    xcd_split(blockIdx.x, P.R, P.xcd, hb, m);
    const int j = fan_member(P, hb);
    gemv_reduce_block<BATCH>(P.partials[j], P.svh[j], P.out[j], P.out_kind, P.R, P.N[j], P.n_kc, hb - P.hb0[j], m);
}

// ---------------------------------------------------------------- per-bit-width launchers

struct DequantArgs {
    const int16_t* trellis; int k16, n16; int codebook;
    const uint16_t* suh; const uint16_t* svh; uint16_t* out; hipStream_t stream;
    bool nk;                 // write [n][k] instead of [k][n]
};
struct GemvArgs {
    const uint16_t* x; const int16_t* trellis; const uint16_t* suh; const uint16_t* svh;
    void* out; int out_kind; int R, K, N; GemvPlan plan; int codebook;
    float* partials; hipStream_t stream;
};

struct GemmArgs {
    const u32x4_t* xd; const int16_t* trellis; int K, N; GemmPlan plan; int codebook; float4_t* partials; bool xcd;
    hipStream_t stream;
};

// Defined in exl3_dense_inst.hip, one translation unit per BITS.
template <int BITS> int launch_dequant(const DequantArgs& a);
template <int BITS> int launch_gemv(const GemvArgs& a);
template <int BITS> int launch_gemm(const GemmArgs& a);
template <int BITS> int launch_gemv_fan(const FanParams& P, int codebook, hipStream_t stream);

}  // namespace exl3
