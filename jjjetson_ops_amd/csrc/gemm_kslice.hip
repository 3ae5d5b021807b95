// Mid-batch GEMM (about 17 to 1000 tokens) of Q4_0 weights x Q8_1 activations on
// gfx950 int8 matrix cores: the K range of an output tile is cut over the waves of
// one workgroup.
//
// Math is the reference's per-block epilogue (src/cuda/mm_q4_0_q8_1.cu:71-93,
// summed over K at :256-269):
//     y[m][n] = sum_b d_w[n,b] * (sumi[n,m,b] * d_x[m,b] - 8 * s_x[m,b])
// with the exact int32 block sums of v_mfma_i32_32x32x32_i8 read as fp32 through the
// 1.5*2^23 accumulator bias (mfma_q4q8_tile.hpp), two fp32 FMAs per element and block,
// and the s_x term on an f16 MFMA.
//
// What bounds it, and the design that follows
//   * A batch of tens or hundreds of tokens has too few 64- or 128-row tiles for 256
//     CUs: N=4096, K=11008, 48 tokens ran 128 workgroups of four waves, each wave
//     walking all of K, at 52 us.  Here a workgroup is WK waves that each own a
//     contiguous K slice of the SAME (32*RT rows) x (32*CT tokens) tile, so a small
//     output still fills the chip with waves (18 us).  The slices' partial sums are
//     added through LDS in slice order; no workspace, no atomics, no second launch, and
//     the result does not depend on timing.
//   * A wave shares nothing with the others inside the K loop, so there is no barrier in
//     it.  A stage (128 of K: one Q8_1 superblock) moves to the wave's own LDS with LDS
//     DMA (activations: 1 KB contiguous runs; weights: 64 nibble bytes or one 72-byte
//     run per row), is read into registers, and the DMA of the next stage starts into
//     the same bytes while this one is computed.  Direct loads of the MFMA operands
//     (16 bytes every 144 for the activation) touch a cache line per lane pair and ran
//     at half the speed (K=4096, N=14336, 64 tokens: 33 us against 22).
//   * One buffer per wave, not a ring: deeper rings hid no more latency and cost
//     residency (64 x 64 tiles, 256 tokens, N=14336, block_q4_0: 83 us with two weight
//     slots, 59 with one).
//   * The 64 x 64 forms' loop is bound by instruction issue: a wave issues a two-operand
//     VALU instruction every 5.0 clocks and a three-operand one every 6.1, a SIMD every 2.5
//     and 3.1 from two waves on, and MFMA time adds to it almost in full (K=11008,
//     N=4096, 777 tokens: 651 VALU instructions per wave and stage, 512 of them the epilogue;
//     waves are ready but not issued for 21% of their cycles and wait for 16%; MFMA busy 18%;
//     the two rounds of workgroups are 81% full).  The 32 x 32 form waits: K=11008, N=4096,
//     24 tokens is 128 workgroups, half the CUs, whose waves wait for 67% of their cycles.
//     What is minimised is instructions per 32x32 block: weights are expanded with one load of
//     two blocks per lane pair and v_permlane32_swap (no duplicated work in the two lane
//     halves), scales are widened to fp32 once per stage, d_x stays an fp32 register (a
//     v_fma_mix would issue at two thirds of the rate), and the next block's MFMA is
//     issued before the epilogue that the previous one feeds (sched_barrier: left alone,
//     the scheduler sinks it behind that epilogue, 5-10% slower).
//   * Tile shapes: kslice_pick() below.
#include <hip/hip_fp16.h>

#include <type_traits>

#include "mfma_q4q8_tile.hpp"
#include "q4q8_common.hpp"
#include "q8_1_quant.hpp"

namespace jjo {
namespace {

typedef uint32_t u32x3 __attribute__((ext_vector_type(3)));

// One wave's staging area: activations [32*CT][144], weights per row tile (split: 32 x 64
// nibble bytes and 32 x 8 scale bytes; block_q4_0: 32 rows x 6 chunks of 12 bytes at a
// 16-byte stride, the layout of a 12-byte LDS DMA), fp32 scales [RT][4][32].
template <int RT, int CT, bool SPLIT>
struct KsliceLds {
    static constexpr int kXBytes = 32 * CT * kQ8BlockBytes;
    static constexpr int kXRuns = (kXBytes + 1023) / 1024;  // the last may be half a run
    static constexpr int kWTile = SPLIT ? 2048 + 256 : 3072;
    static constexpr int kOffW = kXBytes;
    static constexpr int kOffScale = kOffW + RT * kWTile;
    static constexpr int kWave = kOffScale + RT * 512;
};

// A lane's source offsets of one row tile's weights (first row r0 below the tile's base,
// `last` the highest valid row there).
template <bool SPLIT>
__device__ __forceinline__ void kslice_offsets(uint32_t (&off)[3], int r0, int last, int nb) {
    const int lane = threadIdx.x & 63;
    if constexpr (SPLIT) {
        // lane l: row l/4 of 16, block (l%4) ^ ((row/4)%4): the 16 rows that read one block
        // then fall in 16 different 16-byte bank groups
#pragma unroll
        for (int i = 0; i < 2; ++i)
            off[i] = (uint32_t)min(r0 + 16 * i + (lane >> 2), last) * nb * 16 + 16 * ((lane & 3) ^ ((lane >> 4) & 3));
        off[2] = (uint32_t)min(r0 + (lane & 31), last) * nb * 2 + 4 * (lane >> 5);
    } else {
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            const int c = 64 * i + lane;
            off[i] = (uint32_t)min(r0 + c / 6, last) * nb * kQ4BlockBytes + 12 * (c % 6);
        }
    }
}

// One wave's K loop over stages s_beg..s_end-1 of its (32*RT rows) x (32*CT tokens) tile:
// acc = sum_b d_w/8 * (sumi * d_x) - d_w * s_x (an eighth of the result).  `stage` is the
// wave's own LDS; rows and tokens past the tile's end re-read the last valid one.
// wq / wd: per row tile, the weight run (nibble plane when split) and the scale plane at
// the tile's first row; woff: the lane's byte offsets below them (kslice_offsets).
// SPREAD: the next stage's DMA goes out one instruction per block instead of in one burst,
// where the waves' bursts queue for each other (64 x 64 tiles: 256 tokens N=4096 K=4096 18.4
// -> 16.9 us, 512 tokens N=14336 96 -> 92.5).  Smaller tiles and the experts' short slices
// need its earlier start more (E=8 top-2 FFN, 32 tokens: 225 us in a burst, 259 spread).
template <int RT, int CT, bool SPLIT, bool SPREAD>
__device__ __forceinline__ void kslice_loop(f32x16 (&acc)[RT][CT], uint8_t *stage, const uint8_t *const (&wq)[RT],
                                            const uint8_t *const (&wd)[RT], const uint32_t (&woff)[RT][3],
                                            const uint8_t *xb, size_t x_stride, uint32_t xlim, int s_beg, int s_end) {
    using L = KsliceLds<RT, CT, SPLIT>;
    const int lane = threadIdx.x & 63, l32 = lane & 31, hh = lane >> 5;
    const uint32_t stage_lds = (uint32_t)(uintptr_t)stage;
    float *wde = reinterpret_cast<float *>(stage + L::kOffScale);
    // Inline asm: the compiler would order every later LDS access behind these; their
    // completion is waited for at the top of a stage.
    constexpr int kPieces = 3 * RT + L::kXRuns;
    // One DMA instruction of a stage.  The spread form takes them in this order: the weights,
    // which come from further away, first.
    auto dma_piece = [&](int k, int s) {
        if (k >= 3 * RT) {
            const int i = k - 3 * RT;
            const uint32_t m0v = __builtin_amdgcn_readfirstlane(stage_lds + i * 1024);
            if ((i + 1) * 1024 <= L::kXBytes || lane < 32)
                asm volatile("global_load_lds_dwordx4 %0, %1"
                             :
                             : "v"(min((uint32_t)(i * 1024 + lane * 16), xlim)), "s"(xb + (size_t)s * x_stride),
                               "{m0}"(m0v)
                             : "memory");
            return;
        }
        const int rt = k / 3, i = k % 3;
        const uint32_t m0v = __builtin_amdgcn_readfirstlane(stage_lds + L::kOffW + rt * L::kWTile + i * 1024);
        if constexpr (!SPLIT)
            asm volatile("global_load_lds_dwordx3 %0, %1"
                         :
                         : "v"(woff[rt][i]), "s"(wq[rt] + (size_t)s * (4 * kQ4BlockBytes)), "{m0}"(m0v)
                         : "memory");
        else if (i < 2)
            asm volatile("global_load_lds_dwordx4 %0, %1"
                         :
                         : "v"(woff[rt][i]), "s"(wq[rt] + (size_t)s * 64), "{m0}"(m0v)
                         : "memory");
        else
            asm volatile("global_load_lds_dword %0, %1"
                         :
                         : "v"(woff[rt][i]), "s"(wd[rt] + (size_t)s * 8), "{m0}"(m0v)
                         : "memory");
    };
    // A whole stage in one burst: the activations, then the weights.
    auto dma = [&](int s) {
#pragma unroll
        for (int k = 0; k < kPieces; ++k) dma_piece((k + 3 * RT) % kPieces, s);
    };

    i32x16 bias;
#pragma unroll
    for (int v = 0; v < 16; ++v) bias[v] = (int32_t)kBiasBits;
    asm volatile("" : "+v"(bias));
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int ct = 0; ct < CT; ++ct)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[rt][ct][v] = 0.0f;

    // Order of a stage's four blocks: a lane holds blocks 2*hh and 2*hh+1 of its row, so the
    // first half-wave swap completes blocks 0 and 2, the second blocks 1 and 3.
    constexpr int kOrder[4] = {0, 2, 1, 3};
    constexpr int kJobs = 4 * RT * CT;  // 32x32 blocks of a stage
    if (s_beg < s_end) dma(s_beg);
    if constexpr (SPREAD) {
        for (int s = s_beg; s < s_end - 1; ++s) {
#define KSLICE_MORE true
#include "gemm_kslice_stage.inc"
#undef KSLICE_MORE
        }
        if (s_beg < s_end) {
            const int s = s_end - 1;
#define KSLICE_MORE false
#include "gemm_kslice_stage.inc"
#undef KSLICE_MORE
        }
    } else {
        for (int s = s_beg; s < s_end; ++s) {
#define KSLICE_MORE false
#include "gemm_kslice_stage.inc"
#undef KSLICE_MORE
        }
    }
}

template <int RT, int CT, int WK, bool SPLIT, int WAVES_PER_SIMD>
__global__ __launch_bounds__(64 * WK, WAVES_PER_SIMD) void gemm_kslice_kernel(
    const uint8_t *__restrict__ w, const uint8_t *__restrict__ xq, float *__restrict__ y, int K, int N, int M,
    int row_tiles, int tok_tiles) {
    using L = KsliceLds<RT, CT, SPLIT>;
    extern __shared__ __align__(16) uint8_t smem[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

    // Workgroups go round-robin over the 8 XCDs: each XCD takes one contiguous eighth of the
    // tiles, the token tiles of a row tile following each other, so its weights come from
    // HBM (nearly) once and no XCD gets more than one tile above the mean.
    const int tiles = row_tiles * tok_tiles, per_xcd = (tiles + 7) >> 3;
    const int tile = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
    if (tile >= tiles) return;  // uniform over the workgroup
    const int row_tile = tile / tok_tiles, tok_tile = tile % tok_tiles;
    const int n0 = row_tile * 32 * RT, m0 = tok_tile * 32 * CT;
    const int nb = K / kQK, nsb = K / kQSuper;

    f32x16 acc[RT][CT];
    const uint8_t *wq[RT], *wd[RT];
    uint32_t woff[RT][3];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        wq[rt] = w + (size_t)n0 * nb * (SPLIT ? 16 : kQ4BlockBytes);
        wd[rt] = w + ((size_t)N * 16 + (size_t)n0 * 2) * nb;  // split: the scale plane
        kslice_offsets<SPLIT>(woff[rt], 32 * rt, N - 1 - n0, nb);
    }
    kslice_loop<RT, CT, SPLIT, RT * CT == 4>(acc, smem + wave * L::kWave, wq, wd, woff, xq + (size_t)m0 * kQ8BlockBytes,
                               (size_t)M * kQ8BlockBytes, min(32 * CT, M - m0) * kQ8BlockBytes - 16,
                               (int)((int64_t)wave * nsb / WK), (int)((int64_t)(wave + 1) * nsb / WK));

    // ---- add the K slices in slice order, y[m][n] = 8 * sum ----
    __syncthreads();  // every wave is done with its staging area
    f32x4 *red = reinterpret_cast<f32x4 *>(smem);
    constexpr int kItems = RT * CT * 256;
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int ct = 0; ct < CT; ++ct)
#pragma unroll
            for (int q = 0; q < 4; ++q)
                red[wave * kItems + (rt * CT + ct) * 256 + q * 64 + lane] =
                    f32x4{acc[rt][ct][4 * q], acc[rt][ct][4 * q + 1], acc[rt][ct][4 * q + 2], acc[rt][ct][4 * q + 3]};
    __syncthreads();
    // Eight consecutive threads take the 32 rows of one token: 128 contiguous bytes of y.
    for (int it = tid; it < kItems; it += 64 * WK) {
        const int qh = it & 7, tok = (it >> 3) & 31, tile = it >> 8;
        const int src = tile * 256 + (qh >> 1) * 64 + tok + 32 * (qh & 1);
        f32x4 v = red[src];
#pragma unroll
        for (int i = 1; i < WK; ++i) v += red[i * kItems + src];
        v *= 8.0f;
        const int m = m0 + 32 * (tile % CT) + tok, n = n0 + 32 * (tile / CT) + 4 * qh;
        if (m >= M) continue;
        float *yr = y + (size_t)m * N + n;
        if (n + 3 < N) {
            *reinterpret_cast<f32x4a4 *>(yr) = v;
        } else {
#pragma unroll
            for (int k = 0; k < 4; ++k)
                if (n + k < N) yr[k] = v[k];
        }
    }
}

// ---- grouped (MoE) form: workgroups over (64-row tile, token tile of an expert) ----
// Token tiles of 32*CT routes, listed expert by expert; a tile with at most 32 routes runs
// the one-column loop.  kSwiglu: row tile x is gate rows 32x..32x+31 (first row tile) and up
// rows 32x..32x+31 (second), and instead of storing them the workgroup writes the Q8_1
// bytes of silu(gate) * up of those 32 intermediate values: one Q8_1 group per route.
// Every output element is summed in the same order in all of these forms (K slices of the
// same waves, the same order inside a slice).
template <int CT, int WK, bool SPLIT, bool kSwiglu>
__global__ __launch_bounds__(64 * WK, 2) void gemm_kslice_grouped_kernel(
    const uint8_t *__restrict__ w, const uint8_t *__restrict__ w2, const uint8_t *__restrict__ xq,
    float *__restrict__ y, uint8_t *__restrict__ midq, int K, int N, int M, int n_split,
    const int32_t *__restrict__ expert_offsets, int n_experts, const int32_t *__restrict__ route_dst) {
    constexpr int RT = 2;
    extern __shared__ __align__(16) uint8_t smem[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nb = K / kQK, nsb = K / kQSuper;

    // Tile blockIdx.y of the concatenated per-expert tile lists, 64 experts per step.
    // Ranges are clamped to [0, M]: a malformed table drops routes, it reads nothing outside.
    int t = blockIdx.y, m0 = -1, m_end = 0, expert = 0;
    for (int e0 = 0; e0 < n_experts && m0 < 0; e0 += 64) {
        const int ei = e0 + lane;
        int beg = 0, end = 0;
        if (ei < n_experts) {
            beg = min(max(expert_offsets[ei], 0), M);
            end = min(max(expert_offsets[ei + 1], beg), M);
        }
        const int tiles = (end - beg + 32 * CT - 1) / (32 * CT);
        int incl = tiles;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const int o = __shfl_up(incl, d);
            if (lane >= d) incl += o;
        }
        const int total = __shfl(incl, 63);
        if (t < total) {
            const int f = __builtin_ctzll(__ballot(incl > t));  // the expert holding tile t
            m0 = __shfl(beg, f) + (t - (__shfl(incl, f) - __shfl(tiles, f))) * (32 * CT);
            m_end = __shfl(end, f);
            expert = e0 + f;
        } else {
            t -= total;
        }
    }
    if (m0 < 0) return;  // uniform over the workgroup
    m0 = __builtin_amdgcn_readfirstlane(m0);
    m_end = __builtin_amdgcn_readfirstlane(m_end);
    expert = __builtin_amdgcn_readfirstlane(expert);

    // Row tile rt: rows r0.. of one matrix with `rows_e` rows per expert (n_split % 64 == 0,
    // so a 64-row tile of two stacked matrices lies in one of them).
    const uint8_t *wq[RT], *wd[RT];
    uint32_t woff[RT][3];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        const uint8_t *mat = w;
        int rows_e = N, r0 = blockIdx.x * 64 + 32 * rt;
        if constexpr (kSwiglu) {
            mat = rt == 0 ? w : w2;
            rows_e = n_split;
            r0 = blockIdx.x * 32;
        } else if (w2 != nullptr) {
            const bool second = r0 >= n_split;
            mat = second ? w2 : w;
            rows_e = second ? N - n_split : n_split;
            r0 -= second ? n_split : 0;
        }
        const size_t row = (size_t)expert * rows_e + min(r0, rows_e - 1);
        wq[rt] = mat + row * nb * (SPLIT ? 16 : kQ4BlockBytes);
        wd[rt] = mat + ((size_t)n_experts * rows_e * 16 + row * 2) * nb;  // split: the scale plane
        kslice_offsets<SPLIT>(woff[rt], 0, max(rows_e - 1 - r0, 0), nb);
    }
    const uint8_t *xb = xq + (size_t)m0 * kQ8BlockBytes;
    const size_t x_stride = (size_t)M * kQ8BlockBytes;
    const int s_beg = (int)((int64_t)wave * nsb / WK), s_end = (int)((int64_t)(wave + 1) * nsb / WK);
    f32x4 *red = reinterpret_cast<f32x4 *>(smem);

    auto run = [&](auto ct_tag) {
        constexpr int C = decltype(ct_tag)::value;
        const int valid = min(32 * C, m_end - m0);
        f32x16 acc[RT][C];
        kslice_loop<RT, C, SPLIT, false>(acc, smem + wave * KsliceLds<RT, C, SPLIT>::kWave, wq, wd, woff, xb, x_stride,
                                  valid * kQ8BlockBytes - 16, s_beg, s_end);
        __syncthreads();  // every wave is done with its staging area
        constexpr int kTile = C * 256, kItems = RT * kTile;
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
#pragma unroll
            for (int ct = 0; ct < C; ++ct)
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    red[wave * kItems + (rt * C + ct) * 256 + q * 64 + lane] = f32x4{
                        acc[rt][ct][4 * q], acc[rt][ct][4 * q + 1], acc[rt][ct][4 * q + 2], acc[rt][ct][4 * q + 3]};
        __syncthreads();
        auto sum = [&](int src) {
            f32x4 v = red[src];
#pragma unroll
            for (int i = 1; i < WK; ++i) v += red[i * kItems + src];
            return v * 8.0f;
        };
        // Eight consecutive threads take the 32 rows of one token.
        for (int it = tid; it < (kSwiglu ? kTile : kItems); it += 64 * WK) {
            const int qh = it & 7, tok = (it >> 3) & 31, tile = it >> 8;
            const int src = tile * 256 + (qh >> 1) * 64 + tok + 32 * (qh & 1);
            const int m = m0 + 32 * (tile % C) + tok;
            if constexpr (kSwiglu) {
                const f32x4 g = sum(src), u = sum(kTile + src);
                uint32_t ds;  // every lane of the wave is active here (the group butterfly)
                const uint32_t qv = quantize_group8(swiglu(g.x, u.x), swiglu(g.y, u.y), swiglu(g.z, u.z),
                                                    swiglu(g.w, u.w), &ds);
                if (m < m_end) {
                    const int grp = blockIdx.x & 3;  // 32-group of the superblock
                    uint8_t *blk = midq + ((size_t)(blockIdx.x >> 2) * M + m) * kQ8BlockBytes;
                    *reinterpret_cast<uint32_t *>(blk + 16 + 32 * grp + 4 * qh) = qv;
                    if (qh == 0) *reinterpret_cast<uint32_t *>(blk + 4 * grp) = ds;
                }
            } else if (m < m_end) {
                const f32x4 v = sum(src);
                const int n = blockIdx.x * 64 + 32 * (tile / C) + 4 * qh;
                float *yr = y + (size_t)(route_dst != nullptr ? route_dst[m] : m) * N + n;
                if (n + 3 < N) {
                    *reinterpret_cast<f32x4a4 *>(yr) = v;
                } else {
#pragma unroll
                    for (int k = 0; k < 4; ++k)
                        if (n + k < N) yr[k] = v[k];
                }
            }
        }
    };
    if (CT == 1 || m_end - m0 <= 32)
        run(std::integral_constant<int, 1>{});
    else
        run(std::integral_constant<int, CT>{});
}

template <int CT, int WK, bool SPLIT, bool kSwiglu>
hipError_t launch_grouped(const void *w, const void *w2, const void *xq, float *y, void *midq, int K, int N, int M,
                          int n_split, const int32_t *offsets, int n_experts, const int32_t *route_dst,
                          hipStream_t stream) {
    auto kern = gemm_kslice_grouped_kernel<CT, WK, SPLIT, kSwiglu>;
    const size_t stage = WK * (size_t)KsliceLds<2, CT, SPLIT>::kWave, red = (size_t)WK * 2 * CT * 4096;
    const size_t lds = stage > red ? stage : red;
    hipError_t e = ensure_dynamic_lds((const void *)kern, lds);
    if (e != hipSuccess) return e;
    // Upper bound on the token tiles over all experts.
    const dim3 grid(kSwiglu ? n_split / 32 : (N + 63) / 64, (M + 32 * CT - 1) / (32 * CT) + n_experts);
    hipLaunchKernelGGL(kern, grid, dim3(64 * WK), lds, stream, (const uint8_t *)w, (const uint8_t *)w2,
                       (const uint8_t *)xq, y, (uint8_t *)midq, K, N, M, n_split, offsets, n_experts, route_dst);
    return hipGetLastError();
}

template <int RT, int CT, int WK, int WAVES_PER_SIMD>
hipError_t launch(const void *w, const void *xq, float *y, int K, int N, int M, bool split, hipStream_t stream) {
    auto kern = split ? gemm_kslice_kernel<RT, CT, WK, true, WAVES_PER_SIMD>
                      : gemm_kslice_kernel<RT, CT, WK, false, WAVES_PER_SIMD>;
    const size_t stage = WK * (size_t)(split ? KsliceLds<RT, CT, true>::kWave : KsliceLds<RT, CT, false>::kWave);
    const size_t red = (size_t)WK * RT * CT * 4096, lds = stage > red ? stage : red;
    hipError_t e = ensure_dynamic_lds((const void *)kern, lds);
    if (e != hipSuccess) return e;
    const int64_t rows = ((int64_t)N + 32 * RT - 1) / (32 * RT), toks = ((int64_t)M + 32 * CT - 1) / (32 * CT);
    const int64_t grid = (rows * toks + 7) / 8 * 8;  // kslice_accepts bounds it
    hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(64 * WK), lds, stream, (const uint8_t *)w,
                       (const uint8_t *)xq, y, K, N, M, (int)rows, (int)toks);
    return hipGetLastError();
}

// The tile shapes with their estimated time: a launch runs in rounds of `resident` workgroups
// per CU; a round costs round_us + stage_us per 128-value stage, a (last) round of at most one
// workgroup per CU alone_us + alone_stage_us per stage, of which `idle` is left when the chip is
// nearly empty.  Fitted to K=128..14336, N=256..151936, 17..3072 tokens, the mean of the two
// layouts (they differ by 2-6%, and one table gives both the same shape and so the same bits):
// an estimate is off by 7-10% (one standard deviation), 15-20% for one in twenty.
struct Shape {
    int rt, ct, waves, resident;
    double fixed, round_us, stage_us, alone_us, alone_stage_us, idle;
};
constexpr Shape kShapes[] = {
    {1, 1, 8, 2, 2.45, 1.26, 0.238, 0.777, 0.151, 0.812},  // N=4096, K=4096, 48 tokens: 8.6 / 8.2 us
    {1, 2, 8, 1, 1.83, 2.14, 0.225, 2.14, 0.225, 1.0},     // 100 tokens: 11.7 / 11.3
    {2, 2, 8, 1, 2.55, 2.67, 0.362, 2.67, 0.365, 1.0},     // N=8192, 128 tokens: 17.8 / 17.2
    {2, 2, 4, 2, 2.31, 2.76, 0.682, 2.76, 0.394, 1.0},     // N=4096, 512 tokens: 27.7 / 27.1
};

int64_t shape_tiles(const Shape &s, int N, int M) {
    return (((int64_t)N + 32 * s.rt - 1) / (32 * s.rt)) * (((int64_t)M + 32 * s.ct - 1) / (32 * s.ct));
}

}  // namespace

// A launch holds less than 2^32 threads in x: 2^23 workgroups of eight waves, which one tile
// per 32 rows and tokens reaches at N = 2^28, 17 tokens.
bool kslice_accepts(int shape, int K, int N, int M) {
    if (shape < 0 || shape >= (int)(sizeof(kShapes) / sizeof(kShapes[0])) || M > 65535 || K >= kMaxTileK) return false;
    const Shape &s = kShapes[shape];
    return (shape_tiles(s, N, M) + 7) / 8 * 8 * 64 * s.waves < 1LL << 32;
}

int kslice_pick(int K, int N, int M, double *us) {
    const int64_t cus = device_cu_count();
    int best = 0;
    for (int i = 0; i < (int)(sizeof(kShapes) / sizeof(kShapes[0])); ++i) {
        const Shape &s = kShapes[i];
        const int64_t g = shape_tiles(s, N, M), slots = s.resident * cus, rem = g % slots;
        const double stages = K / kQSuper, round = s.round_us + s.stage_us * stages;
        const double busy = g < cus ? (double)g / cus : 1.0;
        const double alone = s.alone_us + s.alone_stage_us * stages * (s.idle + (1.0 - s.idle) * busy);
        const double t = s.fixed + (double)(g / slots) * round + (rem == 0 ? 0.0 : rem > cus ? round : alone);
        if (i == 0 || t < *us) {
            best = i;
            *us = t;
        }
    }
    return best;
}

hipError_t launch_gemm_kslice(const void *w, const void *xq, float *y, int K, int N, int M, bool split, int shape,
                              hipStream_t stream) {
    if (!kslice_accepts(shape, K, N, M)) return hipErrorInvalidValue;
    switch (shape) {
        case 0: return launch<1, 1, 8, 4>(w, xq, y, K, N, M, split, stream);
        case 1: return launch<1, 2, 8, 2>(w, xq, y, K, N, M, split, stream);
        case 2: return launch<2, 2, 8, 2>(w, xq, y, K, N, M, split, stream);
        default: return launch<2, 2, 4, 2>(w, xq, y, K, N, M, split, stream);
    }
}

hipError_t launch_gemm_kslice_grouped(const void *w, const void *w2, const void *xq, float *y, void *midq, int K,
                                      int N, int M, int n_split, const int32_t *offsets, int n_experts,
                                      const int32_t *route_dst, bool split, int cols, hipStream_t stream) {
    // Four waves: two workgroups share a CU, three at 32 routes with SwiGLU (167 registers;
    // 170 without), and an expert's ragged last tile ends sooner than with eight (E=64
    // top-8, 100 tokens, FFN: 137 us against 195).
    auto go = [&](auto ct, auto sp, auto sw) {
        return launch_grouped<decltype(ct)::value, 4, decltype(sp)::value, decltype(sw)::value>(
            w, w2, xq, y, midq, K, N, M, n_split, offsets, n_experts, route_dst, stream);
    };
    auto with_layout = [&](auto ct, auto sw) {
        return split ? go(ct, std::true_type{}, sw) : go(ct, std::false_type{}, sw);
    };
    auto with_cols = [&](auto sw) {
        return cols == 1 ? with_layout(std::integral_constant<int, 1>{}, sw)
                         : with_layout(std::integral_constant<int, 2>{}, sw);
    };
    return midq != nullptr ? with_cols(std::true_type{}) : with_cols(std::false_type{});
}

}  // namespace jjo
