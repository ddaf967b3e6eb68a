// Prefill GEMM on MFMA for gfx950: C[M][N] = A[M][I] . Q[I][N] with Q decoded
// from the trellis on the fly, FP16 operands, FP32 accumulation.  This is the
// narrow core: calls of fewer than 256 rows, and layers whose width is not a
// multiple of 256 (reference src/wmma_tiled.hip:87-269, src/gemm.hip:15-76);
// the rest run the wide core (gemm_wide.hpp).
//
// Bound: the trellis decode (VALU) and, with few rows, latency.  K splits in
// narrow_splits parts (a function of the layer only); a workgroup of four waves
// owns 64 output columns and 16 TM rows of one part, small enough (32 KiB of
// LDS) for two to five workgroups per CU, so that one's decode covers another's
// barrier and loads.  Per stage of 128 channels:
//   * every lane decodes one chunk: wave w the two input blocks of K32 step w,
//     lanes 0-31 block 2w, lanes 32-63 block 2w + 1 (8 lanes per 16-column tile,
//     four tiles), and stores its column fragments in MFMA B-operand order in
//     LDS (double-buffered);
//   * the four waves multiply as WM x (4 / WM): TM / WM row tiles by WM column
//     tiles each, B fragments from LDS, A fragments from global memory (the L1
//     serves the waves that share them) one stage ahead, in MFMA A-operand
//     order, which the input-stage kernel wrote: one coalesced 16-byte load per
//     lane and fragment.  WM balances the two sources: more waves along M read
//     fewer A fragments twice and more B ones;
//   * raw core rows go to planes[split][M][N] whatever the split count; in a pass
//     of one 16-row block the last workgroup of a 128-column group folds them and
//     applies the output stage itself, otherwise a second launch does
//     (plane_finish_kernel).
// Per-output accumulation: MFMA K32 steps in ascending K from +0 (the order
// inside one MFMA step is the hardware's), then the planes in ascending split
// order from +0; so a row has the same bits in every such call.
//
// Measured against 128 x 128 and 256 x 128 tiles of the same order (64 KiB of
// LDS, two waves along each dimension; 320 workgroups on 5120^2 that multiplied
// 128 rows whatever M was), prepared plans back to back on one buffer, same bits:
// 5120^2 K5 M = 16 / 24 / 64 / 128 / 200 23.7 / 24.5 / 27.6 / 30.8 / 40.7 -> 13.6 /
// 15.1 / 19.4 / 24.5 / 30.0 us, 4096 -> 12288 K6 29.0 / 29.4 / 32.1 / 35.8 / 50.4 ->
// 16.6 / 18.6 / 23.9 / 31.1 / 41.9 us, 1152 -> 5120 K4 M = 16 / 128 25.2 / 30.2 ->
// 11.8 / 16.5 us; 5120 -> 1152 K4 M = 512 / 4096 31.6 / 142.5 -> 24.8 / 120.6 us.
//
// MFMA 16x16x32 f16 operand layout (lane l, e = 0..7 / 0..3):
//   A: A[l % 16][8 (l / 16) + e]      B: B[8 (l / 16) + e][l % 16]
//   D: D[4 (l / 16) + e][l % 16]
#pragma once
#include <type_traits>

#include "backend.hpp"
#include "gemv_kernel.hpp"
#include "stages.hpp"

namespace stx {

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef float float4_t __attribute__((ext_vector_type(4)));

struct GemmArgs {
    const uint32_t* trellis;
    const uint16_t* svh;
    const float* bias;
    const _Float16* afrag;    // core input in fragment order: [ceil(M/16)][I/32][64 lanes][8]
    uint64_t afrag_bytes;
    float* y;                 // [M][N]
    uint32_t M, I, N;
    float alpha, beta;
    uint32_t col_block0;      // wide kernel: first column block of the launch,
    uint32_t col_blocks;      // column blocks launched,
    uint32_t tiles;           // and tiles (column blocks x row blocks)
    // Wide kernel K-split handoff (x > 0): x tiles of the launch split at half
    // of K between a head and a tail workgroup, 256 q whole tiles.
    uint32_t q, x;
    float* handoff;           // [x][8 waves][128 accumulators][64 lanes]
    uint32_t* flags;          // [x], 0 at launch; narrow kernel with the fold: arrivals per 128-column group
    uint32_t poll_limit;      // tail's polls before it takes a tile over
    // K split: `splits` workgroups per tile (narrow kernel: grid z, I/splits
    // channels each; wide kernel: grid y, stage ranges) write their raw core
    // rows to planes[s][M][N], folded in ascending s from +0 before the output
    // stage.
    uint32_t splits;
    float* planes;
#if STX_STAGE_CLOCK
    // Instrumented build only: per-wave phase cycle records of the wide
    // kernel, [workgroup][8 waves][16] (null: none written).
    unsigned long long* clock;
#endif
};

// Byte offset of the A fragment (row block rb, 32-channel block kb) of lane l.
__host__ __device__ __forceinline__ uint64_t afrag_offset(uint32_t rb, uint32_t kb, uint32_t I, uint32_t lane) {
    return ((uint64_t(rb) * (I / 32) + kb) * 64 + lane) * 16;
}

constexpr int NARROW_BSTAGE_BYTES = 4 * 4 * 64 * 16;   // 4 tiles x 4 K32 steps x 64 lanes x 16 B

// Register budget: three workgroups per CU from 128 rows on (92-128 VGPRs at 128,
// so four fit), four below.  The 256-row instances take 160-168 VGPRs, and at 6, 7
// and 8 bits, whose chunks are longer, 1-10 more go to scratch (8-12, 20, 24-28
// bytes per lane); M = 200 on 4096 -> 12288 K6 / K7 / K8 41.9 / 42.6 / 43.6 us.
template <int K, int CB, int TM, bool FOLD>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(TM >= 8 ? 3 : 4)))
void gemm_narrow_kernel(const uint32_t* trellis, const _Float16* afrag, uint32_t input,
                                                         uint32_t output, uint32_t splits, uint32_t rows,
                                                         GemmArgs args) {
    // What the first loads need comes as scalar arguments, preloaded into SGPRs.
    GemmArgs a = args;
    a.trellis = trellis;
    a.afrag = afrag;
    a.I = input;
    a.N = output;
    a.splits = splits;
    a.M = rows;
    a.afrag_bytes = uint64_t((rows + 15) / 16 * 16) * input * 2;
    constexpr int WM = TM >= 8 ? 4 : TM >= 2 ? 2 : 1, WN = 4 / WM;   // waves along M and N
    constexpr int RT = TM / WM, CT = 4 / WN;              // row and column tiles per wave
    constexpr int D = RT >= 4 ? 2 : 3;                    // chunk ring: stages in flight
    // A ring: K32 steps in flight.  Four (a whole stage) up to two row tiles per
    // wave; with four, two, which leaves registers for three workgroups per CU.
    constexpr int AD = RT >= 4 ? 2 : 4;
    __shared__ __align__(16) unsigned char smem[2 * NARROW_BSTAGE_BYTES];
    const int c = blockIdx.x, mb = blockIdx.y, split = blockIdx.z;
    const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int wm = w / WN, wn = w % WN;
    const int jt = (lane >> 3) & 3, g = lane & 7, odd = lane >> 5;
    const uint32_t I = a.I, N = a.N, stages = I / 128 / a.splits, kb0 = uint32_t(split) * stages * 4;

    constexpr uint32_t tile_bytes = 32u * K;
    const uint32_t row_bytes = (N >> 4) * tile_bytes;
    const auto wrsrc = make_rsrc(reinterpret_cast<const char*>(a.trellis) +
                                     uint64_t(split) * stages * 8 * row_bytes,
                                 uint32_t(uint64_t(stages) * 8 * row_bytes));
    const auto arsrc = make_rsrc(a.afrag, uint32_t(a.afrag_bytes));
    // The lane's chunk of stage st: tile 4c + jt of block 8 st + 2w + odd.
    const uint32_t lane_off = uint32_t(2 * w + odd) * row_bytes + (4u * c + jt) * tile_bytes + g * 4u * K;
    auto load_stage = [&](Chunk<K>& dst, uint32_t st) {
        const bool live = st < stages;
        load_chunk(dst, wrsrc, lane_off + (live ? 0u : 0x80000000u), live ? st * 8u * row_bytes : 0u);
    };
    // Fragment (column n, k-group) of (tile, K32 step) -> lane 16 * kgroup + n.
    const uint32_t wr = ((jt * 4 + w) * 64 + 32 * odd + g) * 16;
    auto decode_stage = [&](Chunk<K>& src, uint32_t buf) {
        unsigned char* base = smem + buf * NARROW_BSTAGE_BYTES + wr;
        link_chunk(src, g == 0);
        auto frag = [&](auto fc, int l) {
            constexpr int F = decltype(fc)::value;
            const uint32_t f0 = as_u32(decode_pair<K, CB, 0, F>(src)), f1 = as_u32(decode_pair<K, CB, 1, F>(src));
            const uint32_t f2 = as_u32(decode_pair<K, CB, 2, F>(src)), f3 = as_u32(decode_pair<K, CB, 3, F>(src));
            *reinterpret_cast<u32x4*>(base + l * 16) = u32x4{f0, f1, f2, f3};
        };
        frag(std::integral_constant<int, 0>{}, 0);    // rows 0-7 of column g
        frag(std::integral_constant<int, 2>{}, 16);   // rows 8-15
        frag(std::integral_constant<int, 4>{}, 8);    // rows 0-7 of column g + 8
        frag(std::integral_constant<int, 6>{}, 24);   // rows 8-15
    };

    // A fragments of the wave's row tiles: slot t % AD holds K32 step t and is
    // refilled with step t + AD once consumed.  Row tiles past the padded rows
    // read out of range (zeros).
    const uint32_t rb0 = uint32_t(mb) * TM + uint32_t(wm);
    half8_t af[AD][RT];
    // A fragment is the lane's 16 bytes at a scalar offset (row tile and K32
    // step); a row tile past the padded rows takes an out-of-range lane offset
    // at scalar offset 0 instead.
    const uint32_t tiles16 = (a.M + 15) / 16;
    auto load_a = [&](half8_t (&dst)[RT], uint32_t kb32) {
#pragma unroll
        for (int i = 0; i < RT; ++i) {
            const bool live = RT == 1 || rb0 + WM * i < tiles16;   // uniform
            if constexpr (RT == 1) {   // one tile: the whole offset in the lane's (range-checked)
                dst[0] = __builtin_bit_cast(half8_t, __builtin_amdgcn_raw_buffer_load_b128(
                                                         arsrc, uint32_t(afrag_offset(rb0, kb0 + kb32, I, lane)), 0, 0));
                continue;
            }
            const uint32_t at = live ? uint32_t(afrag_offset(rb0 + WM * i, kb0 + kb32, I, 0)) : 0u;
            dst[i] = __builtin_bit_cast(half8_t, __builtin_amdgcn_raw_buffer_load_b128(
                                                     arsrc, uint32_t(lane) * 16u | (live ? 0u : 0x80000000u), at, 0));
        }
    };
    float4_t acc[RT][CT];
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int j = 0; j < CT; ++j) acc[i][j] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};

    Chunk<K> ring[D];
#pragma unroll
    for (int d = 0; d < D; ++d) load_stage(ring[d], d);
#pragma unroll
    for (int k32 = 0; k32 < AD; ++k32) load_a(af[k32], k32);
    decode_stage(ring[0], 0);
    load_stage(ring[0], D);
    __syncthreads();

    for (uint32_t st0 = 0; st0 < stages; st0 += D) {
#pragma unroll
        for (int d = 0; d < D; ++d) {
            const uint32_t st = st0 + d;
            if (st >= stages) break;
            const unsigned char* bbase = smem + (st & 1) * NARROW_BSTAGE_BYTES;
#pragma unroll
            for (int k32 = 0; k32 < 4; ++k32) {
                half8_t bf[CT];
#pragma unroll
                for (int j = 0; j < CT; ++j)
                    bf[j] = *reinterpret_cast<const half8_t*>(bbase + (((CT * wn + j) * 4 + k32) * 64 + lane) * 16);
#pragma unroll
                for (int i = 0; i < RT; ++i)
#pragma unroll
                    for (int j = 0; j < CT; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[k32 % AD][i], bf[j], acc[i][j], 0, 0, 0);
                if (k32 + AD < 4 || st + 1 < stages) load_a(af[k32 % AD], st * 4 + k32 + AD);
                if constexpr (RT >= 4) __builtin_amdgcn_sched_barrier(0);   // bounds the live fragments
            }
            if (st + 1 >= stages) break;
            const int slot = (d + 1) % D;   // compile-time after unrolling
            decode_stage(ring[slot], (st + 1) & 1);
            load_stage(ring[slot], st + 1 + D);
            __syncthreads();
        }
    }

    float* plane = a.planes + uint64_t(split) * a.M * N + 64 * c + 16 * CT * wn + (lane & 15);
    auto put_plane = [&](auto coherent) {
#pragma unroll
        for (int i = 0; i < RT; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const uint32_t row = 16 * (rb0 + WM * i) + 4 * (lane >> 4) + e;
                if (row < a.M) {
#pragma unroll
                    for (int j = 0; j < CT; ++j) {
                        float* to = plane + uint64_t(row) * N + 16 * j;
                        if constexpr (decltype(coherent)::value) store_coherent(to, acc[i][j][e]);
                        else *to = acc[i][j][e];
                    }
                }
            }
    };
    if constexpr (!FOLD) {
        put_plane(std::false_type{});
        return;
    } else {
        put_plane(std::true_type{});
        // The last of the column group's 2 S workgroups (two halves of 128
        // columns) folds the planes.  The partials are agent-scope stores,
        // complete (waited for, then a barrier) before the arrival; the last
        // arrival reads them with device-coherent loads issued after the counter
        // result, behind a barrier.
        static_assert(16 * TM == kNarrowFoldRows, "the fold serves a pass of one row block");
        __builtin_amdgcn_s_waitcnt(0);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        __syncthreads();
        int* last = reinterpret_cast<int*>(smem);
        const uint32_t cg = uint32_t(c) >> 1;
        if (tid == 0)
            *last = __hip_atomic_fetch_add(a.flags + cg, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ==
                    2 * a.splits - 1;
        __syncthreads();
        if (!*last) return;
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
        // Wave w folds rows w, w + 4, ..., P at a time, lane l columns 2l and 2l + 1:
        // each plane from +0 in ascending split order, then H32 and the output stage
        // (the order and operations of plane_finish_kernel).  Both loops run at most
        // once; written out, the 32 loads' resources are live together and SGPRs
        // spill (106 for 67; 5120^2 K5 at 16 rows 13.8 -> 14.0, 4096^2 K4 11.9 -> 12.2 us).
        constexpr int P = int(kNarrowFoldRows) / 4, SB = int(kNarrowFoldSplits);
        const uint32_t n0 = 128u * cg + 2u * uint32_t(lane);
        const uint32_t svp = ld_global(reinterpret_cast<const uint32_t*>(a.svh + n0));
        const bool has_bias = a.bias != nullptr;
        const auto rb = make_rsrc(a.bias, has_bias ? N * 4u : 0u);
        const gemv_f2_t bias = __builtin_bit_cast(gemv_f2_t, __builtin_amdgcn_raw_buffer_load_b64(rb, n0 * 4u, 0, 0));
        for (uint32_t r0 = uint32_t(w); r0 < a.M; r0 += 4 * P) {
            gemv_f2_t z[P];
#pragma unroll
            for (int i = 0; i < P; ++i) z[i] = gemv_f2_t{0.0f, 0.0f};
            for (uint32_t s0 = 0; s0 < a.splits; s0 += SB) {
                gemv_f2_t v[SB][P];
#pragma unroll
                for (int u = 0; u < SB; ++u)
#pragma unroll
                    for (int i = 0; i < P; ++i) {
                        // Past the last split or row: a valid address again, unused.
                        const uint32_t ss = s0 + u < a.splits ? s0 + u : s0;
                        const uint32_t r = r0 + 4 * i < a.M ? r0 + 4 * i : r0;
                        const auto ps = make_rsrc(a.planes + (uint64_t(ss) * a.M + r) * N, N * 4u);
                        v[u][i] = poll_pair(ps, n0 * 4u, 0);
                    }
#pragma unroll
                for (int u = 0; u < SB; ++u)
                    if (s0 + u < a.splits)
#pragma unroll
                        for (int i = 0; i < P; ++i) {
                            z[i].x = z[i].x + v[u][i].x;
                            z[i].y = z[i].y + v[u][i].y;
                        }
            }
            h32_pairs<P>(z);
#pragma unroll
            for (int i = 0; i < P; ++i) {
                if (r0 + 4 * i >= a.M) break;
                float* yr = a.y + uint64_t(r0 + 4 * i) * N + n0;
                gemv_f2_t o;
                o.x = output_value(z[i].x, uint16_t(svp), has_bias, bias.x, a.alpha, a.beta, yr);
                o.y = output_value(z[i].y, uint16_t(svp >> 16), has_bias, bias.y, a.alpha, a.beta, yr + 1);
                *(__attribute__((address_space(1))) gemv_f2_t*)(yr) = o;
            }
        }
    }
}

struct GemmLaunch {
    GemmArgs args;
    uint32_t codebook;
    uint32_t bm;              // narrow kernel: rows per workgroup (16, 32, 64, 128 or 256)
    uint32_t bn, col_blocks;  // wide kernel: tile width and column blocks launched
    hipStream_t stream;
};

template <int K>
hipError_t gemm_narrow_dispatch(const GemmLaunch& l);

// Row tiles of 16 per workgroup: 1 with the fold, 2, 4, 8 or 16 without.
#define STX_INSTANTIATE_GEMM_NARROW(K)                                                                          \
    template <>                                                                                                \
    hipError_t gemm_narrow_dispatch<K>(const GemmLaunch& l) {                                                   \
        using Fn = void (*)(const uint32_t*, const _Float16*, uint32_t, uint32_t, uint32_t, uint32_t, GemmArgs); \
        static const Fn table[5][3] = {                                                                        \
            {gemm_narrow_kernel<K, 0, 1, true>, gemm_narrow_kernel<K, 1, 1, true>, gemm_narrow_kernel<K, 2, 1, true>}, \
            {gemm_narrow_kernel<K, 0, 2, false>, gemm_narrow_kernel<K, 1, 2, false>, gemm_narrow_kernel<K, 2, 2, false>}, \
            {gemm_narrow_kernel<K, 0, 4, false>, gemm_narrow_kernel<K, 1, 4, false>, gemm_narrow_kernel<K, 2, 4, false>}, \
            {gemm_narrow_kernel<K, 0, 8, false>, gemm_narrow_kernel<K, 1, 8, false>, gemm_narrow_kernel<K, 2, 8, false>}, \
            {gemm_narrow_kernel<K, 0, 16, false>, gemm_narrow_kernel<K, 1, 16, false>, gemm_narrow_kernel<K, 2, 16, false>}}; \
        /* the fold: one row block, and planes that one round trip holds */                                    \
        if (l.bm == 16 && (l.args.M > kNarrowFoldRows || l.args.splits > kNarrowFoldSplits))                   \
            return hipErrorInvalidValue;                                                                       \
        const int ti = l.bm == 16 ? 0 : l.bm == 32 ? 1 : l.bm == 64 ? 2 : l.bm == 128 ? 3 : 4;                  \
        const dim3 grid(l.args.N / 64, (l.args.M + l.bm - 1) / l.bm, l.args.splits);                           \
        const GemmArgs& a = l.args;                                                                            \
        hipLaunchKernelGGL(table[ti][l.codebook], grid, dim3(256), 0, l.stream, a.trellis, a.afrag, a.I, a.N,   \
                           a.splits, a.M, a);                                                                  \
        return hipGetLastError();                                                                              \
    }

}  // namespace stx
