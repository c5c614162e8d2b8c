// Fit-side kernels for MI355X (gfx950): max|X|, batched symmetric Gram, projection onto a
// stored fp16 basis, direct residual / source energies, column extrema and the 8-bit quantizer.
//
// Reference: reelcache/gpu_fitting.py (gram_bases :276-295), reelcache/rank_method.py
// (_symmetric_gram :634-638), reelcache/factorization.py (project_onto_basis :318-434,
// measure_source_energy :692-724), reelcache/node_packets.py (quantize_device :155-173),
// reelcache/_hevc.py (quantize_coefficients :445-472).
//
// Arithmetic contract:
//   * Gram: exact products (16-bit sources on 16-bit MFMA, whose products are exact in fp32;
//     fp32 sources on fp32 MFMA), fp32 accumulation, exactly symmetric output.
//   * Projection P = X Q^T and the reconstruction P Q of the residual: operands converted
//     exactly to FP64, products and sums on v_mfma_f64_16x16x4f64, P rounded once to fp32.
//     The FP64 sum makes P the correctly rounded fp32 value of the exact dot product except
//     within ~1e-13 relative of a rounding boundary, i.e. independent of summation order.
//   * Energies: FP64 sums of (x - r)^2 and x^2 over partials of 16 rows and a part of the channels, totalled in
//     one order and divided by s^2.
//   * P, energies and span traces of a matrix have the same bits in every batch: the launch shape depends on
//     the batch, the order of the sums only on the matrix.
//   * Quantizer: FP64 (v - offset) / scale, round half to even, clamp to [0, 255].
#include <algorithm>
#include <type_traits>

#include "common.h"

namespace rch {
namespace {

constexpr int kThreads = 256;

template <int DT>
constexpr int esize() {
    return DT == RCH_DT_F32 ? 4 : 2;
}

// 16-bit element bits -> float.
template <int DT>
__device__ __forceinline__ float half_bits(uint32_t bits) {
    if constexpr (DT == RCH_DT_BF16) {
        return __uint_as_float(bits << 16);
    } else {
        return static_cast<float>(__builtin_bit_cast(_Float16, static_cast<uint16_t>(bits)));
    }
}

// Order-preserving unsigned key of an fp32 value (larger value -> larger key).
__device__ __forceinline__ uint32_t order_key(float v) {
    const uint32_t u = __float_as_uint(v);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

// Buffer over rows [r0, rows) of a source matrix (empty when r0 >= rows).
template <int DT>
__device__ __forceinline__ __amdgpu_buffer_rsrc_t source_rows(const rch_fit_matrix* M, int channels, int64_t r0) {
    constexpr int E = esize<DT>();
    const int64_t left = M->rows - r0;
    return make_rsrc(M->src_ptr + r0 * M->src_stride * E, left > 0 ? ((left - 1) * M->src_stride + channels) * E : 0);
}

// ---------------------------------------------------------------------------------------------
// max|X|: workgroup (row tile, matrix), one unsigned atomic max of the fp32 bits per workgroup.
// HBM-bound: the absolute values compare as integers in their own width (two 16-bit values per
// v_pk_max_u16), only the maximum is widened; four rows per wave at a time, lanes along the row.  The
// keys of a batch share cache lines, where the atomics queue at about 13 ns each, so a tile is as many
// 16-row sets as leave about kAbsmaxGroups workgroups.
// ---------------------------------------------------------------------------------------------

constexpr int kAbsmaxRows = 16, kAbsmaxGroups = 600, kAbsmaxSets = 32;

template <int DT>
__global__ void __launch_bounds__(kThreads) absmax_kernel(const rch_fit_matrix* __restrict__ mats, int channels, int sets) {
    const rch_fit_matrix* M = mats + blockIdx.y;
    const int64_t first = static_cast<int64_t>(blockIdx.x) * sets * kAbsmaxRows;
    if (first >= M->rows) return;
    constexpr int E = esize<DT>(), kLoads = DT == RCH_DT_F32 ? 2 : 1, kRows = kAbsmaxRows / (kThreads / 64);
    const int groups = channels / 8;  // 8 elements per item
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const uint32_t row_bytes = static_cast<uint32_t>(M->src_stride * E);
    typedef unsigned short us2 __attribute__((ext_vector_type(2)));
    uint32_t m = 0;
    us2 pair = {0, 0};
    for (int set = 0; set < sets; ++set) {
        // Rows past the end read zeros.
        const __amdgpu_buffer_rsrc_t src = source_rows<DT>(M, channels, first + set * kAbsmaxRows);
        for (int g = lane; g < groups; g += 64) {
            u4 w[kRows][kLoads];
#pragma unroll
            for (int r = 0; r < kRows; ++r)
#pragma unroll
                for (int q = 0; q < kLoads; ++q)
                    w[r][q] = __builtin_amdgcn_raw_buffer_load_b128(
                        src, static_cast<uint32_t>(kRows * wave + r) * row_bytes + static_cast<uint32_t>(8 * g * E + 16 * q), 0, 0);
#pragma unroll
            for (int r = 0; r < kRows; ++r)
#pragma unroll
                for (int q = 0; q < kLoads; ++q)
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        if constexpr (DT == RCH_DT_F32) {
                            const uint32_t bits = w[r][q][j] & 0x7fffffffu;
                            m = bits > m ? bits : m;
                        } else {
                            pair = __builtin_elementwise_max(pair, __builtin_bit_cast(us2, w[r][q][j] & 0x7fff7fffu));
                        }
                    }
        }
    }
    if constexpr (DT != RCH_DT_F32) m = __float_as_uint(half_bits<DT>(pair[0] > pair[1] ? pair[0] : pair[1]));
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) {
        const uint32_t o = __shfl_xor(m, d);
        m = o > m ? o : m;
    }
    __shared__ uint32_t part[kThreads / 64];
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < kThreads / 64; ++w) m = part[w] > m ? part[w] : m;
        atomicMax(reinterpret_cast<unsigned int*>(M->absmax_ptr), m);  // vector atomic
    }
}

// ---------------------------------------------------------------------------------------------
// Gram G = X^T X.  Workgroup = one 256 x 256 tile (ti >= tj) of one matrix, 16 waves: wave w
// computes the 64 x 64 quadrant (w / 4, w % 4) as 2 x 2 MFMA 32x32 blocks (on a diagonal tile
// the quadrants above the diagonal are mirrors and are skipped), and stages a quarter of the
// step's rows for 128 channels of one panel.  Rows are staged 32 per step into LDS as
// [channel][row]: each lane loads a channel pair of 8 rows, coalesced along the row, and writes
// the two channels' row runs, so that an MFMA operand (8 consecutive rows of one channel for
// 16-bit sources, 16 for fp32) is one or four 16-byte LDS reads.  Register-prefetched two steps
// ahead, double-buffered LDS, one barrier per step.
//
// The 21 tiles of a 1536-channel matrix run on one XCD (xcd_unit) and sweep the rows together,
// so each row band of X is fetched from HBM about once and then read from that XCD's L2 by the
// six tiles of each panel.  Every output element sums its products in row order, 16 rows (2 for
// fp32) per MFMA, so the result does not depend on the tile size or the rows per step.
// ---------------------------------------------------------------------------------------------

constexpr int kGramTile = 256;
constexpr int kGramThreads = 1024;

// Rows staged per step (a wave stages a quarter of them).  Measured on MI355X, 32-row steps with
// loads two steps ahead beat 64-row steps (which leave registers for one step ahead only).
template <int DT>
constexpr int gram_rows() {
    return 32;
}

template <int DT>
constexpr int gram_pitch() {
    return gram_rows<DT>() * esize<DT>() + 16;  // bytes per staged channel
}

template <int DT>
struct GramStage {
    typedef typename std::conditional<DT == RCH_DT_F32, u2, uint32_t>::type word;
    word d[gram_rows<DT>() / 4];  // rows r0 .. of this lane's channel pair
};

template <int DT>
__device__ __forceinline__ void gram_load(GramStage<DT>& st, const rch_fit_matrix* M, int channels, int64_t r0, int c) {
    constexpr int E = esize<DT>();
    const __amdgpu_buffer_rsrc_t src = source_rows<DT>(M, channels, r0);
    const uint32_t offset = c < channels ? static_cast<uint32_t>(c * E) : kOutOfRange;
    const uint32_t row_bytes = static_cast<uint32_t>(M->src_stride * E);
#pragma unroll
    for (int r = 0; r < gram_rows<DT>() / 4; ++r) {
        if constexpr (DT == RCH_DT_F32)
            st.d[r] = __builtin_amdgcn_raw_buffer_load_b64(src, offset + r * row_bytes, 0, 0);
        else
            st.d[r] = __builtin_amdgcn_raw_buffer_load_b32(src, offset + r * row_bytes, 0, 0);
    }
}

// The stage's two channels, each as a run of rows/4 consecutive rows at row offset
// group * rows / 4 of the channel's staged row block.
template <int DT>
__device__ __forceinline__ void gram_store(const GramStage<DT>& st, unsigned char* tile, int lane, int group) {
    constexpr int P = gram_pitch<DT>();
    unsigned char* c0 = tile + (2 * lane) * P;
    unsigned char* c1 = c0 + P;
    if constexpr (DT == RCH_DT_F32) {
        static_assert(gram_rows<DT>() == 32, "fp32 stages hold 8 rows per lane");
        const u4 a0 = {st.d[0][0], st.d[1][0], st.d[2][0], st.d[3][0]};
        const u4 a1 = {st.d[4][0], st.d[5][0], st.d[6][0], st.d[7][0]};
        const u4 b0 = {st.d[0][1], st.d[1][1], st.d[2][1], st.d[3][1]};
        const u4 b1 = {st.d[4][1], st.d[5][1], st.d[6][1], st.d[7][1]};
        *reinterpret_cast<u4*>(c0 + 32 * group) = a0;
        *reinterpret_cast<u4*>(c0 + 32 * group + 16) = a1;
        *reinterpret_cast<u4*>(c1 + 32 * group) = b0;
        *reinterpret_cast<u4*>(c1 + 32 * group + 16) = b1;
    } else {
        constexpr int kRuns = gram_rows<DT>() / 32;  // 8-row runs (16 bytes) per lane and channel
        static_assert(kRuns >= 1 && 8 * kRuns == sizeof(st.d) / sizeof(st.d[0]), "stage rows");
#pragma unroll
        for (int run = 0; run < kRuns; ++run) {  // rows 8 run .. 8 run + 7 of the stage
            u4 lo, hi;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const uint32_t even = st.d[8 * run + 2 * q], odd = st.d[8 * run + 2 * q + 1];
                lo[q] = (even & 0xffffu) | (odd << 16);
                hi[q] = (even >> 16) | (odd & 0xffff0000u);
            }
            *reinterpret_cast<u4*>(c0 + 16 * kRuns * group + 16 * run) = lo;
            *reinterpret_cast<u4*>(c1 + 16 * kRuns * group + 16 * run) = hi;
        }
    }
}

template <int DT>
__device__ __forceinline__ void gram_mfma(f16v (&acc)[2][2], const unsigned char* ti, const unsigned char* tj, int wm,
                                          int wn, int lane) {
    constexpr int P = gram_pitch<DT>();
    const int h = lane >> 5, col = lane & 31;
    const unsigned char* a_base = ti + (wm * 64 + col) * P;
    const unsigned char* b_base = tj + (wn * 64 + col) * P;
    if constexpr (DT == RCH_DT_F32) {
        // Lane half h holds rows 16h .. 16h + 15; MFMA step s takes row 16h + s.
        f4 a[2][4], b[2][4];
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                a[x][q] = *reinterpret_cast<const f4*>(a_base + x * 32 * P + 64 * h + 16 * q);
                b[x][q] = *reinterpret_cast<const f4*>(b_base + x * 32 * P + 64 * h + 16 * q);
            }
#pragma unroll
        for (int s = 0; s < 16; ++s)
#pragma unroll
            for (int x = 0; x < 2; ++x)
#pragma unroll
                for (int y = 0; y < 2; ++y)
                    acc[x][y] =
                        __builtin_amdgcn_mfma_f32_32x32x2f32(a[x][s >> 2][s & 3], b[y][s >> 2][s & 3], acc[x][y], 0, 0, 0);
    } else {
        // 16-row MFMA steps; lane half h holds rows 16 ks + 8h .. + 7.
#pragma unroll
        for (int ks = 0; ks < gram_rows<DT>() / 16; ++ks) {
            u4 a[2], b[2];
#pragma unroll
            for (int x = 0; x < 2; ++x) {
                a[x] = *reinterpret_cast<const u4*>(a_base + x * 32 * P + 32 * ks + 16 * h);
                b[x] = *reinterpret_cast<const u4*>(b_base + x * 32 * P + 32 * ks + 16 * h);
            }
#pragma unroll
            for (int x = 0; x < 2; ++x)
#pragma unroll
                for (int y = 0; y < 2; ++y) {
                    if constexpr (DT == RCH_DT_BF16)
                        acc[x][y] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf8, a[x]),
                                                                            __builtin_bit_cast(bf8, b[y]), acc[x][y], 0, 0, 0);
                    else
                        acc[x][y] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(h8, a[x]),
                                                                           __builtin_bit_cast(h8, b[y]), acc[x][y], 0, 0, 0);
                }
        }
    }
}

template <int DT>
__global__ void __launch_bounds__(kGramThreads) gram_kernel(const rch_fit_matrix* __restrict__ mats, int channels,
                                                            int tiles, int grid) {
    constexpr int P = gram_pitch<DT>();
    __shared__ __attribute__((aligned(16))) unsigned char lds[2][2][kGramTile * P];

    const int unit = xcd_unit(blockIdx.x, grid);  // the tiles of one matrix share an XCD's L2
    const int mat = unit / tiles;
    int ti = 0, rest = unit - mat * tiles;
    while (rest > ti) {  // tile index -> (ti, tj), row-major over the lower triangle
        rest -= ti + 1;
        ++ti;
    }
    const int tj = rest;
    const bool diagonal = ti == tj;
    const rch_fit_matrix* M = mats + mat;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    // Staging role: panel (0: the ti columns, 1: the tj columns), 128-channel half, 8-row group.
    const int panel = wave >> 3, half = (wave >> 2) & 1, group = wave & 3;
    // A diagonal tile stages one panel: the other panel's waves load from an out-of-range column
    // (the buffer loads return zeros without a memory access), so every wave runs the same
    // straight-line loop and the loads stay in flight across the MFMAs.
    const int c = diagonal && panel == 1 ? channels : (panel ? tj : ti) * kGramTile + 128 * half + 2 * lane;
    // MFMA role: the 64 x 64 quadrant (wm, wn).
    const int wm = wave >> 2, wn = wave & 3;
    const bool computes = !(diagonal && wm < wn);
    constexpr int kRows = gram_rows<DT>();
    const int steps = static_cast<int>((M->rows + kRows - 1) / kRows);

    f16v acc[2][2];
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y) acc[x][y] = f16v{};

    // 16-bit rows are loaded two steps ahead into alternating register stages: the loads for
    // step s + 2 are issued before step s's MFMAs and written to LDS after step s + 1's, so two
    // steps of MFMA work cover their latency.  Rows past the end read as zeros (empty buffer), so
    // the loads and stores need no conditions and the loop stays straight-line, which keeps the
    // compiler's waits on the older stage only.
    unsigned char* staged = lds[0][panel] + 128 * half * P;  // this wave's rows in buffer 0
    constexpr int kBuffer = 2 * kGramTile * P;                // buffer 1 = buffer 0 + kBuffer
    auto mfma_step = [&](int step) {
        const int buf = step & 1;
        if (computes) gram_mfma<DT>(acc, lds[buf][0], diagonal ? lds[buf][0] : lds[buf][1], wm, wn, lane);
        return staged + (buf ^ 1) * kBuffer;  // where the next step's rows go
    };
    if constexpr (DT != RCH_DT_F32) {
        GramStage<DT> sa, sb;
        gram_load<DT>(sa, M, channels, kRows / 4 * group, c);
        gram_load<DT>(sb, M, channels, kRows + kRows / 4 * group, c);
        gram_store<DT>(sa, staged, lane, group);
        __syncthreads();
        auto step_body = [&](int step, GramStage<DT>& ahead, const GramStage<DT>& next) {
            gram_load<DT>(ahead, M, channels, static_cast<int64_t>(step + 2) * kRows + kRows / 4 * group, c);
            gram_store<DT>(next, mfma_step(step), lane, group);
            __syncthreads();
        };
        for (int step = 0; step < steps; step += 2) {
            step_body(step, sa, sb);
            if (step + 1 < steps) step_body(step + 1, sb, sa);
        }
    } else {  // fp32 stages are twice as large: one step ahead keeps the loop within 128 VGPRs
        GramStage<DT> st;
        gram_load<DT>(st, M, channels, kRows / 4 * group, c);
        gram_store<DT>(st, staged, lane, group);
        __syncthreads();
        for (int step = 0; step < steps; ++step) {
            gram_load<DT>(st, M, channels, static_cast<int64_t>(step + 1) * kRows + kRows / 4 * group, c);
            gram_store<DT>(st, mfma_step(step), lane, group);
            __syncthreads();
        }
    }
    if (!computes) return;

    // Accumulator element e of lane l: row 8 (e / 4) + 4 (l / 32) + e % 4, column l % 32.
    RCH_GLOBAL float* G = gout<float>(M->gram_ptr);
    const int64_t ld = M->gram_stride;
    const int h = lane >> 5, col = lane & 31;
    const bool lower_only = diagonal && wm == wn;  // a quadrant on the diagonal: its lower half, mirrored
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y) {
            const int ib = ti * kGramTile + wm * 64 + x * 32;
            const int64_t j = tj * kGramTile + wn * 64 + y * 32 + col;
            if (j >= channels) continue;
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int64_t i0 = ib + 8 * g + 4 * h;  // rows i0 .. i0 + 3 (channels % 8 == 0: all or none in range)
                if (i0 >= channels) continue;
                if (!lower_only) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) G[(i0 + r) * ld + j] = acc[x][y][4 * g + r];
                    // Mirror: G[j][i0 .. i0 + 3] is one 16-byte store.
                    const f4 v = {acc[x][y][4 * g], acc[x][y][4 * g + 1], acc[x][y][4 * g + 2], acc[x][y][4 * g + 3]};
                    *reinterpret_cast<RCH_GLOBAL f4*>(G + j * ld + i0) = v;
                } else {
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int64_t i = i0 + r;
                        if (i >= j) {  // lower triangle, mirrored
                            G[i * ld + j] = acc[x][y][4 * g + r];
                            G[j * ld + i] = acc[x][y][4 * g + r];
                        }
                    }
                }
            }
        }
}

// ---------------------------------------------------------------------------------------------
// Projection P = X Q^T on v_mfma_f64_16x16x4f64: D[m = token][n = rank] = sum_c X[token][c] Q[rank][c].
// Per 32-channel step a lane (i = l % 16, group g = l / 16) holds channels 8g .. 8g + 7 of its token
// rows and of its basis rows (16-byte loads), and MFMA step s takes channel 8g + s from every group.  The
// f64 accumulator holds element v of lane l at row (l / 16) + 4v, column l % 16: token g + 4v, rank i of
// the block.
//
// Every element is the sum of two chains, over the first and the second half of the channel steps, each run
// by a wave of its own, whatever the shape of the launch: the bits of P do not depend on the batch, which
// chooses the shape.
//   * kShared: a wave owns 32 tokens and half of the channels; the four waves of a half share a step's
//     converted basis operands through LDS (two parts, one barrier a step), so a wave loads and converts a
//     quarter of them and each feeds two of its products; workgroup = 128 tokens x 64 ranks, eight waves.
//   * kDeep: for batches whose last round of those would leave CUs idle: a wave owns 16 tokens, 16 or 32 ranks
//     and half of the channels, and keeps kProjectDeep steps of loads in flight; workgroup = 32 tokens.
//   * kGram: the sources are the basis rows themselves, the channel steps dealt to four waves, and the FP64
//     sums are stored as they are, G = Q Q^T.
// Bound by the FP64 matrix rate; the next step's loads are issued before a step's products and the step body
// has no branch, so their latency is covered.  The vector instructions do not hide under FP64 products, and the
// rate depends on the operands' bits: products of full 53-bit operands alone reach 46-49 TFLOP/s, a large
// library product 68.
// bf16 [4680, 1536] at rank 96 (MI355X): one matrix 105 us with 64-token workgroups of one wave per 16 tokens
// and loads in the step, 38 now (34 with four chains per element, whose partial sums a wave of kShared has no
// registers for); 60 matrices 1563 us, 1396 with every wave converting its own basis operands, 1306 now.
// ---------------------------------------------------------------------------------------------

// Eight consecutive source elements as loaded, and as doubles.
template <int DT>
struct Eight {
    u4 w[DT == RCH_DT_F32 ? 2 : 1];
};
template <int DT>
__device__ __forceinline__ Eight<DT> load_eight(__amdgpu_buffer_rsrc_t rsrc, uint32_t offset) {
    Eight<DT> e;
    e.w[0] = __builtin_amdgcn_raw_buffer_load_b128(rsrc, offset, 0, 0);
    if constexpr (DT == RCH_DT_F32) e.w[1] = __builtin_amdgcn_raw_buffer_load_b128(rsrc, offset + 16, 0, 0);
    return e;
}
template <int DT>
__device__ __forceinline__ double eight_at(const Eight<DT>& e, int i) {
    if constexpr (DT == RCH_DT_F32) return static_cast<double>(__uint_as_float(e.w[i >> 2][i & 3]));
    else return static_cast<double>(half_bits<DT>((e.w[0][i >> 1] >> (16 * (i & 1))) & 0xffffu));
}

constexpr int kProjectDeep = 3;  // 4 and 6 measure the same

enum class Project { kShared, kDeep, kGram };

// Waves of a workgroup, tokens of a wave, and first channel of the second half.
template <Project SHAPE>
constexpr int kProjectWaves = SHAPE == Project::kShared ? 8 : 4;
template <Project SHAPE>
constexpr int kProjectTiles = SHAPE == Project::kShared ? 2 : 1;  // of 16 tokens
__device__ __forceinline__ int project_middle(int channels) { return min(channels, 32 * (((channels + 31) / 32 + 1) / 2)); }

// Order of the padded FP64 k x k matrices of the span kernels.
__device__ __forceinline__ int padded_order(int rank) { return (rank + 15) & ~15; }

template <int DT, Project SHAPE, int NB>
__device__ __forceinline__ void project_ranks(const rch_fit_matrix* M, int channels, int r0, int64_t wt, int wave, int lane,
                                              double* shared) {
    constexpr int E = esize<DT>();
    constexpr bool GRAM = SHAPE == Project::kGram;
    static_assert(!GRAM || DT == RCH_DT_F16, "the basis Gram runs on fp16 rows");
    constexpr int TB = kProjectTiles<SHAPE>, kWaves = kProjectWaves<SHAPE>;
    const int half = GRAM ? 0 : wave / (kWaves / 2), middle = project_middle(channels);
    const int begin = half ? middle : 0, end = GRAM || half ? channels : middle;  // of this wave's channels
    const int rank = static_cast<int>(M->rank);
    const int64_t rows = GRAM ? rank : M->rows;
    const int g = lane >> 4, i16 = lane & 15;
    const __amdgpu_buffer_rsrc_t qs = make_rsrc(M->basis_ptr, ((rank - 1) * M->basis_stride + channels) * 2);
    const __amdgpu_buffer_rsrc_t xs = GRAM ? qs : source_rows<DT>(M, channels, wt);
    uint32_t x_row[TB], q_row[NB];
#pragma unroll
    for (int t = 0; t < TB; ++t) {
        if constexpr (GRAM) x_row[t] = wt + i16 < rank ? static_cast<uint32_t>((wt + i16) * M->basis_stride * 2) : kOutOfRange;
        else x_row[t] = static_cast<uint32_t>((16 * t + i16) * M->src_stride * E);
    }
#pragma unroll
    for (int b = 0; b < NB; ++b)  // rows past the rank read zeros
        q_row[b] = r0 + 16 * b + i16 < rank ? static_cast<uint32_t>((r0 + 16 * b + i16) * M->basis_stride * 2) : kOutOfRange;
    Eight<DT> x_now[TB], x_next[TB];
    auto load_x = [&](int c0) __attribute__((always_inline)) {
        const int c = c0 + 8 * g;  // channels % 8 == 0: a group is whole or past the end
        const uint32_t past = c < end ? 0u : kOutOfRange;
#pragma unroll
        for (int t = 0; t < TB; ++t) x_next[t] = load_eight<DT>(xs, (x_row[t] + static_cast<uint32_t>(c * E)) | past);
    };
    auto q_at = [&](int b, int c0, int first) __attribute__((always_inline)) {  // from channel `first` of a group
        const int c = c0 + 8 * g;
        return (q_row[b] + static_cast<uint32_t>((c + first) * 2)) | (c < end ? 0u : kOutOfRange);
    };
    d4 acc[TB][NB];
#pragma unroll
    for (int t = 0; t < TB; ++t)
#pragma unroll
        for (int b = 0; b < NB; ++b) acc[t][b] = d4{};
    // basis(b, s): channel s of rank block b.
    auto products = [&](const Eight<DT> (&x)[TB], auto&& basis) __attribute__((always_inline)) {
        double xv[TB][8];
#pragma unroll
        for (int t = 0; t < TB; ++t)
#pragma unroll
            for (int s = 0; s < 8; ++s) xv[t][s] = eight_at<DT>(x[t], s);
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int s = 0; s < 8; ++s) {
                const double qv = basis(b, s);
#pragma unroll
                for (int t = 0; t < TB; ++t)
                    acc[t][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(xv[t][s], qv, acc[t][b], 0, 0, 0);
            }
    };
    auto advance = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < TB; ++t) x_now[t] = x_next[t];
    };
    d4 sum[NB];  // of the 16 tokens that this wave stores
    if constexpr (SHAPE == Project::kShared) {  // wave w of a half converts channels 2w, 2w + 1 of every group for its four
        static_assert(kWaves == 8, "four waves share a step's eight channels");
        constexpr int kStep = 8 * NB * 64;
        const int pair_at = 2 * (wave & 3);
        double* const staged = shared + 2 * half * kStep;
        uint32_t pair[NB];
        auto load_pair = [&](int c0) __attribute__((always_inline)) {
#pragma unroll
            for (int b = 0; b < NB; ++b) pair[b] = __builtin_amdgcn_raw_buffer_load_b32(qs, q_at(b, c0, pair_at), 0, 0);
        };
        auto stage = [&](int at) __attribute__((always_inline)) {
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                double* to = staged + at + (8 * b + pair_at) * 64 + lane;
                to[0] = static_cast<double>(half_bits<RCH_DT_F16>(pair[b] & 0xffffu));
                to[64] = static_cast<double>(half_bits<RCH_DT_F16>(pair[b] >> 16));
            }
        };
        load_x(begin), load_pair(begin);
        stage(0), advance();
        __syncthreads();
        // Both halves take the first half's count of steps (a step past the end multiplies zeros).
        for (int c = 0, at = 0; c < middle; c += 32, at = kStep - at) {
            load_x(begin + c + 32), load_pair(begin + c + 32);
            products(x_now, [&](int b, int s) { return staged[at + (8 * b + s) * 64 + lane]; });
            stage(kStep - at), advance();  // this part was last read before the previous barrier
            __syncthreads();
        }
        // Each half stores one of the two tiles: the other's sums go to the wave that shares the tokens.
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int v = 0; v < 4; ++v) shared[((wave * NB + b) * 4 + v) * 64 + lane] = half ? acc[0][b][v] : acc[1][b][v];
        __syncthreads();
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int v = 0; v < 4; ++v)
                sum[b][v] = (half ? acc[1][b][v] : acc[0][b][v]) + shared[(((wave ^ 4) * NB + b) * 4 + v) * 64 + lane];
        wt += 16 * half;
    } else if constexpr (SHAPE == Project::kDeep) {
        Eight<DT> x[kProjectDeep][TB];
        Eight<RCH_DT_F16> q[kProjectDeep][NB];
        auto load = [&](int c0, Eight<DT> (&x_to)[TB], Eight<RCH_DT_F16> (&q_to)[NB]) __attribute__((always_inline)) {
            load_x(c0);
#pragma unroll
            for (int t = 0; t < TB; ++t) x_to[t] = x_next[t];
#pragma unroll
            for (int b = 0; b < NB; ++b) q_to[b] = load_eight<RCH_DT_F16>(qs, q_at(b, c0, 0));
        };
#pragma unroll
        for (int d = 0; d < kProjectDeep; ++d) load(begin + 32 * d, x[d], q[d]);
        for (int c0 = begin; c0 < end; c0 += 32 * kProjectDeep) {
#pragma unroll
            for (int d = 0; d < kProjectDeep; ++d) {  // a step past the end multiplies zeros
                products(x[d], [&](int b, int s) { return eight_at<RCH_DT_F16>(q[d][b], s); });
                load(c0 + 32 * (d + kProjectDeep), x[d], q[d]);
            }
        }
        if (half) {
#pragma unroll
            for (int b = 0; b < NB; ++b)
#pragma unroll
                for (int v = 0; v < 4; ++v) shared[(((wave & 1) * NB + b) * 4 + v) * 64 + lane] = acc[0][b][v];
        }
        __syncthreads();
        if (half) return;
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int v = 0; v < 4; ++v) sum[b][v] = acc[0][b][v] + shared[((wave * NB + b) * 4 + v) * 64 + lane];
    } else {
        Eight<RCH_DT_F16> q_now[NB], q_next[NB];
        auto load_q = [&](int c0) __attribute__((always_inline)) {
#pragma unroll
            for (int b = 0; b < NB; ++b) q_next[b] = load_eight<RCH_DT_F16>(qs, q_at(b, c0, 0));
        };
        auto advance_q = [&]() __attribute__((always_inline)) {
#pragma unroll
            for (int b = 0; b < NB; ++b) q_now[b] = q_next[b];
        };
        load_x(32 * wave), load_q(32 * wave);
        advance(), advance_q();
        for (int c0 = 32 * wave; c0 < channels; c0 += 32 * kWaves) {
            load_x(c0 + 32 * kWaves), load_q(c0 + 32 * kWaves);
            products(x_now, [&](int b, int s) { return eight_at<RCH_DT_F16>(q_now[b], s); });
            advance(), advance_q();
        }
        // Block b of every wave is added, in wave order, by wave b.
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int v = 0; v < 4; ++v) shared[((b * kWaves + wave) * 4 + v) * 64 + lane] = acc[0][b][v];
        __syncthreads();
        if (wave >= NB) return;
        d4 entry = d4{};
#pragma unroll
        for (int w = 0; w < kWaves; ++w)
#pragma unroll
            for (int v = 0; v < 4; ++v) entry[v] += shared[((wave * kWaves + w) * 4 + v) * 64 + lane];
        const int kp = padded_order(rank), k = r0 + 16 * wave + i16;  // rows and columns past the rank are zeros
#pragma unroll
        for (int v = 0; v < 4; ++v) gout<double>(M->gram_ptr)[(wt + g + 4 * v) * kp + k] = entry[v];
        return;
    }
    RCH_GLOBAL float* out = gout<float>(M->coef_ptr);
    unsigned int* ext = reinterpret_cast<unsigned int*>(M->extrema_ptr);
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        const int k = r0 + 16 * b + i16;  // this lane's rank
        uint32_t lo = 0u, hi = 0u;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int64_t token = wt + g + 4 * v;
            const float value = static_cast<float>(sum[b][v]);
            if (token < rows) {
                if (k < rank) out[token * M->coef_stride + k] = value;  // 16 lanes: 64 contiguous bytes of a row
                const uint32_t key = order_key(value);
                lo = ~key > lo ? ~key : lo;
                hi = key > hi ? key : hi;
            }
        }
        if (ext) {
#pragma unroll
            for (int d = 16; d <= 32; d <<= 1) {  // over the 4 token groups
                const uint32_t ol = __shfl_xor(lo, d), oh = __shfl_xor(hi, d);
                lo = ol > lo ? ol : lo;
                hi = oh > hi ? oh : hi;
            }
            if (g == 0 && k < rank) {
                atomicMax(ext + k, lo);  // vector atomics
                atomicMax(ext + rank + k, hi);
            }
        }
    }
}

// Tokens of a project_kernel workgroup: its halves' waves share them.
template <Project SHAPE>
constexpr int kProjectTokens = 16 * kProjectTiles<SHAPE> * kProjectWaves<SHAPE> / 2;

template <int DT, Project SHAPE>
__global__ void __launch_bounds__(64 * kProjectWaves<SHAPE>, 4) project_kernel(const rch_fit_matrix* __restrict__ mats,
                                                                              int channels, int chunk) {
    constexpr bool kShared = SHAPE == Project::kShared;
    // The basis operands of two steps of four rank blocks per half, then the exchanged sums: the same size.
    __shared__ double shared[kShared ? 2 * 2 * 8 * 4 * 64 : 2 * 2 * 4 * 64];
    const rch_fit_matrix* M = mats + blockIdx.z;
    const int rank = static_cast<int>(M->rank);
    const int64_t t0 = static_cast<int64_t>(blockIdx.x) * kProjectTokens<SHAPE>;
    const int r0 = blockIdx.y * chunk;  // chunk: 16 or 32 ranks, kShared also 48 or 64
    if (t0 >= M->rows || r0 >= rank) return;  // whole workgroup
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int64_t wt = t0 + 16 * kProjectTiles<SHAPE> * (wave % (kProjectWaves<SHAPE> / 2));  // first token of this wave
    const int blocks = min(chunk >> 4, (rank - r0 + 15) >> 4);  // 16-rank blocks of this chunk (uniform)
    if (blocks == 1) project_ranks<DT, SHAPE, 1>(M, channels, r0, wt, wave, lane, shared);
    else if (!kShared || blocks == 2) project_ranks<DT, SHAPE, 2>(M, channels, r0, wt, wave, lane, shared);
    if constexpr (kShared) {
        if (blocks == 3) project_ranks<DT, SHAPE, 3>(M, channels, r0, wt, wave, lane, shared);
        else if (blocks >= 4) project_ranks<DT, SHAPE, 4>(M, channels, r0, wt, wave, lane, shared);
    }
}

// ---------------------------------------------------------------------------------------------
// Residual energies on v_mfma_f64_16x16x4f64: D[m = token][n = channel] = sum_k P[token][k] Q[k][c].
// Workgroup = some tokens of one matrix and every gridDim.z-th part of its 64-channel groups.  A group is
// four 16 x 16 blocks per 16 tokens whose columns interleave: column i of block b is channel 4i + b of the
// group, so after the four blocks lane l (i = l % 16, g = l / 16) holds channels 4i .. 4i + 3 of tokens
// g + 4v (v = 0..3, the f64 accumulator's row (l / 16) + 4v): X and the residual move as 4-channel vectors,
// 16 lanes covering 64 contiguous channels of a row.  Per 16-rank step a lane
// takes P[token i][4g .. 4g + 3] (the A operand; MFMA step j takes rank 4g + j) and, for each j,
// Q[4g + j][4i .. 4i + 3] (one 8-byte load: the B operands of the four blocks).
//
// Two shapes:
//   * SHARED: a wave owns 32 of the workgroup's 128 tokens and all waves walk the same channel groups,
//     sharing a step's converted basis operands through LDS (two halves, one barrier a step): a wave loads
//     and converts a quarter of them and each feeds two of its products.
//   * for batches that would leave CUs idle: 16 tokens, a channel group per wave.
// Bound by the FP64 matrix rate (rank 0, the source energy alone: by HBM), with the vector instructions
// beside it: they do not hide under FP64 products.  The next step's operands are loaded before a step's
// products and a group's source elements before all of its products.
// bf16 [4680, 1536] (MI355X, with the totals): one matrix at rank 96 137 -> 42 us; 60 at rank 96 1808 us with
// 16-token workgroups, 1527 with 32-token ones of unshared operands, 1450 now (57 TFLOP/s); 60 at ranks 32 to
// 128 1350 -> 1285 us; source energy alone of one 8 us, of 60 169.
// ---------------------------------------------------------------------------------------------

// The 4 channels of tokens g + 4v (v = 0..3) of a lane's 64-channel group, as raw 16-bit pairs
// (or fp32 words).
template <int DT>
struct SourceQuad {
    using word = std::conditional_t<DT == RCH_DT_F32, u4, u2>;
    word w[4];
};

// A partial energy sums 16 tokens and one part of the channels, a run of 64-channel groups, whatever the
// shape of the launch: a lane adds its elements in order, then the wave its lanes.  So the bits of a matrix's
// energies do not depend on the batch that it is measured in, which chooses the shape.
__host__ __device__ __forceinline__ int residual_groups(int channels) { return (channels + 63) >> 6; }
__host__ __device__ __forceinline__ int residual_part_groups(int channels) {
    return (residual_groups(channels) + RCH_RESIDUAL_PARTS - 1) / RCH_RESIDUAL_PARTS;
}
__host__ __device__ __forceinline__ int residual_parts(int channels) {
    const int each = residual_part_groups(channels);
    return (residual_groups(channels) + each - 1) / each;
}

// v plus the value `Turn` lanes on within the row of 16 lanes.
template <int Turn>
__device__ __forceinline__ double add_turned(double v) {
    const u2 w = __builtin_bit_cast(u2, v);
    const u2 o = {static_cast<uint32_t>(__builtin_amdgcn_mov_dpp(static_cast<int>(w[0]), 0x120 + Turn, 0xf, 0xf, true)),
                  static_cast<uint32_t>(__builtin_amdgcn_mov_dpp(static_cast<int>(w[1]), 0x120 + Turn, 0xf, 0xf, true))};
    return v + __builtin_bit_cast(double, o);
}

// Sums over the wave of the TB tiles' two energies: lanes 0-15 and 16-31 return src[0] and src[TB - 1], lanes
// 32-47 and 48-63 err[0] and err[TB - 1].  Per value a tree over lane distances 32, 16, 8, 4, 2, 1.
template <int TB>
__device__ __forceinline__ double residual_sums(const double (&src)[TB], const double (&err)[TB], int lane) {
    double half[TB];
#pragma unroll
    for (int t = 0; t < TB; ++t) {  // the lower half keeps src, the upper half err
        const double give = lane < 32 ? err[t] : src[t];
        half[t] = (lane < 32 ? src[t] : err[t]) + __shfl_xor(give, 32);
    }
    const bool odd = lane & 16;
    const double give = odd ? half[0] : half[TB - 1];
    double sum = (odd ? half[TB - 1] : half[0]) + __shfl_xor(give, 16);
    sum = add_turned<8>(sum);
    sum = add_turned<4>(sum);
    sum = add_turned<2>(sum);
    return add_turned<1>(sum);
}

// Tokens of a residual_kernel workgroup, and channel parts that its waves work on at once.
template <bool SHARED>
constexpr int kResidualTokens = SHARED ? 32 * (kThreads / 64) : 16;
template <bool SHARED>
constexpr int kResidualAtOnce = SHARED ? 1 : kThreads / 64;

template <int DT, bool SHARED>
__global__ void __launch_bounds__(kThreads, 2) residual_kernel(const rch_fit_matrix* __restrict__ mats, int channels) {
    constexpr int E = esize<DT>(), TB = SHARED ? 2 : 1, kWaves = kThreads / 64;
    constexpr int kStep = 16 * 64;  // basis operands of a 16-rank step, [j: rank 4g + j][block][lane]
    static_assert(kWaves == 4, "wave j shares the rows of ranks 4g + j");
    __shared__ double staged[SHARED ? 2 * kStep : 1];
    const rch_fit_matrix* M = mats + blockIdx.y;
    const int64_t rows = M->rows;
    const int rank = static_cast<int>(M->rank);
    const int64_t t0 = static_cast<int64_t>(blockIdx.x) * kResidualTokens<SHARED>;
    if (t0 >= rows) return;  // whole workgroup
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int g = lane >> 4, i16 = lane & 15;
    const int64_t wt = SHARED ? t0 + 32 * wave : t0, left = rows - wt;  // rows past the end read zeros
    const __amdgpu_buffer_rsrc_t xs = source_rows<DT>(M, channels, wt);
    const __amdgpu_buffer_rsrc_t ps = make_rsrc(M->coef_ptr + wt * M->coef_stride * 4,
                                                rank > 0 && left > 0 ? ((left - 1) * M->coef_stride + rank) * 4 : 0);
    const __amdgpu_buffer_rsrc_t qs = make_rsrc(M->basis_ptr, rank > 0 ? ((rank - 1) * M->basis_stride + channels) * 2 : 0);
    const uint32_t q_stride = static_cast<uint32_t>(M->basis_stride * 2);
    RCH_GLOBAL float* resid = M->resid_ptr ? gout<float>(M->resid_ptr) : nullptr;
    uint32_t p_row[TB], x_row[TB][4];
#pragma unroll
    for (int t = 0; t < TB; ++t) {
        p_row[t] = static_cast<uint32_t>((16 * t + i16) * M->coef_stride * 4);
#pragma unroll
        for (int v = 0; v < 4; ++v) x_row[t][v] = static_cast<uint32_t>((16 * t + g + 4 * v) * M->src_stride * E);
    }
    auto load_source = [&](int c64, SourceQuad<DT> (&q)[TB]) __attribute__((always_inline)) {
        const int c = c64 + 4 * i16;  // this lane's 4 channels (channels % 8 == 0: all or none in range)
        const uint32_t past = c < channels ? 0u : kOutOfRange;
#pragma unroll
        for (int t = 0; t < TB; ++t)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const uint32_t offset = (x_row[t][v] + static_cast<uint32_t>(c * E)) | past;
                if constexpr (DT == RCH_DT_F32) q[t].w[v] = __builtin_amdgcn_raw_buffer_load_b128(xs, offset, 0, 0);
                else q[t].w[v] = __builtin_amdgcn_raw_buffer_load_b64(xs, offset, 0, 0);
            }
    };
    // Q[k0 + 4g + j][4 channels] (SHARED: j = wave alone) and P[token][k0 + 4g ..].
    u2 q_now[SHARED ? 1 : 4], q_next[SHARED ? 1 : 4];
    u4 p_now[TB], p_next[TB];
    auto load_operands = [&](int c64, int k0) __attribute__((always_inline)) {
        const int c = c64 + 4 * i16, k = k0 + 4 * g;
#pragma unroll
        for (int q = 0; q < (SHARED ? 1 : 4); ++q) {
            const int kq = k + (SHARED ? wave : q);
            const uint32_t offset = (kq < rank && c < channels) ? static_cast<uint32_t>(kq) * q_stride + 2u * c : kOutOfRange;
            q_next[q] = __builtin_amdgcn_raw_buffer_load_b64(qs, offset, 0, 0);
        }
#pragma unroll
        for (int t = 0; t < TB; ++t)
            p_next[t] = __builtin_amdgcn_raw_buffer_load_b128(ps, k < rank ? p_row[t] + static_cast<uint32_t>(k * 4) : kOutOfRange, 0, 0);
    };
    auto basis_at = [](const u2& q, int b) __attribute__((always_inline)) {
        return static_cast<double>(half_bits<RCH_DT_F16>((q[b >> 1] >> (16 * (b & 1))) & 0xffffu));
    };
    auto advance = [&](int k0, int at) __attribute__((always_inline)) {  // the loaded operands are the next step's
        if constexpr (SHARED) {
#pragma unroll
            for (int b = 0; b < 4; ++b) staged[at + (4 * wave + b) * 64 + lane] = basis_at(q_next[0], b);
        } else {
#pragma unroll
            for (int q = 0; q < 4; ++q) q_now[q] = q_next[q];
        }
        if (k0 + 16 > rank) {  // P rows may hold padding beyond the rank; its basis rows read as zero
#pragma unroll
            for (int t = 0; t < TB; ++t)
#pragma unroll
                for (int j = 0; j < 4; ++j) p_next[t][j] = k0 + 4 * g + j < rank ? p_next[t][j] : 0u;
        }
#pragma unroll
        for (int t = 0; t < TB; ++t) p_now[t] = p_next[t];
        if constexpr (SHARED) __syncthreads();
    };

    double src[TB], err[TB];
    d4 acc[TB][4];
    // e = x - r per element: FP64 sums of x^2 and e^2, optional fp32 store.
    auto finish = [&](auto source_only, int c64, const SourceQuad<DT> (&x)[TB]) __attribute__((always_inline)) {
        const int c = c64 + 4 * i16;
#pragma unroll
        for (int t = 0; t < TB; ++t)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                double e[4];
#pragma unroll
                for (int b = 0; b < 4; ++b) {
                    double a;
                    if constexpr (DT == RCH_DT_F32) a = static_cast<double>(__uint_as_float(x[t].w[v][b]));
                    else a = static_cast<double>(half_bits<DT>((x[t].w[v][b >> 1] >> (16 * (b & 1))) & 0xffffu));
                    src[t] = fma(a, a, src[t]);
                    if constexpr (source_only.value) {
                        e[b] = a;
                    } else {
                        e[b] = a - acc[t][b][v];
                        err[t] = fma(e[b], e[b], err[t]);
                    }
                }
                const int token = 16 * t + g + 4 * v;
                if (resid && c < channels && token < left) {
                    const f4 out = {static_cast<float>(e[0]), static_cast<float>(e[1]), static_cast<float>(e[2]),
                                    static_cast<float>(e[3])};
                    *reinterpret_cast<RCH_GLOBAL f4*>(resid + (wt + token) * channels + c) = out;
                }
            }
    };
    const int parts = residual_parts(channels), each = residual_part_groups(channels);
    const int stride = kResidualAtOnce<SHARED> * static_cast<int>(gridDim.z);
    auto clear = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < TB; ++t) src[t] = err[t] = 0.0;
    };
    // The wave's parts are stored together at the end, lane i16 the i16-th: a store in the loop would hold up the
    // loads behind it, which complete in order.
    double kept = 0.0;
    int done = 0;
    auto end_part = [&]() __attribute__((always_inline)) {
        const double sum = residual_sums<TB>(src, err, lane);
        kept = i16 == done ? sum : kept;
        ++done;
        clear();
    };
    // The 64-channel groups of this wave's parts in turn; past the channels at the end.
    auto part_end = [&](int part) __attribute__((always_inline)) { return min(64 * each * (part + 1), channels); };
    auto next_group = [&](int& part, int& c64) __attribute__((always_inline)) {
        c64 += 64;
        if (c64 < part_end(part)) return;
        part += stride;
        c64 = part < parts ? 64 * each * part : channels;
    };
    const int first_part = kResidualAtOnce<SHARED> * static_cast<int>(blockIdx.z) + (SHARED ? 0 : wave);
    const int first = first_part < parts ? 64 * each * first_part : channels;
    int part = first_part;
    int part_next = part, next = first;  // of the group after the current one
    next_group(part_next, next);
    SourceQuad<DT> x_now[TB];
    clear();
    if (rank > 0) {
        load_operands(first, 0);
        advance(0, 0);
        int at = 0;
        for (int c64 = first; c64 < channels;) {
            load_source(c64, x_now);  // in flight under the group's products
#pragma unroll
            for (int t = 0; t < TB; ++t)
#pragma unroll
                for (int b = 0; b < 4; ++b) acc[t][b] = d4{};
            for (int k0 = 0; k0 < rank; k0 += 16) {
                const bool last = k0 + 16 >= rank;
                const int k_next = last ? 0 : k0 + 16;
                load_operands(last ? next : c64, k_next);
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    double pa[TB];
#pragma unroll
                    for (int t = 0; t < TB; ++t) pa[t] = static_cast<double>(__uint_as_float(p_now[t][j]));
#pragma unroll
                    for (int b = 0; b < 4; ++b) {
                        double qb;
                        if constexpr (SHARED) qb = staged[at + (4 * j + b) * 64 + lane];
                        else qb = basis_at(q_now[j], b);
#pragma unroll
                        for (int t = 0; t < TB; ++t) acc[t][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(pa[t], qb, acc[t][b], 0, 0, 0);
                    }
                }
                at = kStep - at;  // this half was last read before the previous barrier
                advance(k_next, at);
            }
            finish(std::false_type{}, c64, x_now);
            if (c64 + 64 >= part_end(part)) end_part();  // uniform
            part = part_next, c64 = next;
            next_group(part_next, next);
        }
    } else {  // the source energy alone (the residual is the source): one group ahead
        SourceQuad<DT> x_next[TB];
        load_source(first, x_now);
        for (int c64 = first; c64 < channels;) {
            load_source(next, x_next);
            finish(std::true_type{}, c64, x_now);
            if (c64 + 64 >= part_end(part)) {
#pragma unroll
                for (int t = 0; t < TB; ++t) err[t] = src[t];
                end_part();
            }
            part = part_next, c64 = next;
            next_group(part_next, next);
#pragma unroll
            for (int t = 0; t < TB; ++t) x_now[t] = x_next[t];
        }
    }
    const int64_t tile = (wt >> 4) + (TB > 1 ? g & 1 : 0);  // residual_sums: 16 lanes per tile and energy
    if (i16 < done && (TB > 1 || !(g & 1)) && 16 * tile < rows)
        gout<double>(M->partial_ptr)[2 * (tile * parts + first_part + stride * i16) + (g >> 1)] = kept;
}

// Sum of the partials of each matrix, one workgroup per matrix: thread t takes partials t, t + 1024, ... in
// order, then its wave's lanes and the waves in order; divided by s^2 (s = max|X|).  The order depends on the
// matrix's rows and channels alone.
constexpr int kTotalThreads = 1024;
typedef double d2 __attribute__((ext_vector_type(2)));

__global__ void __launch_bounds__(kTotalThreads) energy_total_kernel(const rch_fit_matrix* __restrict__ mats, int channels) {
    constexpr int kWaves = kTotalThreads / 64;
    __shared__ double sums[2][kWaves];
    const rch_fit_matrix* M = mats + blockIdx.x;
    const int64_t count = ((M->rows + 15) >> 4) * residual_parts(channels);
    const RCH_GLOBAL d2* p = gin<d2>(M->partial_ptr);
    double a = 0.0, b = 0.0;
    for (int64_t t0 = threadIdx.x; t0 < count; t0 += 4 * kTotalThreads) {
        d2 v[4];  // four loads in flight
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = t0 + i * kTotalThreads < count ? p[t0 + i * kTotalThreads] : d2{};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            a += v[i][0];
            b += v[i][1];
        }
    }
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) {
        a += __shfl_xor(a, d);
        b += __shfl_xor(b, d);
    }
    if ((threadIdx.x & 63) == 0) {
        sums[0][threadIdx.x >> 6] = a;
        sums[1][threadIdx.x >> 6] = b;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < kWaves; ++w) {
            a += sums[0][w];
            b += sums[1][w];
        }
        const float smax = __uint_as_float(*gin<unsigned int>(M->absmax_ptr));
        if (smax != 0.0f) {
            const double s = static_cast<double>(smax);
            a = a / s / s;
            b = b / s / s;
        }
        RCH_GLOBAL double* out = gout<double>(M->energy_ptr);
        out[0] = a;
        out[1] = b;
    }
}

// ---------------------------------------------------------------------------------------------
// Column extrema (workgroup = 64 rows, a thread per column) and the FP64 quantizer of fp32 [rows, cols]
// matrices.  Both are latency-bound at archive sizes.  The quantizer spreads a tile's rows and columns
// over all threads: one [4680, 96] matrix takes 5 us (15 us with a thread per column and 64 rows in
// turn), 60 of mixed ranks 42 us (76).  The extrema, spread the same way over 4 or 16 waves, took 10
// and 12 us against 10: they wait for their atomics.
// ---------------------------------------------------------------------------------------------

__global__ void __launch_bounds__(kThreads) extrema_kernel(const float* __restrict__ values, int64_t rows, int cols,
                                                           int64_t stride, unsigned int* __restrict__ keys) {
    const int64_t r0 = static_cast<int64_t>(blockIdx.x) * 64;
    const int64_t r1 = rows - r0 < 64 ? rows : r0 + 64;
    for (int c = threadIdx.x; c < cols; c += kThreads) {
        uint32_t lo = 0u, hi = 0u;
        for (int64_t r = r0; r < r1; ++r) {
            const uint32_t k = order_key(values[r * stride + c]);
            lo = ~k > lo ? ~k : lo;
            hi = k > hi ? k : hi;
        }
        atomicMax(keys + c, lo);  // vector atomics
        atomicMax(keys + cols + c, hi);
    }
}

constexpr int kQuantizeRows = 16;  // rows per workgroup

// Codes of rows [r0, r0 + kQuantizeRows): a thread takes four consecutive columns of a row.
__device__ __forceinline__ void quantize_rows(const RCH_GLOBAL float* values, int64_t r0, int64_t rows, int cols, int64_t stride,
                                              const RCH_GLOBAL double* scale, const RCH_GLOBAL double* offset,
                                              RCH_GLOBAL uint8_t* codes, int64_t code_stride) {
    const int groups = (cols + 3) >> 2;
    const int left = static_cast<int>(rows - r0 < kQuantizeRows ? rows - r0 : kQuantizeRows);
    const bool vec = ((reinterpret_cast<int64_t>(values) | (stride * 4)) & 15) == 0;
    const bool words = ((reinterpret_cast<int64_t>(codes) | code_stride) & 3) == 0;
    for (int i = threadIdx.x; i < left * groups; i += kThreads) {
        const int row = i / groups, c = 4 * (i - row * groups);
        const RCH_GLOBAL float* v = values + (r0 + row) * stride + c;
        const bool whole = c + 4 <= cols;
        float x[4];
        if (vec && whole) {
            const f4 w = *reinterpret_cast<const RCH_GLOBAL f4*>(v);
#pragma unroll
            for (int j = 0; j < 4; ++j) x[j] = w[j];
        } else {
#pragma unroll
            for (int j = 0; j < 4; ++j) x[j] = c + j < cols ? v[j] : 0.0f;
        }
        uint32_t word = 0u;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if (c + j >= cols) continue;
            const double sc = scale[c + j], of = offset[c + j];
            double q = 0.0;
            if (sc > 0.0) q = rint((static_cast<double>(x[j]) - of) / sc);
            q = q < 0.0 ? 0.0 : (q > 255.0 ? 255.0 : q);
            word |= static_cast<uint32_t>(static_cast<uint8_t>(q)) << (8 * j);
        }
        RCH_GLOBAL uint8_t* out = codes + (r0 + row) * code_stride + c;
        if (words && whole) {
            *reinterpret_cast<RCH_GLOBAL uint32_t*>(out) = word;
        } else {
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (c + j < cols) out[j] = static_cast<uint8_t>(word >> (8 * j));
        }
    }
}

__global__ void __launch_bounds__(kThreads) quantize_kernel(const float* __restrict__ values, int64_t rows, int cols,
                                                            int64_t stride, const double* __restrict__ scale,
                                                            const double* __restrict__ offset,
                                                            uint8_t* __restrict__ codes, int64_t code_stride) {
    quantize_rows(gin<float>(reinterpret_cast<int64_t>(values)), static_cast<int64_t>(blockIdx.x) * kQuantizeRows, rows, cols,
                  stride, gin<double>(reinterpret_cast<int64_t>(scale)), gin<double>(reinterpret_cast<int64_t>(offset)),
                  gout<uint8_t>(reinterpret_cast<int64_t>(codes)), code_stride);
}

__global__ void __launch_bounds__(kThreads) quantize_batched_kernel(const rch_quantize_job* __restrict__ jobs) {
    const rch_quantize_job* J = jobs + blockIdx.y;
    const int64_t r0 = static_cast<int64_t>(blockIdx.x) * kQuantizeRows;
    if (r0 >= J->rows) return;
    const int cols = static_cast<int>(J->cols);
    const RCH_GLOBAL double* affine = gin<double>(J->affine_ptr);
    quantize_rows(gin<float>(J->values_ptr), r0, J->rows, cols, J->stride, affine, affine + cols, gout<uint8_t>(J->codes_ptr),
                  J->code_stride);
}

// ---------------------------------------------------------------------------------------------
// Batched FP64 Cholesky factor and triangular inverse (the planner's CholeskyQR steps): one
// 8-wave workgroup per k x k matrix, held in LDS (padded to whole 16-blocks with the identity).
// Bound by the chain of dependent pivots, so the work is blocked by 16 to keep everything but that
// chain off it: a column-at-a-time form with one workgroup barrier per factor column and per inverse
// row took 202 us for 60 matrices of order 96 (44 for 32), this one 73 (19) us (MI355X).
//
// Factorization, per 16-row panel: each wave holds the panel's diagonal block (lanes 0-15, one
// column each; every wave factors it, so no barrier is needed inside a panel) and 48 further
// columns (lanes 16-63); a step broadcasts the pivot and the pivot row's panel entries by readlane.
// Two barriers per panel: before and after the trailing update A -= R_p^T R_p (16 x 16 tiles, four
// elements per lane).
//
// Inverse X = R^-1: wave J computes block column J from the bottom with no barrier.  Block (I, J)
// sums S = sum_{I < P <= J} R_IP X_PJ (four rows per lane) and finishes by substitution in R_II (lane
// = column).  X_PJ is kept in the unused lower triangle, at block (J, P).
//
// Every element's products are rounded, then added in one fixed order (factor: pivot rows
// ascending; inverse: rows descending), whatever the blocking: no fused or matrix-unit products,
// whose different rounding would move near-tied row signs of the planner's directions.
// ---------------------------------------------------------------------------------------------

constexpr int kCholThreads = 512;
constexpr int kCholWaves = kCholThreads / 64;
constexpr int kCholBlocks = RCH_CHOLESKY_MAX_K / 16;
constexpr int kCholPitch = RCH_CHOLESKY_MAX_K + 1;
static_assert(RCH_CHOLESKY_MAX_K % 16 == 0 && kCholBlocks <= kCholWaves, "one wave per block column");

__device__ __forceinline__ double broadcast_lane(double v, int lane) {
    const u2 w = __builtin_bit_cast(u2, v);
    return __builtin_bit_cast(double, (u2{static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(w[0]), lane)),
                                          static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(w[1]), lane))}));
}

struct CholeskyShared {
    double m[RCH_CHOLESKY_MAX_K * kCholPitch];   // A, then R; below the diagonal blocks X transposed by blocks
    double inverse_diagonal[kCholBlocks][16 * 16];  // X_JJ
    double pivot_inverse[RCH_CHOLESKY_MAX_K];    // 1 / R[j][j]
    int failed_at;
};

// Factors the padded matrix in shared.m (upper triangle; visible to the workgroup) and inverts the
// factor; store(row, column, value) takes the upper-triangular X in blocks.  Returns 0, or the order of
// the first leading minor that is not positive definite (no X then).  Uniform over the workgroup.
template <class Store>
__device__ __forceinline__ int cholesky_invert(CholeskyShared& shared, int k, Store store) {
    constexpr int P = kCholPitch;
    double* const m = shared.m;
    double* const pivot_inverse = shared.pivot_inverse;
    auto& inverse_diagonal = shared.inverse_diagonal;
    int& failed_at = shared.failed_at;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int i16 = lane & 15, g = lane >> 4;
    const int blocks = (k + 15) >> 4, kp = 16 * blocks;
    for (int J = 0; J < blocks; ++J) {
        const int j0 = 16 * J;
        const int right = kp - j0 - 16;  // columns beside the diagonal block
        double v[16];
        if (wave == 0 || 48 * wave < right) {
            // Lower-triangle entries of the diagonal block's lanes are unset: they feed nothing and
            // are not written back.
            const int c = lane < 16 ? j0 + lane : j0 + 48 * wave + lane;
#pragma unroll
            for (int r = 0; r < 16; ++r) v[r] = c < kp ? m[(j0 + r) * P + c] : 0.0;
            int failed = 0;
#pragma unroll
            for (int j = 0; j < 16; ++j) {
                const double d = broadcast_lane(v[j], j);  // uniform
                if (failed == 0 && (!(d > 0.0) || !(d < INFINITY))) failed = j0 + j + 1;
                if (failed == 0) {
                    const double inv = 1.0 / sqrt(d);
                    v[j] *= inv;
                    if (wave == 0 && lane == 0) pivot_inverse[j0 + j] = inv;
#pragma unroll
                    for (int i = j + 1; i < 16; ++i) v[i] = v[i] - broadcast_lane(v[j], i) * v[j];
                }
            }
            if (wave == 0 && lane == 0) failed_at = failed;
            if (c < kp && lane >= 16) {
#pragma unroll
                for (int r = 0; r < 16; ++r) m[(j0 + r) * P + c] = v[r];
            }
        }
        __syncthreads();
        if (failed_at) break;  // uniform
        // The diagonal block goes back only now: every panel wave has read it.
        if (wave == 0 && lane < 16) {
#pragma unroll
            for (int r = 0; r < 16; ++r)
                if (r <= lane) m[(j0 + r) * P + j0 + lane] = v[r];
        }
        // Trailing tiles (ti <= tj) behind the panel, dealt to the waves.
        const int left = blocks - J - 1, count = left * (left + 1) / 2;
        for (int t = wave; t < count; t += kCholWaves) {
            int tj = 0, rest = t;
            while (rest > tj) {
                rest -= tj + 1;
                ++tj;
            }
            const int row = j0 + 16 + 16 * rest, col = j0 + 16 + 16 * tj;
            double acc[4];
#pragma unroll
            for (int v = 0; v < 4; ++v) acc[v] = m[(row + g + 4 * v) * P + col + i16];
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const double rc = m[(j0 + r) * P + col + i16];
#pragma unroll
                for (int v = 0; v < 4; ++v) acc[v] = acc[v] - m[(j0 + r) * P + row + g + 4 * v] * rc;
            }
#pragma unroll
            for (int v = 0; v < 4; ++v) m[(row + g + 4 * v) * P + col + i16] = acc[v];
        }
        __syncthreads();
    }
    if (failed_at) return failed_at;
    if (wave < blocks) {
        const int J = wave;
        for (int I = J; I >= 0; --I) {
            double* const slot = m + 16 * J * P + 16 * I;  // block (J, I): holds S, then X_IJ
            if (I < J) {
                double sum[4] = {0.0, 0.0, 0.0, 0.0};  // rows g + 4v, column i16
                for (int Q = J; Q > I; --Q) {
                    const double* r_iq = m + (16 * I + g) * P + 16 * Q;
                    const double* x_qj = Q == J ? inverse_diagonal[J] + i16 : m + 16 * J * P + 16 * Q + i16;
                    const int pitch = Q == J ? 16 : P;
#pragma unroll
                    for (int p = 15; p >= 0; --p) {
                        const double xv = x_qj[p * pitch];
#pragma unroll
                        for (int v = 0; v < 4; ++v) sum[v] = sum[v] + r_iq[4 * v * P + p] * xv;
                    }
                }
#pragma unroll
                for (int v = 0; v < 4; ++v) slot[(g + 4 * v) * P + i16] = sum[v];
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // other lanes of this wave read it
            }
            // Substitution: lane c holds column c of R_II and of S (the four lane groups repeat it).
            double t[16], sum[16], y[16];
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                t[r] = r <= i16 ? m[(16 * I + r) * P + 16 * I + i16] : 0.0;
                sum[r] = I < J ? slot[r * P + i16] : 0.0;
            }
#pragma unroll
            for (int i = 15; i >= 0; --i) {
                const double value = ((I == J && i == i16 ? 1.0 : 0.0) - sum[i]) * pivot_inverse[16 * I + i];
                y[i] = I == J && i > i16 ? 0.0 : value;
#pragma unroll
                for (int r = 0; r < i; ++r) sum[r] = sum[r] + broadcast_lane(t[r], i) * y[i];
            }
            if (lane < 16) {
                double* const to = I == J ? inverse_diagonal[J] + i16 : slot + i16;
                const int pitch = I == J ? 16 : P;
#pragma unroll
                for (int r = 0; r < 16; ++r) to[r * pitch] = y[r];
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            const int col = 16 * J + i16;
#pragma unroll
            for (int r = 0; r < 16; ++r)
                if ((r & 3) == g) store(16 * I + r, col, y[r]);
        }
    }
    return 0;
}

// Upper triangle of A (order k) into shared.m, padded to whole blocks with the identity.
__device__ __forceinline__ void cholesky_load(CholeskyShared& shared, const RCH_GLOBAL double* A, int k, int pitch) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, kp = padded_order(k);
    if (threadIdx.x == 0) shared.failed_at = 0;
    for (int i = wave; i < kp; i += kCholWaves)
        for (int c = i + lane; c < kp; c += 64)
            shared.m[i * kCholPitch + c] = (i < k && c < k) ? A[i * pitch + c] : (i == c ? 1.0 : 0.0);
    __syncthreads();
}

__global__ void __launch_bounds__(kCholThreads) cholesky_inverse_kernel(const double* __restrict__ a,
                                                                         double* __restrict__ x,
                                                                         int32_t* __restrict__ info, int k) {
    __shared__ CholeskyShared shared;
    const int64_t base = static_cast<int64_t>(blockIdx.x) * k * k;
    RCH_GLOBAL double* X = gout<double>(reinterpret_cast<int64_t>(x)) + base;
    cholesky_load(shared, gin<double>(reinterpret_cast<int64_t>(a)) + base, k, k);
    const int failed = cholesky_invert(shared, k, [&](int row, int col, double value) {
        if (row < k && col < k) X[row * k + col] = value;
    });
    if (threadIdx.x == 0) info[blockIdx.x] = failed;
    // The identity for a failed member, else zeros below the diagonal blocks.
    for (int e = threadIdx.x; e < k * k; e += kCholThreads) {
        const int row = e / k, col = e - row * k;
        if (failed) X[e] = row == col ? 1.0 : 0.0;
        else if ((row >> 4) > (col >> 4)) X[e] = 0.0;
    }
}

// ---------------------------------------------------------------------------------------------
// Terms of a stored basis view Q (order k <= RCH_CHOLESKY_MAX_K) and its coefficients P: the span trace
// trace(G^-1 C) with G = Q Q^T and C = P^T P, the Cholesky status of G, ||G - I||_inf, max |G_ii|,
// ||G||_inf and ||G^-1||_inf, in FP64.  Four launches for a batch of any ranks in place of some twenty
// library launches per rank group; each is latency- or FP64-rate-bound at a few tens of us:
//   * basis_gram_kernel: G (the projection's channel-split body on the basis rows);
//   * basis_terms_kernel: factor, X = R^-1, W = X X^T = G^-1 and the norms, one workgroup per matrix;
//   * span_trace_kernel: sum over tiles of W o C.  A workgroup keeps its token range's share of C in
//     accumulators and multiplies it by W at the end, so C is never written;
//   * span_total_kernel: the workgroups' sums in order.
// ---------------------------------------------------------------------------------------------

__global__ void __launch_bounds__(kThreads) basis_gram_kernel(const rch_fit_matrix* __restrict__ mats, int channels) {
    __shared__ double partial[2 * 4 * 4 * 64];  // the four waves' sums of two 16-column blocks
    const rch_fit_matrix* M = mats + blockIdx.z;
    const int kp = padded_order(static_cast<int>(M->rank));
    const int t0 = 16 * blockIdx.x, r0 = 32 * blockIdx.y;
    if (t0 >= kp || r0 >= kp) return;  // whole workgroup
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (t0 == 0 && r0 == 0 && threadIdx.x == 0)  // basis_terms_kernel puts the time since in its place
        gout<uint64_t>(M->energy_ptr)[6] = wall_clock64();
    if (r0 + 16 < kp) project_ranks<RCH_DT_F16, Project::kGram, 2>(M, channels, r0, t0, wave, lane, partial);
    else project_ranks<RCH_DT_F16, Project::kGram, 1>(M, channels, r0, t0, wave, lane, partial);
}

__global__ void __launch_bounds__(kCholThreads) basis_terms_kernel(const rch_fit_matrix* __restrict__ mats, double tick) {
    __shared__ CholeskyShared shared;
    constexpr int P = kCholPitch;
    const rch_fit_matrix* M = mats + blockIdx.x;
    const int k = static_cast<int>(M->rank), kp = padded_order(k), blocks = kp >> 4;
    const RCH_GLOBAL double* G = gin<double>(M->gram_ptr);
    RCH_GLOBAL double* W = gout<double>(M->gram_ptr) + kp * kp;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int i16 = lane & 15, g = lane >> 4;
    cholesky_load(shared, G, k, kp);
    // Row norms of G: four threads per row (k <= 128 rows), then the largest of the workgroup.
    const int row = tid >> 2, part = tid & 3;
    double eta = 0.0, largest = 0.0, norm = 0.0;
    if (row < k) {
        for (int c = part; c < k; c += 4) {
            const double v = G[row * kp + c];
            norm += fabs(v);
            eta += fabs(c == row ? v - 1.0 : v);
            if (c == row) largest = fabs(v);
        }
    }
    const int failed = cholesky_invert(shared, k, [](int, int, double) {});
    __syncthreads();
    // W_IJ = sum_{Q >= J} X_IQ X_JQ^T for I <= J, into the blocks R no longer needs.
    double* const m = shared.m;
    if (!failed) {
        auto x_at = [&](int I, int Q) -> const double* {
            return I == Q ? shared.inverse_diagonal[I] : m + 16 * Q * P + 16 * I;
        };
        for (int t = wave; t < blocks * (blocks + 1) / 2; t += kCholWaves) {
            int J = 0, I = t;
            while (I > J) {
                I -= J + 1;
                ++J;
            }
            d4 acc = d4{};
            for (int Q = J; Q < blocks; ++Q) {
                const double* left = x_at(I, Q);
                const double* right = x_at(J, Q);
                const int lp = I == Q ? 16 : P, rp = J == Q ? 16 : P;
#pragma unroll
                for (int s = 0; s < 4; ++s)
                    acc = __builtin_amdgcn_mfma_f64_16x16x4f64(left[i16 * lp + 4 * s + g], right[i16 * rp + 4 * s + g], acc, 0, 0, 0);
            }
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                m[(16 * I + g + 4 * v) * P + 16 * J + i16] = acc[v];
                W[(16 * I + g + 4 * v) * kp + 16 * J + i16] = acc[v];
            }
        }
    }
    __syncthreads();
    double inverse_norm = 0.0;
    if (row < k) {
        // Upper blocks hold W; entries below the diagonal blocks come from the transposed place.
        for (int c = part; c < k; c += 4)
            inverse_norm += fabs((c >> 4) >= (row >> 4) ? m[row * P + c] : m[c * P + row]);
    }
#pragma unroll
    for (int d = 1; d <= 2; d <<= 1) {
        norm += __shfl_xor(norm, d);
        eta += __shfl_xor(eta, d);
        largest = fmax(largest, __shfl_xor(largest, d));
        inverse_norm += __shfl_xor(inverse_norm, d);
    }
    // A NaN must survive the maximum: row sums that are not finite become infinity.
    norm = norm < INFINITY ? norm : INFINITY;
    eta = eta < INFINITY ? eta : INFINITY;
    inverse_norm = inverse_norm < INFINITY ? inverse_norm : INFINITY;
#pragma unroll
    for (int d = 4; d <= 32; d <<= 1) {
        norm = fmax(norm, __shfl_xor(norm, d));
        eta = fmax(eta, __shfl_xor(eta, d));
        largest = fmax(largest, __shfl_xor(largest, d));
        inverse_norm = fmax(inverse_norm, __shfl_xor(inverse_norm, d));
    }
    __syncthreads();
    double* const best = shared.pivot_inverse;
    if (lane == 0) {
        best[4 * wave] = eta;
        best[4 * wave + 1] = largest;
        best[4 * wave + 2] = norm;
        best[4 * wave + 3] = inverse_norm;
    }
    __syncthreads();
    if (tid == 0) {
        RCH_GLOBAL double* out = gout<double>(M->energy_ptr);
        out[0] = 0.0;
        out[1] = static_cast<double>(failed);
        for (int q = 0; q < 4; ++q) {
            double v = best[q];
            for (int w = 1; w < kCholWaves; ++w) v = fmax(v, best[4 * w + q]);
            out[2 + q] = v;
        }
        if (failed) out[5] = INFINITY;
        out[6] = static_cast<double>(wall_clock64() - gin<uint64_t>(M->energy_ptr)[6]) * tick;
    }
}

constexpr int kSpanThreads = 512;
constexpr int kSpanWaves = kSpanThreads / 64;
constexpr int kSpanTokens = 32;  // tokens staged at a time
constexpr int kSpanRange = 96;   // fewest tokens of a range
constexpr int kSpanTiles = (kCholBlocks * (kCholBlocks + 1) / 2 + kSpanWaves - 1) / kSpanWaves;  // per wave

// Tokens of a range (one workgroup, one partial sum), by the matrix's rows alone: its trace then has the same
// bits in every batch.  96 tokens or, beyond RCH_SPAN_SPLITS of those, an equal share: one matrix at rank 96
// takes 118 us (all four launches; 64 tokens 117, 256 125), 60 at ranks 32 to 128 283 (300, 291).
__device__ __forceinline__ int64_t span_range(int64_t rows) {
    const int64_t share = (rows + RCH_SPAN_SPLITS - 1) / RCH_SPAN_SPLITS;
    const int64_t whole = (share + kSpanTokens - 1) / kSpanTokens * kSpanTokens;
    return whole > kSpanRange ? whole : kSpanRange;
}

// Workgroup (token range, matrix): the 16 x 16 tiles (ti <= tj) of C are dealt to the waves; 32 tokens
// of P at a time are staged in LDS as doubles, the next 32 loaded meanwhile.
__global__ void __launch_bounds__(kSpanThreads) span_trace_kernel(const rch_fit_matrix* __restrict__ mats) {
    constexpr int kPitch = RCH_CHOLESKY_MAX_K + 16;
    __shared__ double staged[kSpanTokens * kPitch];
    __shared__ double sums[kSpanWaves];
    const rch_fit_matrix* M = mats + blockIdx.y;
    const int k = static_cast<int>(M->rank), kp = padded_order(k), blocks = kp >> 4;
    const int tiles = blocks * (blocks + 1) / 2;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int i16 = lane & 15, g = lane >> 4;
    const int64_t per = span_range(M->rows);
    const int64_t begin = blockIdx.x * per, end = begin + per < M->rows ? begin + per : M->rows;
    if (begin >= M->rows) return;  // whole workgroup
    int ti[kSpanTiles], tj[kSpanTiles];
    d4 acc[kSpanTiles];
#pragma unroll
    for (int q = 0; q < kSpanTiles; ++q) {
        int J = 0, I = wave + kSpanWaves * q;
        while (I > J) {
            I -= J + 1;
            ++J;
        }
        ti[q] = 16 * I;
        tj[q] = 16 * J;
        acc[q] = d4{};
    }
    // Thread -> (token, columns 8 part .. 8 part + 7) of a 32-token stage.
    const int token = tid >> 4, part = tid & 15;
    const bool mine = 8 * part < kp;
    float next[8];
    auto load = [&](int64_t t0) {
#pragma unroll
        for (int j = 0; j < 8; ++j) next[j] = 0.0f;
        if (mine && t0 + token < end) {
            const RCH_GLOBAL float* p = gin<float>(M->coef_ptr) + (t0 + token) * M->coef_stride + 8 * part;
#pragma unroll
            for (int j = 0; j < 8; ++j)
                if (8 * part + j < k) next[j] = p[j];
        }
    };
    load(begin);
    for (int64_t t0 = begin; t0 < end; t0 += kSpanTokens) {
        if (mine) {
#pragma unroll
            for (int j = 0; j < 8; ++j) staged[token * kPitch + 8 * part + j] = static_cast<double>(next[j]);
        }
        __syncthreads();
        load(t0 + kSpanTokens);
#pragma unroll
        for (int q = 0; q < kSpanTiles; ++q) {
            if (wave + kSpanWaves * q >= tiles) continue;  // uniform
#pragma unroll
            for (int s = 0; s < kSpanTokens / 4; ++s) {
                const double* r = staged + (4 * s + g) * kPitch + i16;
                acc[q] = __builtin_amdgcn_mfma_f64_16x16x4f64(r[ti[q]], r[tj[q]], acc[q], 0, 0, 0);
            }
        }
        __syncthreads();
    }
    const RCH_GLOBAL double* W = gin<double>(M->gram_ptr) + kp * kp;
    double sum = 0.0;
#pragma unroll
    for (int q = 0; q < kSpanTiles; ++q) {
        if (wave + kSpanWaves * q >= tiles) continue;
        double tile = 0.0;
#pragma unroll
        for (int v = 0; v < 4; ++v) tile = fma(W[(ti[q] + g + 4 * v) * kp + tj[q] + i16], acc[q][v], tile);
        sum += ti[q] == tj[q] ? tile : 2.0 * tile;
    }
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) sum += __shfl_xor(sum, d);
    if (lane == 0) sums[wave] = sum;
    __syncthreads();
    if (tid == 0) {
        for (int w = 1; w < kSpanWaves; ++w) sum += sums[w];
        gout<double>(M->partial_ptr)[blockIdx.x] = sum;
    }
}

// The span trace of each matrix from its workgroups' sums, in order (0 when G is not positive definite).
__global__ void __launch_bounds__(64) span_total_kernel(const rch_fit_matrix* __restrict__ mats, int n) {
    const int mat = blockIdx.x * 64 + threadIdx.x;
    if (mat >= n) return;
    const rch_fit_matrix* M = mats + mat;
    RCH_GLOBAL double* out = gout<double>(M->energy_ptr);
    const int64_t per = span_range(M->rows);
    const int ranges = static_cast<int>((M->rows + per - 1) / per);
    double sum = 0.0;
    for (int s = 0; s < ranges; ++s) sum += gin<double>(M->partial_ptr)[s];
    out[0] = out[1] == 0.0 ? sum : 0.0;
}

// ---------------------------------------------------------------------------------------------
// Seeded Gaussian columns (start blocks of the subspace solvers)
//
// Counter-based Philox-4x32-10 (Salmon, Moraes, Dror, Shaw, "Parallel random numbers: as easy as
// 1, 2, 3", SC 2011): the key is the job's 64-bit seed, the counter the index of a group of four
// elements, so every element has a fixed value whatever the launch shape.  Box-Muller turns each
// pair of 32-bit words into two standard normals.
// ---------------------------------------------------------------------------------------------

__device__ __forceinline__ void philox4x32_10(uint32_t (&c)[4], uint32_t k0, uint32_t k1) {
#pragma unroll
    for (int round = 0; round < 10; ++round) {
        const uint64_t p0 = static_cast<uint64_t>(0xD2511F53u) * c[0];
        const uint64_t p1 = static_cast<uint64_t>(0xCD9E8D57u) * c[2];
        const uint32_t hi0 = static_cast<uint32_t>(p0 >> 32), lo0 = static_cast<uint32_t>(p0);
        const uint32_t hi1 = static_cast<uint32_t>(p1 >> 32), lo1 = static_cast<uint32_t>(p1);
        c[0] = hi1 ^ c[1] ^ k0;
        c[1] = lo1;
        c[2] = hi0 ^ c[3] ^ k1;
        c[3] = lo0;
        k0 += 0x9E3779B9u;
        k1 += 0xBB67AE85u;
    }
}

__global__ void __launch_bounds__(256) gaussian_kernel(const rch_gauss_job* __restrict__ jobs) {
    const rch_gauss_job& J = jobs[blockIdx.y];
    const int64_t total = J.rows * J.cols;
    const int64_t group = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;  // elements 4 group .. + 3
    if (4 * group >= total) return;
    uint32_t c[4] = {static_cast<uint32_t>(group), static_cast<uint32_t>(group >> 32), 0u, 0u};
    philox4x32_10(c, static_cast<uint32_t>(J.seed), static_cast<uint32_t>(static_cast<uint64_t>(J.seed) >> 32));
    float z[4];
#pragma unroll
    for (int pair = 0; pair < 2; ++pair) {
        // Uniforms in (0, 1]: (word + 1) * 2^-32 keeps log away from zero.
        const float u1 = (static_cast<float>(c[2 * pair]) + 1.0f) * 2.3283064365386963e-10f;
        const float u2 = static_cast<float>(c[2 * pair + 1]) * 2.3283064365386963e-10f;
        const float r = sqrtf(-2.0f * logf(u1));
        z[2 * pair] = r * cosf(6.283185307179586f * u2);
        z[2 * pair + 1] = r * sinf(6.283185307179586f * u2);
    }
    RCH_GLOBAL float* dst = gout<float>(J.dst_ptr);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int64_t e = 4 * group + i;
        if (e < total) {
            const int64_t r = e / J.cols, col = e - r * J.cols;
            dst[r * J.stride + col] = z[i];
        }
    }
}

// The projection's 128-token workgroups run in rounds of one per CU.  They win while the last round is nearly
// full, else the finer shape, n matrices [4680, 1536] of bf16 (MI355X, us, kShared / kDeep; groups of kShared in
// brackets):
//   rank 96: 3 [222] 85 / 90, 4 [296] 153 / 107, 6 [444] 154 / 161, 8 [592] 227 / 206, 10 [740] 226 / 259,
//            12 [888] 297 / 302, 24 [1776] 514 / 596, 60 [4440] 1306 / 1465;
//   rank 32: 12 [444] 112 / 108, 20 [740] 165 / 178, 24 [888] 216 / 207, 30 [1110] 266 / 262, 60 [2220] 470 / 501;
//   fp32, rank 96: 8 225 / 205, 10 233 / 259, 12 299 / 310.
// In the finer shape 16-rank chunks balance few waves better, and 32-rank ones convert less: 38 / 38 us at one
// matrix of rank 96 (1758 tiles of 16 x 16), 62 / 65 at 3516, 113 / 107 at 7032; [390, 1536]: 12 / 19.
constexpr int64_t kChipCus = 256, kProjectNarrowTiles = 6000;
// The residual's 128-token form against the 16-token one, in 32-token groups: rank 96 49 / 41 us at 147 (one
// matrix), 66 / 64 at 294, 91 / 94 at 441, 104 / 117 at 588, 207 / 243 at 1176; rank 32 31 / 29 at 294, 47 / 49 at
// 588, 87 / 96 at 1176; fp32 the same within 2 us.  The source energy alone would stay with the 16-token form (60
// matrices 169 / 161), but one rule serves both.
static_assert(RCH_RESIDUAL_PARTS <= 16, "a wave keeps its parts' sums in 16 lanes");
constexpr int64_t kResidualSharedGroups = 500;  // of 32 tokens
// Workgroups that the channel splits aim at, and the fewest and most splits of the 128-token ones, which are
// long and at mixed ranks unequal (60 matrices at ranks 32 to 128: one 1415 us, three 1288, six 1276; a batch
// without bases, whose workgroups then end before their loads overlap, takes 169 at three and 191 at six).
constexpr int64_t kResidualSplitAim = 2000, kResidualSharedSplits = 3, kResidualSharedMost = 8;
constexpr int64_t kResidualSplits = 4;  // of 16-token tiles: a wave's first loads then serve one or two groups

int check_matrices(const rch_fit_matrix* mats, int n, int channels, const char* what) {
    if (!mats || n <= 0 || n > 65535) return fail(RCH_E_CONFIG, "%s: 1 <= n_mats <= 65535 required", what);
    if (channels <= 0 || channels % 8 != 0 || channels > (1 << 20))
        return fail(RCH_E_CONFIG, "%s: channels must be a positive multiple of 8", what);
    return RCH_OK;
}

}  // namespace
}  // namespace rch

using namespace rch;

#define RCH_DISPATCH_DTYPE_BLOCK(dtype, what, KERNEL, GRID, BLOCK, ...)                                             \
    switch (dtype) {                                                                                                \
        case RCH_DT_BF16: hipLaunchKernelGGL(KERNEL<RCH_DT_BF16>, GRID, dim3(BLOCK), 0, s, __VA_ARGS__); break;     \
        case RCH_DT_F16: hipLaunchKernelGGL(KERNEL<RCH_DT_F16>, GRID, dim3(BLOCK), 0, s, __VA_ARGS__); break;       \
        case RCH_DT_F32: hipLaunchKernelGGL(KERNEL<RCH_DT_F32>, GRID, dim3(BLOCK), 0, s, __VA_ARGS__); break;       \
        default: return fail(RCH_E_CONFIG, "%s: source dtype must be bf16, f16 or f32", what);                      \
    }

extern "C" {

int rch_fit_matrix_size(void) { return static_cast<int>(sizeof(rch_fit_matrix)); }

int rch_fit_absmax(const rch_fit_matrix* mats_dev, int n_mats, int channels, int64_t max_rows, int src_dtype,
                   void* stream) {
    if (int status = check_matrices(mats_dev, n_mats, channels, "rch_fit_absmax")) return status;
    if (max_rows <= 0 || (max_rows + kAbsmaxRows - 1) / kAbsmaxRows > 0x7fffffff)
        return fail(RCH_E_CONFIG, "rch_fit_absmax: invalid max_rows");
    const int64_t tiles = (max_rows + kAbsmaxRows - 1) / kAbsmaxRows;
    const int64_t wanted = tiles * n_mats / kAbsmaxGroups;
    const int sets = static_cast<int>(wanted < 1 ? 1 : (wanted > kAbsmaxSets ? kAbsmaxSets : wanted));
    const dim3 grid(static_cast<unsigned>((tiles + sets - 1) / sets), static_cast<unsigned>(n_mats));
    hipStream_t s = as_stream(stream);
    RCH_DISPATCH_DTYPE_BLOCK(src_dtype, "rch_fit_absmax", absmax_kernel, grid, kThreads, mats_dev, channels, sets);
    return check_launch("rch_fit_absmax");
}

int rch_fit_gram(const rch_fit_matrix* mats_dev, int n_mats, int channels, int src_dtype, void* stream) {
    if (int status = check_matrices(mats_dev, n_mats, channels, "rch_fit_gram")) return status;
    const int t = (channels + kGramTile - 1) / kGramTile;
    const int64_t tiles = static_cast<int64_t>(t) * (t + 1) / 2;
    if (tiles * n_mats > 0x7fffffff) return fail(RCH_E_CONFIG, "rch_fit_gram: too many tiles");
    const int grid = static_cast<int>(tiles * n_mats);
    hipStream_t s = as_stream(stream);
    RCH_DISPATCH_DTYPE_BLOCK(src_dtype, "rch_fit_gram", gram_kernel, dim3(grid), kGramThreads, mats_dev, channels,
                             static_cast<int>(tiles), grid);
    return check_launch("rch_fit_gram");
}

int rch_fit_project(const rch_fit_matrix* mats_dev, int n_mats, int channels, int64_t max_rows, int max_rank,
                    int src_dtype, void* stream) {
    if (int status = check_matrices(mats_dev, n_mats, channels, "rch_fit_project")) return status;
    if (max_rows <= 0 || max_rank <= 0 || (max_rows + 63) / 64 > 0x7fffffff || max_rank > channels)
        return fail(RCH_E_CONFIG, "rch_fit_project: invalid max_rows / max_rank");
    hipStream_t s = as_stream(stream);
    const unsigned z = static_cast<unsigned>(n_mats);
    // The fewest rank chunks of at most 64 ranks, as equal as 16-rank blocks allow.
    const int blocks = (max_rank + 15) / 16;
    int chunks = (blocks + 3) / 4, chunk = 16 * ((blocks + chunks - 1) / chunks);
    const int64_t groups = (max_rows + 127) / 128 * chunks * n_mats, rounds = (groups + kChipCus - 1) / kChipCus;
    if (7 * groups >= 6 * kChipCus * rounds) {
        const dim3 grid(static_cast<unsigned>((max_rows + 127) / 128), static_cast<unsigned>(chunks), z);
        switch (src_dtype) {
            case RCH_DT_BF16: hipLaunchKernelGGL((project_kernel<RCH_DT_BF16, Project::kShared>), grid, dim3(64 * kProjectWaves<Project::kShared>), 0, s, mats_dev, channels, chunk); break;
            case RCH_DT_F16: hipLaunchKernelGGL((project_kernel<RCH_DT_F16, Project::kShared>), grid, dim3(64 * kProjectWaves<Project::kShared>), 0, s, mats_dev, channels, chunk); break;
            case RCH_DT_F32: hipLaunchKernelGGL((project_kernel<RCH_DT_F32, Project::kShared>), grid, dim3(64 * kProjectWaves<Project::kShared>), 0, s, mats_dev, channels, chunk); break;
            default: return fail(RCH_E_CONFIG, "rch_fit_project: source dtype must be bf16, f16 or f32");
        }
    } else {
        chunk = (max_rows + 15) / 16 * blocks * n_mats < kProjectNarrowTiles ? 16 : 32;
        chunks = (max_rank + chunk - 1) / chunk;
        const dim3 grid(static_cast<unsigned>((max_rows + 31) / 32), static_cast<unsigned>(chunks), z);
        switch (src_dtype) {
            case RCH_DT_BF16: hipLaunchKernelGGL((project_kernel<RCH_DT_BF16, Project::kDeep>), grid, dim3(64 * kProjectWaves<Project::kDeep>), 0, s, mats_dev, channels, chunk); break;
            case RCH_DT_F16: hipLaunchKernelGGL((project_kernel<RCH_DT_F16, Project::kDeep>), grid, dim3(64 * kProjectWaves<Project::kDeep>), 0, s, mats_dev, channels, chunk); break;
            case RCH_DT_F32: hipLaunchKernelGGL((project_kernel<RCH_DT_F32, Project::kDeep>), grid, dim3(64 * kProjectWaves<Project::kDeep>), 0, s, mats_dev, channels, chunk); break;
            default: return fail(RCH_E_CONFIG, "rch_fit_project: source dtype must be bf16, f16 or f32");
        }
    }
    return check_launch("rch_fit_project");
}

int rch_fit_residual(const rch_fit_matrix* mats_dev, int n_mats, int channels, int64_t max_rows, int src_dtype,
                     void* stream) {
    if (int status = check_matrices(mats_dev, n_mats, channels, "rch_fit_residual")) return status;
    if (max_rows <= 0 || (max_rows + 15) / 16 > 0x7fffffff) return fail(RCH_E_CONFIG, "rch_fit_residual: invalid max_rows");
    hipStream_t s = as_stream(stream);
    // 128-token workgroups, the channels split where those are few, while their waves fill the chip, else
    // 16-token ones, the channels split as well.
    const bool shared = (max_rows + 31) / 32 * n_mats >= kResidualSharedGroups;
    const int tokens = shared ? kResidualTokens<true> : kResidualTokens<false>;
    const int at_once = shared ? kResidualAtOnce<true> : kResidualAtOnce<false>;
    const int64_t groups = (max_rows + tokens - 1) / tokens * n_mats;
    const int64_t wanted = std::max<int64_t>((kResidualSplitAim + groups - 1) / groups, shared ? kResidualSharedSplits : 1);
    const int64_t most = std::min<int64_t>((residual_parts(channels) + at_once - 1) / at_once,
                                           shared ? kResidualSharedMost : kResidualSplits);
    const int splits = static_cast<int>(std::min(wanted, most));
    const dim3 grid(static_cast<unsigned>((max_rows + tokens - 1) / tokens), static_cast<unsigned>(n_mats),
                    static_cast<unsigned>(splits));
    switch (src_dtype) {
        case RCH_DT_BF16:
            if (shared) hipLaunchKernelGGL((residual_kernel<RCH_DT_BF16, true>), grid, dim3(kThreads), 0, s, mats_dev, channels);
            else hipLaunchKernelGGL((residual_kernel<RCH_DT_BF16, false>), grid, dim3(kThreads), 0, s, mats_dev, channels);
            break;
        case RCH_DT_F16:
            if (shared) hipLaunchKernelGGL((residual_kernel<RCH_DT_F16, true>), grid, dim3(kThreads), 0, s, mats_dev, channels);
            else hipLaunchKernelGGL((residual_kernel<RCH_DT_F16, false>), grid, dim3(kThreads), 0, s, mats_dev, channels);
            break;
        case RCH_DT_F32:
            if (shared) hipLaunchKernelGGL((residual_kernel<RCH_DT_F32, true>), grid, dim3(kThreads), 0, s, mats_dev, channels);
            else hipLaunchKernelGGL((residual_kernel<RCH_DT_F32, false>), grid, dim3(kThreads), 0, s, mats_dev, channels);
            break;
        default: return fail(RCH_E_CONFIG, "rch_fit_residual: source dtype must be bf16, f16 or f32");
    }
    if (int status = check_launch("rch_fit_residual")) return status;
    hipLaunchKernelGGL(energy_total_kernel, dim3(n_mats), dim3(kTotalThreads), 0, s, mats_dev, channels);
    return check_launch("rch_fit_residual (totals)");
}

int rch_column_extrema(const float* values_dev, int64_t rows, int cols, int64_t stride, uint32_t* keys_dev,
                       void* stream) {
    if (!values_dev || !keys_dev || rows <= 0 || cols <= 0 || stride < cols || (rows + 63) / 64 > 0x7fffffff)
        return fail(RCH_E_CONFIG, "rch_column_extrema: invalid arguments");
    hipLaunchKernelGGL(extrema_kernel, dim3(static_cast<unsigned>((rows + 63) / 64)), dim3(kThreads), 0,
                       as_stream(stream), values_dev, rows, cols, stride, reinterpret_cast<unsigned int*>(keys_dev));
    return check_launch("rch_column_extrema");
}

int rch_quantize(const float* values_dev, int64_t rows, int cols, int64_t stride, const double* scale_dev,
                 const double* offset_dev, uint8_t* codes_dev, int64_t code_stride, void* stream) {
    if (!values_dev || !scale_dev || !offset_dev || !codes_dev || rows <= 0 || cols <= 0 || stride < cols ||
        code_stride < cols || (rows + kQuantizeRows - 1) / kQuantizeRows > 0x7fffffff)
        return fail(RCH_E_CONFIG, "rch_quantize: invalid arguments");
    hipLaunchKernelGGL(quantize_kernel, dim3(static_cast<unsigned>((rows + kQuantizeRows - 1) / kQuantizeRows)), dim3(kThreads), 0,
                       as_stream(stream), values_dev, rows, cols, stride, scale_dev, offset_dev, codes_dev, code_stride);
    return check_launch("rch_quantize");
}

int rch_cholesky_inverse(const double* a_dev, double* x_dev, int32_t* info_dev, int n, int k, void* stream) {
    if (!a_dev || !x_dev || !info_dev || n <= 0 || k <= 0 || k > RCH_CHOLESKY_MAX_K)
        return fail(RCH_E_CONFIG, "rch_cholesky_inverse: 1 <= k <= %d and device buffers required", RCH_CHOLESKY_MAX_K);
    hipLaunchKernelGGL(cholesky_inverse_kernel, dim3(static_cast<unsigned>(n)), dim3(kCholThreads), 0, as_stream(stream),
                       a_dev, x_dev, info_dev, k);
    return check_launch("rch_cholesky_inverse");
}

int rch_fit_span(const rch_fit_matrix* mats_dev, int n_mats, int channels, int64_t max_rows, int max_rank,
                 int with_coefficients, void* stream) {
    if (int status = check_matrices(mats_dev, n_mats, channels, "rch_fit_span")) return status;
    if (max_rank <= 0 || max_rank > RCH_CHOLESKY_MAX_K || (with_coefficients && max_rows <= 0))
        return fail(RCH_E_CONFIG, "rch_fit_span: 1 <= max_rank <= %d and positive max_rows required", RCH_CHOLESKY_MAX_K);
    hipStream_t s = as_stream(stream);
    const unsigned n = static_cast<unsigned>(n_mats);
    static const int khz = [] {  // of the clock that the terms' time is read from: the same on every gfx950
        int device = 0, rate = 0;
        const bool known = hipGetDevice(&device) == hipSuccess &&
                           hipDeviceGetAttribute(&rate, hipDeviceAttributeWallClockRate, device) == hipSuccess;
        return known && rate > 0 ? rate : 100000;
    }();
    hipLaunchKernelGGL(basis_gram_kernel, dim3((max_rank + 15) / 16, (max_rank + 31) / 32, n), dim3(kThreads), 0, s, mats_dev,
                       channels);
    hipLaunchKernelGGL(basis_terms_kernel, dim3(n), dim3(kCholThreads), 0, s, mats_dev, 1e-3 / khz);
    if (with_coefficients) {
        const int64_t ranges = std::min<int64_t>((max_rows + kSpanRange - 1) / kSpanRange, RCH_SPAN_SPLITS);
        hipLaunchKernelGGL(span_trace_kernel, dim3(static_cast<unsigned>(ranges), n), dim3(kSpanThreads), 0, s, mats_dev);
        hipLaunchKernelGGL(span_total_kernel, dim3((n + 63) / 64), dim3(64), 0, s, mats_dev, n_mats);
    }
    return check_launch("rch_fit_span");
}

int rch_fit_gaussian(const rch_gauss_job* jobs_dev, int n_jobs, int64_t max_elements, void* stream) {
    if (!jobs_dev || n_jobs <= 0 || n_jobs > 65535 || max_elements <= 0 || (max_elements + 1023) / 1024 > 0x7fffffff)
        return fail(RCH_E_CONFIG, "rch_fit_gaussian: invalid arguments");
    const dim3 grid(static_cast<unsigned>((max_elements + 1023) / 1024), static_cast<unsigned>(n_jobs));
    hipLaunchKernelGGL(gaussian_kernel, grid, dim3(256), 0, as_stream(stream), jobs_dev);
    return check_launch("rch_fit_gaussian");
}

int rch_quantize_batched(const rch_quantize_job* jobs_dev, int n_jobs, int64_t max_rows, void* stream) {
    if (!jobs_dev || n_jobs <= 0 || n_jobs > 65535 || max_rows <= 0 ||
        (max_rows + kQuantizeRows - 1) / kQuantizeRows > 0x7fffffff)
        return fail(RCH_E_CONFIG, "rch_quantize_batched: invalid arguments");
    const dim3 grid(static_cast<unsigned>((max_rows + kQuantizeRows - 1) / kQuantizeRows), static_cast<unsigned>(n_jobs));
    hipLaunchKernelGGL(quantize_batched_kernel, grid, dim3(kThreads), 0, as_stream(stream), jobs_dev);
    return check_launch("rch_quantize_batched");
}

}  // extern "C"
