// Dense 16-row panels of a hybrid plan on FP32 matrix cores.
//
// The reference pads column patterns up to denser kernel patterns by its ILP
// cost model (sbench/ilp_pad/nano_solver.py:76-116) and calls a tile dense
// past a density threshold (sbench/padding_reordering.py:36, 0.30).  A
// hybrid plan takes the 16-row panels at or above its threshold out of the
// register-tiled packing and stores them dense for v_mfma_f32_16x16x4_f32:
// per panel and 16-column K group g, lane l holds the four k-steps it feeds,
//   A[row = l % 16][k = 16 g + 4 j + l / 16],  j = 0..3,
// as one 16-byte word (one load per lane per K group).
//
// An output tile is kTP panels (16 kTP rows) x kNTiles 16-column MFMA tiles:
// 128 x 128, 64 x 64 or 32 x 64.  A large tile reads A and B from L2
// least often, a small one gives more workgroups and a shorter chain, so fewer
// K splits, whose partials are written and read again.  A workgroup is 8 waves,
// two per SIMD: wave w computes the panels of half w / 4 against a quarter
// w % 4 of the columns (eight 16 x 16 accumulators of a 128 x 128 tile, one of
// 32 x 64).  K advances in stages of 64 (4 groups) through two LDS buffers
// holding the stage's A words (as stored) and B block in MFMA B-operand order,
//   lb[group q][column tile t][lane l] = B[16 q + 4 j + l / 16][16 t + l % 16], j = 0..3,
// the lane index XORed with t % 4: the four lanes of a writing quarter-wave
// that share a column group hit different banks (792 conflict cycles a stage
// without, 264 with).  Per stage: the next stage's global loads are issued
// first, the MFMAs of group q run while group q + 1's operands are read from
// LDS, the next stage's words are written to the other buffer in the middle of
// group 1 (in group 2 they hold up the narrow B loads of widths that 4 does not
// divide: 720 x 2751 x 727 takes 49.0 us, 44.8 so), and the one barrier sits
// before group 3, whose MFMAs hide the next stage's first reads.  Loads two
// stages ahead gave no more (156 us against 154 at 1024 x 16384 x 512): large
// products run at 0.76 of the matrix cores' cycles.
//
// K is cut into ranges, one chain of additions each, and ranges into groups (long
// ones each its own, short ones at most eight); a range's sum joins its group's,
// the groups' sums are added in order.  A workgroup takes whole groups, so tile
// and split change no bit of C.
// With S > 1 workgroups per tile each stores its groups' sums (lane order) to a
// workspace, and dense_tiles_reduce adds them in order and writes C: results
// repeat bit for bit.
//
// Workgroups map to (split, tile) split-major, blocks b, b + 8, ... on one
// XCD taking consecutive logical ids: with S = 8 each XCD owns one K range,
// whose A and B slices fit its L2.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "srt_internal.h"

namespace srt {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kSG = 4;              // 16-column K groups per stage (64 k)
constexpr int kWaves = 8;
constexpr int kThreads = 64 * kWaves;
constexpr int kXcds = 8;
constexpr int kMaxRanges = 32;
constexpr int kFewGroups = 8;

// Workspace words (f32x4) of one (group, tile): every wave's accumulators.
constexpr int64_t tile_words(int tp, int nt16) { return (int64_t)tp * nt16 * 64; }

template <bool kVecB, int kTP, int kNTiles>
__global__ void __launch_bounds__(kThreads)
    dense_tiles_kernel(int ndense, int G, int PT, int NT, int S, int SPC, int CPG, int GPS, const f32x4 *__restrict__ apack,
                       uint32_t a_bytes, const int32_t *__restrict__ panel_row, const float *__restrict__ B,
                       int64_t ldb, uint32_t b_bytes, float *__restrict__ C, int64_t ldc, f32x4 *__restrict__ ws,
                       int M, int N, int K) {
    constexpr int kTN = 16 * kNTiles;               // columns of a tile
    constexpr int kPM = kTP / 2, kPN = kNTiles / 4;  // panels and column tiles of a wave
    constexpr int kAW = kTP * kSG * 64 / kThreads;  // A words of a thread per stage
    constexpr int kBC = kNTiles / 2;                // B columns of a thread per stage
    typedef float fb __attribute__((ext_vector_type(kBC)));
    __shared__ f32x4 la[2][kTP][kSG][64];
    __shared__ f32x4 lb[2][kSG][kNTiles][64];
    const int T = PT * NT, total = T * S;
    const int b = blockIdx.x;
    const int L = (total % kXcds == 0) ? (b % kXcds) * (total / kXcds) + b / kXcds : b;
    const int split = L / T, tile = L % T;
    const int pt = tile / NT, nt = tile % NT;
    const int stages = (G + kSG - 1) / kSG;
    const int s0 = split * GPS * CPG * SPC, s1 = min(stages, s0 + GPS * CPG * SPC);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    const int mw = wave >> 2, nw = wave & 3;

    // Buffer loads: an offset past the resource's extent reads 0, so groups
    // past G, rows past K, columns past N and panels past the list need no
    // branch (the stage after the last reads zeros, written but never used).
    const __amdgpu_buffer_rsrc_t brsrc =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(B), (short)0, (int)b_bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t arsrc =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<f32x4 *>(apack), (short)0, (int)a_bytes, 0x00020000);

    // A staging: word e = tid + 512 r of the stage's [kTP panels][4 groups][64 lanes]
    f32x4 ra[kAW];
    fb rb[4];
    auto load_a = [&](int s, bool ok) {
#pragma unroll
        for (int r = 0; r < kAW; ++r) {
            const int e = threadIdx.x + kThreads * r;
            const int p = e / (kSG * 64), q = (e >> 6) % kSG, l = e & 63;
            const int d = pt * kTP + p, g = s * kSG + q;
            const uint32_t off = (ok & (d < ndense) & (g < G))
                                     ? ((uint32_t)(d * G + g) * 64u + (uint32_t)l) * 16u
                                     : 0xffffffffu;
            ra[r] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(arsrc, off, 0, 0));
        }
    };
    auto write_a = [&](int buf) {
#pragma unroll
        for (int r = 0; r < kAW; ++r) {
            const int e = threadIdx.x + kThreads * r;
            la[buf][e / (kSG * 64)][(e >> 6) % kSG][e & 63] = ra[r];
        }
    };
    // B staging: thread owns rows 16 q + 4 j + kr (j = 0..3) x kBC columns of
    // the tile (512 threads = 16 (q, kr) x 32 c4)
    const int c4 = threadIdx.x & 31, qk = threadIdx.x >> 5;
    const int bq = qk >> 2, bkr = qk & 3;
    const int bn = nt * kTN + kBC * c4;
    auto load_b = [&](int s, bool ok) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int k = s * (16 * kSG) + 16 * bq + 4 * j + bkr;
            const bool rowok = ok & (k < K);
            if constexpr (kVecB) {
                const uint32_t at = ((uint32_t)k * (uint32_t)ldb + (uint32_t)bn) * 4u;
                const uint32_t off = (rowok & (bn < N)) ? at : 0xffffffffu;
                if constexpr (kBC == 4)
                    rb[j] = __builtin_bit_cast(fb, __builtin_amdgcn_raw_buffer_load_b128(brsrc, off, 0, 0));
                else
                    rb[j] = __builtin_bit_cast(fb, __builtin_amdgcn_raw_buffer_load_b64(brsrc, off, 0, 0));
            } else {
#pragma unroll
                for (int c = 0; c < kBC; ++c) {
                    const uint32_t at = ((uint32_t)k * (uint32_t)ldb + (uint32_t)(bn + c)) * 4u;
                    const uint32_t off = (rowok & (bn + c < N)) ? at : 0xffffffffu;
                    rb[j][c] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(brsrc, off, 0, 0));
                }
            }
        }
    };
    auto write_b = [&](int buf) {
#pragma unroll
        for (int c = 0; c < kBC; ++c) {
            const int col = kBC * c4 + c;
            lb[buf][bq][col >> 4][(bkr * 16 + (col & 15)) ^ (col >> 4 & 3)] = f32x4{rb[0][c], rb[1][c], rb[2][c], rb[3][c]};
        }
    };

    f32x4 acc[kPM][kPN], group[kPM][kPN], sum[kPM][kPN];  // chain, sum of a group's chains, of groups
#pragma unroll
    for (int p = 0; p < kPM; ++p)
#pragma unroll
        for (int t = 0; t < kPN; ++t) acc[p][t] = group[p][t] = sum[p][t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    f32x4 a[2][kPM], bw[2][kPN];  // operands of two groups: one in use, one being read
    auto rd = [&](int buf, int q, int h) {
#pragma unroll
        for (int p = 0; p < kPM; ++p) a[h][p] = la[buf][kPM * mw + p][q][lane];
#pragma unroll
        for (int t = 0; t < kPN; ++t) bw[h][t] = lb[buf][q][kPN * nw + t][lane ^ ((kPN * nw + t) & 3)];
    };
    auto mm = [&](int h) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int p = 0; p < kPM; ++p)
#pragma unroll
                for (int t = 0; t < kPN; ++t)
                    acc[p][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[h][p][j], bw[h][t][j], acc[p][t], 0, 0, 0);
    };
    constexpr int kMF = 4 * kPM * kPN;  // MFMAs of a group
    constexpr int kRD = kPM + kPN;      // LDS reads of a group
    constexpr int kH = kMF / 16 > 0 ? kMF / 16 : 1;

    load_a(s0, true);
    load_b(s0, true);
    write_a(0);
    write_b(0);
    __syncthreads();
    rd(0, 0, 0);
    int chain = 0, groups = 0;
    for (int s = s0; s < s1;) {
        const int end = min(s1, s + SPC);
        for (; s < end; ++s) {
            const int buf = (s - s0) & 1;
            const bool more = s + 1 < s1;
            load_a(s + 1, more);
            load_b(s + 1, more);
            rd(buf, 1, 1);
            mm(0);
            rd(buf, 2, 0);
            mm(1);
            write_a(buf ^ 1);
            write_b(buf ^ 1);
            rd(buf, 3, 1);
            mm(0);
            // that order, interleaved: global loads first; each group's next
            // operands after its first two MFMAs; the other buffer's writes in
            // the middle of group 1
            __builtin_amdgcn_sched_group_barrier(0x020, kAW + 4, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, kH, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, kRD, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, kMF - kH, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, kH, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, kRD, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, kMF / 2 - kH, 0);
            __builtin_amdgcn_sched_group_barrier(0x200, kAW + kBC, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, kMF / 2, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, kH, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, kRD, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, kMF - kH, 0);
            __builtin_amdgcn_sched_barrier(0);
            __syncthreads();
            __builtin_amdgcn_sched_barrier(0);
            rd(buf ^ 1, 0, 0);  // the next stage's group 0 (after the last stage: unused words)
            mm(1);
            __builtin_amdgcn_sched_group_barrier(0x100, kRD, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, kMF, 0);
        }
        // the end of a range joins its group's sum
#pragma unroll
        for (int p = 0; p < kPM; ++p)
#pragma unroll
            for (int t = 0; t < kPN; ++t) {
                group[p][t] = chain == 0 ? acc[p][t] : group[p][t] + acc[p][t];
                acc[p][t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            }
        if (++chain < CPG && s < s1) continue;
        chain = 0;  // the end of a group
        if (S == 1) {
#pragma unroll
            for (int p = 0; p < kPM; ++p)
#pragma unroll
                for (int t = 0; t < kPN; ++t) sum[p][t] = groups == 0 ? group[p][t] : sum[p][t] + group[p][t];
        } else {
            f32x4 *out =
                ws + ((int64_t)((split * GPS + groups) * T + tile) * kWaves + wave) * (kPM * kPN) * 64 + lane;
#pragma unroll
            for (int p = 0; p < kPM; ++p)
#pragma unroll
                for (int t = 0; t < kPN; ++t) out[(p * kPN + t) * 64] = group[p][t];
        }
        ++groups;
    }
    if (S == 1) {
        // D layout: lane l holds rows 4 (l / 16) .. + 3 of column l % 16
#pragma unroll
        for (int p = 0; p < kPM; ++p) {
            const int d = pt * kTP + kPM * mw + p;
            if (d >= ndense) continue;
            const int row0 = panel_row[d];
#pragma unroll
            for (int t = 0; t < kPN; ++t) {
                const int n = nt * kTN + 16 * (kPN * nw + t) + (lane & 15);
                if (n >= N) continue;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int row = row0 + 4 * (lane >> 4) + r;
                    if (row < M) C[(int64_t)row * ldc + n] = sum[p][t][r];
                }
            }
        }
    }
}

// One thread per (tile, wave, accumulator, lane): the Q groups' sums added in
// order, then written to C.
template <int kTP, int kNTiles>
__global__ void __launch_bounds__(256)
    dense_tiles_reduce(int ndense, int PT, int NT, int Q, const f32x4 *__restrict__ ws,
                       const int32_t *__restrict__ panel_row, float *__restrict__ C, int64_t ldc, int M, int N) {
    constexpr int kPM = kTP / 2, kPN = kNTiles / 4;
    constexpr int kTileWords = (int)tile_words(kTP, kNTiles);
    const int T = PT * NT;
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= (int64_t)T * kTileWords) return;
    const int tile = (int)(i / kTileWords), w0 = (int)(i % kTileWords);
    const int lane = w0 & 63, pt2 = (w0 >> 6) % (kPM * kPN), wave = (w0 >> 6) / (kPM * kPN);
    const int pt = tile / NT, nt = tile % NT;
    const int mw = wave >> 2, nw = wave & 3, p = pt2 / kPN, t = pt2 % kPN;
    const int d = pt * kTP + kPM * mw + p;
    const int n = nt * 16 * kNTiles + 16 * (kPN * nw + t) + (lane & 15);
    if (d >= ndense || n >= N) return;
    const int64_t stride = (int64_t)T * kTileWords;
    f32x4 v = ws[i];
    const f32x4 *p1 = ws + i + stride;
    int left = Q - 1;
    for (; left >= 4; left -= 4, p1 += 4 * stride) {  // four loads in flight
        f32x4 w[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) w[u] = p1[u * stride];
#pragma unroll
        for (int u = 0; u < 4; ++u) v += w[u];
    }
    if (left == 3) {
        const f32x4 w0 = p1[0], w1 = p1[stride], w2 = p1[2 * stride];
        v += w0;
        v += w1;
        v += w2;
    } else {
        for (; left > 0; --left, p1 += stride) v += p1[0];
    }
    const int row0 = panel_row[d];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int row = row0 + 4 * (lane >> 4) + r;
        if (row < M) C[(int64_t)row * ldc + n] = v[r];
    }
}

// Tile and K split of a launch.  K is cut into the ranges that fill the chip
// with 128 x 128 tiles, at most 32 (SPC stages each); CPG ranges form a group; a
// workgroup takes GPS of the Q groups.
struct DenseGrid {
    int tp, nt16, PT, NT, SPC, CPG, Q, GPS, S;
};

int dense_ranges(int ndense, int stages, int N, int *stages_each) {
    const int tiles = ((ndense + 7) / 8) * ((N + 127) / 128);
    const int ranges = std::max(1, std::min({kMaxRanges, 256 / std::max(tiles, 1), stages}));
    *stages_each = (stages + ranges - 1) / ranges;
    return (stages + *stages_each - 1) / *stages_each;  // no empty range
}

// The launch of least modelled time among the tiles and splits that the
// workspace holds; another than 128 x 128 tiles with a workgroup per group has
// to gain 6 %.  The model, in us: a launch, a stage of a workgroup's chain, the
// matrix work of the CU with most workgroups, the operand bytes, and for a
// split the second launch and its partials.  Least squares over 123 problems
// (256..4096 rows and depth, 32..2048 columns); its choice takes 1.02 of the
// fastest launch's time on average, 128 x 128 tiles with a workgroup per range,
// the only launch before, 1.35 (512 x 512 x 128: 12.0 us, now 6.8; 512 x 2048 x
// 256: 21.3, now 13.5; 4096 x 4096 x 64: 47.0, now 28.8; 2048 x 2048 x 1024: 83
// both).
DenseGrid dense_grid(int ndense, int G, int N, size_t ws_words) {
    static constexpr struct {
        int tp, nt16;
        double stage;
    } kTiles[] = {{8, 8, 0.0}, {4, 4, .099}, {2, 4, .174}};
    const int stages = std::max(1, (G + kSG - 1) / kSG);
    DenseGrid best{}, g;
    const int ranges = dense_ranges(ndense, stages, N, &g.SPC);
    // A range of three stages or more is its own group, which keeps 128 x 128
    // tiles busy; shorter ones form at most eight, since their partials would
    // cost more (2920 x 2692 x 128, 11 ranges of 4 stages: 36.8 us in 6 groups,
    // 30.1 in 11; 761 x 1012 x 192, 16 of 1: 13.0 in 8, 16.9 in 16).
    g.CPG = g.SPC >= 3 ? 1 : (ranges + kFewGroups - 1) / kFewGroups;
    g.Q = (ranges + g.CPG - 1) / g.CPG;
    double best_t = -1.0;
    for (const auto &tile : kTiles) {
        g.tp = tile.tp;
        g.nt16 = tile.nt16;
        g.PT = (ndense + g.tp - 1) / g.tp;
        g.NT = (N + 16 * g.nt16 - 1) / (16 * g.nt16);
        const int64_t T = (int64_t)g.PT * g.NT;
        // the last one, all groups in one workgroup, needs no workspace
        for (g.GPS = 1;; g.GPS = std::min(2 * g.GPS, g.Q)) {
            g.S = (g.Q + g.GPS - 1) / g.GPS;
            const int64_t words = g.Q * T * tile_words(g.tp, g.nt16);
            if (g.S == 1 || (size_t)words <= ws_words) {
                const double chain = std::min(stages, g.SPC * g.CPG * g.GPS);
                double t = 6.6 + tile.stage * chain + 4.32 / 64 * chain * ((g.S * T + 255) / 256) * (g.tp * g.nt16) +
                           0.222 / 4096 * g.S * T * chain * (g.tp + g.nt16);
                if (g.S > 1) t += 0.63 + 0.88e-6 * 4 * (2 * g.Q + 1) * T * tile_words(g.tp, g.nt16);
                if (best_t < 0)
                    best_t = .94 * t, best = g;
                else if (t < best_t)
                    best_t = t, best = g;
            }
            if (g.GPS == g.Q) break;
        }
    }
    return best;
}

}  // namespace

// What 128 x 128 tiles with a workgroup per range would take at n columns or
// any fewer (fewer columns are split further, so they may take more), at most
// 256 tiles or 16 MB; groups are fewer and the padding of smaller tiles is
// less, so no launch takes more.
size_t dense_panels_workspace_bytes(int ndense, int G, int n) {
    if (ndense <= 0 || n <= 0) return 0;
    const int stages = std::max(1, (G + kSG - 1) / kSG), pt = (ndense + 7) / 8;
    int64_t most = 0;
    for (int nt = 1; nt <= (n + 127) / 128 && (int64_t)pt * nt <= 128; ++nt) {
        int each = 0;
        const int ranges = dense_ranges(ndense, stages, 128 * nt, &each);
        if (ranges > 1) most = std::max(most, (int64_t)ranges * pt * nt);
    }
    return (size_t)most * tile_words(8, 8) * sizeof(f32x4);
}

template <int kTP, int kNTiles>
static hipError_t launch_dense_tiles(const DenseGrid &g, bool vec, int ndense, int G, const void *apack,
                                     uint32_t a_bytes, const int32_t *panel_row, const float *B, int64_t ldb,
                                     uint32_t b_bytes, float *C, int64_t ldc, int M, int N, int K, void *ws,
                                     hipStream_t s) {
    const dim3 grid((unsigned)(g.PT * g.NT * g.S));
    if (vec)
        hipLaunchKernelGGL((dense_tiles_kernel<true, kTP, kNTiles>), grid, dim3(kThreads), 0, s, ndense, G, g.PT,
                           g.NT, g.S, g.SPC, g.CPG, g.GPS, static_cast<const f32x4 *>(apack), a_bytes, panel_row, B, ldb,
                           b_bytes, C, ldc, static_cast<f32x4 *>(ws), M, N, K);
    else
        hipLaunchKernelGGL((dense_tiles_kernel<false, kTP, kNTiles>), grid, dim3(kThreads), 0, s, ndense, G, g.PT,
                           g.NT, g.S, g.SPC, g.CPG, g.GPS, static_cast<const f32x4 *>(apack), a_bytes, panel_row, B, ldb,
                           b_bytes, C, ldc, static_cast<f32x4 *>(ws), M, N, K);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || g.S == 1) return e;
    const int64_t threads = (int64_t)g.PT * g.NT * tile_words(kTP, kNTiles);
    hipLaunchKernelGGL((dense_tiles_reduce<kTP, kNTiles>), dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, s,
                       ndense, g.PT, g.NT, g.Q, static_cast<const f32x4 *>(ws), panel_row, C, ldc, M, N);
    return hipGetLastError();
}

hipError_t launch_dense_panels(int ndense, int G, const void *apack, const int32_t *panel_row, const float *B,
                               int64_t ldb, float *C, int64_t ldc, int M, int N, int K, void *ws, size_t ws_bytes,
                               hipStream_t s) {
    if (ndense <= 0 || N <= 0) return hipSuccess;
    // byte offsets are 32-bit (buffer loads); the extent must stay below the
    // 0xffffffff offset that marks a zero read
    const int64_t a_bytes = (int64_t)ndense * G * 64 * 16, b_bytes = (int64_t)K * ldb * 4;
    if (a_bytes >= 0xffffffffLL || b_bytes >= 0xffffffffLL) return hipErrorInvalidValue;
    const DenseGrid g = dense_grid(ndense, G, N, ws ? ws_bytes / sizeof(f32x4) : 0);
    const bool vec = N % 4 == 0 && ldb % 4 == 0 && (uintptr_t)B % 16 == 0;
    auto launch = g.tp == 8   ? launch_dense_tiles<8, 8>
                  : g.tp == 4 ? launch_dense_tiles<4, 4>
                              : launch_dense_tiles<2, 4>;
    return launch(g, vec, ndense, G, apack, (uint32_t)a_bytes, panel_row, B, ldb, (uint32_t)b_bytes, C, ldc, M, N, K,
                  ws, s);
}

}  // namespace srt
