// Streamed executor: C = A . B for packings whose chains run in column order
// (M_r = 1: every panel is one row, every packed column one nonzero).
//
// Why it exists.  The gather executor (exec_kernel.h) fetches one B row slice
// per packed column through the vector L1, which returns 64 bytes per clock
// and CU: 16 clocks per packed column and 256 C columns, and that rate bounds
// it.  The LDS of this chip returns 256 bytes per clock and CU for 16-byte
// lane reads (measured, conflict free: 252; 126 for 8- and 4-byte reads), so
// the same slice costs 4 clocks from there.  A column-ordered chain can be cut
// at any column, so B is walked in tiles of T rows that fit the LDS, whatever
// K is, and the result is still the sequential fused multiply-add chain.
//
// A workgroup owns W waves x R rows of C and one slice of 64 * V columns:
// lane l holds columns n0 + l * V .. + V of its wave's R rows.  Per tile:
//   - the B rows of the next tile are loaded into registers (kStageChunks
//     16-byte chunks per thread), one barrier makes the current tile visible,
//   - every wave runs its entries of the tile from the LDS,
//   - the registers are written to the other LDS buffer.
// Entries reach the wave through the scalar unit as blocks of S: S values,
// then S LDS byte offsets.  Four consecutive slots share an accumulator row
// (its number sits in the low byte of the first one's offset; offsets are
// multiples of 256 * V), so a block costs S / 4 uniform branches however the
// rows' nonzeros fall.  A row's entries of a tile are padded to four with an
// identity: value -0.0 against a row of +0.0 leaves every accumulator, signed
// zero and NaN included, as it is.
//
// Measured (4096 x 1024 at 80 % times 1024 x 2048): 110.7 us, the gather
// executor 168.7 (31.1 and 20.4 TFLOP/s).  What bounds it is instruction
// issue: per entry a wave issues V multiply-adds, an LDS read and about one
// scalar instruction, 4.3 and 4.4 clocks of a SIMD each (8 multiply-adds and 8
// scalar instructions together take 44 clocks), and waits for its scalar
// loads; LDS reads alone would take 51 us, the multiply-adds 22.  Half the
// bytes per entry (16-bit row words) took 138 us, since unpacking costs scalar
// instructions; entries through vector registers (DPP broadcasts 139 us,
// readlane 280) and blocks fetched into the L2 a tile ahead (142) were slower.
// Staging costs a workgroup the L2's 64 bytes per clock and CU, shared by its
// W * R rows: with few rows (little work) the gather executor is the faster.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "exec_kernel.h"
#include "srt_internal.h"

namespace srt {
namespace {

constexpr int kStageChunks = 4;  // 16-byte chunks of a tile held per thread

// B rows of one tile: kStageChunks chunks per thread of W waves.
constexpr int tile_rows(int V, int W) { return kStageChunks * 64 * W / (16 * V); }

// Entries per block, the unit of the scalar loads and of the reads in flight:
// as many as the row registers (2 x S x V) leave room for.
constexpr int block_slots(int V) { return V == 4 ? 8 : 16; }

// In the low byte of a block's first offset.
constexpr uint32_t kLastFlag = 16;  // the last block of a tile that is not the last
constexpr uint32_t kEndFlag = 32;   // the wave's last block

typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));
typedef float f2u __attribute__((ext_vector_type(2), aligned(4)));

template <int S>
__device__ __forceinline__ void load_words(const uint32_t *__restrict__ p, uint32_t (&out)[S]) {
    uint32_t __attribute__((ext_vector_type(S))) v;
    __builtin_memcpy(&v, p, sizeof(v));
#pragma unroll
    for (int i = 0; i < S; ++i) out[i] = v[i];
}

template <int V, int S>
struct Stream {
    typename VecOf<V>::type rows[S];  // B rows of the block
    uint32_t vals[S];                 // its values
    uint32_t offs[S];                 // offsets of the block after it
};

template <int V, int S>
__device__ __forceinline__ void read_rows(typename VecOf<V>::type (&rows)[S], const uint32_t (&offs)[S],
                                          const char *__restrict__ lds_lane) {
#pragma unroll
    for (int s = 0; s < S; ++s) {
        const uint32_t o = s % 4 == 0 ? offs[s] & ~0xffu : offs[s];
        rows[s] = *reinterpret_cast<const typename VecOf<V>::type *>(lds_lane + o);
    }
}

// Four slots into one accumulator row.
template <int V, int S>
__device__ __forceinline__ void quad_fmas(float (&acc)[V], const typename VecOf<V>::type (&rows)[S],
                                          const uint32_t (&vals)[S], int s0) {
#pragma unroll
    for (int s = s0; s < s0 + 4; ++s) {
        const float a = __builtin_bit_cast(float, vals[s]);
#pragma unroll
        for (int j = 0; j < V; ++j) acc[j] = __builtin_fmaf(a, lane_elem<V>(rows[s], j), acc[j]);
    }
}

template <int V, int R, int S>
__device__ __forceinline__ void block_fmas(float (&acc)[R][V], const typename VecOf<V>::type (&rows)[S],
                                           const uint32_t (&vals)[S], const uint32_t (&meta)[S / 4]) {
#define SRT_ROW(n)                                                       \
    case n:                                                              \
        if constexpr (n < R) quad_fmas<V, S>(acc[n], rows, vals, 4 * q); \
        break
#pragma unroll
    for (int q = 0; q < S / 4; ++q) {
        if constexpr (R == 1) {
            quad_fmas<V, S>(acc[0], rows, vals, 4 * q);
        } else {
            switch (meta[q] & (R - 1)) {
                SRT_ROW(0);
                SRT_ROW(1);
                SRT_ROW(2);
                SRT_ROW(3);
                SRT_ROW(4);
                SRT_ROW(5);
                SRT_ROW(6);
                SRT_ROW(7);
            }
        }
    }
#undef SRT_ROW
}

// Chunk c of this thread: row k0 + i / CH, columns n0 + 4 * (i % CH) .. + 4.
// Rows past K repeat the last one and columns past N read as zero (outside
// the buffer) or as the next row's: no entry and no stored lane uses them.
template <int V>
__device__ __forceinline__ void stage_load(float4 (&reg)[kStageChunks], __amdgpu_buffer_rsrc_t B, uint32_t row_bytes,
                                           int K, bool whole, int n0, int k0) {
    constexpr int CH = 16 * V;
#pragma unroll
    for (int c = 0; c < kStageChunks; ++c) {
        const int i = threadIdx.x + c * blockDim.x;
        const int k = k0 + i / CH < K ? k0 + i / CH : K - 1;
        const uint32_t off = (uint32_t)k * row_bytes + (uint32_t)(n0 + i % CH * 4) * 4u;
        if (whole) {  // uniform: every column of the slice exists
            reg[c] = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(B, off, 0, 0));
        } else {
            reg[c].x = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(B, off, 0, 0));
            reg[c].y = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(B, off + 4, 0, 0));
            reg[c].z = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(B, off + 8, 0, 0));
            reg[c].w = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(B, off + 12, 0, 0));
        }
    }
}

template <int V>
__device__ __forceinline__ void stage_store(const float4 (&reg)[kStageChunks], float *__restrict__ tile) {
#pragma unroll
    for (int c = 0; c < kStageChunks; ++c) {
        const int i = threadIdx.x + c * blockDim.x;
        *reinterpret_cast<float4 *>(tile + 4 * i) = reg[c];
    }
}

// The B tiles of one workgroup's slice: the current one in the LDS, the next
// one in registers.
template <int V>
struct Tiles {
    __amdgpu_buffer_rsrc_t rsrc;
    uint32_t row_bytes;
    int K, n0, T, n_tiles, t;
    bool whole;
    float *lds;  // tile buffer 0, a row of zeros, tile buffer 1 (n_tiles > 1)
    float4 reg[kStageChunks];

    __device__ __forceinline__ void fetch(int tile) {
        stage_load<V>(reg, rsrc, row_bytes, K, whole, n0, tile * T);
    }
    __device__ __forceinline__ void put(int tile) {
        stage_store<V>(reg, lds + (tile & 1 ? (T + 1) * 64 * V : 0));
    }
    // From tile t to t + 1.  Its buffer was last read before the barrier that
    // opened tile t, which every wave has passed.
    __device__ __forceinline__ void advance() {
        ++t;
        put(t);
        __syncthreads();
        if (t + 1 < n_tiles) fetch(t + 1);
    }
};

// One block: open the next tile if this block closes one, read the next
// block's rows, load the words after that, multiply.
template <int V, int R, int S>
__device__ __forceinline__ void stream_step(float (&acc)[R][V], const Stream<V, S> &in, Stream<V, S> &out,
                                            uint32_t (&meta)[S / 4], const uint32_t *__restrict__ blocks,
                                            uint32_t &at, Tiles<V> &tiles, const char *__restrict__ lds_lane) {
    // Scalar loads and LDS reads share one wait counter and scalar loads may
    // return out of order.  Everything this block needs was asked for by the
    // one before: one wait here, none between the loads issued below and the
    // multiply-adds.
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
    uint32_t now[S / 4];
#pragma unroll
    for (int q = 0; q < S / 4; ++q) {
        now[q] = meta[q];
        meta[q] = in.offs[4 * q];
    }
    if (now[0] & kLastFlag) tiles.advance();
    read_rows<V, S>(out.rows, in.offs, lds_lane);
    load_words<S>(blocks + at * (2 * S), out.vals);
    load_words<S>(blocks + at * (2 * S) + 3 * S, out.offs);
    ++at;
    block_fmas<V, R, S>(acc, in.rows, in.vals, now);
}

template <int V, int R>
__global__ void __launch_bounds__(1024)
    stream_kernel(const uint32_t *__restrict__ blocks, const uint32_t *__restrict__ first,
                  const int32_t *__restrict__ rows_of, const float *__restrict__ B, int64_t ldb,
                  float *__restrict__ C, int64_t ldc, int N, int K, int n_wg, int n_tiles, int xcd_remap) {
    constexpr int S = block_slots(V);
    extern __shared__ float lds[];
    const int waves = blockDim.x >> 6;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    int b = blockIdx.x;
    if (xcd_remap) b = xcd_swizzle(b, gridDim.x);
    const int slice = b / n_wg;
    const int wg = b - slice * n_wg;
    const int n0 = slice * (64 * V);
    const char *lds_lane = reinterpret_cast<const char *>(lds) + lane * 4 * V;
    Tiles<V> tiles;
    tiles.row_bytes = (uint32_t)ldb * 4u;
    tiles.K = K;
    tiles.n0 = n0;
    tiles.T = kStageChunks * 64 * waves / (16 * V);
    tiles.n_tiles = n_tiles;
    tiles.t = 0;
    tiles.whole = n0 + 64 * V <= N;
    tiles.lds = lds;
    tiles.rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(B), (short)0,
                                                   (int)((uint32_t)(K - 1) * tiles.row_bytes + (uint32_t)N * 4u),
                                                   0x00020000);
    tiles.fetch(0);
    uint32_t at = first[wg * waves + wave];
    Stream<V, S> s0, s1;
    uint32_t meta[S / 4];
    load_words<S>(blocks + at * (2 * S) + S, s1.offs);
    load_words<S>(blocks + at * (2 * S), s0.vals);
    load_words<S>(blocks + at * (2 * S) + 3 * S, s0.offs);
    ++at;
    float acc[R][V];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int j = 0; j < V; ++j) acc[r][j] = 0.0f;
    if (threadIdx.x < 64 * V) lds[tiles.T * 64 * V + threadIdx.x] = 0.0f;
    tiles.put(0);
    __syncthreads();
    if (n_tiles > 1) tiles.fetch(1);
#pragma unroll
    for (int q = 0; q < S / 4; ++q) meta[q] = s1.offs[4 * q];
    read_rows<V, S>(s0.rows, s1.offs, lds_lane);
    while (true) {  // two blocks per trip: the stages alternate without copies
        const uint32_t end0 = meta[0] & kEndFlag;
        stream_step<V, R, S>(acc, s0, s1, meta, blocks, at, tiles, lds_lane);
        if (end0) break;
        const uint32_t end1 = meta[0] & kEndFlag;
        stream_step<V, R, S>(acc, s1, s0, meta, blocks, at, tiles, lds_lane);
        if (end1) break;
    }

    const int n = n0 + lane * V;
    if (n >= N) return;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int row = rows_of[(wg * waves + wave) * R + r];
        if (row >= 0) {
            float *c = C + (int64_t)row * ldc + n;
            if (V == 1 || n + V <= N) {
                if constexpr (V == 4) {
                    f4u v = {acc[r][0], acc[r][1], acc[r][2], acc[r][3]};
                    __builtin_nontemporal_store(v, reinterpret_cast<f4u *>(c));
                } else if constexpr (V == 2) {
                    f2u v = {acc[r][0], acc[r][1]};
                    __builtin_nontemporal_store(v, reinterpret_cast<f2u *>(c));
                } else {
                    __builtin_nontemporal_store(acc[r][0], c);
                }
            } else {
#pragma unroll
                for (int j = 0; j < V; ++j)
                    if (n + j < N) c[j] = acc[r][j];
            }
        }
    }
}

// ---------------------------------------------------------------- schedule
// First entry of row `row` with column >= k (entries are column ordered).
__device__ __forceinline__ int64_t entry_at(const int32_t *__restrict__ cols, int64_t lo, int64_t hi, int k) {
    while (lo < hi) {
        const int64_t mid = (lo + hi) >> 1;
        if (cols[mid] < k) lo = mid + 1; else hi = mid;
    }
    return lo;
}

// One wavefront per stream wave: blocks of each tile (lane = tile, 64 at a
// time) and in all.  Every tile has at least one block.
__global__ void stream_count_kernel(int n_waves, int R, int S, int T, int n_tiles, const int32_t *__restrict__ rows_of,
                                    const int64_t *__restrict__ col_ptr, const int32_t *__restrict__ cols,
                                    int32_t *__restrict__ tile_blocks, uint32_t *__restrict__ total) {
    const int w = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
    if (w >= n_waves) return;
    const int lane = threadIdx.x & 63;
    uint32_t sum = 0;
    for (int t = lane; t < n_tiles; t += 64) {
        int quads = 0;
        for (int r = 0; r < R; ++r) {
            const int row = rows_of[w * R + r];
            if (row < 0) continue;
            const int64_t lo = col_ptr[row], hi = col_ptr[row + 1];
            const int64_t a = entry_at(cols, lo, hi, t * T), e = entry_at(cols, a, hi, (t + 1) * T);
            quads += (int)((e - a + 3) / 4);
        }
        const int blk = quads > 0 ? (quads * 4 + S - 1) / S : 1;
        tile_blocks[(int64_t)w * n_tiles + t] = blk;
        sum += blk;
    }
    for (int off = 32; off > 0; off >>= 1) sum += __shfl_xor(sum, off);
    if (lane == 0) total[w] = sum;
}

// One wavefront per stream wave writes its blocks, lanes over the slots of a
// tile: slot -> (row, entry) through the running quads of the wave's rows.
__global__ void stream_fill_kernel(int n_waves, int R, int S, int V, int T, int n_tiles,
                                   const int32_t *__restrict__ rows_of, const int64_t *__restrict__ col_ptr,
                                   const int32_t *__restrict__ cols, const float *__restrict__ vals,
                                   const int32_t *__restrict__ tile_blocks, const uint32_t *__restrict__ first,
                                   uint32_t *__restrict__ blocks) {
    const int w = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
    if (w >= n_waves) return;
    const int lane = threadIdx.x & 63;
    const uint32_t row_bytes = 256u * V;
    const uint32_t zero_row = (uint32_t)T * row_bytes;
    int64_t at = first[w];
    // lane r < R walks its row's entries tile by tile
    const int my = lane < R ? rows_of[w * R + lane] : -1;
    int64_t pos = my >= 0 ? col_ptr[my] : 0;
    const int64_t hi = my >= 0 ? col_ptr[my + 1] : 0;
    for (int t = 0; t < n_tiles; ++t) {
        const int64_t e = my >= 0 ? entry_at(cols, pos, hi, (t + 1) * T) : 0;
        const int cnt = (int)(e - pos);
        int quads_end = (cnt + 3) / 4;  // inclusive running quads over lanes 0..lane
        for (int off = 1; off < 8; off <<= 1) {
            const int up = __shfl_up(quads_end, off);
            if (lane >= off) quads_end += up;
        }
        const int blk = tile_blocks[(int64_t)w * n_tiles + t];
        const uint32_t buffer = t & 1 ? zero_row + row_bytes : 0;
        for (int s0 = 0; s0 < blk * S; s0 += 64) {
            const int s = s0 + lane;
            int r = 0, begin = 0;
            for (int q = 0; q < R; ++q) {
                const int end = __shfl(quads_end, q);
                if (s / 4 >= end) {
                    r = q + 1;
                    begin = end;
                }
            }
            const bool in = r < R;
            const int src = in ? r : 0;
            const int64_t p0 = __shfl(pos, src);
            const int n = __shfl(cnt, src);
            const int idx = s - 4 * begin;
            float v = -0.0f;
            uint32_t o = zero_row;
            if (in && idx < n) {
                v = vals[p0 + idx];
                o = buffer + (uint32_t)(cols[p0 + idx] - t * T) * row_bytes;
            }
            if (s % 4 == 0) o |= (uint32_t)src;
            if (s == (blk - 1) * S) o |= t + 1 < n_tiles ? kLastFlag : kEndFlag;
            if (s < blk * S) {
                const int64_t bk = at + s / S;
                blocks[bk * (2 * S) + s % S] = __builtin_bit_cast(uint32_t, v);
                blocks[bk * (2 * S) + S + s % S] = o;
            }
        }
        at += blk;
        pos = my >= 0 ? e : 0;
    }
}

template <int V, int R>
hipError_t launch_vr(const StreamLaunch &a, hipStream_t s) {
    const int T = tile_rows(V, a.waves);
    const int n_tiles = (a.K + T - 1) / T;
    const size_t lds = (size_t)(n_tiles > 1 ? 2 : 1) * T * 256 * V + 256 * V;
    const long long grid = (long long)a.n_wg * ((a.N + 64 * V - 1) / (64 * V));
    if (grid > 0x7fffffffLL) return hipErrorInvalidConfiguration;
    if (lds > 65536) {
        static const hipError_t raised =
            hipFuncSetAttribute(reinterpret_cast<const void *>(&stream_kernel<V, R>),
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_limit());
        if (raised != hipSuccess) return raised;
    }
    hipLaunchKernelGGL((stream_kernel<V, R>), dim3((unsigned)grid), dim3(64 * a.waves), lds, s, a.blocks, a.first,
                       a.rows_of, a.B, a.ldb, a.C, a.ldc, a.N, a.K, a.n_wg, n_tiles, a.xcd_remap);
    return hipGetLastError();
}

template <int V>
hipError_t launch_v(const StreamLaunch &a, hipStream_t s) {
    switch (a.R) {
        case 1: return launch_vr<V, 1>(a, s);
        case 2: return launch_vr<V, 2>(a, s);
        case 4: return launch_vr<V, 4>(a, s);
        default: return launch_vr<V, 8>(a, s);
    }
}

}  // namespace

int stream_tile_rows(int V, int waves) { return tile_rows(V, waves); }
int stream_block_words(int V) { return 2 * block_slots(V); }

hipError_t launch_stream(const StreamLaunch &a, hipStream_t s) {
    if (a.N <= 0 || a.K <= 0 || a.n_wg <= 0) return hipSuccess;
    switch (a.V) {
        case 4: return launch_v<4>(a, s);
        case 2: return launch_v<2>(a, s);
        default: return launch_v<1>(a, s);
    }
}

hipError_t launch_stream_count(int n_waves, int R, int V, int waves, int K, const int32_t *rows_of,
                               const int64_t *col_ptr, const int32_t *cols, int32_t *tile_blocks, uint32_t *total,
                               hipStream_t s) {
    const int T = tile_rows(V, waves);
    hipLaunchKernelGGL(stream_count_kernel, dim3((n_waves + 3) / 4), dim3(256), 0, s, n_waves, R, block_slots(V), T,
                       (K + T - 1) / T, rows_of, col_ptr, cols, tile_blocks, total);
    return hipGetLastError();
}

hipError_t launch_stream_fill(int n_waves, int R, int V, int waves, int K, const int32_t *rows_of,
                              const int64_t *col_ptr, const int32_t *cols, const float *vals,
                              const int32_t *tile_blocks, const uint32_t *first, uint32_t *blocks, hipStream_t s) {
    const int T = tile_rows(V, waves);
    hipLaunchKernelGGL(stream_fill_kernel, dim3((n_waves + 3) / 4), dim3(256), 0, s, n_waves, R, block_slots(V), V, T,
                       (K + T - 1) / T, rows_of, col_ptr, cols, vals, tile_blocks, first, blocks);
    return hipGetLastError();
}

}  // namespace srt
