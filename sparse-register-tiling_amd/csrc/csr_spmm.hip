// HIP CSR SpMM baseline: the reference's AVX-512 row-times-panel kernel
// (sbench/SOP/_C/pytorch_csr_wrapper.cpp:70-102, dispatch :140-191) laid out
// for 64-wide wavefronts.  One wavefront owns one row of A and a 64*V-column
// slice of B/C; each lane reads V consecutive B columns per stored entry and
// keeps V fp32 accumulators.  Per output element the accumulation is one fused
// multiply-add per stored entry in storage order, like the reference.
//
// The row's indices and values come 64 at a time, one per lane, in one
// coalesced load each (the next 64 while these run), and reach the wave as
// scalars by readlane; 16 B rows are on their way while 16 are
// multiplied.  Loads through the scalar unit, four entries at a time, left the
// wave waiting twice (indices, then rows) for every four entries.  A row is one
// chain, so the longest row's latency is the floor where the rows are few:
// 2048 x 512 at 90 % x 256 takes 12.4 us (46.8 with the scalar loads at one
// float per lane), 1024 x 4096 at 70 % x 512 132 (672).
#include <hip/hip_runtime.h>

#include "exec_kernel.h"
#include "srt_internal.h"

namespace srt {

namespace {

// B rows multiplied while as many are on their way (8: 17.9 us instead of 14.2
// for 2048 x 512 at 90 % x 256 in a graph).
constexpr int kBatch = 16;

// BIG: B is larger than the 4 GiB a buffer descriptor and a 32-bit offset reach.
template <typename I, int V, bool BIG>
__global__ void __launch_bounds__(256)
    csr_kernel(int m, int k, int n, I nnz, const I *__restrict__ rowptr,
               const I *__restrict__ colind, const float *__restrict__ vals,
               const float *__restrict__ B, int64_t ldb, float *__restrict__ C, int64_t ldc,
               int row_groups) {
    typedef typename VecAt4<V>::type vec;
    const int waves = blockDim.x >> 6;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    const int b = xcd_swizzle(blockIdx.x, gridDim.x);
    const int ntile = b / row_groups;
    const int rg = b - ntile * row_groups;
    const int row = rg * waves + wave;
    if (row >= m) return;
    // The lane's columns; the last lane moves back where V does not divide n
    // (n >= V): it repeats columns of the lane before it, bit for bit.
    const int col = ntile * (64 * V) + lane * V;
    const bool active = col < n;
    const int cl = !active ? 0 : col + V <= n ? col : n - V;
    BRows<V> rows;
    if constexpr (!BIG) {
        rows.rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(B), (short)0,
                                                      (int)(uint32_t)(((int64_t)(k - 1) * ldb + n) * 4), 0x00020000);
        rows.voff = (uint32_t)cl * 4u;
        rows.row_bytes = 1;  // offsets arrive in bytes
    }
    float acc[V];
#pragma unroll
    for (int j = 0; j < V; ++j) acc[j] = 0.0f;
    // Entries outside [0, nnz) and column indices outside [0, k) are never
    // dereferenced: rows are clamped to the arrays, bad columns are skipped.
    I q = rowptr[row];
    I end = rowptr[row + 1];
    q = q < 0 ? 0 : (q > nnz ? nnz : q);
    end = end > nnz ? nnz : (end < q ? q : end);
    // Lane l holds entry l of 64: B row offset (bytes, or rows when BIG) and
    // value; a lane without one holds row 0 and is not multiplied.
    // Ends are compared as differences: within 64 entries of the largest I a
    // sum past the end wraps to an index below the arrays.
    I c = -1;
    float a = 0.0f;
    auto fetch = [&](I at) {
        c = -1;
        if (lane < end - at) {
            c = colind[at + lane];
            a = vals[at + lane];
        }
    };
    int off = 0, val = 0;
    auto take = [&]() {
        const bool ok = c >= 0 && c < (I)k;
        off = !ok ? 0 : BIG ? (int)c : (int)((uint32_t)c * ((uint32_t)ldb * 4u));
        val = __builtin_bit_cast(int, ok ? a : 0.0f);
    };
    vec r0[kBatch], r1[kBatch];
    auto load = [&](vec (&r)[kBatch], int j) {
#pragma unroll
        for (int u = 0; u < kBatch; ++u) {
            if constexpr (BIG)
                r[u] = *reinterpret_cast<const vec *>(B + (int64_t)__builtin_amdgcn_readlane(off, j + u) * ldb + cl);
            else
                r[u] = rows.load(__builtin_amdgcn_readlane(off, j + u));
        }
    };
    auto add = [&](const vec (&r)[kBatch], int from, int j, int count) {
#pragma unroll
        for (int u = 0; u < kBatch; ++u)
            if (u < count) {
                const float v = __builtin_bit_cast(float, __builtin_amdgcn_readlane(from, j + u));
#pragma unroll
                for (int i = 0; i < V; ++i) {
                    if constexpr (V == 1) acc[i] = __builtin_fmaf(v, r[u], acc[i]);
                    else acc[i] = __builtin_fmaf(v, r[u][i], acc[i]);
                }
            }
    };
    fetch(q);
    if (q < end) {
        take();
        load(r0, 0);
    }
    for (; end - q > 64; q += 64) {
        fetch(q + 64);
        load(r1, 16);
        add(r0, val, 0, kBatch);
        load(r0, 32);
        add(r1, val, 16, kBatch);
        load(r1, 48);
        add(r0, val, 32, kBatch);
        const int last = val;
        take();
        load(r0, 0);
        add(r1, last, 48, kBatch);
    }
    // The last 1 to 64 entries.
    const int left = (int)(end - q);
    if (left > 16) load(r1, 16);
    add(r0, val, 0, left);
    if (left > 16) {
        if (left > 32) load(r0, 32);
        add(r1, val, 16, left - 16);
    }
    if (left > 32) {
        if (left > 48) load(r1, 48);
        add(r0, val, 32, left - 32);
    }
    if (left > 48) add(r1, val, 48, left - 48);
    if (active) {
        vec o;
        if constexpr (V == 1) {
            o = acc[0];
        } else {
#pragma unroll
            for (int j = 0; j < V; ++j) o[j] = acc[j];
        }
        __builtin_nontemporal_store(o, reinterpret_cast<vec *>(C + (int64_t)row * ldc + cl));
    }
}

// Many rows of few entries, two or four floats per lane.  The kernel above asks
// for 16 B rows whatever a row holds, and its registers leave three or four
// waves a SIMD; here there are eight.  A wave takes its row's entries four at a
// time, indices and values through the scalar unit.  A row of more than kLongRow
// entries is the whole workgroup's: each of its four waves takes a quarter of
// the columns at one float per lane, 64 entries a load and 16 B rows ahead, as
// above.  us above and here: 40000 rows of 1 entry x 352 41.0 and 20.7, of 8 51.4
// and 36.0; 5000 rows of 4 x 1616 26.1 and 15.0; 20000 of 8 x 256, ten of them of
// 5000, 128 and 150 (759 four entries at a time).
constexpr int kLongRow = 32;

template <typename I, int V>
__global__ void __launch_bounds__(256)
    csr_short_kernel(int m, int k, int n, I nnz, const I *__restrict__ rowptr, const I *__restrict__ colind,
                     const float *__restrict__ vals, const float *__restrict__ B, int64_t ldb, float *__restrict__ C,
                     int64_t ldc, int row_groups) {
    typedef typename VecAt4<V>::type vec;
    constexpr int W = 4;  // waves, rows of a workgroup
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    const int b = xcd_swizzle(blockIdx.x, gridDim.x);
    const int ntile = b / row_groups;
    const int row0 = (b - ntile * row_groups) * W;
    // Entries of a row, inside [0, nnz) whatever the row pointers hold.
    auto range = [&](int row, I &q, I &end) {
        q = rowptr[row];
        end = rowptr[row + 1];
        q = q < 0 ? 0 : (q > nnz ? nnz : q);
        end = end > nnz ? nnz : (end < q ? q : end);
    };
    const __amdgpu_buffer_rsrc_t rsrc =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(B), (short)0,
                                          (int)(uint32_t)(((int64_t)(k - 1) * ldb + n) * 4), 0x00020000);
    const uint32_t row_bytes = (uint32_t)ldb * 4u;
    const int row = row0 + wave;
    I q = 0, end = 0;
    __shared__ int long_row[W];
    if (row < m) range(row, q, end);
    if (lane == 0) long_row[wave] = end - q > kLongRow;
    __syncthreads();
    int rest = 0;  // rows that are the workgroup's
#pragma unroll
    for (int i = 0; i < W; ++i) rest |= long_row[i] << i;
    rest = __builtin_amdgcn_readfirstlane(rest);
    if (row < m && end - q <= kLongRow) {
        const int col = ntile * (64 * V) + lane * V;
        const bool active = col < n;
        const int cl = !active ? 0 : col + V <= n ? col : n - V;
        const BRows<V> from{rsrc, (uint32_t)cl * 4u, 1};
        vec acc = {};
        vec r[4];
        float a[4];
        auto load = [&](int u) {
            const I c = colind[q + u];
            const bool ok = c >= 0 && c < (I)k;
            r[u] = from.load((int)((uint32_t)(ok ? c : 0) * row_bytes));
            a[u] = ok ? vals[q + u] : 0.0f;
        };
        auto add = [&](int u) {
#pragma unroll
            for (int i = 0; i < V; ++i) acc[i] = __builtin_fmaf(a[u], r[u][i], acc[i]);
        };
        for (; end - q >= 4; q += 4) {
#pragma unroll
            for (int u = 0; u < 4; ++u) load(u);
#pragma unroll
            for (int u = 0; u < 4; ++u) add(u);
        }
        for (; q < end; ++q) {
            load(0);
            add(0);
        }
        if (active) __builtin_nontemporal_store(acc, reinterpret_cast<vec *>(C + (int64_t)row * ldc + cl));
    }
    const int col = ntile * (64 * V) + wave * (16 * V) + lane;
    const bool active = lane < 16 * V && col < n;
    const BRows<1> from{rsrc, (uint32_t)(active ? col : 0) * 4u, 1};
#pragma unroll 1
    for (; rest; rest &= rest - 1) {
        const int i = __builtin_ctz(rest);
        range(row0 + i, q, end);
        constexpr int D = 16;  // rows multiplied while as many are on their way
        float r0[D], r1[D], acc = 0.0f, a = 0.0f;
        I c = -1;
        int at = 0, val = 0;
        auto fetch = [&](I from) {
            c = -1;
            if (lane < end - from) {
                c = colind[from + lane];
                a = vals[from + lane];
            }
        };
        auto take = [&]() {
            const bool ok = c >= 0 && c < (I)k;
            at = ok ? (int)((uint32_t)c * row_bytes) : 0;
            val = __builtin_bit_cast(int, ok ? a : 0.0f);
        };
        auto ask = [&](float (&r)[D], int j) {
#pragma unroll
            for (int u = 0; u < D; ++u) r[u] = from.load(__builtin_amdgcn_readlane(at, j + u));
        };
        auto sum = [&](const float (&r)[D], int from, int j, int count) {
#pragma unroll
            for (int u = 0; u < D; ++u)
                if (u < count)
                    acc = __builtin_fmaf(__builtin_bit_cast(float, __builtin_amdgcn_readlane(from, j + u)), r[u], acc);
        };
        fetch(q);
        take();
        ask(r0, 0);
        for (; end - q > 64; q += 64) {
            fetch(q + 64);
            ask(r1, D);
            sum(r0, val, 0, D);
            ask(r0, 2 * D);
            sum(r1, val, D, D);
            ask(r1, 3 * D);
            sum(r0, val, 2 * D, D);
            const int last = val;
            take();
            ask(r0, 0);
            sum(r1, last, 3 * D, D);
        }
        const int left = (int)(end - q);  // 1 to 64
        if (left > D) ask(r1, D);
        sum(r0, val, 0, left);
        if (left > D) {
            if (left > 2 * D) ask(r0, 2 * D);
            sum(r1, val, D, left - D);
        }
        if (left > 2 * D) {
            if (left > 3 * D) ask(r1, 3 * D);
            sum(r0, val, 2 * D, left - 2 * D);
        }
        if (left > 3 * D) sum(r1, val, 3 * D, left - 3 * D);
        if (active) __builtin_nontemporal_store(acc, C + (int64_t)(row0 + i) * ldc + col);
    }
}

template <typename I, int V>
hipError_t launch_csr_t(int m, int k, int n, int64_t nnz, const I *rowptr, const I *colind,
                        const float *vals, const float *B, int64_t ldb, float *C, int64_t ldc,
                        hipStream_t s) {
    const int waves = 4;
    const int row_groups = (m + waves - 1) / waves;
    const int n_tiles = (n + 64 * V - 1) / (64 * V);
    const long long nblocks = (long long)row_groups * n_tiles;
    if (nblocks == 0) return hipSuccess;
    if (nblocks > 0x7fffffffLL) return hipErrorInvalidConfiguration;
    const bool big = (int64_t)k * ldb * (int64_t)sizeof(float) > (int64_t)0xffffffffLL || k < 1;
    auto kernel = big ? csr_kernel<I, V, true> : csr_kernel<I, V, false>;
    // Few entries a row, and workgroups enough (four per CU) that the time is
    // work and not latency: with fewer, and from 12 entries on, the kernels are
    // even or the other one leads (600 rows of 4 x 352: 3.5 us, 3.7 short).
    if constexpr (V > 1)
        if (!big && nblocks >= 1024 && nnz <= 8 * (int64_t)m) kernel = csr_short_kernel<I, V>;
    hipLaunchKernelGGL(kernel, dim3((unsigned)nblocks), dim3(64 * waves), 0, s, m, k, n, (I)nnz, rowptr, colind, vals, B,
                       ldb, C, ldc, row_groups);
    return hipGetLastError();
}

template <typename I>
hipError_t launch_csr_i(int m, int k, int n, int64_t nnz, const void *rowptr, const void *colind,
                        const float *vals, const float *B, int64_t ldb, float *C, int64_t ldc, int V,
                        hipStream_t s) {
    const I *rp = (const I *)rowptr;
    const I *ci = (const I *)colind;
    switch (V) {
        case 4: return launch_csr_t<I, 4>(m, k, n, nnz, rp, ci, vals, B, ldb, C, ldc, s);
        case 2: return launch_csr_t<I, 2>(m, k, n, nnz, rp, ci, vals, B, ldb, C, ldc, s);
        default: return launch_csr_t<I, 1>(m, k, n, nnz, rp, ci, vals, B, ldb, C, ldc, s);
    }
}

}  // namespace

hipError_t launch_csr(int m, int k, int n, int64_t nnz, const void *rowptr, const void *colind,
                      int index_bytes, const float *vals, const float *B, int64_t ldb, float *C,
                      int64_t ldc, int vec_width, hipStream_t s) {
    if (index_bytes == 8)
        return launch_csr_i<int64_t>(m, k, n, nnz, rowptr, colind, vals, B, ldb, C, ldc, vec_width, s);
    return launch_csr_i<int32_t>(m, k, n, nnz, rowptr, colind, vals, B, ldb, C, ldc, vec_width, s);
}

}  // namespace srt
