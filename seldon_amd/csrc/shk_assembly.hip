// shk_assembly.hip -- CSR assembly from coordinates on the device
// (Seldon's ConvertMatrix_from_Coordinates for RowSparse).
//
// Seldon sorts the entries by row with its bottom-up MergeSort, counts the
// rows into Ptr, then sorts each row by column with the same MergeSort
// (matrix_sparse/Matrix_Conversions.cxx:1288-1335).  That merge takes from
// the right run only on a strictly smaller key (vector/Functions_Arrays.cxx:
// 412-480), so it is stable: the result is the entries ordered by
// (row, column), entries with equal (row, column) -- duplicates, which this
// conversion keeps -- in their input order.
//
// Entries are dealt, values with them, to buckets of 2^s consecutive rows, s
// chosen so that a bucket fits a work-group's LDS, in two splits of at most
// 256 parts each (one where that is enough); a work-group then orders its
// bucket in LDS.  The input index rides in the key, so no step has to keep an
// order.  28.3M entries of a 1M-row power-law matrix: splits 230 us each (3.9
// TB/s), buckets 478 us (LDS reads), count and starts 60, the two scans of
// the indices 71 each; 1.20 ms in all against 2.60 with a radix sort of
// packed keys, which moves each key and index five times and then gathers the
// values, a cache line each.  (Dealt in one split, straight to 16384 buckets:
// 790 us, two entries a cache line.)
//
// Entries that do not suit it (few of them, a bucket over the LDS, more
// buckets than a work-group can count) take that stable LSD radix sort, the
// entry index as payload, which gives the same order.
#include <cstring>

#include <rocprim/device/device_radix_sort.hpp>

#include "shk_internal.hpp"

namespace shk {

// Packed keys, the entry index as payload, and the largest row / column
// (integer atomics: max is order-independent) and a flag for an index below
// zero after the shift.
__global__ __launch_bounds__(kBlock) void k_coo_scan(int64_t nnz, const int *row, const int *col, int index,
                                                     int *stats /* [0] max row, [1] max col, [2] bad */)
{
    int mr = -1, mc = -1, bad = 0;
    const int64_t step = (int64_t)gridDim.x * kBlock;
    for (int64_t i = blockIdx.x * (int64_t)kBlock + threadIdx.x; i < nnz; i += 4 * step) {
        int r[4], c[4];
#pragma unroll
        for (int u = 0; u < 4; u++) {  // past the end: the first entry again
            const int64_t e = i + u * step < nnz ? i + u * step : i;
            r[u] = row[e];
            c[u] = col[e];
        }
#pragma unroll
        for (int u = 0; u < 4; u++) {
            r[u] -= index;
            c[u] -= index;
            bad |= (r[u] < 0) | (c[u] < 0);
            mr = max(mr, r[u]);
            mc = max(mc, c[u]);
        }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        mr = max(mr, __shfl_xor(mr, off, kWave));
        mc = max(mc, __shfl_xor(mc, off, kWave));
        bad |= __shfl_xor(bad, off, kWave);
    }
    // a wavefront raises what is still below its own: two atomics each on the
    // same words took four times as long as the scan
    if ((threadIdx.x & (kWave - 1)) == 0) {
        if (__hip_atomic_load(&stats[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < mr) atomicMax(&stats[0], mr);
        if (__hip_atomic_load(&stats[1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < mc) atomicMax(&stats[1], mc);
        if (bad) atomicOr(&stats[2], 1);
    }
}

// ---- buckets -------------------------------------------------------------
constexpr int kCooThreads = 1024;
constexpr int kCooTile = 4096;        // entries of a splitting work-group
constexpr int kCooDigits = 256;       // parts of one split
constexpr int kCooGroups = 256;       // work-groups of the count
constexpr int kCooMaxBuckets = 36864; // counted in LDS (144 KiB)
constexpr int kCooMaxRowBits = 10;    // rows of a bucket
constexpr int kCooRunBits = 5, kCooRun = 1 << kCooRunBits;  // entries of a row ordered by counting
// fewer entries: the sort, which has no count to wait for (3000 entries 104 us
// against 120 in buckets, 30000 entries 153 against 124)
constexpr int kCooFew = 16384;
constexpr int kCooAhead = kCooTile / kCooThreads;  // entries in flight per thread

// How an entry's key is packed, from the top: its row within its part, its
// column, its place in the input.  Keys of one part are all different and
// order as the result does.
struct CooPack {
    int rowbits;  // of the row, within a bucket
    int split;    // of the bucket, within a first part
    int col, idx;
};

// entries of each bucket in this work-group's share of the input
__global__ __launch_bounds__(kCooThreads) void k_coo_count(int64_t nnz, int64_t chunk, const int *__restrict__ row,
                                                           int index, int s, int nb, int *__restrict__ table)
{
    extern __shared__ int coo_lds[];
    for (int b = threadIdx.x; b < nb; b += kCooThreads) coo_lds[b] = 0;
    __syncthreads();
    const int64_t i0 = blockIdx.x * chunk, i1 = min(nnz, i0 + chunk);
    for (int64_t i = i0 + threadIdx.x; i < i1; i += kCooAhead * kCooThreads) {
        int r[kCooAhead];
#pragma unroll
        for (int u = 0; u < kCooAhead; u++) {
            const int64_t e = i + u * kCooThreads;
            r[u] = e < i1 ? row[e] - index : -1;
        }
#pragma unroll
        for (int u = 0; u < kCooAhead; u++)
            if (r[u] >= 0) atomicAdd(&coo_lds[r[u] >> s], 1);
    }
    __syncthreads();
    for (int b = threadIdx.x; b < nb; b += kCooThreads) table[(size_t)blockIdx.x * nb + b] = coo_lds[b];
}

__global__ __launch_bounds__(kBlock) void k_coo_sizes(int groups, int nb, const int *__restrict__ table,
                                                      int *__restrict__ size)
{
    const int b = blockIdx.x * kBlock + threadIdx.x;
    if (b >= nb) return;
    int tot = 0;
#pragma unroll 16
    for (int g = 0; g < groups; g++) tot += table[(size_t)g * nb + b];
    size[b] = tot;
}

// Inclusive sums over the work-group's first kWave * kWave threads at most
// (every thread calls; part holds a word per wavefront).
static __device__ __forceinline__ int coo_sums(int v, int *part)
{
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
        const int w = __shfl_up(v, o, kWave);
        if (lane >= o) v += w;
    }
    __syncthreads();  // the last use of part
    if (lane == kWave - 1) part[wave] = v;
    __syncthreads();
    for (int w = 0; w < wave; w++) v += part[w];
    return v;
}

// One work-group: the buckets' starts from their sizes (base[nb]: all
// entries), the cursors of both splits, the first tile of each first part,
// and the largest bucket.
__global__ __launch_bounds__(kCooThreads) void k_coo_bases(int nb, int split, const int *__restrict__ size,
                                                           int *__restrict__ base, int *__restrict__ cursor,
                                                           int *__restrict__ first_cursor,
                                                           int *__restrict__ first_tile, int *__restrict__ most)
{
    extern __shared__ int coo_lds[];  // nb + 1
    __shared__ int part[kCooThreads / kWave], top;
    const int t = threadIdx.x, per = (nb + kCooThreads - 1) / kCooThreads;
    const int b0 = min(nb, t * per), b1 = min(nb, b0 + per);
    if (t == 0) top = 0;
    for (int b = t; b < nb; b += kCooThreads) coo_lds[b] = size[b];
    __syncthreads();
    int tot = 0, mx = 0;
    for (int b = b0; b < b1; b++) {
        tot += coo_lds[b];
        mx = max(mx, coo_lds[b]);
    }
    atomicMax(&top, mx);
    const int end = coo_sums(tot, part);
    int at = end - tot;
    for (int b = b0; b < b1; b++) {
        const int c = coo_lds[b];
        coo_lds[b] = at;
        at += c;
    }
    if (t == kCooThreads - 1) coo_lds[nb] = end;
    __syncthreads();
    for (int b = t; b <= nb; b += kCooThreads) base[b] = cursor[b] = coo_lds[b];
    const int parts = (nb + (1 << split) - 1) >> split;
    int tiles = 0;
    if (t < parts) {
        const int p0 = coo_lds[t << split], p1 = coo_lds[min(nb, (t + 1) << split)];
        first_cursor[t] = p0;
        tiles = (p1 - p0 + kCooTile - 1) / kCooTile;
    }
    const int tile = coo_sums(tiles, part);
    if (t < parts) first_tile[t + 1] = tile;
    if (t == 0) {
        first_tile[0] = 0;
        *most = top;
    }
}

// One tile dealt to at most kCooDigits parts: brought together by part in LDS,
// so that what goes to one part is written as a run.  A tile takes its room
// in a part from the part's cursor: the order within a part is whatever it
// turns out to be, the keys hold what the result needs.  First: from the
// input to first parts (split of rows by their top bits); else a first part's
// tile to its buckets.
template <typename T, bool First>
__global__ __launch_bounds__(kCooThreads) void k_coo_split(int64_t nnz, const int *__restrict__ row,
                                                           const int *__restrict__ col, int index, CooPack pk,
                                                           int parts, const int *__restrict__ base, int nb,
                                                           const int *__restrict__ first_tile,
                                                           int *__restrict__ cursor,
                                                           const uint64_t *__restrict__ key_in,
                                                           const T *__restrict__ val_in,
                                                           uint64_t *__restrict__ key_out, T *__restrict__ val_out)
{
    __shared__ uint64_t keys[kCooTile];
    __shared__ T vals[kCooTile];
    __shared__ unsigned char digit[kCooTile];
    __shared__ int count[kCooDigits], start[kCooDigits], off[kCooDigits], part[kCooThreads / kWave], which;
    const int t = threadIdx.x, low = pk.col + pk.idx;
    if (t < kCooDigits) count[t] = 0;
    int64_t i0 = (int64_t)blockIdx.x * kCooTile;
    int n;
    if constexpr (First) {
        n = (int)min((int64_t)kCooTile, nnz - i0);
    } else {
        if ((int)blockIdx.x >= first_tile[parts]) return;
        if (t < parts && first_tile[t] <= (int)blockIdx.x && (int)blockIdx.x < first_tile[t + 1]) which = t;
        __syncthreads();
        const int p = which, p1 = base[min(nb, (p + 1) << pk.split)];
        i0 = base[p << pk.split] + (int64_t)((int)blockIdx.x - first_tile[p]) * kCooTile;
        n = (int)min((int64_t)kCooTile, p1 - i0);
        cursor += p << pk.split;
    }
    uint64_t k[kCooAhead];
    T v[kCooAhead];
    int d[kCooAhead], place[kCooAhead];
    if constexpr (First) {
        int r[kCooAhead], c[kCooAhead];
#pragma unroll
        for (int u = 0; u < kCooAhead; u++) {
            const int j = u * kCooThreads + t;
            r[u] = j < n ? row[i0 + j] - index : 0;
            c[u] = j < n ? col[i0 + j] - index : 0;
            v[u] = j < n ? val_in[i0 + j] : (T)0;
        }
#pragma unroll
        for (int u = 0; u < kCooAhead; u++) {
            const int bits = pk.rowbits + pk.split;
            d[u] = r[u] >> bits;
            k[u] = ((((uint64_t)(r[u] & ((1 << bits) - 1)) << pk.col) | (unsigned)c[u]) << pk.idx) |
                   (uint64_t)(i0 + u * kCooThreads + t);
        }
    } else {
#pragma unroll
        for (int u = 0; u < kCooAhead; u++) {
            const int j = u * kCooThreads + t;
            k[u] = j < n ? key_in[i0 + j] : 0;
            v[u] = j < n ? val_in[i0 + j] : (T)0;
        }
#pragma unroll
        for (int u = 0; u < kCooAhead; u++) {
            d[u] = (int)(k[u] >> (low + pk.rowbits));
            k[u] &= (1ull << (low + pk.rowbits)) - 1ull;
        }
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kCooAhead; u++)
        if (u * kCooThreads + t < n) place[u] = atomicAdd(&count[d[u]], 1);
    __syncthreads();
    const int c = t < kCooDigits ? count[t] : 0;
    const int to = c > 0 ? atomicAdd(&cursor[t], c) : 0;
    const int st = coo_sums(c, part) - c;
    if (t < kCooDigits) {
        start[t] = st;
        off[t] = to - st;
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kCooAhead; u++)
        if (u * kCooThreads + t < n) {
            const int q = start[d[u]] + place[u];
            keys[q] = k[u];
            vals[q] = v[u];
            digit[q] = (unsigned char)d[u];
        }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kCooAhead; u++) {
        const int j = u * kCooThreads + t;
        if (j < n) {
            const size_t o = (size_t)(off[digit[j]] + j);
            key_out[o] = keys[j];
            val_out[o] = vals[j];
        }
    }
}

// One bucket: entries grouped by row in LDS, then each row ordered there, in
// runs of 32 by counting the run's smaller keys (lanes of one run read the
// same words), then by merging runs two by two: an entry looks itself up in
// the run beside its own.  A row of L entries costs 32 + sum(log2) LDS reads
// an entry; counting the whole row, L reads, took 772 us where this takes 478
// (28.3M entries, rows of 4 to 512).
template <typename T, int CAP>
__global__ __launch_bounds__(kCooThreads) void k_coo_bucket(int m, CooPack pk, const int *__restrict__ base,
                                                            const uint64_t *__restrict__ key_in,
                                                            const T *__restrict__ val_in, int *__restrict__ ptr,
                                                            int *__restrict__ ind, T *__restrict__ val_out)
{
    extern __shared__ uint64_t coo_keys[];  // [CAP], then CAP values
    __shared__ int start[(1 << kCooMaxRowBits) + 1], fill[1 << kCooMaxRowBits], part[kCooThreads / kWave], longest;
    T *vals = (T *)(coo_keys + CAP);
    constexpr int K = CAP / kCooThreads;
    const int t = threadIdx.x, b = blockIdx.x, rows = 1 << pk.rowbits, low = pk.col + pk.idx;
    const int at = base[b], cnt = base[b + 1] - at;
    if (t < rows) fill[t] = 0;
    if (t == 0) longest = 0;
    uint64_t e[K];
    T v[K];
    int place[K];
#pragma unroll
    for (int k = 0; k < K; k++)
        if (k * kCooThreads + t < cnt) {
            e[k] = key_in[(size_t)at + k * kCooThreads + t];
            v[k] = val_in[(size_t)at + k * kCooThreads + t];
        }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < K; k++)
        if (k * kCooThreads + t < cnt) place[k] = atomicAdd(&fill[e[k] >> low], 1);
    __syncthreads();
    const int mine = t < rows ? fill[t] : 0;
    const int st = coo_sums(mine, part) - mine;
    if (mine > kCooRun) atomicMax(&longest, mine);
    if (t < rows) {
        start[t] = st;
        const int r = (b << pk.rowbits) + t;
        if (r < m) ptr[r] = at + st;
    }
    if (t == 0) {
        start[rows] = cnt;
        if (b == (int)gridDim.x - 1) ptr[m] = at + cnt;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < K; k++)
        if (k * kCooThreads + t < cnt) {
            const int q = start[e[k] >> low] + place[k];
            coo_keys[q] = e[k];
            vals[q] = v[k];
        }
    __syncthreads();
    // the entries again, lanes beside each other in one row
    int pos[K], q0[K], q1[K];
#pragma unroll
    for (int k = 0; k < K; k++) {
        const int q = k * kCooThreads + t;
        if (q >= cnt) continue;
        e[k] = coo_keys[q];
        v[k] = vals[q];
        const int r = (int)(e[k] >> low);
        q0[k] = start[r];
        q1[k] = start[r + 1];
        const int r0 = q - ((q - q0[k]) & (kCooRun - 1)), r1 = min(r0 + kCooRun, q1[k]);
        pos[k] = r0;
#pragma unroll 4
        for (int j = r0; j < r1; j++) pos[k] += coo_keys[j] < e[k];
    }
    const int top = longest;  // 0: no row of more than one run
    for (int w = kCooRun, lg = kCooRunBits; w < top; w <<= 1, lg++) {
        __syncthreads();
#pragma unroll
        for (int k = 0; k < K; k++)
            if (k * kCooThreads + t < cnt) coo_keys[pos[k]] = e[k];
        __syncthreads();
#pragma unroll
        for (int k = 0; k < K; k++) {
            if (k * kCooThreads + t >= cnt || q1[k] - q0[k] <= w) continue;
            const int run = (pos[k] - q0[k]) >> lg;
            const int other = q0[k] + (run ^ 1) * w;
            int n = min(w, q1[k] - other), lo = 0;  // n <= 0: no run beside it
            while (n > 0) {
                const int half = n >> 1;
                if (coo_keys[other + lo + half] < e[k]) {
                    lo += half + 1;
                    n -= half + 1;
                } else n = half;
            }
            pos[k] += lo - (run & 1) * w;
        }
    }
    const unsigned cmask = (1u << pk.col) - 1u;  // at most 31 bits
#pragma unroll
    for (int k = 0; k < K; k++)
        if (k * kCooThreads + t < cnt) {
            ind[(size_t)at + pos[k]] = (int)((unsigned)(e[k] >> pk.idx) & cmask);
            val_out[(size_t)at + pos[k]] = v[k];
        }
}

__global__ __launch_bounds__(kBlock) void k_coo_keys(int64_t nnz, const int *row, const int *col, int index,
                                                     int colbits, uint64_t *key, uint32_t *idx)
{
    for (int64_t i = blockIdx.x * (int64_t)kBlock + threadIdx.x; i < nnz; i += (int64_t)gridDim.x * kBlock) {
        key[i] = ((uint64_t)(uint32_t)(row[i] - index) << colbits) | (uint32_t)(col[i] - index);
        idx[i] = (uint32_t)i;
    }
}

// Sorted entries -> column indices, values (gathered by entry index) and the
// row pointer: the first entry of each run of equal rows writes the pointers
// of its row and of the empty rows before it; the last entry closes the rest.
template <typename T>
__global__ __launch_bounds__(kBlock) void k_coo_fill(int64_t nnz, int m, int colbits, const uint64_t *key,
                                                     const uint32_t *idx, const T *val, int *ptr, int *ind,
                                                     T *val_out)
{
    const uint64_t cmask = (colbits >= 64) ? ~0ull : ((1ull << colbits) - 1);
    for (int64_t i = blockIdx.x * (int64_t)kBlock + threadIdx.x; i < nnz; i += (int64_t)gridDim.x * kBlock) {
        const uint64_t k = key[i];
        const int r = (int)(k >> colbits);
        ind[i] = (int)(k & cmask);
        val_out[i] = val[idx[i]];
        const int rprev = i == 0 ? -1 : (int)(key[i - 1] >> colbits);
        for (int q = rprev + 1; q <= r; q++) ptr[q] = (int)i;
        if (i == nnz - 1)
            for (int q = r + 1; q <= m; q++) ptr[q] = (int)nnz;
    }
}

__global__ __launch_bounds__(kBlock) void k_fill_int(int64_t n, int v, int *x)
{
    for (int64_t i = blockIdx.x * (int64_t)kBlock + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBlock) x[i] = v;
}

static int bits_for(int v)
{
    int b = 0;
    while (b < 31 && (1 << b) <= v) b++;
    return b;
}

// The bucket path; *done = false when the entries do not suit it (nothing has
// been written then).  A bucket may be about half full on average, so that
// uneven ones still fit; the smaller LDS size, two work-groups per CU, where
// its buckets can be counted.  The scratch it needs is no more than the
// sort's (val_out holds the values between the two splits); without it the
// sort below reports what is missing.
template <typename T>
static int coo_buckets(shk_ctx ctx, int64_t nnz, const int *row, const int *col, const T *val, int index, int m,
                       int colbits, int *ptr, int *ind, T *val_out, bool *done)
{
    *done = false;
    if (nnz <= kCooFew || nnz >= INT32_MAX) return SHK_OK;
    const double per_row = std::max((double)nnz / m, 1e-3);
    CooPack pk;
    pk.col = colbits;
    pk.idx = bits_for((int)nnz - 1);
    int nb = 0;
    for (int cap : {4096, 8192}) {
        pk.rowbits = kCooMaxRowBits;
        while (pk.rowbits > 0 && per_row * (1 << pk.rowbits) > 0.55 * cap) pk.rowbits--;
        nb = (int)(((int64_t)m + (1 << pk.rowbits) - 1) >> pk.rowbits);
        if (nb <= kCooMaxBuckets) break;
    }
    if (nb > kCooMaxBuckets) return SHK_OK;
    // two splits of about as many parts each, or one
    const bool twice = nb > kCooDigits;
    pk.split = twice ? (bits_for(nb - 1) + 1) / 2 : 0;
    if (pk.rowbits + pk.split + pk.col + pk.idx > 64) return SHK_OK;
    const int parts = (nb + (1 << pk.split) - 1) >> pk.split;
    hipStream_t st = ctx->stream;
    const int64_t chunk =
        std::max<int64_t>(kCooTile, ((nnz + kCooGroups - 1) / kCooGroups + kCooTile - 1) / kCooTile * kCooTile);
    const int groups = (int)((nnz + chunk - 1) / chunk), tiles = (int)((nnz + kCooTile - 1) / kCooTile);
    auto al = [](size_t v) { return (v + 255) & ~(size_t)255; };
    const size_t kb = al(sizeof(uint64_t) * (size_t)nnz), vb = al(sizeof(T) * (size_t)nnz),
                 bb = al(sizeof(int) * ((size_t)nb + 1)), pb = al(sizeof(int) * (kCooDigits + 1));
    // the count's table is read before the keys are written over it
    const size_t table_bytes = sizeof(int) * (size_t)groups * nb;
    const size_t big = std::max(kb * (twice ? 2 : 1) + vb, al(table_bytes));
    if (!spare_ws2(ctx, big + 3 * bb + 3 * pb)) return SHK_OK;
    char *w = (char *)ctx->ws2;
    uint64_t *key = (uint64_t *)w, *key0 = (uint64_t *)(w + kb + vb);
    T *v = (T *)(w + kb);
    int *table = (int *)w;
    w += big;
    int *size = (int *)w, *base = (int *)(w + bb), *cursor = (int *)(w + 2 * bb);
    w += 3 * bb;
    int *first_cursor = (int *)w, *first_tile = (int *)(w + pb), *most = (int *)(w + 2 * pb);
    const size_t lds = sizeof(int) * ((size_t)nb + 1);
    hipLaunchKernelGGL(k_coo_count, dim3(groups), dim3(kCooThreads), lds, st, nnz, chunk, row, index, pk.rowbits,
                       nb, table);
    hipLaunchKernelGGL(k_coo_sizes, dim3((nb + kBlock - 1) / kBlock), dim3(kBlock), 0, st, groups, nb,
                       (const int *)table, size);
    hipLaunchKernelGGL(k_coo_bases, dim3(1), dim3(kCooThreads), lds, st, nb, pk.split, (const int *)size, base,
                       cursor, first_cursor, first_tile, most);
    SHK_HIP(hipGetLastError());
    int h = 0;
    SHK_HIP(hipMemcpyAsync(&h, most, sizeof(int), hipMemcpyDeviceToHost, st));
    SHK_HIP(hipStreamSynchronize(st));
    if (h > 8192) return SHK_OK;
    hipLaunchKernelGGL((k_coo_split<T, true>), dim3(tiles), dim3(kCooThreads), 0, st, nnz, row, col, index, pk,
                       parts, (const int *)base, nb, (const int *)first_tile, first_cursor,
                       (const uint64_t *)nullptr, val, twice ? key0 : key, twice ? val_out : v);
    if (twice)  // every first part ends in a tile of its own
        hipLaunchKernelGGL((k_coo_split<T, false>), dim3(tiles + parts), dim3(kCooThreads), 0, st, nnz,
                           (const int *)nullptr, (const int *)nullptr, 0, pk, parts, (const int *)base, nb,
                           (const int *)first_tile, cursor, (const uint64_t *)key0, (const T *)val_out, key, v);
    const int cap = h <= 4096 ? 4096 : 8192;
    const size_t blds = (sizeof(uint64_t) + sizeof(T)) * (size_t)cap;
    if (cap == 4096)
        hipLaunchKernelGGL((k_coo_bucket<T, 4096>), dim3(nb), dim3(kCooThreads), blds, st, m, pk,
                           (const int *)base, (const uint64_t *)key, (const T *)v, ptr, ind, val_out);
    else
        hipLaunchKernelGGL((k_coo_bucket<T, 8192>), dim3(nb), dim3(kCooThreads), blds, st, m, pk,
                           (const int *)base, (const uint64_t *)key, (const T *)v, ptr, ind, val_out);
    SHK_HIP(hipGetLastError());
    ctx->count[SHK_COUNT_COO_BUCKETS]++;
    *done = true;
    return SHK_OK;
}

template <typename T>
static int coo_to_csr_typed(shk_ctx ctx, int64_t nnz, const int *row, const int *col, const T *val, int index,
                            int m_min, int n_min, int m_cap, int *m_out, int *n_out, int *ptr, int *ind,
                            T *val_out)
{
    hipStream_t st = ctx->stream;
    int *stats = (int *)ctx->scalars;  // 3 ints
    const int init[3] = {-1, -1, 0};
    SHK_HIP(hipMemcpyAsync(stats, init, sizeof(init), hipMemcpyHostToDevice, st));
    const int nb = red_blocks(nnz);
    if (nnz > 0) hipLaunchKernelGGL(k_coo_scan, dim3(nb), dim3(kBlock), 0, st, nnz, row, col, index, stats);
    int h[3];
    SHK_HIP(hipMemcpyAsync(h, stats, sizeof(h), hipMemcpyDeviceToHost, st));
    SHK_HIP(hipStreamSynchronize(st));
    SHK_CHECK(h[2] == 0, SHK_ERR_ARG, "coo_to_csr: an index is below the base index");
    // m = max(row) + 1 and at least the matrix's previous size; with no
    // entries Seldon's GetNormInf gives 0, so m >= 1 (Matrix_Conversions.cxx:
    // 1310-1316)
    const int m = std::max(std::max(h[0], 0) + 1, m_min);
    const int n = std::max(std::max(h[1], 0) + 1, n_min);
    *m_out = m;
    *n_out = n;
    if (!ptr) return SHK_OK;  // dimensions only
    SHK_CHECK(m <= m_cap, SHK_ERR_DIM, "coo_to_csr: the row pointer holds fewer than m + 1 entries");
    if (nnz == 0) {
        hipLaunchKernelGGL(k_fill_int, dim3(red_blocks(m + 1)), dim3(kBlock), 0, st, (int64_t)m + 1, 0, ptr);
        SHK_HIP(hipGetLastError());
        return SHK_OK;
    }
    SHK_CHECK(nnz < ((int64_t)1 << 32), SHK_ERR_ARG, "coo_to_csr: more than 2^32 - 1 entries");
    const int colbits = bits_for(n - 1), rowbits = std::max(bits_for(m - 1), colbits == 0 ? 1 : 0);
    bool done = false;
    SHK_TRY(coo_buckets<T>(ctx, nnz, row, col, val, index, m, colbits, ptr, ind, val_out, &done));
    if (done) return SHK_OK;
    // workspace: keys and indices, in and out, then rocPRIM's temporary
    const size_t kb = ((size_t)nnz * 8 + 255) & ~(size_t)255, ib = ((size_t)nnz * 4 + 255) & ~(size_t)255;
    size_t tmp_bytes = 0;
    SHK_HIP(rocprim::radix_sort_pairs(nullptr, tmp_bytes, (const uint64_t *)nullptr, (uint64_t *)nullptr,
                                      (const uint32_t *)nullptr, (uint32_t *)nullptr, (size_t)nnz, 0,
                                      colbits + rowbits, st));
    SHK_TRY(ensure_ws2(ctx, 2 * kb + 2 * ib + tmp_bytes + 256));
    char *w = (char *)ctx->ws2;
    uint64_t *k0 = (uint64_t *)w, *k1 = (uint64_t *)(w + kb);
    uint32_t *i0 = (uint32_t *)(w + 2 * kb), *i1 = (uint32_t *)(w + 2 * kb + ib);
    void *tmp = w + 2 * kb + 2 * ib;
    hipLaunchKernelGGL(k_coo_keys, dim3(nb), dim3(kBlock), 0, st, nnz, row, col, index, colbits, k0, i0);
    SHK_HIP(rocprim::radix_sort_pairs(tmp, tmp_bytes, (const uint64_t *)k0, k1, (const uint32_t *)i0, i1,
                                      (size_t)nnz, 0, colbits + rowbits, st));
    hipLaunchKernelGGL(k_coo_fill<T>, dim3(nb), dim3(kBlock), 0, st, nnz, m, colbits, (const uint64_t *)k1,
                       (const uint32_t *)i1, val, ptr, ind, val_out);
    SHK_HIP(hipGetLastError());
    return SHK_OK;
}

}  // namespace shk

using namespace shk;

extern "C" {

int shk_coo_to_csr(shk_ctx ctx, shk_dtype dt, int64_t nnz, const int *drow, const int *dcol, const void *dval,
                   int index, int m_min, int n_min, int m_cap, int *m, int *n, int *dptr, int *dind,
                   void *dval_out)
{
    SHK_CHECK(ctx && m && n, SHK_ERR_ARG, "coo_to_csr: null argument");
    SHK_CHECK(nnz >= 0, SHK_ERR_ARG, "coo_to_csr: negative entry count");
    SHK_CHECK(dt == SHK_F64 || dt == SHK_F32, SHK_ERR_ARG, "coo_to_csr: bad dtype");
    if (nnz > 0) {
        SHK_TRY(check_device_ptr(drow, "row"));
        SHK_TRY(check_device_ptr(dcol, "col"));
        SHK_TRY(check_device_ptr(dval, "val"));
        if (dptr) {
            SHK_TRY(check_device_ptr(dind, "ind out"));
            SHK_TRY(check_device_ptr(dval_out, "val out"));
        }
    }
    if (dt == SHK_F64)
        return coo_to_csr_typed<double>(ctx, nnz, drow, dcol, (const double *)dval, index, m_min, n_min, m_cap, m,
                                        n, dptr, dind, (double *)dval_out);
    return coo_to_csr_typed<float>(ctx, nnz, drow, dcol, (const float *)dval, index, m_min, n_min, m_cap, m, n,
                                   dptr, dind, (float *)dval_out);
}

}  // extern "C"
