// shk_dia.hpp -- the diagonal-slice copy of a matrix and its SpMV kernel.
//
// Stencil and banded matrices in natural order repeat a few column offsets
// (col - row) row after row.  Rows are taken in slices of 64, one row per
// lane, and a slice's entries are stored by offset: step k of a slice holds,
// for one offset, the values of the rows that have an entry there, at 64
// consecutive positions, with one 64-bit mask of those rows.  An entry then
// costs its value alone (V bytes, plus 16 bytes per 64-row step) where the
// other layouts read a 2- or 4-byte column with it, and a step's x reads are
// 64 consecutive elements whose address needs no load, so they are issued
// together with the values instead of after them.
//
// Within a row the steps are in increasing offset, so in increasing column:
// the order the row is stored in (the build refuses rows whose columns are
// not strictly increasing).  Lanes outside a step's mask keep their sum
// untouched, so row sums are Seldon's `temp += data[j] * X(ind[j])`
// (Functions_MatVect.cxx:424-430) term for term.  RowSymSparse rows hold the
// steps of their stored upper part first, then the "direct" steps of the
// transposed part (Functions_MatVect.cxx:553-563).
//
// Every slice of a matrix has the same number of steps (dia_steps, the
// largest any slice needs), so positions need no table.  The build is on the
// device, from the row arrays, and gives up where the steps would cost more
// than kDiaFill times the entries: irregular matrices keep the other layouts.
#pragma once

namespace shk {

constexpr int kDiaMaxSteps = 32;
// slots (64 per step and slice) per stored entry, at most: past 1.25 the
// padding costs what the saved columns gain (12 against 8 bytes FP64, less
// the other layouts' own overheads)
constexpr double kDiaFill = 1.25;
constexpr int64_t kDiaSlack = 4096;  // slots a small matrix may add to that
constexpr int kDiaWaves = kBlock / kWave;  // slices per work-group of the build

struct alignas(16) DiaStep {
    uint64_t mask;  // rows (lanes) of the slice with an entry at this offset
    int off;        // col - row
    int direct;     // RowSymSparse: a transposed-part step
};

// raise *p to v; almost every wavefront finds it there already, and the read
// spares an atomic on one address (100K of them were 0.5 ms)
__device__ __forceinline__ void dia_max(int *p, int v)
{
    if (__hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < v) atomicMax(p, v);
}

struct DiaView {
    int steps;              // per slice
    int groups;             // work-group steps: a slice per wavefront each
    int q;                  // groups per XCD
    const DiaStep *step;    // [slices * steps]
};

// One slice's rows: the steps' values and x reads are all issued before the
// first is used (KS steps at a time; KS = 0: any number, eight at a time).
template <typename T, int MODE, int KS>
__device__ __forceinline__ T dia_row(const SpmvArgs<T> &a, const DiaView &v, int slice, int row, int lane, T y0)
{
    constexpr int U = KS ? KS : 8;
    const int steps = KS ? KS : v.steps;
    const DiaStep *sp = v.step + (size_t)slice * steps;
    const T *vp = a.val + (size_t)slice * steps * kWave + lane;
    const uint64_t bit = 1ull << lane;
    T acc = MODE == kArray ? y0 : (T)0;
    bool direct = false;  // RowSymSparse: y formed, transposed part started
    for (int k0 = 0; k0 < steps; k0 += U) {
        T vv[U], xv[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int k = KS ? u : min(k0 + u, steps - 1);
            const DiaStep s = sp[k];
            vv[u] = vp[(size_t)k * kWave];
            xv[u] = a.x[(s.mask & bit) ? row + s.off : 0];
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int k = k0 + u;
            if (!KS && k >= steps) break;
            const DiaStep s = sp[k];
            if (MODE == kSym && s.direct && !direct) {
                acc = y0 + a.alpha * acc;
                direct = true;
            }
            const T val = vv[u];
            const T pr = (MODE == kArray || (MODE == kSym && direct)) ? (a.alpha * val) * xv[u] : val * xv[u];
            const T sum = acc + pr;
            acc = (s.mask & bit) ? sum : acc;
        }
    }
    if (MODE == kArray || (MODE == kSym && direct)) return acc;
    return y0 + a.alpha * acc;
}

// Work-groups of one XCD take consecutive groups of that XCD's contiguous
// range together, so the x lines neighbouring slices share stay in its L2.
// Work-groups of 256 threads up to 4096 slices, so small matrices reach every
// CU, of 1024 above, at most two per CU: each leaves one partial per fused
// dot, and every work-group of the next kernel sums them all (2048 partials
// instead of 512 made the vector kernels of a 2M-row BiCgStab iteration 22 to
// 33% slower).
template <typename T, int MODE, int KS>
__global__ __launch_bounds__(1024, 8) void k_dia(SpmvArgs<T> a, DiaView v)
{
    if (a.skip && *a.skip) return;
    const int lane = threadIdx.x & (kWave - 1);
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int xcd = blockIdx.x % kNumXcd, stride = gridDim.x / kNumXcd;
    const int end = min(v.groups, (xcd + 1) * v.q);
    T c[2] = {(T)0, (T)0};
    for (int g = xcd * v.q + (int)(blockIdx.x / kNumXcd); g < end; g += stride) {
        const int slice = g * (int)(blockDim.x / kWave) + w;
        const int row = slice * kWave + lane;
        if (slice * kWave >= a.m) break;  // wave-uniform: the last group's empty slices
        const bool in = row < a.m;
        const T y0 = panel_y0<T, MODE>(a, in ? row : -1);
        const T y = dia_row<T, MODE, KS>(a, v, slice, row, lane, y0);
        if (in) spmv_epilogue<T, MODE>(a, row, y, c);
    }
    if (a.dot0 != kDotNone || a.dot1 != kDotNone) block_partial<T, 2>(c, a.partials, gridDim.x, blockIdx.x);
}

// Launch on the matrix's diagonal-slice copy (a.m, pointers and partials set
// by the caller); returns the grid.
template <typename T>
int launch_dia(shk_csr A, SpmvArgs<T> &a);

}  // namespace shk
