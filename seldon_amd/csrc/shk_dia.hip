// shk_dia.hip -- the diagonal-slice copy: its build on the device, value
// updates and the SpMV launch.  Layout and kernel: shk_dia.hpp.
#include <algorithm>
#include <vector>

#include "shk_kernels.hpp"

namespace shk {

namespace {

// The steps of one slice, by one wavefront: each lane walks its row's entries
// and every step takes the smallest offset any lane is at.  The stored part
// [ptr, mid) comes first, then the transposed part [mid, ptr end) (mid null:
// one part).  fill = false fills flag[] = {most steps of a slice; a row's
// columns do not increase or there are more than kDiaMaxSteps; largest row -
// col; largest col - row}; fill = true writes the steps and, per slot, the entry's position (src; -1 where the row has
// none).
__global__ __launch_bounds__(kBlock) void k_dia_build(int m, const int *ptr, const int *mid, const uint32_t *ind,
                                                      int steps, DiaStep *step, int *src, int *flag, bool fill)
{
    const int slice = blockIdx.x * kDiaWaves + (int)(threadIdx.x >> 6);
    const int lane = threadIdx.x & (kWave - 1);
    if (slice * kWave >= m) return;
    const int row = slice * kWave + lane;
    const bool in = row < m;
    int j = in ? ptr[row] : 0;
    const int end = in ? ptr[row + 1] : 0;
    const int split = in && mid ? mid[row] : end;
    const size_t s0 = (size_t)slice * steps;
    int k = 0, left = 0, right = 0;
    bool ok = true;
    for (int part = 0; part < (mid ? 2 : 1); part++) {
        const int e = part == 0 ? split : end;
        int last = -1;
        for (;;) {
            const int col = j < e ? (int)(ind[j] & ~kLowerFlag) : 0;
            if (j < e && col <= last) ok = false;
            const int off = j < e ? col - row : INT32_MAX;
            int lo = off;
            for (int o = 32; o > 0; o >>= 1) lo = min(lo, __shfl_xor(lo, o, kWave));
            if (lo == INT32_MAX || k == kDiaMaxSteps || (fill && k == steps)) {
                if (lo != INT32_MAX) ok = false;
                break;
            }
            left = max(left, -lo);
            right = max(right, lo);
            const bool act = j < e && off == lo;
            const uint64_t mask = __builtin_amdgcn_ballot_w64(act);
            if (fill) {
                if (lane == 0) step[s0 + k] = DiaStep{mask, lo, part};
                src[(s0 + k) * kWave + lane] = act ? j : -1;
            }
            if (act) {
                last = col;
                j++;
            }
            k++;
        }
    }
    if (!fill) {
        if (!ok) atomicOr(flag + 1, 1);
        if (lane == 0) {
            dia_max(flag, k);
            dia_max(flag + 2, left);
            dia_max(flag + 3, right);
        }
    } else {
        for (; k < steps; k++) {
            if (lane == 0) step[s0 + k] = DiaStep{0ull, 0, mid ? 1 : 0};
            src[(s0 + k) * kWave + lane] = -1;
        }
    }
}

// positions in the device row arrays -> positions in the caller's (src_of:
// RowSymSparse, whose rows are expanded)
__global__ __launch_bounds__(kBlock) void k_dia_map(int64_t n, const int64_t *src_of, int *src)
{
    for (int64_t i = blockIdx.x * (int64_t)kBlock + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBlock)
        if (src[i] >= 0) src[i] = (int)src_of[src[i]];
}

template <typename T>
__global__ __launch_bounds__(kBlock) void k_dia_vals(int64_t n, const int *__restrict__ src, const T *__restrict__ from,
                                                     T *__restrict__ to)
{
    for (int64_t i = blockIdx.x * (int64_t)kBlock + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBlock) {
        const int q = src[i];
        to[i] = q >= 0 ? from[q] : (T)0;
    }
}

inline int64_t dia_slots(shk_csr A) { return (int64_t)((A->m + kWave - 1) / kWave) * A->dia_steps * kWave; }

}  // namespace

int dia_build(shk_csr A, const int *ptr, const int *mid, const uint32_t *ind, const int64_t *src_of, bool *applies)
{
    *applies = false;
    if (A->m == 0 || A->nnz_dev == 0) return SHK_OK;
    hipStream_t s = A->ctx->stream;
    const int slices = (A->m + kWave - 1) / kWave;
    const dim3 grid((slices + kDiaWaves - 1) / kDiaWaves), blk(kBlock);
    int *flag = nullptr, h[4] = {0, 0, 0, 0};
    hipError_t e = spare_malloc(A->ctx, (void **)&flag, sizeof(h));
    if (e == hipErrorOutOfMemory) return SHK_OK;
    SHK_HIP(e);
    e = hipMemcpyAsync(flag, h, sizeof(h), hipMemcpyHostToDevice, s);
    if (e == hipSuccess) {
        hipLaunchKernelGGL(k_dia_build, grid, blk, 0, s, A->m, ptr, mid, ind, 0, (DiaStep *)nullptr, (int *)nullptr,
                           flag, false);
        e = hipMemcpyAsync(h, flag, sizeof(h), hipMemcpyDeviceToHost, s);
    }
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    hipFree(flag);
    SHK_HIP(e);
    const int64_t slots = (int64_t)slices * h[0] * kWave;
    if (h[1] || h[0] == 0 || slots > (int64_t)(kDiaFill * (double)A->nnz_dev) + kDiaSlack) return SHK_OK;
    A->dia_steps = h[0];
    A->dia_left = h[2];
    A->dia_right = h[3];
    A->dia_block = slices <= 4096 ? kBlock : 1024;
    A->dia_groups = (int)(((int64_t)slices * kWave + A->dia_block - 1) / A->dia_block);
    e = spare_malloc(A->ctx, &A->dia_step, sizeof(DiaStep) * (size_t)slices * h[0]);
    if (e == hipSuccess) e = spare_malloc(A->ctx, (void **)&A->dia_src, sizeof(int) * (size_t)slots);
    if (e == hipSuccess) e = spare_malloc(A->ctx, &A->dia_val, dsize(A->dtype) * (size_t)slots);
    if (e == hipErrorOutOfMemory) {  // the layout already there serves
        dia_free(A);
        return SHK_OK;
    }
    SHK_HIP(e);
    hipLaunchKernelGGL(k_dia_build, grid, blk, 0, s, A->m, ptr, mid, ind, h[0], (DiaStep *)A->dia_step, A->dia_src,
                       (int *)nullptr, true);
    if (src_of)
        hipLaunchKernelGGL(k_dia_map, dim3(red_blocks(slots)), blk, 0, s, slots, src_of, A->dia_src);
    SHK_HIP(hipGetLastError());
    *applies = true;
    return SHK_OK;
}

int dia_set_values(shk_csr A, const void *dval)
{
    if (!A->dia_val) return SHK_OK;
    const int64_t n = dia_slots(A);
    if (A->dtype == SHK_F64)
        hipLaunchKernelGGL(k_dia_vals<double>, dim3(red_blocks(n)), dim3(kBlock), 0, A->ctx->stream, n,
                           (const int *)A->dia_src, (const double *)dval, (double *)A->dia_val);
    else
        hipLaunchKernelGGL(k_dia_vals<float>, dim3(red_blocks(n)), dim3(kBlock), 0, A->ctx->stream, n,
                           (const int *)A->dia_src, (const float *)dval, (float *)A->dia_val);
    SHK_HIP(hipGetLastError());
    return SHK_OK;
}

void dia_free(shk_csr A)
{
    hipFree(A->dia_step);
    hipFree(A->dia_src);
    hipFree(A->dia_val);
    A->dia_step = A->dia_val = nullptr;
    A->dia_src = nullptr;
    A->dia_steps = A->dia_groups = 0;
}

// Work-groups of a product with fused dots: persistent, two 1024-thread ones
// per CU at most (see k_dia).
int dia_grid(shk_csr A)
{
    const int q = (A->dia_groups + kNumXcd - 1) / kNumXcd;
    return kNumXcd * std::min(q, std::max(1, A->ctx->num_cus * (2048 / A->dia_block) / kNumXcd));
}

template <typename T, int MODE>
static void launch_dia_mode(shk_csr A, const SpmvArgs<T> &a, const DiaView &v, dim3 grid, dim3 blk)
{
    hipStream_t s = A->ctx->stream;
    switch (v.steps) {
#define SHK_DIA_CASE(k) \
    case k: hipLaunchKernelGGL((k_dia<T, MODE, k>), grid, blk, 0, s, a, v); break;
        SHK_DIA_CASE(1)
        SHK_DIA_CASE(2)
        SHK_DIA_CASE(3)
        SHK_DIA_CASE(4)
        SHK_DIA_CASE(5)
        SHK_DIA_CASE(6)
        SHK_DIA_CASE(7)
        SHK_DIA_CASE(8)
        SHK_DIA_CASE(9)
#undef SHK_DIA_CASE
    default: hipLaunchKernelGGL((k_dia<T, MODE, 0>), grid, blk, 0, s, a, v); break;
    }
}

template <typename T>
int launch_dia(shk_csr A, SpmvArgs<T> &a)
{
    const bool dots = a.dot0 != kDotNone || a.dot1 != kDotNone;
    // without dots nothing counts the work-groups: small ones, each a single
    // step, dealt out as CUs come free
    const int block = dots ? A->dia_block : kBlock;
    const int groups = dots ? A->dia_groups : (int)(((int64_t)A->m + kBlock - 1) / kBlock);
    const int q = (groups + kNumXcd - 1) / kNumXcd;
    const DiaView v{A->dia_steps, groups, q, (const DiaStep *)A->dia_step};
    const dim3 grid(dots ? dia_grid(A) : kNumXcd * q), blk(block);
    a.val = (const T *)A->dia_val;
    if (A->storage == SHK_ARRAYROWSPARSE) launch_dia_mode<T, kArray>(A, a, v, grid, blk);
    else if (A->storage == SHK_ROWSYMSPARSE) launch_dia_mode<T, kSym>(A, a, v, grid, blk);
    else launch_dia_mode<T, kCsr>(A, a, v, grid, blk);
    return (int)grid.x;
}
template int launch_dia<double>(shk_csr, SpmvArgs<double> &);
template int launch_dia<float>(shk_csr, SpmvArgs<float> &);

}  // namespace shk
