// shk_resident.hip -- one Cg solve on chip (shk_resident.hpp): the kernel and
// its launch.
#include <algorithm>

#include "shk_resident.hpp"
#include "shk_solver_state.hpp"

namespace shk {

constexpr int kResThreads = 512;
constexpr long long kResWaitSeconds = 2;
// A launch leaves a solve after SHK_OPT_CG_ITERS iterations (2^15: 0.13 s at
// 4 us each) and the next one carries it on: contexts of other threads get
// their turn on the GPU, however long a solve is.  Solves whose max_iter is
// within that take kernels without the provision (LONG), which in the others
// costs registers: 256^2 4.07 -> 4.15 us per iteration, with Jacobi 4.53 -> 5.19,
// 1000^2 10.0 -> 10.1 and 14.3 -> 14.3.

template <typename T>
struct ResSolve {
    int m, left, right, steps, share, k, iters;
    const DiaStep *step;
    const T *val, *diag, *x0;
    T *r;                 // in: the residual; out: the solution, or the residual (each member its own rows)
    ll_word *zw, *slot;
    long long limit;
    KState<T> *st;
};

template <typename T, int RPT, int KS, bool JAC, bool LONG>
__global__ __launch_bounds__(kResThreads, 2) void k_cg_resident(ResSolve<T> a)
{
    extern __shared__ char res_lds[];
    __shared__ ResShared<T> sh;
    KState<T> *st = a.st;
    if (st->skip) return;
    const int tid = threadIdx.x;
    if (tid == 0) sh.bad = 0;
    ResTeam t{a.k, (int)blockIdx.x, LlBuf(a.slot, 2 * a.k * res_slot_words<T>()), 0u, &st->res_stall, a.limit,
              res_every(a.limit)};
    const LlBuf zw(a.zw, (int64_t)a.m * ll_words<T>());
    ResRows R;
    R.r0 = 0;
    R.r1 = a.m;
    R.m0 = min(a.m, t.j * a.share);
    R.m1 = min(a.m, R.m0 + a.share);
    R.left = a.left;
    R.right = a.right;
    R.slice0 = R.m0 / kWave;
    R.steps = R.stride = a.steps;
    R.step = a.step;
    res_window(R);
    T x[RPT], r[RPT];
#pragma unroll
    for (int u = 0; u < RPT; u++) {
        const int row = R.m0 + u * kResThreads + tid;
        x[u] = row < R.m1 ? a.x0[row] : (T)0;
        r[u] = row < R.m1 ? a.r[row] : (T)0;
    }
    const int nb0 = st->nb_iter;
    ResIter<T> it{st->facteur, st->tol, st->max_iter, nb0, 0, st->rho, (T)0, nullptr};
    if (LONG) {  // the launch's share of iterations ends the loop too
        it.max_iter = (int)min((int64_t)nb0 + a.iters, (int64_t)st->max_iter);
        it.rho_1 = st->rho_1;
        it.p = st->res_left;
    }
    double *hist = st->hist;
    int *hist_it = st->hist_it;
    const int hist_cap = st->hist_cap;
    int hist_len = st->hist_len;
    double last = LONG ? st->last_res : 0.0;
    const bool lead = blockIdx.x == 0 && tid == 0;
    unsigned zepoch = 0u;
    __syncthreads();
    // Iteration::Finished (Iterative.cxx:272-319); every member decides alike,
    // the first records it
    const bool ok = res_cg<T, kResThreads, RPT, KS, JAC, LONG>(
        R, a.val, a.diag, x, r, zw, (T *)res_lds, it, t, sh, zepoch, [&](int nb, T rr) {
            const double reste = it.facteur * (double)sqrt_t(rr);
            last = reste;
            if (lead && hist_len < hist_cap) {
                hist[hist_len] = reste;
                hist_it[hist_len] = nb;
            }
            hist_len++;
            return reste < it.tol || nb >= it.max_iter;
        });
    const bool paused = LONG && ok && !it.code && !(last < it.tol) && it.nb < st->max_iter;
    if (!ok) return;
#pragma unroll
    for (int u = 0; u < RPT; u++) {
        const int row = R.m0 + u * kResThreads + tid;
        if (row < R.m1) {
            a.r[row] = LONG && paused ? r[u] : x[u];
            if (LONG && paused) {
                T *left = st->res_left;
                left[row] = ((const T *)res_lds)[row - R.lo];
                left[a.m + row] = x[u];
            }
        }
    }
    if (lead) {
        st->nb_iter = it.nb;
        st->hist_len = hist_len;
        if (it.nb > 0) st->last_res = last;
        if (LONG && paused) {
            st->rho_1 = it.rho_1;
            st->res_paused = 1;
            return;
        }
        if (it.code) {
            st->fail = 1;
            st->error_code = it.code;
        }
        st->done = st->skip = 1;
        st->res_ran = 1;
    }
}

// sum words and z words to epoch 0
template <typename T>
__global__ __launch_bounds__(kBlock) void k_res_clear(int64_t nz, ll_word *zw, int ns, ll_word *slot, KState<T> *st,
                                                     T *left)
{
    if (st->skip) return;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        st->res_paused = 0;
        st->res_left = left;
    }
    for (int64_t i = blockIdx.x * (int64_t)kBlock + threadIdx.x; i < nz; i += (int64_t)gridDim.x * kBlock) zw[i] = 0;
    if (blockIdx.x == 0)
        for (int i = threadIdx.x; i < ns; i += kBlock) slot[i] = 0;
}

// x from the members' results, when all of them came to the end
template <typename T>
__global__ __launch_bounds__(kBlock) void k_res_out(int64_t n, const T *__restrict__ from, T *__restrict__ x,
                                                    const KState<T> *st)
{
    if (!st->res_ran || st->res_stall) return;
    for (int64_t i = blockIdx.x * (int64_t)kBlock + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBlock) x[i] = from[i];
}

// Rows per thread (a member per CU, kResThreads threads each).  Few rows per
// thread keep the sweep over them short, few members the sums: measured on
// 2-D Laplacians, us per iteration with 2 / 4 / 8 rows: 64^2 3.8 / 4.2 / 3.3,
// 256^2 4.0 / 4.2 / 5.0, 512^2 6.8 / 5.4 / 5.5, 64^3 with Jacobi 13.9 / 13.2;
// so two rows up to 128 members of them, then four, and eight only where four
// no longer reach (1000^2: 10.0 against 32.0 for launched kernels).  Seven-step
// rows spill at eight.
static int res_rows_per_thread(int m, int steps, int cus)
{
    for (int r : {2, 4})
        if ((int64_t)m <= (int64_t)r * kResThreads * std::min(cus, 128)) return r;
    return (int64_t)m <= (int64_t)4 * kResThreads * cus || steps > 5 ? 4 : 8;
}

// Stencils of up to seven offsets whose rows, with the band around a member's
// share, fit the members' registers and LDS.
bool cg_resident_fits(shk_csr A)
{
    if (!A->dia_val || A->dia_steps > 7) return false;
    const int cus = std::min(A->ctx->num_cus, kResMaxTeam), rpt = res_rows_per_thread(A->m, A->dia_steps, cus);
    const int64_t share = (int64_t)rpt * kResThreads, halo = (int64_t)A->dia_left + A->dia_right;
    return (A->m + share - 1) / share <= cus && (size_t)(share + halo + 1) * dsize(A->dtype) <= kResLds &&
           share + halo < 0xffff;
}

int cg_resident_groups(shk_csr A)
{
    const int share = res_rows_per_thread(A->m, A->dia_steps, std::min(A->ctx->num_cus, kResMaxTeam)) * kResThreads;
    return (A->m + share - 1) / share;
}

template <typename T, int RPT, int KS>
static void res_launch(const ResSolve<T> &a, dim3 grid, size_t lds, bool jac, bool lng, hipStream_t s)
{
    const dim3 blk(kResThreads);
    if (jac && lng) hipLaunchKernelGGL((k_cg_resident<T, RPT, KS, true, true>), grid, blk, lds, s, a);
    else if (jac) hipLaunchKernelGGL((k_cg_resident<T, RPT, KS, true, false>), grid, blk, lds, s, a);
    else if (lng) hipLaunchKernelGGL((k_cg_resident<T, RPT, KS, false, true>), grid, blk, lds, s, a);
    else hipLaunchKernelGGL((k_cg_resident<T, RPT, KS, false, false>), grid, blk, lds, s, a);
}

template <typename T>
int cg_resident(shk_ctx ctx, shk_csr A, const T *diag, T *x, T *r, void *zw, void *slot, KState<T> *st, T *pause,
                bool carry)
{
    const int rpt = res_rows_per_thread(A->m, A->dia_steps, std::min(ctx->num_cus, kResMaxTeam));
    hipStream_t s = ctx->stream;
    ResSolve<T> a{};
    a.m = A->m;
    a.left = A->dia_left;
    a.right = A->dia_right;
    a.steps = A->dia_steps;
    a.share = rpt * kResThreads;
    a.k = cg_resident_groups(A);
    a.step = (const DiaStep *)A->dia_step;
    a.val = (const T *)A->dia_val;
    a.diag = diag;
    a.x0 = carry ? pause + A->m : x;
    a.r = r;
    a.zw = (ll_word *)zw;
    a.slot = (ll_word *)slot;
    a.st = st;
    SHK_TRY(wait_ticks(ctx, kResWaitSeconds, &a.limit));
    a.iters = (int)ctx->opt[SHK_OPT_CG_ITERS];
    const int64_t nz = (int64_t)A->m * ll_words<T>();
    hipLaunchKernelGGL(k_res_clear<T>, dim3(red_blocks(nz)), dim3(kBlock), 0, s, nz, a.zw,
                       2 * a.k * res_slot_words<T>(), a.slot, st, pause);
    const dim3 grid(a.k);
    const size_t lds = (size_t)(a.share + a.left + a.right + 1) * sizeof(T);
    const bool jac = diag != nullptr, lng = pause != nullptr;
    if (a.steps <= 5) {
        if (rpt == 2) res_launch<T, 2, 5>(a, grid, lds, jac, lng, s);
        else if (rpt == 4) res_launch<T, 4, 5>(a, grid, lds, jac, lng, s);
        else res_launch<T, 8, 5>(a, grid, lds, jac, lng, s);
    } else {
        if (rpt == 2) res_launch<T, 2, 7>(a, grid, lds, jac, lng, s);
        else res_launch<T, 4, 7>(a, grid, lds, jac, lng, s);
    }
    hipLaunchKernelGGL(k_res_out<T>, dim3(red_blocks(A->m)), dim3(kBlock), 0, s, (int64_t)A->m, (const T *)r, x,
                       (const KState<T> *)st);
    SHK_HIP(hipGetLastError());
    return SHK_OK;
}
template int cg_resident<double>(shk_ctx, shk_csr, const double *, double *, double *, void *, void *,
                                 KState<double> *, double *, bool);
template int cg_resident<float>(shk_ctx, shk_csr, const float *, float *, float *, void *, void *, KState<float> *,
                                float *, bool);

}  // namespace shk
