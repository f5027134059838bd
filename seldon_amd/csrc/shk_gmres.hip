// shk_gmres.hip -- the orthogonalisation of one GMRES step in one kernel.
//
// Modified Gram-Schmidt (Gmres.cxx:127-140) needs every (V_k, w) before the
// next update of w, so it is i + 1 passes over w with a sum between them.  As
// one kernel per pass each read w, V_{k-1} and V_k and wrote w (32 bytes per
// FP64 element) and paid a launch.  Here every work-group keeps its part of w
// in registers for all passes and V_k from its dot to its update, so a pass
// reads V_k alone (8 bytes per element), and V_{k+1} is loaded while the sum
// of pass k travels (the epoch words of shk_resident.hpp).  The norm, the
// scaled V_{i+1} and the step's rotations follow in the same kernel.
//
// Same operations per element as before (w += (-h) V_k, V_{i+1} = w (1 / h)),
// the dots in another fixed order.
//
// Bound by the sum (3.2 us over 128 work-groups) and, at 2M rows and more, by
// reading V_k.  Per iteration of GMRES(30) + Jacobi, FP64, a kernel per pass
// -> this: 24^3 rows 104 -> 38 us, 64^3 119 -> 50, 100^3 170 -> 75, 128^3
// 335 -> 120; GMRES(50) on the 4M-row power-law matrix 800 -> 440 (its SpMV
// 290 of them), FP32 390 -> 244.  (A ninth wavefront for the sums alone, V two
// passes ahead: 47 at 64^3, 124 at 128^3, and 16 vectors no longer fit.)
#include <algorithm>

#include "shk_resident.hpp"
#include "shk_solver_state.hpp"

namespace shk {

constexpr int kGoThreads = 512;
constexpr int kGoWaitSeconds = 2;
constexpr int kGoMaxVec = 16;  // 16-byte vectors of w per thread, at most (w, V_k, V_{k+1}: 192 VGPRs)

template <typename T>
struct GmOrtho {
    const T *V;          // V_0; V_k ldv elements after V_{k-1}, zero from n on
    T *vnext;            // V_{i+1}
    const T *w;
    int64_t ldv;         // a multiple of 32
    int i, k;            // the Arnoldi step; work-groups
    unsigned epoch;      // sums posted by the launches before this one
    ll_word *slot;
    long long limit;
    KState<T> *st;
};

template <typename T>
struct GoVec;
template <>
struct GoVec<double> {
    typedef double type __attribute__((ext_vector_type(2)));
};
template <>
struct GoVec<float> {
    typedef float type __attribute__((ext_vector_type(4)));
};

template <typename T, int NV>
__global__ __launch_bounds__(kGoThreads, 2) void k_gm_ortho(GmOrtho<T> a)
{
    using Vec = typename GoVec<T>::type;
    constexpr int N = 16 / (int)sizeof(T);
    extern __shared__ double go_lds[];  // the step's column of H, cosines, sines
    __shared__ ResShared<T> sh;
    KState<T> *st = a.st;
    if (st->skip || st->res_stall) return;
    const int tid = threadIdx.x, i = a.i;
    const bool lead = blockIdx.x == 0;
    double *hc = go_lds, *rc = hc + i + 2, *rs = rc + i + 1;
    if (tid == 0) sh.bad = 0;
    double gs0 = 0.0, gs1 = 0.0;
    if (lead) {
        for (int k = tid; k < i; k += kGoThreads) {
            rc[k] = st->gc[k];
            rs[k] = st->gsn[k];
        }
        if (tid == 0) {
            gs0 = st->gs[i];
            gs1 = st->gs[i + 1];
        }
    }
    ResTeam t{a.k, (int)blockIdx.x, LlBuf(a.slot, 2 * a.k * res_slot_words<T>()), a.epoch, &st->res_stall, a.limit,
               res_every(a.limit)};
    // vector q of this thread: byte q kGoThreads 16 after `at`; past ldv reads
    // are 0 and writes dropped
    const int bytes = (int)(a.ldv * (int64_t)sizeof(T));
    const int at = ((int)blockIdx.x * NV * kGoThreads + tid) * 16;
    auto load = [&](const T *from, Vec (&v)[NV]) {
        const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(const_cast<T *>(from), (short)0, bytes, 0x00020000);
#pragma unroll
        for (int q = 0; q < NV; q++)
            v[q] = __builtin_bit_cast(Vec, __builtin_amdgcn_raw_buffer_load_b128(r, at, q * kGoThreads * 16, 0));
    };
    // pass k with V_k in `cur`; V_{k+1} loads into `next` while the sum travels
    // (two sets taken in turn: a copy between them would wait for the loads)
    Vec w[NV], va[NV], vb[NV];
    auto pass = [&](const Vec (&cur)[NV], Vec (&next)[NV], int k) {
        T c[1] = {(T)0};
#pragma unroll
        for (int q = 0; q < NV; q++)
#pragma unroll
            for (int e = 0; e < N; e++) c[0] += cur[q][e] * w[q][e];
        // many loads hold the post up behind them in the CU's memory pipeline
        // (16 vectors: 128.7 us per iteration at 128^3 rows, 120.2 with the
        // post first), few are better on their way while the work-group meets
        // (2 vectors, 64^3 rows: 50.0 against 52.2)
        constexpr bool kPostFirst = NV >= 8;
        if constexpr (kPostFirst) res_post<T, 1, kGoThreads>(c, t, sh);
        __builtin_amdgcn_sched_barrier(0);
        load(a.V + (size_t)min(k + 1, i) * a.ldv, next);  // the last pass reads its own V_i again, unused
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (!kPostFirst) res_post<T, 1, kGoThreads>(c, t, sh);
        if (!res_wait<T, 1, kGoThreads>(c, t, sh)) return false;
        const double h = (double)c[0];
        if (lead && tid == 0) hc[k] = h;
        const T m = (T)(-h);
        if (m != (T)0) {
#pragma unroll
            for (int q = 0; q < NV; q++)
#pragma unroll
                for (int e = 0; e < N; e++) w[q][e] += m * cur[q][e];
        }
        return true;
    };
    load(a.w, w);
    load(a.V, va);
    __syncthreads();  // sh.bad
    for (int k = 0;; k += 2) {
        if (!pass(va, vb, k)) return;
        if (k + 1 > i) break;
        if (!pass(vb, va, k + 1)) return;
        if (k + 2 > i) break;
    }
    T c[1] = {(T)0};
#pragma unroll
    for (int q = 0; q < NV; q++)
#pragma unroll
        for (int e = 0; e < N; e++) c[0] += w[q][e] * w[q][e];
    res_post<T, 1, kGoThreads>(c, t, sh);
    if (!res_wait<T, 1, kGoThreads>(c, t, sh)) return;
    double hi = (double)sqrt_t(c[0]);
    const T scale = hi != 0.0 ? (T)(1.0 / hi) : (T)1;
    // ordinary stores under a bounds test: what may follow a 16-byte store is
    // the compiler's to arrange (buffer stores whose offset was in a register
    // got no wait before the next write to their data, and V_{i+1} came out
    // wrong now and then where the registers were used again)
#pragma unroll
    for (int q = 0; q < NV; q++) {
        const int o = at + q * kGoThreads * 16;
        if (o < bytes) *(Vec *)((char *)a.vnext + o) = w[q] * scale;
    }
    if (!lead) return;
    // FinGmStep's end of step on the LDS column (Gmres.cxx:135-162)
    if (tid == 0) {
        st->gm_hi = hi;
        st->gm_scale = scale;
        double x = hc[0];
        for (int k = 0; k < i; k++) {
            double y = hc[k + 1];
            dev_applyrot(x, y, rc[k], rs[k]);
            hc[k] = x;
            x = y;
        }
        hc[i] = x;
        if (hi != 0.0) {
            double cs, sn;
            dev_genrot(hc[i], hi, cs, sn);
            dev_applyrot(gs0, gs1, cs, sn);
            st->gc[i] = cs;
            st->gsn[i] = sn;
            st->gs[i] = gs0;
            st->gs[i + 1] = gs1;
        }
        st->gm_inner_nb++;
        st->nb_iter++;
        st->gm_i = i + 1;
        if (it_finished(st, fabs(gs1), st->gm_inner_nb, st->gm_inner_max)) {
            st->gm_cycle_done = 1;
            st->skip = 1;
        }
    }
    __syncthreads();
    double *H = st->H + (size_t)i * (st->gm_m + 1);
    for (int k = tid; k <= i; k += kGoThreads) H[k] = hc[k];
}

// sum words to epoch 0
__global__ void k_go_clear(int n, ll_word *slot)
{
    for (int j = threadIdx.x; j < n; j += blockDim.x) slot[j] = 0;
}

// Vectors per thread: few work-groups make the sums short, few vectors the
// pass.  The smallest count that needs no more than 128 work-groups (measured
// at 32 / 64 / 128 / 256: 64^3 rows 52.8 / 49.8 / 51.3 / 51.2 us per
// iteration, 100^3 86.6 / 85.8 / 80.2 / 86.1, 128^3 134 / 135 / 134 / 136).
static int go_vectors(int64_t vecs, int cus)
{
    int nv = 2;
    while (nv < kGoMaxVec && vecs > (int64_t)nv * kGoThreads * std::min(cus, 128)) nv *= 2;
    return nv;
}

template <typename T>
bool gm_ortho_fits(shk_ctx ctx, int64_t ldv, int m)
{
    const int cus = std::min(ctx->num_cus, kResMaxTeam);
    return ldv * (int64_t)sizeof(T) / 16 <= (int64_t)kGoMaxVec * kGoThreads * cus && m <= 1000;
}

// work-groups of a step
template <typename T>
int gm_ortho_groups(shk_ctx ctx, int64_t ldv)
{
    const int64_t vecs = ldv * (int64_t)sizeof(T) / 16;
    const int64_t per = (int64_t)go_vectors(vecs, std::min(ctx->num_cus, kResMaxTeam)) * kGoThreads;
    return (int)((vecs + per - 1) / per);
}

size_t gm_ortho_words() { return 2 * (size_t)kResMaxTeam * res_slot_words<double>(); }

template <typename T>
int gm_ortho_start(shk_ctx ctx, void *slot)
{
    hipLaunchKernelGGL(k_go_clear, dim3(1), dim3(kBlock), 0, ctx->stream, (int)gm_ortho_words(), (ll_word *)slot);
    SHK_HIP(hipGetLastError());
    return SHK_OK;
}

template <typename T>
int gm_ortho(shk_ctx ctx, const T *V, int64_t ldv, T *w, int i, unsigned *epoch, void *slot, KState<T> *st)
{
    const int64_t vecs = ldv * (int64_t)sizeof(T) / 16;
    const int nv = go_vectors(vecs, std::min(ctx->num_cus, kResMaxTeam));
    GmOrtho<T> a{};
    a.V = V;
    a.vnext = const_cast<T *>(V) + (size_t)(i + 1) * ldv;
    a.w = w;
    a.ldv = ldv;
    a.i = i;
    a.k = gm_ortho_groups<T>(ctx, ldv);
    a.epoch = *epoch;
    a.slot = (ll_word *)slot;
    a.st = st;
    SHK_TRY(wait_ticks(ctx, kGoWaitSeconds, &a.limit));
    *epoch += (unsigned)i + 2;
    const size_t lds = sizeof(double) * 3 * ((size_t)i + 2);
    const dim3 grid(a.k), blk(kGoThreads);
    hipStream_t s = ctx->stream;
    switch (nv) {
    case 2: hipLaunchKernelGGL((k_gm_ortho<T, 2>), grid, blk, lds, s, a); break;
    case 4: hipLaunchKernelGGL((k_gm_ortho<T, 4>), grid, blk, lds, s, a); break;
    case 8: hipLaunchKernelGGL((k_gm_ortho<T, 8>), grid, blk, lds, s, a); break;
    default: hipLaunchKernelGGL((k_gm_ortho<T, 16>), grid, blk, lds, s, a); break;
    }
    SHK_HIP(hipGetLastError());
    return SHK_OK;
}

template bool gm_ortho_fits<double>(shk_ctx, int64_t, int);
template bool gm_ortho_fits<float>(shk_ctx, int64_t, int);
template int gm_ortho_groups<double>(shk_ctx, int64_t);
template int gm_ortho_groups<float>(shk_ctx, int64_t);
template int gm_ortho_start<double>(shk_ctx, void *);
template int gm_ortho_start<float>(shk_ctx, void *);
template int gm_ortho<double>(shk_ctx, const double *, int64_t, double *, int, unsigned *, void *, KState<double> *);
template int gm_ortho<float>(shk_ctx, const float *, int64_t, float *, int, unsigned *, void *, KState<float> *);

}  // namespace shk
