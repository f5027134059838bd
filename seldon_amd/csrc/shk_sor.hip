// shk_sor.hip -- Seldon's SOR / SSOR sweeps on the device.
//
// SOR(A, X, B, omega, iter, type_ssor) runs iter forward sweeps when
// type_ssor % 2 == 0, then iter backward sweeps when type_ssor % 3 == 0.
//
// General storages (matrix_sparse/Relaxation_MatVect.cxx:41-95 RowSparse,
// :106-167 ArrayRowSparse) update X row after row:
//   temp = sum_k a_jk X(ind_k)          (the whole row, stored order)
//   temp = B(j) - temp + ajj * X(j)
//   X(j) = (1 - omega) * X(j) + omega * temp / ajj
// with the rows in increasing order (forward) or decreasing (backward).  A
// row reads the new X of the rows swept before it and the old X of the
// others.
//
// A sweep is one kernel.  The new values go to words that say which sweep
// wrote them ({sweep number, 32 bits of the value}, as in shk_resident.hpp);
// a row polls the words of the rows it needs, forms its own value and writes
// its word.  X itself, which holds every old value, is only read during the
// sweep and takes the new values after it, so a row never has to wait for the
// readers of its old value.  Rows are taken in the order of the dependence
// levels (a row's level is one more than the highest it reads a new value
// from), 64 rows of one level at most at a time, by wavefronts that draw the
// next piece from a counter: the lowest unfinished piece is always being
// worked on and needs only finished ones, so every wait ends whatever part of
// the GPU the kernel gets.  Every row sees exactly the operands of the
// sequential sweep, in its order: the results are bitwise Seldon's.
//
// The words and counters of a sweep are of one call at a time (SorWork): a
// context's direct calls follow each other and share one set, and every
// capture has its own, since replays may overlap direct calls and each other.
//
// Bound by the chain of levels: a word's way from one work-group to another
// and the division behind it, 1.0 us per level on 2-D grids, 1.7 on the 128^3
// one.  (A launch per level cost 9 us, one work-group stepping through small
// levels 2.5.)  Symmetric sweep, FP64, before -> after: 128^3
// convection-diffusion (2 x 382 levels) 5.81 -> 1.36 ms, 64^3 2.51 -> 0.54,
// 16^3 0.194 -> 0.135; 256^2 Laplacian RowSparse 2.56 -> 1.09, RowSymSparse
// 2.02 -> 1.04; 50K-row power-law matrix 85.6 -> 43.7.
//
// RowSymSparse (:179-300, upper triangle stored) splits each sweep in two
// passes.  Forward: Z(j) = (1-w)/w ajj X(j) + (B(j) - sum_{p>j} a_jp X(p))
// from the old X (one launch over all rows), then the lower solve
// X(p) = (Z(p) - sum_{j<p} a_jp X(j)) * (w / ajj), the sum over column p of
// the stored triangle in Seldon's scatter order (rows increasing), by levels.
// Backward: Y(j) = sum_{i<j} a_ij X(i) (old X, same order) and
// Z(j) = (1-w)/w ajj X(j) + B(j) - Y(j) in one launch, then the upper solve
// X(j) = (Z(j) - sum_{p>j} a_jp X(p)) w / ajj in decreasing levels.
//
// omega is applied in the type C++ gives (value, omega): a double omega on
// float values makes each relaxation step double, rounded once on the store.
#include <algorithm>
#include <string>
#include <vector>

#include "shk_resident.hpp"

namespace shk {

constexpr int kSorBatch = 8;              // entries of a row in flight at a time
constexpr long long kSorWaitSeconds = 4;  // a wait before the sweep is left to one work-group

constexpr int kSorOwnPolls = 1 << 20;     // looks at a word the wavefront wrote itself, at most

// device counters of the sweeps
struct SorState {
    unsigned ticket, stall, sweep;
};

// What a sweep writes besides X, in one allocation.
struct SorWork {
    SorState *state = nullptr;
    // the new value of each row, in the order of rows[d]: a piece writes
    // consecutive words, and the rows it waits for stand close together in the
    // levels before it (by row number a 64-row piece of a 3-D grid polls up to
    // 192 cache lines: 2.18 instead of 1.36 ms at 128^3)
    ll_word *word = nullptr;
    void *z = nullptr;                // RowSymSparse: the half-step vector
    unsigned long long capture = 0;   // the capture it is of (0: direct calls),
    hipStream_t stream = nullptr;     // on this stream of it
};

struct SorPlan {
    int m = 0, storage = 0, dtype = 0;
    int *ptr = nullptr, *ind = nullptr;  // the stored rows
    void *val = nullptr, *diag = nullptr;
    int *tptr = nullptr, *tind = nullptr;  // RowSymSparse: strict upper entries by column
    void *tval = nullptr;                  // (rows increasing)
    int *rows[2] = {nullptr, nullptr};     // forward, backward: rows by level
    int *pos[2] = {nullptr, nullptr};      // where each row stands in rows[d]
    int2 *piece[2] = {nullptr, nullptr};   // {first of rows[d], count}: up to 64 rows of one level
    int npiece[2] = {0, 0};
    std::vector<SorWork> work;             // [0]: direct calls
};

// ---- row operations ------------------------------------------------------
// Each names its rows' entries (ptr, ind, val), says whether entry column c
// is read new, old or not at all, loads what else a row needs (before it
// waits), and forms the row's value from the sum of its entries in stored
// order.
enum SorRead { kSorOld, kSorNew, kSorNone };

// general storages: one row of the sweep
template <typename T, typename W>
struct SorRow {
    const int *ptr, *ind;
    const T *val, *diag, *B;
    const T *X;
    W omega;
    bool forward;
    static constexpr bool kSubtract = false;
    __device__ __forceinline__ SorRead read(int j, int c) const
    {
        return (forward ? c < j : c > j) ? kSorNew : kSorOld;
    }
    struct Row {
        T ajj, xj, b;
    };
    __device__ __forceinline__ Row load(int j) const { return Row{diag[j], X[j], B[j]}; }
    __device__ __forceinline__ T start(const Row &) const { return (T)0; }
    __device__ __forceinline__ T value(const Row &r, T temp) const
    {
        temp = r.b - temp + r.ajj * r.xj;
        return (T)(((W)1 - omega) * (W)r.xj + omega * (W)temp / (W)r.ajj);
    }
};

// RowSymSparse forward solve: X(p) = (Z(p) - sum_j a_jp X(j)) * (w / ajj)
template <typename T, typename W>
struct SymForward {
    const int *ptr, *ind;  // strict upper entries by column
    const T *val, *diag, *Z;
    const T *X;
    W omega;
    static constexpr bool kSubtract = true;
    __device__ __forceinline__ SorRead read(int, int) const { return kSorNew; }
    struct Row {
        T z;
        W f;
    };
    __device__ __forceinline__ Row load(int p) const { return Row{Z[p], omega / (W)diag[p]}; }
    __device__ __forceinline__ T start(const Row &r) const { return r.z; }
    __device__ __forceinline__ T value(const Row &r, T x) const { return (T)((W)x * r.f); }
};

// RowSymSparse backward solve: X(j) = (Z(j) - sum_{p != j} a_jp X(p)) w / ajj
template <typename T, typename W>
struct SymBackward {
    const int *ptr, *ind;
    const T *val, *diag, *Z;
    const T *X;
    W omega;
    static constexpr bool kSubtract = false;
    __device__ __forceinline__ SorRead read(int j, int c) const { return c == j ? kSorNone : kSorNew; }
    struct Row {
        T z, ajj;
    };
    __device__ __forceinline__ Row load(int j) const { return Row{Z[j], diag[j]}; }
    __device__ __forceinline__ T start(const Row &) const { return (T)0; }
    __device__ __forceinline__ T value(const Row &r, T temp) const
    {
        return (T)((W)(r.z - temp) * omega / (W)r.ajj);
    }
};

// no word carries a sweep number yet: sweeps count from 1
__global__ __launch_bounds__(kBlock) void k_sor_clear(int64_t n, ll_word *words, SorState *st)
{
    const int64_t i0 = blockIdx.x * (int64_t)kBlock + threadIdx.x;
    if (i0 == 0) *st = SorState{0u, 0u, 0u};
    for (int64_t i = i0; i < n; i += (int64_t)gridDim.x * kBlock) words[i] = 0;
}

// the next sweep: its number, and its counters to their start
__global__ void k_sor_begin(SorState *st)
{
    st->ticket = 0u;
    st->stall = 0u;
    st->sweep++;
}

// One sweep: wavefronts draw pieces until none is left.  `rescue`: only when
// the sweep before it gave up waiting (a GPU shared with long-running work),
// by a single wavefront, which takes the pieces in order: every word it needs
// is one it has written itself, so it waits for nobody.
template <typename T, class Words, class Op>
__global__ __launch_bounds__(kBlock) void k_sor_sweep(int m, const int *__restrict__ rows, const int *__restrict__ pos,
                                                      const int2 *__restrict__ piece, int npiece, Op op,
                                                      ll_word *words, SorState *st, long long limit, bool rescue,
                                                      unsigned *rescued)
{
    if (rescue && !st->stall) return;
    if (rescue && threadIdx.x == 0) atomicAdd(rescued, 1u);
    const unsigned sweep = st->sweep;
    const Words w(words, (int64_t)m * ll_words<T>());
    const int lane = threadIdx.x & (kWave - 1);
    auto draw = [&](int after) {
        if (rescue) return after + 1;
        int q = 0;
        if (lane == 0) q = (int)atomicAdd(&st->ticket, 1u);
        return __builtin_amdgcn_readfirstlane(q);
    };
    for (int q = draw(-1); q < npiece;) {
        const int next = draw(q);  // on its way while this piece waits
        const int2 pc = piece[q];
        const bool in = lane < pc.y;
        const int j = rows[pc.x + (in ? lane : 0)];
        const int p0 = op.ptr[j], len = in ? op.ptr[j + 1] - p0 : 0;
        int most = len;
        for (int o = 32; o > 0; o >>= 1) most = max(most, __shfl_xor(most, o, kWave));
        const typename Op::Row row = op.load(j);
        T acc = op.start(row);
        for (int k0 = 0; k0 < most; k0 += kSorBatch) {
            int c[kSorBatch], how[kSorBatch];
            T v[kSorBatch], x[kSorBatch];
#pragma unroll
            for (int u = 0; u < kSorBatch; u++) {
                const int k = k0 + u < len ? p0 + k0 + u : 0;
                c[u] = op.ind[k];
                v[u] = op.val[k];
            }
            unsigned need = 0u;  // entries some lane reads new
#pragma unroll
            for (int u = 0; u < kSorBatch; u++) {
                how[u] = k0 + u < len ? (int)op.read(j, c[u]) : (int)kSorNone;
                if (__builtin_amdgcn_ballot_w64(how[u] == kSorNew)) need |= 1u << u;
                x[u] = how[u] == kSorOld ? op.X[c[u]] : (T)0;
                c[u] = how[u] == kSorNew ? pos[c[u]] : pc.x;  // the word to poll
            }
            if (need) {
                const long long t0 = wall_clock64();
                for (int n = 1;; n++) {
                    asm volatile("" ::: "memory");  // the words are read again
                    // every word is on its way before the first is looked at
                    typename Words::template Raw<T> raw[kSorBatch];
#pragma unroll
                    for (int u = 0; u < kSorBatch; u++)
                        if (need >> u & 1u)
                            raw[u] = w.template read<T>((int64_t)c[u] * ll_words<T>());
                    bool all = true;
#pragma unroll
                    for (int u = 0; u < kSorBatch; u++)
                        if (need >> u & 1u) {
                            T y;
                            const bool got = Words::value(raw[u], y, sweep);
                            if (how[u] == kSorNew) {
                                x[u] = y;
                                all &= got;
                            }
                        }
                    if (!__builtin_amdgcn_ballot_w64(!all)) break;
                    if (rescue) {
                        if (n == kSorOwnPolls) break;
                    } else if ((n & 255) == 0 || limit <= 0) {
                        const bool late = wall_clock64() - t0 >= limit;
                        if (late) __hip_atomic_store(&st->stall, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                        if (late || __hip_atomic_load(&st->stall, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) return;
                    }
                }
            }
#pragma unroll
            for (int u = 0; u < kSorBatch; u++)
                if (how[u] != kSorNone) {
                    const T t = v[u] * x[u];
                    acc = Op::kSubtract ? acc - t : acc + t;
                }
        }
        if (in) ll_put(w, (int64_t)(pc.x + lane) * ll_words<T>(), op.value(row, acc), sweep);
        q = next;
    }
}

// X from the sweep's words
template <typename T, class Words>
__global__ __launch_bounds__(kBlock) void k_sor_out(int m, const int *__restrict__ pos, ll_word *words,
                                                    T *__restrict__ X, const SorState *st)
{
    const Words w(words, (int64_t)m * ll_words<T>());
    const unsigned sweep = st->sweep;
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= m) return;
    T v;
    ll_get(w, (int64_t)pos[i] * ll_words<T>(), v, sweep);
    X[i] = v;
}

// ---- RowSymSparse explicit halves ----------------------------------------
// forward: Z(j) = (1-w)/w ajj X(j) + (B(j) - sum_{p != j} a_jp X(p))
template <typename T, typename W>
__global__ __launch_bounds__(kBlock) void k_sor_sym_f1(int m, const int *__restrict__ ptr, const int *__restrict__ ind,
                                                       const T *__restrict__ val, const T *__restrict__ diag,
                                                       const T *__restrict__ B, const T *__restrict__ X,
                                                       T *__restrict__ Z, W omega)
{
    const int j = blockIdx.x * kBlock + threadIdx.x;
    if (j >= m) return;
    T temp = (T)0;
    for (int k = ptr[j]; k < ptr[j + 1]; k++)
        if (ind[k] != j) temp += val[k] * X[ind[k]];
    temp = B[j] - temp;
    Z[j] = (T)(((W)1 - omega) / omega * (W)diag[j] * (W)X[j] + (W)temp);
}

// backward: Z(j) = (1-w)/w ajj X(j) + B(j) - sum_{i<j} a_ij X(i)
template <typename T, typename W>
__global__ __launch_bounds__(kBlock) void k_sor_sym_b1(int m, const int *__restrict__ tptr,
                                                       const int *__restrict__ tind, const T *__restrict__ tval,
                                                       const T *__restrict__ diag, const T *__restrict__ B,
                                                       const T *__restrict__ X, T *__restrict__ Z, W omega)
{
    const int j = blockIdx.x * kBlock + threadIdx.x;
    if (j >= m) return;
    T y = (T)0;
    for (int k = tptr[j]; k < tptr[j + 1]; k++) y += tval[k] * X[tind[k]];
    Z[j] = (T)(((W)1 - omega) / omega * (W)diag[j] * (W)X[j] + (W)B[j] - (W)y);
}

// ---- plan ----------------------------------------------------------------
// Rows of one sweep direction (dir 0: rows 0..m-1, dir 1: m-1..0) by level,
// and the levels cut into pieces of up to 64 rows.
static void sor_levels(int m, const std::vector<int> &ptr, const std::vector<int> &ind, int dir,
                       std::vector<int> &rows, std::vector<int> &pos, std::vector<int2> &piece)
{
    std::vector<int> lev(m, 0);
    int nlev = 0;
    for (int q = 0; q < m; q++) {
        const int j = dir == 0 ? q : m - 1 - q;
        int L = 0;
        for (int k = ptr[j]; k < ptr[j + 1]; k++) {
            const int c = ind[k];
            const bool before = dir == 0 ? c < j : c > j;  // swept before j: read new
            if (before) L = std::max(L, lev[c] + 1);
        }
        lev[j] = L;
        nlev = std::max(nlev, L + 1);
    }
    std::vector<int> off((size_t)nlev + 1, 0);
    for (int j = 0; j < m; j++) off[(size_t)lev[j] + 1]++;
    for (int l = 0; l < nlev; l++) off[(size_t)l + 1] += off[l];
    std::vector<int> next(off.begin(), off.end() - 1);
    rows.assign(m, 0);
    pos.assign(m, 0);
    for (int j = 0; j < m; j++) {
        pos[j] = next[lev[j]]++;
        rows[pos[j]] = j;
    }
    piece.clear();
    for (int l = 0; l < nlev; l++)
        for (int q = off[l]; q < off[(size_t)l + 1]; q += kWave)
            piece.push_back(make_int2(q, std::min(kWave, off[(size_t)l + 1] - q)));
}

// Seldon's A(j, j) on RowSparse (matrix_sparse/Matrix_Sparse.cxx:1054-1084):
// the scan moves on while the column is below j and stops at the row's last
// entry; the entry it stops on counts if its column is j, else a_jj = 0.
template <typename T>
static T rowsparse_diag(const std::vector<int> &ptr, const std::vector<int> &ind, const std::vector<T> &val, int j)
{
    const int first = ptr[j], last = ptr[(size_t)j + 1] - 1;
    if (last < first) return (T)0;
    int k = first;
    while (k < last && ind[k] < j) k++;
    return ind[k] == j ? val[k] : (T)0;
}

template <typename V>
static hipError_t put(V **dst, const std::vector<V> &src, hipStream_t s)
{
    hipError_t e = hipMalloc((void **)dst, sizeof(V) * std::max<size_t>(src.size(), 1));
    if (e == hipSuccess && !src.empty())
        e = hipMemcpyAsync(*dst, src.data(), sizeof(V) * src.size(), hipMemcpyHostToDevice, s);
    return e;
}

// state, words and (RowSymSparse) the half-step vector of P's sweeps
template <typename T>
static hipError_t sor_work_alloc(const SorPlan *P, SorWork &w)
{
    auto al = [](size_t v) { return (v + 255) & ~(size_t)255; };
    const size_t sb = al(sizeof(SorState)), wb = al(sizeof(ll_word) * ll_words<T>() * (size_t)P->m),
                 zb = P->storage == SHK_ROWSYMSPARSE ? sizeof(T) * (size_t)P->m : 0;
    char *p = nullptr;
    const hipError_t e = hipMalloc((void **)&p, sb + wb + zb);
    if (e != hipSuccess) return e;
    w.state = (SorState *)p;
    w.word = (ll_word *)(p + sb);
    w.z = p + sb + wb;
    return hipSuccess;
}

template <typename T>
static void sor_clear(const SorPlan *P, const SorWork &w, hipStream_t s)
{
    const int64_t n = (int64_t)P->m * ll_words<T>();
    hipLaunchKernelGGL(k_sor_clear, dim3(red_blocks(n)), dim3(kBlock), 0, s, n, w.word, w.state);
}

// What a call on the context's stream may write.  Direct calls follow each
// other: a context has one stream, and is synchronised where that changes.
// Captured calls of one capture and stream follow each other too; their words
// start from nothing on every replay.
template <typename T>
static int sor_work(shk_ctx ctx, SorPlan *P, SorWork &out)
{
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    unsigned long long id = 0;
    if (hipStreamGetCaptureInfo(ctx->stream, &cs, &id) != hipSuccess) (void)hipGetLastError();
    if (cs != hipStreamCaptureStatusActive) {
        out = P->work[0];
        return SHK_OK;
    }
    for (size_t i = 1; i < P->work.size(); i++)
        if (P->work[i].capture == id && P->work[i].stream == ctx->stream) {
            out = P->work[i];
            return SHK_OK;
        }
    SorWork w;
    w.capture = id;
    w.stream = ctx->stream;
    // an allocation is no part of the capture
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
    SHK_HIP(hipThreadExchangeStreamCaptureMode(&mode));
    const hipError_t e = sor_work_alloc<T>(P, w);
    (void)hipThreadExchangeStreamCaptureMode(&mode);
    if (e != hipSuccess) return fail(SHK_ERR_NOMEM, std::string("sor: device memory: ") + hipGetErrorString(e));
    sor_clear<T>(P, w, ctx->stream);
    P->work.push_back(w);
    out = w;
    return SHK_OK;
}

template <typename T>
static int sor_build(shk_csr A, SorPlan **out)
{
    std::vector<int> ptr, ind;
    std::vector<T> val;
    SHK_TRY(stored_arrays<T>(A, ptr, ind, val));
    const int m = A->m;
    const bool sym = A->storage == SHK_ROWSYMSPARSE;
    // ajj: RowSparse reads A(j, j); ArrayRowSparse and RowSymSparse add the
    // row's diagonal entries onto 0 (Relaxation_MatVect.cxx:136-140, :217-225)
    std::vector<T> diag(m, (T)0);
    for (int j = 0; j < m; j++) {
        if (A->storage == SHK_ROWSPARSE) {
            diag[j] = rowsparse_diag(ptr, ind, val, j);
            continue;
        }
        for (int k = ptr[j]; k < ptr[(size_t)j + 1]; k++) {
            SHK_CHECK(!sym || ind[k] >= j, SHK_ERR_ARG, "sor: a RowSymSparse entry below the diagonal");
            if (ind[k] == j) diag[j] += val[k];
        }
    }
    std::vector<int> rows[2], pos[2], tptr, tind;
    std::vector<T> tval;
    std::vector<int2> piece[2];
    if (sym) {
        // strict upper entries gathered by column, rows increasing (a stable
        // counting sort of the row-major entries)
        tptr.assign((size_t)m + 1, 0);
        for (int j = 0; j < m; j++)
            for (int k = ptr[j]; k < ptr[(size_t)j + 1]; k++)
                if (ind[k] != j) tptr[(size_t)ind[k] + 1]++;
        for (int p = 0; p < m; p++) tptr[(size_t)p + 1] += tptr[p];
        tind.resize(tptr[m]);
        tval.resize(tptr[m]);
        std::vector<int> next(tptr.begin(), tptr.end() - 1);
        for (int j = 0; j < m; j++)
            for (int k = ptr[j]; k < ptr[(size_t)j + 1]; k++)
                if (ind[k] != j) {
                    const int q = next[ind[k]]++;
                    tind[q] = j;
                    tval[q] = val[k];
                }
        // the forward solve's row p reads the X(j) of its column entries, the
        // backward solve's row j the X(p) of its row entries
        sor_levels(m, tptr, tind, 0, rows[0], pos[0], piece[0]);
        sor_levels(m, ptr, ind, 1, rows[1], pos[1], piece[1]);
    } else {
        for (int d = 0; d < 2; d++) sor_levels(m, ptr, ind, d, rows[d], pos[d], piece[d]);
    }
    SorPlan *P = new SorPlan;
    P->m = m;
    P->storage = A->storage;
    P->dtype = A->dtype;
    for (int d = 0; d < 2; d++) P->npiece[d] = (int)piece[d].size();
    hipStream_t s = A->ctx->stream;
    hipError_t e = put(&P->ptr, ptr, s);
    if (e == hipSuccess) e = put(&P->ind, ind, s);
    if (e == hipSuccess) e = put((T **)&P->val, val, s);
    if (e == hipSuccess) e = put((T **)&P->diag, diag, s);
    for (int d = 0; d < 2 && e == hipSuccess; d++) e = put(&P->rows[d], rows[d], s);
    for (int d = 0; d < 2 && e == hipSuccess; d++) e = put(&P->pos[d], pos[d], s);
    for (int d = 0; d < 2 && e == hipSuccess; d++) e = put(&P->piece[d], piece[d], s);
    P->work.emplace_back();
    if (e == hipSuccess) e = sor_work_alloc<T>(P, P->work[0]);
    if (e == hipSuccess) sor_clear<T>(P, P->work[0], s);
    if (sym) {
        if (e == hipSuccess) e = put(&P->tptr, tptr, s);
        if (e == hipSuccess) e = put(&P->tind, tind, s);
        if (e == hipSuccess) e = put((T **)&P->tval, tval, s);
    }
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    if (e != hipSuccess) {
        sor_free(P);
        return fail(SHK_ERR_NOMEM, std::string("sor: device memory: ") + hipGetErrorString(e));
    }
    *out = P;
    return SHK_OK;
}

void sor_free(SorPlan *P)
{
    if (!P) return;
    hipFree(P->ptr);
    hipFree(P->ind);
    hipFree(P->val);
    hipFree(P->diag);
    hipFree(P->tptr);
    hipFree(P->tind);
    hipFree(P->tval);
    hipFree(P->rows[0]);
    hipFree(P->rows[1]);
    hipFree(P->pos[0]);
    hipFree(P->pos[1]);
    hipFree(P->piece[0]);
    hipFree(P->piece[1]);
    for (const SorWork &w : P->work) hipFree(w.state);
    delete P;
}

static inline dim3 grid_for(int count) { return dim3((count + kBlock - 1) / kBlock); }

// One sweep's triangular part.  Four wavefronts per work-group and one
// work-group per CU at most: more of them than the levels can use only poll
// (128^3 with 64 / 128 / 256 / 512 work-groups: 1.78 / 1.40 / 1.36 / 1.45 ms).
template <typename T, class Words, class Op>
static void launch_sweep(shk_ctx ctx, const SorPlan *P, const SorWork &w, long long limit, int d, const Op &op, T *X)
{
    hipStream_t s = ctx->stream;
    const int np = P->npiece[d], waves = kBlock / kWave;
    const dim3 grid(std::max(1, std::min((np + waves - 1) / waves, ctx->num_cus))), blk(kBlock);
    unsigned *rescued = ctx->red.ticket + kRescuedSlot;
    hipLaunchKernelGGL(k_sor_begin, dim3(1), dim3(1), 0, s, w.state);
    hipLaunchKernelGGL((k_sor_sweep<T, Words, Op>), grid, blk, 0, s, P->m, (const int *)P->rows[d],
                       (const int *)P->pos[d], (const int2 *)P->piece[d], np, op, w.word, w.state, limit, false, rescued);
    hipLaunchKernelGGL((k_sor_sweep<T, Words, Op>), dim3(1), dim3(kWave), 0, s, P->m, (const int *)P->rows[d],
                       (const int *)P->pos[d], (const int2 *)P->piece[d], np, op, w.word, w.state, limit, true, rescued);
    hipLaunchKernelGGL((k_sor_out<T, Words>), grid_for(P->m), blk, 0, s, P->m, (const int *)P->pos[d], w.word, X,
                       (const SorState *)w.state);
}

// 32-bit buffer offsets reach 2 GiB of words (134M FP64 rows)
template <typename T, class Op>
static void run_sweep(shk_ctx ctx, const SorPlan *P, const SorWork &w, long long limit, int d, const Op &op, T *X)
{
    if ((int64_t)P->m * ll_words<T>() * (int64_t)sizeof(ll_word) < ctx->opt[SHK_OPT_BUFFER_BYTES])
        launch_sweep<T, LlBuf>(ctx, P, w, limit, d, op, X);
    else
        launch_sweep<T, LlPtr>(ctx, P, w, limit, d, op, X);
}

template <typename T, typename W>
static int sor_run(shk_ctx ctx, SorPlan *P, T *X, const T *B, W omega, int iter, int type_ssor)
{
    hipStream_t s = ctx->stream;
    const T *val = (const T *)P->val, *diag = (const T *)P->diag, *tval = (const T *)P->tval;
    SorWork w;
    SHK_TRY(sor_work<T>(ctx, P, w));
    long long limit = 0;
    SHK_TRY(wait_ticks(ctx, kSorWaitSeconds, &limit));
    T *Z = (T *)w.z;
    auto sweep = [&](int d) {
        if (P->storage != SHK_ROWSYMSPARSE) {
            run_sweep<T>(ctx, P, w, limit, d, SorRow<T, W>{P->ptr, P->ind, val, diag, B, X, omega, d == 0}, X);
        } else if (d == 0) {
            hipLaunchKernelGGL((k_sor_sym_f1<T, W>), grid_for(P->m), dim3(kBlock), 0, s, P->m, P->ptr, P->ind, val,
                               diag, B, (const T *)X, Z, omega);
            run_sweep<T>(ctx, P, w, limit, 0, SymForward<T, W>{P->tptr, P->tind, tval, diag, Z, X, omega}, X);
        } else {
            hipLaunchKernelGGL((k_sor_sym_b1<T, W>), grid_for(P->m), dim3(kBlock), 0, s, P->m, P->tptr, P->tind,
                               tval, diag, B, (const T *)X, Z, omega);
            run_sweep<T>(ctx, P, w, limit, 1, SymBackward<T, W>{P->ptr, P->ind, val, diag, Z, X, omega}, X);
        }
    };
    if (type_ssor % 2 == 0)
        for (int i = 0; i < iter; i++) sweep(0);
    if (type_ssor % 3 == 0)
        for (int i = 0; i < iter; i++) sweep(1);
    SHK_HIP(hipGetLastError());
    return SHK_OK;
}

}  // namespace shk

using namespace shk;

extern "C" {

int shk_sor(shk_ctx ctx, shk_csr A, void *dx, const void *db, double omega, shk_dtype omega_type, int iter,
            int type_ssor)
{
    SHK_CHECK(ctx && A && A->ctx == ctx, SHK_ERR_ARG, "sor: null or foreign argument");
    SHK_CHECK(A->storage == SHK_ROWSPARSE || A->storage == SHK_ARRAYROWSPARSE || A->storage == SHK_ROWSYMSPARSE,
              SHK_ERR_ARG, "sor: unknown storage");
    SHK_CHECK(omega_type == SHK_F64 || omega_type == SHK_F32, SHK_ERR_ARG, "sor: bad omega type");
    SHK_CHECK(A->m == A->n, SHK_ERR_DIM, "sor: the matrix must be square");
    SHK_CHECK(iter >= 0, SHK_ERR_ARG, "sor: negative iteration count");
    if (A->m == 0 || iter == 0 || (type_ssor % 2 != 0 && type_ssor % 3 != 0)) return SHK_OK;
    SHK_TRY(check_device_ptr(dx, "x"));
    SHK_TRY(check_device_ptr(db, "b"));
    if (!A->sor) {
        SorPlan *P = nullptr;
        SHK_TRY(A->dtype == SHK_F64 ? sor_build<double>(A, &P) : sor_build<float>(A, &P));
        A->sor = P;
    }
    SorPlan *P = A->sor;
    if (A->dtype == SHK_F64)
        return sor_run<double, double>(ctx, P, (double *)dx, (const double *)db, omega, iter, type_ssor);
    if (omega_type == SHK_F64)
        return sor_run<float, double>(ctx, P, (float *)dx, (const float *)db, omega, iter, type_ssor);
    return sor_run<float, float>(ctx, P, (float *)dx, (const float *)db, (float)omega, iter, type_ssor);
}

}  // extern "C"
