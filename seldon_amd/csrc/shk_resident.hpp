// shk_resident.hpp -- Cg with the whole system held on chip.
//
// A Cg iteration on a system of some 10^4 .. 10^6 rows moves little data but
// has two sums that every row waits for; as separate kernels each costs a
// launch and a cold start, and every vector goes through memory again.  Here a
// team of work-groups holds the system for the whole solve: a member owns a
// contiguous run of rows, keeps their matrix values (diagonal-slice form,
// shk_dia.hpp), x and r in registers and p in LDS, and meets the others
// only in the two sums.
//
// p of the other members' rows ("halo": the columns the band reaches past the
// member's rows) is not fetched: a member keeps its own copy of it in its LDS
// window and applies the same p = beta p + z there, with the z its owner
// published before the sum that gave beta.  So an iteration has exactly two
// exchanges: (p, q), and |r|^2 [with (r, z)] together with the halo's z.
//
// Everything exchanged is written as 64-bit words {epoch, 32 bits of the
// value}, each valid by itself, stored and loaded as relaxed device-scope
// atomics: a reader polls the word until it holds the epoch it waits for.
// No fence, no cache write-back or invalidation, no flag to order after the
// data.  (A counter barrier with device-scope release and acquire cost
// 25 us per iteration on the 256^2 Laplacian, more than the launches it
// replaced; this exchange measures 1.2 us over 8 work-groups, 1.9 over 32,
// 2.2 over 64, 3.7 over 256.)  A word is rewritten only after a sum that its
// readers entered after reading it, so one z word per row and two
// alternating sets of sum words are enough.
//
// Each row's sums and updates are Seldon's (Cg.cxx:45-116) operation for
// operation; sums over rows go lane, wave, work-group, member in a fixed
// order.  Every wait is bounded by the wall clock: a wait that runs out sets
// *stall, every member leaves, and the caller solves another way.
//
// What bounds it is latency: the two exchanges, the two divisions and the
// square root behind them, and, on 3-D grids, the halo (two planes per
// member).  Cg per iteration, launched kernels -> this (FP64): 2-D Laplacian
// 64^2 16 -> 4.0 us, 256^2 16.2 -> 4.0, 512^2 20 -> 5.5, 1000^2 35 -> 10; 3-D
// diffusion with Jacobi 40^3 22 -> 7.4, 64^3 26 -> 13.2, 78^3 34 -> 19.7.
#pragma once

#include "shk_kernels.hpp"

namespace shk {

typedef unsigned long long ll_word;

template <typename T>
constexpr int ll_words() { return (int)sizeof(T) / 4; }

// Raw buffer accesses at device scope (sc1, bit 4 of the cache policy): a
// double's two words go as one 16-byte access, which asks the memory side
// once where two 8-byte loads of neighbouring words would ask twice.
constexpr int kLlAux = 16;
typedef unsigned ll_u4 __attribute__((ext_vector_type(4)));
typedef unsigned ll_u2 __attribute__((ext_vector_type(2)));

struct LlBuf {
    template <typename T>
    using Raw = typename std::conditional<sizeof(T) == 8, ll_u4, ll_u2>::type;
    __amdgpu_buffer_rsrc_t rsrc;
    __device__ __forceinline__ LlBuf(ll_word *base, int64_t words)
        : rsrc(__builtin_amdgcn_make_buffer_rsrc(base, (short)0, (int)(words * 8), 0x00020000))
    {
    }
    // a value's words as they stand, and the value they hold (false: not of
    // this epoch)
    template <typename T>
    __device__ __forceinline__ Raw<T> read(int64_t w) const
    {
        if constexpr (sizeof(T) == 8) return __builtin_amdgcn_raw_buffer_load_b128(rsrc, (int)w * 8, 0, kLlAux);
        else return __builtin_amdgcn_raw_buffer_load_b64(rsrc, (int)w * 8, 0, kLlAux);
    }
    static __device__ __forceinline__ bool value(const ll_u4 &q, double &v, unsigned epoch)
    {
        v = __builtin_bit_cast(double, (uint64_t)q[0] | ((uint64_t)q[2] << 32));
        return (q[1] == epoch) & (q[3] == epoch);
    }
    static __device__ __forceinline__ bool value(const ll_u2 &q, float &v, unsigned epoch)
    {
        v = __builtin_bit_cast(float, q[0]);
        return q[1] == epoch;
    }
};

// word index w of the buffer (of a double's first word)
__device__ __forceinline__ void ll_put(const LlBuf &b, int64_t w, double v, unsigned epoch)
{
    const uint64_t bits = __builtin_bit_cast(uint64_t, v);
    const ll_u4 q = {(unsigned)bits, epoch, (unsigned)(bits >> 32), epoch};
    __builtin_amdgcn_raw_buffer_store_b128(q, b.rsrc, (int)w * 8, 0, kLlAux);
}
__device__ __forceinline__ void ll_put(const LlBuf &b, int64_t w, float v, unsigned epoch)
{
    const ll_u2 q = {__builtin_bit_cast(unsigned, v), epoch};
    __builtin_amdgcn_raw_buffer_store_b64(q, b.rsrc, (int)w * 8, 0, kLlAux);
}
// The same words past a buffer's 2 GiB: 8-byte atomics on 64-bit addresses.
struct LlPtr {
    ll_word *p;
    __device__ __forceinline__ LlPtr(ll_word *base, int64_t) : p(base) {}
    __device__ __forceinline__ void store(int64_t w, unsigned v, unsigned epoch) const
    {
        __hip_atomic_store(p + w, (ll_word)epoch << 32 | v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    template <typename T>
    struct Raw {
        ll_word q[ll_words<T>()];
    };
    template <typename T>
    __device__ __forceinline__ Raw<T> read(int64_t w) const
    {
        Raw<T> r;
#pragma unroll
        for (int i = 0; i < ll_words<T>(); i++)
            r.q[i] = __hip_atomic_load(p + w + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return r;
    }
    static __device__ __forceinline__ bool value(const Raw<double> &r, double &v, unsigned epoch)
    {
        v = __builtin_bit_cast(double, (r.q[0] & 0xffffffffull) | (r.q[1] << 32));
        return ((unsigned)(r.q[0] >> 32) == epoch) & ((unsigned)(r.q[1] >> 32) == epoch);
    }
    static __device__ __forceinline__ bool value(const Raw<float> &r, float &v, unsigned epoch)
    {
        v = __builtin_bit_cast(float, (unsigned)r.q[0]);
        return (unsigned)(r.q[0] >> 32) == epoch;
    }
};
__device__ __forceinline__ void ll_put(const LlPtr &b, int64_t w, double v, unsigned epoch)
{
    const uint64_t bits = __builtin_bit_cast(uint64_t, v);
    b.store(w, (unsigned)bits, epoch);
    b.store(w + 1, (unsigned)(bits >> 32), epoch);
}
__device__ __forceinline__ void ll_put(const LlPtr &b, int64_t w, float v, unsigned epoch)
{
    b.store(w, __builtin_bit_cast(unsigned, v), epoch);
}
template <class Words, typename T>
__device__ __forceinline__ bool ll_get(const Words &b, int64_t w, T &v, unsigned epoch)
{
    return Words::value(b.template read<T>(w), v, epoch);
}

// Sum over each 16-lane row, in every lane, by DPP (no LDS round trip).
template <int CTRL>
__device__ __forceinline__ float dpp_move(float v)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), CTRL, 0xf, 0xf, true));
}
template <int CTRL>
__device__ __forceinline__ double dpp_move(double v)
{
    const uint64_t b = __builtin_bit_cast(uint64_t, v);
    const unsigned lo = (unsigned)__builtin_amdgcn_mov_dpp((int)(unsigned)b, CTRL, 0xf, 0xf, true);
    const unsigned hi = (unsigned)__builtin_amdgcn_mov_dpp((int)(unsigned)(b >> 32), CTRL, 0xf, 0xf, true);
    return __builtin_bit_cast(double, (uint64_t)lo | ((uint64_t)hi << 32));
}
template <typename T>
__device__ __forceinline__ T row16_sum(T v)
{
    v += dpp_move<0xB1>(v);   // quad_perm [1,0,3,2]
    v += dpp_move<0x4E>(v);   // quad_perm [2,3,0,1]
    v += dpp_move<0x141>(v);  // row_half_mirror
    v += dpp_move<0x140>(v);  // row_mirror
    return v;
}
__device__ __forceinline__ float lane_value(float v, int lane)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), lane));
}
__device__ __forceinline__ double lane_value(double v, int lane)
{
    const uint64_t b = __builtin_bit_cast(uint64_t, v);
    const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)b, lane);
    const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(b >> 32), lane);
    return __builtin_bit_cast(double, (uint64_t)lo | ((uint64_t)hi << 32));
}
// the wave's sum, the same in every lane
template <typename T>
__device__ __forceinline__ T wave_total(T v)
{
    v = row16_sum(v);
    return (lane_value(v, 0) + lane_value(v, 16)) + (lane_value(v, 32) + lane_value(v, 48));
}

constexpr int kResMaxTeam = 256;   // members, one polling lane each
template <typename T>
constexpr int res_slot_words() { return 2 * ll_words<T>(); }  // two sums

struct ResTeam {
    int k, j;             // members, this one
    LlBuf slot;           // [2][k][res_slot_words]
    unsigned epoch;       // of the last sum posted (0: none)
    unsigned *stall;
    long long limit;      // wall-clock ticks a wait may take
    unsigned every;       // looks between two at the clock, less one (2^k - 1)
};
__host__ __device__ constexpr unsigned res_every(long long limit) { return limit > 0 ? 63u : 0u; }

// Work-group scratch of the sums.
template <typename T>
struct ResShared {
    T wave[2][2][16];     // [phase][value][wave]
    T part[2][4];         // [value][polling wave]
    int bad;              // a wait of this work-group ran out
};

// A bounded wait: false when the time is up (after the first look with a limit
// of 0) or another member gave up.
template <class Ready>
__device__ __forceinline__ bool res_poll(const ResTeam &t, Ready ready)
{
    asm volatile("" ::: "memory");  // no word read before this call
    if (ready()) return true;
    const long long t0 = wall_clock64();
    for (unsigned n = 0;; n++) {
        asm volatile("" ::: "memory");  // the words are read again
        if (ready()) return true;
        if ((n & t.every) == t.every) {
            if (__hip_atomic_load(t.stall, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) return false;
            if (wall_clock64() - t0 >= t.limit) {
                __hip_atomic_store(t.stall, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                return false;
            }
        }
    }
}

// The sum of v over the team's threads, in two halves: post publishes this
// member's share, wait gives every thread the total (and, across both, orders
// LDS as a barrier does).  Between them the caller may wait for other words.
template <typename T, int NV, int NT>
__device__ __forceinline__ void res_post(const T (&v)[NV], ResTeam &t, ResShared<T> &sh)
{
    constexpr int NW = NT / kWave;
    const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
    const unsigned ph = ++t.epoch & 1u;
#pragma unroll
    for (int i = 0; i < NV; i++) {
        const T s = wave_total(v[i]);
        if (lane == 0) sh.wave[ph][i][w] = s;
    }
    __syncthreads();
    if (t.k > 1 && w == 0) {
        const int mine = (int)(ph * t.k + t.j) * res_slot_words<T>();
#pragma unroll
        for (int i = 0; i < NV; i++) {
            const T s = row16_sum((lane & 15) < NW ? sh.wave[ph][i][lane & 15] : (T)0);
            if (lane == 0) ll_put(t.slot, mine + i * ll_words<T>(), s, t.epoch);
        }
    }
}

template <typename T, int NV, int NT>
__device__ __forceinline__ bool res_wait(T (&v)[NV], ResTeam &t, ResShared<T> &sh)
{
    constexpr int NW = NT / kWave;
    const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
    const unsigned ph = t.epoch & 1u;
    if (t.k == 1) {
#pragma unroll
        for (int i = 0; i < NV; i++) v[i] = row16_sum((lane & 15) < NW ? sh.wave[ph][i][lane & 15] : (T)0);
        return true;
    }
    const int npoll = (t.k + kWave - 1) / kWave;  // polling waves
    if (w < npoll) {
        const int q = w * kWave + lane;
        T s[NV];
#pragma unroll
        for (int i = 0; i < NV; i++) s[i] = (T)0;
        if (q < t.k) {
            const int from = (int)(ph * t.k + q) * res_slot_words<T>();
            const bool ok = res_poll(t, [&]() {
                LlBuf::Raw<T> raw[NV];
#pragma unroll
                for (int i = 0; i < NV; i++) raw[i] = t.slot.template read<T>(from + i * ll_words<T>());
                bool all = true;
#pragma unroll
                for (int i = 0; i < NV; i++) all &= LlBuf::value(raw[i], s[i], t.epoch);
                return all;
            });
            if (!ok) sh.bad = 1;
        }
#pragma unroll
        for (int i = 0; i < NV; i++) {
            const T p = wave_total(s[i]);
            if (lane == 0) sh.part[i][w] = p;
        }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NV; i++) {
        T s = sh.part[i][0];
        for (int q = 1; q < npoll; q++) s += sh.part[i][q];
        v[i] = s;
    }
    return sh.bad == 0;
}

// One member's part of a system.  Rows are absolute (indices into x, r, d and
// z); slices of 64 rows count from the system's first row.
struct ResRows {
    int r0, r1;           // the system
    int m0, m1;           // this member's rows (m0 - r0 a multiple of 64)
    int lo, hi;           // its window: [m0 - left band, m1 + right band) within the system
    int left, right;      // the band: largest row - col and col - row
    int slice0;           // diagonal-slice index of row m0
    int steps, stride;    // steps in use, steps stored per slice
    const DiaStep *step;
};

__device__ __forceinline__ void res_window(ResRows &R)
{
    R.lo = max(R.r0, R.m0 - R.left);
    R.hi = min(R.r1, R.m1 + R.right);
}

// What the solve starts from and how it ended.
template <typename T>
struct ResIter {
    double facteur, tol;
    int max_iter;
    int nb;               // iterations done
    int code;             // breakdown (0: none)
    T rho;                // (r, z) at the start
    T rho_1;              // (r, z) of the iteration that head ended the loop after
    const T *p;           // p to carry on from, by row
};

// halo elements per thread fetched while the sum before them is on its way
// (all of a 2-D grid's); the rest follow it (4 and 8 ahead, 8 and 16 in
// flight: within 3% of this on the 64^3 grid, whose halo is two planes)
constexpr int kResAhead = 2;
constexpr int kResBatch = 4;  // of those, in flight together

// The loop of Cg.cxx:72-113 from r = b - A x, x, after the first Finished(r)
// (which did not end it).  x[u], r[u] hold row m0 + (u NW + wave) 64 + lane.
// Returns false when a wait ran out.  `head(nb, |r|^2)` runs after every
// iteration on each thread alike and says whether Finished(r) ends the solve.
// LONG: with it.nb > 0 the loop goes on where another launch's head ended it,
// from that x, r, p and it.
template <typename T, int NT, int RPT, int KS, bool JAC, bool LONG, class Head>
__device__ __forceinline__ bool res_cg(const ResRows &R, const T *val, const T *diag, T (&x)[RPT], T (&r)[RPT],
                                       const LlBuf &zw, T *win, ResIter<T> &it, ResTeam &t, ResShared<T> &sh,
                                       unsigned &zepoch, Head head)
{
    constexpr int NW = NT / kWave;
    const int tid = threadIdx.x, lane = tid & (kWave - 1);
    const int w = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int nsl = (R.m1 - R.m0 + kWave - 1) / kWave;
    const uint64_t bit = 1ull << lane;
    // Values, and each entry's window index (16 bits, two to a register).  A
    // row without an entry at a step reads the window's spare element, which
    // is 0, with a value of 0: adding that +0 leaves every sum as it was,
    // since a sum of -0 becomes the +0 of `0 + temp` at the row's end anyway.
    // (Masks and offsets read from memory in the loop cost 8 us per iteration
    // at 8 rows per thread: scalar loads share their counter with LDS reads.)
    constexpr int KP = (KS + 1) / 2;
    const int spare = R.hi - R.lo;
    T a[RPT][KS];
    unsigned at[RPT][KP];
#pragma unroll
    for (int u = 0; u < RPT; u++) {
        const int sl = u * NW + w;
        const bool live = sl < nsl;
        const size_t s0 = (size_t)(R.slice0 + (live ? sl : 0)) * R.stride;
        const int own = R.m0 + sl * kWave + lane - R.lo;
#pragma unroll
        for (int k = 0; k < KP; k++) at[u][k] = 0u;
#pragma unroll
        for (int k = 0; k < KS; k++) {
            const bool have = live && k < R.steps;
            const DiaStep q = R.step[s0 + (have ? k : 0)];
            const bool act = have && (q.mask & bit);
            a[u][k] = act ? val[(s0 + (have ? k : 0)) * kWave + lane] : (T)0;
            at[u][k / 2] |= (unsigned)(act ? own + q.off : spare) << (16 * (k & 1));
        }
    }
    if (tid == 0) win[spare] = (T)0;
    const int nleft = R.m0 - R.lo, nhalo = nleft + (R.hi - R.m1);
    // row of halo element h (the window minus the member's own rows)
    auto halo_row = [&](int h) { return h < nleft ? R.lo + h : R.m1 + (h - nleft); };
    // z of the rows another member's window reaches
    auto publish = [&](int row, T z) {
        if (t.k > 1 && (row >= R.m1 - R.left || row < R.m0 + R.right)) ll_put(zw, row * ll_words<T>(), z, zepoch);
    };
    T rho = it.rho, rho_1 = (T)1, beta = (T)0, z[RPT];
    const bool carried = LONG && it.nb > 0;
    if (LONG && carried) {
        for (int i = tid; i < R.hi - R.lo; i += NT) win[i] = it.p[R.lo + i];
    }
    zepoch++;
#pragma unroll
    for (int u = 0; u < RPT; u++) {
        const int row = R.m0 + (u * NW + w) * kWave + lane;
        z[u] = JAC && row < R.m1 ? r[u] / diag[row] : r[u];
        if (row < R.m1) publish(row, z[u]);
    }
    bool ok = true;
    // N halo values from element h0 on: every word is on its way before the
    // first is looked at (checked one by one, the loads took turns: 64^3 15.6
    // instead of 13.2 us per iteration); lanes past the halo's end poll its
    // last element
    auto fetch = [&](auto &zh, int h0) {
        constexpr int N = sizeof(zh) / sizeof(T);
        if (h0 >= nhalo) return;
        const bool got = res_poll(t, [&]() {
            LlBuf::Raw<T> raw[N];
#pragma unroll
            for (int q = 0; q < N; q++)
                if (h0 + q * NT < nhalo) {
                    const int h = min(h0 + q * NT + tid, nhalo - 1);
                    raw[q] = zw.template read<T>(halo_row(h) * ll_words<T>());
                }
            bool all = true;
#pragma unroll
            for (int q = 0; q < N; q++)
                if (h0 + q * NT < nhalo) all &= LlBuf::value(raw[q], zh[q], zepoch);
            return all;
        });
        if (!got) sh.bad = 1;
    };
    // First ? p = z : { p *= beta; p += 1 * z } for N halo elements from h0 on
    auto advance = [&](const auto &zh, int h0, bool first) {
        constexpr int N = sizeof(zh) / sizeof(T);
#pragma unroll
        for (int q = 0; q < N; q++) {
            const int h = h0 + q * NT + tid;
            if (h < nhalo) {
                const int i = halo_row(h) - R.lo;
                T v = zh[q];
                if (!first) {
                    v = win[i] * beta;
                    v += (T)1 * zh[q];
                }
                win[i] = v;
            }
        }
    };
    T za[kResAhead];
#pragma unroll
    for (int q = 0; q < kResAhead; q++) za[q] = (T)0;
    if (JAC || (LONG && carried)) {  // rho = (r, z), summed as below
        T c[1] = {(T)0};
#pragma unroll
        for (int u = 0; u < RPT; u++) c[0] += r[u] * z[u];
        res_post<T, 1, NT>(c, t, sh);
        fetch(za, 0);
        ok = res_wait<T, 1, NT>(c, t, sh);
        rho = c[0];
        if (rho == (T)0) {
            it.code = 1;
            return ok;
        }
        if (LONG && carried) beta = rho / it.rho_1;
    } else {
        fetch(za, 0);
    }
    for (;;) {
        // First ? p = z : { p *= beta; p += 1 * z }, own rows and halo
        const bool first = it.nb == 0;
#pragma unroll
        for (int u = 0; u < RPT; u++) {
            const int row = R.m0 + (u * NW + w) * kWave + lane;
            if (row < R.m1) {
                T v = z[u];
                if (!first) {
                    v = win[row - R.lo] * beta;
                    v += (T)1 * z[u];
                }
                win[row - R.lo] = v;
            }
        }
        advance(za, 0, first);
        for (int h0 = kResAhead * NT; h0 < nhalo; h0 += kResBatch * NT) {
            T zb[kResBatch];
#pragma unroll
            for (int q = 0; q < kResBatch; q++) zb[q] = (T)0;
            fetch(zb, h0);
            advance(zb, h0, first);
        }
        __syncthreads();
        if (sh.bad) return false;
        // q = A p, (p, q)
        T c[1] = {(T)0}, qv[RPT];
#pragma unroll
        for (int u = 0; u < RPT; u++) {
            const int sl = u * NW + w;
            qv[u] = (T)0;
            if (sl < nsl) {
                const int row = R.m0 + sl * kWave + lane;
                T pv[KS];
#pragma unroll
                for (int k = 0; k < KS; k++) pv[k] = win[(at[u][k / 2] >> (16 * (k & 1))) & 0xffffu];
                const T own = win[row < R.m1 ? row - R.lo : spare];
                T acc = (T)0;
#pragma unroll
                for (int k = 0; k < KS; k++) acc += a[u][k] * pv[k];
                qv[u] = (T)0 + acc;  // Mlt: 0 + 1 * temp
                c[0] += own * qv[u];
            }
        }
        res_post<T, 1, NT>(c, t, sh);
        ok = res_wait<T, 1, NT>(c, t, sh);
        if (!ok) return false;
        if (c[0] == (T)0) {
            it.code = 2;
            return true;
        }
        const T alpha = rho / c[0], malpha = -alpha;
        T s[2] = {(T)0, (T)0};
        zepoch++;
#pragma unroll
        for (int u = 0; u < RPT; u++) {
            const int row = R.m0 + (u * NW + w) * kWave + lane;
            if (row < R.m1) {
                if (alpha != (T)0) x[u] += alpha * win[row - R.lo];
                if (malpha != (T)0) r[u] += malpha * qv[u];
                z[u] = JAC ? r[u] / diag[row] : r[u];
                publish(row, z[u]);
                s[0] += r[u] * r[u];
                if (JAC) s[1] += r[u] * z[u];
            }
        }
        constexpr int NV = JAC ? 2 : 1;
        T tot[NV];
        tot[0] = s[0];
        if (JAC) tot[NV - 1] = s[1];
        res_post<T, NV, NT>(tot, t, sh);
        fetch(za, 0);
        ok = res_wait<T, NV, NT>(tot, t, sh);
        if (!ok) return false;
        rho_1 = rho;
        it.nb++;
        if (head(it.nb, tot[0])) {
            if (LONG) it.rho_1 = rho_1;
            return true;
        }
        rho = tot[NV - 1];
        if (rho == (T)0) {
            it.code = 1;
            return true;
        }
        beta = rho / rho_1;
    }
}

}  // namespace shk
