// One workgroup per system: factorisation, solves and whole Newton steps of
// systems whose factors fit one workgroup's LDS (plan: sys_plan.hpp).
//
// A small grid is bound by latency, not by arithmetic or memory: the level
// sweeps of the batched kernels launch some 45 kernels per Newton step, each
// 4 to 25 us long for a few microseconds' chain of dependent loads.  Here a
// scenario's network state, Jacobian, factors and solution stay in LDS for
// the whole step, so one launch does it and global memory sees the state
// once.  A front of at most 16 rows takes 16 lanes (a row per lane in
// registers, pivot rows broadcast by DPP), four fronts to a wave; a front of at
// most 32 rows takes a wave, and larger ones, or a level of one or two, the
// whole workgroup, the front's elements in registers and the pivot row and
// column passed through LDS.
//
// What bounds it is latency: on 118 buses FP64 a Newton step takes 72 us, 30 of
// them the 43 pivots of the shared fronts one after another (0.7 us each, with
// one barrier and, per thread, the update of 8 elements), 13 the levels of quads
// and wave fronts, 20 the solve, 4.5 the residual and stop test (a wave alone on
// its SIMD issues an instruction about every 9 cycles).  Solves: 118 buses x1
// FP64 1.92 -> 0.41 ms (captured mixed 1.67 -> 0.34), x300 mixed 2.73 -> 0.50,
// x1,024 FP64 3.14 -> 1.44.
#include "sys_kernels.hpp"
#include "hip_common.hpp"

#include <algorithm>
#include <type_traits>

namespace cupf::kern {
namespace {

constexpr unsigned long long kNanBits = 0x7FF8000000000000ULL;

// The pivot rule of the batched kernels without branches: |pivot| <= low
// becomes +-rep and raises the flag (static pivots: both are eps; else a zero
// pivot becomes 1).
template <typename T>
struct PivotRule {
    T low, rep;
    bool sign;
    __device__ __forceinline__ PivotRule(double eps, int static_piv)
        : low(static_piv ? T(eps) : T(0)), rep(static_piv ? T(eps) : T(1)), sign(static_piv != 0) {}
    __device__ __forceinline__ bool small(T piv) const { return (piv < T(0) ? -piv : piv) <= low; }
    __device__ __forceinline__ T replaced(T piv) const { return sign && piv < T(0) ? -rep : rep; }
};

// 1 / d by Newton's iteration from the hardware estimate, within an ulp where it
// is a normal number, else something that is not.
__device__ __forceinline__ double reciprocal(double d) {
    double r = __builtin_amdgcn_rcp(d);
    r = __builtin_fma(__builtin_fma(-d, r, 1.0), r, r);
    return __builtin_fma(__builtin_fma(-d, r, 1.0), r, r);
}
__device__ __forceinline__ float reciprocal(float d) {
    const float r = __builtin_amdgcn_rcpf(d);
    return __builtin_fmaf(__builtin_fmaf(-d, r, 1.f), r, r);
}

// a / d from r = 1 / d: the product and one residual correction, which round
// as the division does (no difference in 10^8 pairs of either type) at a
// quarter of its latency.  No number where r is none, a is infinite or the
// quotient overflows: a factorisation looks at its reciprocals, a solve at its
// results, and both start again by division then (factor_matrix, solve_system).
__device__ __forceinline__ double quotient(double a, double d, double r) {
    const double q = a * r;
    return __builtin_fma(__builtin_fma(-d, q, a), r, q);
}
__device__ __forceinline__ float quotient(float a, float d, float r) {
    const float q = a * r;
    return __builtin_fmaf(__builtin_fmaf(-d, q, a), r, q);
}
template <bool EXACT, typename T>
__device__ __forceinline__ T over(T a, T d, T r) {
    return EXACT ? a / d : quotient(a, d, r);
}

__device__ __forceinline__ double nfma(double a, double b, double c) { return __builtin_fma(-a, b, c); }
__device__ __forceinline__ float nfma(float a, float b, float c) { return __builtin_fmaf(-a, b, c); }
__device__ __forceinline__ double mul_add(double a, double b, double c) { return __builtin_fma(b, a, c); }
__device__ __forceinline__ float mul_add(float a, float b, float c) { return __builtin_fmaf(b, a, c); }

// lane `k`'s value (k uniform)
__device__ __forceinline__ float lane_value(float x, int k) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), k));
}
__device__ __forceinline__ double lane_value(double x, int k) {
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(x), k),
                            __builtin_amdgcn_readlane(__double2loint(x), k));
}
// lane K's value of each group of 16 lanes (row_newbcast)
template <int K>
__device__ __forceinline__ float row_value(float x) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0x150 + K, 0xf, 0xf, true));
}
template <int K>
__device__ __forceinline__ double row_value(double x) {
    const long long v = __double_as_longlong(x);
    return __longlong_as_double(__builtin_amdgcn_update_dpp(v, v, 0x150 + K, 0xf, 0xf, true));
}

// Orders a wave's LDS accesses (performed in order by the hardware) for the
// compiler.
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Pivot row and column buffers: a share for each of eight waves, or all of
// them for a shared front.
constexpr int kWaveBuf = 128, kSysBuf = 8 * kWaveBuf;
constexpr int kSysMark = 4;           // elements of Sys::mark (16 or 32 bytes)

// The tables and arrays of one system in LDS.  `a` holds the factors at 0 and
// the scratch region (contribution blocks, then work vectors) at scr.
template <typename T>
struct Sys {
    T* a;
    T* dinv;
    T* y;
    T* buf;                           // the front teams' pivot rows and columns
    int* mark;                        // see any_thread()
    int scr;
    const SysFront* front;
    const int* level;
    const int* slice;
    const unsigned short* list;       // the whole blob as u16
    const unsigned short* adds;       // global
    int o_task, o_rows, o_gptr, o_gsrc, o_perm;
    int num_levels;
};

// A front's sizes and the offsets of its parts in Sys::a.
struct Front {
    int fs, K, uc, us, ls, fo, lo, co, wo, first, rows, gptr, slice0, slices;
    // element (i, j) while the front is being factored
    __device__ __forceinline__ int at(int i, int j) const {
        const int below = j < K ? lo + (i - K) * ls + j : co + (i - K) * uc + (j - K);
        return i < K ? fo + i * us + j : below;
    }
    // row i's first element among the pivot columns
    __device__ __forceinline__ int row(int i) const { return i < K ? fo + i * us : lo + (i - K) * ls; }
};

template <typename T>
__device__ __forceinline__ Front load_front(const Sys<T>& S, int p) {
    const SysFront f = S.front[p];
    Front o;
    o.fs = f.size & 0xffff;
    o.K = f.size >> 16;
    o.uc = o.fs - o.K;
    o.us = o.fs | 1;
    o.ls = o.K | 1;
    o.fo = f.fo;
    o.lo = f.fo + o.K * o.us;
    o.co = S.scr + f.co;
    o.wo = S.scr + f.wo;
    o.first = f.first;
    o.rows = S.o_rows + f.rows;
    o.gptr = S.o_gptr + f.rows;
    o.slice0 = f.slice0;
    o.slices = f.slices;
    return o;
}

// Adds the children's contribution blocks into front f: 16-lane group g of
// `groups` takes every groups-th slice, a destination per lane; four slices'
// list entries are in flight together (they come from L2).
template <typename T>
__device__ __forceinline__ void add_children(const Sys<T>& S, const Front& f, int g, int groups) {
    const int r = int(threadIdx.x) & 15;
    for (int q0 = g; q0 < f.slices; q0 += 4 * groups) {
        unsigned w[4];
        const unsigned short* list[4];
        int dst[4], s0[4], s1[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            w[u] = unsigned(S.slice[f.slice0 + min(q0 + u * groups, f.slices - 1)]);
            list[u] = S.adds + (w[u] & ((1u << kSysSliceShift) - 1)) * 16 + r;
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            dst[u] = list[u][0];
            s0[u] = list[u][16];
            s1[u] = list[u][32];                                // the list ends with a spare row
        }
        T v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) v[u] = S.a[dst[u]];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int width = int(w[u] >> kSysSliceShift);
            const T x0 = S.a[s0[u]];
            const T x1 = S.a[width > 1 ? s1[u] : s0[u]];
            v[u] += x0;
            v[u] += width > 1 ? x1 : T(0);
            for (int k = 2; k < width; ++k) v[u] += S.a[list[u][16 * (1 + k)]];
        }
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (q0 + u * groups < f.slices) S.a[dst[u]] = v[u];
    }
}

// Compile-time pivot steps k0 .. 15 (the DPP broadcasts take the lane as an
// immediate).
template <int K0, int K1, class F>
__device__ __forceinline__ void each(F f) {
    if constexpr (K0 < K1) {
        f(std::integral_constant<int, K0>{});
        each<K0 + 1, K1>(f);
    }
}
template <int K0, class F>
__device__ __forceinline__ void each_down(F f) {
    if constexpr (K0 >= 0) {
        f(std::integral_constant<int, K0>{});
        each_down<K0 - 1>(f);
    }
}

// LU steps on 16-lane groups, row r = lane of the group, x its row: K pivots
// (kmax, uniform: the most of the wave's groups).  Leaves 1 / pivot r in rinv.
// Four steps run straight through, so the next pivot's reciprocal chain
// overlaps the column updates; steps past K change nothing.  A replaced pivot
// leaves the chain through a branch that is hardly ever taken.
template <int k, typename T>
__device__ __forceinline__ void eliminate_step(T (&x)[16], int r, int K, const PivotRule<T>& rule, int& flag,
                                               T& rinv) {
    const bool on = k < K, below = on && r > k;
    const T raw = row_value<k>(x[k]);
    T piv = on ? raw : T(1);
    if (__builtin_expect(__any(on && rule.small(raw)), 0)) {
        const bool low = on && rule.small(raw);
        flag |= low;
        piv = low ? rule.replaced(raw) : piv;
        x[k] = low && r == k ? piv : x[k];
    }
    const T ri = reciprocal(piv);
    rinv = r == k ? ri : rinv;
    const T l = quotient(below ? x[k] : T(0), piv, ri);
    x[k] = below ? l : x[k];
    const T nl = -l;
#pragma unroll
    for (int j = k + 1; j < 16; ++j) x[j] = mul_add(nl, row_value<k>(x[j]), x[j]);
}

template <int k0, typename T>
__device__ __forceinline__ void eliminate16(T (&x)[16], int r, int K, int kmax,
                                            const PivotRule<T>& rule, int& flag, T& rinv) {
    if constexpr (k0 < 16) {
        if (k0 < kmax) {                                        // uniform
            eliminate_step<k0>(x, r, K, rule, flag, rinv);
            eliminate_step<k0 + 1>(x, r, K, rule, flag, rinv);
            eliminate_step<k0 + 2>(x, r, K, rule, flag, rinv);
            eliminate_step<k0 + 3>(x, r, K, rule, flag, rinv);
            eliminate16<k0 + 4>(x, r, K, kmax, rule, flag, rinv);
        }
    }
}

// largest value over the four 16-lane groups (each uniform in its group)
__device__ __forceinline__ int over_groups(int v) {
    return max(max(__builtin_amdgcn_readlane(v, 0), __builtin_amdgcn_readlane(v, 16)),
               max(__builtin_amdgcn_readlane(v, 32), __builtin_amdgcn_readlane(v, 48)));
}

// Four fronts of at most 16 rows, one per 16 lanes: contribution blocks added
// in LDS, the rows factored in registers.
template <typename T>
__device__ __forceinline__ void factor_quad(const Sys<T>& S, const unsigned short* ids,
                                            const PivotRule<T>& rule, int& flag) {
    const int lane = int(threadIdx.x) & 63, r = lane & 15;
    const int p = ids[lane >> 4];
    const bool have = p != 0xffff;
    const Front f = load_front(S, have ? p : int(ids[0]));
    const int fs = have ? f.fs : 0, K = have ? f.K : 0;
    if (have) {
        for (int e = r; e < f.uc * f.uc; e += 16) S.a[f.co + e] = T(0);
        wave_sync();
        add_children(S, f, 0, 1);
    }
    wave_sync();
    const int kmax = over_groups(K);
    const int rr = min(r, f.fs - 1);
    const int lo = f.row(rr), hi = rr < f.K ? f.fo + rr * f.us : f.co + (rr - f.K) * f.uc - f.K;
    T x[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) {
        const int jj = min(j, f.fs - 1);
        const T v = S.a[(jj < f.K ? lo : hi) + jj];
        x[j] = r < fs && j < fs ? v : T(0);
    }
    T rinv = T(1);
    eliminate16<0>(x, r, K, kmax, rule, flag, rinv);
#pragma unroll
    for (int j = 0; j < 16; ++j)
        if (r < fs && j < fs) S.a[(j < f.K ? lo : hi) + j] = x[j];
    if (r < K) S.dinv[f.first + r] = rinv;
}

// One front by a team of TR x TC threads (a wave, or with ALL the whole
// workgroup), thread (ti, tj) holding the elements of rows ti + TR a and
// columns tj + TC b in registers for the whole elimination.  A pivot step
// reads the pivot row and column from the team's buffers, where their owners
// put them at the end of the step before: one synchronisation a pivot, and no
// triangular solves or trailing passes.  Finished rows and columns go to their
// places a thread per position, so the updates need no masks (what they do to
// finished elements is never read).
template <typename T, int RA, int RB, int TR, int TC, bool ALL>
__device__ __forceinline__ void factor_front(const Sys<T>& S, int p, T* buf, const PivotRule<T>& rule, int& flag) {
    constexpr int kRows = TR * RA, kCols = TC * RB;             // buf: [2][kRows + kCols]
    static_assert(2 * (kRows + kCols) <= (ALL ? kSysBuf : kWaveBuf), "the team's buffers");
    const int tid = ALL ? int(threadIdx.x) : int(threadIdx.x) & 63;
    const int ti = tid / TC, tj = tid % TC;
    auto sync = [] {
        if (ALL) __syncthreads();
        else wave_sync();
    };
    const Front f = load_front(S, p);
    for (int e = tid; e < f.uc * f.uc; e += TR * TC) S.a[f.co + e] = T(0);
    sync();
    add_children(S, f, tid >> 4, TR * TC / 16);
    sync();
    T x[RA][RB];
#pragma unroll
    for (int a = 0; a < RA; ++a) {
        const int i = min(ti + TR * a, f.fs - 1);
        const int lo = f.row(i), hi = i < f.K ? lo : f.co + (i - f.K) * f.uc - f.K;
#pragma unroll
        for (int b = 0; b < RB; ++b) {
            const int j = min(tj + TC * b, f.fs - 1);
            x[a][b] = S.a[(j < f.K ? lo : hi) + j];
        }
    }
    const int mine = min(tid, f.fs - 1);
    const int my_row = f.row(mine);
    each<0, RA>([&](auto ac) {                                  // pivots TR a .. TR a + TR - 1
        constexpr int a0 = ac.value, bc = a0 * TR / TC, tc0 = a0 * TR % TC;
        static_assert(TC % TR == 0, "a block of pivots stays in one column register");
        if constexpr (a0 * TR < 64)
            for (int kk = 0; kk < TR && TR * a0 + kk < f.K; ++kk) {
                const int k = TR * a0 + kk;
                T* cb = buf + (kk & 1) * (kRows + kCols);
                T* rb = cb + kRows;
                if (ti == kk) {
#pragma unroll
                    for (int b = 0; b < RB; ++b) rb[tj + TC * b] = x[a0][b];
                }
                if (tj == tc0 + kk) {
#pragma unroll
                    for (int a = 0; a < RA; ++a) cb[ti + TR * a] = x[a][bc];
                }
                sync();
                T piv = rb[k];
                T u[RB], c[RA];
#pragma unroll
                for (int b = 0; b < RB; ++b) u[b] = rb[tj + TC * b];
#pragma unroll
                for (int a = 0; a < RA; ++a) c[a] = cb[ti + TR * a];
                const T my_c = cb[mine], my_u = rb[mine];
                if (__builtin_expect(__any(rule.small(piv)), 0)) {      // the same for all
                    flag = 1;
                    piv = rule.replaced(piv);
                }
                const T r = reciprocal(piv);
                // column / pivot as the column times the reciprocal and its
                // error, one rounding: an instruction a quotient less
                const T rerr = nfma(piv, r, T(1)) * r;
                const T my_l = mul_add(r, my_c, my_c * rerr);
                T l[RA];
#pragma unroll
                for (int a = 0; a < RA; ++a) l[a] = mul_add(r, c[a], c[a] * rerr);
#pragma unroll
                for (int a = 0; a < RA; ++a)
#pragma unroll
                    for (int b = 0; b < RB; ++b) x[a][b] = nfma(l[a], u[b], x[a][b]);
                // position `mine` of the finished row and column
                if (tid >= k && tid < f.fs) {
                    S.a[my_row + k] = tid == k ? piv : my_l;
                    S.a[f.fo + k * f.us + tid] = tid == k ? piv : my_u;
                    if (tid == k) S.dinv[f.first + k] = r;
                }
            }
    });
#pragma unroll
    for (int a = 0; a < RA; ++a) {
        const int i = ti + TR * a;
        const int hi = f.co + (i - f.K) * f.uc - f.K;
#pragma unroll
        for (int b = 0; b < RB; ++b) {
            const int j = tj + TC * b;
            if (i >= f.K && j >= f.K && i < f.fs && j < f.fs) S.a[hi + j] = x[a][b];
        }
    }
    sync();
}

template <typename T, int NT>
__device__ __forceinline__ void factor_system(const Sys<T>& S, double eps, int static_piv, int& flag) {
    const PivotRule<T> rule(eps, static_piv);
    const int wave = int(threadIdx.x) >> 6, waves = int(blockDim.x) >> 6;
    for (int L = 0; L < S.num_levels; ++L) {
        const int* lv = S.level + L * kSysLevelInts;
        const unsigned short* task = S.list + S.o_task + lv[0];
        const int quads = lv[1], fronts = lv[2], shared = lv[3];
        for (int t = wave; t < fronts + quads; t += waves) {
            if (t >= fronts) factor_quad(S, task + fronts + 4 * (t - fronts), rule, flag);
            else factor_front<T, 4, 4, 8, 8, false>(S, task[t], S.buf + wave * kWaveBuf, rule, flag);
        }
        __syncthreads();
        for (int t = 0; t < shared; ++t) {
            const int p = task[fronts + 4 * quads + t];
            if ((S.front[p].size & 0xffff) <= 64) factor_front<T, 4, 64 * 16 / NT, 16, NT / 16, true>(S, p, S.buf, rule, flag);
            else factor_front<T, kSysMaxRows / 16, (kSysMaxRows * 16 + NT - 1) / NT, 16, NT / 16, true>(S, p, S.buf, rule, flag);
        }
    }
}

// One front by one wave, in LDS and by division.
template <typename T>
__device__ __forceinline__ void factor_dividing(const Sys<T>& S, int p, const PivotRule<T>& rule, int& flag) {
    const int lane = int(threadIdx.x) & 63;
    const Front f = load_front(S, p);
    for (int e = lane; e < f.uc * f.uc; e += 64) S.a[f.co + e] = T(0);
    wave_sync();
    add_children(S, f, lane >> 4, 4);
    wave_sync();
    for (int k = 0; k < f.K; ++k) {
        T piv = S.a[f.at(k, k)];
        if (rule.small(piv)) {
            flag = 1;
            piv = rule.replaced(piv);
        }
        wave_sync();
        if (lane == 0) {
            const T r = reciprocal(piv);
            S.a[f.at(k, k)] = piv;
            S.dinv[f.first + k] = __builtin_isnormal(r) ? r : T(__builtin_nanf(""));    // the solves divide
        }
        for (int i = k + 1 + lane; i < f.fs; i += 64) {
            const T l = S.a[f.at(i, k)] / piv;
            S.a[f.at(i, k)] = l;
            for (int j = k + 1; j < f.fs; ++j) S.a[f.at(i, j)] = nfma(l, S.a[f.at(k, j)], S.a[f.at(i, j)]);
        }
        wave_sync();
    }
}

// A pointer into LDS, as the functions below take them: behind a call the
// compiler could not tell the address space otherwise.
template <typename X>
using Lds = __attribute__((address_space(3))) X*;
template <typename X>
__device__ __forceinline__ Lds<X> lds(X* p) {
    return (Lds<X>)p;
}

// All fronts so.  A function of its own, as divide_solve(): inlined, their
// registers and code slow the plain path by 1-4%.
template <typename T>
__device__ __attribute__((noinline)) int divide_factors(Lds<T> a, Lds<T> dinv, int scr, Lds<const int> ints, int o_level,
                                                        int o_slice, const unsigned short* adds, int o_task,
                                                        int num_levels, double eps, int static_piv) {
    Sys<T> S{};
    S.a = (T*)a;
    S.dinv = (T*)dinv;
    S.scr = scr;
    S.front = (const SysFront*)(const int*)ints;
    S.level = (const int*)ints + o_level;
    S.slice = (const int*)ints + o_slice;
    S.list = (const unsigned short*)(const int*)ints;
    S.adds = adds;
    const PivotRule<T> rule(eps, static_piv);
    int flag = 0;
    for (int L = 0; L < num_levels; ++L) {
        const int* lv = S.level + L * kSysLevelInts;
        const unsigned short* task = S.list + o_task + lv[0];
        for (int t = int(threadIdx.x) >> 6; t < lv[2] + 4 * lv[1] + lv[3]; t += int(blockDim.x) >> 6)
            if (task[t] != 0xffff) factor_dividing(S, task[t], rule, flag);
        __syncthreads();
    }
    return flag;
}

template <typename T>
__device__ __forceinline__ int divide_factors(const Sys<T>& S, double eps, int static_piv) {
    const int* ints = reinterpret_cast<const int*>(S.front);
    return divide_factors<T>(lds(S.a), lds(S.dinv), S.scr, lds(ints), int(S.level - ints), int(S.slice - ints), S.adds,
                             S.o_task, S.num_levels, eps, static_piv);
}

// Back to 0 once every thread has read it.
template <typename T>
__device__ __forceinline__ void clear_mark(const Sys<T>& S) {
    __syncthreads();
    if (threadIdx.x == 0) *S.mark = 0;
    __syncthreads();
}

// Whether `yes` holds on any thread of the workgroup (one barrier).  S.mark is 0
// before and after; two calls have a barrier between them.
template <typename T>
__device__ __forceinline__ bool any_thread(const Sys<T>& S, bool yes) {
    if (yes) *S.mark = 1;
    __syncthreads();
    if (__builtin_expect(*S.mark == 0, 1)) return false;
    clear_mark(S);
    return true;
}

// The factors of the matrix that load() puts into the factors' place (it ends
// with a barrier).  A pivot whose reciprocal is no normal number has it all done
// again by division, unless hopeless() finds a NaN among this thread's inputs.
template <typename T, int NT, class F, class G>
__device__ __forceinline__ void factor_matrix(const Sys<T>& S, int n, double eps, int static_piv, int& flag,
                                              F load, G hopeless) {
    load();
    factor_system<T, NT>(S, eps, static_piv, flag);
    bool normal = true;
    for (int k = int(threadIdx.x); k < n; k += NT) normal = normal && __builtin_isnormal(S.dinv[k]);
    if (!any_thread(S, !normal) || any_thread(S, hopeless())) return;
    flag = 0;
    load();
    flag = divide_factors(S, eps, static_piv);
}

// Solve sweeps on y (permuted order).  Fronts of at most 16 rows four to a
// wave, the others a wave each; a row per lane, the solved entries broadcast.

// Position l's right-hand side: its own entry (a pivot's) and the children's
// work-vector elements that land there, in child order.
template <typename T>
__device__ __forceinline__ T gather(const Sys<T>& S, const Front& f, int l) {
    T v = l < f.K ? S.y[f.first + min(l, f.K - 1)] : T(0);
    const int g0 = S.list[f.gptr + l], g1 = S.list[f.gptr + l + 1];
    for (int g = g0; g < g1; g += 4) {
        int at[4];
        T x[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) at[u] = S.list[S.o_gsrc + min(g + u, g1 - 1)];
#pragma unroll
        for (int u = 0; u < 4; ++u) x[u] = S.a[at[u]];
#pragma unroll
        for (int u = 0; u < 4; ++u) v += g + u < g1 ? x[u] : T(0);
    }
    return v;
}

template <bool TRANS, typename T>
__device__ __forceinline__ void forward_quad(const Sys<T>& S, const unsigned short* ids) {
    const int lane = int(threadIdx.x) & 63, r = lane & 15;
    const int p = ids[lane >> 4];
    const bool have = p != 0xffff;
    const Front f = load_front(S, have ? p : int(ids[0]));
    const int K = have ? f.K : 0;
    const int rr = min(r, f.fs - 1), row = f.row(rr);
    T c[16];
#pragma unroll
    for (int k = 0; k < 16; ++k) {
        const int kk = min(k, f.K - 1);
        c[k] = TRANS ? S.a[f.fo + kk * f.us + rr] : S.a[row + kk];
    }
    const int rk = min(r, f.K - 1);
    const T dg = TRANS ? S.a[f.fo + rk * f.us + rk] : T(1), di = TRANS ? S.dinv[f.first + rk] : T(1);
    T z = gather(S, f, rr);
    each<0, 16>([&](auto kc) {
        constexpr int k = kc.value;
        if (TRANS) z = r == k && k < K ? quotient(z, dg, di) : z;   // U11^T: non-unit
        const T zk = row_value<k>(z);
        z = r > k && k < K ? nfma(c[k], zk, z) : z;
    });
    if (have && r < f.fs) {
        if (r < f.K) S.y[f.first + r] = z;
        else S.a[f.wo + r] = z;
    }
}

template <bool TRANS, typename T>
__device__ __forceinline__ void backward_quad(const Sys<T>& S, const unsigned short* ids) {
    const int lane = int(threadIdx.x) & 63, r = lane & 15;
    const int p = ids[lane >> 4];
    const bool have = p != 0xffff;
    const Front f = load_front(S, have ? p : int(ids[0]));
    const int fs = have ? f.fs : 0;
    const int rk = min(r, f.K - 1);
    T c[16];                                                    // row rk of U (row of L^T)
#pragma unroll
    for (int j = 0; j < 16; ++j) {
        const int jj = min(j, f.fs - 1);
        c[j] = TRANS ? S.a[f.row(jj) + rk] : S.a[f.fo + rk * f.us + jj];
    }
    const T dg = TRANS ? T(1) : S.a[f.fo + rk * f.us + rk], di = TRANS ? T(1) : S.dinv[f.first + rk];
    T z = S.y[r < f.K ? f.first + r : int(S.list[f.rows + min(r, f.fs - 1)])];
    each_down<15>([&](auto jc) {
        constexpr int j = jc.value;
        if (!TRANS) z = r == j && j < f.K ? quotient(z, dg, di) : z;        // U11: non-unit
        const T xj = row_value<j>(z);
        z = r < j && r < f.K && j < fs ? nfma(c[j], xj, z) : z;
    });
    if (have && r < f.K) S.y[f.first + r] = z;
}

template <bool TRANS, bool EXACT, typename T>
__device__ __forceinline__ void forward_front(const Sys<T>& S, int p) {
    const int lane = int(threadIdx.x) & 63;
    const Front f = load_front(S, p);
    // the first 64 rows a lane each, the others after the pivots
    const int l0 = min(lane, f.fs - 1), row = f.row(l0);
    T z = gather(S, f, l0);
#pragma unroll (EXACT ? 1 : 8)
    for (int k = 0; k < f.K; ++k) {
        const T c = TRANS ? S.a[f.fo + k * f.us + l0] : S.a[row + k];
        T zk = lane_value(z, k);
        if (TRANS) {                                            // U11^T: non-unit
            zk = over<EXACT>(zk, S.a[f.fo + k * f.us + k], S.dinv[f.first + k]);
            z = lane == k ? zk : z;
        }
        z = lane > k ? nfma(c, zk, z) : z;
    }
    if (lane < f.K) S.y[f.first + lane] = z;
    else if (lane < f.fs) S.a[f.wo + lane] = z;
    if (f.fs > 64) {
        wave_sync();
        for (int l = 64 + lane; l < f.fs; l += 64) {            // K <= 64
            T v = gather(S, f, l);
#pragma unroll (EXACT ? 1 : 4)
            for (int k = 0; k < f.K; ++k)
                v = nfma(TRANS ? S.a[f.fo + k * f.us + l] : S.a[f.lo + (l - f.K) * f.ls + k], S.y[f.first + k], v);
            S.a[f.wo + l] = v;
        }
    }
}

template <bool TRANS, bool EXACT, typename T>
__device__ __forceinline__ void backward_front(const Sys<T>& S, int p) {
    const int lane = int(threadIdx.x) & 63;
    const Front f = load_front(S, p);
    for (int l = f.K + lane; l < f.fs; l += 64) S.a[f.wo + l] = S.y[S.list[f.rows + l]];
    wave_sync();
    const int i = min(lane, f.K - 1);
    T z = S.y[f.first + i];
#pragma unroll (EXACT ? 1 : 8)
    for (int j = f.K; j < f.fs; ++j)
        z = nfma(TRANS ? S.a[f.lo + (j - f.K) * f.ls + i] : S.a[f.fo + i * f.us + j], S.a[f.wo + j], z);
#pragma unroll (EXACT ? 1 : 8)
    for (int k = f.K - 1; k >= 0; --k) {
        const T c = TRANS ? S.a[f.fo + k * f.us + i] : S.a[f.fo + i * f.us + k];
        T xk = lane_value(z, k);
        if (!TRANS) {                                           // U11: non-unit
            xk = over<EXACT>(xk, S.a[f.fo + k * f.us + k], S.dinv[f.first + k]);
            z = lane == k ? xk : z;
        }
        z = lane < k ? nfma(c, xk, z) : z;
    }
    if (lane < f.K) S.y[f.first + lane] = z;
}

// EXACT: pivots by division, every front on a wave.
template <bool TRANS, bool EXACT, typename T>
__device__ __forceinline__ void sweep_system(const Sys<T>& S) {
    const int wave = int(threadIdx.x) >> 6, waves = int(blockDim.x) >> 6;
    for (int s = 0; s < 2 * S.num_levels; ++s) {
        const bool fwd = s < S.num_levels;
        const int* lv = S.level + (fwd ? s : 2 * S.num_levels - 1 - s) * kSysLevelInts;
        const unsigned short* task = S.list + S.o_task + lv[0];
        const int quads = lv[1], fronts = lv[2], shared = lv[3];
        for (int t = wave; t < fronts + quads + shared; t += waves) {
            if (t >= fronts && t < fronts + quads) {
                const unsigned short* ids = task + fronts + 4 * (t - fronts);
                for (int g = 0; EXACT && g < 4 && ids[g] != 0xffff; ++g) {
                    if (fwd) forward_front<TRANS, true>(S, ids[g]);
                    else backward_front<TRANS, true>(S, ids[g]);
                }
                if (!EXACT && fwd) forward_quad<TRANS>(S, ids);
                if (!EXACT && !fwd) backward_quad<TRANS>(S, ids);
            } else {
                const int p = task[t < fronts ? t : t + 3 * quads];
                if (fwd) forward_front<TRANS, EXACT>(S, p);
                else backward_front<TRANS, EXACT>(S, p);
            }
        }
        __syncthreads();
    }
}

template <bool TRANS, typename T>
__device__ __attribute__((noinline)) void divide_solve(Lds<T> a, Lds<T> dinv, Lds<T> y, int scr, Lds<const int> ints,
                                                       int o_level, int o_task, int o_rows, int o_gptr, int o_gsrc,
                                                       int num_levels) {
    Sys<T> S{};
    S.a = (T*)a;
    S.dinv = (T*)dinv;
    S.y = (T*)y;
    S.scr = scr;
    S.front = (const SysFront*)(const int*)ints;
    S.level = (const int*)ints + o_level;
    S.list = (const unsigned short*)(const int*)ints;
    S.o_task = o_task;
    S.o_rows = o_rows;
    S.o_gptr = o_gptr;
    S.o_gsrc = o_gsrc;
    S.num_levels = num_levels;
    sweep_system<TRANS, true>(S);
}

template <bool TRANS, typename T>
__device__ __forceinline__ void divide_solve(const Sys<T>& S) {
    const int* ints = reinterpret_cast<const int*>(S.front);
    divide_solve<TRANS, T>(lds(S.a), lds(S.dinv), lds(S.y), S.scr, lds(ints), int(S.level - ints), S.o_task, S.o_rows,
                           S.o_gptr, S.o_gsrc, S.num_levels);
}

// On this thread's elements.
template <typename T>
__device__ __forceinline__ bool factors_hold_nan(const Sys<T>& S) {
    bool nan = false;
    for (int e = int(threadIdx.x); e < S.scr; e += int(blockDim.x)) nan = nan || S.a[e] != S.a[e];
    return nan;
}

// y = A^-1 y (or A^-T y); load() puts the right-hand side into y.  A result that
// is not finite is computed again by division, unless the factors hold a NaN.
template <bool TRANS, typename T, class F>
__device__ __forceinline__ void solve_system(const Sys<T>& S, int n, F load) {
    load();
    __syncthreads();
    sweep_system<TRANS, false>(S);
    bool finite = true;
    for (int k = int(threadIdx.x); k < n; k += int(blockDim.x)) finite = finite && __builtin_isfinite(S.y[k]);
    if (any_thread(S, !finite)) {
        if (any_thread(S, factors_hold_nan(S))) return;
        load();
        __syncthreads();
        divide_solve<TRANS>(S);
    }
}

__device__ __forceinline__ bool gate_closed(const int* gate) { return gate && *gate; }

// Carves the workgroup's LDS: the front-type arrays (8-byte aligned lengths),
// then the tables.  Returns the first free byte.
template <typename T>
__device__ __forceinline__ unsigned char* carve(const SysDevice& d, unsigned char* at, Sys<T>& S) {
    auto take = [&](int elems) {
        T* p = reinterpret_cast<T*>(at);
        at += (size_t(elems) * sizeof(T) + 15) / 16 * 16;
        return p;
    };
    S.a = take(d.fac + d.scratch);
    S.scr = d.fac;
    S.dinv = take(d.n);
    S.y = take(d.n);
    S.buf = take(kSysBuf + kSysMark);
    S.mark = reinterpret_cast<int*>(S.buf + kSysBuf);
    int4* blob = reinterpret_cast<int4*>(at);
    for (int e = int(threadIdx.x); e < d.blob_quads; e += int(blockDim.x)) blob[e] = d.blob[e];
    const int* ints = reinterpret_cast<const int*>(at);
    S.front = reinterpret_cast<const SysFront*>(ints);
    S.level = ints + d.o_level;
    S.list = reinterpret_cast<const unsigned short*>(ints);
    if (threadIdx.x == 0) {
        S.a[d.fac + d.scratch - 1] = T(0);                      // the zero element
        *S.mark = 0;
    }
    S.slice = ints + d.o_slice;
    S.adds = d.adds;
    S.o_task = d.o_task;
    S.o_rows = d.o_rows;
    S.o_gptr = d.o_gptr;
    S.o_gsrc = d.o_gsrc;
    S.o_perm = d.o_perm;
    S.num_levels = d.num_levels;
    return at + size_t(d.blob_quads) * 16;
}

template <typename T, int NT>
__global__ __launch_bounds__(NT, 2) void k_sys_factor(SysDevice d, const double* __restrict__ A, int Bp,
                                                   T* __restrict__ store, double eps, int static_piv,
                                                   int* __restrict__ sing) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    Sys<T> S;
    carve(d, smem, S);
    const int b = blockIdx.x, tid = threadIdx.x;
    int flag = 0;
    factor_matrix<T, NT>(S, d.n, eps, static_piv, flag, [&] {
        for (int e = tid; e < d.fac; e += NT) S.a[e] = T(0);
        __syncthreads();
        for (int k0 = tid; k0 < d.nnz; k0 += 4 * NT) {
            int at[4];
            double v[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int k = min(k0 + u * NT, d.nnz - 1);
                at[u] = d.slot_pos[k];
                v[u] = A[(long long)k * Bp + b];
            }
#pragma unroll
            for (int u = 0; u < 4; ++u)
                if (k0 + u * NT < d.nnz) S.a[at[u]] = T(v[u]);
        }
        __syncthreads();
    }, [&] {
        bool nan = false;
        for (int k = tid; k < d.nnz; k += NT) nan = nan || __builtin_isnan(A[(long long)k * Bp + b]);
        return nan;
    });
    T* out = store + (long long)b * (d.fac + d.n);
    for (int e = tid; e < d.fac; e += NT) out[e] = S.a[e];
    for (int e = tid; e < d.n; e += NT) out[d.fac + e] = S.dinv[e];
    if (flag && !gate_closed(d.gate)) atomicOr(sing + b, 1);
}

template <typename T, bool TRANS, typename TX, int NT>
__global__ __launch_bounds__(NT, 2) void k_sys_solve(SysDevice d, const T* __restrict__ store,
                                                  const double* __restrict__ rhs, int Bp,
                                                  TX* __restrict__ x) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    Sys<T> S;
    carve(d, smem, S);
    const int b = blockIdx.x, tid = threadIdx.x;
    const T* in = store + (long long)b * (d.fac + d.n);
    for (int e0 = tid; e0 < d.fac; e0 += 8 * NT) {              // eight loads in flight
        T v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = in[min(e0 + u * NT, d.fac - 1)];
#pragma unroll
        for (int u = 0; u < 8; ++u)
            if (e0 + u * NT < d.fac) S.a[e0 + u * NT] = v[u];
    }
    for (int e = tid; e < d.n; e += NT) S.dinv[e] = in[d.fac + e];
    __syncthreads();
    const unsigned short* perm = S.list + S.o_perm;
    solve_system<TRANS>(S, d.n, [&] {
        for (int k = tid; k < d.n; k += NT) S.y[k] = T(rhs[(long long)perm[k] * Bp + b]);
    });
    for (int k = tid; k < d.n; k += NT) x[(long long)perm[k] * Bp + b] = TX(S.y[k]);
}

// ---- fused Newton steps -----------------------------------------------------
struct Bus {
    double2* V;
    double2* I;       // Ybus V
    double2* vn;      // V / |V|
    double* F;        // mismatch, then the refinement's right-hand side
    double* dx;       // Newton step
};

// Ybus entry k for scenario b
__device__ __forceinline__ double2 y_value(const NrDevice& nr, int k, int Bp, int b) {
    return nr.yb ? nr.yb[(long long)k * Bp + b] : nr.y[k];
}

// V_i conj(I_i) - S_i in the batched residual kernel's operations
__device__ __forceinline__ double2 mismatch(const Bus& n, int i, double2 sb) {
#pragma clang fp contract(off)
    const double2 v = n.V[i], I = n.I[i];
    const double nI = -I.y;
    const double pr = v.x * I.x - v.y * nI;
    const double pi = v.x * nI + v.y * I.x;
    return make_double2(pr - sb.x, pi - sb.y);
}

// Row currents, |V|-normalised voltages and the mismatch of this thread's
// buses, in the batched residual kernel's operations and order; returns the
// norm's bits over its rows.
template <int NT>
__device__ __forceinline__ unsigned long long evaluate(const NrDevice& nr, const Bus& n,
                                                       const double2* __restrict__ Sb, int Bp, int b) {
#pragma clang fp contract(off)
    double m = 0.0;
    bool nan = false;
    for (int i = threadIdx.x; i < nr.n_bus; i += NT) {
        double ir = 0.0, ii = 0.0;
        const int k0 = nr.yp[i], k1 = nr.yp[i + 1];
        for (int kk = k0; kk < k1; kk += 4) {
            double2 y[4], v[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int k = min(kk + u, k1 - 1);
                y[u] = y_value(nr, k, Bp, b);
                v[u] = n.V[nr.yi[k]];
            }
#pragma unroll
            for (int u = 0; u < 4; ++u)
                if (kk + u < k1) {
                    ir += y[u].x * v[u].x - y[u].y * v[u].y;
                    ii += y[u].x * v[u].y + y[u].y * v[u].x;
                }
        }
        n.I[i] = make_double2(ir, ii);
        const double2 v = n.V[i];
        const double vm = fmax(hypot(v.x, v.y), 1e-8);
        n.vn[i] = make_double2(v.x / vm, v.y / vm);
        const int r1 = nr.row_pvpq[i];
        if (r1 < 0) continue;
        const double2 f = mismatch(n, i, Sb[(long long)i * Bp + b]);
        const double fr = f.x, fi = f.y;
        n.F[r1] = fr;
        m = fmax(m, fabs(fr));
        nan |= fr != fr;
        const int r2 = nr.row_pq[i];
        if (r2 >= 0) {
            n.F[r2] = fi;
            m = fmax(m, fabs(fi));
            nan |= fi != fi;
        }
    }
    return nan ? kNanBits : (unsigned long long)__double_as_longlong(m);
}

// dS_i/dVa_j and dS_i/d|V|_j of Ybus entry (i, j): real parts the P rows',
// imaginary parts the Q rows' (k_jacobian's operations).
__device__ __forceinline__ void entry_jacobian(const Bus& n, double2 y, int i, int j, double2& dva,
                                               double2& dvm) {
#pragma clang fp contract(off)
    const double2 vi = n.V[i], vj = n.V[j], vnj = n.vn[j];
    const double ja_r = vi.y, ja_i = -vi.x;                     // -j V_i
    const double cr = y.x * vj.x - y.y * vj.y;
    const double nci = -(y.x * vj.y + y.y * vj.x);
    dva = make_double2(ja_r * cr - ja_i * nci, ja_r * nci + ja_i * cr);
    const double wr = y.x * vnj.x - y.y * vnj.y;
    const double nwi = -(y.x * vnj.y + y.y * vnj.x);
    dvm = make_double2(vi.x * wr - vi.y * nwi, vi.x * nwi + vi.y * wr);
    if (i == j) {                                               // j V_i conj(I_i), conj(I_i) Vn_i
        const double2 I = n.I[i], vni = n.vn[i];
        const double nI = -I.y;
        const double sr = vi.x * I.x - vi.y * nI;
        const double si = vi.x * nI + vi.y * I.x;
        dva.x += -si;
        dva.y += sr;
        dvm.x += I.x * vni.x - nI * vni.y;
        dvm.y += I.x * vni.y + nI * vni.x;
    }
}

template <typename T, int NT>
__global__ __launch_bounds__(NT, 2) void k_sys_newton(SysDevice d, NrDevice nr, SysNet net, SysNewton o,
                                                   const double2* __restrict__ Sb,
                                                   double2* __restrict__ V, double* __restrict__ Va,
                                                   double* __restrict__ Vm, double* __restrict__ normF,
                                                   double* __restrict__ bmax, int* __restrict__ ctl,
                                                   unsigned long long* __restrict__ sync2, int Bp,
                                                   double eps, int static_piv, int* __restrict__ sing) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    __shared__ int word[2];                                     // stop, skip refinement
    __shared__ unsigned long long red[NT / 64];
    const int b = blockIdx.x, tid = threadIdx.x;
    if (!o.first) {
        const int stop = ctl[0], skip = ctl[1];
        if (stop && !o.finish) return;                          // the same for every thread
        if (tid == 0) {
            word[0] = 0;
            word[1] = o.finish ? !(o.refine > 0 && bmax[0] <= o.refine_below) : skip;
        }
    }
    Sys<T> S;
    unsigned char* at = carve(d, smem, S);
    Bus n;
    n.V = reinterpret_cast<double2*>(at);
    n.I = n.V + nr.n_bus;
    n.vn = n.I + nr.n_bus;
    n.F = reinterpret_cast<double*>(n.vn + nr.n_bus);
    n.dx = n.F + d.n;
    for (int i = tid; i < nr.n_bus; i += NT) {
        const double2 v = V[(long long)i * Bp + b];
        n.V[i] = v;
        if (o.seed) {
            Va[(long long)i * Bp + b] = atan2(v.y, v.x);
            Vm[(long long)i * Bp + b] = hypot(v.x, v.y);
        }
    }
    __syncthreads();
    unsigned long long bits = 0;
    // the norm of the residual just evaluated, the batch maximum and (by the
    // last workgroup) the control word
    auto conclude = [&](bool first) {
        for (int w = 32; w > 0; w >>= 1) {
            const unsigned long long v = __shfl_xor(bits, w);
            bits = max(bits, v);
        }
        if ((tid & 63) == 0) red[tid >> 6] = bits;
        __syncthreads();
        if (tid == 0) {
            for (int w = 1; w < NT / 64; ++w) bits = max(bits, red[w]);
            normF[b] = __longlong_as_double((long long)bits);
            const bool finite = (bits & 0x7ff0000000000000ull) != 0x7ff0000000000000ull;
            // the tolerant pass looks at finite norms only: 0 none, else bits + 1
            const unsigned long long mine = o.tolerant ? (finite ? bits + 1 : 0) : bits;
            unsigned long long all = mine;
            bool last = true;
            if (gridDim.x > 1) {
                atomicMax(sync2, mine);
                __threadfence();
                last = atomicAdd(sync2 + 1, 1ull) == gridDim.x - 1;
                if (last) {
                    __threadfence();
                    all = atomicExch(sync2, 0ull);
                    atomicExch(sync2 + 1, 0ull);
                }
            }
            if (last) {
                const double m = o.tolerant ? (all ? __longlong_as_double((long long)(all - 1)) : -1.0)
                                            : __longlong_as_double((long long)all);
                const int completed = (first ? 0 : ctl[2]) + 1;
                bool stop = o.tolerant ? m < 0.0 : !isfinite(m);
                stop = stop || m <= o.tol || completed >= o.limit;
                const bool want = !stop && o.refine > 0 && m <= o.refine_below;
                const int hist = first ? 0 : ctl[4];
                bmax[0] = m;
                ctl[0] = stop ? 1 : 0;
                ctl[1] = want ? 0 : 1;
                ctl[2] = completed;
                ctl[3] = (stop || want) ? 1 : 0;
                ctl[4] = (want && completed <= 31) ? (hist | (1 << (completed - 1))) : hist;
                word[0] = stop ? 1 : 0;
                word[1] = want ? 0 : 1;
            }
        }
        __syncthreads();
    };
    for (int pass = 0;; ++pass) {
        bits = evaluate<NT>(nr, n, Sb, Bp, b);
        if (pass > 0 || o.first) conclude(pass == 0);
        else __syncthreads();
        if (pass == o.steps || word[0]) break;
        const int solves = word[1] ? 1 : 1 + o.refine;
        auto load_jacobian = [&] {
            for (int e = tid; e < d.fac; e += NT) S.a[e] = T(0);
            __syncthreads();
            for (int k = tid; k < nr.nnzY; k += NT) {
                const int4 at4 = net.ydst[k];
                double2 dva, dvm;
                entry_jacobian(n, y_value(nr, k, Bp, b), net.yrow[k], nr.yi[k], dva, dvm);
                if (at4.x >= 0) S.a[at4.x] = T(dva.x);
                if (at4.y >= 0) S.a[at4.y] = T(dva.y);
                if (at4.z >= 0) S.a[at4.z] = T(dvm.x);
                if (at4.w >= 0) S.a[at4.w] = T(dvm.y);
            }
            __syncthreads();
        };
        const unsigned short* perm = S.list + S.o_perm;
        load_jacobian();
        int flag = 0;
        factor_system<T, NT>(S, eps, static_piv, flag);
        // As factor_matrix() and solve_system(), with the reciprocals and results
        // looked at on the way and told over the barriers that are there anyway:
        // kLook until one asks for divisions, then kDivide, or kLeave where there
        // is a NaN
        enum { kLook, kLeave, kDivide } mode = kLook;
        for (int it = 0; it < solves; ++it) {
            // refinement: F - J dx, a bus's two rows per thread; the mismatch
            // itself is formed again from the row currents (F then holds the
            // residual), as it is to start the solves again
            for (int i = tid; (it > 0 || mode == kDivide) && i < nr.n_bus; i += NT) {
                const int r1 = nr.row_pvpq[i], r2 = nr.row_pq[i];
                if (r1 < 0) continue;
                double ap = 0.0, aq = 0.0;
                for (int k = nr.yp[i]; it > 0 && k < nr.yp[i + 1]; ++k) {
                    const int j = nr.yi[k];
                    double2 dva, dvm;
                    entry_jacobian(n, y_value(nr, k, Bp, b), i, j, dva, dvm);
                    const int c1 = nr.row_pvpq[j], c2 = nr.row_pq[j];
                    const double xa = c1 >= 0 ? n.dx[c1] : 0.0, xm = c2 >= 0 ? n.dx[c2] : 0.0;
                    ap = fma(dva.x, xa, fma(dvm.x, xm, ap));
                    aq = fma(dva.y, xa, fma(dvm.y, xm, aq));
                }
                const double2 fi = mismatch(n, i, Sb[(long long)i * Bp + b]);
                n.F[r1] = fi.x - ap;
                if (r2 >= 0) n.F[r2] = fi.y - aq;
            }
            __syncthreads();
            bool ask = false;
            for (int k = tid; k < d.n; k += NT) {
                S.y[k] = T(n.F[perm[k]]);
                ask = ask || !__builtin_isnormal(S.dinv[k]);
            }
            if (ask && mode == kLook) *S.mark = 1;
            __syncthreads();
            if (__builtin_expect(*S.mark, 0)) {                 // before the first solve, or never
                clear_mark(S);
                bool nan = false;
                for (int i = tid; i < nr.n_bus; i += NT) nan = nan || n.V[i].x != n.V[i].x || n.V[i].y != n.V[i].y;
                mode = any_thread(S, nan) ? kLeave : kDivide;
                if (mode == kDivide) {
                    load_jacobian();
                    flag = divide_factors(S, eps, static_piv);
                }
            }
            if (__builtin_expect(mode == kDivide, 0))
                divide_solve<false>(S);
            else
                sweep_system<false, false>(S);
            ask = false;
            for (int k = tid; k < d.n; k += NT) {
                const T y = S.y[k];
                ask = ask || !__builtin_isfinite(y);
                n.dx[perm[k]] = it > 0 ? n.dx[perm[k]] + double(y) : double(y);
            }
            if (ask && mode == kLook) *S.mark = 1;
            __syncthreads();
            if (__builtin_expect(*S.mark, 0)) {
                clear_mark(S);
                mode = any_thread(S, factors_hold_nan(S)) ? kLeave : kDivide;
                if (mode == kDivide) it = -1;                   // the solves again
            }
        }
        if (flag) atomicOr(sing + b, 1);
        for (int i = tid; i < nr.n_bus; i += NT) {
            const long long g = (long long)i * Bp + b;
            const int r1 = nr.row_pvpq[i], r2 = nr.row_pq[i];
            double va = Va[g], vm = Vm[g];
            if (r1 >= 0) va -= n.dx[r1];
            if (r2 >= 0) vm -= n.dx[r2];
            Va[g] = va;
            Vm[g] = vm;
            double sn, cs;
            sincos(va, &sn, &cs);
            const double2 v = make_double2(vm * cs, vm * sn);
            V[g] = v;
            n.V[i] = v;
        }
        if (o.finish) return;
        __syncthreads();
    }
}

// Threads of a workgroup: eight waves while a workgroup has its CU to itself
// (by the batch or by its LDS), four when they share CUs.
constexpr int kSysWide = 512, kSysNarrow = 256;
constexpr int kSysCus = 256;

}  // namespace

size_t sys_lds_bytes(const SysPlan& p, int elem, int n_bus) {
    auto up = [](size_t v) { return (v + 15) / 16 * 16; };
    size_t t = up(size_t(p.fac + p.scratch) * elem) + 2 * up(size_t(p.n) * elem) + (kSysBuf + kSysMark) * size_t(elem) +
               p.blob.size() * sizeof(int);
    if (n_bus > 0) t += size_t(n_bus) * 3 * sizeof(double2) + size_t(p.n) * 2 * sizeof(double);
    return t;
}

template <int NT>
void raise_all() {
    raise_lds((const void*)k_sys_factor<double, NT>, kSysLdsMax);
    raise_lds((const void*)k_sys_factor<float, NT>, kSysLdsMax);
    raise_lds((const void*)k_sys_solve<double, false, double, NT>, kSysLdsMax);
    raise_lds((const void*)k_sys_solve<double, true, double, NT>, kSysLdsMax);
    raise_lds((const void*)k_sys_solve<double, false, float, NT>, kSysLdsMax);
    raise_lds((const void*)k_sys_solve<double, true, float, NT>, kSysLdsMax);
    raise_lds((const void*)k_sys_solve<float, false, double, NT>, kSysLdsMax);
    raise_lds((const void*)k_sys_solve<float, true, double, NT>, kSysLdsMax);
    raise_lds((const void*)k_sys_solve<float, false, float, NT>, kSysLdsMax);
    raise_lds((const void*)k_sys_solve<float, true, float, NT>, kSysLdsMax);
    raise_lds((const void*)k_sys_newton<double, NT>, kSysLdsMax);
    raise_lds((const void*)k_sys_newton<float, NT>, kSysLdsMax);
}

void sys_prepare() {
    static OncePerDevice first_use;
    first_use([] {
        raise_all<kSysWide>();
        raise_all<kSysNarrow>();
    });
}

// go(threads) with the workgroup size for B scenarios as a compile-time value
template <class F>
void with_threads(int B, size_t lds, F go) {
    if (B <= kSysCus || 2 * lds > kSysLdsMax) go(std::integral_constant<int, kSysWide>{});
    else go(std::integral_constant<int, kSysNarrow>{});
    CUPF_HIP(hipGetLastError());
}

template <typename T>
void sys_factor(const SysDevice& d, const double* A, int B, int Bp, T* store, double pivot_eps,
                int static_piv, int* sing, size_t lds, hipStream_t s) {
    with_threads(B, lds, [&](auto nt) {
        constexpr int NT = decltype(nt)::value;
        k_sys_factor<T, NT><<<B, NT, lds, s>>>(d, A, Bp, store, pivot_eps, static_piv, sing);
    });
}

template <typename T, typename TX>
void sys_solve(const SysDevice& d, const T* store, const double* rhs, int B, int Bp, TX* x,
               bool transpose, size_t lds, hipStream_t s) {
    with_threads(B, lds, [&](auto nt) {
        constexpr int NT = decltype(nt)::value;
        if (transpose) k_sys_solve<T, true, TX, NT><<<B, NT, lds, s>>>(d, store, rhs, Bp, x);
        else k_sys_solve<T, false, TX, NT><<<B, NT, lds, s>>>(d, store, rhs, Bp, x);
    });
}

template <typename T>
void sys_newton(const SysDevice& d, const NrDevice& nr, const SysNet& net, const SysNewton& o,
                const double2* S, double2* V, double* Va, double* Vm, double* normF, double* bmax,
                int* ctl, unsigned long long* sync2, int B, int Bp, double pivot_eps,
                int static_piv, int* sing, size_t lds, hipStream_t s) {
    with_threads(B, lds, [&](auto nt) {
        constexpr int NT = decltype(nt)::value;
        k_sys_newton<T, NT><<<B, NT, lds, s>>>(d, nr, net, o, S, V, Va, Vm, normF, bmax, ctl, sync2, Bp,
                                               pivot_eps, static_piv, sing);
    });
}

#define CUPF_SYS(T)                                                                                  \
    template void sys_factor<T>(const SysDevice&, const double*, int, int, T*, double, int, int*,    \
                                size_t, hipStream_t);                                                \
    template void sys_solve<T, double>(const SysDevice&, const T*, const double*, int, int, double*, \
                                       bool, size_t, hipStream_t);                                   \
    template void sys_solve<T, float>(const SysDevice&, const T*, const double*, int, int, float*,   \
                                      bool, size_t, hipStream_t);                                    \
    template void sys_newton<T>(const SysDevice&, const NrDevice&, const SysNet&, const SysNewton&,  \
                                const double2*, double2*, double*, double*, double*, double*, int*,  \
                                unsigned long long*, int, int, double, int, int*, size_t, hipStream_t);
CUPF_SYS(double)
CUPF_SYS(float)

}  // namespace cupf::kern
