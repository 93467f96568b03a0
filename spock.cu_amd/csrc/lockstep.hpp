// The lockstep SuperMann solve of many instances of ONE problem (src/cache.cuh:1008-1132), shared
// by the engines of shared batches.  An engine policy E supplies the lane-to-instance mapping and
// the operators:
//   E::ctx()                 wave, nw, gl (this lane's instance) and writer (the lane that writes
//                            the instance's per-instance records; several lanes may serve one
//                            instance and then hold identical per-instance state);
//   E::view<T>(region, rows, c)  v[e] = element e of this lane's instance;
//   E::pass<U>(n, c, ld, st) an iterate-wide pass in which every (element, instance) pair is
//                            visited by exactly one lane;
//   E::sum / E::max          per-instance combination of per-lane partials, in a fixed order;
//   E::applyT, E::reduceEll, E::adjDots  the CP operator and the [L*; L] reductions.
// SuperMann runs in lockstep outer iterations with per-lane decisions: the buffer roles rotate
// uniformly where every lane takes the same step, and per-lane masked copies replace the rotations
// where lanes branch (K0 vs line search, K1/K2/K3).
#pragma once
#include "engine.hpp"

#include <hip/hip_runtime.h>
#include <math.h>

#include <type_traits>

namespace spk {

template <typename T>
using LP = const SPK_CONST LaneInst<T> &;

namespace ls {

constexpr int MAXM = 4;  // Anderson memory supported by the engines of shared batches

// Device wall-clock per phase, accumulated by thread 0 into LDS (uniform control flow, so
// thread 0's view is the workgroup's).
struct LaneClock {
    long last;
    long *acc;
    __device__ __forceinline__ void mark(int ph) {
        const long t = wall_clock64();
        if (threadIdx.x == 0) acc[ph] += t - last;
        last = t;
    }
    __device__ __forceinline__ void skip() { last = wall_clock64(); }
};

template <typename T>
struct DotMax {
    T dot, mx, cross;  // cross = sum over primal elements of x_p . (L* y_d)
};

template <typename T>
struct Cross2 {
    T c1, c2;
};

template <typename T>
struct V2 {
    T a, b;
};
template <typename T>
struct V4 {
    T a, b, c, d;
};
template <typename T, int M>
struct VH {  // two vector values and M history values of one element
    T a, b, h[M];
};
template <typename T, int M>
struct V4H {
    T a, b, c, d, h[M];
};

__device__ __forceinline__ bool anyLane(bool v) { return __syncthreads_or(v ? 1 : 0) != 0; }

// Least squares argmin ||Y g - r|| from the Gram matrix: Cholesky of G + 1e-12 max(diag) I in FP64.
__device__ __forceinline__ bool gramSolve(const double (&G)[MAXM][MAXM], const double (&gb)[MAXM], int m,
                                          double (&g)[MAXM]) {
    double Lm[MAXM][MAXM];
    double dmax = 0.;
#pragma unroll
    for (int i = 0; i < MAXM; i++)
        if (i < m) dmax = fmax(dmax, G[i][i]);
    if (!(dmax > 0.)) return false;
    const double ridge = 1e-12 * dmax;
    bool ok = true;
#pragma unroll
    for (int i = 0; i < MAXM; i++) {
#pragma unroll
        for (int j = 0; j < MAXM; j++) {
            Lm[i][j] = 0.;
            if (i < m && j <= i) {
                double v = G[i][j] + (i == j ? ridge : 0.);
#pragma unroll
                for (int k = 0; k < MAXM; k++)
                    if (k < j) v -= Lm[i][k] * Lm[j][k];
                if (i == j) {
                    ok = ok && (v > 0.);
                    Lm[i][i] = sqrt(fmax(v, 0.));
                } else {
                    Lm[i][j] = v / Lm[j][j];
                }
            }
        }
    }
    if (!ok) return false;
    double y[MAXM];
#pragma unroll
    for (int i = 0; i < MAXM; i++) {
        y[i] = 0.;
        if (i < m) {
            double v = gb[i];
#pragma unroll
            for (int k = 0; k < MAXM; k++)
                if (k < i) v -= Lm[i][k] * y[k];
            y[i] = v / Lm[i][i];
        }
    }
#pragma unroll
    for (int i = MAXM - 1; i >= 0; i--) {
        g[i] = 0.;
        if (i < m) {
            double v = y[i];
#pragma unroll
            for (int k = 0; k < MAXM; k++)
                if (k > i && k < m) v -= Lm[k][i] * g[k];
            g[i] = v / Lm[i][i];
        }
    }
    return true;
}

// ---------------------------------------------------------------- iterate-wide passes
// Never inlined: inside the solve its own state (Gram matrix, counters, tolerances: over 100 registers)
// left the passes' loads in flight to be spilled to memory (1,000 FP64 instances of the 229-node problem, 63
// of 256 CUs: residual and direction passes 2.5 + 2.0 ms an iteration, now 1.4 + 0.9; the 4,096 FP32
// instances, bound by HBM, 1.36 + 1.16 ms, now 1.35 + 0.82).
template <typename T>
struct ColumnSums {
    T rr;                  // |r|^2
    double yy[MAXM], yr[MAXM];  // <Y_head, Y_s> and <Y_s, r>
};

// r = z - T(z), ||r||^2 and, in the same pass, the new Anderson column (src/cache.cuh:861-896) with its
// Gram entries: Y_head = r - r_prev, S_head = (z - z_prev) - Y_head, of M columns.  Sums per lane.
template <typename T, typename E, int M>
__device__ __noinline__ ColumnSums<T> columnPass(const LaneInst<T> *Pp, T *zIn, T *cIn, T *rpIn, T *zpIn, T *rIn, int headIn) {
    LP<T> P = *cst(uniformPtr(Pp));
    const auto c = E::ctx();
    const long n = P.sIter, B = P.B;
    const int head = __builtin_amdgcn_readfirstlane(headIn);
    auto V = [&](T *p) { return E::template view<T>(uniformPtr(p), n, c); };
    const auto Yh = V(P.hY + (long) head * n * B), Sh = V(P.hS + (long) head * n * B);
    const auto rr = V(rIn), cc = V(cIn), rp = V(rpIn), z = V(zIn), zp = V(zpIn);
    constexpr int O = M > 1 ? M - 1 : 1;  // the other columns: slots head + 1 .. head + M - 1
    typename E::template View<T> Yo[O];
#pragma unroll
    for (int i = 0; i < O; i++) Yo[i] = V(P.hY + (long) ((head + 1 + i) % M) * n * B);
    T sr = T(0);
    double hh = 0., hr = 0., oh[O], orr[O];
#pragma unroll
    for (int i = 0; i < O; i++) oh[i] = orr[i] = 0.;
    E::template pass<4>(
        n, c,
        [&](long e) {
            V4H<T, O> v;
            v.a = z[e];
            v.b = cc[e];
            v.c = rp[e];
            v.d = zp[e];
#pragma unroll
            for (int i = 0; i < M - 1; i++) v.h[i] = Yo[i][e];
            return v;
        },
        [&](long e, const V4H<T, O> &v) {
            const T r = v.a - v.b;
            rr[e] = r;
            sr += r * r;
            const T dr = r - v.c;
            Yh[e] = dr;
            Sh[e] = (v.a - v.d) - dr;
            const double drd = (double) dr, rd = (double) r;
            hh += drd * drd;
            hr += drd * rd;
#pragma unroll
            for (int i = 0; i < M - 1; i++) {
                oh[i] += drd * (double) v.h[i];
                orr[i] += (double) v.h[i] * rd;
            }
        });
    ColumnSums<T> a;
    a.rr = sr;
#pragma unroll
    for (int q = 0; q < MAXM; q++) {
        a.yy[q] = q == head ? hh : 0.;
        a.yr[q] = q == head ? hr : 0.;
#pragma unroll
        for (int i = 0; i < M - 1; i++) {
            a.yy[q] = q == (head + 1 + i) % M ? oh[i] : a.yy[q];
            a.yr[q] = q == (head + 1 + i) % M ? orr[i] : a.yr[q];
        }
    }
    return a;
}

// d = -S g - r; K0 lanes write cand = z_prev + d (src/cache.cuh:897-898, 1055-1057).
template <typename T>
struct Coeffs {
    T g[MAXM];
};

template <typename T, typename E, int M>
__device__ __noinline__ void directionPass(const LaneInst<T> *Pp, T *rpIn, T *zpIn, T *dIn, T *cIn, Coeffs<T> k, bool blind) {
    LP<T> P = *cst(uniformPtr(Pp));
    const auto c = E::ctx();
    const long n = P.sIter, B = P.B;
    auto V = [&](T *p) { return E::template view<T>(uniformPtr(p), n, c); };
    typename E::template View<T> Ss[M];
#pragma unroll
    for (int i = 0; i < M; i++) Ss[i] = V(P.hS + (long) i * n * B);
    const auto rp = V(rpIn), zp = V(zpIn), dd = V(dIn), cc = V(cIn);
    E::template pass<4>(
        n, c,
        [&](long e) {
            VH<T, M> v;
            v.a = rp[e];
            v.b = zp[e];
#pragma unroll
            for (int i = 0; i < M; i++) v.h[i] = Ss[i][e];
            return v;
        },
        [&](long e, const VH<T, M> &v) {
            T sg = T(0);
#pragma unroll
            for (int i = 0; i < M; i++) sg += v.h[i] * k.g[i];
            const T d = -sg - v.a;
            if (blind) cc[e] = v.b + d;
            else dd[e] = d;
        });
}

// f<M>() for the Anderson memory m (1 .. MAXM).
template <typename F>
__device__ __forceinline__ void withMemory(int m, F f) {
    if (m == 3) f(std::integral_constant<int, 3>{});
    else if (m == 1) f(std::integral_constant<int, 1>{});
    else if (m == 2) f(std::integral_constant<int, 2>{});
    else f(std::integral_constant<int, 4>{});
}

// out = a - f b for the lanes with `take` (f = 0: a copy).
template <typename T, typename E>
__device__ __noinline__ void takePass(long n, T *outIn, T *aIn, T *bIn, T f, bool take) {
    const auto c = E::ctx();
    n = __builtin_amdgcn_readfirstlane((int) n);  // an iterate's size is an int (spk_problem_sizes)
    auto V = [&](T *p) { return E::template view<T>(uniformPtr(p), n, c); };
    const auto out = V(outIn), a = V(aIn);
    if (bIn == nullptr) {
        E::template pass<8>(n, c, [&](long e) -> T { return a[e]; }, [&](long e, T v) {
            if (take) out[e] = v;
        });
        return;
    }
    const auto b = V(bIn);
    E::template pass<8>(n, c, [&](long e) { return V2<T>{a[e], b[e]}; }, [&](long e, const V2<T> &v) {
        if (take) out[e] = v.a - v.b * f;
    });
}

// The line search's trial point: ds = tau d, z = z_prev + ds (src/cache.cuh:1063-1065).
template <typename T, typename E>
__device__ __noinline__ void trialPass(long n, T *dIn, T *zpIn, T *dsIn, T *zIn, T tau, bool ls) {
    const auto c = E::ctx();
    n = __builtin_amdgcn_readfirstlane((int) n);
    auto V = [&](T *p) { return E::template view<T>(uniformPtr(p), n, c); };
    const auto d = V(dIn), zp = V(zpIn), ds = V(dsIn), z = V(zIn);
    E::template pass<8>(n, c, [&](long e) { return V2<T>{d[e], zp[e]}; }, [&](long e, const V2<T> &v) {
        if (ls) {
            const T s = v.a * tau;
            ds[e] = s;
            z[e] = v.b + s;
        }
    });
}

// r = z - T(z), |r|^2 and <r, ds> (ds == nullptr: r only).  Sums per lane.
template <typename T, typename E>
__device__ __noinline__ V2<T> residualPass(long n, T *zIn, T *cIn, T *dsIn, T *rIn) {
    const auto c = E::ctx();
    n = __builtin_amdgcn_readfirstlane((int) n);
    auto V = [&](T *p) { return E::template view<T>(uniformPtr(p), n, c); };
    const auto rr = V(rIn), z = V(zIn), cc = V(cIn);
    V2<T> a{T(0), T(0)};
    if (dsIn == nullptr) {
        E::template pass<8>(n, c, [&](long e) { return V2<T>{z[e], cc[e]}; },
                            [&](long e, const V2<T> &v) { rr[e] = v.a - v.b; });
        return a;
    }
    const auto ds = V(dsIn);
    E::template pass<8>(n, c, [&](long e) { return V4<T>{z[e], cc[e], ds[e], T(0)}; }, [&](long e, const V4<T> &v) {
        const T d = v.a - v.b;
        rr[e] = d;
        a.a += d * d;
        a.b += d * v.c;
    });
    return a;
}

}  // namespace ls

// ---------------------------------------------------------------- the lockstep solve
template <typename T, typename E>
__device__ void lockstepSolve(const LaneInst<T> *Pp, Out *outs, double *lds, long *phaseAcc) {
    using namespace ls;
    using VW = typename E::template View<T>;
    LP<T> P = *cst(Pp);
    if (threadIdx.x < NUM_PHASES) phaseAcc[threadIdx.x] = 0;
    __syncthreads();
    LaneClock clk{wall_clock64(), phaseAcc};
    const auto c = E::ctx();
    const long n = P.sIter, B = P.B;
    const int gl = c.gl;
    const bool real = gl < P.count;
    const int m = P.andBuff;
    auto V = [&](T *p) { return E::template view<T>(p, n, c); };
    T *Z = P.work[0], *C = P.work[1], *ZP = P.work[2], *RR = P.work[3], *RP = P.work[4], *BK = P.work[5];
    T *C2 = P.work[6], *D = P.work[7], *DS = P.work[8];
    const long t0 = wall_clock64();
    const bool resume = P.resume != 0;
    LaneGroupSave *gs = P.gsave + blockIdx.x;
    long itStart = 0, ticksBefore = 0;
    int headSaved = m - 1;
    // a resume of a workgroup whose solve has ended leaves its results as they are
    if (resume && __builtin_amdgcn_readfirstlane(gs->finished)) return;
    if (resume) {  // roles of the six rotating buffers, ring head, next iteration (uniform)
        T **roles[6] = {&Z, &C, &ZP, &RR, &RP, &BK};
#pragma unroll
        for (int i = 0; i < 6; i++) *roles[i] = P.work[__builtin_amdgcn_readfirstlane(gs->roles[i])];
        headSaved = __builtin_amdgcn_readfirstlane(gs->head);
        const long itv = gs->it;
        itStart = ((long) __builtin_amdgcn_readfirstlane((int) (itv >> 32)) << 32) |
                  (unsigned) __builtin_amdgcn_readfirstlane((int) itv);
        ticksBefore = gs->ticks;
    }
    // initialiseIter / initialisePrev (src/cache.cuh:611-632)
    if (!resume) {
        const VW zio = V(P.zio), rio = V(P.rio), z = V(Z), zp = V(ZP), rp = V(RP);
        const bool spock = P.method == METHOD_SPOCK, warm = P.warm != 0;
        E::template pass<16>(
            n, c, [&](long e) { return V2<T>{zio[e], rio[e]}; },
            [&](long e, const V2<T> &v) {
                z[e] = v.a;
                if (spock) {
                    zp[e] = warm ? v.a : T(1);
                    rp[e] = warm ? v.b : T(1);
                }
            });
    }
    __syncthreads();
    double G[MAXM][MAXM], gb[MAXM];
#pragma unroll
    for (int i = 0; i < MAXM; i++) {
        gb[i] = 0.;
#pragma unroll
        for (int j = 0; j < MAXM; j++) G[i][j] = 0.;
    }
    int head = headSaved;
    bool active = real;
    const T given = (real && P.tolFixed) ? P.tolFixed[gl] : T(0);
    bool initFlag = !(given > T(0));
    int status = ST_NOTRUN;
    long iters = 0;
    T tol = initFlag ? T(0) : given, lastErr = T(NAN), wLast = T(NAN);
    const T c0 = T(0.99), c1 = T(0.99), c2 = T(0.99), beta = T(0.5), sigma = T(0.1), lambda = T(1);
    const T inf = T(INFINITY);
    T zeta = inf, w = inf, wSafe = inf;
    long k0 = 0, k1 = 0, k2 = 0, k2bt = 0, k3 = 0, nT = 0, nEll = 0;
    long it0 = 0;  // the workgroup iteration this lane's solve started at (later than 0 after a refill)
    if (resume) {  // this lane's SuperMann state
        const LaneSave &sv = P.save[gl];
#pragma unroll
        for (int i = 0; i < MAXM; i++) {
            gb[i] = sv.gb[i];
#pragma unroll
            for (int j = 0; j < MAXM; j++) G[i][j] = sv.G[i][j];
        }
        tol = (T) sv.tol;
        lastErr = (T) sv.lastErr;
        wLast = (T) sv.wLast;
        zeta = (T) sv.zeta;
        w = (T) sv.w;
        wSafe = (T) sv.wSafe;
        iters = sv.iters;
        k0 = sv.k0; k1 = sv.k1; k2 = sv.k2; k2bt = sv.k2bt; k3 = sv.k3; nT = sv.nT; nEll = sv.nEll;
        status = sv.status;
        active = sv.active != 0;
        initFlag = sv.initFlag != 0;
        it0 = sv.it0;
    }
    // the iteration cap is only tested at error checks (src/cache.cuh:937-940): a lane's last outer
    // iteration is the first check index at or beyond maxIters of its own count; without a cap a
    // lane still running after 2e6 iterations ends with its current iterate
    const long hardCap =
        P.maxIters > 0 ? (P.maxIters + P.checkPeriod - 1) / P.checkPeriod * P.checkPeriod + 1 : 2000000;
    long it;
    bool chunkExit = false;
    for (it = itStart;; it++) {
        const bool capNow = active && it - it0 >= hardCap;
        if (anyLane(capNow)) {  // the current iterate is the output
            takePass<T, E>(n, P.zio, Z, nullptr, T(0), capNow);
            takePass<T, E>(n, P.rio, RR, nullptr, T(0), capNow);
            __syncthreads();
        }
        if (capNow) {
            status = ST_OUTOFITER;
            iters = it - it0;
            active = false;
        }
        if (!anyLane(active)) break;
        // uniform: save and leave.  The time slice is thread 0's clock, made uniform by the
        // workgroup-wide vote, so every wave leaves at the same iteration.
        if (P.chunkIters > 0 &&
            (it >= itStart + P.chunkIters ||
             (P.chunkTicks > 0. && it > itStart &&
              anyLane(threadIdx.x == 0 && (double) (wall_clock64() - t0) >= P.chunkTicks)))) {
            chunkExit = true;
            break;
        }
        if (it != 0 && P.method == METHOD_SPOCK) {  // acceptCandidate: z <- cand
            T *t = Z;
            Z = C;
            C = t;
        }
        clk.mark(PH_OTHER);
        E::applyT(Pp, Z, C, phaseAcc);
        clk.skip();
        if (active) nT++;
        T sRR;
        const bool spock = P.method == METHOD_SPOCK;
        if (spock) head = (head + 1) % m;
        const bool checkIt = (it - it0) % P.checkPeriod == 0;
        if (!spock) {
            // r = z - T(z): of the plain method only the error checks read it, and the iteration cap, which
            // outputs the residual of the iteration before it
            if (!anyLane(active && (checkIt || it - it0 + 1 >= hardCap))) {
                T *t = Z;
                Z = C;
                C = t;
                clk.mark(PH_RES);
                continue;
            }
            residualPass<T, E>(n, Z, C, nullptr, RR);
            __syncthreads();
            sRR = T(0);
        } else {
            ColumnSums<T> a;
            withMemory(m, [&](auto M) { a = columnPass<T, E, M()>(Pp, Z, C, RP, ZP, RR, head); });
            sRR = (T) E::sum((double) a.rr, lds, c);
#pragma unroll
            for (int q = 0; q < MAXM; q++) {
                if (q < m) {
                    a.yy[q] = E::sum(a.yy[q], lds, c);
                    a.yr[q] = E::sum(a.yr[q], lds, c);
                }
            }
#pragma unroll
            for (int s2 = 0; s2 < MAXM; s2++) {
                if (s2 < m) {
#pragma unroll
                    for (int hh = 0; hh < MAXM; hh++) {
                        if (hh == head) {
                            G[hh][s2] = a.yy[s2];
                            G[s2][hh] = a.yy[s2];
                        }
                    }
                    gb[s2] = a.yr[s2];
                }
            }
        }
        clk.mark(PH_RES);
        // <r, M r> = ||r||^2 - 2 gamma r_p . L* r_d; the full [L*; L] only at the error checks
        T mx = T(0), crossRR = T(0);
        if (anyLane(active && checkIt)) {
            const DotMax<T> dm = E::reduceEll(Pp, RR, RR, lds);
            mx = dm.mx;
            crossRR = dm.cross;
        } else if (spock) {
            crossRR = E::adjDots(Pp, RR, RR, lds, false).c1;
        }
        const T dotRR = sRR - T(2) * P.gamma * crossRR;
        if (active && (spock || checkIt)) nEll++;
        clk.mark(PH_ELL);
        bool done = false;
        if (active && checkIt) {  // computeError (src/cache.cuh:910-961)
            if (initFlag) {
                tol = fmax(P.tolAbs, P.tolRel * mx);
                initFlag = false;
            } else {
                lastErr = mx;
                int code = ST_NOTRUN;
                if (mx <= tol) code = ST_CONVERGED;
                if (P.maxIters && it - it0 >= P.maxIters) code = ST_OUTOFITER;
                if (P.maxTicks > 0 && (it - it0) % 1000 == 0 &&
                    (double) (wall_clock64() - t0 + ticksBefore) >= P.maxTicks)
                    code = ST_OUTOFTIME;
                if (code != ST_NOTRUN) {
                    status = code;
                    iters = it - it0;
                    done = true;
                }
            }
        }
        if (anyLane(done)) {  // accepted candidate and its residual are the solve's output
            takePass<T, E>(n, P.zio, C, nullptr, T(0), done);
            takePass<T, E>(n, P.rio, RR, nullptr, T(0), done);
            __syncthreads();
        }
        if (done) active = false;
        if (P.method == METHOD_CP) {
            T *t = Z;
            Z = C;
            C = t;
            continue;
        }
        {  // backup (src/cache.cuh:804-806)
            T *t = BK;
            BK = C;
            C = t;
        }
        w = sqrt(dotRR);
        if (active) wLast = w;
        clk.mark(PH_ACOL);
        {  // saveToPrev as role moves
            T *t = ZP;
            ZP = Z;
            Z = t;
            t = RP;
            RP = RR;
            RR = t;
        }
        double gs[MAXM];
#pragma unroll
        for (int q = 0; q < MAXM; q++) gs[q] = 0.;
        const bool useLS = (it - it0 >= m) && gramSolve(G, gb, m, gs);
        clk.mark(PH_ALS);
        const bool blind = active && (w <= c0 * zeta);
        Coeffs<T> gg;
#pragma unroll
        for (int s2 = 0; s2 < MAXM; s2++) gg.g[s2] = (useLS && s2 < m) ? (T) gs[s2] : T(0);
        withMemory(m, [&](auto M) { directionPass<T, E, M()>(Pp, RP, ZP, D, C, gg, blind); });
        __syncthreads();
        clk.mark(PH_AAPPLY);
        if (blind) {
            zeta = w;
            k0++;
        }
        bool ls = active && !blind;
        T tau = T(1);
        for (int in = 0; in < P.maxInner; in++) {  // line search (src/cache.cuh:1063-1099)
            if (!anyLane(ls)) break;
            trialPass<T, E>(n, D, ZP, DS, Z, tau, ls);
            __syncthreads();
            clk.mark(PH_LINE);
            E::applyT(Pp, Z, C2, phaseAcc);
            clk.skip();
            if (ls) nT++;
            // r~ = z - T(z), ||r~||^2 and r~ . ds
            const V2<T> sums = residualPass<T, E>(n, Z, C2, DS, RR);
            const T sRRt = (T) E::sum((double) sums.a, lds, c);
            const T sRD = (T) E::sum((double) sums.b, lds, c);
            clk.mark(PH_RES);
            // <r~, M r~> and <r~, M ds> from two adjoints (src/cache.cuh:1066,1080)
            const Cross2<T> cr = E::adjDots(Pp, RR, DS, lds, true);
            const T wTilde = sqrt(sRRt - T(2) * P.gamma * cr.c1);
            const T dotRD = sRD - P.gamma * cr.c2;
            if (ls) nEll++;
            clk.mark(PH_ELL);
            const bool takeK1 = ls && (w <= wSafe) && (wTilde <= c1 * w);
            if (anyLane(takeK1)) {  // K1: cand <- z
                takePass<T, E>(n, C, Z, nullptr, T(0), takeK1);
                __syncthreads();
            }
            if (takeK1) {
                wSafe = wTilde + pow(c2, T(it - it0));
                k1++;
            }
            const bool still = ls && !takeK1;
            const T rho = wTilde * wTilde - dotRD;
            const bool takeK2 = still && (rho >= sigma * wTilde * w);
            if (anyLane(takeK2)) {  // K2: cand <- z_prev - f r
                const T f = lambda * rho / (wTilde * wTilde);
                takePass<T, E>(n, C, ZP, RR, f, takeK2);
                __syncthreads();
            }
            if (takeK2) k2++;
            const bool back = still && !takeK2;
            if (back) {
                tau *= beta;
                k2bt++;
            }
            const bool takeK3 = back && (in >= P.maxInner - 1);
            if (anyLane(takeK3)) {  // K3: restore the plain CP step
                takePass<T, E>(n, C, BK, nullptr, T(0), takeK3);
                __syncthreads();
            }
            if (takeK3) k3++;
            ls = back;
            clk.mark(PH_LINE);
        }
    }
    // A resumable (chunked) launch keeps everything a resume or a refill needs, whether it ended
    // at the chunk's end or because every lane had finished; results report the progress so far.
    if (P.chunkIters > 0) {
        if (threadIdx.x == 0) {
            gs->finished = chunkExit ? 0 : 1;
            T *cur[6] = {Z, C, ZP, RR, RP, BK};
            for (int i = 0; i < 6; i++)
                for (int j = 0; j < 6; j++)
                    if (cur[i] == P.work[j]) gs->roles[i] = j;
            gs->head = head;
            gs->it = it;
            gs->ticks = ticksBefore + (long) (wall_clock64() - t0);
        }
        if (c.wave == 0 && c.writer) {
            LaneSave &sv = P.save[gl];
            for (int i = 0; i < MAXM; i++) {
                sv.gb[i] = gb[i];
                for (int j = 0; j < MAXM; j++) sv.G[i][j] = G[i][j];
            }
            sv.tol = (double) tol;
            sv.lastErr = (double) lastErr;
            sv.wLast = (double) wLast;
            sv.zeta = (double) zeta;
            sv.w = (double) w;
            sv.wSafe = (double) wSafe;
            sv.iters = active ? it - it0 : iters;
            sv.k0 = k0; sv.k1 = k1; sv.k2 = k2; sv.k2bt = k2bt; sv.k3 = k3; sv.nT = nT; sv.nEll = nEll;
            sv.status = status;
            sv.active = active ? 1 : 0;
            sv.initFlag = initFlag ? 1 : 0;
            sv.it0 = it0;
        }
    } else if (threadIdx.x == 0) {
        gs->finished = 1;
    }
    if (active) iters = it - it0;
    __syncthreads();
    if (c.wave == 0 && c.writer && real) {
        Out &o = outs[gl];
        o.status = status;
        o.iters = iters;
        o.err = (double) lastErr;
        o.tol = (double) tol;
        o.w = (double) wLast;
        o.k0 = k0;
        o.k1 = k1;
        o.k2 = k2;
        o.k2bt = k2bt;
        o.k3 = k3;
        o.nT = nT;
        o.nEll = nEll;
        for (int i = 0; i < NUM_PHASES; i++) o.ticks[i] = phaseAcc[i];
    }
}

}  // namespace spk
