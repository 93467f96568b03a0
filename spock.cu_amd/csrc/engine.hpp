// Device-side data model of the fused SPOCK engine (shared by the kernels and the host glue).
#pragma once
#include <hip/hip_runtime.h>

#include "gridbar.hpp"

namespace spk {

// Per-node factor table on the device: entry for node n starts at data + idx[n] * rows * cols (tab()).
template <typename T>
struct DTab {
    const T *data = nullptr;
    const int *idx = nullptr;
    int rows = 0, cols = 0;
};

// A pointer every lane holds the same value of, moved to scalar registers: loads through it
// become scalar loads (needed inside non-inlined functions, whose arguments arrive per lane).
template <typename T>
__device__ __forceinline__ T *uniformPtr(T *p) {
    const unsigned long long v = reinterpret_cast<unsigned long long>(p);
    const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned) v);
    const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned) (v >> 32));
    return reinterpret_cast<T *>(((unsigned long long) hi << 32) | lo);
}

// Constant address space: the descriptor, the tree arrays and the factor tables are never written
// while a solve runs, and wave-uniform reads through such pointers become scalar loads.
#define SPK_CONST __attribute__((address_space(4)))
#define SPK_GLOBAL __attribute__((address_space(1)))
#define SPK_LDS __attribute__((address_space(3)))
template <typename T>
using CP = const SPK_CONST T *;
template <typename T>
using GP = SPK_GLOBAL T *;

template <typename T>
__device__ __forceinline__ CP<T> cst(const T *p) {
    return (CP<T>) p;
}

// Node n's entry of a per-node table, as a constant-space pointer.
template <typename T>
__device__ __forceinline__ CP<T> tab(const SPK_CONST DTab<T> &t, int n) {
    return cst(t.data) + (size_t) cst(t.idx)[n] * t.rows * t.cols;
}

// The same table packed for the tile engine's products: per distinct matrix and block of 64 rows,
// [16-column group][16-row tile][lane][4], lane l holding M[16 t + l % 16][16 k + 4 s + l / 16] at
// position s, zero past the matrix, with 1, 2 or 4 row tiles in a block of up to 16, 32 or 64 rows.
// `stride` entries per matrix.
template <typename T>
struct PTab {
    const T *data = nullptr;
    const int *idx = nullptr;
    int rows = 0, cols = 0, stride = 0;
};

// One solve instance: problem sizes, device tables, state buffers and options.
template <typename T>
struct Inst {
    int N, nl, nlf, S, E, nx, nu, yD, nD, ncost, lcost, ncon, lcon, con3, con5;
    long oU, oX, oY, oT, oS, sPrim, oI, oII, oIII, oIV, oV, oVI, sDual, sIter;
    T gamma, gammaRecip;
    const int *anc, *chFrom, *numCh, *stageFrom, *stageTo;
    DTab<T> BTr, AB, K, KTr, ABKTr, APB, cholL, cholU, RtInv, NN, b, sQ, sR, q, r, trans, lsQ, lq, ltrans;
    DTab<T> nG, nLB, nUB, lG, lLB, lUB, nGT, lGT;
    DTab<T> e, Pe;  // affine dynamics (zero tables when linear)
    int affine;
    // state (iterate-sized unless noted)
    T *z, *zPrev, *cand, *backup, *res, *resPrev, *dir, *dirS;
    T *hS, *hY;    // Anderson histories (iterate and residual differences), andBuff columns each
    T *qd, *dd;    // dynamics sweep intermediates: nx*N and nu*nl
    const T *x0s;  // scaled initial state (nx)
    // options
    T tolAbs, tolRel;  // already multiplied by min(scaling) when preconditioned
    T tolFixed;        // > 0: accept when the error is <= tolFixed from the first check on
    long maxIters;
    int maxInner, andBuff, checkPeriod, method, warm, lsMethod, dynInverse;
    double maxTicks;  // wall-clock cap in device ticks (0 = none)
    T *gpart;         // grid mode: 2 x GRID_MAXK x GRID_MAXWG reduction partials
    int chain;        // grid mode: from this stage on node k of a stage is the only child of node k of the one before
    unsigned *gbar;   // grid mode: the barrier's GRID_BAR_WORDS words, zero before the first launch
    // debug trace (enableDebug, src/cache.cuh:947-959); dbg == nullptr: off.  One record of
    // DBG_WORDS doubles per error check, at most dbgCap; dbgE (sPrim) carries err0's running
    // vector from check to check and from solve to solve
    double *dbg;
    long dbgCap;
    T *dbgE;
    int slot;  // this instance's index in the batch (its result record); descriptors may be reordered
};

// A debug record: outer iteration, calls to L and L* so far, err0, err1, err2, err3.
constexpr int DBG_WORDS = 6;

// Grid mode limits: values per grid reduction and workgroups per cooperative launch.
constexpr int GRID_MAXK = 16;
constexpr int GRID_MAXWG = 1024;
static_assert(GRID_MAXWG / GRID_GROUPS < GRID_BAR_ROUND, "arrivals at one counter of the grid barrier");

// Block-interleaved layout of a region of `rows` rows: instances are grouped in blocks of w (64
// for the lane engine, 16 for the tile engine) and each block stores rows x w words contiguously,
// element e of instance b at ((b / w) * rows + e) * w + b % w.
__host__ __device__ inline size_t laneIndex(long rows, long e, long b, long w = 64) {
    return ((size_t) (b / w) * rows + e) * w + (b % w);
}

// SuperMann state of one lane kept between the launches of a chunked solve.
struct LaneSave {
    double G[4][4], gb[4];
    double tol, lastErr, wLast, zeta, w, wSafe;
    long iters, k0, k1, k2, k2bt, k3, nT, nEll;
    long it0;  // workgroup iteration at which this lane's current solve started
    int status, active, initFlag, pad;
};

// Per-workgroup state of a chunked solve: buffer roles (indices of z, cand, zPrev, res, resPrev,
// backup into work[0..5]), Anderson ring head, whether the workgroup's solve has ended (its
// results are final and a resume returns at once), next outer iteration and device ticks spent.
struct LaneGroupSave {
    int roles[6];
    int head, finished;
    long it, ticks;
};

// Many instances of ONE problem in the block-interleaved layout: a wave whose lanes are the 64
// instances of one block moves 64 consecutive words per access, a workgroup's state is one
// contiguous slab per region, and the factor tables are read at wave-uniform addresses (scalar
// loads shared by the wave).
template <typename T>
struct LaneInst {
    int N, nl, nlf, S, E, nx, nu, yD, nD, ncost, lcost, ncon, lcon, con3, con5;
    long oU, oX, oY, oT, oS, sPrim, oI, oII, oIII, oIV, oV, oVI, sDual, sIter;
    T gamma, gammaRecip;
    const int *anc, *chFrom, *numCh, *stageFrom, *stageTo;
    DTab<T> BTr, AB, K, KTr, ABKTr, APB, cholL, cholU, RtInv, NN, b, sQ, sR, q, r, trans, lsQ, lq, ltrans;
    DTab<T> nG, nLB, nUB, lG, lLB, lUB, nGT, lGT;
    DTab<T> e, Pe;  // affine dynamics (zero tables when linear)
    int affine;
    // tile engine: packed factors (GTx, GTu: the state and the input rows of nGT)
    PTab<T> pBTr, pAB, pK, pKTr, pABKTr, pAPB, pRtInv, pNN, psQ, psR, plsQ, pG, pGTx, pGTu, plG, plGT;
    long B;     // padded instance count (multiple of 64); a region of r rows holds r * B words
    int count;  // instances in use
    T *work[9];   // rotating roles z, cand, zPrev, res, resPrev, backup + cand2, dir, dirS
    T *zio, *rio; // accepted iterate and its residual (warm-start input, solve output)
    T *hS, *hY;   // Anderson rings, andBuff slots of sIter x B each
    T *qd, *dd;   // dynamics sweep intermediates (nx*N and nu*nl rows)
    const T *x0s; // scaled initial states (nx rows)
    const T *tolFixed;  // per-instance given tolerance (> 0), or nullptr
    T tolAbs, tolRel;
    long maxIters;
    int maxInner, andBuff, checkPeriod, method, warm;
    double maxTicks;
    long chunkIters;          // > 0: stop after this many outer iterations, state saved for a resume
    double chunkTicks;        // > 0 (chunked solves): also stop, after at least one outer iteration, once
                              // the launch has run this many wall-clock ticks
    int resume;               // 1: continue the saved solve
    LaneSave *save;           // B entries
    LaneGroupSave *gsave;     // B / 64 entries
};

// Phases timed inside the solve (wall_clock64 ticks, summed over the solve).
enum Phase { PH_ADJ = 0, PH_PROJ = 1, PH_DUAL = 2, PH_RES = 3, PH_ELL = 4, PH_ACOL = 5, PH_ALS = 6, PH_AAPPLY = 7,
             PH_LINE = 8, PH_OTHER = 9, NUM_PHASES = 10 };

struct Out {
    int status;
    int pad;
    long iters;
    double err, tol, w;
    long k0, k1, k2, k2bt, k3, nT, nEll;
    long ticks[NUM_PHASES];  // device wall-clock ticks spent per phase (thread 0's view)
    long nDbg;               // debug records written by the last solve
    long nonfinite;          // debug: first non-finite entry of the candidate (-1: none)
};

enum Method { METHOD_SPOCK = 0, METHOD_CP = 1 };
enum DevKinds { CON_NO_DEV = 0, CON_RECT_DEV = 1, CON_POLY_DEV = 2, COST_QUAD_DEV = 0, COST_QUADLIN_DEV = 1,
                COST_LIN_DEV = 2 };

// A linear cost's dual "projection" (src/costs.cuh:296-301: k_projectRectangle of
// src/definitions.cu:39-48 with lower bound -inf and the epigraph entry as upper bound): the cost
// entry is clamped to at most the epigraph entry, which is kept.  Not the Euclidean projection
// onto {c <= t}; restated as the reference computes it.
template <typename T>
__host__ __device__ __forceinline__ T projBelow(T c, T t) { return c >= t ? t : c; }
// ST_NONFINITE: debug mode found a non-finite candidate entry and stopped the solve, where the
// reference's isFinite throws (src/cache.cuh:52-62, :912)
enum Status { ST_NOTRUN = -1, ST_CONVERGED = 0, ST_OUTOFITER = 1, ST_OUTOFTIME = 2, ST_NONFINITE = 3 };

constexpr int MAXR = 4;  // row chunks of 64 per wave task (rows <= 256)
constexpr int MAXV = 4;  // vector chunks of 64 held in registers (length <= 256)

}  // namespace spk
