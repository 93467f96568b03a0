// Fused SPOCK engine for gfx950: one workgroup owns one problem instance and runs the
// whole SuperMann/Anderson solve (src/cache.cuh:1008-1132) inside a single launch.
// Grid mode: for one large tree, every workgroup of a cooperative launch works on the same
// instance; the work distribution below then spans the grid, barriers are grid barriers and
// reductions combine per-workgroup partials (in a fixed order, so every workgroup takes the
// same branch decisions).
//
// Work decomposition inside the workgroup: a "node task" is handled by one 64-lane
// wavefront with lanes over the rows of the node's blocks; stage-sequential sweeps are separated
// by workgroup barriers; iterate-wide passes are block-strided; reductions use
// cross-lane shuffles and an LDS combine in a fixed order (bitwise repeatable).
//
// Operator semantics follow the reference (file:line cited per function); outputs the
// reference leaves unwritten (t[0] of L*, the IV block of node 0 of L) are zero here.
#include "engine.hpp"

#include <hip/hip_runtime.h>
#include <math.h>

#include <utility>

#ifndef SPK_MAX_THREADS
#define SPK_MAX_THREADS 512
#endif

namespace spk {

// ------------------------------------------------------------------ wave primitives
__device__ __forceinline__ double bcastLane(double v, int src) {
    int lo = __double2loint(v), hi = __double2hiint(v);
    lo = __builtin_amdgcn_readlane(lo, src);
    hi = __builtin_amdgcn_readlane(hi, src);
    return __hiloint2double(hi, lo);
}

__device__ __forceinline__ float bcastLane(float v, int src) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), src));
}

template <typename T>
__device__ __forceinline__ T waveSum(T v) {
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

template <typename T>
__device__ __forceinline__ T waveMax(T v) {
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v = fmax(v, __shfl_xor(v, o, 64));
    return v;
}

// The descriptor is read through the constant address space (scalar loads, kept in scalar
// registers), the state through the global one: with the descriptor in LDS behind generic pointers
// every field was a flat load per lane, waited for on its own, and every branch on one an exec mask.
// Together with the unconditional loads and the shared code of mvChunk: 0.85 -> 0.33 ms per
// application of T on the 229-node FP64 instance with 32 workgroups, 0.25 -> 0.08 ms on the 31-node one.
template <typename T>
using IP = const SPK_CONST Inst<T> &;

template <typename T>
__device__ __forceinline__ GP<T> glb(T *p) {
    return (GP<T>) uniformPtr(p);
}

// Work distribution of a thread: tid/nt and wave/nw index the threads and waves that share one
// instance (the workgroup, or the whole grid in grid mode); ltid/lw/lnw are workgroup-local.
struct Tc {
    unsigned lane;
    unsigned row;  // the row of a node's blocks (of each 64) this lane holds
    int wave, nw, tid, nt;
    int ltid, lw, lnw;
    int grid;
    void *gpart;  // grid mode: two buffers of GRID_MAXK x GRID_MAXWG reduction partials
};

__device__ __forceinline__ Tc threadCtx(int grid = 0, void *gpart = nullptr) {
    Tc c;
    c.ltid = threadIdx.x;
    c.lw = __builtin_amdgcn_readfirstlane(c.ltid >> 6);
    c.lnw = blockDim.x >> 6;
    c.grid = __builtin_amdgcn_readfirstlane(grid);
    c.gpart = gpart;
    c.tid = c.grid ? (int) (blockIdx.x * blockDim.x + threadIdx.x) : c.ltid;
    c.nt = c.grid ? (int) (gridDim.x * blockDim.x) : (int) blockDim.x;
    c.lane = threadIdx.x & 63;
    c.row = 4 * (c.lane & 15) + (c.lane >> 4);  // rowOf
    c.wave = c.grid ? (int) blockIdx.x * c.lnw + c.lw : c.lw;
    c.nw = c.nt >> 6;
    return c;
}

// Grid reductions done so far by this workgroup; selects the partials buffer.
__device__ __forceinline__ SPK_LDS int *gridSeq() {
    __shared__ int seq;
    return (SPK_LDS int *) &seq;
}

// The grid barrier of this workgroup; its first thread alone uses it.
struct GridBar {
    unsigned long long mem;
    unsigned passed;  // value of the flags after the last barrier
};
__device__ __forceinline__ SPK_LDS GridBar *gridBar() {
    __shared__ GridBar bar;
    return (SPK_LDS GridBar *) &bar;
}

// Before a kernel's first barrier or reduction.
__device__ __forceinline__ void startGrid(const Tc &c, unsigned *gbar) {
    if (c.ltid == 0) {
        *gridSeq() = 0;
        if (c.grid) {
            GridMem mem{gbar};
            gridBar()->mem = (unsigned long long) gbar;
            gridBar()->passed = gridPassed(mem, blockIdx.x);
        }
    }
    __syncthreads();
}

// Barrier over all workgroups of the (cooperative, so co-resident) grid.  The stages of T are a few
// microseconds of work between two of them, so this is most of a large tree's time.  What bounds it are the trips
// to memory and the accesses to one address, one after the other; workgroups therefore arrive in groups (by
// index, so mostly of one XCD), the last of each group arrives at the root, and each group waits on a flag of
// its own.  With 1,024 words written by each workgroup and read by another: 32 / 128 / 256 workgroups 3.4 / 4.9 /
// 8.5 us; one counter that all add to and poll 2.7 / 7.2 / 13.7; cooperative_groups' grid barrier 5.6 / 15.8 / 29.2.
__device__ __noinline__ void gridBarrier() {
    // every wave's writes have left before the workgroup's first thread releases them to the other XCDs
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_s_waitcnt(0);
    __builtin_amdgcn_s_barrier();
    if (threadIdx.x == 0) {
        GridMem mem{reinterpret_cast<unsigned *>(gridBar()->mem)};
        gridBar()->passed = gridPass(mem, blockIdx.x, gridDim.x, gridBar()->passed);
    }
    __syncthreads();
}

// Barrier over the threads that share the instance.
__device__ __forceinline__ void sync(const Tc &c) {
    if (c.grid) gridBarrier();
    else __syncthreads();
}

// Grid mode: combine the workgroup values v[0..K) of every workgroup.  Each workgroup publishes its
// values, then every wave reads all partials lane-strided and reduces them with the same shuffle
// tree, so all threads of the grid hold bitwise identical results.  Two partial buffers alternate:
// a workgroup can only start overwriting one after every workgroup passed the barrier of the
// reduction in between, which is after its reads of the same buffer.
template <typename T, int K, bool MAX>
__device__ __forceinline__ void gridCombine(T (&v)[K], const Tc &c) {
    static_assert(K <= GRID_MAXK, "too many values per grid reduction");
    const int seq = *gridSeq();  // advanced below, behind the grid barrier; read again behind a block barrier
    T *part = static_cast<T *>(c.gpart) + (size_t) (seq & 1) * GRID_MAXK * GRID_MAXWG;
    if (c.ltid == 0)
#pragma unroll
        for (int i = 0; i < K; i++) part[i * GRID_MAXWG + blockIdx.x] = v[i];
    gridBarrier();
    if (c.ltid == 0) *gridSeq() = seq + 1;
    const int nb = gridDim.x;
#pragma unroll
    for (int i = 0; i < K; i++) {
        T a = T(0);
        for (int b = c.lane; b < nb; b += 64) {
            const T p = part[i * GRID_MAXWG + b];
            a = MAX ? fmax(a, p) : a + p;
        }
        v[i] = MAX ? waveMax(a) : waveSum(a);
    }
}

// Per-phase wall-clock accounting; mark() is called right after a workgroup barrier so the
// interval covers the whole phase.
struct PhaseClock {
    long last;
    long acc[NUM_PHASES];
    __device__ void start() {
        last = wall_clock64();
        for (int i = 0; i < NUM_PHASES; i++) acc[i] = 0;
    }
    __device__ __forceinline__ void mark(int ph) {
        const long t = wall_clock64();
        acc[ph] += t - last;
        last = t;
    }
};

template <typename T, int K>
__device__ __forceinline__ void zero(T (&a)[K]) {
#pragma unroll
    for (int i = 0; i < K; i++) a[i] = T(0);
}

// v[c] holds element row + 64 c of a vector of length len (0 beyond)
template <typename T, int V, typename F>
__device__ __forceinline__ void loadV(T (&v)[V], int len, unsigned row, F f) {
#pragma unroll
    for (int c = 0; c < V; c++) {
        const unsigned k = row + 64 * c;
        v[c] = T(0);
        if (64 * c < len && k < (unsigned) len) v[c] = f(k);
    }
}

template <typename T, int V, typename P>
__device__ __forceinline__ void loadPtr(T (&v)[V], P p, int len, unsigned row) {
    loadV(v, len, row, [&](unsigned k) -> T { return p[k]; });
}

// ------------------------------------------------------------------ products of a node
// Rows of a node's blocks sit in lanes by rowOf(): lane 16 g + q holds row 4 q + g of each 64.  A
// product y += M v (M column major, up to 64 columns) then runs as four column groups of 16 lanes:
// lane 16 g + q loads rows 4 q .. 4 q + 3 of columns g, g + 4, ... (16 bytes a load in FP32, two such
// loads in FP64), the vector entry it needs, v[4 s + g], is in lane s of its own 16 (a row broadcast),
// and the four groups' sums meet in two swaps between lane rows that leave row 4 q + g in lane
// 16 g + q again.  This is bound by instruction issue and latency, so what counts is that a step of
// four columns is one or two loads, a broadcast and four multiply-adds (one column at a time with
// lanes over rows: 15 instructions a column; T of the 229-node FP64 instance in one workgroup
// 1.22 ms, now 0.75).  All loads of a chunk are issued before the first is used and none is
// conditional: rows past the end repeat the last four, and up to 7 columns past the end are read
// against v = 0 (the tables are padded for it) before the remaining blocks of 8 columns are skipped.
__device__ __forceinline__ unsigned rowOf(unsigned lane) { return 4 * (lane & 15) + (lane >> 4); }
__device__ __forceinline__ int laneOf(int row) { return 16 * (row & 3) + (row >> 2); }  // row < 64

template <int S>
__device__ __forceinline__ float rowBcast(float v) {  // lane S of each 16
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x150 + S, 0xf, 0xf, true));
}
template <int S>
__device__ __forceinline__ double rowBcast(double v) {
    return __longlong_as_double(__builtin_amdgcn_update_dpp(0LL, __double_as_longlong(v), 0x150 + S, 0xf, 0xf, true));
}

// Four consecutive rows of a column, at element alignment.
template <typename T>
struct Quad;
template <>
struct Quad<float> {
    typedef float V __attribute__((ext_vector_type(4), aligned(4)));
    V a;
    __device__ __forceinline__ void load(CP<float> p) { a = *(const SPK_CONST V *) p; }
    __device__ __forceinline__ float get(int i) const { return a[i]; }
};
template <>
struct Quad<double> {
    typedef double V __attribute__((ext_vector_type(2), aligned(8)));
    V a, b;
    __device__ __forceinline__ void load(CP<double> p) {
        a = *(const SPK_CONST V *) p;
        b = *(const SPK_CONST V *) (p + 2);
    }
    __device__ __forceinline__ double get(int i) const { return i < 2 ? a[i] : b[i - 2]; }
};

// a + b where both hold values of both 32-lane halves (16-lane rows): lanes of the lower half (even
// rows) get the sum of a over the pair, the others the sum of b.
__device__ __forceinline__ float halfSum32(float a, float b) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float halfSum16(float a, float b) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ double halfSum32(double a, double b) {
    const auto lo = __builtin_amdgcn_permlane32_swap(__double2loint(a), __double2loint(b), false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap(__double2hiint(a), __double2hiint(b), false, false);
    return __hiloint2double(hi[0], lo[0]) + __hiloint2double(hi[1], lo[1]);
}
__device__ __forceinline__ double halfSum16(double a, double b) {
    const auto lo = __builtin_amdgcn_permlane16_swap(__double2loint(a), __double2loint(b), false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap(__double2hiint(a), __double2hiint(b), false, false);
    return __hiloint2double(hi[0], lo[0]) + __hiloint2double(hi[1], lo[1]);
}

template <typename T, int RR>
struct RowVals {
    T a[RR];
};

// p[rc][i] += the columns 4 (S0 + s) + g, s < NS, of four rows, of a chunk with `cols` columns.
template <typename T, int RR, int S0, int NS>
__device__ __forceinline__ void mvSteps(T (&p)[RR][4], CP<T> M, const unsigned (&off)[RR], int ld, int cols, T v) {
    Quad<T> m[NS][RR];
#pragma unroll
    for (int s = 0; s < NS; s += 2) {
        if (4 * (S0 + s) < cols) {
#pragma unroll
            for (int u = s; u < s + 2; u++) {
                CP<T> col = M + (size_t) (4 * (S0 + u)) * ld;
#pragma unroll
                for (int rc = 0; rc < RR; rc++) m[u][rc].load(col + off[rc]);
            }
        }
    }
    [&]<int... B>(std::integer_sequence<int, B...>) {
        ([&] {
            if (4 * (S0 + 2 * B) < cols) {
                const T x0 = rowBcast<S0 + 2 * B>(v), x1 = rowBcast<S0 + 2 * B + 1>(v);
#pragma unroll
                for (int rc = 0; rc < RR; rc++) {
#pragma unroll
                    for (int i = 0; i < 4; i++) p[rc][i] += m[2 * B][rc].get(i) * x0;
#pragma unroll
                    for (int i = 0; i < 4; i++) p[rc][i] += m[2 * B + 1][rc].get(i) * x1;
                }
            }
        }(), ...);
    }(std::make_integer_sequence<int, NS / 2>{});
}

// acc + M v over one chunk of up to 64 columns, RR chunks of 64 rows.  Never inlined: with a copy of
// this code at each of its call sites the phases of a solve missed the instruction cache all the time
// (229-node FP64 instance, 32 workgroups, one column at a time: 1.6 ms of tree sweeps per application
// of T inlined, 0.28 ms called).
template <typename T, int RR>
__device__ __noinline__ RowVals<T, RR> mvChunk(RowVals<T, RR> acc, const T *Mp, int rows, int ldIn, int colsIn, T v) {
    CP<T> M = cst(uniformPtr(Mp));
    const int ld = __builtin_amdgcn_readfirstlane(ldIn), cols = __builtin_amdgcn_readfirstlane(colsIn);
    const unsigned lane = threadIdx.x & 63, q = lane & 15, g = lane >> 4;
    unsigned off[RR];
    T p[RR][4];
#pragma unroll
    for (int rc = 0; rc < RR; rc++) {
        off[rc] = min(64 * rc + 4 * q, ((unsigned) rows - 1) & ~3u) + g * ld;
#pragma unroll
        for (int i = 0; i < 4; i++) p[rc][i] = T(0);
    }
    // up to 128 registers of matrix entries in flight in FP64
    if constexpr (RR == 1) {
        mvSteps<T, RR, 0, 16>(p, M, off, ld, cols, v);
    } else if constexpr (RR == 2) {
        mvSteps<T, RR, 0, 8>(p, M, off, ld, cols, v);
        if (32 < cols) mvSteps<T, RR, 8, 8>(p, M, off, ld, cols, v);
    } else {
        mvSteps<T, RR, 0, 4>(p, M, off, ld, cols, v);
        if (16 < cols) mvSteps<T, RR, 4, 4>(p, M, off, ld, cols, v);
        if (32 < cols) mvSteps<T, RR, 8, 4>(p, M, off, ld, cols, v);
        if (48 < cols) mvSteps<T, RR, 12, 4>(p, M, off, ld, cols, v);
    }
#pragma unroll
    for (int rc = 0; rc < RR; rc++)
        acc.a[rc] += halfSum16(halfSum32(p[rc][0], p[rc][2]), halfSum32(p[rc][1], p[rc][3]));
    return acc;
}

template <typename T, int RR, int R, int V>
__device__ __forceinline__ void mvRows(T (&acc)[R], CP<T> M, int rows, int ld, int cols, const T (&v)[V]) {
    RowVals<T, RR> a;
#pragma unroll
    for (int rc = 0; rc < RR; rc++) a.a[rc] = acc[rc];
#pragma unroll
    for (int vc = 0; vc < V; vc++)
        if (64 * vc < cols)
            a = mvChunk<T, RR>(a, (const T *) (M + (size_t) (64 * vc) * ld), rows, ld, min(64, cols - 64 * vc), v[vc]);
#pragma unroll
    for (int rc = 0; rc < RR; rc++) acc[rc] = a.a[rc];
}

// acc[rc] (row rowOf(lane) + 64 rc) += sum_{c < cols} M[row + c * ld] * v(c), M column major, v 0
// beyond its length.
template <typename T, int R, int V>
__device__ __forceinline__ void mvAcc(T (&acc)[R], CP<T> M, int rows, int ld, int cols, const T (&v)[V]) {
    if constexpr (R == 1) {
        mvRows<T, 1>(acc, M, rows, ld, cols, v);
    } else {
        if (rows <= 64) mvRows<T, 1>(acc, M, rows, ld, cols, v);
        else if (rows <= 128) mvRows<T, 2>(acc, M, rows, ld, cols, v);
        else mvRows<T, 4>(acc, M, rows, ld, cols, v);
    }
}

// Sum of K per-thread values over the workgroup, identical result in every thread.
template <typename T, int K>
__device__ __forceinline__ void blockSum(T (&v)[K], SPK_LDS T *lds, const Tc &c) {
#pragma unroll
    for (int i = 0; i < K; i++) v[i] = waveSum(v[i]);
    if (c.lane == 0)
#pragma unroll
        for (int i = 0; i < K; i++) lds[i * 32 + c.lw] = v[i];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < K; i++) {
        T s = T(0);
        for (int w = 0; w < c.lnw; w++) s += lds[i * 32 + w];
        v[i] = s;
    }
    __syncthreads();
    if (c.grid) gridCombine<T, K, false>(v, c);
}

template <typename T>
__device__ __forceinline__ T blockMax(T v, SPK_LDS T *lds, const Tc &c) {
    v = waveMax(v);
    if (c.lane == 0) lds[c.lw] = v;
    __syncthreads();
    T s = T(0);
    for (int w = 0; w < c.lnw; w++) s = fmax(s, lds[w]);
    __syncthreads();
    if (c.grid) {
        T a[1] = {s};
        gridCombine<T, 1, true>(a, c);
        s = a[0];
    }
    return s;
}

// ------------------------------------------------------------------ projections
// Box projection in the arithmetic form of src/definitions.cu:38-52.
template <typename T>
__device__ __forceinline__ T projBox(T v, T lb, T ub) {
    const int lower = (v <= lb), upper = (v >= ub);
    const T lbi = isinf(lb) ? T(0) : T(lower) * lb;
    const T ubi = isinf(ub) ? T(0) : T(upper) * ub;
    return v * T(1 - lower) * T(1 - upper) + lbi + ubi;
}

// f(rc, r) for every row r = row + 64 rc < rows of this row.
template <int R, typename F>
__device__ __forceinline__ void eachRow(int rows, unsigned row, F f) {
#pragma unroll
    for (int rc = 0; rc < R; rc++) {
        const unsigned r = row + 64 * rc;
        if (64 * rc < rows && r < (unsigned) rows) f(rc, r);
    }
}

// ------------------------------------------------------------------ L* per node
// src/operator.cuh:63-82; src/costs.cuh:162-195 (quadratic), :418-458 (quadratic+linear);
// src/constraints.cuh:171-191 (rectangle), :265-286 (polyhedron).
template <typename T, int R>
struct AdjOut {
    T x[R];  // rows nx
    T u[R];  // rows nu (nonleaf only)
    T y;        // row < yD (nonleaf only)
    T s, t;     // uniform scalars
};

template <typename T, int R, int V>
__device__ __forceinline__ void adjNode(IP<T> P, GP<T> dual, int n, unsigned row, AdjOut<T, R> &o) {
    const int nx = P.nx, nu = P.nu, nxu = nx + nu, d4 = nxu + 2;
    zero(o.x);
    zero(o.u);
    o.y = T(0);
    o.s = T(0);
    o.t = T(0);
    T v[V], w[R];
    if (n < P.nl) {
        const T II = dual[P.oII + n];
        o.s = II;
        if (row < (unsigned) P.yD) o.y = (dual + (P.oI + (long) n * P.yD))[row] - tab(P.b, n)[row] * II;
        GP<T> d3 = dual + (P.oIII + (long) n * P.con3);
        if (P.ncon == CON_RECT_DEV) {
            eachRow<R>(nx, row, [&](int rc, unsigned r) { o.x[rc] = d3[r]; });
            GP<T> d3u = d3 + nx;
            eachRow<R>(nu, row, [&](int rc, unsigned r) { o.u[rc] = d3u[r]; });
        } else if (P.ncon == CON_POLY_DEV) {
            loadPtr(v, d3, P.con3, row);
            CP<T> GT = tab(P.nGT, n);
            mvAcc(o.x, GT, nx, nxu, P.con3, v);
            mvAcc(o.u, GT + nx, nu, nxu, P.con3, v);
        }
        const int c0 = cst(P.chFrom)[n], nc = cst(P.numCh)[n];
#pragma unroll 1
        for (int ci = 0; ci < nc; ci++) {  // children accumulate in order (src/costs.cuh:172-177)
            const int j = c0 + ci;
            if (P.ncost == COST_LIN_DEV) {  // x_i += q_j sum_j, u_i += r_j sum_j (src/costs.cuh:274-285)
                const T sj = dual[P.oIV + j];
                CP<T> qj = tab(P.q, j), rj = tab(P.r, j);
                eachRow<R>(nx, row, [&](int rc, unsigned r) { o.x[rc] += qj[r] * sj; });
                eachRow<R>(nu, row, [&](int rc, unsigned r) { o.u[rc] += rj[r] * sj; });
                continue;
            }
            GP<T> iv = dual + (P.oIV + (long) j * d4);
            const T a = iv[nxu], bb = iv[nxu + 1];
            loadPtr(v, iv, nx, row);
            zero(w);
            mvAcc(w, tab(P.sQ, j), nx, nx, nx, v);
            if (P.ncost == COST_QUADLIN_DEV) {
                CP<T> qj = tab(P.q, j);
                eachRow<R>(nx, row, [&](int rc, unsigned r) { w[rc] = w[rc] - T(0.5) * qj[r] * a - T(0.5) * qj[r] * bb; });
            }
#pragma unroll
            for (int rc = 0; rc < R; rc++) o.x[rc] += w[rc];
            loadPtr(v, iv + nx, nu, row);
            zero(w);
            mvAcc(w, tab(P.sR, j), nu, nu, nu, v);
            if (P.ncost == COST_QUADLIN_DEV) {
                CP<T> rj = tab(P.r, j);
                eachRow<R>(nu, row, [&](int rc, unsigned r) { w[rc] = w[rc] - T(0.5) * rj[r] * a - T(0.5) * rj[r] * bb; });
            }
#pragma unroll
            for (int rc = 0; rc < R; rc++) o.u[rc] += w[rc];
        }
    } else {
        const int l = n - P.nl;
        GP<T> d5 = dual + (P.oV + (long) l * P.con5);
        if (P.lcon == CON_RECT_DEV) {
            eachRow<R>(nx, row, [&](int rc, unsigned r) { o.x[rc] = d5[r]; });
        } else if (P.lcon == CON_POLY_DEV) {
            loadPtr(v, d5, P.con5, row);
            mvAcc(o.x, tab(P.lGT, l), nx, nx, P.con5, v);
        }
        if (P.lcost == COST_LIN_DEV) {  // x_l += q sum_l, s_l = set_l (src/costs.cuh:289-292)
            const T sl = dual[P.oVI + l];
            CP<T> lq = tab(P.lq, l);
            eachRow<R>(nx, row, [&](int rc, unsigned r) { o.x[rc] += lq[r] * sl; });
            o.s = dual[P.oVI + P.nlf + l];
        } else {
            GP<T> vi = dual + (P.oVI + (long) l * (nx + 2));
            const T a = vi[nx], bb = vi[nx + 1];
            loadPtr(v, vi, nx, row);
            zero(w);
            mvAcc(w, tab(P.lsQ, l), nx, nx, nx, v);
#pragma unroll
            for (int rc = 0; rc < R; rc++) o.x[rc] += w[rc];
            if (P.lcost == COST_QUADLIN_DEV) {
                CP<T> lq = tab(P.lq, l);
                eachRow<R>(nx, row,
                           [&](int rc, unsigned r) { o.x[rc] = o.x[rc] - T(0.5) * lq[r] * a - T(0.5) * lq[r] * bb; });
            }
            o.s = (a + bb) * T(0.5);
        }
    }
    if (P.ncost == COST_LIN_DEV) {
        o.t = dual[P.oIV + P.N + n];  // t <- set, every node (src/costs.cuh:286)
    } else if (n >= 1) {
        GP<T> iv = dual + (P.oIV + (long) n * d4);
        o.t = (iv[nxu] + iv[nxu + 1]) * T(0.5);
    }
}

// ------------------------------------------------------------------ L per node
// src/operator.cuh:41-60; src/costs.cuh:126-160 (quadratic), :379-416 (quadratic+linear);
// src/constraints.cuh:158-169 (rectangle), :251-263 (polyhedron).
// pv(base, k): element base + k of the primal vector, base wave-uniform.
// The handler H receives each dual block of node n as register values:
//   blockI(n, yk (row < yD), IIval)
//   blockElem(dualIndexBase, vals, rows, lb table entry, ub table entry)  [III and V]
//   blockSoc(dualIndexBase, xs (rows nx), us (rows nu, may be 0 rows), h, transEntry)  [IV and VI]
template <typename T, int R, int V, typename PV, typename H>
__device__ __forceinline__ void opNode(IP<T> P, int n, unsigned row, PV pv, H &h) {
    const int nx = P.nx, nu = P.nu, nxu = nx + nu;
    T v[V], v2[V], acc[R], acc2[R];
    if (n < P.nl) {
        const long xn = P.oX + (long) n * nx, un = P.oU + (long) n * nu;
        // I and II
        const T yk = (row < (unsigned) P.yD) ? pv(P.oY + (long) n * P.yD, row) : T(0);
        const T bk = (row < (unsigned) P.yD) ? tab(P.b, n)[row] : T(0);
        const T by = waveSum(bk * yk);
        const T IIval = pv(P.oS + n, 0) - by;
        h.blockI(n, yk, IIval);
        // III
        if (P.ncon == CON_RECT_DEV) {
            zero(acc);
            zero(acc2);
            eachRow<R>(nx, row, [&](int rc, unsigned r) { acc[rc] = pv(xn, r); });
            eachRow<R>(nu, row, [&](int rc, unsigned r) { acc2[rc] = pv(un, r); });
            const long base = P.oIII + (long) n * P.con3;
            h.blockElem(base, acc, nx, tab(P.nLB, n), tab(P.nUB, n));
            h.blockElem(base + nx, acc2, nu, tab(P.nLB, n) + nx, tab(P.nUB, n) + nx);
        } else if (P.ncon == CON_POLY_DEV) {
            loadV(v, nx, row, [&](unsigned k) { return pv(xn, k); });
            loadV(v2, nu, row, [&](unsigned k) { return pv(un, k); });
            zero(acc);
            CP<T> G = tab(P.nG, n);
            mvAcc(acc, G, P.con3, P.con3, nx, v);
            mvAcc(acc, G + (size_t) P.con3 * nx, P.con3, P.con3, nu, v2);
            h.blockElem(P.oIII + (long) n * P.con3, acc, P.con3, tab(P.nLB, n), tab(P.nUB, n));
        }
    }
    // IV
    if (P.ncost == COST_LIN_DEV) {  // (sum_n, set_n) = (q_n' x_anc + r_n' u_anc, t_n), node 0: (0, t_0)
        T sum = T(0);              // (src/costs.cuh:261-267)
        if (n >= 1) {
            const int a = cst(P.anc)[n];
            CP<T> qn = tab(P.q, n), rn = tab(P.r, n);
            T pq = T(0), pr = T(0);
            eachRow<V>(nx, row, [&](int, unsigned k) { pq += qn[k] * pv(P.oX + (long) a * nx, k); });
            eachRow<V>(nu, row, [&](int, unsigned k) { pr += rn[k] * pv(P.oU + (long) a * nu, k); });
            sum = waveSum(pq) + waveSum(pr);
        }
        h.blockLin(P.oIV + n, P.oIV + P.N + n, sum, pv(P.oT + n, 0));
    } else {
        zero(acc);
        zero(acc2);
        T hv = T(0);
        if (n >= 1) {
            const int a = cst(P.anc)[n];
            loadV(v, nx, row, [&](unsigned k) { return pv(P.oX + (long) a * nx, k); });
            loadV(v2, nu, row, [&](unsigned k) { return pv(P.oU + (long) a * nu, k); });
            mvAcc(acc, tab(P.sQ, n), nx, nx, nx, v);
            mvAcc(acc2, tab(P.sR, n), nu, nu, nu, v2);
            hv = pv(P.oT + n, 0) * T(0.5);
            if (P.ncost == COST_QUADLIN_DEV) {
                CP<T> qn = tab(P.q, n), rn = tab(P.r, n);
                T pq = T(0), pr = T(0);
                eachRow<V>(nx, row, [&](int c, unsigned k) { pq += qn[k] * v[c]; });
                eachRow<V>(nu, row, [&](int c, unsigned k) { pr += rn[k] * v2[c]; });
                hv = hv + T(-0.5) * waveSum(pq);
                hv = hv + T(-0.5) * waveSum(pr);
            }
        }
        h.blockSoc(P.oIV + (long) n * (nxu + 2), acc, nx, acc2, nu, hv, tab(P.trans, n));
    }
    // V and VI
    if (n >= P.nl) {
        const int l = n - P.nl;
        const long xn = P.oX + (long) n * nx;
        loadV(v, nx, row, [&](unsigned k) { return pv(xn, k); });
        if (P.lcon == CON_RECT_DEV) {
            zero(acc);
            eachRow<R>(nx, row, [&](int rc, unsigned) { acc[rc] = v[rc]; });
            h.blockElem(P.oV + (long) l * P.con5, acc, nx, tab(P.lLB, l), tab(P.lUB, l));
        } else if (P.lcon == CON_POLY_DEV) {
            zero(acc);
            mvAcc(acc, tab(P.lG, l), P.con5, P.con5, nx, v);
            h.blockElem(P.oV + (long) l * P.con5, acc, P.con5, tab(P.lLB, l), tab(P.lUB, l));
        }
        if (P.lcost == COST_LIN_DEV) {  // (q' x_l, s_l) (src/costs.cuh:269-272)
            CP<T> lq = tab(P.lq, l);
            T pq = T(0);
            eachRow<V>(nx, row, [&](int c, unsigned k) { pq += lq[k] * v[c]; });
            h.blockLin(P.oVI + l, P.oVI + P.nlf + l, waveSum(pq), pv(P.oS + n, 0));
            return;
        }
        zero(acc);
        zero(acc2);
        mvAcc(acc, tab(P.lsQ, l), nx, nx, nx, v);
        T hs = pv(P.oS + n, 0) * T(0.5);
        if (P.lcost == COST_QUADLIN_DEV) {
            CP<T> lq = tab(P.lq, l);
            T pq = T(0);
            eachRow<V>(nx, row, [&](int c, unsigned k) { pq += lq[k] * v[c]; });
            hs = hs + T(-0.5) * waveSum(pq);
        }
        h.blockSoc(P.oVI + (long) l * (nx + 2), acc, nx, acc2, 0, hs, tab(P.ltrans, l));
    }
}

// ---------------------------------------------------------------- L handlers
// Raw store of L values into out (dual-local indices).
template <typename T, int R>
struct StoreL {
    IP<T> P;
    GP<T> out;
    unsigned row;
    __device__ __forceinline__ void blockI(int n, T yk, T IIval) {
        if (row < (unsigned) P.yD) (out + (P.oI + (long) n * P.yD))[row] = yk;
        if (row == 0) out[P.oII + n] = IIval;
    }
    __device__ __forceinline__ void blockElem(long base, const T (&a)[R], int rows, CP<T>, CP<T>) {
        GP<T> ob = out + base;
        eachRow<R>(rows, row, [&](int rc, unsigned r) { ob[r] = a[rc]; });
    }
    __device__ __forceinline__ void blockSoc(long base, const T (&xs)[R], int nxr, const T (&us)[R], int nur, T hv, CP<T>) {
        GP<T> ob = out + base;
        eachRow<R>(nxr, row, [&](int rc, unsigned r) { ob[r] = xs[rc]; });
        eachRow<R>(nur, row, [&](int rc, unsigned r) { (ob + nxr)[r] = us[rc]; });
        if (row == 0) {
            ob[nxr + nur] = hv;
            ob[nxr + nur + 1] = hv;
        }
    }
    __device__ __forceinline__ void blockLin(long eSum, long eSet, T sum, T set) {
        if (row == 0) {
            out[eSum] = sum;
            out[eSet] = set;
        }
    }
};

// Dual prox of the CP step (src/cache.cuh:770-789): a = L*gamma + z_d; w = a/gamma + c;
// cand_d = gamma (w - Pi(w)).  Pi: masked NNOC (src/risks.cuh:99-106, definitions.cu:430-443),
// NNOC (src/cones.cuh:134-137), box (src/constraints.cuh:70-74), SOC (src/projections.cuh:102-128).
template <typename T, int R>
struct ProxL {
    IP<T> P;
    GP<T> zd, cd;
    unsigned row;
    __device__ __forceinline__ T wOf(T Lv, T z, T trans) const { return (Lv * P.gamma + z) * P.gammaRecip + trans; }
    __device__ __forceinline__ void blockI(int n, T yk, T IIval) {
        if (row < (unsigned) P.yD) {
            const long base = P.oI + (long) n * P.yD;
            const T w = wOf(yk, (zd + base)[row], T(0));
            const int idx = ((int) row < 2 * cst(P.numCh)[n]) && (w < T(0));
            const T p = T(1 - idx) * w;
            (cd + base)[row] = (w - p) * P.gamma;
        }
        if (row == 0) {
            const long k = P.oII + n;
            const T w = wOf(IIval, zd[k], T(0));
            const T p = fmax(T(0), w);
            cd[k] = (w - p) * P.gamma;
        }
    }
    __device__ __forceinline__ void blockElem(long base, const T (&a)[R], int rows, CP<T> lb, CP<T> ub) {
        GP<T> zb = zd + base, cb = cd + base;
        eachRow<R>(rows, row, [&](int rc, unsigned r) {
            const T w = wOf(a[rc], zb[r], T(0));
            const T p = projBox(w, lb[r], ub[r]);
            cb[r] = (w - p) * P.gamma;
        });
    }
    __device__ __forceinline__ void blockSoc(long base, const T (&xs)[R], int nxr, const T (&us)[R], int nur, T hv,
                                             CP<T> tr) {
        T wx[R], wu[R];
        T ss = T(0);
        GP<T> zx = zd + base, zu = zx + nxr, zh = zu + nur, cx = cd + base, cu = cx + nxr, ch = cu + nur;
        CP<T> tu = tr + nxr, th = tu + nur;
#pragma unroll
        for (int rc = 0; rc < R; rc++) {
            const unsigned r = row + 64 * rc;
            wx[rc] = T(0);
            wu[rc] = T(0);
            if (64 * rc < nxr && r < (unsigned) nxr) {
                wx[rc] = wOf(xs[rc], zx[r], tr[r]);
                ss += wx[rc] * wx[rc];
            }
            if (64 * rc < nur && r < (unsigned) nur) {
                wu[rc] = wOf(us[rc], zu[r], tu[r]);
                ss += wu[rc] * wu[rc];
            }
        }
        const T w1 = wOf(hv, zh[0], th[0]);
        const T w2 = wOf(hv, zh[1], th[1]);
        ss = waveSum(ss) + w1 * w1;
        const T nrm = sqrt(ss), tl = w2;
        const int i1 = nrm <= tl;
        const int i2 = (nrm <= -tl) && !i1;
        const int i3 = !i1 && !i2;
        const T sc = (nrm + tl) / (T(2) * nrm + T(1 - i3));
        const T mult = T(1 - i2) * (T(i3) * sc + T(1 - i3));
        eachRow<R>(nxr, row, [&](int rc, unsigned r) { cx[r] = (wx[rc] - wx[rc] * mult) * P.gamma; });
        eachRow<R>(nur, row, [&](int rc, unsigned r) { cu[r] = (wu[rc] - wu[rc] * mult) * P.gamma; });
        if (row == 0) {
            const T p1 = w1 * mult;
            const int i1b = (1 - i2) * (1 - i3);
            const T p2 = T(i1b) * (w2 * T(1 - i2)) + T((1 - i1b) * (1 - i2)) * (T(i3) * (sc * nrm - T(1)) + T(1));
            ch[0] = (w1 - p1) * P.gamma;
            ch[1] = (w2 - p2) * P.gamma;
        }
    }
    // linear cost: the cost entry clamped to at most the epigraph entry, which is kept
    // (src/costs.cuh:296-301 with k_projectRectangle, lower bound -inf)
    __device__ __forceinline__ void blockLin(long eSum, long eSet, T sum, T set) {
        if (row == 0) {
            const T ws = wOf(sum, zd[eSum], T(0)), wt = wOf(set, zd[eSet], T(0));
            cd[eSum] = (ws - projBelow(ws, wt)) * P.gamma;
            cd[eSet] = (wt - wt) * P.gamma;
        }
    }
};

// Reduction handler for ell(y) = [L* y_d; L y_p]: accumulates sum x . (y - gamma ell) and
// max |y / gamma - ell| over the dual part (src/cache.cuh:722-734 and :917-931).
template <typename T, int R>
struct ReduceL {
    IP<T> P;
    GP<T> xd, yd;  // dual parts of the partner and input vectors
    unsigned row;
    T dot, mx;
    __device__ __forceinline__ void acc(T x, T y, T ell) {
        dot += x * (ell * (-P.gamma) + y);
        mx = fmax(mx, fabs(y * P.gammaRecip - ell));
    }
    __device__ __forceinline__ void blockI(int n, T yk, T IIval) {
        const long base = P.oI + (long) n * P.yD, k = P.oII + n;
        if (row < (unsigned) P.yD) acc((xd + base)[row], (yd + base)[row], yk);
        if (row == 0) acc(xd[k], yd[k], IIval);
    }
    __device__ __forceinline__ void blockElem(long base, const T (&a)[R], int rows, CP<T>, CP<T>) {
        GP<T> xb = xd + base, yb = yd + base;
        eachRow<R>(rows, row, [&](int rc, unsigned r) { acc(xb[r], yb[r], a[rc]); });
    }
    __device__ __forceinline__ void blockSoc(long base, const T (&xs)[R], int nxr, const T (&us)[R], int nur, T hv, CP<T>) {
        GP<T> xx = xd + base, yx = yd + base, xu = xx + nxr, yu = yx + nxr, xh = xu + nur, yh = yu + nur;
#pragma unroll
        for (int rc = 0; rc < R; rc++) {
            const unsigned r = row + 64 * rc;
            if (64 * rc < nxr && r < (unsigned) nxr) acc(xx[r], yx[r], xs[rc]);
            if (64 * rc < nur && r < (unsigned) nur) acc(xu[r], yu[r], us[rc]);
        }
        if (row == 0) {
            acc(xh[0], yh[0], hv);
            acc(xh[1], yh[1], hv);
        }
    }
    __device__ __forceinline__ void blockLin(long eSum, long eSet, T sum, T set) {
        if (row == 0) {
            acc(xd[eSum], yd[eSum], sum);
            acc(xd[eSet], yd[eSet], set);
        }
    }
};

// ---------------------------------------------------------------- T phases
// modifyPrimal + proxRootS (src/cache.cuh:748-753, 639-642): cand_p = z_p - gamma L*(z_d); s_0 -= gamma.
// Leaf tasks also seed the dynamics sweep with q_leaf = -xbar_leaf (src/dynamics.cuh:79-81).
template <typename T, int R, int V>
__device__ __noinline__ void phaseAdjAxpy(const Inst<T> *Pp, int grid, T *zIn, T *candIn) {
    IP<T> P = *cst(uniformPtr(Pp));
    const Tc c = threadCtx(grid);
    GP<T> z = glb(zIn), cand = glb(candIn), qd = (GP<T>) P.qd;
    GP<T> zd = z + P.sPrim;
    const T g = -P.gamma;
    const int nx = P.nx, nu = P.nu;
    const unsigned row = c.row;
    for (int n = c.wave; n < P.N; n += c.nw) {
        AdjOut<T, R> o;
        adjNode<T, R, V>(P, zd, n, row, o);
        const long xn = P.oX + (long) n * nx, un = P.oU + (long) n * nu, yn = P.oY + (long) n * P.yD;
        eachRow<R>(nx, row, [&](int rc, unsigned r) {
            const T v = o.x[rc] * g + (z + xn)[r];
            (cand + xn)[r] = v;
            if (n >= P.nl) (qd + (long) n * nx)[r] = -v;
        });
        if (n < P.nl) {
            eachRow<R>(nu, row, [&](int rc, unsigned r) { (cand + un)[r] = o.u[rc] * g + (z + un)[r]; });
            if (row < (unsigned) P.yD) (cand + yn)[row] = o.y * g + (z + yn)[row];
        }
        if (row == 0) {
            T sv = o.s * g + z[P.oS + n];
            if (n == 0) sv -= P.gamma;
            cand[P.oS + n] = sv;
            cand[P.oT + n] = o.t * g + z[P.oT + n];
        }
    }
}

// Backward sweep step for node i (src/dynamics.cuh:85-139).  With affine dynamics the children's
// q enter as q_j + P_j e_j (src/dynamics.cuh:93-97).
template <typename T, int R, int V>
__device__ __forceinline__ void dynBackwardNode(IP<T> P, GP<T> cand, int i, int stage, unsigned row) {
    const int nx = P.nx, nu = P.nu;
    GP<T> ubar = cand + (P.oU + (long) i * nu);
    GP<T> xbar = cand + (P.oX + (long) i * nx);
    GP<T> qd = (GP<T>) P.qd;
    T v[V], w[R], acc[R];
    zero(acc);
    const int c0 = cst(P.chFrom)[i], nc = cst(P.numCh)[i];
    const bool mine = row < (unsigned) nu;
    auto loadQ = [&](int j) {
        GP<T> qj = qd + (long) j * nx;
        if (P.affine) {
            CP<T> pe = tab(P.Pe, j);
            loadV(v, nx, row, [&](unsigned k) -> T { return qj[k] + pe[k]; });
        } else {
            loadPtr(v, qj, nx, row);
        }
    };
    const T ub = mine ? ubar[row] : T(0);
#pragma unroll 1
    for (int ci = 0; ci < nc; ci++) {
        const int j = c0 + ci;
        loadQ(j);
        zero(w);
        mvAcc(w, tab(P.BTr, j), nu, nu, nx, v);
#pragma unroll
        for (int rc = 0; rc < R; rc++) acc[rc] = (ci == 0) ? w[rc] : acc[rc] + w[rc];
    }
    // d = R~^-1 (u - sum B'q) with R~ = L L': one matvec with the precomputed inverse, or the
    // two triangular solves of potrs
    T d = mine ? (-acc[0] + ub) : T(0);
    if (P.dynInverse) {
        T dvin[V], dout[R];
        zero(dvin);
        dvin[0] = d;
        zero(dout);
        mvAcc(dout, tab(P.RtInv, i), nu, nu, nu, dvin);
        d = mine ? dout[0] : T(0);
    } else {
        CP<T> L = tab(P.cholL, i);
        for (int k = 0; k < nu; k++) {
            const T dk = bcastLane(d, laneOf(k)) / L[k + (size_t) k * nu];
            if ((int) row == k) d = dk;
            else if ((int) row > k && mine) d -= L[row + (size_t) k * nu] * dk;
        }
        CP<T> U = tab(P.cholU, i);
        for (int k = nu - 1; k >= 0; k--) {
            const T dk = bcastLane(d, laneOf(k)) / U[k + (size_t) k * nu];
            if ((int) row == k) d = dk;
            else if ((int) row < k) d -= U[row + (size_t) k * nu] * dk;
        }
    }
    if (mine) ((GP<T>) P.dd + (long) i * nu)[row] = d;
    if (stage == 0) return;
    // q_i = sum_j (APB_j d_i + ABKTr_j q_j) + K_i'(d_i - u_i) - x_i
    T dv[V];
    zero(dv);
    dv[0] = d;
    zero(acc);
#pragma unroll 1
    for (int ci = 0; ci < nc; ci++) {
        const int j = c0 + ci;
        zero(w);
        mvAcc(w, tab(P.APB, j), nx, nx, nu, dv);
        if (nc > 1) loadQ(j);  // a single child's q is still in v
        mvAcc(w, tab(P.ABKTr, j), nx, nx, nx, v);
#pragma unroll
        for (int rc = 0; rc < R; rc++) acc[rc] = (ci == 0) ? w[rc] : acc[rc] + w[rc];
    }
    dv[0] = mine ? d - ub : T(0);
    zero(w);
    mvAcc(w, tab(P.KTr, i), nx, nx, nu, dv);
    eachRow<R>(nx, row, [&](int rc, unsigned r) { (qd + (long) i * nx)[r] = (acc[rc] + w[rc]) - xbar[r]; });
}

// Kernel projection for nonleaf node i (src/cache.cuh:650-676); padded child slots enter as 0.
template <typename T, int R, int V>
__device__ __forceinline__ void kernelNode(IP<T> P, GP<T> cand, int i, unsigned row) {
    const int yD = P.yD, E = P.E, nc = cst(P.numCh)[i], c0 = cst(P.chFrom)[i];
    // this row's entry of [y; t of the children; s of the children], or none
    const int k = (int) row;
    const bool isY = k < yD, isT = !isY && k < yD + E && k - yD < nc;
    const bool isS = k >= yD + E && k < yD + 2 * E && k - yD - E < nc;
    const bool any = isY || isT || isS;
    const long at = isY ? P.oY + (long) i * yD + k : isT ? P.oT + c0 + (k - yD) : P.oS + c0 + (k - yD - E);
    T vin[V], w[R];
    zero(vin);
    if (any) vin[0] = cand[at];
    zero(w);
    mvAcc(w, tab(P.NN, i), P.nD, P.nD, P.nD, vin);
    if (any) cand[at] = w[0];
}

// Forward rollout for node i (src/dynamics.cuh:144-173); affine dynamics add e_j to each child.  Member m of a
// team of g waves takes every g-th child; u is computed by all of them.
template <typename T, int R, int V>
__device__ __forceinline__ void dynForwardNode(IP<T> P, GP<T> cand, int i, unsigned row, int m = 0, int g = 1) {
    const int nx = P.nx, nu = P.nu;
    T xv[V], uv[V], w[R];
    GP<T> xi = cand + (P.oX + (long) i * nx);
    if (i == 0) {
        loadPtr(xv, cst(P.x0s), nx, row);
        if (m == 0) eachRow<V>(nx, row, [&](int c, unsigned k) { xi[k] = xv[c]; });
    } else {
        loadPtr(xv, xi, nx, row);
    }
    const bool mine = row < (unsigned) nu;
    const T di = mine ? ((GP<T>) P.dd + (long) i * nu)[row] : T(0);
    zero(w);
    mvAcc(w, tab(P.K, i), nu, nu, nx, xv);
    const T u = mine ? w[0] + di : T(0);
    if (m == 0 && mine) (cand + (P.oU + (long) i * nu))[row] = u;
    zero(uv);
    uv[0] = u;
    const int c0 = cst(P.chFrom)[i], nc = cst(P.numCh)[i];
#pragma unroll 1
    for (int ci = m; ci < nc; ci += g) {
        const int j = c0 + ci;
        CP<T> AB = tab(P.AB, j);
        zero(w);
        mvAcc(w, AB, nx, nx, nx, xv);
        mvAcc(w, AB + (size_t) nx * nx, nx, nx, nu, uv);
        CP<T> ej = tab(P.e, j);
        GP<T> xj = cand + (P.oX + (long) j * nx);
        eachRow<R>(nx, row, [&](int rc, unsigned r) { xj[r] = P.affine ? w[rc] + ej[r] : w[rc]; });
    }
}

// Stages with fewer nodes than half the waves (near the root, and all of them when a tree is spread over
// the device) give each node to a team of waves of one workgroup: a node's products are a chain of trips to memory,
// and a team takes its children side by side.  Team size: the largest power of two that fits the waves (and the
// slots below), or 1.  Projections of one T: 341 nodes, nx = 100, 4 children, FP64, 128 workgroups 253 -> 121 us;
// 1,365 nodes FP32, 256 workgroups 254 -> 138; 229 nodes, 9 of 11 stages without branching, 32 workgroups 167 -> 131.
template <int R>
constexpr int TEAM_ROUNDS = R == 1 ? 2 : 1;  // children of a member; wider nodes need fewer and keep LDS small

template <typename T, int R>
struct TeamLds {
    T bq[8][TEAM_ROUNDS<R>][64];      // B'q of a member's children
    T xq[8][TEAM_ROUNDS<R>][64 * R];  // their parts of q
};

template <int R>
__device__ __forceinline__ int teamSize(const Tc &c, int nodes, int children) {
    int g = 1;
    while (2 * g <= c.lnw && c.lnw % (2 * g) == 0 && nodes * 2 * g <= c.nw) g *= 2;
    return children <= TEAM_ROUNDS<R> * g ? g : 1;
}

// dynBackwardNode by member m of a team of g waves whose first is wave w0 of the workgroup: the same sums in the
// same order up to 64 states (beyond, a wave alone adds APB d to the first 64 columns of ABKTr q and then the others,
// a team adds the columns first).  With waves to spare (2 nc <= g) member nc + c takes the product with q of child c.  All waves
// of the workgroup come here together; i < 0: no node.
template <typename T, int R, int V>
__device__ __forceinline__ void dynBackwardTeam(IP<T> P, GP<T> cand, int i, int stage, unsigned row, int m, int g, int w0,
                                                SPK_LDS TeamLds<T, R> *lds) {
    constexpr int K = TEAM_ROUNDS<R>;
    const int nx = P.nx, nu = P.nu;
    const bool mine = row < (unsigned) nu;
    const int c0 = i < 0 ? 0 : cst(P.chFrom)[i], nc = i < 0 ? 0 : cst(P.numCh)[i];
    const bool split = 2 * nc <= g;
    GP<T> qd = (GP<T>) P.qd;
    T rq[K][R], w[R];
    const T ub = i >= 0 && mine ? (cand + (P.oU + (long) i * nu))[row] : T(0);
#pragma unroll
    for (int k = 0; k < K; k++) {
        zero(rq[k]);
        const int ci = split && m >= nc ? m - nc : m + k * g;
        if (ci >= nc || (split && k > 0)) continue;
        const int j = c0 + ci;
        GP<T> qj = qd + (long) j * nx;
        T v[V];
        if (P.affine) {
            CP<T> pe = tab(P.Pe, j);
            loadV(v, nx, row, [&](unsigned k) -> T { return qj[k] + pe[k]; });
        } else {
            loadPtr(v, qj, nx, row);
        }
        if (m < nc || !split) {
            zero(w);
            mvAcc(w, tab(P.BTr, j), nu, nu, nx, v);
            lds->bq[w0 + m][k][row] = w[0];
        }
        if (stage > 0 && (m >= nc || !split)) {
            mvAcc(rq[k], tab(P.ABKTr, j), nx, nx, nx, v);
            if (split) {
#pragma unroll
                for (int rc = 0; rc < R; rc++) lds->xq[w0 + m][0][row + 64 * rc] = rq[k][rc];
            }
        }
    }
    __syncthreads();
    T d = T(0);
    if (i >= 0 && !(split && stage > 0 && m >= nc && m > 2 * nc)) {
        T acc = T(0);
        for (int ci = 0; ci < nc; ci++) {
            const T b = lds->bq[w0 + ci % g][ci / g][row];
            acc = ci == 0 ? b : acc + b;
        }
        d = mine ? (-acc + ub) : T(0);
        if (P.dynInverse) {
            T dvin[V], dout[R];
            zero(dvin);
            dvin[0] = d;
            zero(dout);
            mvAcc(dout, tab(P.RtInv, i), nu, nu, nu, dvin);
            d = mine ? dout[0] : T(0);
        } else {
            CP<T> L = tab(P.cholL, i);
            for (int k = 0; k < nu; k++) {
                const T dk = bcastLane(d, laneOf(k)) / L[k + (size_t) k * nu];
                if ((int) row == k) d = dk;
                else if ((int) row > k && mine) d -= L[row + (size_t) k * nu] * dk;
            }
            CP<T> U = tab(P.cholU, i);
            for (int k = nu - 1; k >= 0; k--) {
                const T dk = bcastLane(d, laneOf(k)) / U[k + (size_t) k * nu];
                if ((int) row == k) d = dk;
                else if ((int) row < k) d -= U[row + (size_t) k * nu] * dk;
            }
        }
        if (m == 0 && mine) ((GP<T>) P.dd + (long) i * nu)[row] = d;
    }
    if (stage == 0) return;
    T dv[V];
    zero(dv);
    dv[0] = d;
#pragma unroll
    for (int k = 0; k < K; k++) {
        const int ci = m + k * g;
        if (ci >= nc) continue;
        zero(w);
        mvAcc(w, tab(P.APB, c0 + ci), nx, nx, nu, dv);
#pragma unroll
        for (int rc = 0; rc < R; rc++) lds->xq[w0 + m][k][row + 64 * rc] = w[rc] + rq[k][rc];
    }
    // the member that finishes the node: one without children if there is one
    const int last = split ? min(2 * nc, g - 1) : nc < g ? nc : 0;
    zero(w);
    if (i >= 0 && m == last) {
        dv[0] = mine ? d - ub : T(0);
        mvAcc(w, tab(P.KTr, i), nx, nx, nu, dv);
    }
    __syncthreads();
    if (i >= 0 && m == last) {
        GP<T> xbar = cand + (P.oX + (long) i * nx);
        eachRow<R>(nx, row, [&](int rc, unsigned r) {
            T acc = T(0);
            for (int ci = 0; ci < nc; ci++) {
                T x = lds->xq[w0 + ci % g][ci / g][r];
                if (split) x += lds->xq[w0 + nc + ci][0][r];
                acc = ci == 0 ? x : acc + x;
            }
            (qd + (long) i * nx)[r] = (acc + w[rc]) - xbar[r];
        });
    }
}

// Dynamics projection + kernel projection on cand (in place).  The kernel projection touches
// (y, t, s) only, so it shares the first backward stage's barrier interval.
// Where the tree no longer branches, the same waves have a node and its child, and no other workgroup
// waits for them: a workgroup barrier ends such a stage (229 nodes, 7 such stages, 32 workgroups: projections of
// one T 131 -> 110 us).
template <typename T, int R, int V>
__device__ __noinline__ void phaseProjections(const Inst<T> *Pp, int grid, T *candIn, bool doDyn, bool doKernel) {
    IP<T> P = *cst(uniformPtr(Pp));
    const Tc c = threadCtx(grid);
    GP<T> cand = glb(candIn);
    __shared__ TeamLds<T, R> teamLds;
    SPK_LDS TeamLds<T, R> *team = (SPK_LDS TeamLds<T, R> *) &teamLds;
    if (doDyn) {
        for (int stage = P.S - 2; stage >= 0; stage--) {
            const int f = cst(P.stageFrom)[stage], nStage = cst(P.stageTo)[stage] - f + 1;
            const int extra = (doKernel && stage == P.S - 2) ? P.nl : 0;
            const int g = teamSize<R>(c, nStage, P.E);
            if (g > 1) {
                const int m = c.lw % g, w0 = c.lw - m, node = c.wave / g;
                if ((c.wave - c.lw) / g < nStage)
                    dynBackwardTeam<T, R, V>(P, cand, node < nStage ? f + node : -1, stage, c.row, m, g, w0, team);
                for (int task = c.wave; task < extra; task += c.nw) kernelNode<T, R, V>(P, cand, task, c.row);
            } else {
                for (int task = c.wave; task < nStage + extra; task += c.nw) {
                    if (task < nStage) dynBackwardNode<T, R, V>(P, cand, f + task, stage, c.row);
                    else kernelNode<T, R, V>(P, cand, task - nStage, c.row);
                }
            }
            if (stage > P.chain) __syncthreads();
            else sync(c);
        }
        for (int stage = 0; stage <= P.S - 2; stage++) {
            const int f = cst(P.stageFrom)[stage], nStage = cst(P.stageTo)[stage] - f + 1;
            const int g = teamSize<R>(c, nStage, 0);
            for (int task = c.wave / g; task < nStage; task += c.nw / g)
                dynForwardNode<T, R, V>(P, cand, f + task, c.row, c.lw % g, g);
            if (stage >= P.chain && stage < P.S - 2) __syncthreads();
            else sync(c);
        }
    } else if (doKernel) {
        for (int task = c.wave; task < P.nl; task += c.nw) kernelNode<T, R, V>(P, cand, task, c.row);
        sync(c);
    }
}

// modifyDual + proximalDual (src/cache.cuh:770-789) on 2 x-bar - z_p.
template <typename T, int R, int V>
__device__ __noinline__ void phaseDualProx(const Inst<T> *Pp, int grid, T *zIn, T *candIn) {
    IP<T> P = *cst(uniformPtr(Pp));
    const Tc c = threadCtx(grid);
    GP<T> z = glb(zIn), cand = glb(candIn);
    ProxL<T, R> h{P, z + P.sPrim, cand + P.sPrim, c.row};
    auto pv = [&](long base, unsigned k) -> T { return (cand + base)[k] * T(2) - (z + base)[k]; };
    for (int n = c.wave; n < P.N; n += c.nw) opNode<T, R, V>(P, n, c.row, pv, h);
    sync(c);
}

// The CP operator T (src/cache.cuh:796-801): cand = T(z).
template <typename T, int R, int V>
__device__ __forceinline__ void applyT(const Inst<T> *P, const Tc &c, T *z, T *cand, PhaseClock *clk = nullptr) {
    phaseAdjAxpy<T, R, V>(P, c.grid, z, cand);
    sync(c);
    if (clk) clk->mark(PH_ADJ);
    phaseProjections<T, R, V>(P, c.grid, cand, true, true);
    if (clk) clk->mark(PH_PROJ);
    phaseDualProx<T, R, V>(P, c.grid, z, cand);
    if (clk) clk->mark(PH_DUAL);
}

// sum x.(y - gamma ell(y)) and max |y/gamma - ell(y)| with ell(y) = [L* y_d; L y_p]; mx[0] and mx[1]
// are the maxima over the primal and the dual part (err1 and err2 of the debug trace).
template <typename T>
struct EllSums {
    T dot, mxPrim, mxDual;
};

template <typename T, int R, int V>
__device__ __noinline__ EllSums<T> reduceEllNodes(const Inst<T> *Pp, int grid, T *xIn, T *yIn) {
    IP<T> P = *cst(uniformPtr(Pp));
    const Tc c = threadCtx(grid);
    GP<T> x = glb(xIn), y = glb(yIn);
    const int nx = P.nx, nu = P.nu;
    const unsigned row = c.row;
    T dot = T(0), mx = T(0);
    auto acc = [&](T xk, T yk, T ell) {
        dot += xk * (ell * (-P.gamma) + yk);
        mx = fmax(mx, fabs(yk * P.gammaRecip - ell));
    };
    GP<T> yd = y + P.sPrim;
    ReduceL<T, R> h{P, x + P.sPrim, yd, row, T(0), T(0)};
    auto pv = [&](long base, unsigned k) -> T { return (y + base)[k]; };
    for (int n = c.wave; n < P.N; n += c.nw) {
        AdjOut<T, R> o;
        adjNode<T, R, V>(P, yd, n, row, o);
        const long xn = P.oX + (long) n * nx, un = P.oU + (long) n * nu, yn = P.oY + (long) n * P.yD;
#pragma unroll
        for (int rc = 0; rc < R; rc++) {
            const unsigned r = row + 64 * rc;
            if (64 * rc < nx && r < (unsigned) nx) acc((x + xn)[r], (y + xn)[r], o.x[rc]);
            if (n < P.nl && 64 * rc < nu && r < (unsigned) nu) acc((x + un)[r], (y + un)[r], o.u[rc]);
        }
        if (n < P.nl && row < (unsigned) P.yD) acc((x + yn)[row], (y + yn)[row], o.y);
        if (row == 0) {
            acc(x[P.oS + n], y[P.oS + n], o.s);
            acc(x[P.oT + n], y[P.oT + n], o.t);
        }
        opNode<T, R, V>(P, n, row, pv, h);
    }
    return EllSums<T>{dot + h.dot, mx, h.mx};
}

// -2 gamma sum r_p . (L* r_d): as r_p . (L* r_d) = (L r_p) . r_d, this and |r|^2 (from the residual's
// pass) make <r, M r>, the squared M-norm that SuperMann needs between the error checks, from one adjoint
// instead of [L*; L] (229-node FP64 instance in one workgroup: 0.35 -> 0.17 ms an iteration).  No digits cancel:
// <r, M r> is 0.63 to 1.07 of |r|^2 on residuals of 1 to 512 iterations of nine problems (31 to 229 nodes, 3 to
// 100 states).  Error in FP32 against 64 bits on these 264: root mean square 5.0e-8, at most 2.0e-7; of [L*; L]
// 6.5e-8 and 2.1e-7.
template <typename T, int R, int V>
__device__ __noinline__ T adjDotNodes(const Inst<T> *Pp, int grid, T *rIn) {
    IP<T> P = *cst(uniformPtr(Pp));
    const Tc c = threadCtx(grid);
    GP<T> r = glb(rIn);
    const int nx = P.nx, nu = P.nu;
    T dot = T(0);
    auto acc = [&](T rk, T ell) { dot += rk * ell; };
    for (int n = c.wave; n < P.N; n += c.nw) {
        AdjOut<T, R> o;
        adjNode<T, R, V>(P, r + P.sPrim, n, c.row, o);
        GP<T> xn = r + (P.oX + (long) n * nx), un = r + (P.oU + (long) n * nu);
        eachRow<R>(nx, c.row, [&](int rc, unsigned k) { acc(xn[k], o.x[rc]); });
        if (n < P.nl) {
            eachRow<R>(nu, c.row, [&](int rc, unsigned k) { acc(un[k], o.u[rc]); });
            if (c.row < (unsigned) P.yD) acc((r + (P.oY + (long) n * P.yD))[c.row], o.y);
        }
        if (c.row == 0) {
            acc(r[P.oS + n], o.s);
            acc(r[P.oT + n], o.t);
        }
    }
    return dot * (T(-2) * P.gamma);
}

// SPLIT: also the maxima over the primal and the dual part apart, in split[0] and split[1].
template <typename T, int R, int V, bool SPLIT = false>
__device__ __forceinline__ void reduceEll(const Inst<T> *P, const Tc &c, T *x, T *y, SPK_LDS T *lds, T &dotOut,
                                          T &maxOut, T *split = nullptr) {
    const EllSums<T> s = reduceEllNodes<T, R, V>(P, c.grid, x, y);
    T v[1] = {s.dot};
    blockSum(v, lds, c);
    dotOut = v[0];
    if constexpr (SPLIT) {
        split[0] = blockMax(s.mxPrim, lds, c);
        split[1] = blockMax(s.mxDual, lds, c);
        maxOut = fmax(split[0], split[1]);
    } else {
        maxOut = blockMax(fmax(s.mxPrim, s.mxDual), lds, c);
    }
}

// ---------------------------------------------------------------- iterate-wide passes
// Every thread issues U independent loads before it stores anything, so a single
// workgroup keeps U * blockDim loads in flight while it streams an iterate.
template <int U, typename Ld, typename St>
__device__ __forceinline__ void stream(long n, const Tc &c, Ld ld, St st) {
    using Vals = decltype(ld(0L));
    const long nt = c.nt;
    long k = c.tid;
    for (; k + (U - 1) * nt < n; k += U * nt) {
        Vals v[U];
#pragma unroll
        for (int u = 0; u < U; u++) v[u] = ld(k + u * nt);
#pragma unroll
        for (int u = 0; u < U; u++) st(k + u * nt, v[u]);
    }
    for (; k < n; k += nt) st(k, ld(k));
}

template <typename T>
struct V2 {
    T a, b;
};
template <typename T>
struct V4 {
    T a, b, c, d;
};

// ---------------------------------------------------------------- Anderson direction
// src/cache.cuh:861-904 with the least squares argmin ||Y g - r|| solved by Householder QR
// (geqrf + ormqr + trsm).  Y and S are rings of andBuff columns; logical column 0 is the newest.
// Only R and the first m entries of Q'r are needed, so the rows of [Y | r] are factored where they
// are read: each thread folds its rows, 4 at a time, into an m x (m + 1) triangle in
// registers, and the triangles are folded pairwise across the lanes, then the waves, then the workgroups
// (a tree of Householder factorisations, each as stable as the one of the whole matrix).  One pass over
// m + 1 vectors and one grid barrier; column by column it took 4 m + 2 such passes and 2 m + 2 reductions
// (229-node FP64 instance, m = 3, per iteration: one workgroup 0.395 ms, now 0.045; 32 workgroups 0.088,
// now 0.019).
template <typename T, int M, int B>
__device__ __forceinline__ void foldRows(T (&R)[M][M + 1], T (&A)[B][M + 1]) {
#pragma unroll
    for (int k = 0; k < M; k++) {
        T sigma = T(0);
#pragma unroll
        for (int i = 0; i < B; i++) sigma += A[i][k] * A[i][k];
        const T alpha = R[k][k];
        const T nrm = sqrt(alpha * alpha + sigma);
        const bool flat = sigma == T(0);
        const T beta = flat ? alpha : (alpha >= T(0) ? -nrm : nrm);
        const T tau = flat ? T(0) : (beta - alpha) / beta;
        const T scale = flat ? T(0) : T(1) / (alpha - beta);
        R[k][k] = beta;
#pragma unroll
        for (int i = 0; i < B; i++) A[i][k] *= scale;
#pragma unroll
        for (int j = k + 1; j <= M; j++) {
            T w = R[k][j];
#pragma unroll
            for (int i = 0; i < B; i++) w += A[i][k] * A[i][j];
            w *= tau;
            R[k][j] -= w;
#pragma unroll
            for (int i = 0; i < B; i++) A[i][j] -= w * A[i][k];
        }
    }
}

// R <- the factor of both lanes' triangles, the lower lane's on top, for lanes `step` apart.
template <typename T, int M>
__device__ __forceinline__ void foldLanes(T (&R)[M][M + 1], int step, unsigned lane) {
    T A[M][M + 1];
    const bool upper = (lane & step) != 0;
#pragma unroll
    for (int i = 0; i < M; i++)
#pragma unroll
        for (int j = 0; j <= M; j++) {
            A[i][j] = T(0);
            if (j >= i) {
                const T mine = R[i][j], other = __shfl_xor(mine, step, 64);
                R[i][j] = upper ? other : mine;
                A[i][j] = upper ? mine : other;
            }
        }
    foldRows<T, M, M>(R, A);
}

template <typename T, int M>
__device__ __noinline__ void andersonLeastSquares(const Inst<T> *Pp, int grid, int head, T *rIn, SPK_LDS T *lds,
                                                  double (&gs)[8]) {
    constexpr int B = 4;  // rows folded at a time
    constexpr int NV = M * (M + 1) / 2 + M;  // entries of a triangle; 8 waves of them fit the LDS buffer
    static_assert(NV * SPK_MAX_THREADS / 64 <= 16 * 32, "LDS buffer");
    IP<T> P = *cst(uniformPtr(Pp));
    const Tc c = threadCtx(grid, P.gpart);
    head = __builtin_amdgcn_readfirstlane(head);
    const long n = P.sIter;
    // workgroups that take rows: all whose triangles fit in one partials buffer
    const int nb = c.grid ? min((int) gridDim.x, GRID_MAXK * GRID_MAXWG / NV) : 1;
    const long nt = (long) nb * blockDim.x;
    GP<T> col[M + 1];
#pragma unroll
    for (int lc = 0; lc < M; lc++) col[lc] = (GP<T>) P.hY + (long) ((head - lc + M) % M) * n;
    col[M] = glb(rIn);
    T R[M][M + 1];
#pragma unroll
    for (int i = 0; i < M; i++) zero(R[i]);
    auto entries = [&](auto f) {  // f(position, entry) over the triangle
        int q = 0;
#pragma unroll
        for (int i = 0; i < M; i++)
#pragma unroll
            for (int j = i; j <= M; j++) f(q++, R[i][j]);
    };
    if (c.tid < nt) {
#pragma unroll 1
        for (long k0 = c.tid; k0 < n; k0 += B * nt) {
            T A[B][M + 1];
#pragma unroll
            for (int i = 0; i < B; i++) {
                const long k = k0 + i * nt;
#pragma unroll
                for (int j = 0; j <= M; j++) A[i][j] = col[j][k < n ? k : k0];
            }
#pragma unroll
            for (int i = 1; i < B; i++)
#pragma unroll
                for (int j = 0; j <= M; j++) A[i][j] = k0 + i * nt < n ? A[i][j] : T(0);
            foldRows<T, M, B>(R, A);
        }
    }
#pragma unroll 1
    for (int o = 1; o < 64; o <<= 1) foldLanes<T, M>(R, o, c.lane);
    if (c.lane == 0) entries([&](int q, T &e) { lds[c.lw * NV + q] = e; });
    __syncthreads();
    entries([&](int q, T &e) { e = (int) c.lane < c.lnw ? lds[c.lane * NV + q] : T(0); });
#pragma unroll 1
    for (int o = c.lnw > 4 ? 4 : c.lnw > 2 ? 2 : c.lnw / 2; o >= 1; o >>= 1) foldLanes<T, M>(R, o, c.lane);
    if (c.grid) {
        const int seq = *gridSeq();
        GP<T> part = (GP<T>) c.gpart + (size_t) (seq & 1) * GRID_MAXK * GRID_MAXWG;
        if (c.ltid == 0 && (int) blockIdx.x < nb) entries([&](int q, T &e) { part[blockIdx.x * NV + q] = e; });
        gridBarrier();
        if (c.ltid == 0) *gridSeq() = seq + 1;
        entries([&](int q, T &e) { e = (int) c.lane < nb ? part[c.lane * NV + q] : T(0); });
#pragma unroll 1
        for (int b = c.lane + 64; b < nb; b += 64) {
            T A[M][M + 1];
            int q = 0;
#pragma unroll
            for (int i = 0; i < M; i++)
#pragma unroll
                for (int j = 0; j <= M; j++) A[i][j] = j >= i ? (T) part[b * NV + q++] : T(0);
            foldRows<T, M, M>(R, A);
        }
#pragma unroll 1
        for (int o = 1; o < 64; o <<= 1) foldLanes<T, M>(R, o, c.lane);
    }
    // lane 0's triangle in every lane, then back substitution
    entries([&](int, T &e) { e = bcastLane(e, 0); });
    T g[M];
#pragma unroll
    for (int q = M - 1; q >= 0; q--) {
        T v = R[q][M];
#pragma unroll
        for (int j = q + 1; j < M; j++) v -= R[q][j] * g[j];
        g[q] = v / R[q][q];
    }
#pragma unroll
    for (int lc = 0; lc < M; lc++) gs[(head - lc + M) % M] = (double) g[lc];
    __syncthreads();
}

// New Anderson column (src/cache.cuh:863-868): Y_h = r - r_prev, S_h = (z - z_prev) - Y_h.
// With the Gram least squares it also accumulates, in FP64, <Y_h, Y_s> for every slot s and
// <Y_s, r> for every slot, and updates the slot-indexed Gram matrix G held in LDS.
template <typename T>
__device__ __noinline__ void andersonColumn(const Inst<T> *Pp, int grid, int head, T *RIn, T *RPIn, T *ZIn, T *ZPIn,
                                            bool gram, SPK_LDS double *G, SPK_LDS double *gb, SPK_LDS double *ldsd) {
    IP<T> P = *cst(uniformPtr(Pp));
    const Tc c = threadCtx(grid, P.gpart);
    GP<T> Rv = glb(RIn), RP = glb(RPIn), Z = glb(ZIn), ZP = glb(ZPIn);
    head = __builtin_amdgcn_readfirstlane(head);
    const long n = P.sIter;
    const int m = P.andBuff;
    GP<T> Yh = (GP<T>) P.hY + (long) head * n, Sh = (GP<T>) P.hS + (long) head * n;
    if (!gram) {
        stream<8>(
            n, c, [&](long k) { return V4<T>{Rv[k], RP[k], Z[k], ZP[k]}; },
            [&](long k, const V4<T> &v) {
                const T dr = v.a - v.b;
                Yh[k] = dr;
                Sh[k] = (v.c - v.d) - dr;
            });
        sync(c);
        return;
    }
    double acc[16];
#pragma unroll
    for (int q = 0; q < 16; q++) acc[q] = 0.;
    GP<T> Ys[8];
#pragma unroll
    for (int s2 = 0; s2 < 8; s2++) Ys[s2] = (GP<T>) P.hY + (long) (s2 < m ? s2 : 0) * n;
    stream<4>(
        n, c, [&](long k) { return V4<T>{Rv[k], RP[k], Z[k], ZP[k]}; },
        [&](long k, const V4<T> &v) {
            const T dr = v.a - v.b;
            Yh[k] = dr;
            Sh[k] = (v.c - v.d) - dr;
            const double drd = (double) dr, rd = (double) v.a;
#pragma unroll
            for (int s2 = 0; s2 < 8; s2++) {
                if (s2 < m) {
                    const double ys = (s2 == head) ? drd : (double) Ys[s2][k];
                    acc[s2] += drd * ys;
                    acc[8 + s2] += ys * rd;
                }
            }
        });
    blockSum(acc, ldsd, c);
    if (c.ltid == 0) {
        for (int s2 = 0; s2 < m; s2++) {
            G[head * 8 + s2] = acc[s2];
            G[s2 * 8 + head] = acc[s2];
            gb[s2] = acc[8 + s2];
        }
    }
    sync(c);
}

// Least squares argmin ||Y g - r|| from the Gram matrix: Cholesky of G + eps * max(diag) I in
// FP64 (uniform in every thread).  Returns false when the factorisation breaks down.
__device__ __forceinline__ bool gramSolve(const SPK_LDS double *G, const SPK_LDS double *gb, int m, double (&g)[8]) {
    double Lm[8][8];
    double dmax = 0.;
    for (int i = 0; i < m; i++) dmax = fmax(dmax, G[i * 8 + i]);
    if (!(dmax > 0.)) return false;
    const double ridge = 1e-12 * dmax;
#pragma unroll
    for (int i = 0; i < 8; i++) {
#pragma unroll
        for (int j = 0; j < 8; j++) {
            if (i < m && j <= i) {
                double v = G[i * 8 + j] + (i == j ? ridge : 0.);
#pragma unroll
                for (int k = 0; k < 8; k++)
                    if (k < j) v -= Lm[i][k] * Lm[j][k];
                if (i == j) {
                    if (!(v > 0.)) return false;
                    Lm[i][i] = sqrt(v);
                } else {
                    Lm[i][j] = v / Lm[j][j];
                }
            }
        }
    }
    double y[8];
#pragma unroll
    for (int i = 0; i < 8; i++) {
        y[i] = 0.;
        if (i < m) {
            double v = gb[i];
#pragma unroll
            for (int k = 0; k < 8; k++)
                if (k < i) v -= Lm[i][k] * y[k];
            y[i] = v / Lm[i][i];
        }
    }
#pragma unroll
    for (int i = 7; i >= 0; i--) {
        g[i] = 0.;
        if (i < m) {
            double v = y[i];
#pragma unroll
            for (int k = 0; k < 8; k++)
                if (k > i && k < m) v -= Lm[k][i] * g[k];
            g[i] = v / Lm[i][i];
        }
    }
    return true;
}

// d = -S g - r (src/cache.cuh:897-898); with toCand the K0 update cand = z_prev + d is written
// directly (src/cache.cuh:1055-1057) and d itself is not stored.
template <typename T>
__device__ __noinline__ void andersonApply(const Inst<T> *Pp, int grid, const double (&gs)[8], bool useLS, T *RIn,
                                           T *ZPIn, T *outIn, bool toCand) {
    IP<T> P = *cst(uniformPtr(Pp));
    const Tc c = threadCtx(grid);
    GP<T> Rv = glb(RIn), ZP = glb(ZPIn), out = glb(outIn);
    const long n = P.sIter;
    const int m = P.andBuff;
    T gg[8];
    GP<T> Ss[8];
#pragma unroll
    for (int s2 = 0; s2 < 8; s2++) {
        gg[s2] = (useLS && s2 < m) ? (T) gs[s2] : T(0);
        Ss[s2] = (GP<T>) P.hS + (long) (s2 < m ? s2 : 0) * n;
    }
    if (!useLS) {
        stream<8>(
            n, c, [&](long k) { return V2<T>{Rv[k], ZP[k]}; },
            [&](long k, const V2<T> &v) {
                const T d = -v.a;
                out[k] = toCand ? v.b + d : d;
            });
    } else {
        stream<4>(
            n, c, [&](long k) { return V2<T>{Rv[k], ZP[k]}; },
            [&](long k, const V2<T> &v) {
                T sg = T(0);
#pragma unroll
                for (int s2 = 0; s2 < 8; s2++)
                    if (s2 < m) sg += Ss[s2][k] * gg[s2];
                const T d = -sg - v.a;
                out[k] = toCand ? v.b + d : d;
            });
    }
    sync(c);
}

// r = z - cand; returns this thread's part of |r|^2.
template <typename T>
__device__ __forceinline__ T residualPass(IP<T> P, const Tc &c, T *zIn, T *candIn, T *rIn) {
    GP<T> z = glb(zIn), cand = glb(candIn), r = glb(rIn);
    T sr = T(0);
    stream<8>(
        P.sIter, c, [&](long k) { return V2<T>{z[k], cand[k]}; },
        [&](long k, const V2<T> &v) {
            const T d = v.a - v.b;
            r[k] = d;
            sr += d * d;
        });
    return sr;
}

// ---------------------------------------------------------------- debug trace
// Index of the first non-finite entry of v[0, n), or -1.  The index travels through the block's
// T-valued max reduction as n - k, exact while n < 2^24 in FP32 (2^53 in FP64).
template <typename T>
__device__ __noinline__ long firstNonfinite(const T *v, long n, SPK_LDS T *lds, int grid, void *gpart) {
    const Tc c = threadCtx(grid, gpart);
    T bad = T(0);
    for (long k = c.tid; k < n; k += c.nt)
        if (!isfinite(v[k])) bad = fmax(bad, T(n - k));
    bad = blockMax(bad, lds, c);
    return bad > T(0) ? n - (long) bad : -1;
}

// One record of the reference's debug caches at an error check (src/cache.cuh:947-959):
//   err1, err2  the max-norms of the primal and dual parts of r/gamma - [L*; L] r   (split)
//   err3        ||z - cand||_2 = ||r||_2
//   err0        the reference computes e <- cand_prim - e on a vector e that starts at zero and
//               is only zeroed by reset() (its L* product goes to another buffer, so it does not
//               enter e), then ||e||_2; restated as computed, with e in P.dbgE
//   callsL      calls to L and L* counted so far: two per application of T (src/cache.cuh:704-716,
//               :750, :773); the host adds the count of earlier solves
template <typename T>
__device__ __noinline__ void debugRecord(const Inst<T> *Pp, int grid, SPK_LDS T *lds, long it, long callsL,
                                         const T (&split)[2], const T *RR, const T *C, long &nDbg) {
    IP<T> P = *cst(uniformPtr(Pp));
    const Tc c = threadCtx(grid, P.gpart);
    T acc[2] = {T(0), T(0)};
    for (long k = c.tid; k < P.sIter; k += c.nt) acc[0] += RR[k] * RR[k];
    T *E = P.dbgE;
    for (long k = c.tid; k < P.sPrim; k += c.nt) {
        const T e = C[k] - E[k];
        E[k] = e;
        acc[1] += e * e;
    }
    blockSum(acc, lds, c);
    if (nDbg < P.dbgCap && c.tid == 0) {
        double *r = P.dbg + nDbg * DBG_WORDS;
        r[0] = (double) it;
        r[1] = (double) callsL;
        r[2] = sqrt((double) acc[1]);
        r[3] = (double) split[0];
        r[4] = (double) split[1];
        r[5] = sqrt((double) acc[0]);
    }
    nDbg++;
    sync(c);
}

// ---------------------------------------------------------------- the solve
// SuperMann with Anderson directions (src/cache.cuh:1008-1132) and runCp (:967-1002).
// The six iterate buffers rotate by pointer instead of being copied: acceptCandidate,
// backup/restore and saveToPrev are pointer moves.
template <typename T, int R, int V>
__device__ void solveInstance(const Inst<T> *Pp, Out &out, SPK_LDS T *lds, SPK_LDS double *ldsd, int grid) {
    IP<T> P = *cst(uniformPtr(Pp));
    const Tc c = threadCtx(grid, P.gpart);
    const long n = P.sIter;
    const int m = P.andBuff;
    const bool gram = P.lsMethod == 1;
    __shared__ double gramMat[64], gramRhs[8];
    SPK_LDS double *G = (SPK_LDS double *) gramMat, *gb = (SPK_LDS double *) gramRhs;
    T *Z = P.z, *C = P.cand, *ZP = P.zPrev, *RR = P.res, *RP = P.resPrev, *BK = P.backup;
    T *D = P.dir, *DS = P.dirS;
    int head = m - 1;
    const long t0 = wall_clock64();
    long nT = 0, nEll = 0, nDbg = 0, nonfinite = -1;
    PhaseClock clk;
    clk.start();
    // initialisePrev / initialiseIter (src/cache.cuh:611-632)
    if (P.method == METHOD_SPOCK) {
        if (P.warm) {
            stream<8>(
                n, c, [&](long k) { return V2<T>{Z[k], RR[k]}; },
                [&](long k, const V2<T> &v) {
                    ZP[k] = v.a;
                    RP[k] = v.b;
                });
        } else {
            stream<8>(
                n, c, [&](long k) { return 0; },
                [&](long k, int) {
                    ZP[k] = T(1);
                    RP[k] = T(1);
                });
        }
    }
    if (c.ltid < 64) G[c.ltid] = 0.;
    startGrid(c, P.gbar);
    sync(c);
    // a given tolerance (> 0) skips the reference's first-check calibration, so warm starts and
    // polish solves are accepted against the threshold of the cold solve they continue
    bool initFlag = !(P.tolFixed > T(0));
    int status = ST_NOTRUN;
    long iters = 0;
    T tol = initFlag ? T(0) : P.tolFixed, lastErr = T(NAN), wLast = T(NAN);
    const T c0 = T(0.99), c1 = T(0.99), c2 = T(0.99), beta = T(0.5), sigma = T(0.1), lambda = T(1);
    const T inf = T(INFINITY);
    T zeta = inf, w = inf, wSafe = inf;
    long k0 = 0, k1 = 0, k2 = 0, k2bt = 0, k3 = 0;
    // the iteration cap is only tested at error checks (src/cache.cuh:937-940): the last outer
    // iteration is the first check index at or beyond maxIters
    const long hardCap =
        P.maxIters > 0 ? (P.maxIters + P.checkPeriod - 1) / P.checkPeriod * P.checkPeriod + 1 : 2000000;
    long it = 0;
    for (it = 0; it < hardCap; it++) {
        if (it != 0 && P.method == METHOD_SPOCK) {  // acceptCandidate: z <- cand
            T *tmp = Z;
            Z = C;
            C = tmp;
        }
        clk.mark(PH_OTHER);
        applyT<T, R, V>(Pp, c, Z, C, &clk);
        nT++;
        // computeError (src/cache.cuh:910-961): r = z - cand
        if (P.dbg) {  // isFinite(candidate) (src/cache.cuh:912): stop at the first non-finite entry
            const long bad = firstNonfinite<T>(C, n, lds, grid, P.gpart);
            if (bad >= 0) {
                status = ST_NONFINITE;
                iters = it;
                nonfinite = bad;
                break;
            }
        }
        const T sumR = residualPass<T>(P, c, Z, C, RR);
        sync(c);
        clk.mark(PH_RES);
        bool haveDot = false;
        T dotRR = T(0);
        if (it % P.checkPeriod == 0) {
            T mx;
            if (P.dbg) {
                T split[2];
                reduceEll<T, R, V, true>(Pp, c, RR, RR, lds, dotRR, mx, split);
                debugRecord<T>(Pp, grid, lds, it, 2 * nT, split, RR, C, nDbg);
            } else {
                reduceEll<T, R, V>(Pp, c, RR, RR, lds, dotRR, mx);
            }
            nEll++;
            haveDot = true;
            clk.mark(PH_ELL);
            if (initFlag) {
                tol = fmax(P.tolAbs, P.tolRel * mx);
                initFlag = false;
            } else {
                lastErr = mx;
                int code = ST_NOTRUN;
                if (mx <= tol) code = ST_CONVERGED;
                if (P.maxIters && it >= P.maxIters) code = ST_OUTOFITER;
                if (P.maxTicks > 0 && it % 1000 == 0) {
                    // threads read the clock at different moments: decide on the latest reading
                    const T late = (double) (wall_clock64() - t0) >= P.maxTicks ? T(1) : T(0);
                    if (blockMax(late, lds, c) > T(0)) code = ST_OUTOFTIME;
                }
                if (code != ST_NOTRUN) {
                    status = code;
                    iters = it;
                }
            }
        }
        if (status != ST_NOTRUN || P.method == METHOD_CP) {  // acceptCandidate (and stop)
            T *tmp = Z;
            Z = C;
            C = tmp;
            if (status != ST_NOTRUN) break;
            continue;
        }
        {  // backup (src/cache.cuh:804-806): keep T(z) aside, continue in a fresh buffer
            T *tmp = BK;
            BK = C;
            C = tmp;
        }
        // normM(r) (src/cache.cuh:740-742)
        if (!haveDot) {
            T v[1] = {adjDotNodes<T, R, V>(Pp, grid, RR) + sumR};
            blockSum(v, lds, c);
            dotRR = v[0];
            nEll++;
            clk.mark(PH_ELL);
        }
        w = sqrt(dotRR);
        wLast = w;
        // delta iterate/residual, new Anderson column, then saveToPrev as pointer moves
        head = (head + 1) % m;
        andersonColumn<T>(Pp, grid, head, RR, RP, Z, ZP, gram, G, gb, ldsd);
        clk.mark(PH_ACOL);
        {
            T *tmp = ZP;
            ZP = Z;
            Z = tmp;
            tmp = RP;
            RP = RR;
            RR = tmp;
        }
        // updateDirection (src/cache.cuh:861-904); r now lives in RP
        double gs[8];
#pragma unroll
        for (int q = 0; q < 8; q++) gs[q] = 0.;
        bool useLS = false;
        if (it >= m) {
            if (gram) {
                useLS = gramSolve(G, gb, m, gs);
            } else {
                SPK_LDS T *ldsT = (SPK_LDS T *) ldsd;
                switch (m) {
                    case 1: andersonLeastSquares<T, 1>(Pp, grid, head, RP, ldsT, gs); break;
                    case 2: andersonLeastSquares<T, 2>(Pp, grid, head, RP, ldsT, gs); break;
                    case 3: andersonLeastSquares<T, 3>(Pp, grid, head, RP, ldsT, gs); break;
                    case 4: andersonLeastSquares<T, 4>(Pp, grid, head, RP, ldsT, gs); break;
                    case 5: andersonLeastSquares<T, 5>(Pp, grid, head, RP, ldsT, gs); break;
                    case 6: andersonLeastSquares<T, 6>(Pp, grid, head, RP, ldsT, gs); break;
                    case 7: andersonLeastSquares<T, 7>(Pp, grid, head, RP, ldsT, gs); break;
                    default: andersonLeastSquares<T, 8>(Pp, grid, head, RP, ldsT, gs); break;
                }
                useLS = true;
            }
        }
        clk.mark(PH_ALS);
        const bool blind = w <= c0 * zeta;
        andersonApply<T>(Pp, grid, gs, useLS, RP, ZP, blind ? C : D, blind);
        clk.mark(PH_AAPPLY);
        if (blind) {  // K0 blind update (src/cache.cuh:1055-1061)
            zeta = w;
            k0++;
            continue;
        }
        T tau = T(1);
        for (int in = 0; in < P.maxInner; in++) {  // line search (src/cache.cuh:1063-1099)
            stream<8>(
                n, c, [&](long k) { return V2<T>{D[k], ZP[k]}; },
                [&](long k, const V2<T> &v) {
                    const T ds = v.a * tau;
                    DS[k] = ds;
                    Z[k] = v.b + ds;
                });
            sync(c);
            clk.mark(PH_LINE);
            applyT<T, R, V>(Pp, c, Z, C, &clk);
            nT++;
            const T sumT = residualPass<T>(P, c, Z, C, RR);
            sync(c);
            clk.mark(PH_RES);
            T dot[1] = {adjDotNodes<T, R, V>(Pp, grid, RR) + sumT};
            blockSum(dot, lds, c);
            nEll++;
            clk.mark(PH_ELL);
            const T wTilde = sqrt(dot[0]);
            if (w <= wSafe && wTilde <= c1 * w) {  // K1: cand <- z
                T *tmp = C;
                C = Z;
                Z = tmp;
                wSafe = wTilde + pow(c2, T(it));
                k1++;
                break;
            }
            T dotRD, mx;
            reduceEll<T, R, V>(Pp, c, RR, DS, lds, dotRD, mx);
            nEll++;
            clk.mark(PH_ELL);
            const T rho = wTilde * wTilde - dotRD;
            if (rho >= sigma * wTilde * w) {  // K2
                const T f = lambda * rho / (wTilde * wTilde);
                stream<8>(
                    n, c, [&](long k) { return V2<T>{RR[k], ZP[k]}; },
                    [&](long k, const V2<T> &v) {
                        const T rk = v.a * f;
                        RR[k] = rk;
                        C[k] = v.b - rk;
                    });
                sync(c);
                k2++;
                break;
            } else {
                tau *= beta;
                k2bt++;
            }
            if (in >= P.maxInner - 1) {  // K3: restore the plain CP step
                T *tmp = C;
                C = BK;
                BK = tmp;
                k3++;
            }
        }
    }
    if (status == ST_NOTRUN) {
        status = ST_OUTOFITER;
        iters = it;
    }
    // the accepted iterate must end in P.z and the last residual in P.res; both sources are
    // read before either destination is written, so rotated roles cannot clobber each other
    if (Z != P.z || RR != P.res) {
        T *dz = P.z, *dr = P.res;
        stream<8>(
            n, c, [&](long k) { return V2<T>{Z[k], RR[k]}; },
            [&](long k, const V2<T> &v) {
                dz[k] = v.a;
                dr[k] = v.b;
            });
    }
    sync(c);
    if (c.tid == 0) {
        out.nDbg = nDbg;
        out.nonfinite = nonfinite;
        out.status = status;
        out.iters = iters;
        out.err = (double) lastErr;
        out.tol = (double) tol;
        out.w = (double) wLast;
        out.k0 = k0;
        out.k1 = k1;
        out.k2 = k2;
        out.k2bt = k2bt;
        out.k3 = k3;
        out.nT = nT;
        out.nEll = nEll;
        clk.mark(PH_OTHER);
        for (int i = 0; i < NUM_PHASES; i++) out.ticks[i] = clk.acc[i];
    }
}

// grid = 0: workgroup k solves instance k.  grid = 1 (cooperative launch, count = 1): every
// workgroup works on instance 0.
template <typename T, int R, int V>
__global__ void __launch_bounds__(SPK_MAX_THREADS) k_solve(const Inst<T> *__restrict__ insts, Out *outs, int count,
                                                int grid) {
    __shared__ T lds[8 * 32];
    __shared__ double ldsd[16 * 32];
    const int k = grid ? 0 : (int) blockIdx.x;
    if (k >= count) return;
    solveInstance<T, R, V>(insts + k, outs[insts[k].slot], (SPK_LDS T *) lds, (SPK_LDS double *) ldsd, grid);
}

// ---------------------------------------------------------------- single-operator kernels
// Debug entry points used by the parity tests: they read P.z and write P.cand.
enum DebugOp { OP_L = 0, OP_LADJ = 1, OP_DYN = 2, OP_KERNEL = 3, OP_T = 4, OP_ELL = 5, OP_DUAL = 6 };

template <typename T, int R, int V>
__global__ void __launch_bounds__(SPK_MAX_THREADS) k_debug(const Inst<T> *__restrict__ insts, Out *outs, int count, int op,
                                                int grid) {
    __shared__ T ldsBuf[8 * 32];
    SPK_LDS T *lds = (SPK_LDS T *) ldsBuf;
    const int kInst = grid ? 0 : (int) blockIdx.x;
    if (kInst >= count) return;
    const Inst<T> *Pp = insts + kInst;
    IP<T> P = *cst(Pp);
    const Tc c = threadCtx(grid, P.gpart);
    startGrid(c, P.gbar);
    GP<T> z = (GP<T>) P.z, cand = (GP<T>) P.cand;
    if (op == OP_L) {
        StoreL<T, R> h{P, cand + P.sPrim, c.row};
        auto pv = [&](long base, unsigned k) -> T { return (z + base)[k]; };
        for (int n = c.wave; n < P.N; n += c.nw) opNode<T, R, V>(P, n, c.row, pv, h);
    } else if (op == OP_LADJ) {
        for (int n = c.wave; n < P.N; n += c.nw) {
            AdjOut<T, R> o;
            adjNode<T, R, V>(P, z + P.sPrim, n, c.row, o);
            eachRow<R>(P.nx, c.row, [&](int rc, unsigned r) { cand[P.oX + (long) n * P.nx + r] = o.x[rc]; });
            if (n < P.nl) {
                eachRow<R>(P.nu, c.row, [&](int rc, unsigned r) { cand[P.oU + (long) n * P.nu + r] = o.u[rc]; });
                if (c.row < (unsigned) P.yD) cand[P.oY + (long) n * P.yD + c.row] = o.y;
            }
            if (c.row == 0) {
                cand[P.oS + n] = o.s;
                cand[P.oT + n] = o.t;
            }
        }
    } else if (op == OP_DYN || op == OP_KERNEL) {
        for (long k = c.tid; k < P.sPrim; k += c.nt) cand[k] = z[k];
        sync(c);
        if (op == OP_DYN)
            for (int n = c.wave; n < P.N; n += c.nw)
                if (n >= P.nl)
                    for (int r = c.lane; r < P.nx; r += 64)
                        ((GP<T>) P.qd)[(long) n * P.nx + r] = -cand[P.oX + (long) n * P.nx + r];
        sync(c);
        phaseProjections<T, R, V>(Pp, grid, P.cand, op == OP_DYN, op == OP_KERNEL);
    } else if (op == OP_T) {
        applyT<T, R, V>(Pp, c, P.z, P.cand);
    } else if (op == OP_DUAL) {  // Cache::getDual (src/cache.cuh:371-376): dual prox of the given primal
        phaseDualProx<T, R, V>(Pp, grid, P.z, P.cand);
    } else if (op == OP_ELL) {
        T dot, mx;
        reduceEll<T, R, V>(Pp, c, P.z, P.cand, lds, dot, mx);
        if (c.tid == 0) {
            outs[P.slot].w = (double) dot;
            outs[P.slot].err = (double) mx;
        }
    }
}

// Explicit instantiations: register chunk classes (R, V) = (1,1) for dims <= 64, and (4,4) for
// dims <= 256.  The library compiles this file once per type and class (SPK_KERNEL_T, SPK_KERNEL_CLASS).
template __global__ void k_solve<SPK_KERNEL_T, SPK_KERNEL_CLASS, SPK_KERNEL_CLASS>(const Inst<SPK_KERNEL_T> *, Out *, int,
                                                                                 int);
template __global__ void k_debug<SPK_KERNEL_T, SPK_KERNEL_CLASS, SPK_KERNEL_CLASS>(const Inst<SPK_KERNEL_T> *, Out *, int,
                                                                                 int, int);

}  // namespace spk
