// Tile engine: many instances of ONE problem, 16 per workgroup, the per-node products on the
// matrix cores.
//
// Layout (LaneInst with width 16): element e of instance b of every state region is at
// ((b / 16) * rows + e) * 16 + b % 16, so a workgroup's state is one contiguous slab per region
// and four consecutive rows of its 16 instances are 64 consecutive words.
//
// Lane l of a wave serves instance j = l % 16 and row group g = l / 16.  A node's product of a
// factor M (r x c, packed in operand order) with the 16 instances' vectors X (c x 16) is a GEMM on
// v_mfma_{f32,f64}_16x16x4: the A operand is a 16 x 4 block of M (lane l holds M[r0 + l%16][k0 + l/16]),
// the B operand four rows of X (lane l holds X[k0 + l/16][l%16], its own instance's entry) and each
// lane receives four rows of its instance (RowMap: rows 4g .. 4g + 3 of each 16-row tile in FP32,
// rows g, g + 4, g + 8, g + 12 in FP64).  The elementwise parts of the operators use the same row
// ownership, so a lane only ever reads back what it wrote itself.  Intermediate vectors a wave
// needs again as a B operand (R~^-1 e, d, u of the tree sweeps) pass through its own LDS slice.
// Per-instance sums are per-lane partials, combined across the four row groups by cross-lane
// shuffles (the same value in all four lanes) and across waves through LDS in wave order.
//
// Operator semantics are those of the other engines and of the reference (src/operator.cuh:41-82,
// src/dynamics.cuh:74-174, src/cache.cuh:650-801); the SuperMann control is the shared lockstep
// solve (lockstep.hpp).  As in the lane engine the dynamics sweep applies the precomputed
// (L L')^-1 and the Anderson least squares is the FP64 Gram solve.
#include "engine.hpp"
#include "lockstep.hpp"

#include <hip/hip_runtime.h>
#include <math.h>

#include <type_traits>

// Launch bound of this compilation: 512 threads (two waves per SIMD, up to 256 registers each) or 1024
// (four waves per SIMD, 128 registers each: more waves to hide memory latency, more spills).  The
// library is built once per bound; the 1024 build's kernels carry the suffix _x1024.
#ifndef SPK_TILE_MAX_THREADS
#define SPK_TILE_MAX_THREADS 512
#endif
#if SPK_TILE_MAX_THREADS == 512
#define SPK_TILE_KERNEL(name) name
#else
#define SPK_TILE_KERNEL_CAT2(a, b) a##_x##b
#define SPK_TILE_KERNEL_CAT(a, b) SPK_TILE_KERNEL_CAT2(a, b)
#define SPK_TILE_KERNEL(name) SPK_TILE_KERNEL_CAT(name, SPK_TILE_MAX_THREADS)
#endif
namespace spk {
namespace tile {
using namespace ls;

constexpr int W = 16;                                // instances per workgroup
constexpr int MAXW = SPK_TILE_MAX_THREADS / 64;      // waves per workgroup
constexpr int STG = 32 * W;                          // words of one LDS staging slice (32 rows)

template <typename T>
struct AccT;
template <>
struct AccT<float> {
    typedef float type __attribute__((ext_vector_type(4)));
};
template <>
struct AccT<double> {
    typedef double type __attribute__((ext_vector_type(4)));
};
template <typename T>
using Acc = typename AccT<T>::type;

__device__ __forceinline__ Acc<float> mfma(float a, float b, Acc<float> c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ Acc<double> mfma(double a, double b, Acc<double> c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

struct Ctx {
    int lane, g, j, wave, nw;
    int gl;       // this lane's instance
    bool writer;  // the row group 0 lane writes the instance's records
};

__device__ __forceinline__ Ctx ctx() {
    Ctx c;
    c.lane = threadIdx.x & 63;
    c.g = c.lane >> 4;
    c.j = c.lane & 15;
    c.wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    c.nw = blockDim.x >> 6;
    c.gl = blockIdx.x * W + c.j;
    c.writer = c.g == 0;
    return c;
}

__device__ __forceinline__ int rowGroup() { return (threadIdx.x >> 4) & 3; }
__device__ __forceinline__ int instLane() { return threadIdx.x & 15; }

// View of a region: v[e] is element e of this lane's instance (per-lane e), a global-memory access.
template <typename T>
struct TV {
    T *p;   // this workgroup's slab of the region
    int j;  // instance within the workgroup
    // the lane's part of the address is a 32-bit byte offset from a scalar base: a workgroup's slab of a
    // region stays below 4 GiB (a batch of larger ones, at least 64 instances and 19 regions, exceeds the card)
    __device__ __forceinline__ SPK_GLOBAL T &operator[](long e) const {
        return *(SPK_GLOBAL T *) ((SPK_GLOBAL char *) p + ((unsigned) e * W + j) * (unsigned) sizeof(T));
    }
    __device__ __forceinline__ TV shift(long e0) const { return TV{p + e0 * W, j}; }
};

// A wave's LDS staging slices.
template <typename T>
using SP = SPK_LDS T *;

template <typename T>
__device__ __forceinline__ TV<T> tview(T *region, long rows, int j) {
    return TV<T>{region + (long) blockIdx.x * rows * W, j};
}

// Sum (max) over the four lanes of one instance; every one of them receives the same value.
template <typename T>
__device__ __forceinline__ T sumG(T v) {
    v += __shfl_xor(v, 16);
    v += __shfl_xor(v, 32);
    return v;
}
template <typename T>
__device__ __forceinline__ T maxG(T v) {
    v = fmax(v, __shfl_xor(v, 16));
    v = fmax(v, __shfl_xor(v, 32));
    return v;
}

// Which lane receives which row of a product: v_mfma_f32_16x16x4f32 gives lane (g, j) rows
// 16 t + 4 g + q of tile t in its four accumulator entries q, v_mfma_f64_16x16x4f64 rows
// 16 t + 4 q + g.  Lane g owns those rows of every node block, (r / 4) % 4 == g in FP32 and
// r % 4 == g in FP64.
template <typename T>
struct RowMap;
template <>
struct RowMap<float> {
    __device__ static __forceinline__ int row(int t, int g, int q) { return 16 * t + 4 * g + q; }
};
template <>
struct RowMap<double> {
    __device__ static __forceinline__ int row(int t, int g, int q) { return 16 * t + 4 * q + g; }
};

// The rows r < len this lane owns, f(r) for each.
template <typename T, typename F>
__device__ __forceinline__ void forRows(int len, F f) {
    const int g = rowGroup();
    for (int t = 0; 16 * t < len; t++) {
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int r = RowMap<T>::row(t, g, q);
            if (r < len) f(r);
        }
    }
}

template <typename T, int NT>
__device__ __forceinline__ void zeroTiles(Acc<T> (&a)[NT]) {
#pragma unroll
    for (int t = 0; t < NT; t++) a[t] = Acc<T>{T(0), T(0), T(0), T(0)};
}

// Row block r0 .. (a multiple of 64) of node n's packed factor (PTab): 1, 2 or 4 row tiles.
template <typename T>
__device__ __forceinline__ CP<T> packed(const SPK_CONST PTab<T> &t, int n, int r0) {
    return cst(t.data) + (size_t) cst(t.idx)[n] * t.stride + (size_t) (r0 >> 6) * ((t.cols + 15) >> 4) * 1024;
}

// acc[t] += M[16 t + i][c] x(c) summed over c < cols for the row tiles of M; x(c) is this lane's instance's
// entry c.  The factors are packed for this (PTab): 16 columns of a row tile are one run of 64 lanes x 4
// entries, so an operand of four k-steps is one 16-byte load a lane (two in FP64) at a scalar base, with
// no clamping (the padding is zero), where the column-major table took four 4-byte loads of four 64-byte
// runs each, and their addresses.  The vector's entries of up to
// 64 columns are requested together in FP32 (16 in FP64, whose registers they would take).  Code size
// matters at 17 call sites: with the factor's loads and the products of 64 columns unrolled as well T was
// 300 KB of code and 3 times slower.  Columns past the end enter with a valid entry of x against the
// packing's zeros.
template <typename T, int NT, typename XF>
__device__ __forceinline__ void mma(Acc<T> (&acc)[NT], CP<T> M, int cols, XF x) {
    typedef T Vec4 __attribute__((ext_vector_type(4)));
    const int g = rowGroup();
    const SPK_CONST Vec4 *base = (const SPK_CONST Vec4 *) M;
    const unsigned lane = threadIdx.x & 63;
    auto loadX = [&](int c0, T *b) {
#pragma unroll
        for (int s = 0; s < 4; s++) b[s] = x(min(c0 + 4 * s + g, cols - 1));
    };
    auto step = [&](const T *b) {
        Vec4 a[NT];
#pragma unroll
        for (int t = 0; t < NT; t++) a[t] = base[t * 64 + lane];
        base += NT * 64;
#pragma unroll
        for (int s = 0; s < 4; s++)
#pragma unroll
            for (int t = 0; t < NT; t++) acc[t] = mfma(a[t][s], b[s], acc[t]);
    };
    if constexpr (sizeof(T) == 4) {
#pragma unroll 1
        for (int c0 = 0; c0 < cols; c0 += 64) {
            T b[16];
#pragma unroll
            for (int k = 0; k < 4; k++)
                if (c0 + 16 * k < cols) loadX(c0 + 16 * k, b + 4 * k);
#pragma unroll
            for (int k = 0; k < 4; k++)
                if (c0 + 16 * k < cols) step(b + 4 * k);
        }
    } else {
#pragma unroll 1
        for (int c0 = 0; c0 < cols; c0 += 16) {
            T b[4];
            loadX(c0, b);
            step(b);
        }
    }
}

// The wave's LDS slice: the accumulators of 64 rows, or two staged vectors of 32 rows.
template <typename T>
__device__ __forceinline__ SP<T> waveStage() {
    __shared__ __align__(32) T stage[MAXW * 2 * STG];
    return (SP<T>) (stage + (threadIdx.x >> 6) * 2 * STG);
}

// f(row, value) for the rows < `rows` of a row block that this lane owns, straight from the registers
// (for few rows or a short f: the code of f is repeated for every one).
template <int NT, typename T, typename F>
__device__ __forceinline__ void eachOut(Acc<T> (&acc)[NT], int rows, F f) {
    const int g = rowGroup();
#pragma unroll
    for (int t = 0; t < NT; t++) {
        if (16 * t < rows) {
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int r = RowMap<T>::row(t, g, q);
                T v = acc[t][q];
                if (r < rows) f(r, v);
                acc[t][q] = v;
            }
        }
    }
}

// The same through the lane's own words of the LDS slice, so that one loop over the row tiles serves
// any number of them (each lane's four values of a tile are contiguous: no bank conflicts).  The
// return value of f replaces the staged one; again(f) visits the rows once more.
template <typename T>
struct StagedOut {
    typedef T Vec4 __attribute__((ext_vector_type(4)));
    SPK_LDS Vec4 *st;
    int rows;
    template <int NT>
    __device__ __forceinline__ StagedOut(const Acc<T> (&acc)[NT], int nrows) : rows(nrows) {
        st = (SPK_LDS Vec4 *) waveStage<T>() + (threadIdx.x & 63);
#pragma unroll
        for (int t = 0; t < NT; t++) st[t * 64] = acc[t];
    }
    template <bool KEEP, typename F>
    __device__ __forceinline__ void each(F f) {
        const int g = rowGroup();
#pragma unroll 1
        for (int t = 0; 16 * t < rows; t++) {
            Vec4 v = st[t * 64];
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int r = RowMap<T>::row(t, g, q);
                if (r < rows) v[q] = f(r, v[q]);
            }
            if (KEEP) st[t * 64] = v;
        }
    }
};

// out(r, y_r) for every row r < rows this lane owns, y = the sum of the products terms(acc, r0)
// accumulates (calls of mma on the row block at r0 of each term's matrix), 64 rows at a time.
// STAGED: the outputs pass through the LDS slice (which must be free), else straight from registers.
template <int NT, bool STAGED, typename T, typename Terms, typename F>
__device__ __forceinline__ void gemvBlock(int r0, int rows, Terms &terms, F &out) {
    Acc<T> a[NT];
    zeroTiles<T>(a);
    terms(a, r0);
    if constexpr (STAGED) {
        StagedOut<T> s(a, rows);
        s.template each<false>([&](int r, T v) {
            out(r0 + r, v);
            return v;
        });
    } else {
        eachOut<NT, T>(a, rows, [&](int r, T v) { out(r0 + r, v); });
    }
}

template <typename T, bool STAGED = true, typename Terms, typename F>
__device__ __forceinline__ void gemv(int rows, Terms terms, F out) {
#pragma unroll 1
    for (int r0 = 0; r0 < rows; r0 += 64) {
        const int rr = min(64, rows - r0);
        if (rr > 32) gemvBlock<4, STAGED, T>(r0, rr, terms, out);
        else if (rr <= 16) gemvBlock<1, STAGED, T>(r0, rr, terms, out);
        else gemvBlock<2, STAGED, T>(r0, rr, terms, out);
    }
}

template <typename T>
__device__ __forceinline__ T projBox(T v, T lb, T ub) {  // src/definitions.cu:38-52
    const int lower = (v <= lb), upper = (v >= ub);
    const T lbi = isinf(lb) ? T(0) : T(lower) * lb;
    const T ubi = isinf(ub) ? T(0) : T(upper) * ub;
    return v * T(1 - lower) * T(1 - upper) + lbi + ubi;
}

// ------------------------------------------------------------------ rows of a node's block
// Row (t, q) of the lane in a block of rows: a scalar base, the lane's own offset and an immediate, so a
// block's loads are one instruction each and all in flight together.  They are not conditional: rows past
// the block read what follows it in the region (the state buffer is padded by 64 rows) and are not used.
template <typename T>
__device__ __forceinline__ unsigned rowLane() {
    return ((unsigned) RowMap<T>::row(0, rowGroup(), 0) * W + instLane()) * (unsigned) sizeof(T);
}

template <typename T>
__device__ __forceinline__ SPK_GLOBAL T &rowAt(const TV<T> &v, long e0, unsigned lo, int t, int q) {
    return *(SPK_GLOBAL T *) ((SPK_GLOBAL char *) (v.p + e0 * W) + lo + RowMap<T>::row(t, 0, q) * W * (int) sizeof(T));
}

template <typename T, int NT>
__device__ __forceinline__ void loadRows(const TV<T> &v, long e0, unsigned lo, T (&out)[NT][4]) {
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
        for (int q = 0; q < 4; q++) out[t][q] = rowAt(v, e0, lo, t, q);
}

// The same of a per-node vector of a table (padded by 64 entries).
template <typename T, int NT>
__device__ __forceinline__ void loadRows(CP<T> p, T (&out)[NT][4]) {
    const int r0 = RowMap<T>::row(0, rowGroup(), 0);
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
        for (int q = 0; q < 4; q++) out[t][q] = (p + RowMap<T>::row(t, 0, q))[r0];
}

// f(t, q, r) for the rows r < `rows` of a block of up to NT tiles.
template <typename T, int NT, typename F>
__device__ __forceinline__ void eachRow(int rows, F f) {
    const int g = rowGroup();
#pragma unroll
    for (int t = 0; t < NT; t++) {
        if (16 * t < rows) {
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int r = RowMap<T>::row(t, g, q);
                if (r < rows) f(t, q, r);
            }
        }
    }
}

// What a handler reads of the rows of a block besides the products.  In FP32 it is requested before the
// products, so that it arrives with their operands; in FP64 after them, two row tiles at a time (the
// registers do not hold more).
template <typename T, int NT>
struct Pre {
    T a[NT][4], b[NT][4];
};
template <typename T>
constexpr bool EARLY = sizeof(T) == 4;

// f(first tile, its accumulators) for the parts of NT row tiles that are handled together.
template <typename T, int NT, typename F>
__device__ __forceinline__ void eachPart(Acc<T> (&a)[NT], F f) {
    constexpr int CH = EARLY<T> ? NT : (NT < 2 ? NT : 2);
#pragma unroll
    for (int t0 = 0; t0 < NT; t0 += CH) {
        Acc<T> part[CH];
#pragma unroll
        for (int t = 0; t < CH; t++) part[t] = a[t0 + t];
        f(t0, part);
#pragma unroll
        for (int t = 0; t < CH; t++) a[t0 + t] = part[t];
    }
}

// ------------------------------------------------------------------ L* per node
// src/operator.cuh:63-82; src/costs.cuh:162-195 (quadratic), :418-458 (quadratic+linear);
// src/constraints.cuh:171-191 (rectangle), :265-286 (polyhedron).
// The handler gets every entry of this lane's instance in exactly one lane: one(kind, k, value) with kind
// 2 = y (k < yD), 3 = s, 4 = t, and for blocks of x (kind 0) and u (kind 1) rows, at element e0 of the
// primal part, load(e0, lo, pre) and then rows(kind, k0, e0, lo, rows, values, pre).
// A node is a chain of memory round trips (about 2 us each when all CUs are busy), so they are few: the
// operands of up to 64 columns, the constraint's dual rows and the handler's rows go out together.
template <int NT, typename T, typename H, typename Terms, typename Extra>
__device__ __forceinline__ void adjBlock(const TV<T> &d, int kind, int k0, long e0, long ec, bool rect, int rows, Terms &terms,
                                         Extra &extra, H &h) {
    const unsigned lo = rowLane<T>();
    Pre<T, NT> all;
    T crAll[NT][4];
    if (EARLY<T>) {
        h.load(e0, lo, all);
        if (rect) loadRows(d, ec, lo, crAll);
    }
    Acc<T> acc[NT];
    zeroTiles<T>(acc);
    terms(acc, k0);
    eachPart<T, NT>(acc, [&](int t0, auto &a) {
        constexpr int CH = std::extent_v<std::remove_reference_t<decltype(a)>>;
        auto finish = [&](auto &pre, auto &cr) {
            if (rect) {
#pragma unroll
                for (int t = 0; t < CH; t++)
#pragma unroll
                    for (int q = 0; q < 4; q++) a[t][q] += cr[t][q];
            }
            extra(a, k0 + 16 * t0, rows - 16 * t0);
            h.rows(kind, k0 + 16 * t0, e0 + 16 * t0, lo, rows - 16 * t0, a, pre);
        };
        if constexpr (EARLY<T>) {
            finish(all, crAll);
        } else if (16 * t0 < rows) {
            Pre<T, CH> pre;
            T cr[CH][4];
            h.load(e0 + 16 * t0, lo, pre);
            if (rect) loadRows(d, ec + 16 * t0, lo, cr);
            finish(pre, cr);
        }
    });
}

template <typename T, typename H>
__device__ __forceinline__ void adjNode(LP<T> P, const TV<T> &d, int n, H &h) {
    const int nx = P.nx, nu = P.nu, nxu = nx + nu, d4 = nxu + 2;
    const bool first = rowGroup() == 0;
    auto blocks = [&](int kind, long e0, long ec, bool rect, int rows, auto terms, auto extra) {
#pragma unroll 1
        for (int r0 = 0; r0 < rows; r0 += 64) {
            const int rr = min(64, rows - r0);
            if (rr > 32) adjBlock<4>(d, kind, r0, e0 + r0, ec + r0, rect, rr, terms, extra, h);
            else if (rr <= 16) adjBlock<1>(d, kind, r0, e0 + r0, ec + r0, rect, rr, terms, extra, h);
            else adjBlock<2>(d, kind, r0, e0 + r0, ec + r0, rect, rr, terms, extra, h);
        }
    };
    if (n < P.nl) {
        const T II = d[P.oII + n];
        if (first) h.one(3, 0, II);
        CP<T> bn = tab(P.b, n);
        forRows<T>(P.yD, [&](int k) { h.one(2, k, d[P.oI + (long) n * P.yD + k] - bn[k] * II); });
        const long b3 = P.oIII + (long) n * P.con3;
        const int c0 = cst(P.chFrom)[n], nc = cst(P.numCh)[n];
#pragma unroll 1
        for (int part = 0; part < 2; part++) {  // x rows, then u rows
            const int rows = part == 0 ? nx : nu;
            blocks(
                part, part == 0 ? P.oX + (long) n * nx : P.oU + (long) n * nu, b3 + part * nx, P.ncon == CON_RECT_DEV, rows,
                [&](auto &acc, int r0) {
                    if (P.ncon == CON_POLY_DEV)
                        mma<T>(acc, packed(part == 0 ? P.pGTx : P.pGTu, n, r0), P.con3, [&](int cc) { return d[b3 + cc]; });
                    if (P.ncost == COST_LIN_DEV) return;  // elementwise below
                    for (int ci = 0; ci < nc; ci++) {  // children accumulate (src/costs.cuh:172-177)
                        const long iv = P.oIV + (long) (c0 + ci) * d4 + part * nx;
                        mma<T>(acc, packed(part == 0 ? P.psQ : P.psR, c0 + ci, r0), rows, [&](int cc) { return d[iv + cc]; });
                    }
                },
                [&](auto &acc, int r0, int rr) {
                    if (P.ncost == COST_LIN_DEV) {  // q_j sum_j, r_j sum_j (src/costs.cuh:274-285)
                        for (int ci = 0; ci < nc; ci++) {
                            const int j = c0 + ci;
                            CP<T> qj = (part == 0 ? tab(P.q, j) : tab(P.r, j)) + r0;
                            const T sj = d[P.oIV + j];
                            eachOut<std::extent_v<std::remove_reference_t<decltype(acc)>>, T>(acc, rr,
                                                                                             [&](int r, T &v) { v += qj[r] * sj; });
                        }
                    } else if (P.ncost == COST_QUADLIN_DEV) {
                        for (int ci = 0; ci < nc; ci++) {
                            const int j = c0 + ci;
                            const long iv = P.oIV + (long) j * d4;
                            const T a = d[iv + nxu], bb = d[iv + nxu + 1];
                            CP<T> qj = (part == 0 ? tab(P.q, j) : tab(P.r, j)) + r0;
                            eachOut<std::extent_v<std::remove_reference_t<decltype(acc)>>, T>(acc, rr, [&](int r, T &v) {
                                const T qr = qj[r];
                                v = v - T(0.5) * qr * a - T(0.5) * qr * bb;
                            });
                        }
                    }
                });
        }
    } else {
        const int l = n - P.nl;
        const long b5 = P.oV + (long) l * P.con5;
        const bool lin = P.lcost == COST_LIN_DEV;  // block VI = (sum of every leaf; set of every leaf)
        const long vi = P.oVI + (long) l * (lin ? 1 : nx + 2);
        const T a = lin ? T(0) : d[vi + nx], bb = lin ? T(0) : d[vi + nx + 1];
        blocks(
            0, P.oX + (long) n * nx, b5, P.lcon == CON_RECT_DEV, nx,
            [&](auto &acc, int r0) {
                if (P.lcon == CON_POLY_DEV) mma<T>(acc, packed(P.plGT, l, r0), P.con5, [&](int cc) { return d[b5 + cc]; });
                if (!lin) mma<T>(acc, packed(P.plsQ, l, r0), nx, [&](int cc) { return d[vi + cc]; });
            },
            [&](auto &acc, int r0, int rr) {
                if (!lin && P.lcost != COST_QUADLIN_DEV) return;
                CP<T> lq = tab(P.lq, l) + r0;
                const T sl = lin ? d[vi] : T(0);  // q sum_l (src/costs.cuh:289-292)
                eachOut<std::extent_v<std::remove_reference_t<decltype(acc)>>, T>(acc, rr, [&](int r, T &v) {
                    const T qr = lq[r];
                    if (lin) v += qr * sl;
                    else v = v - T(0.5) * qr * a - T(0.5) * qr * bb;
                });
            });
        if (first) h.one(3, 0, lin ? d[P.oVI + P.nlf + l] : (a + bb) * T(0.5));
    }
    if (first) {
        if (P.ncost == COST_LIN_DEV) {
            h.one(4, 0, d[P.oIV + P.N + n]);  // t <- set, every node (src/costs.cuh:286)
        } else if (n >= 1) {
            const long iv = P.oIV + (long) n * d4;
            h.one(4, 0, (d[iv + nxu] + d[iv + nxu + 1]) * T(0.5));
        } else {
            h.one(4, 0, T(0));
        }
    }
}

// ------------------------------------------------------------------ L per node
// src/operator.cuh:41-60; src/costs.cuh:126-160, :379-416; src/constraints.cuh:158-169, :251-263.
// pv(e) is element e of the primal vector, pv.rows(e0, lo, v) the lane's rows of a block.
// Handler: elemI(n, k, v), elemII(n, v) (row group 0 only), elemBox(e, v, lb, ub) for polyhedral rows;
// load(e0, lo, pre) and boxRows(e0, lo, rows, v, lb, ub, pre) for the box blocks III and V.  SOC blocks
// (IV and VI): socBegin(); with up to 64 states socIn(e0, lo, rows, values, pre, trans) for its row tiles,
// m = socScale(base, dim, h, trans) for its last two entries, which both carry h, and socOut(e0, lo, rows,
// values, m); with more, socPart(e, v, trans) for the owned rows of all but the last two entries and
// socEnd(base, n1, n2, h, trans).
template <int NT, typename T, typename PV, typename H>
__device__ __forceinline__ void boxTiles(long e0, long eb, int rows, CP<T> lb, CP<T> ub, PV &pv, H &h) {
    const unsigned lo = rowLane<T>();
#pragma unroll 1
    for (int r0 = 0; r0 < rows; r0 += 16 * NT) {
        Pre<T, NT> pre;
        T v[NT][4], l[NT][4], u[NT][4];
        pv.rows(e0 + r0, lo, v);
        h.load(eb + r0, lo, pre);
        loadRows(lb + r0, l);
        loadRows(ub + r0, u);
        h.boxRows(eb + r0, lo, min(16 * NT, rows - r0), v, l, u, pre);
    }
}

template <typename T, typename PV, typename H>
__device__ __forceinline__ void boxRows(long e0, long eb, int rows, CP<T> lb, CP<T> ub, PV &pv, H &h) {
    if (!EARLY<T> || rows <= 16) boxTiles<1>(e0, eb, rows, lb, ub, pv, h);
    else boxTiles<2>(e0, eb, rows, lb, ub, pv, h);
}

template <int NX, int NU, typename T, typename XF, typename UF, typename H>
__device__ __forceinline__ void socBlock(CP<T> MX, int nx, XF xf, CP<T> MU, int nu, UF uf, long base, T hv, CP<T> tr, H &h) {
    const unsigned lo = rowLane<T>();
    Pre<T, NX> px;
    Pre<T, NU> pu;
    if (EARLY<T>) {
        h.load(base, lo, px);
        if (nu > 0) h.load(base + nx, lo, pu);
    }
    Acc<T> ax[NX], au[NU];
    zeroTiles<T>(ax);
    zeroTiles<T>(au);
    mma<T>(ax, MX, nx, xf);
    if (nu > 0) mma<T>(au, MU, nu, uf);
    h.socBegin();
    auto in = [&](auto &acc, int n, long e0, CP<T> trn, auto &all) {
        constexpr int NT = std::extent_v<std::remove_reference_t<decltype(acc)>>;
        eachPart<T, NT>(acc, [&](int t0, auto &a) {
            constexpr int CH = std::extent_v<std::remove_reference_t<decltype(a)>>;
            if constexpr (EARLY<T>) {
                h.socIn(e0, lo, n, a, all, trn);
            } else if (16 * t0 < n) {
                Pre<T, CH> pre;
                h.load(e0 + 16 * t0, lo, pre);
                h.socIn(e0 + 16 * t0, lo, n - 16 * t0, a, pre, trn + 16 * t0);
            }
        });
    };
    in(ax, nx, base, tr, px);
    if (nu > 0) in(au, nu, base + nx, tr + nx, pu);
    const T mult = h.socScale(base, nx + nu + 2, hv, tr);
    h.socOut(base, lo, nx, ax, mult);
    if (nu > 0) h.socOut(base + nx, lo, nu, au, mult);
}

// By the row tiles of the state and input parts (nx <= 64, nu <= 32).
template <typename T, typename XF, typename UF, typename H>
__device__ __forceinline__ void socTiles(CP<T> MX, int nx, XF xf, CP<T> MU, int nu, UF uf, long base, T hv, CP<T> tr, H &h) {
    if (nx <= 16) {
        if (nu <= 16) socBlock<1, 1, T>(MX, nx, xf, MU, nu, uf, base, hv, tr, h);
        else socBlock<1, 2, T>(MX, nx, xf, MU, nu, uf, base, hv, tr, h);
    } else if (nx <= 32) {
        if (nu <= 16) socBlock<2, 1, T>(MX, nx, xf, MU, nu, uf, base, hv, tr, h);
        else socBlock<2, 2, T>(MX, nx, xf, MU, nu, uf, base, hv, tr, h);
    } else {
        if (nu <= 16) socBlock<4, 1, T>(MX, nx, xf, MU, nu, uf, base, hv, tr, h);
        else socBlock<4, 2, T>(MX, nx, xf, MU, nu, uf, base, hv, tr, h);
    }
}

template <typename T, typename PV, typename H>
__device__ __forceinline__ void opNode(LP<T> P, int n, PV &pv, H &h) {
    const int nx = P.nx, nu = P.nu, nxu = nx + nu;
    const int g = rowGroup();
    if (n < P.nl) {
        CP<T> bn = tab(P.b, n);
        T by = T(0);
        forRows<T>(P.yD, [&](int k) {
            const T yk = pv(P.oY + (long) n * P.yD + k);
            by += bn[k] * yk;
            h.elemI(n, k, yk);
        });
        by = sumG(by);
        if (g == 0) h.elemII(n, pv(P.oS + n) - by);
        const long base = P.oIII + (long) n * P.con3;
        if (P.ncon == CON_RECT_DEV) {
            CP<T> lb = tab(P.nLB, n), ub = tab(P.nUB, n);
            boxRows(P.oX + (long) n * nx, base, nx, lb, ub, pv, h);
            boxRows(P.oU + (long) n * nu, base + nx, nu, lb + nx, ub + nx, pv, h);
        } else if (P.ncon == CON_POLY_DEV) {
            CP<T> lb = tab(P.nLB, n), ub = tab(P.nUB, n);
            gemv<T>(
                P.con3,
                [&](auto &acc, int r0) {
                    mma<T>(acc, packed(P.pG, n, r0), nxu, [&](int cc) {
                        return cc < nx ? pv(P.oX + (long) n * nx + cc) : pv(P.oU + (long) n * nu + cc - nx);
                    });
                },
                [&](int r, T v) { h.elemBox(base + r, v, lb[r], ub[r]); });
        }
    }
    if (P.ncost == COST_LIN_DEV) {  // IV: (q_n' x_anc + r_n' u_anc, t_n), node 0 (0, t_0) (src/costs.cuh:261-267)
        T sum = T(0);
        if (n >= 1) {
            const int a = cst(P.anc)[n];
            CP<T> qn = tab(P.q, n), rn = tab(P.r, n);
            T pq = T(0), pr = T(0);
            forRows<T>(nx, [&](int k) { pq += qn[k] * pv(P.oX + (long) a * nx + k); });
            forRows<T>(nu, [&](int k) { pr += rn[k] * pv(P.oU + (long) a * nu + k); });
            sum = sumG(pq) + sumG(pr);
        }
        if (g == 0) h.lin(P.oIV + n, P.oIV + P.N + n, sum, pv(P.oT + n));
    } else {  // IV
        const long base = P.oIV + (long) n * (nxu + 2);
        CP<T> tr = tab(P.trans, n);
        if (n >= 1) {
            const int a = cst(P.anc)[n];
            auto xa = [&](int cc) { return pv(P.oX + (long) a * nx + cc); };
            auto ua = [&](int cc) { return pv(P.oU + (long) a * nu + cc); };
            T hv = pv(P.oT + n) * T(0.5);
            if (P.ncost == COST_QUADLIN_DEV) {
                CP<T> qn = tab(P.q, n), rn = tab(P.r, n);
                T pq = T(0), pr = T(0);
                forRows<T>(nx, [&](int k) { pq += qn[k] * xa(k); });
                forRows<T>(nu, [&](int k) { pr += rn[k] * ua(k); });
                pq = sumG(pq);
                pr = sumG(pr);
                hv = hv + T(-0.5) * pq;
                hv = hv + T(-0.5) * pr;
            }
            if (nx <= 64) {  // the block's entries stay in registers
                socTiles<T>(packed(P.psQ, n, 0), nx, xa, packed(P.psR, n, 0), nu, ua, base, hv, tr, h);
            } else {
                h.socBegin();
                gemv<T>(
                    nx, [&](auto &acc, int r0) { mma<T>(acc, packed(P.psQ, n, r0), nx, xa); },
                    [&](int r, T v) { h.socPart(base + r, v, tr[r]); });
                gemv<T>(
                    nu, [&](auto &acc, int r0) { mma<T>(acc, packed(P.psR, n, r0), nu, ua); },
                    [&](int r, T v) { h.socPart(base + nx + r, v, tr[nx + r]); });
                h.socEnd(base, nx, nu, hv, tr);
            }
        } else {
            h.socBegin();
            forRows<T>(nx, [&](int r) { h.socPart(base + r, T(0), tr[r]); });
            forRows<T>(nu, [&](int r) { h.socPart(base + nx + r, T(0), tr[nx + r]); });
            h.socEnd(base, nx, nu, T(0), tr);
        }
    }
    if (n >= P.nl) {  // V and VI
        const int l = n - P.nl;
        const long b5 = P.oV + (long) l * P.con5;
        if (P.lcon == CON_RECT_DEV) {
            boxRows(P.oX + (long) n * nx, b5, nx, tab(P.lLB, l), tab(P.lUB, l), pv, h);
        } else if (P.lcon == CON_POLY_DEV) {
            CP<T> lb = tab(P.lLB, l), ub = tab(P.lUB, l);
            gemv<T>(
                P.con5,
                [&](auto &acc, int r0) { mma<T>(acc, packed(P.plG, l, r0), nx, [&](int cc) { return pv(P.oX + (long) n * nx + cc); }); },
                [&](int r, T v) { h.elemBox(b5 + r, v, lb[r], ub[r]); });
        }
        if (P.lcost == COST_LIN_DEV) {  // VI: (q' x_l, s_l) (src/costs.cuh:269-272)
            CP<T> lq = tab(P.lq, l);
            T pq = T(0);
            forRows<T>(nx, [&](int k) { pq += lq[k] * pv(P.oX + (long) n * nx + k); });
            pq = sumG(pq);
            if (g == 0) h.lin(P.oVI + l, P.oVI + P.nlf + l, pq, pv(P.oS + n));
            return;
        }
        const long base = P.oVI + (long) l * (nx + 2);
        CP<T> tr = tab(P.ltrans, l);
        auto xl = [&](int cc) { return pv(P.oX + (long) n * nx + cc); };
        T hs = pv(P.oS + n) * T(0.5);
        if (P.lcost == COST_QUADLIN_DEV) {
            CP<T> lq = tab(P.lq, l);
            T pq = T(0);
            forRows<T>(nx, [&](int k) { pq += lq[k] * xl(k); });
            pq = sumG(pq);
            hs = hs + T(-0.5) * pq;
        }
        if (nx <= 16) {
            socBlock<1, 1, T>(packed(P.plsQ, l, 0), nx, xl, (CP<T>) nullptr, 0, xl, base, hs, tr, h);
        } else if (nx <= 32) {
            socBlock<2, 1, T>(packed(P.plsQ, l, 0), nx, xl, (CP<T>) nullptr, 0, xl, base, hs, tr, h);
        } else if (nx <= 64) {
            socBlock<4, 1, T>(packed(P.plsQ, l, 0), nx, xl, (CP<T>) nullptr, 0, xl, base, hs, tr, h);
        } else {
            h.socBegin();
            gemv<T>(
                nx, [&](auto &acc, int r0) { mma<T>(acc, packed(P.plsQ, l, r0), nx, xl); },
                [&](int r, T v) { h.socPart(base + r, v, tr[r]); });
            h.socEnd(base, nx, 0, hs, tr);
        }
    }
}

// Primal vectors of opNode: 2 xbar - z, and one vector.
template <typename T>
struct Reflected {
    TV<T> cand, z;
    __device__ __forceinline__ T operator()(long e) const { return cand[e] * T(2) - z[e]; }
    template <int NT>
    __device__ __forceinline__ void rows(long e0, unsigned lo, T (&v)[NT][4]) const {
        T c[NT][4];
        loadRows(cand, e0, lo, c);
        loadRows(z, e0, lo, v);
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int q = 0; q < 4; q++) v[t][q] = c[t][q] * T(2) - v[t][q];
    }
};
template <typename T>
struct Plain {
    TV<T> y;
    __device__ __forceinline__ T operator()(long e) const { return y[e]; }
    template <int NT>
    __device__ __forceinline__ void rows(long e0, unsigned lo, T (&v)[NT][4]) const { loadRows(y, e0, lo, v); }
};

// Dual prox of the CP step (src/cache.cuh:770-789): w = (L gamma + z_d)/gamma + c and
// cand_d = gamma (w - Pi(w)), Pi the masked NNOC (src/risks.cuh:99-106), NNOC (src/cones.cuh:134-137),
// box (src/constraints.cuh:70-74) or SOC (src/projections.cuh:102-128).  SOC blocks of up to 64 states
// keep w in registers (socRegs); larger ones stage it in cand_d (each lane its own rows), accumulate
// |w|^2 and rescale in socEnd.
template <typename T>
struct Prox {
    LP<T> P;
    TV<T> zd, cd;
    T ss;
    __device__ __forceinline__ T wAt(T Lv, T z, T tr) const { return (Lv * P.gamma + z) * P.gammaRecip + tr; }
    __device__ __forceinline__ T wOf(T Lv, long e, T tr) const { return wAt(Lv, zd[e], tr); }
    __device__ __forceinline__ void elemI(int n, int k, T v) {
        const long e = P.oI + (long) n * P.yD + k;
        const T w = wOf(v, e, T(0));
        const int idx = (k < 2 * cst(P.numCh)[n]) && (w < T(0));
        cd[e] = (w - T(1 - idx) * w) * P.gamma;
    }
    __device__ __forceinline__ void elemII(int n, T v) {
        const long e = P.oII + n;
        const T w = wOf(v, e, T(0));
        cd[e] = (w - fmax(T(0), w)) * P.gamma;
    }
    __device__ __forceinline__ void elemBox(long e, T v, T lb, T ub) {
        const T w = wOf(v, e, T(0));
        cd[e] = (w - projBox(w, lb, ub)) * P.gamma;
    }
    template <int NT>
    __device__ __forceinline__ void load(long e0, unsigned lo, Pre<T, NT> &p) const { loadRows(zd, e0, lo, p.a); }
    template <int NT>
    __device__ __forceinline__ void boxRows(long e0, unsigned lo, int rows, T (&v)[NT][4], T (&lb)[NT][4], T (&ub)[NT][4],
                                            Pre<T, NT> &p) {
        eachRow<T, NT>(rows, [&](int t, int q, int) {
            const T w = wAt(v[t][q], p.a[t][q], T(0));
            rowAt(cd, e0, lo, t, q) = (w - projBox(w, lb[t][q], ub[t][q])) * P.gamma;
        });
    }
    __device__ __forceinline__ void socBegin() { ss = T(0); }
    __device__ __forceinline__ void socPart(long e, T v, T tr) {
        const T w = wOf(v, e, tr);
        cd[e] = w;
        ss += w * w;
    }
    // the factor of the block's vector part; the last two entries are written
    __device__ __forceinline__ T socScale(long base, int dim, T hv, CP<T> tr) {
        const long k1 = base + dim - 2, k2 = base + dim - 1;
        const T w1 = wOf(hv, k1, tr[dim - 2]);
        const T w2 = wOf(hv, k2, tr[dim - 1]);
        const T sq = sumG(ss) + w1 * w1;
        const T nrm = sqrt(sq), tl = w2;
        const int i1 = nrm <= tl;
        const int i2 = (nrm <= -tl) && !i1;
        const int i3 = !i1 && !i2;
        const T sc = (nrm + tl) / (T(2) * nrm + T(1 - i3));
        const T mult = T(1 - i2) * (T(i3) * sc + T(1 - i3));
        if (rowGroup() == 0) {
            const T p1 = w1 * mult;
            const int i1b = (1 - i2) * (1 - i3);
            const T p2 = T(i1b) * (w2 * T(1 - i2)) + T((1 - i1b) * (1 - i2)) * (T(i3) * (sc * nrm - T(1)) + T(1));
            cd[k1] = (w1 - p1) * P.gamma;
            cd[k2] = (w2 - p2) * P.gamma;
        }
        return mult;
    }
    template <int NT>
    __device__ __forceinline__ void socIn(long, unsigned, int rows, Acc<T> (&a)[NT], Pre<T, NT> &p, CP<T> tr) {
        T tx[NT][4];
        loadRows(tr, tx);
        eachRow<T, NT>(rows, [&](int t, int q, int) {
            const T w = wAt(a[t][q], p.a[t][q], tx[t][q]);
            a[t][q] = w;
            ss += w * w;
        });
    }
    template <int NT>
    __device__ __forceinline__ void socOut(long e0, unsigned lo, int rows, Acc<T> (&a)[NT], T mult) {
        eachRow<T, NT>(rows, [&](int t, int q, int) {
            const T w = a[t][q];
            rowAt(cd, e0, lo, t, q) = (w - w * mult) * P.gamma;
        });
    }
    __device__ __forceinline__ void socEnd(long base, int n1, int n2, T hv, CP<T> tr) {
        const T mult = socScale(base, n1 + n2 + 2, hv, tr);
        auto rescale = [&](long e) {
            const T w = cd[e];
            cd[e] = (w - w * mult) * P.gamma;
        };
        forRows<T>(n1, [&](int r) { rescale(base + r); });
        forRows<T>(n2, [&](int r) { rescale(base + n1 + r); });
    }
    __device__ __forceinline__ void lin(long eSum, long eSet, T sum, T set) {
        const T ws = wOf(sum, eSum, T(0)), wt = wOf(set, eSet, T(0));
        cd[eSum] = (ws - projBelow(ws, wt)) * P.gamma;
        cd[eSet] = (wt - wt) * P.gamma;
    }
};

template <typename T>
__device__ __forceinline__ long primIndex(LP<T> P, int n, int kind, int k) {
    if (kind == 0) return P.oX + (long) n * P.nx + k;
    if (kind == 1) return P.oU + (long) n * P.nu + k;
    if (kind == 2) return P.oY + (long) n * P.yD + k;
    if (kind == 3) return P.oS + n;
    return P.oT + n;
}

// ell(y) = [L* y_d; L y_p] reductions: sum x.(y - gamma ell) and max |y/gamma - ell|
// (src/cache.cuh:722-734, 917-931), per lane over its own entries; elements are counted from the
// iterate's start in adjNode and from its dual part in opNode.
template <typename T>
struct Red {
    LP<T> P;
    TV<T> x, y;
    T dot, mx;
    long off;  // of the elements the handler is given
    T cross;   // adjoint part: sum of x_p . (L* y_d)
    int n;
    __device__ __forceinline__ void accV(T xk, T yk, T ell) {
        dot += xk * (ell * (-P.gamma) + yk);
        mx = fmax(mx, fabs(yk * P.gammaRecip - ell));
    }
    __device__ __forceinline__ void acc(long e, T ell) { accV(x[e], y[e], ell); }
    template <int NT>
    __device__ __forceinline__ void load(long e0, unsigned lo, Pre<T, NT> &p) const {
        loadRows(x, off + e0, lo, p.a);
        loadRows(y, off + e0, lo, p.b);
    }
    // adjoint
    __device__ __forceinline__ void one(int kind, int k, T v) {
        const long e = primIndex(P, n, kind, k);
        cross += x[e] * v;
        acc(e, v);
    }
    template <int NT>
    __device__ __forceinline__ void rows(int, int, long, unsigned, int rows, Acc<T> (&a)[NT], Pre<T, NT> &p) {
        eachRow<T, NT>(rows, [&](int t, int q, int) {
            cross += p.a[t][q] * a[t][q];
            accV(p.a[t][q], p.b[t][q], a[t][q]);
        });
    }
    // operator
    __device__ __forceinline__ void elemI(int n, int k, T v) { acc(off + P.oI + (long) n * P.yD + k, v); }
    __device__ __forceinline__ void elemII(int n, T v) { acc(off + P.oII + n, v); }
    __device__ __forceinline__ void elemBox(long e, T v, T, T) { acc(off + e, v); }
    template <int NT>
    __device__ __forceinline__ void boxRows(long, unsigned, int rows, T (&v)[NT][4], T (&)[NT][4], T (&)[NT][4], Pre<T, NT> &p) {
        eachRow<T, NT>(rows, [&](int t, int q, int) { accV(p.a[t][q], p.b[t][q], v[t][q]); });
    }
    __device__ __forceinline__ void socBegin() {}
    __device__ __forceinline__ void socPart(long e, T v, T) { acc(off + e, v); }
    template <int NT>
    __device__ __forceinline__ void socIn(long, unsigned, int rows, Acc<T> (&a)[NT], Pre<T, NT> &p, CP<T>) {
        eachRow<T, NT>(rows, [&](int t, int q, int) { accV(p.a[t][q], p.b[t][q], a[t][q]); });
    }
    template <int NT>
    __device__ __forceinline__ void socOut(long, unsigned, int, Acc<T> (&)[NT], T) {}
    __device__ __forceinline__ T socScale(long base, int dim, T hv, CP<T> tr) {
        socEnd(base, dim - 2, 0, hv, tr);
        return T(0);
    }
    __device__ __forceinline__ void socEnd(long base, int n1, int n2, T hv, CP<T>) {
        if (rowGroup() != 0) return;
        const int dim = n1 + n2 + 2;
        acc(off + base + dim - 2, hv);
        acc(off + base + dim - 1, hv);
    }
    __device__ __forceinline__ void lin(long eSum, long eSet, T sum, T set) {
        acc(off + eSum, sum);
        acc(off + eSet, set);
    }
};

// Raw values of L (opNode) and L* (adjNode) into `out` (its dual or primal part).
template <typename T>
struct Store {
    LP<T> P;
    TV<T> out;
    int n;
    template <int NT>
    __device__ __forceinline__ void load(long, unsigned, Pre<T, NT> &) const {}
    __device__ __forceinline__ void one(int kind, int k, T v) { out[primIndex(P, n, kind, k)] = v; }
    template <int NT>
    __device__ __forceinline__ void rows(int, int, long e0, unsigned lo, int rows, Acc<T> (&a)[NT], Pre<T, NT> &) {
        eachRow<T, NT>(rows, [&](int t, int q, int) { rowAt(out, e0, lo, t, q) = a[t][q]; });
    }
    __device__ __forceinline__ void elemI(int n, int k, T v) { out[P.oI + (long) n * P.yD + k] = v; }
    __device__ __forceinline__ void elemII(int n, T v) { out[P.oII + n] = v; }
    __device__ __forceinline__ void elemBox(long e, T v, T, T) { out[e] = v; }
    template <int NT>
    __device__ __forceinline__ void boxRows(long e0, unsigned lo, int rows, T (&v)[NT][4], T (&)[NT][4], T (&)[NT][4], Pre<T, NT> &) {
        eachRow<T, NT>(rows, [&](int t, int q, int) { rowAt(out, e0, lo, t, q) = v[t][q]; });
    }
    __device__ __forceinline__ void socBegin() {}
    __device__ __forceinline__ void socPart(long e, T v, T) { out[e] = v; }
    template <int NT>
    __device__ __forceinline__ void socIn(long e0, unsigned lo, int rows, Acc<T> (&a)[NT], Pre<T, NT> &, CP<T>) {
        eachRow<T, NT>(rows, [&](int t, int q, int) { rowAt(out, e0, lo, t, q) = a[t][q]; });
    }
    template <int NT>
    __device__ __forceinline__ void socOut(long, unsigned, int, Acc<T> (&)[NT], T) {}
    __device__ __forceinline__ T socScale(long base, int dim, T hv, CP<T> tr) {
        socEnd(base, dim - 2, 0, hv, tr);
        return T(0);
    }
    __device__ __forceinline__ void socEnd(long base, int n1, int n2, T hv, CP<T>) {
        if (rowGroup() != 0) return;
        const int dim = n1 + n2 + 2;
        out[base + dim - 2] = hv;
        out[base + dim - 1] = hv;
    }
    __device__ __forceinline__ void lin(long eSum, long eSet, T sum, T set) {
        out[eSum] = sum;
        out[eSet] = set;
    }
};

// ------------------------------------------------------------------ T phases
// modifyPrimal + proxRootS (src/cache.cuh:748-753, 639-642); leaves seed q = -xbar (src/dynamics.cuh:79-81).
template <typename T>
struct Axpy {
    LP<T> P;
    TV<T> z, cand, qd;
    int n;
    template <int NT>
    __device__ __forceinline__ void load(long e0, unsigned lo, Pre<T, NT> &p) const { loadRows(z, e0, lo, p.a); }
    __device__ __forceinline__ void one(int kind, int k, T v) {
        const long e = primIndex(P, n, kind, k);
        T val = v * (-P.gamma) + z[e];
        if (kind == 3 && n == 0) val -= P.gamma;
        cand[e] = val;
    }
    template <int NT>
    __device__ __forceinline__ void rows(int, int k0, long e0, unsigned lo, int rows, Acc<T> (&a)[NT], Pre<T, NT> &p) {
        const bool leaf = n >= P.nl;
        eachRow<T, NT>(rows, [&](int t, int q, int) {
            const T val = a[t][q] * (-P.gamma) + p.a[t][q];
            rowAt(cand, e0, lo, t, q) = val;
            if (leaf) rowAt(qd, (long) n * P.nx + k0, lo, t, q) = -val;
        });
    }
};

template <typename T>
__device__ __forceinline__ void phaseAdj(LP<T> P, const Ctx &c, const TV<T> &z, const TV<T> &cand,
                                         const TV<T> &qd) {
    const TV<T> zd = z.shift(P.sPrim);
    for (int n = c.wave; n < P.N; n += c.nw) {
        Axpy<T> h{P, z, cand, qd, n};
        adjNode(P, zd, n, h);
    }
}

// Backward sweep step for node i (src/dynamics.cuh:85-139) with R~^-1 applied as one product.
// stg: this wave's two LDS slices of 32 rows x 16 instances.  NU: row tiles of the inputs (nu <= 32).
template <int NT, typename T, typename Terms>
__device__ __forceinline__ void dynBackRows(const TV<T> &cand, const TV<T> &qd, long ex, long eq, int r0, int rows, Terms &terms) {
    const unsigned lo = rowLane<T>();
    T xb[NT][4];
    if (EARLY<T>) loadRows(cand, ex + r0, lo, xb);
    Acc<T> acc[NT];
    zeroTiles<T>(acc);
    terms(acc, r0);
    if (!EARLY<T>) loadRows(cand, ex + r0, lo, xb);
    eachRow<T, NT>(rows, [&](int t, int q, int) { rowAt(qd, eq + r0, lo, t, q) = acc[t][q] - xb[t][q]; });
}

template <int NU, typename T>
__device__ __forceinline__ void dynBackward(LP<T> P, const TV<T> &cand, const TV<T> &qd, const TV<T> &dd, int i,
                                            int stage, SP<T> stg) {
    const int nx = P.nx, nu = P.nu;
    const int c0 = cst(P.chFrom)[i], nc = cst(P.numCh)[i];
    const int jj = instLane(), g = rowGroup();
    const unsigned lo = rowLane<T>();
    SP<T> e1 = stg, d1 = stg + STG;
    const long ub0 = P.oU + (long) i * nu;
    T ub[NU][4];
    loadRows(cand, ub0, lo, ub);
    // affine dynamics: the children's q enter as q_j + P_j e_j (src/dynamics.cuh:93-97)
    const bool affine = P.affine != 0;
    auto qv = [&](int j, int cc) { return affine ? qd[(long) j * nx + cc] + tab(P.Pe, j)[cc] : qd[(long) j * nx + cc]; };
    // e = ubar - sum_j B_j' q_j
    Acc<T> au[NU];
    zeroTiles<T>(au);
#pragma unroll 1
    for (int ci = 0; ci < nc; ci++) mma<T>(au, packed(P.pBTr, c0 + ci, 0), nx, [&](int cc) { return qv(c0 + ci, cc); });
    eachRow<T, NU>(nu, [&](int t, int q, int r) { e1[r * W + jj] = -au[t][q] + ub[t][q]; });
    __builtin_amdgcn_wave_barrier();
    // d = R~^-1 e
    zeroTiles<T>(au);
    mma<T>(au, packed(P.pRtInv, i, 0), nu, [&](int cc) -> T { return e1[cc * W + jj]; });
    __builtin_amdgcn_wave_barrier();
    eachRow<T, NU>(nu, [&](int t, int q, int r) {
        rowAt(dd, (long) i * nu, lo, t, q) = au[t][q];
        d1[r * W + jj] = au[t][q];
        e1[r * W + jj] = au[t][q] - ub[t][q];
    });
    __builtin_amdgcn_wave_barrier();
    if (stage == 0) return;
    // q_i = sum_j (APB_j d_i + ABKTr_j q_j) + K_i'(d_i - u_i) - x_i
    auto terms = [&](auto &acc, int r0) {
#pragma unroll 1
        for (int ci = 0; ci < nc; ci++) {
            const int j = c0 + ci;
            mma<T>(acc, packed(P.pAPB, j, r0), nu, [&](int cc) -> T { return d1[cc * W + jj]; });
            mma<T>(acc, packed(P.pABKTr, j, r0), nx, [&](int cc) { return qv(j, cc); });
        }
        mma<T>(acc, packed(P.pKTr, i, r0), nu, [&](int cc) -> T { return e1[cc * W + jj]; });
    };
    const long ex = P.oX + (long) i * nx, eq = (long) i * nx;
#pragma unroll 1
    for (int r0 = 0; r0 < nx; r0 += 64) {
        const int rr = min(64, nx - r0);
        if (rr > 32) dynBackRows<4>(cand, qd, ex, eq, r0, rr, terms);
        else if (rr <= 16) dynBackRows<1>(cand, qd, ex, eq, r0, rr, terms);
        else dynBackRows<2>(cand, qd, ex, eq, r0, rr, terms);
    }
}

// Kernel projection for nonleaf node i (src/cache.cuh:650-676); padded child slots enter as 0.
// In place: every entry is read (as a B operand) before any result is written.
template <typename T>
__device__ __forceinline__ void kernelProj(LP<T> P, const TV<T> &cand, int i) {
    const int yD = P.yD, E = P.E, nc = cst(P.numCh)[i], c0 = cst(P.chFrom)[i];
    auto vin = [&](int k) -> T {
        if (k < yD) return cand[P.oY + (long) i * yD + k];
        if (k < yD + E) return (k - yD < nc) ? cand[P.oT + c0 + (k - yD)] : T(0);
        return (k - yD - E < nc) ? cand[P.oS + c0 + (k - yD - E)] : T(0);
    };
    gemv<T>(
        P.nD, [&](auto &acc, int r0) { mma<T>(acc, packed(P.pNN, i, r0), P.nD, vin); },
        [&](int k, T v) {
            if (k < yD) cand[P.oY + (long) i * yD + k] = v;
            else if (k < yD + E) {
                if (k - yD < nc) cand[P.oT + c0 + (k - yD)] = v;
            } else if (k - yD - E < nc) {
                cand[P.oS + c0 + (k - yD - E)] = v;
            }
        });
}

// Forward rollout for node i (src/dynamics.cuh:144-173); affine dynamics add e_j to each child.
template <int NU, typename T>
__device__ __forceinline__ void dynForward(LP<T> P, const TV<T> &cand, const TV<T> &x0s, const TV<T> &dd, int i,
                                           SP<T> stg) {
    const int nx = P.nx, nu = P.nu;
    const int jj = instLane();
    const unsigned lo = rowLane<T>();
    SP<T> u1 = stg;
    T db[NU][4];
    loadRows(dd, (long) i * nu, lo, db);
    // x_0 is the (scaled) initial state; other nodes' x were written by their parent's step
    auto xv = [&](int cc) { return i == 0 ? x0s[cc] : cand[P.oX + (long) i * nx + cc]; };
    if (i == 0) forRows<T>(nx, [&](int r) { cand[P.oX + r] = x0s[r]; });
    Acc<T> au[NU];
    zeroTiles<T>(au);
    mma<T>(au, packed(P.pK, i, 0), nx, xv);
    eachRow<T, NU>(nu, [&](int t, int q, int r) {
        const T u = au[t][q] + db[t][q];
        rowAt(cand, P.oU + (long) i * nu, lo, t, q) = u;
        u1[r * W + jj] = u;
    });
    __builtin_amdgcn_wave_barrier();
    const int c0 = cst(P.chFrom)[i], nc = cst(P.numCh)[i];
#pragma unroll 1
    for (int ci = 0; ci < nc; ci++) {
        const int j = c0 + ci;
        const long ex = P.oX + (long) j * nx;
        gemv<T, false>(  // u1 stays in the LDS slice for the next child
            nx,
            [&](auto &acc, int r0) {
                mma<T>(acc, packed(P.pAB, j, r0), nx + nu, [&](int cc) -> T { return cc < nx ? xv(cc) : u1[(cc - nx) * W + jj]; });
            },
            [&](int r, T v) {
                if (P.affine) v += tab(P.e, j)[r];
                cand[ex + r] = v;
            });
    }
    __builtin_amdgcn_wave_barrier();
}

template <int NU, typename T>
__device__ __forceinline__ void phaseProjTiles(LP<T> P, const Ctx &c, const TV<T> &cand, const TV<T> &qd, const TV<T> &dd,
                                               const TV<T> &x0s, bool doDyn, bool doKernel, SP<T> stg) {
    if (doDyn) {
        for (int stage = P.S - 2; stage >= 0; stage--) {
            const int f = cst(P.stageFrom)[stage], nStage = cst(P.stageTo)[stage] - f + 1;
            const int extra = (doKernel && stage == P.S - 2) ? P.nl : 0;
            for (int task = c.wave; task < nStage + extra; task += c.nw) {
                if (task < nStage) dynBackward<NU>(P, cand, qd, dd, f + task, stage, stg);
                else kernelProj(P, cand, task - nStage);
            }
            __syncthreads();
        }
        for (int stage = 0; stage <= P.S - 2; stage++) {
            const int f = cst(P.stageFrom)[stage], nStage = cst(P.stageTo)[stage] - f + 1;
            for (int task = c.wave; task < nStage; task += c.nw) dynForward<NU>(P, cand, x0s, dd, f + task, stg);
            __syncthreads();
        }
    } else if (doKernel) {
        for (int task = c.wave; task < P.nl; task += c.nw) kernelProj(P, cand, task);
        __syncthreads();
    }
}

template <typename T>
__device__ __forceinline__ void phaseProj(LP<T> P, const Ctx &c, const TV<T> &cand, const TV<T> &qd, const TV<T> &dd,
                                          const TV<T> &x0s, bool doDyn, bool doKernel, SP<T> stg) {
    if (P.nu <= 16) phaseProjTiles<1>(P, c, cand, qd, dd, x0s, doDyn, doKernel, stg);
    else phaseProjTiles<2>(P, c, cand, qd, dd, x0s, doDyn, doKernel, stg);  // nu <= 32 (checked on the host)
}

// modifyDual + proximalDual (src/cache.cuh:770-789) on 2 xbar - z_p.
template <typename T>
__device__ __forceinline__ void phaseDual(LP<T> P, const Ctx &c, const TV<T> &z, const TV<T> &cand) {
    Prox<T> h{P, z.shift(P.sPrim), cand.shift(P.sPrim), T(0)};
    Reflected<T> pv{cand, z};
    for (int n = c.wave; n < P.N; n += c.nw) opNode(P, n, pv, h);
}

// The CP operator T (src/cache.cuh:796-801): cand = T(z).
template <typename T>
__device__ __noinline__ void applyT(const LaneInst<T> *Pp, T *z, T *cand, long *phaseAcc) {
    LaneClock clk{wall_clock64(), phaseAcc};
    LP<T> P = *cst(uniformPtr(Pp));
    z = uniformPtr(z);
    cand = uniformPtr(cand);
    const Ctx c = ctx();
    const TV<T> zv = tview(z, P.sIter, c.j), cv = tview(cand, P.sIter, c.j);
    const TV<T> qd = tview(P.qd, (long) P.nx * P.N, c.j), dd = tview(P.dd, (long) P.nu * P.nl, c.j);
    const TV<T> x0s = tview(const_cast<T *>(P.x0s), P.nx, c.j);
    phaseAdj(P, c, zv, cv, qd);
    __syncthreads();
    clk.mark(PH_ADJ);
    phaseProj(P, c, cv, qd, dd, x0s, true, true, waveStage<T>());
    clk.mark(PH_PROJ);
    phaseDual(P, c, zv, cv);
    __syncthreads();
    clk.mark(PH_DUAL);
}

// Per-instance combination: the four row-group lanes, then the waves in wave order (LDS).
__device__ __forceinline__ double tileSum(double v, double *lds, const Ctx &c) {
    v = sumG(v);
    __syncthreads();
    if (c.g == 0) lds[c.wave * W + c.j] = v;
    __syncthreads();
    double s = 0.;
    for (int w = 0; w < c.nw; w++) s += lds[w * W + c.j];
    return s;
}

__device__ __forceinline__ double tileMax(double v, double *lds, const Ctx &c) {
    v = maxG(v);
    __syncthreads();
    if (c.g == 0) lds[c.wave * W + c.j] = v;
    __syncthreads();
    double s = 0.;
    for (int w = 0; w < c.nw; w++) s = fmax(s, lds[w * W + c.j]);
    return s;
}

// sum x.(y - gamma ell(y)) and max |y/gamma - ell(y)| per instance.
template <typename T>
__device__ __noinline__ DotMax<T> reduceEll(const LaneInst<T> *Pp, T *x, T *y, double *lds) {
    LP<T> P = *cst(uniformPtr(Pp));
    x = uniformPtr(x);
    y = uniformPtr(y);
    const Ctx c = ctx();
    const TV<T> xv = tview(x, P.sIter, c.j), yv = tview(y, P.sIter, c.j);
    const TV<T> yd = yv.shift(P.sPrim);
    Red<T> h{P, xv, yv, T(0), T(0), 0, T(0), 0};
    Plain<T> pv{yv};
    for (int n = c.wave; n < P.N; n += c.nw) {
        h.n = n;
        h.off = 0;
        adjNode(P, yd, n, h);
        h.off = P.sPrim;
        opNode(P, n, pv, h);
    }
    DotMax<T> r;
    r.dot = (T) tileSum((double) h.dot, lds, c);
    r.mx = (T) tileMax((double) h.mx, lds, c);
    r.cross = (T) tileSum((double) h.cross, lds, c);
    return r;
}

// c1 += x_p . (adjoint), c2 += (adjoint) . y_p.
template <typename T>
struct Dots {
    LP<T> P;
    TV<T> x, y;
    bool withY;
    int n;
    T c1, c2;
    template <int NT>
    __device__ __forceinline__ void load(long e0, unsigned lo, Pre<T, NT> &p) const {
        loadRows(x, e0, lo, p.a);
        if (withY) loadRows(y, e0, lo, p.b);
    }
    __device__ __forceinline__ void one(int kind, int k, T v) {
        const long e = primIndex(P, n, kind, k);
        c1 += x[e] * v;
        if (withY) c2 += v * y[e];
    }
    template <int NT>
    __device__ __forceinline__ void rows(int, int, long, unsigned, int rows, Acc<T> (&a)[NT], Pre<T, NT> &p) {
        eachRow<T, NT>(rows, [&](int t, int q, int) {
            c1 += p.a[t][q] * a[t][q];
            if (withY) c2 += a[t][q] * p.b[t][q];
        });
    }
};

// c1 = sum_p x_p . (L* x_d),  c2 = sum_p x_p . (L* y_d) + (L* x_d) . y_p (see the lane engine).
template <typename T>
__device__ __noinline__ Cross2<T> adjDots(const LaneInst<T> *Pp, T *x, T *y, double *lds, bool withY) {
    LP<T> P = *cst(uniformPtr(Pp));
    x = uniformPtr(x);
    y = uniformPtr(y);
    const Ctx c = ctx();
    const TV<T> xv = tview(x, P.sIter, c.j), yv = tview(y, P.sIter, c.j);
    const TV<T> xd = xv.shift(P.sPrim), yd = yv.shift(P.sPrim);
    T c1 = T(0), c2 = T(0);
    for (int n = c.wave; n < P.N; n += c.nw) {
        Dots<T> h{P, xv, yv, withY, n, c1, c2};
        adjNode(P, xd, n, h);
        c1 = h.c1;
        c2 = h.c2;
        if (withY) {
            Dots<T> hy{P, xv, yv, false, n, c2, T(0)};
            adjNode(P, yd, n, hy);
            c2 = hy.c1;
        }
    }
    Cross2<T> r;
    r.c1 = (T) tileSum((double) c1, lds, c);
    r.c2 = withY ? (T) tileSum((double) c2, lds, c) : T(0);
    return r;
}

// Iterate-wide pass: wave w takes a contiguous range of elements (a multiple of 4 long); lane
// (g, j) visits elements e0 + 4 s + g of instance j, so each access of the wave moves 4 rows x 16
// instances = 64 consecutive words, with U accesses in flight per lane.
template <int U, typename Ld, typename St>
__device__ __forceinline__ void pass(long n, const Ctx &c, Ld ld, St st) {
    using Vals = decltype(ld(0L));
    const long per = (((n + c.nw - 1) / c.nw) + 3) & ~3L;
    const long e0 = (long) c.wave * per, e1 = min(n, e0 + per);
    long b = e0;
#pragma unroll 1
    for (; b + 4 * U <= e1; b += 4 * U) {  // no conditions: all U loads are in flight together
        Vals v[U];
#pragma unroll
        for (int u = 0; u < U; u++) v[u] = ld(b + 4 * u + c.g);
#pragma unroll
        for (int u = 0; u < U; u++) st(b + 4 * u + c.g, v[u]);
    }
#pragma unroll 1
    for (; b < e1; b += 4)
        if (b + c.g < e1) st(b + c.g, ld(b + c.g));
}

// The tile engine as a policy of the lockstep solve.
struct Policy {
    template <typename T>
    using View = TV<T>;
    __device__ static Ctx ctx() { return tile::ctx(); }
    template <typename T>
    __device__ static TV<T> view(T *region, long rows, const Ctx &c) { return tview(region, rows, c.j); }
    template <int U, typename Ld, typename St>
    __device__ static void pass(long n, const Ctx &c, Ld ld, St st) { tile::pass<U>(n, c, ld, st); }
    __device__ static double sum(double v, double *lds, const Ctx &c) { return tileSum(v, lds, c); }
    __device__ static double max(double v, double *lds, const Ctx &c) { return tileMax(v, lds, c); }
    template <typename T>
    __device__ static void applyT(const LaneInst<T> *P, T *z, T *cand, long *phaseAcc) { tile::applyT(P, z, cand, phaseAcc); }
    template <typename T>
    __device__ static DotMax<T> reduceEll(const LaneInst<T> *P, T *x, T *y, double *lds) { return tile::reduceEll(P, x, y, lds); }
    template <typename T>
    __device__ static Cross2<T> adjDots(const LaneInst<T> *P, T *x, T *y, double *lds, bool withY) {
        return tile::adjDots(P, x, y, lds, withY);
    }
};

}  // namespace tile

template <typename T>
__global__ void __launch_bounds__(SPK_TILE_MAX_THREADS) SPK_TILE_KERNEL(k_tile_solve)(const LaneInst<T> *__restrict__ P, Out *outs) {
    __shared__ double lds[tile::MAXW * tile::W];
    __shared__ long phaseAcc[NUM_PHASES];
    lockstepSolve<T, tile::Policy>(P, outs, lds, phaseAcc);
}

// Single operators on every instance (parity tests): z = zio, cand = work[1].
template <typename T>
__global__ void __launch_bounds__(SPK_TILE_MAX_THREADS) SPK_TILE_KERNEL(k_tile_debug)(const LaneInst<T> *__restrict__ Pp, Out *outs,
                                                                     int op) {
    using namespace tile;
    __shared__ double lds[MAXW * W];
    LP<T> P = *cst(Pp);
    const Ctx c = ctx();
    T *z = P.zio, *cand = P.work[1];
    const TV<T> zv = tview(z, P.sIter, c.j), cv = tview(cand, P.sIter, c.j);
    if (op == 0) {  // L
        Store<T> h{P, cv.shift(P.sPrim), 0};
        Plain<T> pv{zv};
        for (int n = c.wave; n < P.N; n += c.nw) opNode(P, n, pv, h);
    } else if (op == 1) {  // L*
        const TV<T> zd = zv.shift(P.sPrim);
        for (int n = c.wave; n < P.N; n += c.nw) {
            Store<T> h{P, cv, n};
            adjNode(P, zd, n, h);
        }
    } else if (op == 2 || op == 3) {  // dynamics / kernel projection of the primal part
        tile::pass<16>(P.sPrim, c, [&](long e) { return zv[e]; }, [&](long e, T v) { cv[e] = v; });
        __syncthreads();
        const TV<T> qd = tview(P.qd, (long) P.nx * P.N, c.j), dd = tview(P.dd, (long) P.nu * P.nl, c.j);
        const TV<T> x0s = tview(const_cast<T *>(P.x0s), P.nx, c.j);
        if (op == 2)
            for (int n = c.wave; n < P.N; n += c.nw)
                if (n >= P.nl) forRows<T>(P.nx, [&](int r) { qd[(long) n * P.nx + r] = -cv[P.oX + (long) n * P.nx + r]; });
        __syncthreads();
        phaseProj(P, c, cv, qd, dd, x0s, op == 2, op == 3, waveStage<T>());
    } else if (op == 4) {  // T
        __shared__ long phaseAcc[NUM_PHASES];
        applyT(Pp, z, cand, phaseAcc);
    } else if (op == 5) {  // ell reductions
        const DotMax<T> r = reduceEll(Pp, z, cand, lds);
        if (c.wave == 0 && c.writer && c.gl < P.count) {
            outs[c.gl].w = (double) r.dot;
            outs[c.gl].err = (double) r.mx;
        }
    }
}

template __global__ void SPK_TILE_KERNEL(k_tile_solve)<float>(const LaneInst<float> *, Out *);
template __global__ void SPK_TILE_KERNEL(k_tile_solve)<double>(const LaneInst<double> *, Out *);
template __global__ void SPK_TILE_KERNEL(k_tile_debug)<float>(const LaneInst<float> *, Out *, int);
template __global__ void SPK_TILE_KERNEL(k_tile_debug)<double>(const LaneInst<double> *, Out *, int);

}  // namespace spk
