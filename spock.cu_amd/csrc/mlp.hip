// Learned warm start: an MLP x0 -> (standardized) primal-dual iterate, trained on solved
// iterates.  Hand-written kernels: a bf16 MFMA GEMM (FP32 accumulation) with fused bias / GELU /
// output affine epilogues, the GELU backward, column sums, the MSE loss and Adam.  Weights are kept
// as FP32 masters with bf16 copies that feed the matrix cores.
#include <hip/hip_runtime.h>
#include <hip/hip_bf16.h>
#include <math.h>

#include "engine.hpp"

namespace spk {
namespace mlp {

__device__ __forceinline__ unsigned short toBf16(float f) {  // round to nearest even
    unsigned int u = __float_as_uint(f);
    if ((u & 0x7f800000u) == 0x7f800000u) return (unsigned short) (u >> 16) | ((u & 0xffff) ? 0x40 : 0);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (unsigned short) (u >> 16);
}
__device__ __forceinline__ float fromBf16(unsigned short h) { return __uint_as_float(((unsigned int) h) << 16); }

__device__ __forceinline__ float gelu(float x) { return 0.5f * x * (1.f + erff(x * 0.70710678118654752f)); }
__device__ __forceinline__ float geluGrad(float x) {
    return 0.5f * (1.f + erff(x * 0.70710678118654752f)) + x * 0.3989422804014327f * expf(-0.5f * x * x);
}

// Adam (bias-corrected) on the FP32 masters of one block of parameters, refreshing the bf16 copies.
struct AdamArgs {
    float *w;
    unsigned short *wb;
    float *m, *v;
    float lr, b1, b2, eps, c1, c2;
};

__device__ __forceinline__ float adamStep(const AdamArgs &a, float gt, float w, float &m, float &v) {
    const float mt = a.b1 * m + (1.f - a.b1) * gt;
    const float vt = a.b2 * v + (1.f - a.b2) * gt * gt;
    m = mt;
    v = vt;
    return w - a.lr * (mt / a.c1) / (sqrtf(vt / a.c2) + a.eps);
}

// The products of the network, by operand layout and epilogue: forward layers (A contiguous along k, B = W
// along its columns), weight gradients (both along their rows), gradients of activations (both along k).
enum Epi {
    FWD_BIAS,    // C = acc + bias (FP32)
    FWD_GELU,    // C = acc + bias (FP32), Cb = gelu(C) (bf16)
    FWD_AFFINE,  // C = (acc + bias) * scale[col] + shift[col] (FP32)
    FWD_LANES,   // the same, rows being the instances of a shared batch in blocks of 16 (instance fastest)
    FWD_MSE,     // d = acc + bias - target: C = 2 d / count (FP32), Cb its bf16 copy, loss += d^2
    DW_STORE,    // C = acc
    DW_ADAM,     // acc is the gradient of the parameters of `adam` (and stored if C is given)
    DA_GELU,     // C = acc . gelu'(Z) (FP32), Cb its bf16 copy
};
constexpr bool kRows(int epi) { return epi < DW_STORE || epi == DA_GELU; }  // A contiguous along k
constexpr bool kCols(int epi) { return epi == DA_GELU; }                    // B contiguous along k

struct GemmArgs {
    const unsigned short *A;  // bf16, element (i, k) at A[i * lda + k], or A[i + k * lda] for weight gradients
    const unsigned short *B;  // bf16, element (k, j) at B[k * ldb + j], or B[k + j * ldb] (gradients of activations)
    long lda, ldb;
    int M, N, K;
    float *C;                 // FP32 output (row-major, ldc)
    long ldc;
    unsigned short *Cb;       // bf16 output (row-major, ldc)
    const float *bias, *scale, *shift;
    const float *Z;           // DA_GELU: the layer's sums (row-major, ldc)
    const float *target;      // FWD_MSE: row `row` is target[rows[row] * ldc ..]
    const int *rows;
    float inv;
    double *loss;             // FWD_MSE: one partial sum per workgroup
    AdamArgs adam;            // DW_ADAM
};

// ---------------------------------------------------------------- CDNA4 GEMM
// C (M x N) = A (M x K) . B (K x N) on v_mfma_f32_16x16x32_bf16 (gfx950).
// Lane layout of the instruction: first operand [i][k] from lane i + 16 (k / 8) item k % 8, second [k][j]
// from lane j + 16 (k / 8) item k % 8, D[i][j] in lane j + 16 (i / 4) item i % 4.  B goes in first, so that a
// lane holds four consecutive columns of a row and the epilogues move 128-bit vectors; FWD_LANES puts A first
// and holds four consecutive instances of a column.
// Both operands sit in LDS k-contiguous ([row][k] and [col][k]) in octets of 8 k, the octets of a row
// exchanged by octetOf(), so that a lane's fragment is one 128-bit read and neither the reads nor the
// writes hit a bank twice.  An operand that is contiguous along k moves to LDS in 128-bit vectors as it is.
// One contiguous along its rows / columns is read in pieces of 4 rows by 8 k (eight 64-bit loads), turned in
// registers by byte permutes and written as four 128-bit octets.  (Single 16-bit writes took most of the
// time of the output layer: 4,096 x 512 x 52,360 in 0.87 ms, now 0.53; the 858 MB it
// writes take 0.19 at the copy rate, and a tile of 8 k-steps waits for memory at its start and end.)  Rows need no alignment: vectors
// are loaded from any even address, so a 50-wide layer reads as the others do.

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
typedef f32x4 __attribute__((aligned(4))) f32x4Any;
typedef u32x4 __attribute__((aligned(2))) u32x4Any;
typedef u32x2 __attribute__((aligned(2))) u32x2Any;

__device__ __forceinline__ int octetOf(int row, int octet) { return octet ^ ((row ^ (row >> 3)) & 7); }

// Loads are unconditional (a branch per vector costs more than the vector): past the last row they read rows
// again, whose results are not used, and in the last k-step past the last k, which then becomes zero.

// Octet k0 .. k0 + 7 of a row of an operand contiguous along k; FULL: all of them are in range.
template <bool FULL>
__device__ __forceinline__ u32x4 loadOctet(const unsigned short *P, long ld, int row, int rowsTotal, int k0, int K) {
    P += (long) min(row, rowsTotal - 1) * ld;
    if (FULL) return *reinterpret_cast<const u32x4Any *>(P + k0);
    unsigned int e[8];
#pragma unroll
    for (int q = 0; q < 8; q++) e[q] = P[min(k0 + q, K - 1)];
    u32x4 o;
#pragma unroll
    for (int q = 0; q < 4; q++) o[q] = (k0 + 2 * q < K ? e[2 * q] : 0u) | (k0 + 2 * q + 1 < K ? e[2 * q + 1] << 16 : 0u);
    return o;
}

// Rows row .. row + 3 of eight k of an operand contiguous along its rows: r[i] holds k0 + i.  At the last rows
// the vector starts earlier, by earlyRows(), and is shifted when it is used.  (With fewer than 4 rows in all it
// reads on into the next k, or into the ROW_PAD elements that follow every operand.)
constexpr int ROW_PAD = 4;

__device__ __forceinline__ int earlyRows(int row, int rowsTotal) { return row - max(0, min(row, rowsTotal - 4)); }

template <bool FULL>
__device__ __forceinline__ void loadPiece(const unsigned short *P, long ld, int row, int rowsTotal, int k0, int K,
                                          u32x2 (&r)[8]) {
    P += row - earlyRows(row, rowsTotal);
#pragma unroll
    for (int i = 0; i < 8; i++) {
        r[i] = *reinterpret_cast<const u32x2Any *>(P + (long) (FULL ? k0 + i : min(k0 + i, K - 1)) * ld);
        if (!FULL && k0 + i >= K) r[i] = u32x2{0, 0};
    }
}

// The octet of row `q` (0 .. 3) of such a piece.
__device__ __forceinline__ u32x4 turned(const u32x2 (&r)[8], int q) {
    u32x4 o;
#pragma unroll
    for (int p = 0; p < 4; p++)
        o[p] = __builtin_amdgcn_perm(r[2 * p + 1][q >> 1], r[2 * p][q >> 1], (q & 1) ? 0x07060302u : 0x05040100u);
    return o;
}

// One thread's part of staging ROWS x BK of an operand: global memory to registers, registers to LDS.
template <bool KC, int ROWS, int BK>
struct Stage {
    static constexpr int OR = BK / 8;                // octets of a row
    static constexpr int N = ROWS * OR / 256;        // octets of a thread
    static constexpr int RQ = ROWS / 4;              // pieces across the rows
    static_assert(KC ? N >= 1 : N % 4 == 0);
    u32x4 oct[KC ? N : 1];
    u32x2 piece[KC ? 1 : N / 4][8];
    int shift = 0;
    template <bool FULL>
    __device__ __forceinline__ void load(const unsigned short *P, long ld, int row0, int rowsTotal, int k0, int K) {
        const int tid = threadIdx.x;
        if constexpr (KC) {
#pragma unroll
            for (int v = 0; v < N; v++)
                oct[v] = loadOctet<FULL>(P, ld, row0 + tid / OR + 256 / OR * v, rowsTotal, k0 + 8 * (tid % OR), K);
        } else {
            shift = 16 * min(earlyRows(row0 + 4 * (tid % RQ), rowsTotal), 3);
#pragma unroll
            for (int v = 0; v < N / 4; v++)
                loadPiece<FULL>(P, ld, row0 + 4 * (tid % RQ), rowsTotal, k0 + 8 * (tid / RQ + 256 / RQ * v), K, piece[v]);
        }
    }
    __device__ __forceinline__ void store(unsigned short *S) const {
        const int tid = threadIdx.x;
        if constexpr (KC) {
#pragma unroll
            for (int v = 0; v < N; v++) {
                const int r = tid / OR + 256 / OR * v;
                *reinterpret_cast<u32x4 *>(S + r * BK + 8 * octetOf(r, tid % OR)) = oct[v];
            }
        } else {
#pragma unroll
            for (int v = 0; v < N / 4; v++) {
                u32x2 w[8];
#pragma unroll
                for (int i = 0; i < 8; i++) {
                    const unsigned long long two = (piece[v][i][0] | ((unsigned long long) piece[v][i][1] << 32)) >> shift;
                    w[i] = u32x2{(unsigned) two, (unsigned) (two >> 32)};
                }
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const int r = 4 * (tid % RQ) + q;
                    *reinterpret_cast<u32x4 *>(S + r * BK + 8 * octetOf(r, tid / RQ + 256 / RQ * v)) = turned(w, q);
                }
            }
        }
    }
};

template <int BK>
__device__ __forceinline__ bf16x8 fragment(const unsigned short *S, int row, int octet) {
    return *reinterpret_cast<const bf16x8 *>(S + row * BK + 8 * octetOf(row, octet));
}

__device__ __forceinline__ f32x4 load4(const float *p, int n) {
    if (n >= 4) return *reinterpret_cast<const f32x4Any *>(p);
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
    for (int t = 0; t < 3; t++)
        if (t < n) v[t] = p[t];
    return v;
}
__device__ __forceinline__ void store4(float *p, f32x4 v, int n) {
    if (n >= 4) {
        *reinterpret_cast<f32x4Any *>(p) = v;
        return;
    }
    for (int t = 0; t < 3; t++)
        if (t < n) p[t] = v[t];
}
__device__ __forceinline__ void store4b(unsigned short *p, f32x4 v, int n) {
    if (n >= 4) {
        *reinterpret_cast<u32x2Any *>(p) =
            u32x2{toBf16(v[0]) | ((unsigned) toBf16(v[1]) << 16), toBf16(v[2]) | ((unsigned) toBf16(v[3]) << 16)};
        return;
    }
    for (int t = 0; t < 3; t++)
        if (t < n) p[t] = toBf16(v[t]);
}

// A lane's four results of a tile at (row, col): columns col .. col + 3, or rows row .. row + 3 (FWD_LANES).
// What the epilogue reads is requested for several tiles ahead of their writes: a read behind a write waits
// for it as well.
struct Operands {
    f32x4 a, b, c;
};

template <int EPI>
__device__ __forceinline__ Operands fetch(const GemmArgs &g, int row, int col) {
    Operands x{};
    if (row >= g.M || col >= g.N) return x;
    const long o = (long) row * g.ldc + col;
    const int n = g.N - col;
    if constexpr (EPI == FWD_LANES) {
        x.a[0] = g.bias[col];
        x.b[0] = g.scale[col];
        x.c[0] = g.shift[col];
    } else if constexpr (EPI < DW_STORE) {
        x.a = load4(g.bias + col, n);
    }
    if constexpr (EPI == FWD_AFFINE) {
        x.b = load4(g.scale + col, n);
        x.c = load4(g.shift + col, n);
    } else if constexpr (EPI == FWD_MSE) {
        x.b = load4(g.target + (long) g.rows[row] * g.ldc + col, n);
    } else if constexpr (EPI == DW_ADAM) {
        x.a = load4(g.adam.w + o, n);
        x.b = load4(g.adam.m + o, n);
        x.c = load4(g.adam.v + o, n);
    } else if constexpr (EPI == DA_GELU) {
        x.a = load4(g.Z + o, n);
    }
    return x;
}

template <int EPI>
__device__ __forceinline__ void finish(const GemmArgs &g, int row, int col, f32x4 v, Operands x, double &loss) {
    if (row >= g.M || col >= g.N) return;
    if constexpr (EPI == FWD_LANES) {
        store4(g.C + ((long) (row >> 4) * g.N + col) * 16 + (row & 15), (v + x.a[0]) * x.b[0] + x.c[0], g.M - row);
        return;
    }
    const long o = (long) row * g.ldc + col;
    const int n = g.N - col;
    if constexpr (EPI == FWD_BIAS) {
        store4(g.C + o, v + x.a, n);
    } else if constexpr (EPI == DW_STORE) {
        store4(g.C + o, v, n);
    } else if constexpr (EPI == FWD_GELU) {
        v += x.a;
        store4(g.C + o, v, n);
#pragma unroll
        for (int t = 0; t < 4; t++) v[t] = gelu(v[t]);
        store4b(g.Cb + o, v, n);
    } else if constexpr (EPI == FWD_AFFINE) {
        store4(g.C + o, (v + x.a) * x.b + x.c, n);
    } else if constexpr (EPI == FWD_MSE) {
        const f32x4 d = v + x.a - x.b;
#pragma unroll
        for (int t = 0; t < 4; t++) {
            if (t < n) loss += (double) d[t] * d[t];
            v[t] = 2.f * d[t] * g.inv;
        }
        store4(g.C + o, v, n);
        store4b(g.Cb + o, v, n);
    } else if constexpr (EPI == DW_ADAM) {
        if (g.C) store4(g.C + o, v, n);
        f32x4 w;
#pragma unroll
        for (int t = 0; t < 4; t++) {
            float mt = x.b[t], st = x.c[t];
            w[t] = adamStep(g.adam, v[t], x.a[t], mt, st);
            x.b[t] = mt;
            x.c[t] = st;
        }
        store4(g.adam.m + o, x.b, n);
        store4(g.adam.v + o, x.c, n);
        store4(g.adam.w + o, w, n);
        store4b(g.adam.wb + o, w, n);
    } else if constexpr (EPI == DA_GELU) {
#pragma unroll
        for (int t = 0; t < 4; t++) v[t] *= geluGrad(x.a[t]);
        store4(g.C + o, v, n);
        store4b(g.Cb + o, v, n);
    }
}

// The workgroup's part of the loss, threads in a fixed tree.
template <int EPI>
__device__ __forceinline__ void lossOut(const GemmArgs &g, double loss, double *red) {
    if constexpr (EPI == FWD_MSE) {
        __syncthreads();
        red[threadIdx.x] = loss;
        __syncthreads();
        for (int s = 128; s > 0; s >>= 1) {
            if (threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
            __syncthreads();
        }
        if (threadIdx.x == 0) g.loss[blockIdx.x] = red[0];
    }
}

// Workgroup -> tile of a tm x tn grid: workgroups are dealt round to the 8 XCDs, and each XCD takes a run
// of tiles, 8 tiles of rows fastest, then the columns: its L2 keeps the rows of A for all the run and a tile
// of B for 8 workgroups (with all 32 row tiles of the 4,096-row output layer first 0.57 instead of 0.55 ms).  False: no tile.
__device__ __forceinline__ bool tileOf(int tm, int tn, int &ti, int &tj) {
    const int run = gridDim.x / 8, t = (blockIdx.x % 8) * run + blockIdx.x / 8;
    const int group = t / (8 * tn), r = t - group * 8 * tn, rows = min(8, tm - 8 * group);
    if (t >= tm * tn) return false;
    ti = 8 * group + r % rows;
    tj = r / rows;
    return true;
}

// Large products: 256 threads, a 128 x 128 tile per workgroup in k-steps of 64, each wave a 64 x 64
// block of 4 x 4 MFMA tiles (64 accumulator registers).  LDS is double buffered, and two more k-steps are on
// their way in registers: a k-step is shorter than a trip to memory.  With split-K (gridDim.z > 1)
// each z-slice writes its partial product to a workspace, summed by k_splitk_reduce.
constexpr int G2_BM = 128, G2_BN = 128, G2_BK = 64;

template <int EPI>
__global__ void __launch_bounds__(256, 2) k_gemm2(GemmArgs g, float *partial) {
    __shared__ __attribute__((aligned(16))) unsigned short lds[4 * G2_BM * G2_BK];
    static_assert(G2_BM == 128 && G2_BN == 128 && sizeof(lds) == G2_BM * G2_BN * sizeof(float));
    unsigned short *As[2] = {lds, lds + G2_BM * G2_BK}, *Bs[2] = {lds + 2 * G2_BM * G2_BK, lds + 3 * G2_BM * G2_BK};
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int ti, tj;
    double loss = 0.;
    if (tileOf((g.M + G2_BM - 1) / G2_BM, (g.N + G2_BN - 1) / G2_BN, ti, tj)) {
        const int i0 = ti * G2_BM, j0 = tj * G2_BN, wi = (wave >> 1) * 64, wj = (wave & 1) * 64;
        // this z-slice's k range, a multiple of the k-step
        const int kPer = ((g.K + gridDim.z - 1) / gridDim.z + G2_BK - 1) / G2_BK * G2_BK;
        const int kBeg = blockIdx.z * kPer, kEnd = min(g.K, kBeg + kPer);
        Operands cols[4] = {};
        if constexpr (EPI == FWD_LANES) {
#pragma unroll
            for (int b = 0; b < 4; b++) cols[b] = fetch<EPI>(g, i0, j0 + wj + 16 * b + (lane & 15));
        }
        f32x4 acc[4][4];
#pragma unroll
        for (int a = 0; a < 4; a++)
#pragma unroll
            for (int b = 0; b < 4; b++) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
        Stage<kRows(EPI), G2_BM, G2_BK> sa[2];
        Stage<kCols(EPI), G2_BN, G2_BK> sb[2];
        const int nk = max(0, kEnd - kBeg) / G2_BK, kTail = kBeg + nk * G2_BK;  // whole k-steps, and the rest
        auto load = [&](int kt, int s) {  // past the end the last one again: a condition would drain what is in flight
            const int k0 = kBeg + min(kt, nk - 1) * G2_BK;
            sa[s].template load<true>(g.A, g.lda, i0, g.M, k0, kEnd);
            sb[s].template load<true>(g.B, g.ldb, j0, g.N, k0, kEnd);
        };
        auto store = [&](int s) {
            sa[s].store(As[s]);
            sb[s].store(Bs[s]);
        };
        auto multiply = [&](int s) {
#pragma unroll
            for (int ks = 0; ks < G2_BK / 8; ks += 4) {
                bf16x8 af[4], bfr[4];
#pragma unroll
                for (int a = 0; a < 4; a++) af[a] = fragment<G2_BK>(As[s], wi + 16 * a + (lane & 15), ks + (lane >> 4));
#pragma unroll
                for (int b = 0; b < 4; b++) bfr[b] = fragment<G2_BK>(Bs[s], wj + 16 * b + (lane & 15), ks + (lane >> 4));
#pragma unroll
                for (int a = 0; a < 4; a++)
#pragma unroll
                    for (int b = 0; b < 4; b++)
                        acc[a][b] = EPI == FWD_LANES
                                        ? __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[a], bfr[b], acc[a][b], 0, 0, 0)
                                        : __builtin_amdgcn_mfma_f32_16x16x32_bf16(bfr[b], af[a], acc[a][b], 0, 0, 0);
            }
        };
        // k-step kt from LDS buffer s, kt + 1 from registers to the other, kt + 3 requested
        auto step = [&](int kt, int s) {
            multiply(s);
            store(s ^ 1);
            load(kt + 3, s ^ 1);
            __syncthreads();
        };
        if (nk > 0) {
            load(0, 0);
            load(1, 1);
            store(0);
            load(2, 0);
            __syncthreads();
            for (int kt = 0;; kt += 2) {
                step(kt, 0);
                if (kt + 1 >= nk) break;
                step(kt + 1, 1);
                if (kt + 2 >= nk) break;
            }
        }
        if (kTail < kEnd) {
            sa[0].template load<false>(g.A, g.lda, i0, g.M, kTail, kEnd);
            sb[0].template load<false>(g.B, g.ldb, j0, g.N, kTail, kEnd);
            store(0);
            __syncthreads();
            multiply(0);
            __syncthreads();
        }
        if constexpr (EPI == FWD_LANES) {
#pragma unroll
            for (int b = 0; b < 4; b++)
#pragma unroll
                for (int a = 0; a < 4; a++)
                    finish<EPI>(g, i0 + wi + 16 * a + 4 * (lane >> 4), j0 + wj + 16 * b + (lane & 15), acc[a][b], cols[b], loss);
        } else {
            // Rows by way of LDS, so that a wave moves 512-byte pieces of two rows: straight from the accumulators
            // it moves 64-byte pieces of 16 rows, each in another page
            // (weight gradient with Adam, 512 x 52,360 x 256: 268 us, now 184: 3.9 of the 4.6 TB/s of a copy)
            f32x4 *S = reinterpret_cast<f32x4 *>(lds);
#pragma unroll
            for (int a = 0; a < 4; a++)
#pragma unroll
                for (int b = 0; b < 4; b++) {
                    const int row = wi + 16 * a + (lane & 15), unit = wj / 4 + 4 * b + (lane >> 4);
                    S[row * 32 + (unit ^ (row & 7))] = acc[a][b];
                }
            __syncthreads();
            const int row = threadIdx.x >> 5, unit = threadIdx.x & 31, col = j0 + 4 * unit;
            auto tile = [&](int it) { return S[(8 * it + row) * 32 + (unit ^ row)]; };
            float *part = EPI >= DW_STORE && gridDim.z > 1 ? partial + (long) blockIdx.z * g.M * g.N : nullptr;
            if (part) {
#pragma unroll
                for (int it = 0; it < 16; it++) {
                    const int r = i0 + 8 * it + row;
                    if (r < g.M && col < g.N) store4(part + (long) r * g.N + col, tile(it), g.N - col);
                }
            } else {
                Operands x[2][4];
#pragma unroll
                for (int q = 0; q < 4; q++) x[0][q] = fetch<EPI>(g, i0 + 8 * q + row, col);
#pragma unroll
                for (int p = 0; p < 4; p++) {
                    if (p < 3) {
#pragma unroll
                        for (int q = 0; q < 4; q++) x[(p + 1) & 1][q] = fetch<EPI>(g, i0 + 8 * (4 * p + 4 + q) + row, col);
                    }
#pragma unroll
                    for (int q = 0; q < 4; q++)
                        finish<EPI>(g, i0 + 8 * (4 * p + q) + row, col, tile(4 * p + q), x[p & 1][q], loss);
                }
            }
        }
    }
    lossOut<EPI>(g, loss, reinterpret_cast<double *>(lds));
}

// Small products (fewer 128 x 128 tiles than CUs, e.g. the 256 x 512 x 512 hidden layers: 8 tiles, 33 us,
// now 7): 32 x 64 tiles, and 256 k at a time in LDS, so that a product waits for memory once per 256 k
// instead of once per 64.  256 threads, each wave 16 x 32.
constexpr int G3_BM = 32, G3_BN = 64, G3_BK = 256;

template <int EPI>
__global__ void __launch_bounds__(256) k_gemm3(GemmArgs g) {
    __shared__ __attribute__((aligned(16))) unsigned short As[G3_BM * G3_BK];
    __shared__ __attribute__((aligned(16))) unsigned short Bs[G3_BN * G3_BK];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int ti, tj;
    double loss = 0.;
    if (tileOf((g.M + G3_BM - 1) / G3_BM, (g.N + G3_BN - 1) / G3_BN, ti, tj)) {
        const int i0 = ti * G3_BM, j0 = tj * G3_BN, wi = (wave >> 1) * 16, wj = (wave & 1) * 32;
        f32x4 acc[2];
        acc[0] = acc[1] = f32x4{0.f, 0.f, 0.f, 0.f};
        Stage<kRows(EPI), G3_BM, G3_BK> sa;
        Stage<kCols(EPI), G3_BN, G3_BK> sb;
        const int nk = g.K / G3_BK, kTail = nk * G3_BK;  // whole k-steps, and the rest
        auto multiply = [&](int octets) {
#pragma unroll 4
            for (int ks = 0; ks < octets; ks += 4) {
                const bf16x8 af = fragment<G3_BK>(As, wi + (lane & 15), ks + (lane >> 4));
#pragma unroll
                for (int b = 0; b < 2; b++) {
                    const bf16x8 bfr = fragment<G3_BK>(Bs, wj + 16 * b + (lane & 15), ks + (lane >> 4));
                    acc[b] = EPI == FWD_LANES ? __builtin_amdgcn_mfma_f32_16x16x32_bf16(af, bfr, acc[b], 0, 0, 0)
                                              : __builtin_amdgcn_mfma_f32_16x16x32_bf16(bfr, af, acc[b], 0, 0, 0);
                }
            }
        };
        if (nk > 0) {
            sa.template load<true>(g.A, g.lda, i0, g.M, 0, g.K);
            sb.template load<true>(g.B, g.ldb, j0, g.N, 0, g.K);
        }
        for (int kt = 0; kt < nk; kt++) {
            if (kt) __syncthreads();
            sa.store(As);
            sb.store(Bs);
            __syncthreads();
            if (kt + 1 < nk) {
                sa.template load<true>(g.A, g.lda, i0, g.M, (kt + 1) * G3_BK, g.K);
                sb.template load<true>(g.B, g.ldb, j0, g.N, (kt + 1) * G3_BK, g.K);
            }
            multiply(G3_BK / 8);
        }
        if (kTail < g.K) {
            sa.template load<false>(g.A, g.lda, i0, g.M, kTail, g.K);
            sb.template load<false>(g.B, g.ldb, j0, g.N, kTail, g.K);
            __syncthreads();
            sa.store(As);
            sb.store(Bs);
            __syncthreads();
            multiply((g.K - kTail + 7) / 8);
        }
        const int row = i0 + wi + (EPI == FWD_LANES ? 4 * (lane >> 4) : lane & 15);
        const int col = j0 + wj + (EPI == FWD_LANES ? lane & 15 : 4 * (lane >> 4));
        Operands x[2];
#pragma unroll
        for (int b = 0; b < 2; b++) x[b] = fetch<EPI>(g, row, col + 16 * b);
#pragma unroll
        for (int b = 0; b < 2; b++) finish<EPI>(g, row, col + 16 * b, acc[b], x[b], loss);
    }
    lossOut<EPI>(g, loss, reinterpret_cast<double *>(As));
}

// The sum of the split-K slices of a product, in slice order, through its epilogue.
template <int EPI>
__global__ void k_splitk_reduce(const float *partial, int slices, GemmArgs g) {
    const long n = (long) g.M * g.N;
    for (long e = blockIdx.x * (long) blockDim.x + threadIdx.x; e < n; e += (long) gridDim.x * blockDim.x) {
        float s = 0.f;
        for (int z = 0; z < slices; z += 8) {
            float v[8];
#pragma unroll
            for (int q = 0; q < 8; q++) v[q] = partial[(long) min(z + q, slices - 1) * n + e];
#pragma unroll
            for (int q = 0; q < 8; q++)
                if (z + q < slices) s += v[q];
        }
        const long o = e / g.N * g.ldc + e % g.N;
        if (EPI == DA_GELU) {
            s *= geluGrad(g.Z[o]);
            g.Cb[o] = toBf16(s);
        }
        g.C[o] = s;
    }
}

// db[j] = sum_i dZ[i][j], and with a.w Adam on these biases.
// 256 threads per 64 columns: thread (c, q) sums rows q, q + 4, ... of column c, then the four
// partials of a column are added in q order (the same order on every run).  16 rows are requested at a
// time: one after the other, 64 rows of 512 columns took 21 us, now 4.
__global__ void __launch_bounds__(256) k_colsum(const float *dZ, int rows, int cols, float *db, AdamArgs a) {
    __shared__ float part[4][64];
    const int c = threadIdx.x & 63, q = threadIdx.x >> 6;
    const int j = blockIdx.x * 64 + c, jc = min(j, cols - 1);
    float s = 0.f;
    for (int i = q; i < rows; i += 64) {
        float v[16];
#pragma unroll
        for (int t = 0; t < 16; t++) v[t] = dZ[(long) min(i + 4 * t, rows - 1) * cols + jc];
#pragma unroll
        for (int t = 0; t < 16; t++)
            if (i + 4 * t < rows) s += v[t];
    }
    part[q][c] = s;
    __syncthreads();
    if (q != 0 || j >= cols) return;
    const float gt = ((part[0][c] + part[1][c]) + part[2][c]) + part[3][c];
    if (db) db[j] = gt;
    if (a.w) {
        a.w[j] = adamStep(a, gt, a.w[j], a.m[j], a.v[j]);
        a.wb[j] = toBf16(a.w[j]);
    }
}

// MSE on standardized outputs: dY = 2 (y - t) / count and per-block partial sums of (y - t)^2.
__global__ void k_mse(const float *Y, const float *Tg, float *dY, unsigned short *dYb, long n, float inv,
                      double *partial) {
    __shared__ double red[256];
    double acc = 0.;
    for (long t = blockIdx.x * (long) blockDim.x + threadIdx.x; t < n; t += (long) gridDim.x * blockDim.x) {
        const float d = Y[t] - Tg[t];
        acc += (double) d * d;
        const float g = 2.f * d * inv;
        dY[t] = g;
        dYb[t] = toBf16(g);
    }
    red[threadIdx.x] = acc;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if (threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) partial[blockIdx.x] = red[0];
}

__global__ void k_adam(AdamArgs a, const float *g, long n) {
    for (long t = blockIdx.x * (long) blockDim.x + threadIdx.x; t < n; t += (long) gridDim.x * blockDim.x) {
        const float wn = adamStep(a, g[t], a.w[t], a.m[t], a.v[t]);
        a.w[t] = wn;
        a.wb[t] = toBf16(wn);
    }
}

__global__ void k_to_bf16(const float *in, unsigned short *out, long n) {
    for (long t = blockIdx.x * (long) blockDim.x + threadIdx.x; t < n; t += (long) gridDim.x * blockDim.x)
        out[t] = toBf16(in[t]);
}

// Minibatch inputs: rows idx[r] of X, FP32 -> bf16.
__global__ void k_gather(const float *X, int in, const int *idx, int rows, unsigned short *Xb) {
    const long total = (long) rows * in;
    for (long t = blockIdx.x * (long) blockDim.x + threadIdx.x; t < total; t += (long) gridDim.x * blockDim.x)
        Xb[t] = toBf16(X[(long) idx[t / in] * in + t % in]);
}

// Per-column mean and standard deviation of an N x cols matrix (two passes, rows in order).
__global__ void k_col_stats(const float *Tg, long rows, long cols, float *mean, float *stdv) {
    const long j = blockIdx.x * (long) blockDim.x + threadIdx.x;
    if (j >= cols) return;
    double s = 0.;
    for (long i = 0; i < rows; i++) s += Tg[i * cols + j];
    const double mu = s / (double) rows;
    double q = 0.;
    for (long i = 0; i < rows; i++) {
        const double d = Tg[i * cols + j] - mu;
        q += d * d;
    }
    const double sd = sqrt(q / (double) rows);
    mean[j] = (float) mu;
    stdv[j] = (float) (sd > 1e-6 * (fabs(mu) + 1e-12) && sd > 1e-12 ? sd : 1.0);
}

__global__ void k_standardize(float *Tg, long rows, long cols, const float *mean, const float *stdv) {
    const long total = rows * cols;
    for (long t = blockIdx.x * (long) blockDim.x + threadIdx.x; t < total; t += (long) gridDim.x * blockDim.x) {
        const long j = t % cols;
        Tg[t] = (Tg[t] - mean[j]) / stdv[j];
    }
}

}  // namespace mlp
}  // namespace spk

// ====================================================================== host side (C ABI)
#include <algorithm>
#include <cstring>
#include <memory>
#include <numeric>
#include <random>
#include <string>
#include <vector>

#include "../../include/spock_amd.h"
#include "common.hpp"

using spk::check;
using spk::DevBuf;
using spk::fail;
namespace M = spk::mlp;

struct spk_mlp {
    spk_ctx *ctx = nullptr;  // holds a reference
    explicit spk_mlp(spk_ctx *c) : ctx(spk::retain(c)) {}
    ~spk_mlp() {
        if (ctx && ctx->stream) (void) hipStreamSynchronize(ctx->stream);
        spk::releaseCtx(ctx);
    }
    spk_mlp(const spk_mlp &) = delete;
    spk_mlp &operator=(const spk_mlp &) = delete;
    std::vector<int> dims;          // in, hidden..., out
    std::vector<long> wOff, bOff;   // parameter offsets (weights [d_l][d_l+1] row-major, then bias)
    long nParams = 0;
    DevBuf w, wb, g, m, v;          // FP32 masters, bf16 copies, gradients, Adam moments
    long step = 0;
    DevBuf inMean, inStd, outMean, outStd;
    std::vector<float> hInMean, hInStd;
    int cap = 0;                    // rows the workspace holds
    DevBuf X, Y, dY, dYb, dZ[2], dZb[2], Tb, idx, partial, Xf;
    int lanesRows = 0;              // rows whose outputs went to a batch instead of Y
    DevBuf splitWs;                 // split-K partial products of the GEMM
    std::vector<std::unique_ptr<DevBuf>> Z, A;
    long nTrain = 0;
    DevBuf trX, trT;
    int layers() const { return (int) dims.size() - 1; }
    int in() const { return dims.front(); }
    int out() const { return dims.back(); }
};

namespace {

dim3 grid1(long n) { return dim3((unsigned) std::min<long>(4096, (n + 255) / 256)); }

constexpr int LOSS_BLOCKS = 1024;  // of k_mse

int tiles(const M::GemmArgs &a, int bm, int bn) { return ((a.M + bm - 1) / bm) * ((a.N + bn - 1) / bn); }

// Split K when the output has too few tiles to fill the device and K is long (the output layer's
// dA = dY W': 8 tiles, K = 52,360): up to 256 workgroups, 16 k-steps each at least.  Operands whose rows
// start off 16-byte boundaries keep one sum per element.
int splitOf(const M::GemmArgs &a, int epi) {
    const int t = tiles(a, M::G2_BM, M::G2_BN);
    if (epi < M::DW_STORE || t >= 128 || a.lda % 8 || a.ldb % 8 || (uintptr_t) a.A % 16 || (uintptr_t) a.B % 16) return 1;
    return std::max(1, std::min(256 / t, a.K / (16 * M::G2_BK)));
}

// Products with fewer 128 x 128 tiles than this go to the 32 x 64 kernel: 8 to 128
// tiles (hidden layers of 256 and 4,096 rows) take 7 us in it and 23 to 32 in the other; 820 tiles (256 x 512 x
// 52,360) 102 and 88 us, 13,120 tiles 1.08 and 0.53 ms.
constexpr int SMALL_TILES = 256;

// Workgroups of an unsplit product (and partial sums of its loss).
int gemmBlocks(const M::GemmArgs &a) {
    const int t = tiles(a, M::G2_BM, M::G2_BN);
    return ((t < SMALL_TILES ? tiles(a, M::G3_BM, M::G3_BN) : t) + 7) / 8 * 8;
}

template <int EPI>
void gemm(spk_mlp *m, const M::GemmArgs &a) {
    hipStream_t st = m->ctx->stream;
    const int split = splitOf(a, EPI);
    if (split > 1) {
        const size_t need = (size_t) split * a.M * a.N * sizeof(float);
        if (m->splitWs.bytes < need) m->splitWs.alloc(need);
        const int t = (tiles(a, M::G2_BM, M::G2_BN) + 7) / 8 * 8;
        hipLaunchKernelGGL(M::k_gemm2<EPI>, dim3(t, 1, split), dim3(256), 0, st, a, m->splitWs.as<float>());
        hipLaunchKernelGGL(M::k_splitk_reduce<EPI>, grid1((long) a.M * a.N), dim3(256), 0, st, m->splitWs.as<float>(), split, a);
    } else if (tiles(a, M::G2_BM, M::G2_BN) < SMALL_TILES) {
        hipLaunchKernelGGL(M::k_gemm3<EPI>, dim3(gemmBlocks(a)), dim3(256), 0, st, a);
    } else {
        hipLaunchKernelGGL(M::k_gemm2<EPI>, dim3(gemmBlocks(a)), dim3(256), 0, st, a, (float *) nullptr);
    }
}

void ensureCap(spk_mlp *m, int rows) {
    if (rows <= m->cap) return;
    const int h = *std::max_element(m->dims.begin() + 1, m->dims.end() - 1);
    const long out = m->out(), in = m->in();
    m->X.alloc(((size_t) rows * in + M::ROW_PAD) * 2);
    m->Xf.alloc((size_t) rows * in * 4);
    m->Y.alloc((size_t) rows * out * 4);
    m->dY.alloc((size_t) rows * out * 4);
    m->dYb.alloc(((size_t) rows * out + M::ROW_PAD) * 2);
    m->Tb.alloc((size_t) rows * out * 4);
    for (int q = 0; q < 2; q++) {
        m->dZ[q].alloc((size_t) rows * h * 4);
        m->dZb[q].alloc(((size_t) rows * h + M::ROW_PAD) * 2);
    }
    m->Z.clear();
    m->A.clear();
    for (int l = 0; l + 1 < m->layers(); l++) {
        m->Z.push_back(std::make_unique<DevBuf>());
        m->A.push_back(std::make_unique<DevBuf>());
        m->Z.back()->alloc((size_t) rows * m->dims[l + 1] * 4);
        m->A.back()->alloc(((size_t) rows * m->dims[l + 1] + M::ROW_PAD) * 2);
    }
    m->cap = rows;
}

const unsigned short *wbf(spk_mlp *m, int l) { return m->wb.as<unsigned short>() + m->wOff[l]; }
const float *bias(spk_mlp *m, int l) { return m->w.as<float>() + m->bOff[l]; }

// Layer l of the forward pass: A = the previous activations, B = W.
M::GemmArgs layer(spk_mlp *m, int l, int rows) {
    M::GemmArgs a{};
    a.A = l == 0 ? m->X.as<unsigned short>() : m->A[l - 1]->as<unsigned short>();
    a.B = wbf(m, l);
    a.M = rows;
    a.K = m->dims[l];
    a.N = m->dims[l + 1];
    a.lda = a.K;
    a.ldb = a.ldc = a.N;
    a.bias = bias(m, l);
    return a;
}

// The hidden layers of `rows` rows whose bf16 inputs are in m->X.
void hiddenLayers(spk_mlp *m, int rows) {
    for (int l = 0; l + 1 < m->layers(); l++) {
        M::GemmArgs a = layer(m, l, rows);
        a.C = m->Z[l]->as<float>();
        a.Cb = m->A[l]->as<unsigned short>();
        gemm<M::FWD_GELU>(m, a);
    }
}

// The output layer: Y gets the standardized outputs, or the denormalized iterate with `denorm`; `lanes`
// gets the denormalized iterate as a shared batch holds it, 16 instances to a block, and then Y does not.
void outputLayer(spk_mlp *m, int rows, bool denorm, float *lanes = nullptr) {
    M::GemmArgs a = layer(m, m->layers() - 1, rows);
    a.C = lanes ? lanes : m->Y.as<float>();
    a.scale = m->outStd.as<float>();
    a.shift = m->outMean.as<float>();
    if (lanes) gemm<M::FWD_LANES>(m, a);
    else if (denorm) gemm<M::FWD_AFFINE>(m, a);
    else gemm<M::FWD_BIAS>(m, a);
    m->lanesRows = lanes ? rows : 0;
    check(hipGetLastError(), "mlp forward");
}

void forward(spk_mlp *m, int rows, bool denorm) {
    hiddenLayers(m, rows);
    outputLayer(m, rows, denorm);
}

// Y of a prediction that went straight to a batch (0.53 ms for 4,096 rows of 52,360, which few callers read), for
// the loss and before the parameters or the normalization it was made with change.
void keepOutputs(spk_mlp *m) {
    if (m->lanesRows) outputLayer(m, m->lanesRows, true);
}

// Adam's arguments for the parameters from offset `off` on.
M::AdamArgs adamAt(const spk_mlp *m, const M::AdamArgs &all, long off) {
    M::AdamArgs a = all;
    a.w += off;
    a.wb += off;
    a.m += off;
    a.v += off;
    return a;
}

// Gradients of the loss whose output gradient is in m->dY / m->dYb (rows of the last forward), kept in
// m->g with `keep`; with `step`, Adam on each layer's parameters as soon as its weights have been used: its
// epilogue has the gradient in registers, where a pass of its own reads it back from memory (output
// layer: product 75 + Adam 145 us, together 184).
void backward(spk_mlp *m, int rows, bool keep, const M::AdamArgs *step) {
    hipStream_t st = m->ctx->stream;
    const unsigned short *dCur = m->dYb.as<unsigned short>();
    const float *dCurF = m->dY.as<float>();
    for (int l = m->layers() - 1; l >= 0; l--) {
        const int Nl = m->dims[l + 1], Kl = m->dims[l], q = l & 1;
        if (l > 0) {  // dZ_{l-1} = (dZ_l W_l') . gelu'(Z_{l-1})  (rows x Kl)
            M::GemmArgs a{};
            a.A = dCur;
            a.B = wbf(m, l);
            a.lda = a.ldb = a.K = Nl;
            a.M = rows;
            a.N = Kl;
            a.ldc = Kl;
            a.C = m->dZ[q].as<float>();
            a.Cb = m->dZb[q].as<unsigned short>();
            a.Z = m->Z[l - 1]->as<float>();
            gemm<M::DA_GELU>(m, a);
        }
        // dW_l = A_{l-1}' dZ_l  (Kl x Nl), db_l = colsum dZ_l
        M::GemmArgs a{};
        a.A = l == 0 ? m->X.as<unsigned short>() : m->A[l - 1]->as<unsigned short>();
        a.B = dCur;
        a.lda = a.M = Kl;
        a.ldb = a.ldc = a.N = Nl;
        a.K = rows;
        float *gw = m->g.as<float>() + m->wOff[l], *gb = m->g.as<float>() + m->bOff[l];
        if (step && splitOf(a, M::DW_ADAM) == 1) {
            a.C = keep ? gw : nullptr;
            a.adam = adamAt(m, *step, m->wOff[l]);
            gemm<M::DW_ADAM>(m, a);
        } else {
            a.C = gw;
            gemm<M::DW_STORE>(m, a);
            const long n = (long) Kl * Nl;
            if (step) hipLaunchKernelGGL(M::k_adam, grid1(n), dim3(256), 0, st, adamAt(m, *step, m->wOff[l]), gw, n);
        }
        hipLaunchKernelGGL(M::k_colsum, dim3((Nl + 63) / 64), dim3(256), 0, st, dCurF, rows, Nl, keep ? gb : nullptr,
                           step ? adamAt(m, *step, m->bOff[l]) : M::AdamArgs{});
        dCur = m->dZb[q].as<unsigned short>();
        dCurF = m->dZ[q].as<float>();
    }
    check(hipGetLastError(), "mlp backward");
}

double mseLoss(spk_mlp *m, int rows, const float *target) {
    const long n = (long) rows * m->out();
    const int blocks = (int) std::min<long>(LOSS_BLOCKS, (n + 255) / 256);
    if (m->partial.bytes < blocks * sizeof(double)) m->partial.alloc(blocks * sizeof(double));
    hipLaunchKernelGGL(M::k_mse, dim3(blocks), dim3(256), 0, m->ctx->stream, m->Y.as<float>(), target, m->dY.as<float>(),
                       m->dYb.as<unsigned short>(), n, 1.f / (float) n, m->partial.as<double>());
    check(hipGetLastError(), "mlp loss");
    std::vector<double> part(blocks);
    check(hipMemcpyAsync(part.data(), m->partial.p, blocks * sizeof(double), hipMemcpyDeviceToHost, m->ctx->stream),
          "loss");
    check(hipStreamSynchronize(m->ctx->stream), "sync");
    double s = 0.;
    for (double v : part) s += v;
    return s / (double) n;
}

M::AdamArgs adamStep(spk_mlp *m, float lr, float b1, float b2, float eps) {
    m->step++;
    return {m->w.as<float>(), m->wb.as<unsigned short>(), m->m.as<float>(), m->v.as<float>(), lr, b1, b2, eps,
            1.f - std::pow(b1, (float) m->step), 1.f - std::pow(b2, (float) m->step)};
}

// Host rows -> normalized FP32 -> bf16 workspace inputs.
template <typename S>
void uploadInputs(spk_mlp *m, const S *x, int rows) {
    ensureCap(m, rows);
    const int in = m->in();
    std::vector<float> xs((size_t) rows * in);
    for (int r = 0; r < rows; r++)
        for (int c = 0; c < in; c++)
            xs[(size_t) r * in + c] = (float) ((x[(size_t) r * in + c] - m->hInMean[c]) / m->hInStd[c]);
    check(hipMemcpyAsync(m->Xf.p, xs.data(), xs.size() * 4, hipMemcpyHostToDevice, m->ctx->stream), "inputs");
    hipLaunchKernelGGL(M::k_to_bf16, grid1((long) xs.size()), dim3(256), 0, m->ctx->stream, m->Xf.as<float>(),
                       m->X.as<unsigned short>(), (long) xs.size());
    check(hipStreamSynchronize(m->ctx->stream), "sync");
}

void refreshBf16(spk_mlp *m) {
    hipLaunchKernelGGL(M::k_to_bf16, grid1(m->nParams), dim3(256), 0, m->ctx->stream, m->w.as<float>(),
                       m->wb.as<unsigned short>(), m->nParams);
    check(hipGetLastError(), "bf16 copy");
}

}  // namespace

extern "C" {

int spk_mlp_create(spk_ctx *ctx, int in, int hidden, int layers, int out, unsigned long long seed, spk_mlp **res) {
    try {
        if (in <= 0 || hidden <= 0 || layers < 0 || out <= 0) throw std::runtime_error("bad MLP dimensions");
        if (!ctx) throw std::runtime_error("null context");
        auto m = std::make_unique<spk_mlp>(ctx);
        check(hipSetDevice(ctx->device), "hipSetDevice");
        m->dims.push_back(in);
        for (int l = 0; l < layers; l++) m->dims.push_back(hidden);
        m->dims.push_back(out);
        long off = 0;
        for (int l = 0; l < m->layers(); l++) {
            m->wOff.push_back(off);
            off += (long) m->dims[l] * m->dims[l + 1];
            m->bOff.push_back(off);
            off += m->dims[l + 1];
        }
        m->nParams = off;
        // He-uniform initialisation from a seeded generator; zero biases
        std::vector<float> p(off, 0.f);
        std::mt19937_64 gen(seed);
        for (int l = 0; l < m->layers(); l++) {
            const float a = std::sqrt(6.f / (float) m->dims[l]) * (l + 1 == m->layers() ? 0.5f : 1.f);
            std::uniform_real_distribution<float> U(-a, a);
            for (long k = 0; k < (long) m->dims[l] * m->dims[l + 1]; k++) p[m->wOff[l] + k] = U(gen);
        }
        m->w.alloc(off * 4);
        m->wb.alloc((off + M::ROW_PAD) * 2);
        m->g.alloc(off * 4);
        m->m.alloc(off * 4);
        m->v.alloc(off * 4);
        check(hipMemcpy(m->w.p, p.data(), off * 4, hipMemcpyHostToDevice), "params");
        check(hipMemsetAsync(m->g.p, 0, off * 4, ctx->stream), "zero");
        check(hipMemsetAsync(m->m.p, 0, off * 4, ctx->stream), "zero");
        check(hipMemsetAsync(m->v.p, 0, off * 4, ctx->stream), "zero");
        refreshBf16(m.get());
        m->hInMean.assign(in, 0.f);
        m->hInStd.assign(in, 1.f);
        std::vector<float> zo(out, 0.f), on(out, 1.f);
        m->inMean.alloc(in * 4);
        m->inStd.alloc(in * 4);
        m->outMean.alloc(out * 4);
        m->outStd.alloc(out * 4);
        check(hipMemcpy(m->inMean.p, m->hInMean.data(), in * 4, hipMemcpyHostToDevice), "norm");
        check(hipMemcpy(m->inStd.p, m->hInStd.data(), in * 4, hipMemcpyHostToDevice), "norm");
        check(hipMemcpy(m->outMean.p, zo.data(), out * 4, hipMemcpyHostToDevice), "norm");
        check(hipMemcpy(m->outStd.p, on.data(), out * 4, hipMemcpyHostToDevice), "norm");
        check(hipStreamSynchronize(ctx->stream), "sync");
        *res = m.release();
        return 0;
    } catch (const std::exception &e) {
        return fail(ctx, e);
    }
}

int spk_mlp_destroy(spk_mlp *m) {
    delete m;
    return 0;
}

long spk_mlp_num_params(const spk_mlp *m) { return m ? m->nParams : -1; }

int spk_mlp_get_params(spk_mlp *m, float *p) {
    try {
        check(hipStreamSynchronize(m->ctx->stream), "sync");
        spk::readBack(m->ctx, p, m->w.as<float>(), m->nParams);
        return 0;
    } catch (const std::exception &e) {
        return fail(m->ctx, e);
    }
}

int spk_mlp_set_params(spk_mlp *m, const float *p) {
    try {
        keepOutputs(m);
        check(hipStreamSynchronize(m->ctx->stream), "sync");
        check(hipMemcpy(m->w.p, p, m->nParams * 4, hipMemcpyHostToDevice), "params");
        refreshBf16(m);
        check(hipStreamSynchronize(m->ctx->stream), "sync");
        return 0;
    } catch (const std::exception &e) {
        return fail(m->ctx, e);
    }
}

int spk_mlp_get_grads(spk_mlp *m, float *p) {
    try {
        check(hipStreamSynchronize(m->ctx->stream), "sync");
        spk::readBack(m->ctx, p, m->g.as<float>(), m->nParams);
        return 0;
    } catch (const std::exception &e) {
        return fail(m->ctx, e);
    }
}

int spk_mlp_get_normalization(spk_mlp *m, float *inMean, float *inStd, float *outMean, float *outStd) {
    try {
        check(hipStreamSynchronize(m->ctx->stream), "sync");
        std::copy(m->hInMean.begin(), m->hInMean.end(), inMean);
        std::copy(m->hInStd.begin(), m->hInStd.end(), inStd);
        check(hipMemcpy(outMean, m->outMean.p, m->out() * 4, hipMemcpyDeviceToHost), "norm");
        check(hipMemcpy(outStd, m->outStd.p, m->out() * 4, hipMemcpyDeviceToHost), "norm");
        return 0;
    } catch (const std::exception &e) {
        return fail(m->ctx, e);
    }
}

int spk_mlp_set_normalization(spk_mlp *m, const float *inMean, const float *inStd, const float *outMean,
                              const float *outStd) {
    try {
        keepOutputs(m);
        check(hipStreamSynchronize(m->ctx->stream), "sync");
        m->hInMean.assign(inMean, inMean + m->in());
        m->hInStd.assign(inStd, inStd + m->in());
        check(hipMemcpy(m->inMean.p, inMean, m->in() * 4, hipMemcpyHostToDevice), "norm");
        check(hipMemcpy(m->inStd.p, inStd, m->in() * 4, hipMemcpyHostToDevice), "norm");
        check(hipMemcpy(m->outMean.p, outMean, m->out() * 4, hipMemcpyHostToDevice), "norm");
        check(hipMemcpy(m->outStd.p, outStd, m->out() * 4, hipMemcpyHostToDevice), "norm");
        return 0;
    } catch (const std::exception &e) {
        return fail(m->ctx, e);
    }
}

int spk_mlp_forward(spk_mlp *m, const float *x, int rows, float *y) {
    try {
        if (rows <= 0) throw std::runtime_error("rows must be positive");
        uploadInputs(m, x, rows);
        forward(m, rows, false);
        if (y) check(hipMemcpyAsync(y, m->Y.p, (size_t) rows * m->out() * 4, hipMemcpyDeviceToHost, m->ctx->stream),
                     "outputs");
        check(hipStreamSynchronize(m->ctx->stream), "sync");
        return 0;
    } catch (const std::exception &e) {
        return fail(m->ctx, e);
    }
}

int spk_mlp_loss_backward(spk_mlp *m, const float *target, int rows, double *loss) {
    try {
        if (rows <= 0 || rows > m->cap) throw std::runtime_error("rows must match the last forward");
        check(hipMemcpyAsync(m->Tb.p, target, (size_t) rows * m->out() * 4, hipMemcpyHostToDevice, m->ctx->stream),
              "targets");
        keepOutputs(m);
        const double l = mseLoss(m, rows, m->Tb.as<float>());
        backward(m, rows, true, nullptr);
        check(hipStreamSynchronize(m->ctx->stream), "sync");
        if (loss) *loss = l;
        return 0;
    } catch (const std::exception &e) {
        return fail(m->ctx, e);
    }
}

int spk_mlp_adam(spk_mlp *m, float lr, float b1, float b2, float eps) {
    try {
        keepOutputs(m);
        hipLaunchKernelGGL(M::k_adam, grid1(m->nParams), dim3(256), 0, m->ctx->stream, adamStep(m, lr, b1, b2, eps),
                           m->g.as<float>(), m->nParams);
        check(hipGetLastError(), "mlp adam");
        check(hipStreamSynchronize(m->ctx->stream), "sync");
        return 0;
    } catch (const std::exception &e) {
        return fail(m->ctx, e);
    }
}

// The training set: targets already in trT (N rows), inputs x0 (host, N rows).
static void finishDataset(spk_mlp *m, int N, const double *x0);

int spk_mlp_dataset(spk_mlp *m, spk_batch *solved, const double *x0) {
    try {
        const int N = spk_batch_count(solved);
        const long out = m->out();
        m->trT.alloc((size_t) N * out * 4);
        if (spk_batch_get_iterates_device(solved, m->trT.as<float>(), out)) throw std::runtime_error(m->ctx->err);
        finishDataset(m, N, x0);
        return 0;
    } catch (const std::exception &e) {
        return fail(m->ctx, e);
    }
}

int spk_mlp_dataset_lanes(spk_mlp *m, spk_batch *solved, int count, const int *lanes, const double *x0) {
    try {
        if (count < 1) throw std::runtime_error("an empty training set");
        const long out = m->out();
        m->trT.alloc((size_t) count * out * 4);
        if (spk_batch_get_lanes_device(solved, count, lanes, m->trT.as<float>(), out)) throw std::runtime_error(m->ctx->err);
        finishDataset(m, count, x0);
        return 0;
    } catch (const std::exception &e) {
        return fail(m->ctx, e);
    }
}

static void finishDataset(spk_mlp *m, int N, const double *x0) {
    {
        const int in = m->in();
        const long out = m->out();
        m->nTrain = N;
        hipStream_t st = m->ctx->stream;
        keepOutputs(m);
        hipLaunchKernelGGL(M::k_col_stats, dim3((unsigned) ((out + 255) / 256)), dim3(256), 0, st, m->trT.as<float>(),
                           (long) N, out, m->outMean.as<float>(), m->outStd.as<float>());
        hipLaunchKernelGGL(M::k_standardize, grid1((long) N * out), dim3(256), 0, st, m->trT.as<float>(), (long) N,
                           out, m->outMean.as<float>(), m->outStd.as<float>());
        check(hipGetLastError(), "dataset");
        // input normalization from the training inputs
        for (int c = 0; c < in; c++) {
            double s = 0., q = 0.;
            for (int r = 0; r < N; r++) s += x0[(size_t) r * in + c];
            const double mu = s / N;
            for (int r = 0; r < N; r++) q += (x0[(size_t) r * in + c] - mu) * (x0[(size_t) r * in + c] - mu);
            const double sd = std::sqrt(q / N);
            m->hInMean[c] = (float) mu;
            m->hInStd[c] = (float) (sd > 1e-12 ? sd : 1.);
        }
        check(hipMemcpy(m->inMean.p, m->hInMean.data(), in * 4, hipMemcpyHostToDevice), "norm");
        check(hipMemcpy(m->inStd.p, m->hInStd.data(), in * 4, hipMemcpyHostToDevice), "norm");
        std::vector<float> xs((size_t) N * in);
        for (int r = 0; r < N; r++)
            for (int c = 0; c < in; c++)
                xs[(size_t) r * in + c] = (float) ((x0[(size_t) r * in + c] - m->hInMean[c]) / m->hInStd[c]);
        m->trX.alloc(xs.size() * 4);
        check(hipMemcpy(m->trX.p, xs.data(), xs.size() * 4, hipMemcpyHostToDevice), "inputs");
        check(hipStreamSynchronize(st), "sync");
    }
}

int spk_mlp_train(spk_mlp *m, int epochs, int minibatch, float lr, unsigned long long seed, double *epochLoss) {
    try {
        if (m->nTrain <= 0) throw std::runtime_error("no training set (spk_mlp_dataset)");
        if (minibatch <= 0) throw std::runtime_error("minibatch must be positive");
        const int mb = (int) std::min<long>(minibatch, m->nTrain);
        ensureCap(m, mb);
        std::vector<int> perm(m->nTrain);
        std::iota(perm.begin(), perm.end(), 0);
        std::mt19937_64 gen(seed);
        hipStream_t st = m->ctx->stream;
        // An epoch is queued without waiting: its indices go up together, its losses come back together.
        const int nb = (int) (m->nTrain / mb);
        const long n = (long) mb * m->out();
        M::GemmArgs o = layer(m, m->layers() - 1, mb);
        const int blocks = gemmBlocks(o);
        std::vector<double> part((size_t) nb * blocks);
        if (m->partial.bytes < part.size() * sizeof(double)) m->partial.alloc(part.size() * sizeof(double));
        if (m->idx.bytes < perm.size() * 4) m->idx.alloc(perm.size() * 4);
        for (int ep = 0; ep < epochs; ep++) {
            std::shuffle(perm.begin(), perm.end(), gen);
            check(hipMemcpyAsync(m->idx.p, perm.data(), perm.size() * 4, hipMemcpyHostToDevice, st), "indices");
            for (int k = 0; k < nb; k++) {
                const bool last = ep + 1 == epochs && k + 1 == nb;  // its outputs and gradients can be read afterwards
                const int *idx = m->idx.as<int>() + (long) k * mb;
                hipLaunchKernelGGL(M::k_gather, grid1((long) mb * m->in()), dim3(256), 0, st, m->trX.as<float>(), m->in(),
                                   idx, mb, m->X.as<unsigned short>());
                hiddenLayers(m, mb);
                if (last) outputLayer(m, mb, false);
                o.C = m->dY.as<float>();
                o.Cb = m->dYb.as<unsigned short>();
                o.target = m->trT.as<float>();
                o.rows = idx;
                o.inv = 1.f / (float) n;
                o.loss = m->partial.as<double>() + (long) k * blocks;
                gemm<M::FWD_MSE>(m, o);
                const M::AdamArgs step = adamStep(m, lr, 0.9f, 0.999f, 1e-8f);
                backward(m, mb, last, &step);
            }
            check(hipMemcpyAsync(part.data(), m->partial.p, part.size() * sizeof(double), hipMemcpyDeviceToHost, st), "loss");
            check(hipStreamSynchronize(st), "sync");
            double acc = 0.;
            for (int k = 0; k < nb; k++) {
                double s = 0.;
                for (int b = 0; b < blocks; b++) s += part[(size_t) k * blocks + b];
                acc += s / (double) n;
            }
            if (epochLoss) epochLoss[ep] = acc / nb;
        }
        return 0;
    } catch (const std::exception &e) {
        return fail(m->ctx, e);
    }
}

int spk_mlp_predict(spk_mlp *m, const double *x0, int rows, spk_batch *dst) {
    try {
        if (rows != spk_batch_count(dst)) throw std::runtime_error("rows must equal the batch count");
        uploadInputs(m, x0, rows);
        if (float *lanes = spk::laneIterates(dst, m->ctx, m->out())) {
            hiddenLayers(m, rows);
            outputLayer(m, rows, true, lanes);
            check(hipStreamSynchronize(m->ctx->stream), "sync");
            return 0;
        }
        forward(m, rows, true);
        check(hipStreamSynchronize(m->ctx->stream), "sync");
        if (spk_batch_set_iterates_device(dst, m->Y.as<float>(), m->out())) throw std::runtime_error(m->ctx->err);
        return 0;
    } catch (const std::exception &e) {
        return fail(m->ctx, e);
    }
}

int spk_mlp_predict_lanes(spk_mlp *m, const double *x0, int rows, spk_batch *dst, const int *lanes) {
    try {
        uploadInputs(m, x0, rows);
        forward(m, rows, true);
        check(hipStreamSynchronize(m->ctx->stream), "sync");
        if (spk_batch_refill_rows(dst, rows, lanes, x0, m->Y.as<float>(), m->out())) throw std::runtime_error(m->ctx->err);
        return 0;
    } catch (const std::exception &e) {
        return fail(m->ctx, e);
    }
}

}  // extern "C"
