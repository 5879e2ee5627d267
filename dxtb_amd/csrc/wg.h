// Workgroup-level FP64 building blocks for gfx950 (one molecule per
// workgroup).  Every function here is called by ALL threads of the
// workgroup (they contain barriers) and assumes blockDim.x == XTB_NT.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#ifndef XTB_NT
#define XTB_NT 512
#endif

namespace xtb {

constexpr int NT = XTB_NT;
constexpr int WAVE = 64;
constexpr int NWAVE = NT / WAVE;

// Address-space-qualified pointers.  A function compiled out of line cannot
// tell whether a plain pointer addresses LDS or global memory and falls back
// to flat instructions (slower, and every wait covers both kinds of access);
// these types keep ds_* and global_* addressing across calls.
typedef __attribute__((address_space(3))) double ldsf;
typedef __attribute__((address_space(3))) int ldsi;
typedef __attribute__((address_space(1))) double glbf;
__device__ inline ldsf* to_lds(double* p) { return (ldsf*)p; }
__device__ inline ldsi* to_lds(int* p) { return (ldsi*)p; }
__device__ inline glbf* to_glb(double* p) { return (glbf*)p; }
__device__ inline const glbf* to_glb(const double* p) { return (const glbf*)p; }

__device__ __forceinline__ int uniform(int x) { return __builtin_amdgcn_readfirstlane(x); }
template <class T>
__device__ __forceinline__ T* uniform(T* p) {
    const uint64_t v = (uint64_t)p;
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
    return (T*)(((uint64_t)hi << 32) | lo);
}
// A uniform value or struct of them as scalars (arguments of an out-of-line
// call arrive in vector registers, which are spilled around the next call).
template <class T>
__device__ __forceinline__ T uniform_copy(const T& x) {
    static_assert(sizeof(T) % 4 == 0, "whole words");
    uint32_t v[sizeof(T) / 4];
    __builtin_memcpy(v, &x, sizeof(T));
#pragma unroll
    for (uint32_t& u : v) u = __builtin_amdgcn_readfirstlane(u);
    T y;
    __builtin_memcpy(&y, v, sizeof(T));
    return y;
}

// DPP move of a double; lanes without a source keep `old`
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp64(double old, double v) {
    const int lo = __builtin_amdgcn_update_dpp(__double2loint(old), __double2loint(v), CTRL, ROWS, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(__double2hiint(old), __double2hiint(v), CTRL, ROWS, 0xf, false);
    return __hiloint2double(hi, lo);
}
// lane `lane` (uniform) of v, on every lane
__device__ __forceinline__ double wave_read(double v, int lane) {
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), lane),
                            __builtin_amdgcn_readlane(__double2loint(v), lane));
}

// Reductions over a wave: up the rows of 16 lanes by row shifts 1, 2, 4, 8,
// then across the rows by row broadcasts; the result, in lane 63, goes to
// every lane as a uniform value.  Register moves only, ~150 cycles; a
// butterfly through LDS permutes took ~600.
__device__ __forceinline__ double wave_sum(double v) {
    v += dpp64<0x111, 0xf>(0.0, v);
    v += dpp64<0x112, 0xf>(0.0, v);
    v += dpp64<0x114, 0xf>(0.0, v);
    v += dpp64<0x118, 0xf>(0.0, v);
    v += dpp64<0x142, 0xa>(0.0, v);
    v += dpp64<0x143, 0xc>(0.0, v);
    return wave_read(v, WAVE - 1);
}

__device__ __forceinline__ double wave_max(double v) {
    v = fmax(v, dpp64<0x111, 0xf>(v, v));
    v = fmax(v, dpp64<0x112, 0xf>(v, v));
    v = fmax(v, dpp64<0x114, 0xf>(v, v));
    v = fmax(v, dpp64<0x118, 0xf>(v, v));
    v = fmax(v, dpp64<0x142, 0xa>(v, v));
    v = fmax(v, dpp64<0x143, 0xc>(v, v));
    return wave_read(v, WAVE - 1);
}

// K sums / maxima over the workgroup at once: v[K] per thread -> v[K] on
// every thread.  `red`: K NWAVE doubles of LDS that no thread still reads
// (they end with a barrier, so calls may follow one another).
template <int K>
__device__ inline void wg_sum_n(double (&v)[K], ldsf* red) {
    const int w = threadIdx.x / WAVE, l = threadIdx.x % WAVE;
#pragma unroll
    for (int k = 0; k < K; ++k) {
        v[k] = wave_sum(v[k]);
        if (l == 0) red[k * NWAVE + w] = v[k];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < K; ++k) {
        double s = 0.0;
#pragma unroll
        for (int i = 0; i < NWAVE; ++i) s += red[k * NWAVE + i];
        v[k] = s;
    }
    __syncthreads();
}
template <int K>
__device__ inline void wg_max_n(double (&v)[K], ldsf* red) {
    const int w = threadIdx.x / WAVE, l = threadIdx.x % WAVE;
#pragma unroll
    for (int k = 0; k < K; ++k) {
        v[k] = wave_max(v[k]);
        if (l == 0) red[k * NWAVE + w] = v[k];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < K; ++k) {
        double s = red[k * NWAVE];
#pragma unroll
        for (int i = 1; i < NWAVE; ++i) s = fmax(s, red[k * NWAVE + i]);
        v[k] = s;
    }
    __syncthreads();
}
__device__ inline double wg_sum(double v, ldsf* red) {
    double x[1] = {v};
    wg_sum_n<1>(x, red);
    return x[0];
}
__device__ inline double wg_max(double v, ldsf* red) {
    double x[1] = {v};
    wg_max_n<1>(x, red);
    return x[0];
}

// Y[e] = a X[e] + b Z[e] (Z null: a X[e]) over `len` contiguous elements, by
// the workgroup, four elements per thread in flight.  Y may alias X or Z
// (element-wise).  No barrier inside.
__device__ inline void wg_axpby(size_t len, double a, const glbf* X, double b, const glbf* Z, glbf* Y) {
    size_t e = threadIdx.x;
    for (; e + 3 * NT < len; e += 4 * NT) {
        double x[4], z[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            x[u] = X[e + u * NT];
            z[u] = Z ? Z[e + u * NT] : 0.0;
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) Y[e + u * NT] = Z ? a * x[u] + b * z[u] : a * x[u];
    }
    for (; e < len; e += NT) Y[e] = Z ? a * X[e] + b * Z[e] : a * X[e];
}

// The same on rows x cols elements of leading dimension ld.
__device__ inline void wg_axpby_rows(int rows, int cols, int ld, double a, const glbf* X, double b, const glbf* Z,
                                     glbf* Y) {
    if (cols == ld) {
        wg_axpby((size_t)rows * ld, a, X, b, Z, Y);
        return;
    }
    for (int r = threadIdx.x / WAVE; r < rows; r += NWAVE)
        for (int c = threadIdx.x % WAVE; c < cols; c += WAVE) {
            const size_t e = (size_t)r * ld + c;
            Y[e] = a * X[e] + b * Z[e];
        }
}

// ---------------------------------------------------------------------------
// FP64 matrix cores.  v_mfma_f64_16x16x4_f64: D(16x16) += A(16x4) B(4x16);
// lane l supplies A[l%16][l/16] and B[l/16][l%16] and holds
// D[l/16 + 4r][l%16] in element r of its 4-vector (checked on gfx950).  So
// element r of an output fragment is exactly the B operand of k-step r of a
// following product: fragments chain without a trip through LDS.
// ---------------------------------------------------------------------------
typedef double v4d __attribute__((ext_vector_type(4)));
typedef double v2d __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) v2d ldsv2;
// pairs of doubles in global memory need no more than a double's alignment
typedef double v2d8 __attribute__((ext_vector_type(2), aligned(8)));
typedef __attribute__((address_space(1))) v2d8 glbv2;

__device__ inline v4d mfma16(double a, double b, v4d c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

__device__ inline v4d v4zero() {
    v4d z = {0.0, 0.0, 0.0, 0.0};
    return z;
}

// ---------------------------------------------------------------------------
// Workgroup GEMM: C = alpha op(A) op(B) + beta C, and its fused forms, by one
// workgroup.
//
// What bounds it at these sizes is not the matrix cores (a 16x16x4 FP64 MFMA
// keeps its SIMD busy for 64 cycles) but fragments without output, and the
// latency around each k panel.  So
// * a workgroup tile is cut to the matrix in 16 x 16 fragments (up to 11 x 11):
//   one tile covers any product up to 176 x 176, larger ones are split evenly;
// * the fragments are dealt to the 8 waves one by one (wave w takes fragments
//   w, w + 8, ...; NF of them, compiled for every count 1..16), so all SIMDs
//   get the same number;
// * a 16-deep panel of both operands is loaded in pairs of doubles without a
//   branch (rows past the end repeat the last one), one panel ahead in
//   registers, and stored to the other LDS stage after three quarters of the
//   panel's MFMAs: one barrier per panel;
// * reads of two fragments' next half panel are issued before the MFMAs of
//   the current one, from addresses kept in registers with the stage and the
//   half panel in the instruction's offset: FP64 MFMAs run at the vector
//   FP64 rate on gfx950, and every vector instruction between them costs its
//   issue time.
// One workgroup alone / 256 of them, n x n x n, us: n = 68: 9.1 / 10.5, 136: 34
// / 44, 171: 59 / 81, 300: 287 / 400, 528: 1329 / 1595 (72 % of a CU's peak
// alone; with all CUs at it the clock falls from 2.4 to 1.85 GHz).  Tiles of
// 128 x 128 to 64 x 64 with a fixed 2 x 4 wave grid, bounds tests on every
// load and 8-byte LDS accesses took 11.4 / 13, 64 / 71, 86 / 97, 371 / 448,
// 1784 / 1904: n = 136 ran four 128-wide tiles at a quarter of their area.
// ---------------------------------------------------------------------------
typedef __attribute__((address_space(1))) char glbc;

constexpr int GEMM_KP = 16;             // k-panel depth
constexpr int GEMM_F = 11;              // fragment rows (columns) of a workgroup tile, at most
constexpr int GEMM_R = 16 * GEMM_F;
constexpr int GEMM_PITCH = 18;          // row pitch of a panel stored [row][k]: conflict-free 16-byte reads
constexpr int GEMM_KPITCH = GEMM_R + 8; // k pitch of a panel stored [k][row]: conflict-free 8-byte reads
constexpr int GEMM_SIDE = GEMM_R * GEMM_PITCH;  // doubles of one operand's panel
constexpr int GEMM_STAGE = 2 * GEMM_SIDE;
constexpr int NGEMM_MFMA_LDS = 2 * GEMM_STAGE;
static_assert(GEMM_KP * GEMM_KPITCH <= GEMM_SIDE, "either layout fits");

// One operand of a workgroup tile: panels of R = 16 F rows.  KM: stored with
// k contiguous, staged as [row][k]; otherwise staged as [k][row].  Each thread loads GE pairs of doubles per
// panel (64 GE >= R).  In a partial last panel of `rem` k, those past the end
// are read at the last valid ones (shift) and zeroed when stored.  Needs K >=
// 2 (KM) or M >= 2 rows (otherwise).
template <bool KM, int GE>
struct GemmSide {
    const glbc* p;
    uint32_t step, shift;
    int R, last, dst;
    uint32_t off[GE];
    __device__ __forceinline__ void init(const glbf* X, int ld, int m0, int M, int F, int rem) {
        const int t = threadIdx.x;
        const uint32_t ld8 = (uint32_t)ld * 8u;
        R = 16 * F;
        last = M - m0 - 1;
        if (KM) {
            // one double back, so that a last panel of one k, read as the pair
            // that ends with it, still has an offset >= 0
            p = (const glbc*)X + (size_t)m0 * ld8 - 8;
            step = 8 * GEMM_KP;
            dst = (t >> 3) * GEMM_PITCH + 2 * (t & 7);
            const int over = 2 * (t & 7) - (rem - 2);
            shift = over > 0 ? (uint32_t)over * 8u : 0u;
#pragma unroll
            for (int e = 0; e < GE; ++e) {
                const int row = (t >> 3) + 64 * e;
                off[e] = (uint32_t)(row < last ? row : last) * ld8 + (uint32_t)(t & 7) * 16u + 8u;
            }
        } else {
            // pairs of rows (m, m + 1): an odd last row is read with the one
            // before it (which lies in the previous tile when it is alone)
            const int base = last > 0 ? 0 : -1;
            p = (const glbc*)X + (ptrdiff_t)(m0 + base) * 8;
            step = GEMM_KP * ld8;
            dst = (t >> 5) * GEMM_KPITCH + 2 * (t & 31);
            const int over = (t >> 5) - (rem - 1);
            shift = over > 0 ? (uint32_t)over * ld8 : 0u;
#pragma unroll
            for (int e = 0; e < GE; ++e) {
                const int m = 2 * (t & 31) + 64 * e;
                off[e] = (uint32_t)(t >> 5) * ld8 + (uint32_t)((m < last - 1 ? m : last - 1) - base) * 8u;
            }
        }
    }
    __device__ __forceinline__ void load(v2d (&st)[GE], bool tail) {
        const uint32_t sh = tail ? shift : 0u;
#pragma unroll
        for (int e = 0; e < GE; ++e) st[e] = *(const glbv2*)(p + (off[e] - sh));
        p += step;
    }
    __device__ __forceinline__ void store(v2d (&st)[GE], ldsf* s, int rem) const {
        const int t = threadIdx.x;
        if (rem) {
#pragma unroll
            for (int e = 0; e < GE; ++e) {
                if (KM) {
                    const int k = 2 * (t & 7);
                    if (k == rem - 1) st[e].x = st[e].y;  // read one k early
                    if (k >= rem) st[e].x = 0.0;
                    if (k + 1 >= rem) st[e].y = 0.0;
                } else if ((t >> 5) >= rem) {
                    st[e].x = 0.0;
                    st[e].y = 0.0;
                }
            }
        }
#pragma unroll
        for (int e = 0; e < GE; ++e) {
            if (KM) {
                if ((t >> 3) + 64 * e < R) *(ldsv2*)(s + dst + 64 * e * GEMM_PITCH) = st[e];
            } else {
                const int m = 2 * (t & 31) + 64 * e;
                if (m < R) {
                    v2d v = st[e];
                    if (m == last) v.x = v.y;  // read one row early
                    *(ldsv2*)(s + dst + 64 * e) = v;
                }
            }
        }
    }
    // this lane's address of fragment row f in stage 0; the k of half panel h
    // are 8 h + 2 lg + j, j = 0, 1 (both operands deal k to the MFMA steps the
    // same way)
    __device__ __forceinline__ const ldsf* at(const ldsf* s, int f, int li, int lg) const {
        return s + (KM ? (16 * f + li) * GEMM_PITCH + 2 * lg : 2 * lg * GEMM_KPITCH + 16 * f + li);
    }
    // stage and half are compile-time constants: they go into the read's offset
    static __device__ __forceinline__ v2d frag(const ldsf* q, int stage, int h) {
        q += stage * GEMM_STAGE;
        if (KM) return *(const ldsv2*)(q + 8 * h);
        const v2d v = {q[8 * h * GEMM_KPITCH], q[(8 * h + 1) * GEMM_KPITCH]};
        return v;
    }
};

// PLAIN: C = alpha op(A) op(B) + beta C; with `sym` (M == N, a symmetric
// product, beta unused) only the fragments on and above the diagonal are
// formed, each also written transposed.  EPI: C = alpha op(A) op(B) + s1 E1 +
// s2 E2, elementwise (E1, E2 with C's leading dimension; C may be E1 or E2, a
// thread reads an element and then writes it).  MULL: C not written; the sums
// a_i = sum_j alpha (op(A) op(B))_ij E1_ij over i, j < nao of a symmetric
// product go to C[i] (0 for i >= nao), from the fragments on and above the
// diagonal: the row sums of each, and the column sums for the rows of its
// mirror image, added per row in a fixed order.  A and B must not overlap C.
enum { GEMM_PLAIN = 0, GEMM_EPI = 1, GEMM_MULL = 2, GEMM_DOT = 3 };

struct GemmOut {
    int M, N;
    double alpha, beta;
    glbf* C;
    int ldc;
    const glbf *E1, *E2;
    double s1, s2;
    int nao;
};

// One workgroup tile of 16 fm x 16 fn at (m0, n0); diag: a diagonal tile of a
// symmetric product.  All threads have passed a barrier since the LDS
// stages' last use.
template <bool TA, bool TB, int NF, int GE, int MODE>
__device__ __forceinline__ void gemm_wg_tile(const GemmOut& g, int m0, int n0, int fm, int fn, int K,
                                             const glbf* A, int lda, const glbf* B, int ldb, bool sym, bool diag,
                                             ldsf* lds) {
    static_assert(NT == 512, "panel loads assume 512 threads");
    const int w = uniform((int)threadIdx.x / WAVE), lane = threadIdx.x % WAVE;
    const int li = lane % 16, lg = lane / 16;
    const int rem = K & 15, np = (K + 15) >> 4;
    GemmSide<!TA, GE> a;
    GemmSide<TB, GE> b;
    a.init(A, lda, m0, g.M, fm, rem);
    b.init(B, ldb, n0, g.N, fn, rem);
    // this wave's fragments (row-major; of a diagonal tile's upper triangle
    // rows d and fm - 1 - d together make a run of fm + 1); idle slots repeat
    // the last fragment and write nothing
    const int T = diag ? fm * (fm + 1) / 2 : fm * fn;
    const int run = diag ? fm + 1 : fn;
    const uint32_t inv = 65536u / (uint32_t)run + 1u;  // q / run, q < 256, run <= 13
    int fr[NF], fc[NF];
    const ldsf *qa[NF], *qb[NF];
#pragma unroll
    for (int t = 0; t < NF; ++t) {
        int q = w + NWAVE * t;
        q = q < T ? q : T - 1;
        const int d = (int)(((uint32_t)q * inv) >> 16), r = q - d * run;
        fr[t] = d;
        fc[t] = r;
        if (diag) {
            const bool lo = r < fm - d;
            fr[t] = lo ? d : fm - 1 - d;
            fc[t] = lo ? d + r : r - 1;
        }
        qa[t] = a.at(lds, fr[t], li, lg);
        qb[t] = b.at(lds + GEMM_SIDE, fc[t], li, lg);
    }
    v4d acc[NF];
#pragma unroll
    for (int t = 0; t < NF; ++t) acc[t] = v4zero();
    auto load = [&](int p, v2d (&sa)[GE], v2d (&sb)[GE]) {
        const bool tail = rem && p == np - 1;
        a.load(sa, tail);
        b.load(sb, tail);
    };
    auto store = [&](int p, int stg, v2d (&sa)[GE], v2d (&sb)[GE]) {
        ldsf* s = lds + stg * GEMM_STAGE;
        const int r = p == np - 1 ? rem : 0;
        a.store(sa, s, r);
        b.store(sb, s + GEMM_SIDE, r);
    };
    // units of two fragments x half a panel (8 k): the reads of a unit are
    // issued one unit ahead, the MFMAs of its two fragments alternate
    constexpr int NU = 2 * ((NF + 1) / 2);
    auto read = [&](int stg, int u, v2d (&x)[2], v2d (&y)[2]) {
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const int t = 2 * (u >> 1) + q;
            if (t < NF) {
                x[q] = a.frag(qa[t], stg, u & 1);
                y[q] = b.frag(qb[t], stg, u & 1);
            }
        }
    };
    auto multiply = [&](int u, const v2d (&x)[2], const v2d (&y)[2]) {
        const int t = 2 * (u >> 1);
        acc[t] = mfma16(x[0].x, y[0].x, acc[t]);
        if (t + 1 < NF) acc[t + 1] = mfma16(x[1].x, y[1].x, acc[t + 1]);
        acc[t] = mfma16(x[0].y, y[0].y, acc[t]);
        if (t + 1 < NF) acc[t + 1] = mfma16(x[1].y, y[1].y, acc[t + 1]);
    };
    auto panel = [&](int p, int stg) {
        __syncthreads();
        v2d x[2][2], y[2][2], sa[GE], sb[GE];
        if (p + 1 < np) load(p + 1, sa, sb);
        read(stg, 0, x[0], y[0]);
        __builtin_amdgcn_sched_barrier(0);
        constexpr int US = NU - (NU + 3) / 4;
#pragma unroll
        for (int u = 0; u < NU; ++u) {
            if (u == US && p + 1 < np) store(p + 1, 1 - stg, sa, sb);
            if (u + 1 < NU) {
                read(stg, u + 1, x[(u + 1) & 1], y[(u + 1) & 1]);
                __builtin_amdgcn_sched_barrier(0);
            }
            multiply(u, x[u & 1], y[u & 1]);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    {
        v2d sa[GE], sb[GE];
        load(0, sa, sb);
        store(0, 0, sa, sb);
    }
    for (int p = 0; p < np; p += 2) {
        panel(p, 0);
        if (p + 1 < np) panel(p + 1, 1);
    }
    // Epilogue, G fragments at a time so that what it reads is in flight
    // together, at clamped places without branches.  Per product of a step at
    // n = 292 with all CUs at it: with two added matrices 75 us (one element
    // after the other, each waiting for its loads: 105), the Mulliken sums
    // with their gathers 242 (308)
    constexpr int G = NF < 4 ? NF : 4;
    auto live = [&](int t) { return w + NWAVE * t < T; };
    auto row = [&](int t, int r) { return m0 + 16 * fr[t] + lg + 4 * r; };
    auto col = [&](int t) { return n0 + 16 * fc[t] + li; };
    const uint32_t ldc = (uint32_t)g.ldc * 8u;
    auto fetch = [&](const glbf* X, int M, int N, int t0, double (&x)[G][4]) {
#pragma unroll
        for (int u = 0; u < G; ++u)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int t = t0 + u < NF ? t0 + u : NF - 1;
                const int gm = row(t, r) < M ? row(t, r) : M - 1, gn = col(t) < N ? col(t) : N - 1;
                x[u][r] = *(const glbf*)((const glbc*)X + ((uint32_t)gm * ldc + (uint32_t)gn * 8u));
            }
    };
    if constexpr (MODE == GEMM_DOT) {
        ldsf* rowp = lds;  // [fn][16 fm] row sums of fragment column c
        ldsf* out = (ldsf*)(uintptr_t)(uint32_t)g.nao;
        double x[G][4];
        fetch(g.E1, g.M, g.N, 0, x);
        __syncthreads();  // every wave has read the last panel
#pragma unroll
        for (int t0 = 0; t0 < NF; t0 += G) {
            if (t0 > 0) fetch(g.E1, g.M, g.N, t0, x);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int u = 0; u < G; ++u) {
                const int t = t0 + u;
                if (t >= NF || !live(t)) continue;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const bool in = row(t, r) < g.M && col(t) < g.N;
                    if (in) *(glbf*)((glbc*)g.C + ((uint32_t)row(t, r) * ldc + (uint32_t)col(t) * 8u)) = acc[t][r];
                    double v = in ? acc[t][r] * x[u][r] : 0.0;
                    v += dpp64<0x111, 0xf>(0.0, v);
                    v += dpp64<0x112, 0xf>(0.0, v);
                    v += dpp64<0x114, 0xf>(0.0, v);
                    v += dpp64<0x118, 0xf>(0.0, v);
                    if (li == 15) rowp[fc[t] * 16 * fm + 16 * fr[t] + lg + 4 * r] = v;
                }
            }
        }
        __syncthreads();
        for (int i = threadIdx.x; i < 16 * fm; i += NT) {
            if (m0 + i >= g.M) continue;
            double s = n0 > 0 ? out[m0 + i] : 0.0;
            for (int c = 0; c < fn; ++c) s += rowp[c * 16 * fm + i];
            out[m0 + i] = s;
        }
        __syncthreads();
        return;
    }
    if constexpr (MODE == GEMM_MULL) {
        ldsf* rowp = lds;                 // [fn][16 fm] row sums of fragment column c
        ldsf* colp = lds + 16 * fm * fn;  // [4 fm][16 fn] column sums of four rows of fragment row r
        double x[G][4];
        fetch(g.E1, g.nao, g.nao, 0, x);
        __syncthreads();  // every wave has read the last panel
#pragma unroll
        for (int t0 = 0; t0 < NF; t0 += G) {
            if (t0 > 0) fetch(g.E1, g.nao, g.nao, t0, x);
#pragma unroll
            for (int u = 0; u < G; ++u) {
                const int t = t0 + u;
                if (t >= NF || !live(t)) continue;
                double cs = 0.0;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    double v = row(t, r) < g.nao && col(t) < g.nao ? g.alpha * acc[t][r] * x[u][r] : 0.0;
                    cs += v;
                    v += dpp64<0x111, 0xf>(0.0, v);
                    v += dpp64<0x112, 0xf>(0.0, v);
                    v += dpp64<0x114, 0xf>(0.0, v);
                    v += dpp64<0x118, 0xf>(0.0, v);
                    if (li == 15) rowp[fc[t] * 16 * fm + 16 * fr[t] + lg + 4 * r] = v;
                }
                colp[(4 * fr[t] + lg) * 16 * fn + 16 * fc[t] + li] = cs;
            }
        }
        __syncthreads();
        for (int i = threadIdx.x; i < 16 * fm; i += NT) {
            if (m0 + i >= g.M) continue;
            double s = g.C[m0 + i];
            for (int c = diag ? i / 16 : 0; c < fn; ++c) s += rowp[c * 16 * fm + i];
            if (diag)
                for (int r = 0; r < i / 16 * 4; ++r) s += colp[r * 16 * fn + i];
            g.C[m0 + i] = s;
        }
        if (!diag)
            for (int i = threadIdx.x; i < 16 * fn; i += NT) {
                if (n0 + i >= g.N) continue;
                double s = g.C[n0 + i];
                for (int r = 0; r < 4 * fm; ++r) s += colp[r * 16 * fn + i];
                g.C[n0 + i] = s;
            }
        __syncthreads();
        return;
    }
    glbc* C = (glbc*)g.C;
    const bool add = MODE == GEMM_PLAIN && !sym && g.beta != 0.0;
#pragma unroll
    for (int t0 = 0; t0 < NF; t0 += G) {
        double x[G][4], y[G][4];
        if (MODE == GEMM_EPI) {
            fetch(g.E1, g.M, g.N, t0, x);
            fetch(g.E2, g.M, g.N, t0, y);
        } else if (add) {
            fetch(g.C, g.M, g.N, t0, x);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < G; ++u) {
            const int t = t0 + u;
            if (t >= NF || !live(t)) continue;
            const int gn = col(t);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int gm = row(t, r);
                double v = g.alpha * acc[t][r];
                if (MODE == GEMM_EPI) v = fma(g.alpha, acc[t][r], fma(g.s1, x[u][r], g.s2 * y[u][r]));
                else if (add) v = fma(g.alpha, acc[t][r], g.beta * x[u][r]);
                if (gm < g.M && gn < g.N) {
                    *(glbf*)(C + ((uint32_t)gm * ldc + (uint32_t)gn * 8u)) = v;
                    if (sym && (!diag || fr[t] != fc[t])) *(glbf*)(C + ((uint32_t)gn * ldc + (uint32_t)gm * 8u)) = v;
                }
            }
        }
    }
    __syncthreads();
}

// `tile`: fm | fn << 8 | sym << 16 | part << 17; part 1, 2: the diagonal tiles
// of a symmetric product only, the others only
template <bool TA, bool TB, int NF, int GE, int MODE>
__device__ __noinline__ void wg_gemm(int M, int N, int K, int tile, double alpha, const glbf* A, int lda,
                                     const glbf* B, int ldb, double beta, glbf* C, int ldc, ldsf* lds,
                                     const glbf* E1, const glbf* E2, double s1, double s2, int nao) {
    // arguments of an out-of-line call arrive in vector registers; they are
    // uniform, and saying so turns the tests into scalar branches and the
    // addresses into a scalar base plus a 32-bit lane offset
    M = uniform(M);
    N = uniform(N);
    K = uniform(K);
    lda = uniform(lda);
    ldb = uniform(ldb);
    tile = uniform(tile);
    A = uniform(A);
    B = uniform(B);
    GemmOut g{M, N, alpha, beta, uniform(C), uniform(ldc), nullptr, nullptr, s1, s2, 0};
    if (MODE != GEMM_PLAIN) g.E1 = uniform(E1);
    if (MODE == GEMM_EPI) g.E2 = uniform(E2);
    if (MODE == GEMM_MULL || MODE == GEMM_DOT) g.nao = uniform(nao);
    const int fm = tile & 255, fn = (tile >> 8) & 255;
    const bool sym = MODE == GEMM_MULL || (MODE == GEMM_PLAIN && (tile >> 16 & 1));
    const int part = tile >> 17;
    if (MODE == GEMM_MULL && part != 2) {
        for (int i = threadIdx.x; i < M; i += NT) g.C[i] = 0.0;
        __syncthreads();
    }
    const int FM = (M + 15) >> 4, FN = (N + 15) >> 4;
    for (int i = 0; i < FM; i += fm)
        for (int j = 0; j < FN; j += fn) {
            if (sym && (j < i || (part && (i == j) != (part == 1)))) continue;
            gemm_wg_tile<TA, TB, NF, GE, MODE>(g, 16 * i, 16 * j, FM - i < fm ? FM - i : fm, FN - j < fn ? FN - j : fn,
                                               K, A, lda, B, ldb, sym, sym && i == j, lds);
        }
}

// Products that the panel loads do not take (fewer than two k, or fewer than
// two rows of an operand stored by rows): an element per thread.
template <bool TA, bool TB, int MODE>
__device__ __noinline__ void wg_gemm_thin(int M, int N, int K, double alpha, const glbf* A, int lda, const glbf* B,
                                          int ldb, double beta, glbf* C, int ldc, const glbf* E1, const glbf* E2,
                                          double s1, double s2, int nao) {
    auto dot = [&](int i, int j) {
        double d = 0.0;
        for (int k = 0; k < K; ++k)
            d = fma(TA ? A[(size_t)k * lda + i] : A[(size_t)i * lda + k],
                    TB ? B[(size_t)j * ldb + k] : B[(size_t)k * ldb + j], d);
        return alpha * d;
    };
    if (MODE == GEMM_MULL) {
        for (int i = threadIdx.x; i < M; i += NT) {
            double a = 0.0;
            for (int j = 0; j < nao && i < nao; ++j) a = fma(dot(i, j), E1[(size_t)i * ldc + j], a);
            C[i] = a;
        }
    } else if (MODE == GEMM_DOT) {
        ldsf* out = (ldsf*)(uintptr_t)(uint32_t)nao;
        for (int i = threadIdx.x; i < M; i += NT) {
            double a = 0.0;
            for (int j = 0; j < N; ++j) {
                const size_t x = (size_t)i * ldc + j;
                const double d = dot(i, j);
                C[x] = d;
                a = fma(d, E1[x], a);
            }
            out[i] = a;
        }
    } else {
        for (int e = threadIdx.x; e < M * N; e += NT) {
            const int i = e / N, j = e - i * N;
            const size_t x = (size_t)i * ldc + j;
            const double d = dot(i, j);
            if (MODE == GEMM_EPI) C[x] = d + fma(s1, E1[x], s2 * E2[x]);
            else C[x] = beta == 0.0 ? d : fma(beta, C[x], d);
        }
    }
    __syncthreads();
}

// The workgroup tile: the whole product if it fits, otherwise the longer side
// is split (evenly) until it does; the wave's fragment count and the panel
// loads per thread follow from it.
template <bool TA, bool TB, int MODE>
__device__ inline void gemm_run(int M, int N, int K, double alpha, const glbf* A, int lda, const glbf* B, int ldb,
                                double beta, glbf* C, int ldc, ldsf* lds, bool sym, const glbf* E1, const glbf* E2,
                                double s1, double s2, int nao) {
    M = uniform(M);
    N = uniform(N);
    K = uniform(K);
    if (M <= 0 || N <= 0) return;
    if (K < 2 || (TA && M < 2) || (!TB && N < 2)) {
        wg_gemm_thin<TA, TB, MODE>(M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, E1, E2, s1, s2, nao);
        return;
    }
    const int FM = (M + 15) >> 4, FN = (N + 15) >> 4;
    int pm = 1, pn = 1, fm = FM, fn = FN;
    while (fm > GEMM_F || fn > GEMM_F) {
        if (sym) fm = fn = (FM + pm) / (pm + 1), ++pm;
        else if (fm > fn) fm = (FM + pm) / (pm + 1), ++pm;
        else fn = (FN + pn) / (pn + 1), ++pn;
    }
    // Several tiles of a symmetric product: the diagonal ones, with half the
    // fragments, and the others in a call each.
    const int big = fm > fn ? fm : fn, split = sym && fm < FM ? 1 : 0;
#pragma unroll 1
    for (int part = split; part <= 2 * split; ++part) {
        const int T = sym && part < 2 ? fm * (fm + 1) / 2 : fm * fn;
        const int nf = (T + 7) >> 3;
        const int tile = fm | fn << 8 | (sym ? 1 : 0) << 16 | part << 17;
#define XTB_G(NF, GE)                                                                                                \
    wg_gemm<TA, TB, NF, GE, MODE>(M, N, K, tile, alpha, A, lda, B, ldb, beta, C, ldc, lds, E1, E2, s1, s2, nao)
#define XTB_G23(NF)             \
    case NF:                    \
        if (big <= 8) XTB_G(NF, 2); \
        else XTB_G(NF, 3);      \
        break;
#define XTB_G3(NF)     \
    case NF:           \
        XTB_G(NF, 3);  \
        break;
        switch (nf) {
            case 1:
                if (big <= 4) XTB_G(1, 1);
                else XTB_G(1, 3);
                break;
            case 2:
                if (big <= 4) XTB_G(2, 1);
                else XTB_G(2, 3);
                break;
            XTB_G23(3) XTB_G23(4) XTB_G23(5) XTB_G23(6) XTB_G23(7) XTB_G23(8)
            XTB_G3(9) XTB_G3(10) XTB_G3(11) XTB_G3(12) XTB_G3(13) XTB_G3(14) XTB_G3(15)
            default: XTB_G(16, 3);
        }
    }
#undef XTB_G3
#undef XTB_G23
#undef XTB_G
}

// C = alpha op(A) op(B) + beta C
template <bool TA, bool TB>
__device__ inline void gemm(int M, int N, int K, double alpha, const glbf* A, int lda,
                            const glbf* B, int ldb, double beta, glbf* C, int ldc, ldsf* lds) {
    gemm_run<TA, TB, GEMM_PLAIN>(M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, lds, false, nullptr, nullptr, 0.0, 0.0,
                                 0);
}

// C = A B + s1 E1 + s2 E2 (row-major, E1 and E2 with C's leading dimension)
__device__ inline void gemm_epi(int M, int N, int K, const glbf* A, int lda, const glbf* B, int ldb,
                                glbf* C, int ldc, const glbf* E1, double s1, const glbf* E2, double s2,
                                ldsf* lds) {
    gemm_run<false, false, GEMM_EPI>(M, N, K, 1.0, A, lda, B, ldb, 0.0, C, ldc, lds, false, E1, E2, s1, s2, 0);
}

// C = A B and, with X of C's shape and leading dimension, the diagonal of C
// X^T: out[i] = sum_j C_ij X_ij (LDS).  A pass of its own over C and X took 5
// us of a step's 68 at n = 68, 43 at n = 289 with all CUs at it; in the product
// 2 and 15 more.
__device__ inline void gemm_dot(int M, int N, int K, const glbf* A, int lda, const glbf* B, int ldb, glbf* C, int ldc,
                                const glbf* X, ldsf* out, ldsf* lds) {
    gemm_run<false, false, GEMM_DOT>(M, N, K, 1.0, A, lda, B, ldb, 0.0, C, ldc, lds, false, X, nullptr, 0.0, 0.0,
                                     (int)(uint32_t)(uintptr_t)out);
}

// C (n x n) = alpha op(A) op(B) for a product known to be symmetric
template <bool TA, bool TB>
__device__ inline void gemm_sym(int n, int K, double alpha, const glbf* A, int lda, const glbf* B, int ldb,
                                glbf* C, int ldc, ldsf* lds) {
    gemm_run<TA, TB, GEMM_PLAIN>(n, n, K, alpha, A, lda, B, ldb, 0.0, C, ldc, lds, true, nullptr, nullptr, 0.0, 0.0, 0);
}

// Mulliken sums out[i] = sum_{j < nao} P_ij S_ij (0 for i >= nao) of the
// symmetric n x n product P = op(A) op(B), which is never stored.  S with
// leading dimension ldS.
template <bool TA, bool TB>
__device__ inline void gemm_sym_mull(int n, int K, const glbf* A, int lda, const glbf* B, int ldb, const glbf* S,
                                     int ldS, int nao, glbf* out, ldsf* lds) {
    gemm_run<TA, TB, GEMM_MULL>(n, n, K, 1.0, A, lda, B, ldb, 0.0, out, ldS, lds, true, S, nullptr, 0.0, 0.0, nao);
}

// Round-robin ("circle method") pairing of n2 (even) players: in round r,
// pair k matches (n2-1, r) for k = 0 and ((r+k) mod (n2-1), (r-k) mod (n2-1))
// otherwise.  Every unordered pair meets once in n2-1 rounds.
__device__ inline void rr_pair(int r, int k, int n2, int& p, int& q) {
    const int m = n2 - 1;
    if (k == 0) { p = m; q = r; }
    else { p = (r + k) % m; q = (r - k + m) % m; }
}

// Occupation classes (cb_lo >= 0): index i has class (i < cb_lo) + (i < cb_hi)
// (doubly, singly, un-occupied for sorted orbitals).  Mode 1 rotates and
// tests only pairs of different classes, which decouples the classes without
// diagonalising inside them (the density of integer occupations needs no
// more); mode 2 only pairs of the same class, which diagonalises inside
// classes that are already decoupled.  Mode 0 (cb_lo < 0): every pair.
__device__ inline int occ_class(int i, int cb_lo, int cb_hi) { return (i < cb_lo) + (i < cb_hi); }
__device__ inline bool pair_in_mode(int mode, int ci, int cj) {
    return mode == 0 || ((ci != cj) == (mode == 1));
}

// ---------------------------------------------------------------------------
// Cyclic two-sided Jacobi with parallel (round-robin) ordering for matrices
// that fit in LDS, one workgroup per matrix.
//
// Round r of the ordering (rr_pair) pairs position k = 0 as (m, r) and
// position k > 0 as (p, q) = (r + k, r - k) mod m, with n2 = n rounded up to
// even, m = n2 - 1 and K = n2 / 2 pairs; m rounds make a sweep.
//
// Storage follows the ring of the m moving indices: the element of indices i
// and j = i + d (mod m), 0 <= d < K, lies at D[d W + i], the elements of the
// fixed index m in a last row at D[K W + i], its diagonal at D[K W + m].  The
// difference d of the elements that two pairs (P, R) share is then the same
// in every round and only the start index moves by one, so an address costs
// one add and a wrap; the packed triangle took a min, max and multiply per
// element.  Consecutive lanes (consecutive R) step by W, W + 1 or W - 1
// doubles: with W = 2 mod 4 at most two of 32 lanes share a bank.
//
// The vectors do not enter the elimination, so a sweep first runs all its
// rounds on D, recording every (c, s) in global memory, and then applies the
// whole sweep to the vectors (ring_vectors).  Bounds: per round two barriers,
// the rotation parameters' dependent divide and square roots on K threads,
// and 8 LDS accesses per 2 x 2 block.  One workgroup, per round with its
// share of the vector pass: 1.04 us at n = 20, 1.65 at 68, 2.2 at 100, 3.8
// at 136, 5.5 at 184, half of it the vectors (a packed triangle walked row by
// row with the vectors rotated in LDS or memory: 2.5 us at n = 20, 5.1 at
// 68, 17.8 at 136).
// ---------------------------------------------------------------------------
struct Ring {
    ldsf* D;
    int n, m, K, W;
    __device__ inline int wrap(int i) const { return i >= m ? i - m : (i < 0 ? i + m : i); }
    // offset of element (i, j), i != j
    __device__ inline int at(int i, int j) const {
        if (i > j) { const int t = i; i = j; j = t; }
        if (j == m) return K * W + i;
        const int d = j - i;
        return d < K ? d * W + i : (m - d) * W + j;
    }
    __device__ inline int diag(int i) const { return i == m ? K * W + m : i; }
};

// The largest n that the rounds cover: 10 of the K (K - 1) / 2 2 x 2 blocks for
// each thread.
constexpr int RING_MAX_N = 202;

// doubles that Ring needs for n with row pitch W (the row of the fixed index
// exists for even n only; it is a dummy otherwise)
__host__ __device__ constexpr int ring_pairs(int n) { return (n + 1) / 2; }
__host__ __device__ constexpr int ring_doubles(int n, int W) {
    return ring_pairs(n) * W + (n % 2 == 0 ? n : 0);
}
static_assert(ring_pairs(RING_MAX_N) * (ring_pairs(RING_MAX_N) - 1) / 2 <= 10 * NT, "ring_rounds<10>");
// row pitch: the next W = 2 mod 4 if the matrix then fits in cap doubles
__host__ __device__ inline int ring_pitch(int n, int cap) {
    const int m = 2 * ring_pairs(n) - 1;
    int W = m;
    while (W % 4 != 2) ++W;
    return ring_doubles(n, W) <= cap ? W : m;
}

// lane l <- lane l - 1 (lane 0 <- first) and lane l <- lane l + 1 (lane 63 <- last)
__device__ __forceinline__ double wave_up(double v, double first) { return dpp64<0x138, 0xf>(first, v); }
__device__ __forceinline__ double wave_down(double v, double last) { return dpp64<0x130, 0xf>(last, v); }

// One recorded sweep applied to C columns of the row-major vectors Ct (row k
// = vector k) by one wave: lane l (and l + 64 with two sets) holds the two
// rows paired at its position in registers, rotates them, and then every row
// moves to its position of the next round: along the top of the ring to the
// left, along the bottom to the right, the top of position 0 fixed.  After
// the m rounds every row is back where it started.  Register traffic only:
// 4 FP64 instructions and 8 moves per column, pair set and round, where
// rotating rows in memory was bound by the latency of 4 accesses per pair.
// `rot`: (c, s) of round r and pair k at rot[2 ring_slot(n, r, k)].
__device__ inline size_t ring_slot(int n, int r, int k) {
    // the fixed index of an odd n is a dummy: its pair is not recorded, so
    // that a sweep takes at most n^2 doubles
    const int K = ring_pairs(n), o = n & 1;
    return (size_t)r * (K - o) + (k - o);
}

template <int SETS, int C>
__device__ __noinline__ void ring_vectors_t(glbf* Ct, int ldc, int n, const glbf* rot, int c0, int ncol) {
    const int lane = threadIdx.x % WAVE;
    const int K = ring_pairs(n), m = 2 * K - 1;
    double top[SETS][C], bot[SETS][C];
    int rt[SETS], rb[SETS];
#pragma unroll
    for (int u = 0; u < SETS; ++u) {
        const int k = lane + WAVE * u;
        rt[u] = k == 0 ? m : k;
        rb[u] = k == 0 ? 0 : m - k;
        if (k >= K || rt[u] >= n) rt[u] = -1;
        if (k >= K) rb[u] = -1;
#pragma unroll
        for (int c = 0; c < C; ++c) {
            const bool in = c < ncol;
            top[u][c] = (in && rt[u] >= 0) ? Ct[(size_t)rt[u] * ldc + c0 + c] : 0.0;
            bot[u][c] = (in && rb[u] >= 0) ? Ct[(size_t)rb[u] * ldc + c0 + c] : 0.0;
        }
    }
    // (c, s) four rounds ahead: pairs past the end repeat the last one (their
    // rows are not stored)
    constexpr int RB = SETS == 1 ? 4 : 2;
    v2d cur[RB][SETS], nxt[RB][SETS];
    auto fetch = [&](int r0, v2d (&x)[RB][SETS]) {
#pragma unroll
        for (int b = 0; b < RB; ++b)
#pragma unroll
            for (int u = 0; u < SETS; ++u) {
                const int r = r0 + b < m ? r0 + b : m - 1;
                const int k = lane + WAVE * u < K ? lane + WAVE * u : K - 1;
                const bool none = k == 0 && (n & 1);
                x[b][u] = *(const glbv2*)(rot + 2 * ring_slot(n, r, none ? 1 : k));
                if (none) x[b][u] = v2d{1.0, 0.0};
            }
    };
    const bool first = lane == 0;
    const int kl = (K - 1) % WAVE;
    fetch(0, cur);
    for (int r0 = 0; r0 < m; r0 += RB) {
        fetch(r0 + RB, nxt);
#pragma unroll
        for (int b = 0; b < RB; ++b) {
            if (r0 + b >= m) break;
#pragma unroll
            for (int c = 0; c < C; ++c) {
#pragma unroll
                for (int u = 0; u < SETS; ++u) {
                    const double x = top[u][c], y = bot[u][c], cs = cur[b][u].x, sn = cur[b][u].y;
                    top[u][c] = cs * x - sn * y;
                    bot[u][c] = sn * x + cs * y;
                }
                if constexpr (SETS == 1) {
                    if (K == 1) continue;  // one pair, nothing moves
                    const double t = top[0][c], e = bot[0][c];
                    const double up = wave_down(t, e);  // position k takes k + 1's top
                    bot[0][c] = wave_up(e, up);         // and k - 1's bottom; 0: the top of 1
                    top[0][c] = first ? t : (lane == kl ? e : up);
                } else {
                    const double t0 = top[0][c], t1 = top[1][c], e0 = bot[0][c], e1 = bot[1][c];
                    const double up0 = wave_down(t0, wave_read(t1, 0)), up1 = wave_down(t1, e1);
                    bot[0][c] = wave_up(e0, up0);
                    bot[1][c] = wave_up(e1, wave_read(e0, WAVE - 1));
                    top[0][c] = first ? t0 : up0;
                    top[1][c] = lane == kl ? e1 : up1;
                }
            }
        }
#pragma unroll
        for (int b = 0; b < RB; ++b)
#pragma unroll
            for (int u = 0; u < SETS; ++u) cur[b][u] = nxt[b][u];
    }
#pragma unroll
    for (int u = 0; u < SETS; ++u)
#pragma unroll
        for (int c = 0; c < C; ++c)
            if (c < ncol) {
                if (rt[u] >= 0) Ct[(size_t)rt[u] * ldc + c0 + c] = top[u][c];
                if (rb[u] >= 0) Ct[(size_t)rb[u] * ldc + c0 + c] = bot[u][c];
            }
}

// A recorded sweep applied to ncol columns of Ct: each wave takes runs of C
// columns.  Up to 64 pairs a lane holds one position, above that two.  C is
// the wave's share ncol / 8 rounded up to a compiled size, so that one run covers
// it (ncol <= 128) or two even ones do (9 up to n = 144, 12 above; 2 x 16 columns
// of two positions would not fit the registers).
__device__ inline void ring_vectors(glbf* Ct, int ldc, int n, int ncol, const glbf* rot) {
    const int w = threadIdx.x / WAVE;
    const int share = (ncol + NWAVE - 1) / NWAVE;
#define XTB_RV(S, C)                                        \
    for (int c0 = w * (C); c0 < ncol; c0 += NWAVE * (C))    \
        ring_vectors_t<S, C>(Ct, ldc, n, rot, c0, ncol - c0)
    if (ring_pairs(n) <= WAVE) {
        if (share <= 4) { XTB_RV(1, 4); }
        else if (share <= 8) { XTB_RV(1, 8); }
        else if (share <= 12) { XTB_RV(1, 12); }
        else { XTB_RV(1, 16); }
    } else {
        if (share <= 18) { XTB_RV(2, 9); }
        else { XTB_RV(2, 12); }
    }
#undef XTB_RV
}

// Smallest tolerance of a Jacobi eigensolve, whatever is asked for: a pivot is
// rotated from 1e-3 of it on, so that the sum of squares under the rotation's
// root stays a normal number.
constexpr double JACOBI_TOL_MIN = 1e-140;

// 1 / x and 1 / sqrt(x) for normal positive x: the hardware estimates with
// Newton steps to full precision (the rotations need no correctly rounded
// division, whose scaling and fix-up steps double the dependent chain)
__device__ inline double fast_rcp(double x) {
    double y = __builtin_amdgcn_rcp(x);
    y = fma(fma(-x, y, 1.0), y, y);
    return fma(fma(-x, y, 1.0), y, y);
}
__device__ inline double fast_rsq(double x) {
    double y = __builtin_amdgcn_rsq(x);
    const double h = 0.5 * x;
    y = fma(fma(-h * y, y, 0.5), y, y);
    return fma(fma(-h * y, y, 0.5), y, y);
}

// 2 x 2 block of the pairs P < R in round 0, the t-th of run d (rows P = d and
// K - 2 - d of the strict triangle joined into runs of K): its elements (p, a),
// (p, b), (q, a), (q, b) lie at D[row + col], and col moves on by one a round,
// around the ring of m.  With one pair only (K = 1) there is no block; the
// answer is then a place inside D that is read and not written.
struct RingBlock {
    int P, R;
    int row[4], col[4];
};
__host__ __device__ constexpr RingBlock ring_block(int K, int W, int d, int t) {
    const int m = 2 * K - 1, E = K * W;
    const bool lo = t < K - 1 - d;
    const int P = lo ? d : (K > 1 ? K - 2 - d : 0), R = lo ? d + 1 + t : t;
    const int p = P, q = P > 0 ? m - P : 0, a = R, b = R > 0 ? m - R : 0;
    const int dm = R - P, dp = R + P;
    const bool fold = dp >= K;
    const int row = (fold ? m - dp : dp) * W;
    return {P, R, {P == 0 ? E : dm * W, P == 0 ? E : row, row, dm * W},
            {P == 0 ? a : p, P == 0 ? b : (fold ? p : b), fold ? a : q, b}};
}

// The rounds of one sweep on D, every thread holding NB of the K (K - 1) / 2
// 2 x 2 blocks P < R.  A block's four addresses and the rounds in which they
// wrap around the ring stay in registers.
template <int NB>
__device__ __noinline__ void ring_rounds(ldsf* D, int n, int W, glbf* rot, ldsf* cs, double skip, int mode, int cb_lo,
                                         int cb_hi) {
    const int K = ring_pairs(n), m = 2 * K - 1, E = K * W;
    const Ring G{D, n, m, K, W};
    const bool even = n % 2 == 0;
    const int nblk = K * (K - 1) / 2;
    const uint32_t inv = (1u << 22) / (uint32_t)K + 1u;  // e / K = e inv >> 22 for e K < 2^22
    ldsf* ad[NB][4];
    ldsf *cp[NB], *cr[NB];
    uint32_t rw[NB];  // byte u: the round after which address u wraps
#pragma unroll
    for (int g = 0; g < NB; ++g) {
        const int e0 = threadIdx.x + g * NT, e = e0 < nblk ? e0 : (nblk > 0 ? nblk - 1 : 0);
        const int d = (int)(((uint32_t)e * inv) >> 22);
        const RingBlock x = ring_block(K, W, d, e - d * K);
        rw[g] = 0;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            ad[g][u] = D + x.row[u] + x.col[u];
            rw[g] |= (uint32_t)(m - 1 - x.col[u]) << (8 * u);
        }
        cp[g] = cs + 2 * x.P;
        cr[g] = cs + 2 * x.R;
    }
    for (int r = 0; r < m; ++r) {
        // rotation parameters, and the pairs' own diagonal blocks: with
        // d = a_qq - a_pp, e = 2 a_pq, t = e sgn(d) / (|d| + sqrt(d^2 + e^2))
        if ((int)threadIdx.x < K) {
            const int k = threadIdx.x;
            const int p = k == 0 ? m : G.wrap(r + k), q = G.wrap(r - k);
            double c = 1.0, s = 0.0;
            if (p < n) {
                const int epq = k == 0 ? E + q : (2 * k < K ? 2 * k * W + q : (m - 2 * k) * W + p);
                const int epp = k == 0 ? E + m : p;
                const double apq = D[epq], app = D[epp], aqq = D[q];
                if (fabs(apq) > skip && pair_in_mode(mode, occ_class(p, cb_lo, cb_hi), occ_class(q, cb_lo, cb_hi))) {
                    const double dd = aqq - app, ee = 2.0 * apq;
                    const double h2 = fma(dd, dd, ee * ee);
                    double t = ee * fast_rcp(fma(h2, fast_rsq(h2), fabs(dd)));
                    if (dd < 0.0) t = -t;
                    c = fast_rsq(fma(t, t, 1.0));
                    s = t * c;
                    D[epp] = fma(-t, apq, app);
                    D[q] = fma(t, apq, aqq);
                    D[epq] = 0.0;
                }
            }
            const v2d v = {c, s};
            *(ldsv2*)(cs + 2 * k) = v;
            if (even || k > 0) *(glbv2*)(rot + 2 * ring_slot(n, r, k)) = v;
        }
        __syncthreads();
        // A <- J^T A J on the 2 x 2 blocks, up to three at a time so that
        // their loads are in flight together
        constexpr int GB = NB < 3 ? NB : 3;
#pragma unroll
        for (int g0 = 0; g0 < NB; g0 += GB) {
            v2d vp[GB], vr[GB];
            double x[GB][4];
#pragma unroll
            for (int g = 0; g < GB; ++g)
                if (g0 + g < NB) {
                    vp[g] = *(ldsv2*)cp[g0 + g];
                    vr[g] = *(ldsv2*)cr[g0 + g];
#pragma unroll
                    for (int u = 0; u < 4; ++u)
                        x[g][u] = (u >= 2 || even || cp[g0 + g] != cs) ? *ad[g0 + g][u] : 0.0;
                }
#pragma unroll
            for (int g = 0; g < GB; ++g)
                if (g0 + g < NB) {
                    const double c1 = vp[g].x, s1 = vp[g].y, c2 = vr[g].x, s2 = vr[g].y;
                    const double r00 = c1 * x[g][0] - s1 * x[g][2], r01 = c1 * x[g][1] - s1 * x[g][3];
                    const double r10 = s1 * x[g][0] + c1 * x[g][2], r11 = s1 * x[g][1] + c1 * x[g][3];
                    x[g][0] = r00 * c2 - r01 * s2;
                    x[g][1] = r00 * s2 + r01 * c2;
                    x[g][2] = r10 * c2 - r11 * s2;
                    x[g][3] = r10 * s2 + r11 * c2;
                    if ((int)threadIdx.x + (g0 + g) * NT < nblk && (s1 != 0.0 || s2 != 0.0)) {
#pragma unroll
                        for (int u = 0; u < 4; ++u)
                            if (u >= 2 || even || cp[g0 + g] != cs) *ad[g0 + g][u] = x[g][u];
                    }
#pragma unroll
                    for (int u = 0; u < 4; ++u)
                        ad[g0 + g][u] += ((rw[g0 + g] >> (8 * u)) & 255u) == (uint32_t)r ? 1 - m : 1;
                }
        }
        __syncthreads();
    }
}

// Diagonalises the symmetric matrix A (full, global, upper triangle read) of
// order n <= RING_MAX_N and applies every rotation to the rows of Ct (Ct[k][mu], row
// k = vector k, mu < ncol), i.e. C <- C J; eigenvalues to `ev`.  `D`: LDS of
// ring_doubles(n, W); `cs`: 2 K doubles of LDS (16-byte aligned); `rot`:
// global scratch of n^2 doubles for a sweep's rotations.  Returns the number
// of sweeps, or -1 when max_sweeps were spent without reaching `tol`
// (absolute, largest off-diagonal element of a pair in mode).
__device__ __noinline__ int wg_jacobi(glbf* A, int n, ldsf* D, int W, glbf* Ct, int ldc, int ncol, glbf* rot,
                                      int max_sweeps, double tol, ldsf* cs, ldsf* red, ldsf* ev, int cb_lo, int cb_hi, bool intra) {
    const int mode = cb_lo < 0 ? 0 : (intra ? 2 : 1);
    n = __builtin_amdgcn_readfirstlane(n);
    W = __builtin_amdgcn_readfirstlane(W);
    const int K = ring_pairs(n), m = 2 * K - 1;
    const Ring G{D, n, m, K, W};
    const int w = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
    for (int i = w; i < n; i += NWAVE)
        for (int j = i + lane; j < n; j += WAVE) D[i == j ? G.diag(i) : G.at(i, j)] = A[(size_t)i * n + j];
    __syncthreads();
    const int per = (K * (K - 1) / 2 + NT - 1) / NT;  // 2 x 2 blocks per thread
    const double skip = 1e-3 * tol;
    int sweep = 0;
    for (;;) {
        // convergence test: largest off-diagonal element
        double off = 0.0;
        for (int i = w; i < n; i += NWAVE) {
            const int ci = occ_class(i, cb_lo, cb_hi);
            for (int j = i + 1 + lane; j < n; j += WAVE)
                if (pair_in_mode(mode, ci, occ_class(j, cb_lo, cb_hi))) off = fmax(off, fabs(D[G.at(i, j)]));
        }
        off = wg_max(off, red);
        if (off <= tol || sweep >= max_sweeps) {
            for (int i = threadIdx.x; i < n; i += NT) ev[i] = D[G.diag(i)];
            __syncthreads();
            return off <= tol ? sweep : -1;
        }
        // the smallest compiled block count that covers the thread's share (1, 2, 3,
        // 5, 7 or 10: the step between them wastes at most a third of a round)
#define XTB_RR(NB) ring_rounds<NB>(D, n, W, rot, cs, skip, mode, cb_lo, cb_hi)
        if (per <= 1) XTB_RR(1);
        else if (per == 2) XTB_RR(2);
        else if (per == 3) XTB_RR(3);
        else if (per <= 5) XTB_RR(5);
        else if (per <= 7) XTB_RR(7);
        else XTB_RR(10);
#undef XTB_RR
        ring_vectors(Ct, ldc, n, ncol, rot);
        __syncthreads();
        ++sweep;
    }
}

// ---------------------------------------------------------------------------
// Block Jacobi for matrices that do not fit in LDS.
//
// Indices are grouped in blocks of JB = 16; a round of the round-robin
// ordering pairs the blocks, and every pair (I, J) defines a subproblem on
// the <= 32 indices of I u J.  One wavefront diagonalises its subproblem in
// LDS with scalar cyclic Jacobi (no workgroup barrier inside), producing an
// orthogonal Q_k.  The workgroup then applies all Q_k of the round to A
// (rows, then columns) and to the vectors Ct, streaming each element once
// per phase and reusing every loaded value 32 times.  Per sweep this moves
// ~3 n^3 bytes instead of the ~32 n^3 of the scalar method.
// ---------------------------------------------------------------------------
constexpr int JB = 16;
constexpr int JS = 2 * JB;               // subproblem dimension
constexpr int JW = 34;                   // row pitch of its ring storage
constexpr int JD = ring_doubles(JS, JW);
constexpr int JWAVE_LDS = JD + JS;       // D, (c, s)
constexpr int NBLOCK_LDS = NWAVE * JWAVE_LDS + 64;  // + flags
// The LDS share of a launch whose largest matrix does not fit: matrices up to
// 161 orbitals among its molecules still take the LDS Jacobi.  Where a large
// molecule's vectors leave less, what its GEMMs and subproblems need will do.
constexpr int NMIXED_LDS = 13052;
constexpr int NMIXED_LDS_MIN = NGEMM_MFMA_LDS > NBLOCK_LDS ? NGEMM_MFMA_LDS : NBLOCK_LDS;
static_assert(NMIXED_LDS_MIN <= NMIXED_LDS, "LDS of the mixed launches");

__device__ inline void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Global index of slot i (0..31) of the subproblem of block pair (I, J):
// slots 0..15 are block I, 16..31 block J; -1 where the index is beyond n
// (partial last block, or the dummy block of an odd block count).
__device__ inline int slot_index(int I, int J, int i, int n) {
    const int g = (i < JB) ? I * JB + i : J * JB + (i - JB);
    return g < n ? g : -1;
}

// lane l of each row of 16 <- lane l - 1 (lane 0 <- first), and <- l + 1 (lane 15 <- last)
__device__ __forceinline__ double row_up(double v, double first) { return dpp64<0x111, 0xf>(first, v); }
__device__ __forceinline__ double row_down(double v, double last) { return dpp64<0x101, 0xf>(last, v); }

// One element of the rows top and bottom of Q^T at position k, rotated, then
// the rows move on around the ring
__device__ __forceinline__ void sub_rotate(double c, double s, int k, double& top, double& bot) {
    const double t = c * top - s * bot, e = s * top + c * bot;
    const double up = row_down(t, e);
    bot = row_up(e, up);
    top = k == 0 ? t : up;
}

// Cyclic Jacobi on a 32 x 32 subproblem by one wavefront, in place on its ring
// storage D (pitch JW; zero rows and columns are never rotated).  The
// rotations Q, D_final = Q^T D_0 Q, go to qg (Q[i][j] at qg[i JS + j]) if any
// was applied; returns 1 then, 0 if D was already diagonal to `tol`.
//
// As in the workgroup's rounds, but all in one wave: every lane computes the
// rotation of position lane % 16 (one LDS trip for its pivots), the lanes hold
// two of the 120 2 x 2 blocks each, and Q stays in registers, 8 columns per
// row of 16 lanes, its rows moving around the ring by row shifts of the lanes.
// A round is bound by that chain.  With n = 296 on the whole GPU a subproblem
// took 22 us so, 4 of them saved by staging with all loads in flight; looking
// up a schedule, packed triangle indices and Q's rows in LDS took 62 us.  (Q's
// update a round late, to fill the rotation's latency, changed nothing; left
// to four waves after the sweep, as on the whole GPU, it comes to 19 us.)
// With LATER, Q is left to the caller (sub_rotate): the rotations of round r go
// to cs + 2 K r (max_sweeps = 1 then).
template <bool LATER>
__device__ __noinline__ int wave_jacobi_sub(ldsf* D, ldsf* cs, glbf* qg, double tol, int max_sweeps, int mode,
                                            unsigned lo_mask, unsigned hi_mask) {
    constexpr int K = JB, m = JS - 1, E = K * JW;
    const int lane = threadIdx.x % WAVE, k = lane % K, g0 = lane / K * 8;
    const Ring G{D, JS, m, K, JW};
    // occupation class of a slot (pairs are selected by mode as in wg_jacobi)
    auto scls = [&](int i) { return (int)((lo_mask >> i) & 1u) + (int)((hi_mask >> i) & 1u); };
    ldsf* ad[2][4];
    ldsf *cp[2], *cr[2];
    uint32_t rw[2];  // byte u: the round after which address u wraps
#pragma unroll
    for (int g = 0; g < 2; ++g) {
        const int e = lane + g * WAVE < K * (K - 1) / 2 ? lane + g * WAVE : K * (K - 1) / 2 - 1;
        const int d = e / K, t = e % K;
        const bool lo = t < K - 1 - d;
        const int P = lo ? d : K - 2 - d, R = lo ? d + 1 + t : t;
        const int q = G.wrap(-P), b = G.wrap(-R);
        const int dm = R - P, dp = R + P;
        const bool fold = dp >= K;
        const int row = (fold ? m - dp : dp) * JW;
        const int i0 = P == 0 ? R : P, i1 = P == 0 ? b : (fold ? P : b), i2 = fold ? R : q;
        ad[g][0] = D + (P == 0 ? E : dm * JW) + i0;
        ad[g][1] = D + (P == 0 ? E : row) + i1;
        ad[g][2] = D + row + i2;
        ad[g][3] = D + dm * JW + b;
        rw[g] = (uint32_t)(m - 1 - i0) | (uint32_t)(m - 1 - i1) << 8 | (uint32_t)(m - 1 - i2) << 16 |
                (uint32_t)(m - 1 - b) << 24;
        cp[g] = cs + 2 * P;
        cr[g] = cs + 2 * R;
    }
    // rows of Q^T at this lane's position: top (k, or the fixed row 31) and
    // bottom (31 - k, or 0), columns g0 .. g0 + 7 of the identity
    const int rt = k == 0 ? m : k, rb = k == 0 ? 0 : m - k;
    double top[8], bot[8];
#pragma unroll
    for (int c = 0; c < 8; ++c) {
        top[c] = rt == g0 + c ? 1.0 : 0.0;
        bot[c] = rb == g0 + c ? 1.0 : 0.0;
    }
    const double skip = 1e-3 * tol;
    int rotated = 0;
    for (int sw = 0; sw < max_sweeps; ++sw) {
        double off = 0.0;
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int d = 1 + 2 * u + (lane >> 5), i = lane & 31;
            if (d < K && i < m && pair_in_mode(mode, scls(i), scls(G.wrap(i + d)))) off = fmax(off, fabs(D[d * JW + i]));
        }
        if (lane < m && pair_in_mode(mode, scls(lane), scls(m))) off = fmax(off, fabs(D[E + lane]));
        off = wave_max(off);
        if (off <= tol) break;
        rotated = 1;
        for (int r = 0; r < m; ++r) {
            const int p = k == 0 ? m : G.wrap(r + k), q = G.wrap(r - k);
            const int epq = k == 0 ? E + q : (2 * k < K ? 2 * k * JW + q : (m - 2 * k) * JW + p);
            const int epp = k == 0 ? E + m : p;
            const double apq = D[epq], app = D[epp], aqq = D[q];
            double c = 1.0, s = 0.0;
            if (fabs(apq) > skip && pair_in_mode(mode, scls(p), scls(q))) {
                const double dd = aqq - app, ee = 2.0 * apq;
                const double h2 = fma(dd, dd, ee * ee);
                double t = ee * fast_rcp(fma(h2, fast_rsq(h2), fabs(dd)));
                if (dd < 0.0) t = -t;
                c = fast_rsq(fma(t, t, 1.0));
                s = t * c;
                if (lane < K) {
                    D[epp] = fma(-t, apq, app);
                    D[q] = fma(t, apq, aqq);
                    D[epq] = 0.0;
                }
            }
            if (lane < K) {
                const v2d v = {c, s};
                *(ldsv2*)(cs + 2 * k + (LATER ? 2 * K * r : 0)) = v;
            }
            wave_sync();
            v2d vp[2], vr[2];
            double x[2][4];
#pragma unroll
            for (int g = 0; g < 2; ++g) {
                vp[g] = *(ldsv2*)(cp[g] + (LATER ? 2 * K * r : 0));
                vr[g] = *(ldsv2*)(cr[g] + (LATER ? 2 * K * r : 0));
#pragma unroll
                for (int u = 0; u < 4; ++u) x[g][u] = *ad[g][u];
            }
            if (!LATER) {
#pragma unroll
                for (int y = 0; y < 8; ++y) sub_rotate(c, s, k, top[y], bot[y]);
            }
#pragma unroll
            for (int g = 0; g < 2; ++g) {
                const double c1 = vp[g].x, s1 = vp[g].y, c2 = vr[g].x, s2 = vr[g].y;
                const double r00 = c1 * x[g][0] - s1 * x[g][2], r01 = c1 * x[g][1] - s1 * x[g][3];
                const double r10 = s1 * x[g][0] + c1 * x[g][2], r11 = s1 * x[g][1] + c1 * x[g][3];
                if ((g == 0 || lane + g * WAVE < K * (K - 1) / 2) && (s1 != 0.0 || s2 != 0.0)) {
                    *ad[g][0] = r00 * c2 - r01 * s2;
                    *ad[g][1] = r00 * s2 + r01 * c2;
                    *ad[g][2] = r10 * c2 - r11 * s2;
                    *ad[g][3] = r10 * s2 + r11 * c2;
                }
#pragma unroll
                for (int u = 0; u < 4; ++u) ad[g][u] += ((rw[g] >> (8 * u)) & 255u) == (uint32_t)r ? 1 - m : 1;
            }
            wave_sync();
        }
    }
    if (!LATER && rotated) {
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            qg[(g0 + c) * JS + rt] = top[c];
            qg[(g0 + c) * JS + rb] = bot[c];
        }
    }
    return rotated;
}

// The subproblem of block pair (I, J) of A (full, global, upper triangle
// read): staged into D (slots beyond n zero), and its diagonalised form
// written back (every element).
// By NW waves; with several the caller has a barrier after (before) it.
template <int NW>
__device__ inline void sub_stage(const glbf* A, int n, int I, int J, ldsf* D) {
    const int t = threadIdx.x % (WAVE * NW), j = t % JS, i0 = t / JS;
    constexpr int U = JS / (2 * NW);
    const Ring G{D, JS, JS - 1, JB, JW};
    const int gj = slot_index(I, J, j, n);
    // all loads in flight (clamped, without branches), then all stores
    double v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int gi = slot_index(I, J, i0 + 2 * NW * u, n);
        const int a = gi < 0 ? 0 : gi, b = gj < 0 ? 0 : gj;
        v[u] = A[(uint32_t)(a < b ? a : b) * (uint32_t)n + (uint32_t)(a < b ? b : a)];
        if (gi < 0 || gj < 0) v[u] = 0.0;
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int i = i0 + 2 * NW * u;
        if (i <= j) D[i == j ? G.diag(i) : G.at(i, j)] = v[u];
    }
    wave_sync();
}
template <int NW>
__device__ inline void sub_unstage(glbf* A, int n, int I, int J, ldsf* D) {
    const int t = threadIdx.x % (WAVE * NW), j = t % JS, i0 = t / JS;
    constexpr int U = JS / (2 * NW);
    const Ring G{D, JS, JS - 1, JB, JW};
    const int gj = slot_index(I, J, j, n);
    double v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int i = i0 + 2 * NW * u;
        v[u] = D[i == j ? G.diag(i) : G.at(i, j)];
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int gi = slot_index(I, J, i0 + 2 * NW * u, n);
        if (gi >= 0 && gj >= 0) A[(uint32_t)gi * (uint32_t)n + (uint32_t)gj] = v[u];
    }
}

// Two-sided tile update on matrix cores (one wavefront):
// A[P_k, P_l] <- Q_k^T A[P_k, P_l] Q_l, written to both triangles.
// A is symmetric before the round, so the tile is read as A[P_l, P_k]
// (row segments, coalesced).  Y = A_kl Q_l stays in registers and feeds the
// second product as its B operand (element r = k-step r).
__device__ __noinline__ void tile_update(glbf* A, int n, const glbf* Qk, const glbf* Ql,
                                         int Ik, int Jk, int Il, int Jl, int idk, int idl) {
    const int lane = threadIdx.x % WAVE, li = lane % 16, lg = lane / 16;
    int gk[2], gl_[2];
#pragma unroll
    for (int b = 0; b < 2; ++b) {
        gk[b] = slot_index(Ik, Jk, b * 16 + li, n);
        gl_[b] = slot_index(Il, Jl, b * 16 + li, n);
    }
    v4d y[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) y[i][j] = v4zero();
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) {
            const int kp = kb * 16 + lg + 4 * kk;
            const int g = slot_index(Il, Jl, kp, n);
            double a[2], bq[2];
#pragma unroll
            for (int bm = 0; bm < 2; ++bm)
                a[bm] = (g >= 0 && gk[bm] >= 0) ? A[(size_t)g * n + gk[bm]] : 0.0;
#pragma unroll
            for (int bn = 0; bn < 2; ++bn)
                bq[bn] = idl ? ((kp == bn * 16 + li) ? 1.0 : 0.0) : Ql[kp * JS + bn * 16 + li];
#pragma unroll
            for (int bm = 0; bm < 2; ++bm)
#pragma unroll
                for (int bn = 0; bn < 2; ++bn) y[bm][bn] = mfma16(a[bm], bq[bn], y[bm][bn]);
        }
    v4d z[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) z[i][j] = v4zero();
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int k = kb * 16 + lg + 4 * r;
            double a[2];
#pragma unroll
            for (int bm = 0; bm < 2; ++bm)
                a[bm] = idk ? ((k == bm * 16 + li) ? 1.0 : 0.0) : Qk[k * JS + bm * 16 + li];
#pragma unroll
            for (int bm = 0; bm < 2; ++bm)
#pragma unroll
                for (int bn = 0; bn < 2; ++bn) z[bm][bn] = mfma16(a[bm], y[kb][bn][r], z[bm][bn]);
        }
#pragma unroll
    for (int bm = 0; bm < 2; ++bm)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int gi = slot_index(Ik, Jk, bm * 16 + lg + 4 * r, n);
            if (gi < 0) continue;
#pragma unroll
            for (int bn = 0; bn < 2; ++bn) {
                const int gj = gl_[bn];
                if (gj < 0) continue;
                A[(size_t)gi * n + gj] = z[bm][bn][r];
                A[(size_t)gj * n + gi] = z[bm][bn][r];
            }
        }
}

// Vector update on matrix cores (one wavefront): rows P_k of the row-major
// matrix X (stride ld), columns c0..c0+63:  X[P_k, c] <- Q_k^T X[P_k, c].
__device__ __noinline__ void rows_update(glbf* X, int n, size_t ld, int ncol, const glbf* Qk,
                                         int Ik, int Jk, int c0) {
    const int lane = threadIdx.x % WAVE, li = lane % 16, lg = lane / 16;
    v4d acc[2][4];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = v4zero();
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) {
            const int kp = kb * 16 + lg + 4 * kk;
            const int g = slot_index(Ik, Jk, kp, n);
            double a[2], b[4];
#pragma unroll
            for (int bm = 0; bm < 2; ++bm) a[bm] = Qk[kp * JS + bm * 16 + li];
#pragma unroll
            for (int bn = 0; bn < 4; ++bn) {
                const int c = c0 + bn * 16 + li;
                b[bn] = (g >= 0 && c < ncol) ? X[(size_t)g * ld + c] : 0.0;
            }
#pragma unroll
            for (int bm = 0; bm < 2; ++bm)
#pragma unroll
                for (int bn = 0; bn < 4; ++bn) acc[bm][bn] = mfma16(a[bm], b[bn], acc[bm][bn]);
        }
#pragma unroll
    for (int bm = 0; bm < 2; ++bm)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int g = slot_index(Ik, Jk, bm * 16 + lg + 4 * r, n);
            if (g < 0) continue;
#pragma unroll
            for (int bn = 0; bn < 4; ++bn) {
                const int c = c0 + bn * 16 + li;
                if (c < ncol) X[(size_t)g * ld + c] = acc[bm][bn][r];
            }
        }
}

// A: full symmetric n x n (row-major, global); Ct: vectors (rows, global);
// Qbuf: global scratch >= (nblocks/2 + 1) * JS * JS doubles.  Returns sweeps
// or -1 when max_sweeps were spent.
template <class CAcc>
__device__ __noinline__ int wg_block_jacobi(glbf* A, int n, CAcc Ct, int ncol, int pad0, int pad1, glbf* Qbuf,
                                            int max_sweeps, double tol,
                                            ldsf* lds, ldsf* red, ldsf* tacc, int inner,
                                            int cb_lo, int cb_hi, bool intra) {
    const int mode = cb_lo < 0 ? 0 : (intra ? 2 : 1);
    // mode 2 skips pairs of pure blocks of different classes; every block then
    // still meets a block of its own class if each class spans two blocks
    const bool skip_cross = mode == 2 && cb_lo >= 2 * JB && n - cb_hi >= 2 * JB;
    const int w = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
    ldsf* D = lds + w * JWAVE_LDS;
    ldsf* cs = D + JD;
    const int nb = (n + JB - 1) / JB;
    const int nb2 = nb + (nb & 1);
    const int npair = nb2 / 2;
    const int ntile = npair * (npair - 1) / 2;
    const int nch = (ncol + WAVE - 1) / WAVE;
    // pairs of blocks that hold nothing but uncoupled indices (pad0 .. pad1,
    // or past the end)
    auto idle = [&](int I, int J) {
        auto in = [&](int b) { return b * JB >= n || (b * JB >= pad0 && (b * JB + JB < n ? b * JB + JB : n) <= pad1); };
        return in(I) && in(J);
    };
    ldsi* ident = reinterpret_cast<ldsi*>(lds + NWAVE * JWAVE_LDS);  // per pair: Q == I
    // symmetrise from the upper triangle
    for (int i = w; i < n; i += NWAVE)
        for (int j = lane; j < i; j += WAVE) A[(size_t)i * n + j] = A[(size_t)j * n + i];
    __syncthreads();
    int sweep = 0;
    for (;;) {
        // (four rows per wave: the loads of four rows in flight)
        double off = 0.0;
        for (int i0 = w * 4; i0 < n; i0 += NWAVE * 4) {
            int ii[4], ci[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                ii[u] = i0 + u < n ? i0 + u : n - 1;
                ci[u] = occ_class(ii[u], cb_lo, cb_hi);
            }
            for (int j = i0 + 1 + lane; j < n; j += WAVE) {
                double a[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) a[u] = A[(size_t)ii[u] * n + j];
                const int cj = occ_class(j, cb_lo, cb_hi);
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    if (j > i0 + u && i0 + u < n && pair_in_mode(mode, ci[u], cj)) off = fmax(off, fabs(a[u]));
            }
        }
        off = wg_max(off, red);
        if (off <= tol) return sweep;
        if (sweep >= max_sweeps) return -1;
        for (int r = 0; r < nb2 - 1; ++r) {
            const double t0 = (double)wall_clock64() * 0.01;
            // 1. subproblems, one wavefront each (invalid slots stay decoupled:
            //    zero rows/columns are never rotated)
            for (int k = w; k < npair; k += NWAVE) {
                int I, J;
                rr_pair(r, k, nb2, I, J);
                if (idle(I, J)) {
                    if (lane == 0) ident[k] = 1;
                    continue;
                }
                unsigned lo_mask = 0u, hi_mask = 0u;
                if (mode != 0) {
                    // slot classes (slots 0..15 block I, 16..31 block J)
                    const int g = slot_index(I, J, lane % JS, n);
                    const unsigned vm = (unsigned)__ballot(lane < JS && g >= 0);
                    lo_mask = (unsigned)__ballot(lane < JS && g >= 0 && g < cb_lo);
                    hi_mask = (unsigned)__ballot(lane < JS && g >= 0 && g < cb_hi);
                    bool skip;
                    if (mode == 1) {
                        // a pair whose valid slots share one class has nothing to decouple
                        skip = (lo_mask == 0u || lo_mask == vm) && (hi_mask == 0u || hi_mask == vm);
                    } else {
                        // two non-empty pure blocks of different classes: no
                        // same-class pair spans them
                        const unsigned vI = vm & 0xFFFFu, vJ = vm >> 16;
                        const unsigned lI = lo_mask & 0xFFFFu, lJ = lo_mask >> 16;
                        const unsigned hI = hi_mask & 0xFFFFu, hJ = hi_mask >> 16;
                        const bool pI = (lI == 0u || lI == vI) && (hI == 0u || hI == vI);
                        const bool pJ = (lJ == 0u || lJ == vJ) && (hJ == 0u || hJ == vJ);
                        const int cI = (lI != 0u) + (hI != 0u), cJ = (lJ != 0u) + (hJ != 0u);
                        skip = skip_cross && vI != 0u && vJ != 0u && pI && pJ && cI != cJ;
                    }
                    if (skip) {
                        if (lane == 0) ident[k] = 1;
                        continue;
                    }
                }
                sub_stage<1>(A, n, I, J, D);
                const int rot =
                    wave_jacobi_sub<false>(D, cs, Qbuf + (size_t)k * JS * JS, tol, inner, mode, lo_mask, hi_mask);
                if (lane == 0) ident[k] = rot ? 0 : 1;
                if (rot) sub_unstage<1>(A, n, I, J, D);
                wave_sync();
            }
            __syncthreads();
            const double t1 = (double)wall_clock64() * 0.01;
            // 2. off-diagonal tiles of A and the vectors, matrix cores
            const int nitem = ntile + npair * nch;
            for (int it = w; it < nitem; it += NWAVE) {
                if (it < ntile) {
                    // tile index -> (k, l), k < l
                    int k = 0, rem = it;
                    while (rem >= npair - 1 - k) { rem -= npair - 1 - k; ++k; }
                    const int l = k + 1 + rem;
                    if (ident[k] && ident[l]) continue;  // both rotations are I
                    int Ik, Jk, Il, Jl;
                    rr_pair(r, k, nb2, Ik, Jk);
                    rr_pair(r, l, nb2, Il, Jl);
                    if (idle(Ik, Jk) || idle(Il, Jl)) continue;  // a tile of zeros
                    tile_update(A, n, Qbuf + (size_t)k * JS * JS, Qbuf + (size_t)l * JS * JS, Ik, Jk,
                                Il, Jl, ident[k], ident[l]);
                } else {
                    const int v = it - ntile;
                    const int k = v / nch, ch = v % nch;
                    if (ident[k]) continue;
                    int Ik, Jk;
                    rr_pair(r, k, nb2, Ik, Jk);
                    rows_update(Ct.a, n, (size_t)Ct.ld, ncol, Qbuf + (size_t)k * JS * JS, Ik, Jk,
                                ch * WAVE);
                }
            }
            __syncthreads();
            const double t2 = (double)wall_clock64() * 0.01;
            if (threadIdx.x == 0) {
                tacc[4] += t1 - t0;
                tacc[5] += t2 - t1;
            }
        }
        ++sweep;
    }
}

struct RowsGlobal {
    glbf* a;
    int ld;
    __device__ inline glbf& at(int k, int mu) const { return a[(size_t)k * ld + mu]; }
};

// Ascending sort of the n <= 2 NT keys src[0..n): key[r] = src[idx[r]], in LDS
// of n entries each.  src may be key itself.
//
// Each thread counts the keys below its own (equal ones in index order, NaN
// as +inf): n LDS broadcasts and four barriers, ~1 us at n = 128 and 3 us at
// 300, where a bitonic network, a barrier per stage (28 and 45), took 3 and 5
// us.
template <class Src>
__device__ inline void wg_sort(Src src, ldsf* key, ldsi* idx, int n) {
    constexpr int Q = 2;
    double v[Q], e[Q];
    int rank[Q];
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        const int j = threadIdx.x + NT * q;
        v[q] = j < n ? src[j] : 0.0;
        e[q] = v[q] == v[q] ? v[q] : INFINITY;
        rank[q] = 0;
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        const int j = threadIdx.x + NT * q;
        if (j < n) key[j] = e[q];
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        const int j = threadIdx.x + NT * q, b0 = j - j % WAVE, b1 = b0 + WAVE < n ? b0 + WAVE : n;
        if (b0 >= n) continue;
#pragma unroll 8
        for (int i = 0; i < b0; ++i) rank[q] += key[i] <= e[q];
#pragma unroll 8
        for (int i = b0; i < b1; ++i) rank[q] += i < j ? key[i] <= e[q] : key[i] < e[q];
#pragma unroll 8
        for (int i = b1; i < n; ++i) rank[q] += key[i] < e[q];
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        const int j = threadIdx.x + NT * q;
        if (j < n) {
            key[rank[q]] = v[q];
            idx[rank[q]] = j;
        }
    }
    __syncthreads();
}

}  // namespace xtb
