// Whole-GPU SCF for one large molecule (thousands of orbitals) on gfx950.
//
// The persistent per-molecule kernel (scf.hip) gives one CU to each molecule,
// the right shape for streams of molecules and the wrong one for a single
// system of n ~ 5000 orbitals.  Here every stage of the same SCF is a grid
// kernel that spreads over all CUs, and the SCF driver runs on the host,
// stream ordered; a few control scalars come back once or twice per step
// through host memory that the kernels write (read_ctl):
//
//   setup   Cholesky orthogonaliser X = L^-1, S = L L^T (or Loewdin's S^-1/2
//           by the coupled Newton-Schulz iteration), on matrix-core GEMMs;
//           the orbitals start as the rows of X
//   step    Fock build F = H0 - 1/2 S o (v_i + v_j)  (scf/base.py:817-859)
//           -> gapped closed shell: perturbative occupied-virtual rotation
//              of the previous step's orbitals (GEMMs), as in scf_kernel.h
//           -> otherwise A = C F C^T and parallel-ordered block Jacobi: one
//              launch solves the 32 x 32 subproblems of a round (a workgroup
//              of four waves each), one applies their rotations to A and to
//              the orbitals on matrix cores
//           -> sort, Fermi smearing (filling.py:201-366), density
//              P = C^T diag(f) C, Mulliken charges, ES2/ES3 potential,
//              Anderson mixing (mixer/anderson.py:163-317), all on device
//   final   the exact step, energies, -TS and the energy-weighted density W
//           for the analytic gradient (types/analytical.py:186-190)
//
// Upstream runs the same SCF (src/dxtb/_src/scf/unrolling/default.py:71-140)
// with LAPACK's eigh per step (scf/unrolling/base.py:142-175).
#include <chrono>
#include <mutex>
#include <vector>

#include "scf_core.h"

namespace xtb {
namespace big {

// control values the host reads back (slots of the `ctl` array)
enum {
    C_EFA = 0, C_EFB, C_FOK, C_KOCC, C_PERM, C_GAPA, C_GAPB, C_DMAX,
    C_AOV, C_KMAX, C_DMIN, C_XF, C_OFF, C_ERR, C_GERSH, C_CONV, C_RESID, C_FSOFT, C_BRANK, C_BDX,
    C_NCTL = 24
};

// The control values' copy in host memory that the device writes (pinned,
// coherent): kernels that end a stretch of work post them, `seq` last.
struct Box {
    double v[C_NCTL];
    unsigned long long seq;
};
struct Post {
    Box* box;  // null: nothing to post
    unsigned long long seq;
};

// by (at least) the first wave, which has written its values to ctl
__device__ inline void post(const double* ctl, const Post& p) {
    if (!p.box || threadIdx.x >= WAVE) return;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
    if (threadIdx.x < C_NCTL)
        __hip_atomic_store(&p.box->v[threadIdx.x], ctl[threadIdx.x], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __threadfence_system();
    if (threadIdx.x == 0) __hip_atomic_store(&p.box->seq, p.seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// ---------------------------------------------------------------------------
// Grid GEMM, C = alpha op(A) op(B) + beta C: wave tiles of 16 FM x 16 FN whose
// MFMA operands are loaded straight from memory into registers, several k
// chunks ahead, with no LDS stage and no barrier in the loop.  (An FP64 MFMA
// takes 64 cycles here, so the 128-byte row segments that a fragment of a
// chunk needs arrive well below the caches' rate, and the vector unit, which
// also runs the FP64 MFMAs, is left alone: a scalar base, 32-bit lane offsets.)
//
// With SPLIT the four waves of a workgroup share one tile and take a quarter
// of k each; their partial sums meet in LDS once, wave w adding and writing
// element w of every fragment.  That shortens the chain of loads that bounds
// small products and gives four times the tiles; without it they are 2 x 2
// tiles with all of k each (large products, where operand re-use counts).
//
// Workgroup b runs on XCD b mod 8; each XCD takes a contiguous run of tiles,
// four tile rows at a time column by column, so that those that run together
// share row and column panels in its L2.  `sym` (M == N, a symmetric product,
// beta unused): tiles on and above the diagonal only, written to both
// triangles.
//
// us at n, k = n / 2 (k n k / n n n / symmetric n n k): n = 148: 3.1 / 3.5 /
// 4, 296: 3.5 / 5.5 / 3.6, 528: 6.2 / 16 / 6.7, 1500: 37 / 130 / 50, 4800: 825
// / 3460 / 840 (65 TFLOP/s); 64- and 128-wide LDS tiles of 8 waves took 7.2 /
// 10.5 / 14.7, 10.6 / 18.7 / 17.9, 17 / 31 / 25, 126 / 245 / 134, 1250 / 4610
// / 1260.
// ---------------------------------------------------------------------------
// One operand of a wave tile.  KM: stored with k contiguous; otherwise by
// rows of k.  A lane's k of a chunk: lg KS + j, j < KS.  Rows past the end
// repeat the last one (their results are not stored).
template <bool KM, int F, int KS>
struct WaveSide {
    const glbc* p;
    uint32_t ldb;
    uint32_t off[F];
    __device__ __forceinline__ void init(const double* X, int ld, int m0, int M, int li, int lg) {
        p = (const glbc*)to_glb(X);
        ldb = (uint32_t)ld * 8u;
#pragma unroll
        for (int f = 0; f < F; ++f) {
            int m = m0 + 16 * f + li;
            m = m < M ? m : M - 1;
            off[f] = KM ? (uint32_t)m * ldb + (uint32_t)(lg * KS * 8) : (uint32_t)(lg * KS) * ldb + (uint32_t)m * 8u;
        }
    }
    __device__ __forceinline__ void fetch(double (&x)[F][KS]) {
#pragma unroll
        for (int f = 0; f < F; ++f) {
            if constexpr (KM) {
#pragma unroll
                for (int j = 0; j < KS; j += 2) {
                    const v2d8 v = *(const glbv2*)(p + off[f] + j * 8);
                    x[f][j] = v.x;
                    x[f][j + 1] = v.y;
                }
            } else {
#pragma unroll
                for (int j = 0; j < KS; ++j) x[f][j] = *(const glbf*)((p + (size_t)j * ldb) + off[f]);
            }
        }
        p += KM ? (size_t)(4 * KS * 8) : (size_t)(4 * KS) * ldb;
    }
    // the last chunk's first rem k; the others are read at the last valid one
    // and count as zero
    __device__ __forceinline__ void fetch_tail(double (&x)[F][KS], int rem, int lg) const {
        const uint32_t unit = KM ? 8u : ldb;
#pragma unroll
        for (int j = 0; j < KS; ++j) {
            const int k = lg * KS + j, kk = k < rem ? k : rem - 1;
#pragma unroll
            for (int f = 0; f < F; ++f) {
                // off holds lg KS units
                const double v = *(const glbf*)(p + (off[f] + (uint32_t)kk * unit - (uint32_t)(lg * KS) * unit));
                x[f][j] = k < rem ? v : 0.0;
            }
        }
    }
};

// EPI: C = alpha op(A) op(B) + s1 E1 + s2 E2, columns from `half` on
// + s3 E1 + s4 E2 of column - half (E1, E2: leading dimension lde).
struct Epi {
    const double *E1, *E2;
    int lde, half;
    double s1, s2, s3, s4;
};

template <bool TA, bool TB, bool EPI, bool SPLIT, int FM, int FN, int KS, int NB>
__global__ void __launch_bounds__(256, 2) k_gemm(int M, int N, int K, double alpha, const double* A, int lda,
                                                 const double* B, int ldb, double beta, double* C, int ldc,
                                                 int sym, int ntiles, const double* Kd, Epi ep) {
    constexpr int KC = 4 * KS, TM = (SPLIT ? 16 : 32) * FM, TN = (SPLIT ? 16 : 32) * FN;
    __shared__ double part[SPLIT ? 3 * FM * FN * 256 : 1];
    const int per = gridDim.x / 8;  // the grid is a multiple of 8
    const int idx = (blockIdx.x % 8) * per + blockIdx.x / 8;
    if (idx >= ntiles) return;
    if (Kd) K = uniform((int)*Kd);  // k from device memory
    const int tm = (M + TM - 1) / TM, tn = (N + TN - 1) / TN;
    int ti, tj;
    if (sym) {
        int r = 0, q = idx;
        while (q >= tn - r) {
            q -= tn - r;
            ++r;
        }
        ti = r;
        tj = r + q;
    } else {
        constexpr int G = 4;
        const int g = idx / (G * tn), r0 = g * G, h = tm - r0 < G ? tm - r0 : G;
        const int q = idx - g * G * tn;
        tj = q / h;
        ti = r0 + (q - tj * h);
    }
    const int lane = threadIdx.x % WAVE, li = lane % 16, lg = lane / 16;
    const int w = uniform((int)threadIdx.x / WAVE);
    int m0 = ti * TM, n0 = tj * TN;
    if (SPLIT) {
        // this wave's quarter of k, in whole chunks
        const int q = ((K + KC - 1) / KC + 3) / 4 * KC;
        const int kb = w * q < K ? w * q : K, ke = kb + q < K ? kb + q : K;
        A += TA ? (size_t)kb * lda : (size_t)kb;
        B += TB ? (size_t)kb : (size_t)kb * ldb;
        K = ke - kb;
    } else {
        m0 += (w / 2) * 16 * FM;
        n0 += (w % 2) * 16 * FN;
        if (m0 >= M || n0 >= N) return;
    }
    WaveSide<!TA, FM, KS> a;
    WaveSide<TB, FN, KS> b;
    a.init(A, lda, m0, M, li, lg);
    b.init(B, ldb, n0, N, li, lg);
    v4d acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = v4zero();
    double xa[NB][FM][KS], xb[NB][FN][KS];
    auto get = [&](int u) {
        a.fetch(xa[u]);
        b.fetch(xb[u]);
        __builtin_amdgcn_sched_barrier(0);
    };
    auto multiply = [&](int u) {
#pragma unroll
        for (int k = 0; k < KS; ++k)
#pragma unroll
            for (int i = 0; i < FM; ++i)
#pragma unroll
                for (int j = 0; j < FN; ++j) acc[i][j] = mfma16(xa[u][i][k], xb[u][j][k], acc[i][j]);
        __builtin_amdgcn_sched_barrier(0);
    };
    const int nfull = K / KC, rem = K - nfull * KC;
    int c = 0;
    if (nfull >= NB) {
        // NB buffers in a ring, each chunk loaded NB - 1 chunks ahead
#pragma unroll
        for (int u = 0; u < NB - 1; ++u) get(u);
        int left = nfull - (NB - 1);  // not loaded yet
        for (; left >= NB; left -= NB) {
#pragma unroll
            for (int u = 0; u < NB; ++u) {
                get((u + NB - 1) % NB);
                multiply(u);
            }
        }
#pragma unroll
        for (int u = 0; u < NB - 1; ++u) {
            if (u < left) get((u + NB - 1) % NB);
            multiply(u);
        }
#pragma unroll
        for (int u = 0; u < NB - 1; ++u)
            if (u < left) multiply((u + NB - 1) % NB);
        c = nfull;
    }
    for (; c < nfull; ++c) {
        get(0);
        multiply(0);
    }
    if (rem) {
        a.fetch_tail(xa[0], rem, lg);
        b.fetch_tail(xb[0], rem, lg);
        multiply(0);
    }
    auto put = [&](int i, int j, int r, double v) {
        const int gm = m0 + 16 * i + lg + 4 * r, gn = n0 + 16 * j + li;
        if (gm >= M || gn >= N) return;
        const size_t e = (size_t)gm * ldc + gn;
        if (EPI) {
            const bool hi = gn >= ep.half;
            const size_t x = (size_t)gm * ep.lde + (hi ? gn - ep.half : gn);
            C[e] = fma(alpha, v, fma(hi ? ep.s3 : ep.s1, ep.E1[x], (hi ? ep.s4 : ep.s2) * ep.E2[x]));
        } else if (sym) {
            C[e] = alpha * v;
            if (ti != tj) C[(size_t)gn * ldc + gm] = alpha * v;
        } else C[e] = beta == 0.0 ? alpha * v : fma(alpha, v, beta * C[e]);
    };
    if constexpr (SPLIT) {
        // element r of a fragment is summed by wave r, in wave order; wave s != r
        // leaves its part in slot s - r - 1 (mod 4)
        auto slot = [&](int f, int r, int s) { return ((((s - r - 1) & 3) * FM * FN + f) * 4 + r) * WAVE + lane; };
#pragma unroll
        for (int f = 0; f < FM * FN; ++f)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (w != r) part[slot(f, r, w)] = acc[f / FN][f % FN][r];
        __syncthreads();
#pragma unroll
        for (int f = 0; f < FM * FN; ++f)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (w == r) {
                    double v = 0.0;
#pragma unroll
                    for (int s = 0; s < 4; ++s) v += s == r ? acc[f / FN][f % FN][r] : part[slot(f, r, s)];
                    put(f / FN, f % FN, r, v);
                }
    } else {
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) put(i, j, r, acc[i][j][r]);
    }
}

// ---------------------------------------------------------------------------
// Elementwise and row kernels.  Row kernels: one wave per row, 8 rows per
// 512-thread workgroup.
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256) k_fock(int n, const double* H0, const double* S, const double* v,
                                              double* F) {
    const int r = blockIdx.y;
    const double vr = v[r];
    for (int c = blockIdx.x * 256 + threadIdx.x; c < n; c += gridDim.x * 256) {
        const size_t e = (size_t)r * n + c;
        F[e] = H0[e] - 0.5 * S[e] * (vr + v[c]);
    }
}

// out[i] = sum_c X[i][c] Y[i][c], i < rows; out[i] = tail[i] for the rest up
// to n
__global__ void __launch_bounds__(NT) k_rowdot(int rows, int n, const double* X, const double* Y, const double* tail,
                                               double* out) {
    const int i = blockIdx.x * NWAVE + threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
    if (i >= n) return;
    if (i >= rows) {
        if (lane == 0) out[i] = tail[i];
        return;
    }
    double d = 0.0;
    for (int c = lane; c < n; c += WAVE) d = fma(X[(size_t)i * n + c], Y[(size_t)i * n + c], d);
    d = wave_sum(d);
    if (lane == 0) out[i] = d;
}

// per-workgroup partials of max |X_ij| over j > i (rows i of this
// workgroup's waves): part[blockIdx.x]
__global__ void __launch_bounds__(NT) k_offmax(int n, const double* A, double* part) {
    __shared__ double red[NWAVE];
    const int w = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
    const int i = blockIdx.x * NWAVE + w;
    double m = 0.0;
    if (i < n)
        for (int j = i + 1 + lane; j < n; j += WAVE) m = fmax(m, fabs(A[(size_t)i * n + j]));
    m = wave_max(m);
    if (lane == 0) red[w] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        double r = red[0];
        for (int k = 1; k < NWAVE; ++k) r = fmax(r, red[k]);
        part[blockIdx.x] = r;
    }
}

// per-workgroup partials of max |d_i| (diagonal of A, or a vector) and of
// the Gershgorin radius max_i sum_j |A_ij| (when A is given)
__global__ void __launch_bounds__(NT) k_rowabs(int n, const double* A, double* part) {
    __shared__ double red[NWAVE];
    const int w = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
    const int i = blockIdx.x * NWAVE + w;
    double s = 0.0;
    if (i < n)
        for (int j = lane; j < n; j += WAVE) s += fabs(A[(size_t)i * n + j]);
    s = wave_sum(s);
    if (lane == 0) red[w] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        double r = red[0];
        for (int k = 1; k < NWAVE; ++k) r = fmax(r, red[k]);
        part[blockIdx.x] = r;
    }
}

// Reduction of per-workgroup partials: ctl[slot] = sum (op 0) or max (op 1) of
// part[b], b < nblk, in a fixed order (deterministic).
__global__ void __launch_bounds__(NT) k_finish(const double* part, int nblk, int op, double* ctl, int slot, Post p) {
    __shared__ double red[NWAVE];
    double a = op == 0 ? 0.0 : -INFINITY;
    for (int b = threadIdx.x; b < nblk; b += NT) a = op == 0 ? a + part[b] : fmax(a, part[b]);
    a = op == 0 ? wg_sum(a, to_lds(red)) : wg_max(a, to_lds(red));
    if (threadIdx.x == 0) ctl[slot] = a;
    post(ctl, p);
}

// What a perturbative step's host decisions need (one workgroup): max |ev|
// over n, and over the partials of k_amplitudes max |A_ia|, max |K_ia|, min
// (e_a - e_i)
__global__ void __launch_bounds__(NT) k_pd_stats(int n, const double* ev, const double* part, int nblk, double* ctl,
                                                 Post p) {
    __shared__ double red[4 * NWAVE];
    double m[4] = {0.0, 0.0, 0.0, -INFINITY};
    for (int i = threadIdx.x; i < n; i += NT) m[0] = fmax(m[0], fabs(ev[i]));
    for (int b = threadIdx.x; b < nblk; b += NT) {
        m[1] = fmax(m[1], part[3 * b]);
        m[2] = fmax(m[2], part[3 * b + 1]);
        m[3] = fmax(m[3], -part[3 * b + 2]);
    }
    wg_max_n<4>(m, to_lds(red));
    if (threadIdx.x == 0) {
        ctl[C_DMAX] = m[0];
        ctl[C_AOV] = m[1];
        ctl[C_KMAX] = m[2];
        ctl[C_DMIN] = -m[3];
    }
    post(ctl, p);
}

// Perturbative amplitudes K_ia <- A_ia / (e_a - e_i) (k x m, row-major);
// partials per workgroup (one wave per row i): max |A_ia|, max |K_ia|,
// min (e_a - e_i)
__global__ void __launch_bounds__(NT) k_amplitudes(int k, int m, double* Kb, const double* ev, double* part) {
    __shared__ double red[3 * NWAVE];
    const int w = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
    const int i = blockIdx.x * NWAVE + w;
    double aov = 0.0, kmax = 0.0, dmin = INFINITY;
    if (i < k) {
        const double ei = ev[i];
        for (int a = lane; a < m; a += WAVE) {
            const double v = Kb[(size_t)i * m + a];
            const double den = ev[k + a] - ei;
            const double amp = v / den;
            aov = fmax(aov, fabs(v));
            dmin = fmin(dmin, den);
            kmax = fmax(kmax, fabs(amp));
            Kb[(size_t)i * m + a] = amp;
        }
    }
    aov = wave_max(aov);
    kmax = wave_max(kmax);
    dmin = -wave_max(-dmin);
    if (lane == 0) {
        red[w] = aov;
        red[NWAVE + w] = kmax;
        red[2 * NWAVE + w] = dmin;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        double a = red[0], b = red[NWAVE], c = red[2 * NWAVE];
        for (int x = 1; x < NWAVE; ++x) {
            a = fmax(a, red[x]);
            b = fmax(b, red[NWAVE + x]);
            c = fmin(c, red[2 * NWAVE + x]);
        }
        part[(size_t)blockIdx.x * 3 + 0] = a;
        part[(size_t)blockIdx.x * 3 + 1] = b;
        part[(size_t)blockIdx.x * 3 + 2] = c;
    }
}

// partials of sum x_e^2 over a contiguous array
__global__ void __launch_bounds__(NT) k_sumsq(size_t len, const double* x, double* part) {
    __shared__ double red[NWAVE];
    double s = 0.0;
    for (size_t e = (size_t)blockIdx.x * NT + threadIdx.x; e < len; e += (size_t)gridDim.x * NT) s = fma(x[e], x[e], s);
    s = wave_sum(s);
    if (threadIdx.x % WAVE == 0) red[threadIdx.x / WAVE] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        double r = 0.0;
        for (int k = 0; k < NWAVE; ++k) r += red[k];
        part[blockIdx.x] = r;
    }
}

// First terms of the two series of a perturbative rotation (k x n):
// R = s1 C + s2 Z and D = s3 C + s4 Z (D may be C itself)
__global__ void __launch_bounds__(256) k_series0(int n, const double* C, const double* Z, double s1, double s2,
                                                 double* R, int ldr, double s3, double s4, double* D, int ldd) {
    const size_t r = blockIdx.y;
    for (int c = blockIdx.x * 256 + threadIdx.x; c < n; c += gridDim.x * 256) {
        const double x = C[r * n + c], z = Z[r * n + c];
        R[r * ldr + c] = s1 * x + s2 * z;
        D[r * ldd + c] = s3 * x + s4 * z;
    }
}

// Y = a X + b Z over `len` contiguous elements (Y may alias X or Z)
__global__ void __launch_bounds__(256) k_axpby(size_t len, double a, const double* X, double b, const double* Z,
                                               double* Y) {
    for (size_t e = (size_t)blockIdx.x * 256 + threadIdx.x; e < len; e += (size_t)gridDim.x * 256)
        Y[e] = a * X[e] + (Z ? b * Z[e] : 0.0);
}

// Newton-Schulz helpers: T <- T + d I; X <- s (X + X^T) / 2 into Y (n x n)
__global__ void __launch_bounds__(256) k_add_diag(int n, double d, double* T) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) T[(size_t)i * n + i] += d;
}

__global__ void __launch_bounds__(256) k_identity(int n, double* T) {
    const int r = blockIdx.y;
    for (int c = blockIdx.x * 256 + threadIdx.x; c < n; c += gridDim.x * 256)
        T[(size_t)r * n + c] = (r == c) ? 1.0 : 0.0;
}

__global__ void __launch_bounds__(256) k_symmetrise(int n, double s, const double* X, double* Y) {
    const int r = blockIdx.y;
    for (int c = blockIdx.x * 256 + threadIdx.x; c < n; c += gridDim.x * 256)
        Y[(size_t)r * n + c] = 0.5 * s * (X[(size_t)r * n + c] + X[(size_t)c * n + r]);
}

// partials of max |T_ij - delta_ij|
__global__ void __launch_bounds__(NT) k_dev_identity(int n, const double* T, double* part) {
    __shared__ double red[NWAVE];
    const int w = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
    const int i = blockIdx.x * NWAVE + w;
    double m = 0.0;
    if (i < n)
        for (int j = lane; j < n; j += WAVE) m = fmax(m, fabs(T[(size_t)i * n + j] - (i == j ? 1.0 : 0.0)));
    m = wave_max(m);
    if (lane == 0) red[w] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        double r = red[0];
        for (int k = 1; k < NWAVE; ++k) r = fmax(r, red[k]);
        part[blockIdx.x] = r;
    }
}

// ---------------------------------------------------------------------------
// Cholesky orthogonaliser X = L^-1, S = L L^T (the per-workgroup version is
// chol_setup in scf_kernel.h), 32-wide panels.  k_chol_diag: one wave factors the
// diagonal block j0 of the lower triangle of L in place and writes its
// inverse to Dg (nb x nb, leading dimension nb); a non-positive pivot sets
// ctl[C_ERR].
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(WAVE) k_chol_diag(double* L, int n, int j0, int nb, double* Dg, double* ctl) {
    const bool ok = chol_block(to_glb(L) + (size_t)j0 * n + j0, n, nb, to_glb(Dg));
    if (!ok && threadIdx.x == 0) ctl[C_ERR] = 1.0;
}

// Y[r][c] = X[r][c] for r < rows, c < cols (leading dimensions ldx, ldy)
__global__ void __launch_bounds__(256) k_copy_block(int rows, int cols, const double* X, int ldx, double* Y,
                                                    int ldy) {
    const int r = blockIdx.y;
    for (int c = blockIdx.x * 256 + threadIdx.x; c < cols; c += gridDim.x * 256)
        Y[(size_t)r * ldy + c] = X[(size_t)r * ldx + c];
}

__global__ void k_post(const double* ctl, Post p) { post(ctl, p); }

__global__ void k_set_slot(double* ctl, int slot, double v) {
    if (threadIdx.x == 0) ctl[slot] = v;
}

// ---------------------------------------------------------------------------
// Block Jacobi on the whole GPU (the per-workgroup version is
// wg_block_jacobi).  Round r of the round-robin order pairs the 16-index
// blocks; k_jsub solves each pair's 32 x 32 subproblem (wave_jacobi_sub and
// sub_rotate), stores its rotation Q_k and the rotated diagonal
// block, and flags Q_k == I; k_japply then applies every Q_k of the round
// to the off-diagonal tiles of A (Q_k^T A_kl Q_l) and to the orbital rows.
// ---------------------------------------------------------------------------
// One workgroup per block pair k of round r.  The first wave runs the rounds of
// a sweep on the subproblem and records the rotations; all four stage it and
// apply the sweep to Q, two columns of Q^T a lane: 18.7 us a launch at n = 296
// and 10.2 at 4800 (everything in one wave 22.5 and 14.3).
constexpr int JSUB_WAVES = 4;
__global__ void __launch_bounds__(JSUB_WAVES * WAVE) k_jsub(double* A_, int n, int r, int nb2, double* Qbuf, int* ident,
                                                            double tol, int inner) {
    __shared__ __align__(16) double buf[JD + 2 * JB * (JS - 1)];
    __shared__ int more;
    glbf* A = to_glb(A_);
    const int b = blockIdx.x, lane = threadIdx.x % WAVE, k = lane % JB;
    ldsf *D = to_lds(buf), *cs = D + JD;
    int I, J;
    rr_pair(r, b, nb2, I, J);
    sub_stage<JSUB_WAVES>(A, n, I, J, D);
    constexpr int m = JS - 1, NC = JS / (4 * JSUB_WAVES);
    const int g0 = (int)threadIdx.x / JB * NC, rt = k == 0 ? m : k, rb = k == 0 ? 0 : m - k;
    double top[NC], bot[NC];
#pragma unroll
    for (int y = 0; y < NC; ++y) {
        top[y] = rt == g0 + y ? 1.0 : 0.0;
        bot[y] = rb == g0 + y ? 1.0 : 0.0;
    }
    int rot = 0;
    __syncthreads();
    for (int sw = 0; sw < inner; ++sw) {
        if (threadIdx.x < WAVE) {
            const int go = wave_jacobi_sub<true>(D, cs, nullptr, tol, 1, 0, 0u, 0u);
            if (threadIdx.x == 0) more = go;
        }
        __syncthreads();
        if (!more) break;
        rot = 1;
#pragma unroll 4
        for (int q = 0; q < m; ++q) {
            const v2d v = *(ldsv2*)(cs + 2 * (JB * q + k));
#pragma unroll
            for (int y = 0; y < NC; ++y) sub_rotate(v.x, v.y, k, top[y], bot[y]);
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) ident[b] = rot ? 0 : 1;
    if (!rot) return;
    glbf* qg = to_glb(Qbuf) + (size_t)b * JS * JS;
#pragma unroll
    for (int y = 0; y < NC; ++y) {
        qg[(g0 + y) * JS + rt] = top[y];
        qg[(g0 + y) * JS + rb] = bot[y];
    }
    sub_unstage<JSUB_WAVES>(A, n, I, J, D);
}

// one wave per work item: the ntile off-diagonal tiles (k < l) of A, then
// npair x nch row chunks (64 columns) of the orbitals
__global__ void __launch_bounds__(NT) k_japply(double* A_, double* Ct_, int n, int r, int nb2,
                                               const double* Qbuf_, const int* ident) {
    glbf* A = to_glb(A_);
    glbf* Ct = to_glb(Ct_);
    const glbf* Qbuf = to_glb(Qbuf_);
    const int npair = nb2 / 2;
    const int ntile = npair * (npair - 1) / 2;
    const int nch = (n + WAVE - 1) / WAVE;
    const int it = __builtin_amdgcn_readfirstlane(blockIdx.x * NWAVE + threadIdx.x / WAVE);
    if (it >= ntile + npair * nch) return;
    if (it < ntile) {
        int k = 0, rem = it;
        while (rem >= npair - 1 - k) {
            rem -= npair - 1 - k;
            ++k;
        }
        const int l = k + 1 + rem;
        if (ident[k] && ident[l]) return;
        int Ik, Jk, Il, Jl;
        rr_pair(r, k, nb2, Ik, Jk);
        rr_pair(r, l, nb2, Il, Jl);
        tile_update(A, n, Qbuf + (size_t)k * JS * JS, Qbuf + (size_t)l * JS * JS, Ik, Jk, Il, Jl, ident[k],
                    ident[l]);
    } else {
        const int v = it - ntile;
        const int k = v / nch, ch = v % nch;
        if (ident[k]) return;
        int Ik, Jk;
        rr_pair(r, k, nb2, Ik, Jk);
        rows_update(Ct, n, (size_t)n, n, Qbuf + (size_t)k * JS * JS, Ik, Jk, ch * WAVE);
    }
}

// Rank of every eigenvalue estimate: skey ascending, sidx its row (equal ones
// in row order, NaN last).  A workgroup ranks 64 of them, each of its waves
// against an eighth of all (uniform loads).  With the smearing below 9.6, 12
// and 57 us at n = 296, 528 and 4800; sorted in the smearing's workgroup (by a
// bitonic network above 512) 11.2, 22.7 and 120.
__global__ void __launch_bounds__(NT) k_rank(int n, const double* __restrict__ ev, double* __restrict__ skey,
                                             int* __restrict__ sidx) {
    __shared__ int part[NWAVE][WAVE];
    const int w = uniform((int)threadIdx.x / WAVE), lane = threadIdx.x % WAVE;
    const int j = blockIdx.x * WAVE + lane, span = (n + NWAVE - 1) / NWAVE;
    const int lo = w * span, hi = lo + span < n ? lo + span : n;
    const double v = j < n ? ev[j] : INFINITY, e = v == v ? v : INFINITY;
    int r = 0;
#pragma unroll 8
    for (int i = lo; i < hi; ++i) {
        const double x = ev[i], y = x == x ? x : INFINITY;
        r += y < e || (y == e && i < j);
    }
    part[w][lane] = r;
    __syncthreads();
    if (w > 0 || j >= n) return;
    r = 0;
    for (int x = 0; x < NWAVE; ++x) r += part[x][lane];
    skey[r] = v;
    sidx[r] = j;
}

// ---------------------------------------------------------------------------
// Fermi smearing (one workgroup) of the sorted estimates: ftot[row] = f_alpha +
// f_beta, occ (alpha, beta, ascending order), and control values:
//   ctl[C_EFA], ctl[C_EFB]   Fermi levels
//   ctl[C_FOK]               1 if both channels converged
//   ctl[C_KOCC]              orbitals with f > 0 (a prefix in sorted order)
//   ctl[C_PERM]              1 if the sort moved any row
//   ctl[C_GAPA], ctl[C_GAPB] frontier gaps skey[ia] - skey[ia-1] (ib), +inf
//                            when the index is outside 1..n-1
//   ctl[C_FSOFT]             largest f (1 - f) of either channel
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(NT) k_fermi(int n, int nao, const double* skey_in, const int* sidx_in, double* ftot,
                                              double* occ, double nel_a, double nel_b, int ia, int ib, double kt,
                                              double thr, int maxiter, double* ctl, Post p) {
    extern __shared__ double lds[];
    ldsf* red = to_lds(lds);
    ldsf* skey = red + RED_DOUBLES;
    ldsi* sidx = reinterpret_cast<ldsi*>(skey + n);
    for (int j = threadIdx.x; j < n; j += NT) {
        skey[j] = skey_in[j];
        sidx[j] = sidx_in[j];
    }
    __syncthreads();
    const Filling fl = fill_orbitals(n, nao, nel_a, nel_b, skey, sidx, to_glb(ftot), red, kt, thr, maxiter, false,
                                     to_glb(occ), to_glb(occ) + n);
    if (threadIdx.x == 0) {
        ctl[C_EFA] = fl.ef[0];
        ctl[C_EFB] = fl.ef[1];
        ctl[C_FOK] = fl.ok ? 1.0 : 0.0;
        ctl[C_KOCC] = (double)fl.kocc;
        ctl[C_PERM] = fl.moved ? 1.0 : 0.0;
        ctl[C_GAPA] = (ia > 0 && ia < n) ? skey[ia] - skey[ia - 1] : INFINITY;
        ctl[C_GAPB] = (ib > 0 && ib < n) ? skey[ib] - skey[ib - 1] : INFINITY;
        ctl[C_FSOFT] = fl.soft;
    }
    post(ctl, p);
}

// G[j] = Ct[sidx[j]]; one workgroup per row.  With ctl: only if the sort moved
// a row (when = C_PERM), or only the occupied rows j < ctl[C_KOCC] (when =
// C_KOCC)
__global__ void __launch_bounds__(256) k_gather(int n, const double* Ct, const int* sidx, const double* ctl, int when,
                                                double* G) {
    const int j = blockIdx.x;
    if (ctl && (when == C_PERM ? ctl[C_PERM] == 0.0 : (double)j >= ctl[C_KOCC])) return;
    const double* src = Ct + (size_t)sidx[j] * n;
    for (int c = threadIdx.x; c < n; c += 256) G[(size_t)j * n + c] = src[c];
}

// H[j] = w_j X[j] for the occupied rows j < ctl[C_KOCC], w_j = ftot[sidx[j]]
// (x ev[sidx[j]] when ev is given), one workgroup per row.  With Ct: X are
// the rows gathered for a sort that moved any, which become Ct's rows; Ct
// itself is X if it moved none.
__global__ void __launch_bounds__(256) k_scale_rows(int n, const double* X, const int* sidx, const double* ftot,
                                                    const double* ev, const double* ctl, double* Ct, double* H) {
    const int j = blockIdx.x;
    const bool perm = ctl[C_PERM] != 0.0, occ = (double)j < ctl[C_KOCC], back = Ct && perm;
    if (!occ && !back) return;
    const int o = sidx[j];
    const double w = ev ? ftot[o] * ev[o] : ftot[o];
    const double* src = Ct && !perm ? Ct : X;
    for (int c = threadIdx.x; c < n; c += 256) {
        const double x = src[(size_t)j * n + c];
        if (back) Ct[(size_t)j * n + c] = x;
        if (occ) H[(size_t)j * n + c] = w * x;
    }
}

// A'_ij = (f_i + f_j)/2 A_ij for the k x k occupied block, f of row i = ftot[i]
__global__ void __launch_bounds__(256) k_scale_pairs(int k, double* A, const double* ftot) {
    const int i = blockIdx.x;
    const double fi = ftot[i];
    for (int j = threadIdx.x; j < k; j += 256) A[(size_t)i * k + j] *= 0.5 * (fi + ftot[j]);
}

// Mulliken (scf/base.py:764-815): q_i = n0_i - (P S)_ii, eorb_i = (P H0)_ii
// (last step only); one wave per row
__global__ void __launch_bounds__(NT) k_mulliken(int n, int nao, const double* P, const double* S, const double* H0,
                                                 const double* n0, int last, double* q, double* eorb) {
    const int i = blockIdx.x * NWAVE + threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
    if (i >= n) return;
    double sq = 0.0, se = 0.0;
    if (i < nao) {
        const double* pr = P + (size_t)i * n;
        const double* sr = S + (size_t)i * n;
        const double* hr = H0 + (size_t)i * n;
        for (int j = lane; j < nao; j += WAVE) {
            sq = fma(pr[j], sr[j], sq);
            if (last) se = fma(pr[j], hr[j], se);
        }
    }
    sq = wave_sum(sq);
    se = wave_sum(se);
    if (lane == 0) {
        q[i] = (i < nao) ? n0[i] - sq : 0.0;
        eorb[i] = (i < nao) ? se : 0.0;
    }
}

// Shell and atom charges, ES2 (gamma q_sh) + ES3 (hd q_at^2) shell potential,
// spread to the orbitals; one wave per shell.  Every workgroup sums all shell
// charges for itself (LDS, nsh doubles): three launches in one.
__global__ void __launch_bounds__(NT) k_potential(int nsh, const int* sh_ao, const int* sh_us, const int* us_l,
                                                  const int* atom_sh0, const int* atom_nsh, const double* q,
                                                  const double* gam, const int* sh_atom, const int* atom_sp,
                                                  const double* sp_gam3, double* qsh_out, double* qat, double* gq,
                                                  double* v) {
    extern __shared__ double lds[];
    ldsf* qsh = to_lds(lds);
    for (int s = threadIdx.x; s < nsh; s += NT) {
        const int o0 = sh_ao[s], nl = 2 * us_l[sh_us[s]] + 1;
        double acc = 0.0;
        for (int x = 0; x < nl; ++x) acc += q[o0 + x];
        qsh[s] = acc;
    }
    __syncthreads();
    const int s = blockIdx.x * NWAVE + threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
    if (s >= nsh) return;
    const double* gr = gam + (size_t)s * nsh;
    double acc = 0.0;
    for (int t = lane; t < nsh; t += WAVE) acc = fma(gr[t], qsh[t], acc);
    acc = wave_sum(acc);
    const int a = sh_atom[s], s0 = atom_sh0[a], ns = atom_nsh[a];
    double qa = 0.0;
    for (int x = 0; x < ns; ++x) qa += qsh[s0 + x];
    const double vs = acc + sp_gam3[atom_sp[a]] * qa * qa;
    const int o0 = sh_ao[s], nl = 2 * us_l[sh_us[s]] + 1;
    if (lane < nl) v[o0 + lane] = vs;
    if (lane == 0) {
        qsh_out[s] = qsh[s];
        gq[s] = acc;
        if (s == s0) qat[a] = qa;
    }
}

// Mixing (one workgroup; the same mixers as the per-molecule kernel):
// Anderson, or Broyden when o.mixer == 1.  ctl[C_CONV] = converged,
// ctl[C_RESID] = the residual's max norm; the Broyden memory's rank and last
// step norm go to ctl[C_BRANK], ctl[C_BDX] for the host's copy of its state
__global__ void __launch_bounds__(NT) k_mix(Mixer mx, Broyden bm, int n, xtb_scf_opts o, double* hx, double* hf,
                                            const double* xnew, const double* xold, double* xout, double* ctl,
                                            Post p) {
    __shared__ double red[RED_DOUBLES];
    const MixOpts mo{o.x_atol, o.x_atol_max, o.damp, o.damp_init, o.diag_offset};
    double resid = 0.0;
    const bool c = o.mixer == 1
        ? broyden(bm, n, n, to_lds(red), mo, o.f_atol, to_glb(hx), to_glb(hf), to_glb(xnew), to_glb(xold),
                  to_glb(xout), &resid)
        : anderson(mx, n, n, to_lds(red), mo, to_glb(hx), to_glb(hf), to_glb(xnew), to_glb(xold), to_glb(xout), &resid);
    if (threadIdx.x == 0) {
        ctl[C_CONV] = c ? 1.0 : 0.0;
        ctl[C_RESID] = resid;
        ctl[C_BRANK] = (double)bm.rank;
        ctl[C_BDX] = bm.dxnorm;
    }
    post(ctl, p);
}

// energies (scf/base.py:514-623) into the result record (one workgroup)
__global__ void __launch_bounds__(NT) k_energies(int n, int nao, int nsh, int nat, const double* eorb,
                                                 const double* qsh, const double* gq, const double* qat,
                                                 const int* atom_sp, const double* sp_gam3, const double* occ,
                                                 double kt, double* out) {
    __shared__ double red[256];
    double acc[4] = {0.0, 0.0, 0.0, 0.0};
    for (int i = threadIdx.x; i < nao; i += NT) acc[0] += eorb[i];
    for (int s = threadIdx.x; s < nsh; s += NT) acc[1] += 0.5 * qsh[s] * gq[s];
    for (int a = threadIdx.x; a < nat; a += NT) {
        const double hd = sp_gam3[atom_sp[a]];
        acc[2] += hd * qat[a] * qat[a] * qat[a] / 3.0;
    }
    const double eps = 2.220446049250313e-16;
    for (int j = threadIdx.x; j < 2 * n; j += NT) {
        const double f = occ[j];
        const double f1 = fmax(f, eps), f2 = fmax(1.0 - f, eps);
        acc[3] += f1 * log(f1) + f2 * log(f2);
    }
    wg_sum_n<4>(acc, to_lds(red));
    if (threadIdx.x == 0) {
        out[XTB_OUT_ESCF] = acc[0] + acc[1] + acc[2];
        out[XTB_OUT_EH0] = acc[0];
        out[XTB_OUT_EES2] = acc[1];
        out[XTB_OUT_EES3] = acc[2];
        out[XTB_OUT_FENERGY] = acc[3] * kt;
    }
}

__global__ void k_copy_emo(int n, const double* skey, int nan_out, double* emo) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) emo[i] = nan_out ? NAN : skey[i];
}

}  // namespace big
}  // namespace xtb

// ===========================================================================
// Host driver
// ===========================================================================
namespace {

using namespace xtb;
using namespace xtb::big;

// result-record slots written from the host (mask bit i: slot i)
struct Rec {
    double v[XTB_OUT_STRIDE];
    uint32_t mask;
};

__global__ void k_put(double* out, Rec r) {
    const int i = threadIdx.x;
    if (i < XTB_OUT_STRIDE && ((r.mask >> i) & 1u)) out[i] = r.v[i];
}

__global__ void k_diag(int n, const double* A, double* ev) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) ev[i] = A[(size_t)i * n + i];
}

// per-workgroup max |x_i|
__global__ void __launch_bounds__(NT) k_vec_absmax(int n, const double* x, double* part) {
    __shared__ double red[NWAVE];
    double m = 0.0;
    for (int i = blockIdx.x * NT + threadIdx.x; i < n; i += gridDim.x * NT) m = fmax(m, fabs(x[i]));
    m = wave_max(m);
    if (threadIdx.x % WAVE == 0) red[threadIdx.x / WAVE] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        double r = red[0];
        for (int k = 1; k < NWAVE; ++k) r = fmax(r, red[k]);
        part[blockIdx.x] = r;
    }
}

inline size_t al32(size_t d) { return (d + 31) & ~(size_t)31; }

struct Layout {
    size_t E, Q, ev, skey, ftot, sidx, ident, part, ctl, qat, gq, total;
};

Layout make_layout(int n, int nsh, int nat) {
    const int nb = (n + JB - 1) / JB, nb2 = nb + (nb & 1), npair = nb2 / 2;
    Layout L;
    size_t o = 0;
    L.E = o; o += al32((size_t)n * n);
    L.Q = o; o += al32((size_t)npair * JS * JS);
    L.ev = o; o += al32(n);
    L.skey = o; o += al32(n);
    L.ftot = o; o += al32(n);
    L.sidx = o; o += al32((n + 1) / 2);
    L.ident = o; o += al32((npair + 1) / 2);
    L.part = o; o += al32(4 * (size_t)n + 4096);
    L.ctl = o; o += al32(C_NCTL);
    L.qat = o; o += al32(nat);
    L.gq = o; o += al32(nsh);
    L.total = o;
    return L;
}

// largest orbital count: the Fermi smearing keeps keys and indices in one
// workgroup's LDS
constexpr int LARGE_MAX_N = 8192;

// Boxes lent to calls, one each from start to end (a call returns only when
// nothing can post to its box any more).  At most MAILS_KEPT idle ones stay
// for later calls: allocating pinned memory synchronises the whole device,
// which other streams' work would feel at every call.
struct Mail {
    Box* box;
    unsigned long long seq;  // of the last post asked for
};
constexpr size_t MAILS_KEPT = 16;
std::mutex mails_mutex;
Mail mails_idle[MAILS_KEPT];
size_t mails_count = 0;

struct MailLease {
    Mail mail{nullptr, 0};
    hipError_t open() {
        {
            std::lock_guard<std::mutex> lock(mails_mutex);
            if (mails_count > 0) {
                mail = mails_idle[--mails_count];
                return hipSuccess;
            }
        }
        const hipError_t e = hipHostMalloc((void**)&mail.box, sizeof(Box),
                                           hipHostMallocPortable | hipHostMallocMapped | hipHostMallocCoherent);
        if (e == hipSuccess) mail.box->seq = 0;
        else mail.box = nullptr;
        return e;
    }
    ~MailLease() {
        if (!mail.box) return;
        {
            std::lock_guard<std::mutex> lock(mails_mutex);
            if (mails_count < MAILS_KEPT) {
                mails_idle[mails_count++] = mail;
                return;
            }
        }
        (void)hipHostFree(mail.box);
    }
};

struct Ctx {
    hipStream_t s;
    const xtb_batch* b;
    const xtb_params* par;
    xtb_scf_opts o;
    const xtb_scf_state* st;
    int n, nao, nsh, nat, nb2, npair;
    double nel_a, nel_b;
    int ia, ib;
    const double *S, *H0, *gam;
    double *F, *Ct, *T, *P, *E;  // n x n; the roles of F, Ct and E rotate
    double *ev, *skey, *ftot, *Qbuf, *part, *ctl, *qat, *gq;
    int *sidx, *ident;
    double h[C_NCTL];  // control values of the last read_ctl
    Mail* mail;
    double gap_a = INFINITY, gap_b = INFINITY;  // frontier gaps of the last sort
    int refresh = 0;                            // perturbative steps since fresh eigenvalues
    hipError_t err = hipSuccess;
    int pd_steps = 0;
    double t_eig = 0.0, t_pd = 0.0;
};

inline void chk(Ctx& c, hipError_t e) {
    if (e != hipSuccess && c.err == hipSuccess) c.err = e;
}
inline void chk_launch(Ctx& c) { chk(c, hipGetLastError()); }

inline double now_s() {
    return std::chrono::duration<double>(std::chrono::steady_clock::now().time_since_epoch()).count();
}

constexpr Post NO_POST{nullptr, 0};

// for the kernel launched last before read_ctl
Post next_post(Ctx& c) { return Post{c.mail->box, ++c.mail->seq}; }

// Waits for the last post and takes its values.  The wait watches host memory
// for ~200 us, then leaves it to the stream.  (A copy and a stream
// synchronisation instead left the GPU idle for ~40 us a time: of 8.5 ms at n
// = 296, 3.1 were such gaps; with fewer reads and fewer, merged kernels the
// same call takes 5.3.)
bool read_ctl(Ctx& c) {
    if (c.err != hipSuccess) return false;
    Box* box = c.mail->box;
    auto there = [&]() { return __atomic_load_n(&box->seq, __ATOMIC_ACQUIRE) == c.mail->seq; };
    const auto t0 = std::chrono::steady_clock::now();
    while (!there()) {
        for (int i = 0; i < 32 && !there(); ++i) __builtin_ia32_pause();
        if (std::chrono::steady_clock::now() - t0 > std::chrono::microseconds(200)) {
            chk(c, hipStreamSynchronize(c.s));
            if (c.err == hipSuccess && !there()) chk(c, hipErrorUnknown);
            break;
        }
    }
    if (c.err != hipSuccess) return false;
    for (int i = 0; i < C_NCTL; ++i) c.h[i] = box->v[i];
    return true;
}

// ctl[slot] = sum / max of nblk partials; posted if it is to be read
void finish(Ctx& c, int nblk, int op, int slot, Post p = NO_POST) {
    hipLaunchKernelGGL(k_finish, dim3(1), dim3(NT), 0, c.s, c.part, nblk, op, c.ctl, slot, p);
    chk_launch(c);
}

template <bool TA, bool TB, bool EPI>
void gemm_t(Ctx& c, int M, int N, int K, double alpha, const double* A, int lda, const double* B, int ldb,
            double beta, double* C, int ldc, bool upper, const Epi& ep = Epi{}, const double* Kd = nullptr) {
    if (M <= 0 || N <= 0) return;
    auto tiles = [&](int t) {
        const int tm = (M + t - 1) / t, tn = (N + t - 1) / t;
        return upper ? tm * (tm + 1) / 2 : tm * tn;
    };
#define XTB_GG(SPLIT, F, KS, NB)                                                                                     \
    {                                                                                                                \
        const int nt = tiles((SPLIT ? 16 : 32) * F), grid = (nt + 7) / 8 * 8;                                        \
        hipLaunchKernelGGL((k_gemm<TA, TB, EPI, SPLIT, F, F, KS, NB>), dim3(grid), dim3(256), 0, c.s, M, N, K,       \
                           alpha, A, lda, B, ldb, beta, C, ldc, upper ? 1 : 0, nt, Kd, ep);                          \
    }
    // the largest tile that still gives the CUs enough workgroups.  us at both
    // sides of the lines: 48-wide tiles (against 32) from ~220 of them, 750 x
    // 1500 x 750 (512) 37 / 44, 500 x 1001 x 500 (231) 15.4 / 14.2, 528^3
    // (121) 15.5 / 15.7; 16-wide below 600 of them, 296^3 (361) 5.4 / 6.8, 350
    // x 700 x 350 (968) 9.2 / 7.5; all of k per wave from 1000 96-wide tiles,
    // 2400 x 4800 x 2400 (1250) 821 / 875, 2400^3 (625) 520 / 460
    if (tiles(96) >= 1000) XTB_GG(false, 3, 2, 2)
    else if (tiles(48) >= 220) XTB_GG(true, 3, 2, 2)
    else if (tiles(16) <= 600) XTB_GG(true, 1, 4, 4)
    else XTB_GG(true, 2, 2, 3)
#undef XTB_GG
    chk_launch(c);
}

// C (n x n, symmetric) = op(A) op(B); with Kd, k is *Kd at run time
template <bool TA, bool TB>
void gemm_sym(Ctx& c, int n, int K, const double* A, int lda, const double* B, int ldb, double* C, int ldc,
              const double* Kd = nullptr) {
    gemm_t<TA, TB, false>(c, n, n, K, 1.0, A, lda, B, ldb, 0.0, C, ldc, true, Epi{}, Kd);
}

void fock(Ctx& c, const double* v) {
    hipLaunchKernelGGL(k_fock, dim3((c.n + 255) / 256, c.n), dim3(256), 0, c.s, c.n, c.H0, c.S, v, c.F);
    chk_launch(c);
}

size_t fermi_lds(int n) { return (RED_DOUBLES + (size_t)n) * 8 + (size_t)n * 4; }

void sort_fermi(Ctx& c, Post p) {
    const xtb_scf_opts& o = c.o;
    hipLaunchKernelGGL(k_rank, dim3((c.n + WAVE - 1) / WAVE), dim3(NT), 0, c.s, c.n, c.ev, c.skey, c.sidx);
    chk_launch(c);
    hipLaunchKernelGGL(k_fermi, dim3(1), dim3(NT), fermi_lds(c.n), c.s, c.n, c.nao, c.skey, c.sidx, c.ftot, c.st->occ,
                       c.nel_a, c.nel_b, c.ia, c.ib, o.kt, o.fermi_thresh, o.fermi_maxiter, c.ctl, p);
    chk_launch(c);
}

void axpby(Ctx& c, size_t len, double a, const double* X, double b, const double* Z, double* Y) {
    const size_t g = (len + 255) / 256;
    hipLaunchKernelGGL(k_axpby, dim3((unsigned)(g < 8192 ? g : 8192)), dim3(256), 0, c.s, len, a, X, b, Z, Y);
    chk_launch(c);
}

// Loewdin orthogonaliser by coupled Newton-Schulz (as ortho_setup in
// scf_kernel.h): Ct <- X = S^-1/2.  Returns false when the iteration did not
// converge (S numerically singular).
bool ortho(Ctx& c) {
    const int n = c.n;
    const size_t nn = (size_t)n * n;
    const int rb = (n + NWAVE - 1) / NWAVE;
    hipLaunchKernelGGL(k_rowabs, dim3(rb), dim3(NT), 0, c.s, n, c.S, c.part);
    chk_launch(c);
    finish(c, rb, 1, C_GERSH, next_post(c));
    if (!read_ctl(c)) return false;
    const double cg = c.h[C_GERSH] * 1.0001;
    double* Y = c.F;
    double* Z = c.Ct;
    double* W = c.P;
    double* T = c.T;
    axpby(c, nn, 1.0 / cg, c.S, 0.0, nullptr, Y);
    hipLaunchKernelGGL(k_identity, dim3((n + 255) / 256, n), dim3(256), 0, c.s, n, Z);
    chk_launch(c);
    int it = 0, extra = -1;
    for (; it < 60; ++it) {
        gemm_t<false, false, false>(c, n, n, n, -0.5, Z, n, Y, n, 0.0, T, n, false);
        hipLaunchKernelGGL(k_add_diag, dim3((n + 255) / 256), dim3(256), 0, c.s, n, 1.5, T);
        chk_launch(c);
        hipLaunchKernelGGL(k_dev_identity, dim3(rb), dim3(NT), 0, c.s, n, T, c.part);
        chk_launch(c);
        finish(c, rb, 1, C_ERR, next_post(c));
        if (!read_ctl(c)) return false;
        const double err = c.h[C_ERR];
        if (extra == 0 || err < 1e-15) break;
        if (extra > 0) --extra;
        else if (err < 1e-9) extra = 1;
        gemm_t<false, false, false>(c, n, n, n, 1.0, Y, n, T, n, 0.0, W, n, false);  // Y T
        gemm_t<false, false, false>(c, n, n, n, 1.0, T, n, Z, n, 0.0, Y, n, false);  // T Z
        double* oldZ = Z;
        Z = Y;
        Y = W;
        W = oldZ;
    }
    // X = Z / sqrt(c), symmetrised, into the orbital buffer (Z is F, Ct or P)
    double* dst = (Z == c.Ct) ? c.E : c.Ct;
    hipLaunchKernelGGL(k_symmetrise, dim3((n + 255) / 256, n), dim3(256), 0, c.s, n, 1.0 / sqrt(cg), Z, dst);
    chk_launch(c);
    if (dst == c.E) {
        double* t = c.Ct;
        c.Ct = c.E;
        c.E = t;
    }
    return it < 60;
}

// Warm start (as in k_scf): the orbitals a previous call left in the state
// (rows in the orbital buffer) become S-orthonormal for the new geometry,
// C <- (C S C^T)^-1/2 C by coupled Newton-Schulz (C S C^T is close to I
// after a small displacement, so a few steps; the symmetric form keeps each
// orbital as close to its old self as possible), and are sorted by their
// energies in the Fock matrix of the kept potential `pot`, so that the first
// step can decouple occupied from virtual orbitals without an eigensolve.
// Returns false, with the orbitals untouched, when C S C^T is too far from
// I (then the caller starts cold).
bool warm_orthonormalise(Ctx& c, const double* pot) {
    const int n = c.n;
    const int rb = (n + NWAVE - 1) / NWAVE;
    // G = C S C^T, the iteration's Y
    gemm_t<false, false, false>(c, n, n, n, 1.0, c.Ct, n, c.S, n, 0.0, c.T, n, false);
    gemm_sym<false, true>(c, n, n, c.T, n, c.Ct, n, c.F, n);
    double* Y = c.F;
    double* Z = c.P;
    double* W = c.E;
    double* T = c.T;
    hipLaunchKernelGGL(k_identity, dim3((n + 255) / 256, n), dim3(256), 0, c.s, n, Z);
    chk_launch(c);
    int it = 0, extra = -1;
    for (; it < 30; ++it) {
        gemm_t<false, false, false>(c, n, n, n, -0.5, Z, n, Y, n, 0.0, T, n, false);
        hipLaunchKernelGGL(k_add_diag, dim3((n + 255) / 256), dim3(256), 0, c.s, n, 1.5, T);
        chk_launch(c);
        hipLaunchKernelGGL(k_dev_identity, dim3(rb), dim3(NT), 0, c.s, n, T, c.part);
        chk_launch(c);
        finish(c, rb, 1, C_ERR, next_post(c));
        if (!read_ctl(c)) return false;
        const double err = c.h[C_ERR];
        // |I - T| = |I - G|/2 at the start: beyond 1/4 the kept orbitals
        // are too far off to be worth keeping
        if (it == 0 && !(err < 0.25)) return false;
        if (extra == 0 || err < 1e-15) break;
        if (extra > 0) --extra;
        else if (err < 1e-9) extra = 1;
        gemm_t<false, false, false>(c, n, n, n, 1.0, Y, n, T, n, 0.0, W, n, false);  // Y T
        gemm_t<false, false, false>(c, n, n, n, 1.0, T, n, Z, n, 0.0, Y, n, false);  // T Z
        double* oldZ = Z;
        Z = Y;
        Y = W;
        W = oldZ;
    }
    if (it >= 30) return false;
    // C <- Z C (Z = G^-1/2), through T
    gemm_t<false, false, false>(c, n, n, n, 1.0, Z, n, c.Ct, n, 0.0, T, n, false);
    chk(c, hipMemcpyAsync(c.Ct, T, sizeof(double) * n * n, hipMemcpyDeviceToDevice, c.s));
    // energy estimates e_i = (C F C^T)_ii, rows sorted by them; the sort's
    // frontier gaps steer the first step's occupied-virtual decoupling
    fock(c, pot);
    gemm_t<false, false, false>(c, n, n, n, 1.0, c.Ct, n, c.F, n, 0.0, T, n, false);
    hipLaunchKernelGGL(k_rowdot, dim3(rb), dim3(NT), 0, c.s, n, n, T, c.Ct, (const double*)nullptr, c.ev);
    chk_launch(c);
    sort_fermi(c, next_post(c));
    hipLaunchKernelGGL(k_gather, dim3(n), dim3(256), 0, c.s, n, c.Ct, c.sidx, (const double*)nullptr, 0, c.F);
    chk_launch(c);
    chk(c, hipMemcpyAsync(c.Ct, c.F, sizeof(double) * n * n, hipMemcpyDeviceToDevice, c.s));
    if (!read_ctl(c)) return false;
    c.gap_a = c.h[C_GAPA];
    c.gap_b = c.h[C_GAPB];
    c.refresh = 1;  // the virtual orbitals' estimates are fresh
    return true;
}

// Cholesky orthogonaliser (as chol_setup in scf_kernel.h): S = L L^T by
// right-looking 32-wide panels (a wave factors each diagonal block, the panel
// solve and the trailing update are grid GEMMs), then X = L^-1 by the
// right-looking triangular inverse: block row j of X <- D_j^-1 X_j, rows
// below -= L_(>j, j) X_j, on the identity.  L in T, X in the orbital buffer,
// R (rows x 32, leading dimension n) in F, the block inverses in P.  Returns
// false when S is not numerically positive definite.
bool ortho_chol(Ctx& c) {
    constexpr int NB = 32;
    const int n = c.n;
    double* L = c.T;
    double* X = c.Ct;
    double* R = c.F;
    double* Dg = c.P;
    chk(c, hipMemcpyAsync(L, c.S, sizeof(double) * n * n, hipMemcpyDeviceToDevice, c.s));
    hipLaunchKernelGGL(k_set_slot, dim3(1), dim3(1), 0, c.s, c.ctl, (int)C_ERR, 0.0);
    chk_launch(c);
    for (int j0 = 0; j0 < n; j0 += NB) {
        const int nb = n - j0 < NB ? n - j0 : NB;
        double* D = Dg + (size_t)j0 * NB;
        hipLaunchKernelGGL(k_chol_diag, dim3(1), dim3(WAVE), 0, c.s, L, n, j0, nb, D, c.ctl);
        chk_launch(c);
        const int mt = n - j0 - nb;
        if (mt > 0) {
            double* Pn = L + (size_t)(j0 + nb) * n + j0;  // panel below the block
            gemm_t<false, true, false>(c, mt, nb, nb, 1.0, Pn, n, D, nb, 0.0, R, n, false);  // b D^-T
            hipLaunchKernelGGL(k_copy_block, dim3(1, mt), dim3(256), 0, c.s, mt, nb, R, n, Pn, n);
            chk_launch(c);
            gemm_t<false, true, false>(c, mt, mt, nb, -1.0, Pn, n, Pn, n, 1.0, Pn + nb, n, false);
        }
    }
    hipLaunchKernelGGL(k_post, dim3(1), dim3(WAVE), 0, c.s, c.ctl, next_post(c));
    chk_launch(c);
    if (!read_ctl(c) || c.h[C_ERR] != 0.0) return false;
    hipLaunchKernelGGL(k_identity, dim3((n + 255) / 256, n), dim3(256), 0, c.s, n, X);
    chk_launch(c);
    for (int j0 = 0; j0 < n; j0 += NB) {
        const int nb = n - j0 < NB ? n - j0 : NB;
        const int w = j0 + nb;  // non-zero columns of block row j
        double* Xj = X + (size_t)j0 * n;
        gemm_t<false, false, false>(c, nb, w, nb, 1.0, Dg + (size_t)j0 * NB, nb, Xj, n, 0.0, R, n,
                                    false);  // D^-1 X_j
        hipLaunchKernelGGL(k_copy_block, dim3((w + 255) / 256, nb), dim3(256), 0, c.s, nb, w, R, n, Xj, n);
        chk_launch(c);
        const int mt = n - w;
        if (mt > 0)
            gemm_t<false, false, false>(c, mt, w, nb, -1.0, L + (size_t)w * n + j0, n, Xj, n, 1.0,
                                        X + (size_t)w * n, n, false);
    }
    return c.err == hipSuccess;
}

// Block Jacobi on A = F (full symmetric); rotations applied to the orbital
// rows.  Tolerance as eig_step in scf_kernel.h.  Eigenvalue estimates -> ev.
// Returns sweeps, or -1 when max_sweeps were spent.
int eig(Ctx& c, double rel_tol, double loose) {
    const double t0 = now_s();
    const int n = c.n;
    const int rb = (n + NWAVE - 1) / NWAVE;
    const int ntile = c.npair * (c.npair - 1) / 2;
    const int nch = (n + WAVE - 1) / WAVE;
    const int nitem = ntile + c.npair * nch;
    // scale of the tolerance: the largest diagonal element of A
    hipLaunchKernelGGL(k_diag, dim3((n + 255) / 256), dim3(256), 0, c.s, n, c.F, c.ev);
    chk_launch(c);
    hipLaunchKernelGGL(k_vec_absmax, dim3(1), dim3(NT), 0, c.s, n, c.ev, c.part);
    chk_launch(c);
    finish(c, 1, 1, C_DMAX);
    double tol = 0.0;
    int sweep = 0;
    for (;;) {
        hipLaunchKernelGGL(k_offmax, dim3(rb), dim3(NT), 0, c.s, n, c.F, c.part);
        chk_launch(c);
        finish(c, rb, 1, C_OFF, next_post(c));
        if (!read_ctl(c)) return -1;
        if (sweep == 0) tol = fmax(fmax(rel_tol * fmax(c.h[C_DMAX], 1.0), loose), JACOBI_TOL_MIN);
        if (c.h[C_OFF] <= tol) break;
        if (sweep >= c.o.jacobi_max_sweeps) {
            sweep = -1;
            break;
        }
        for (int r = 0; r < c.nb2 - 1; ++r) {
            hipLaunchKernelGGL(k_jsub, dim3(c.npair), dim3(JSUB_WAVES * WAVE), 0, c.s, c.F, n, r, c.nb2, c.Qbuf, c.ident, tol,
                               c.o.jacobi_inner);
            chk_launch(c);
            hipLaunchKernelGGL(k_japply, dim3((nitem + NWAVE - 1) / NWAVE), dim3(NT), 0, c.s, c.F, c.Ct, n, r,
                               c.nb2, c.Qbuf, c.ident);
            chk_launch(c);
        }
        ++sweep;
    }
    hipLaunchKernelGGL(k_diag, dim3((n + 255) / 256), dim3(256), 0, c.s, n, c.F, c.ev);
    chk_launch(c);
    c.refresh = 1;  // eigenvalues fresh for the next perturbative step
    c.t_eig += now_s() - t0;
    return sweep;
}

// Perturbative occupied-virtual rotation of a closed shell with k doubly
// occupied rows first (pd_step in scf_kernel.h, with grid GEMMs).  Returns 1
// when done, 0 to ask for Jacobi with Ct and F untouched, -1 to ask for it
// after F served as scratch.
int pd(Ctx& c, int k, double loose, const double* vin) {
    const int n = c.n, m = n - k;
    if (k <= 0 || m <= 0 || 2 * k > n) return 0;
    const double t0 = now_s();
    double* Cv = c.Ct + (size_t)k * n;
    double* Kb = c.P;  // k x m
    const bool refresh = c.refresh == 0 || c.refresh >= 4;
    c.refresh = refresh ? 1 : c.refresh + 1;
    const int rows = refresh ? n : k;
    int ret = 1;
    const int npass = loose > 0.0 ? PD_INEXACT_PASSES : PD_EXACT_PASSES;
    for (int pass = 0; pass < npass; ++pass) {
        if (pass > 0) fock(c, vin);
        gemm_t<false, false, false>(c, rows, n, n, 1.0, c.Ct, n, c.F, n, 0.0, c.T, n, false);  // C F
        gemm_t<false, true, false>(c, k, m, n, 1.0, c.T, n, Cv, n, 0.0, Kb, m, false);        // A_ov
        hipLaunchKernelGGL(k_rowdot, dim3((n + NWAVE - 1) / NWAVE), dim3(NT), 0, c.s, rows, n, c.T, c.Ct, c.skey,
                           c.ev);
        chk_launch(c);
        const int ab = (k + NWAVE - 1) / NWAVE;
        hipLaunchKernelGGL(k_amplitudes, dim3(ab), dim3(NT), 0, c.s, k, m, Kb, c.ev, c.part);
        chk_launch(c);
        hipLaunchKernelGGL(k_pd_stats, dim3(1), dim3(NT), 0, c.s, n, c.ev, c.part, ab, c.ctl, next_post(c));
        chk_launch(c);
        if (!read_ctl(c)) return 0;
        const double tol = fmax(c.o.jacobi_tol * fmax(c.h[C_DMAX], 1.0),
                                loose > 0.0 ? loose : PD_FINAL_REL * c.o.x_atol_max);
        const double aov = c.h[C_AOV], kmax = c.h[C_KMAX], dmin = c.h[C_DMIN];
        if (aov <= tol) { ret = 1; break; }
        const int fail = pass == 0 ? 0 : -1;
        if (!(dmin > 0.0) || !(kmax <= c.o.pd_kmax)) { ret = fail; break; }
        // an exact call's last pass only measures
        if (loose == 0.0 && pass == npass - 1) { ret = fail; break; }
        double* X = c.T;
        double* Z = c.T + (size_t)k * k;
        gemm_sym<false, true>(c, k, m, Kb, m, Kb, m, X, k);                                  // K K^T
        gemm_t<false, false, false>(c, k, n, m, 1.0, Kb, m, Cv, n, 0.0, Z, n, false);         // K C_vir
        hipLaunchKernelGGL(k_sumsq, dim3(256), dim3(NT), 0, c.s, (size_t)k * k, X, c.part);
        chk_launch(c);
        finish(c, 256, 0, C_XF, next_post(c));
        if (!read_ctl(c)) return 0;
        const double xf = sqrt(c.h[C_XF]);
        const double tolj = loose > 0.0 ? fmin(1e-13, fmax(1e-17, 1e-3 * loose)) : 1e-17;
        int J = 0;
        double term = 0.5 * xf;
        bool toolong = false;
        while (term > tolj) {
            ++J;
            term *= xf / ((2.0 * J + 1.0) * (2.0 * J + 2.0));
            if (J > 8) { toolong = true; break; }
        }
        if (toolong) { ret = fail; break; }
        double cc[9], ss[9], ph[9];
        {
            double f = 1.0;  // (2j)!
            for (int j = 0; j <= 8; ++j) {
                if (j > 0) f *= (2.0 * j - 1.0) * (2.0 * j);
                const double sg = (j & 1) ? -1.0 : 1.0;
                cc[j] = sg / f;
                ss[j] = sg / (f * (2.0 * j + 1.0));
                ph[j] = -sg / (f * (2.0 * j + 1.0) * (2.0 * j + 2.0));
            }
        }
        // R = sinc(X) C_occ + phi(X) Z and D = cos(X) C_occ - sinc(X) Z by
        // Horner's rule, side by side (columns 0 .. n and n .. 2n) until the
        // last term, which writes D over C_occ
        double* cur = c.F;
        double* nxt = c.E;
        const int n2 = 2 * n;
        hipLaunchKernelGGL(k_series0, dim3((n + 255) / 256, k), dim3(256), 0, c.s, n, c.Ct, Z, ss[J], ph[J], cur, n2,
                           cc[J], -ss[J], J == 0 ? c.Ct : cur + n, J == 0 ? n : n2);
        chk_launch(c);
        for (int j = J - 1; j > 0; --j) {
            gemm_t<false, false, true>(c, k, n2, k, 1.0, X, k, cur, n2, 0.0, nxt, n2, false,
                                       Epi{c.Ct, Z, n, n, ss[j], ph[j], cc[j], -ss[j]});
            double* t = cur; cur = nxt; nxt = t;
        }
        if (J > 0) {
            gemm_t<false, false, true>(c, k, n, k, 1.0, X, k, cur, n2, 0.0, nxt, n2, false,
                                       Epi{c.Ct, Z, n, n, ss[0], ph[0], 0.0, 0.0});
            gemm_t<false, false, true>(c, k, n, k, 1.0, X, k, cur + n, n2, 0.0, c.Ct, n, false,
                                       Epi{c.Ct, Z, n, n, cc[0], -ss[0], 0.0, 0.0});
            cur = nxt;
        }
        gemm_t<true, false, false>(c, m, n, k, 1.0, Kb, m, cur, n2, 1.0, Cv, n, false);  // C_vir += K^T R
        if (loose > 0.0 && kmax * aov <= tol) { ret = 1; break; }
    }
    c.t_pd += now_s() - t0;
    return ret;
}

// F <- the occupied rows in ascending order, H <- f (or f e, with ev) F
void scaled_occupied(Ctx& c, const double* ev, double* H) {
    hipLaunchKernelGGL(k_gather, dim3(c.n), dim3(256), 0, c.s, c.n, c.Ct, c.sidx, c.ctl, (int)C_KOCC, c.F);
    chk_launch(c);
    hipLaunchKernelGGL(k_scale_rows, dim3(c.n), dim3(256), 0, c.s, c.n, c.F, c.sidx, c.ftot, ev, c.ctl,
                       (double*)nullptr, H);
    chk_launch(c);
}

// one SCF map vin -> vout (scf_step in scf_kernel.h); the sort's control values
// are posted (!sort_rows) or left for the mixing step's post
int step(Ctx& c, const double* vin, double* vout, int& status, double loose, bool allow_bd, bool sort_rows,
         bool final_step, int* decoupled, bool last) {
    const int n = c.n;
    const xtb_scf_opts& o = c.o;
    int cb_lo = -1, cb_hi = -1;
    if ((allow_bd || final_step) && o.bd_gap_kt > 0.0) {
        const double na = c.nel_a, nb = c.nel_b;
        const int ia = (int)rint(na), ib = (int)rint(nb);
        bool ok = fabs(na - ia) < 1e-12 && fabs(nb - ib) < 1e-12 && ib <= ia;
        const double need = o.bd_gap_kt * fmax(o.kt, 9.5e-4);
        if (ok && ia > 0 && ia < n) ok = c.gap_a >= need;
        if (ok && ib > 0 && ib < n) ok = c.gap_b >= need;
        if (ok) { cb_lo = ib; cb_hi = ia; }
    }
    fock(c, vin);
    int sw = 0;
    bool pd_done = false;
    if (final_step) {
        bool intra = false;
        if (cb_lo >= 0 && cb_lo == cb_hi && o.pd_kmax > 0.0) {
            const int r = pd(c, cb_lo, 0.0, vin);
            intra = r > 0;
            if (r != 0) fock(c, vin);  // F may have served as scratch
        }
        pd_done = intra && !o.orbitals;
        if (pd_done && decoupled) *decoupled = cb_lo;
    } else if (cb_lo >= 0 && cb_lo == cb_hi && o.pd_kmax > 0.0) {
        const int r = pd(c, cb_lo, loose, vin);
        pd_done = r > 0;
        if (r < 0) fock(c, vin);
    }
    if (pd_done) {
        ++c.pd_steps;
    } else {
        // A = C F C^T: T = F C^T, A = C T (symmetric) into F
        gemm_t<false, true, false>(c, n, n, n, 1.0, c.F, n, c.Ct, n, 0.0, c.T, n, false);
        gemm_sym<false, false>(c, n, n, c.Ct, n, c.T, n, c.F, n);
        sw = eig(c, o.jacobi_tol, loose);
    }
    if (sw < 0 && final_step) status |= XTB_MOL_JACOBI;
    // sort, Fermi occupations, frontier gaps, occupied prefix
    sort_fermi(c, sort_rows ? NO_POST : next_post(c));
    // density P = C_occ^T diag(f) C_occ in ascending order.  Which rows the
    // sort moved and how many are occupied stays on the device.
    if (sort_rows) {
        // the orbitals' rows into ascending order
        hipLaunchKernelGGL(k_gather, dim3(n), dim3(256), 0, c.s, n, c.Ct, c.sidx, c.ctl, (int)C_PERM, c.F);
        chk_launch(c);
        hipLaunchKernelGGL(k_scale_rows, dim3(n), dim3(256), 0, c.s, n, c.F, c.sidx, c.ftot, (const double*)nullptr,
                           c.ctl, c.Ct, c.T);
        chk_launch(c);
    } else {
        scaled_occupied(c, nullptr, c.T);
    }
    gemm_sym<true, false>(c, n, 0, sort_rows ? c.Ct : c.F, n, c.T, n, c.P, n, c.ctl + C_KOCC);
    // Mulliken charges, shell/atom charges, ES2 + ES3 potential
    const xtb_batch* b = c.b;
    hipLaunchKernelGGL(k_mulliken, dim3((n + NWAVE - 1) / NWAVE), dim3(NT), 0, c.s, n, c.nao, c.P, c.S, c.H0, b->n0,
                       last ? 1 : 0, c.st->q, c.st->eorb);
    chk_launch(c);
    hipLaunchKernelGGL(k_potential, dim3((c.nsh + NWAVE - 1) / NWAVE), dim3(NT), sizeof(double) * c.nsh, c.s, c.nsh,
                       b->sh_ao, b->sh_us, c.par->us_l, b->atom_sh0, b->atom_nsh, c.st->q, c.gam, b->sh_atom,
                       b->atom_sp, c.par->sp_gam3, c.st->qsh, c.qat, c.gq, vout);
    chk_launch(c);
    return sw < 0 ? 0 : sw;
}

// takes the values of a step's sort
bool read_step(Ctx& c, int& status) {
    if (!read_ctl(c)) return false;
    if (c.h[C_FOK] == 0.0) status |= XTB_MOL_FERMI;
    c.gap_a = c.h[C_GAPA];
    c.gap_b = c.h[C_GAPB];
    return true;
}

bool mix(Ctx& c, Mixer& mx, Broyden& bm, const double* xnew, const double* xold, double* xout, double* resid,
         int& status) {
    hipLaunchKernelGGL(k_mix, dim3(1), dim3(NT), 0, c.s, mx, bm, c.n, c.o, c.st->hist_x, c.st->hist_f, xnew, xold,
                       xout, c.ctl, next_post(c));
    chk_launch(c);
    if (!read_step(c, status)) return false;
    // the kernel's own copy of the mixer advanced the same way
    if (c.o.mixer == 1) {
        bm.step += 1;
        bm.rank = (int)c.h[C_BRANK];
        bm.dxnorm = c.h[C_BDX];
    } else {
        mx.step += 1;
        mx.head = (mx.head - 1 + mx.G) % mx.G;
    }
    *resid = c.h[C_RESID];
    return c.h[C_CONV] != 0.0;
}

}  // namespace

extern "C" int32_t xtb_scf_large_workspace(const xtb_batch* batch, int64_t* doubles) {
    if (!batch || !doubles || batch->nmol != 1) return XTB_EINVAL;
    if (batch->max_n > LARGE_MAX_N) return XTB_ETOOBIG;
    *doubles = (int64_t)make_layout(batch->max_n, batch->max_nsh, batch->max_nat).total;
    return XTB_OK;
}

extern "C" int32_t xtb_scf_large(const xtb_batch* batch, const xtb_params* par, const double* S, const double* H0,
                                 const double* gamma, const xtb_scf_opts* opts, const xtb_scf_state* state,
                                 double* work, int64_t work_doubles, void* stream) {
    if (!batch || !par || !S || !H0 || !gamma || !opts || !state || !work) return XTB_EINVAL;
    if (batch->nmol != 1 || batch->max_n <= 0 || batch->has_padding) return XTB_EINVAL;
    if (batch->max_n > LARGE_MAX_N) return XTB_ETOOBIG;
    if (opts->mixer != 0 && opts->mixer != 1) return XTB_EINVAL;
    if (opts->generations < 1 || opts->generations > (opts->mixer == 1 ? BROYDEN_MAXR : MIX_MAXG))
        return XTB_EINVAL;
    if (opts->jacobi_inner < 1 || opts->jacobi_inner > 20 || opts->eig_inexact < 0.0) return XTB_EINVAL;
    if (!state->F || !state->C || !state->T || !state->P || !state->pot || !state->vnew || !state->q ||
        !state->eorb || !state->emo || !state->occ || !state->hist_x || !state->hist_f || !state->qsh ||
        !state->out)
        return XTB_EINVAL;
    const Layout L = make_layout(batch->max_n, batch->max_nsh, batch->max_nat);
    if (work_doubles < (int64_t)L.total) return XTB_EINVAL;
    const double tstart = now_s();
    Ctx c;
    c.s = (hipStream_t)stream;
    MailLease lease;
    if (lease.open() != hipSuccess) return XTB_EHIP;
    c.mail = &lease.mail;
    c.b = batch;
    c.par = par;
    c.o = *opts;
    c.st = state;
    c.n = batch->max_n;
    c.nao = batch->max_n;
    c.nsh = batch->max_nsh;
    c.nat = batch->max_nat;
    const int nb = (c.n + JB - 1) / JB;
    c.nb2 = nb + (nb & 1);
    c.npair = c.nb2 / 2;
    c.S = S;
    c.H0 = H0;
    c.gam = gamma;
    c.F = state->F;
    c.Ct = state->C;
    c.T = state->T;
    c.P = state->P;
    c.E = work + L.E;
    c.Qbuf = work + L.Q;
    c.ev = work + L.ev;
    c.skey = work + L.skey;
    c.ftot = work + L.ftot;
    c.sidx = reinterpret_cast<int*>(work + L.sidx);
    c.ident = reinterpret_cast<int*>(work + L.ident);
    c.part = work + L.part;
    c.ctl = work + L.ctl;
    c.qat = work + L.qat;
    c.gq = work + L.gq;
    static bool attr = false;
    if (!attr) {
        chk(c, hipFuncSetAttribute((const void*)k_fermi, hipFuncAttributeMaxDynamicSharedMemorySize,
                                   (int)fermi_lds(LARGE_MAX_N)));
        attr = true;
    }
    double nel[2] = {0.0, 0.0};
    double prev_status = 1.0;  // a warm start needs a previous call that succeeded
    chk(c, hipMemcpyAsync(nel, batch->mol_nel, sizeof(nel), hipMemcpyDeviceToHost, c.s));
    if (opts->warm_start)
        chk(c, hipMemcpyAsync(&prev_status, state->out + XTB_OUT_STATUS, sizeof(double), hipMemcpyDeviceToHost,
                              c.s));
    chk(c, hipStreamSynchronize(c.s));
    if (c.err != hipSuccess) return XTB_EHIP;
    c.nel_a = nel[0];
    c.nel_b = nel[1];
    c.ia = (int)rint(nel[0]);
    c.ib = (int)rint(nel[1]);
    double* out = state->out;
    int status = 0;
    Rec rec;
    rec.mask = 0u;
    auto put = [&](int slot, double v) {
        rec.v[slot] = v;
        rec.mask |= 1u << slot;
    };
    // nothing may post to the lent box after the call
    auto fail = [&]() {
        (void)hipStreamSynchronize(c.s);
        return XTB_EHIP;
    };
    // warm start from the orbitals and potential a previous call on this
    // state left (a failed re-orthonormalisation starts cold)
    bool warm = opts->warm_start != 0 && prev_status == 0.0;
    if (warm) warm = warm_orthonormalise(c, state->pot);
    const bool ok_ortho = warm || (opts->ortho == 1 ? ortho_chol(c) : ortho(c));
    const double t_ortho = now_s() - tstart;
    if (c.err != hipSuccess) return fail();
    if (!ok_ortho) {
        status |= XTB_MOL_OVERLAP;
        for (int k = 0; k < XTB_OUT_STRIDE; ++k)
            if (k != XTB_OUT_EREP) put(k, 0.0);
        put(XTB_OUT_ESCF, NAN);
        put(XTB_OUT_STATUS, (double)status);
        hipLaunchKernelGGL(k_put, dim3(1), dim3(XTB_OUT_STRIDE), 0, c.s, out, rec);
        chk_launch(c);
        return c.err == hipSuccess ? XTB_OK : fail();
    }
    const int n = c.n;
    if (!warm) chk(c, hipMemsetAsync(state->pot, 0, sizeof(double) * n, c.s));
    const xtb_scf_opts& o = c.o;
    Mixer mx{0, 0, o.generations + 1, !warm && o.soft_start != 0};
    Broyden bm{0, 0, o.generations, 0.0};
    const bool use_broyden = o.mixer == 1;
    int iters = 0, sweeps = 0;
    double resid = 1e-2;
    // first step: a cold start diagonalises to first_tol; a warm start
    // decouples to 1e-2 of that
    const double loose0 = o.eig_inexact > 0.0 ? (warm ? 1e-2 * o.first_tol : o.first_tol) : 0.0;
    const int sw_first = step(c, state->pot, state->vnew, status, loose0, warm && o.eig_inexact > 0.0, true, false,
                              nullptr, false);
    sweeps += sw_first;
    ++iters;
    if (o.mix_guess || use_broyden) {
        mix(c, mx, bm, state->vnew, state->pot, state->pot, &resid, status);
    } else {
        chk(c, hipMemcpyAsync(state->pot, state->vnew, sizeof(double) * n, hipMemcpyDeviceToDevice, c.s));
        hipLaunchKernelGGL(k_post, dim3(1), dim3(WAVE), 0, c.s, c.ctl, next_post(c));
        chk_launch(c);
        read_step(c, status);
    }
    bool converged = false;
    for (int it = 0; it < o.maxiter && c.err == hipSuccess; ++it) {
        // fractional occupations near the Fermi level tighten the inexact
        // eigensolve by 2 kT (as in scf_kernel.h)
        const double soft = c.h[C_FSOFT] > 1e-6 ? fmin(1.0, 2.0 * o.kt) : 1.0;
        sweeps += step(c, state->pot, state->vnew, status, o.eig_inexact * resid * soft, o.eig_inexact > 0.0,
                       true, false, nullptr, false);
        ++iters;
        if (mix(c, mx, bm, state->vnew, state->pot, state->pot, &resid, status)) {
            converged = true;
            break;
        }
    }
    if (use_broyden) {
        // the final density comes from the root search's result (in pot)
        chk(c, hipMemcpyAsync(state->vnew, state->pot, sizeof(double) * n, hipMemcpyDeviceToDevice, c.s));
    }
    if (!converged && o.maxiter > 0) status |= XTB_MOL_MAXITER;
    int kdec = 0;
    const int sw_last = step(c, state->vnew, state->pot, status, 0.0, false, false, o.eig_inexact > 0.0, &kdec, true);
    sweeps += sw_last;
    read_step(c, status);
    hipLaunchKernelGGL(k_energies, dim3(1), dim3(NT), 0, c.s, n, c.nao, c.nsh, c.nat, state->eorb, state->qsh, c.gq,
                       c.qat, batch->atom_sp, par->sp_gam3, state->occ, o.kt, out);
    chk_launch(c);
    hipLaunchKernelGGL(k_copy_emo, dim3((n + 255) / 256), dim3(256), 0, c.s, n, c.skey, kdec > 0 ? 1 : 0,
                       state->emo);
    chk_launch(c);
    if (o.want_w && kdec > 0) {
        // W = C_occ^T A' C_occ with A = C_occ F C_occ^T, A'_ij = (f_i + f_j)/2 A_ij
        // (the final step's input potential; rows not reordered)
        const int k = kdec;
        fock(c, state->vnew);
        gemm_t<false, false, false>(c, k, n, n, 1.0, c.Ct, n, c.F, n, 0.0, c.T, n, false);
        gemm_t<false, true, false>(c, k, k, n, 1.0, c.T, n, c.Ct, n, 0.0, c.F, k, false);
        hipLaunchKernelGGL(k_scale_pairs, dim3(k), dim3(256), 0, c.s, k, c.F, c.ftot);
        chk_launch(c);
        double* R = c.F + (size_t)k * k;
        gemm_t<false, false, false>(c, k, n, k, 1.0, c.F, k, c.Ct, n, 0.0, R, n, false);
        gemm_sym<true, false>(c, n, k, c.Ct, n, R, n, c.T, n);
    } else if (o.want_w) {
        // W = C diag(f e) C^T over the occupied orbitals in ascending order
        scaled_occupied(c, c.ev, c.E);
        gemm_sym<true, false>(c, n, 0, c.F, n, c.E, n, c.T, n, c.ctl + C_KOCC);
    }
    chk(c, hipStreamSynchronize(c.s));
    put(XTB_OUT_ITER, (double)iters);
    put(XTB_OUT_STATUS, (double)status);
    put(XTB_OUT_EFERMI_A, c.h[C_EFA]);
    put(XTB_OUT_EFERMI_B, c.h[C_EFB]);
    put(XTB_OUT_SWEEPS, (double)sweeps);
    put(XTB_OUT_T_ORTHO, t_ortho * 1e6);
    put(XTB_OUT_T_EIGEN, (c.t_eig + c.t_pd) * 1e6);
    put(XTB_OUT_T_PD, c.t_pd * 1e6);
    put(XTB_OUT_PD_STEPS, (double)c.pd_steps);
    put(XTB_OUT_SWEEPS_FIRST, (double)sw_first);
    put(XTB_OUT_SWEEPS_LAST, (double)sw_last);
    put(XTB_OUT_T_TOTAL, (now_s() - tstart) * 1e6);
    hipLaunchKernelGGL(k_put, dim3(1), dim3(XTB_OUT_STRIDE), 0, c.s, out, rec);
    chk_launch(c);
    if (c.err != hipSuccess) return fail();
    // the state's orbital buffer holds the orbitals, whichever buffer they
    // ended in
    if (c.Ct != state->C) {
        chk(c, hipMemcpyAsync(state->C, c.Ct, sizeof(double) * n * n, hipMemcpyDeviceToDevice, c.s));
    }
    return c.err == hipSuccess ? XTB_OK : fail();
}
