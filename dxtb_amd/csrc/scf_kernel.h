// Persistent per-molecule GFN1 SCF on gfx950: one workgroup owns one
// molecule and runs its whole self-consistent cycle without returning to
// the host.  Follows upstream's default ("full") SCF in potential mode
// (src/dxtb/_src/scf/unrolling/default.py:71-140, scf/base.py:651-907):
//
//   v -> F = H0 - 1/2 S o (v_i + v_j)           (Fock build)
//     -> F C = S C e                             (generalized eigensolve)
//     -> f = Fermi(e), P = C diag(f) C^T         (smearing, density)
//     -> q = n0 - diag(P S), e_orb = diag(P H0)  (Mulliken)
//     -> v' = spread(gamma q_sh + hd q_at^2)     (ES2 + ES3 potential)
//   mixed with upstream's Anderson mixer (scf/mixer/anderson.py:163-317).
//
// Eigensolver: the generalized problem is reduced once per geometry with the
// Cholesky factor of S (or the Loewdin S^-1/2 by coupled Newton-Schulz) on
// matrix cores.  Every SCF step transforms F into the basis of the previous
// step's orbitals, A = C^T F C, which is close to diagonal, and finishes it
// with a few sweeps of parallel-ordered cyclic Jacobi whose rotations are
// applied to the stored orbitals: with A in LDS whenever it fits, by block
// Jacobi in memory otherwise.
#pragma once

#include "scf_core.h"

namespace xtb {

struct Lay {
    // LDS layout in doubles (offsets), identical on host and device
    int red, ctx, cs, skey, sidx, ev, ftot, qsh, vsh, gq, qat, big, total_fixed;
};

typedef __attribute__((address_space(1))) int glbi;
typedef __attribute__((address_space(3))) uint32_t ldsu;

struct Mol {
    int m, n, nao, nsh, nat, vec0, sh0, at0;
    size_t mat0, gam0;
    const glbf *S, *H0, *gam;
    glbf *F, *Ct, *T, *P;
    glbf *pot, *vnew, *q, *eorb, *emo, *occ, *qsh_out;
    const glbf *n0, *sp_gam3;                 // reference occupations; third-order parameters
    const glbi *sh_ao, *sh_us, *us_l, *sh_atom, *ao_sh, *atom_sh0, *atom_nsh, *atom_sp;
    double nel_a, nel_b;
    int nvec_total;
};

struct Shared {
    ldsf *red, *cs, *skey, *ev, *ftot, *qsh, *vsh, *gq, *qat, *big;
    ldsi* sidx;
    int big_cap;
    ldsf* tacc;  // stage timers (thread 0)
};

// The padding orbitals of a padded layout have a unit overlap diagonal, zero
// H0 and zero potential: they stay exact eigenvectors at energy 0, coupled to
// nothing.  Between the steps the orbitals' rows are the nr real ones in
// ascending order, then the padding, so that every product of a step runs
// over nr rows and columns.  An eigensolve pairs rows by their place in the
// whole spectrum, padding included (the place decides which rotations
// precede which); for it the padding rows move to row p0, behind the real
// ones of negative energy.  Without padding (or when the state is kept for
// the next call) nr = n.
struct Pad {
    int nr;   // real orbitals
    int at;   // first padding row: nr, or p0
    int p0;   // where they belong in the whole spectrum
};

#ifdef XTB_PD_TIMERS
// phases of the perturbative step (instrumented builds only)
#define PD_MARK(sh, i, t)                                                   \
    do {                                                                    \
        const double t_ = now_us();                                         \
        if (threadIdx.x == 0) (sh).red[RED_DOUBLES - 12 + (i)] += t_ - (t); \
        (t) = t_;                                                           \
    } while (0)
#else
#define PD_MARK(sh, i, t) do { } while (0)
#endif

struct FusedArgs {
    const double* pos;
    double* cn;
    double* S;
    double* H0;
    double* gam;
    double* dedcn;
    double* grad;
};

// The kernels' only argument, at the start of the kernel argument segment:
// functions read what they need of it by scalar loads from there.
struct ScfArgs {
    xtb_batch b;
    xtb_params par;
    const double *S, *H0, *gam;
    xtb_scf_opts o;
    xtb_scf_state st;
    FusedArgs fa;
    int big_cap;
};
typedef const __attribute__((address_space(4))) ScfArgs kargs;

// What the out-of-line functions of a molecule share, in LDS; they take it to
// scalar registers on entry.  By reference it lived in the stack frame, read
// by scratch loads at every use: a 20-orbital energy took 653 us in the
// kernel instead of 533, octane's energy and forces 1874 instead of 1725.
struct Ctx {
    Mol M;
    Shared sh;
    Pad pad;
    int since;  // perturbative steps since the virtual energies were formed (0: never)
    kargs* ka;
    double tacc[12];
};
constexpr int CTX_DOUBLES = 64;
static_assert(sizeof(Ctx) <= 8 * CTX_DOUBLES, "context in LDS");

template <class T>
__device__ __forceinline__ T ctx_load(const ldsf* ctx, size_t off) {
    static_assert(sizeof(T) % 4 == 0, "whole words");
    uint32_t v[sizeof(T) / 4];
    const ldsu* p = (const ldsu*)ctx + off / 4;
#pragma unroll
    for (unsigned i = 0; i < sizeof(T) / 4; ++i) v[i] = __builtin_amdgcn_readfirstlane(p[i]);
    T y;
    __builtin_memcpy(&y, v, sizeof(T));
    return y;
}
template <class T>
__device__ __forceinline__ void ctx_store(ldsf* ctx, size_t off, const T& x) {
    uint32_t v[sizeof(T) / 4];
    __builtin_memcpy(v, &x, sizeof(T));
    ldsu* p = (ldsu*)ctx + off / 4;
#pragma unroll
    for (unsigned i = 0; i < sizeof(T) / 4; ++i) p[i] = v[i];
}
#define CTX_GET(ctx, m) ctx_load<decltype(Ctx::m)>(ctx, offsetof(Ctx, m))
#define CTX_PUT(ctx, m, x) ctx_store<decltype(Ctx::m)>(ctx, offsetof(Ctx, m), x)

template <class T>
__device__ __forceinline__ T karg_load(const __attribute__((address_space(4))) T* x) {
    uint32_t v[sizeof(T) / 4];
    const __attribute__((address_space(4))) uint32_t* p = (const __attribute__((address_space(4))) uint32_t*)x;
#pragma unroll
    for (unsigned i = 0; i < sizeof(T) / 4; ++i) v[i] = p[i];
    T y;
    __builtin_memcpy(&y, v, sizeof(T));
    return y;
}

__host__ __device__ inline int next_pow2(int v) {
    int p = 1;
    while (p < v) p <<= 1;
    return p;
}

constexpr int LDS_DOUBLES = 160 * 1024 / 8;  // of a CU
static_assert((RING_MAX_N + 1) * (RING_MAX_N + 2) / 2 > LDS_DOUBLES, "a matrix that fits the LDS fits the rounds");

// (skey and sidx are rounded up to a power of two: between 184 and 202 orbitals
// the slack is part of the line between the LDS and the block Jacobi)
__host__ __device__ inline Lay make_lay(int nmax, int max_nsh, int max_nat) {
    Lay L;
    const int npow = next_pow2(nmax < 2 ? 2 : nmax);
    int o = 0;
    L.red = o; o += RED_DOUBLES;
    L.ctx = o; o += CTX_DOUBLES;
    L.cs = o; o += 3 * ((nmax < RING_MAX_N ? nmax : RING_MAX_N) / 2 + 2);  // (LDS Jacobi only)
    L.skey = o; o += npow;
    L.sidx = o; o += (npow + 1) / 2;  // ints
    L.ev = o; o += nmax;
    L.ftot = o; o += nmax;
    L.qsh = o; o += max_nsh;
    L.vsh = o; o += max_nsh;
    L.gq = o; o += max_nsh;
    L.qat = o; o += max_nat;
    o = (o + 1) & ~1;
    L.big = o;
    L.total_fixed = o;
    return L;
}

// ---------------------------------------------------------------------------
// eigen step: A (full, in mol.F) -> eigenvalues in sh.ev, rotations applied
// to mol.Ct.  Returns Jacobi sweeps (-1 on failure).
// ---------------------------------------------------------------------------
__device__ __noinline__ int eig_step(const ldsf* ctx, double loose, int cb_lo, int cb_hi, bool intra) {
    const Mol M = CTX_GET(ctx, M);
    const Shared sh = CTX_GET(ctx, sh);
    const xtb_scf_opts o = karg_load(&CTX_GET(ctx, ka)->o);
    const Pad pad = CTX_GET(ctx, pad);
    const int n = M.n, npad = n - pad.nr, max_sweeps = o.jacobi_max_sweeps, inner = o.jacobi_inner;
    const double rel_tol = o.jacobi_tol;
    loose = uniform_copy(loose);
    // scale for the absolute tolerance
    double dmax = 0.0;
    for (int i = threadIdx.x; i < n; i += NT) dmax = fmax(dmax, fabs(M.F[(size_t)i * n + i]));
    dmax = wg_max(dmax, sh.red);
    const double tol = fmax(fmax(rel_tol * fmax(dmax, 1.0), loose), JACOBI_TOL_MIN);
    const int npk = n * (n + 1) / 2;
    int sweeps;
    if (npk <= sh.big_cap) {
        // T is free scratch here and holds a sweep's recorded rotations
        sweeps = wg_jacobi(M.F, n, sh.big, ring_pitch(n, sh.big_cap), M.Ct, n, M.nao, M.T, max_sweeps, tol, sh.cs,
                           sh.red, sh.ev, cb_lo, cb_hi, intra);
    } else {
        // block Jacobi; T is free scratch here and holds the subproblem rotations
        sweeps = wg_block_jacobi(M.F, n, RowsGlobal{M.Ct, n}, M.nao, pad.at, pad.at + npad, M.T, max_sweeps, tol,
                                 sh.big, sh.red, sh.tacc, inner, cb_lo, cb_hi, intra);
        for (int i = threadIdx.x; i < n; i += NT) sh.ev[i] = M.F[(size_t)i * n + i];
    }
    __syncthreads();
    return sweeps;
}

// Loewdin orthogonaliser Ct <- X = S^-1/2 (symmetric, so rows == columns) by
// the coupled Newton-Schulz iteration on matrix cores:
//   Y0 = S/c, Z0 = I;  T = (3I - Z Y)/2;  Y <- Y T;  Z <- T Z
// Y -> (S/c)^1/2 and Z -> (S/c)^-1/2 quadratically once ||I - S/c|| < 1; c is a
// Gershgorin bound on the largest eigenvalue of S.  X = Z / sqrt(c).
__device__ __noinline__ int ortho_setup(const ldsf* ctx, int* status) {
    const Mol M = CTX_GET(ctx, M);
    const Shared sh = CTX_GET(ctx, sh);
    const int n = M.n;
    const size_t nn = (size_t)n * n;
    double rs = 0.0;
    for (int i = threadIdx.x; i < n; i += NT) {
        double a = 0.0;
        for (int j = 0; j < n; ++j) a += fabs(M.S[(size_t)i * n + j]);
        rs = fmax(rs, a);
    }
    const double c = wg_max(rs, sh.red) * 1.0001;
    glbf* Y = M.F;
    glbf* Z = M.Ct;
    glbf* T = M.T;
    glbf* W = M.P;
    const int w = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
    for (int r = w; r < n; r += NWAVE)
        for (int q = lane; q < n; q += WAVE) {
            const size_t e = (size_t)r * n + q;
            Y[e] = M.S[e] / c;
            Z[e] = (r == q) ? 1.0 : 0.0;
        }
    __syncthreads();
    int it = 0;
    int extra = -1;  // iterations left once in the quadratic regime
    for (; it < 60; ++it) {
        gemm<false, false>(n, n, n, -0.5, Z, n, Y, n, 0.0, T, n, sh.big);  // -(Z Y)/2
        double err = 0.0;
        for (int r = w; r < n; r += NWAVE)
            for (int q = lane; q < n; q += WAVE) {
                const size_t e = (size_t)r * n + q;
                const double v = T[e] + ((r == q) ? 1.5 : 0.0);
                err = fmax(err, fabs(v - ((r == q) ? 1.0 : 0.0)));
                T[e] = v;
            }
        err = wg_max(err, sh.red);
        if (extra == 0 || err < 1e-15) break;
        if (extra > 0) --extra;
        else if (err < 1e-9) extra = 1;  // quadratic: one more step reaches rounding level
        gemm<false, false>(n, n, n, 1.0, Y, n, T, n, 0.0, W, n, sh.big);  // Y T
        gemm<false, false>(n, n, n, 1.0, T, n, Z, n, 0.0, Y, n, sh.big);  // T Z (into Y's buffer)
        // rotate buffers: Y <- W, Z <- (T Z) held in Y's buffer
        glbf* oldZ = Z;
        Z = Y;
        Y = W;
        W = oldZ;
    }
    if (it >= 60) *status |= XTB_MOL_OVERLAP;  // S numerically singular
    const double sc = 1.0 / sqrt(c);
    for (size_t e = threadIdx.x; e < nn; e += NT) M.Ct[e] = Z[e] * sc;  // Z may alias Ct
    __syncthreads();
    // symmetrise (rounding)
    for (int r = w; r < n; r += NWAVE)
        for (int q = r + 1 + lane; q < n; q += WAVE) {
            const size_t e = (size_t)r * n + q;
            const double a = 0.5 * (M.Ct[e] + M.Ct[(size_t)q * n + r]);
            M.Ct[e] = a;
            M.Ct[(size_t)q * n + r] = a;
        }
    __syncthreads();
    return 0;
}

// ---------------------------------------------------------------------------
// Orthogonaliser from the Cholesky factor S = L L^T: the rows of X = L^-1 are
// S-orthonormal (X S X^T = I), so Ct <- X starts the SCF like the Loewdin
// X = S^-1/2 does (eigenpairs of the generalised problem do not depend on the
// choice), at about n^3 flops instead of Newton-Schulz's ~10 x 6 n^3.
// Blocked right-looking factorisation with 32-wide panels in T (lower
// triangle): each diagonal block is factored and inverted by one wave
// (chol_block); the panel below (x D^T = b, i.e. x = b D^-T) and the trailing update
// are matrix-core GEMMs.  X follows by block forward substitution L X = I:
// X_i = D_i^-1 (E_i - L_i,<i X_<i), again with GEMMs.  A block padded beyond
// n is the identity.  Scratch: F (up to 32 x n, or mt x 32 with stride n),
// P (the nb x nb inverse, stride nb).
// Returns 0; a non-positive pivot (S not positive definite, where upstream's
// torch.linalg.cholesky raises) sets XTB_MOL_OVERLAP in *status.
// ---------------------------------------------------------------------------
// In-place blocked right-looking Cholesky L L^T = A of the n x n symmetric
// positive definite A (leading dimension ld; lower triangle read and overwritten by L; the strict
// upper triangle is left as it was), 32-wide panels: one wave factors and
// inverts each diagonal block, the panel solve and the trailing update are
// matrix-core GEMMs.  R (>= n rows x 32, leading dimension ld) is
// global scratch; the inverse of block j0's factor goes to Dg + 32 j0
// (leading dimension its width; n x 32 doubles, n x n for n < 32).  Returns
// false when a pivot is not positive.
__device__ __noinline__ bool chol_factor(glbf* L, int n, int ld, glbf* R, glbf* Dg, ldsf* big) {
    L = uniform(L);
    n = uniform(n);
    ld = uniform(ld);
    R = uniform(R);
    Dg = uniform(Dg);
    constexpr int NB = 32;
    const int w = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
    bool bad = false;
    for (int j0 = 0; j0 < n; j0 += NB) {
        const int nb = n - j0 < NB ? n - j0 : NB;
        glbf* D = Dg + (size_t)j0 * NB;
        if (w == 0 && !chol_block(L + (size_t)j0 * ld + j0, ld, nb, D)) bad = true;
        __syncthreads();
        const int mt = n - j0 - nb;
        if (mt > 0) {
            glbf* Pn = L + (size_t)(j0 + nb) * ld + j0;  // panel below the block
            gemm<false, true>(mt, nb, nb, 1.0, Pn, ld, D, nb, 0.0, R, ld, big);  // b D^-T
            for (int r = w; r < mt; r += NWAVE)
                for (int c = lane; c < nb; c += WAVE) Pn[(size_t)r * ld + c] = R[(size_t)r * ld + c];
            __syncthreads();
            gemm<false, true>(mt, mt, nb, -1.0, Pn, ld, Pn, ld, 1.0, Pn + nb, ld, big);
        }
    }
    return !__syncthreads_or(bad);
}

// Cholesky orthogonaliser: L L^T = S, Ct <- X = L^-1 (rows S-orthonormal).
// X by block rows, X_i = D_i^-1 (E_i - L_i,<i X_<i), where only the first
// i0 + nb columns of block row i are non-zero.  L in T, R in F, Dg in P.
__device__ __noinline__ int chol_setup(const ldsf* ctx, int* status) {
    const Mol M = CTX_GET(ctx, M);
    const Shared sh = CTX_GET(ctx, sh);
    constexpr int NB = 32;
    const int n = M.nao, ld = M.n;  // (padding: unit rows and columns)
    const int w = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
    glbf* L = M.T;
    glbf* X = M.Ct;
    glbf* R = M.F;   // NB x n (and mt x NB) scratch
    glbf* Dg = M.P;  // inverses of the diagonal blocks
    for (int r = w; r < n; r += NWAVE)
        for (int c = lane; c < n; c += WAVE) L[(size_t)r * ld + c] = M.S[(size_t)r * ld + c];
    __syncthreads();
    if (!chol_factor(L, n, ld, R, Dg, sh.big)) *status |= XTB_MOL_OVERLAP;
    for (int r = w; r < ld; r += NWAVE)
        for (int c = lane; c < ld; c += WAVE) X[(size_t)r * ld + c] = r == c && r >= n ? 1.0 : 0.0;
    __syncthreads();
    for (int i0 = 0; i0 < n; i0 += NB) {
        const int nb = n - i0 < NB ? n - i0 : NB;
        if (i0 > 0) gemm<false, false>(nb, i0, i0, -1.0, L + (size_t)i0 * ld, ld, X, ld, 0.0, R, ld, sh.big);
        for (int e = threadIdx.x; e < nb * nb; e += NT) {
            const int r = e / nb, c = e % nb;
            R[(size_t)r * ld + i0 + c] = (r == c) ? 1.0 : 0.0;
        }
        __syncthreads();
        gemm<false, false>(nb, i0 + nb, nb, 1.0, Dg + (size_t)i0 * NB, nb, R, ld, 0.0, X + (size_t)i0 * ld, ld, sh.big);
    }
    return 0;
}

// Warm start: the kept orbitals (rows of Ct, S_old-orthonormal, ascending
// energy) are re-orthonormalised against the new overlap by Cholesky
// Gram-Schmidt in their order, C <- L^-1 C with G = C S C^T = L L^T, so the
// lowest orbitals stay within the span of the lowest kept ones.  G and L in
// P, C S and Dg in T, R in F; the forward substitution C_i <- D_i^-1 (C_i -
// L_i,<i C_<i) runs in place by block rows.  Returns false (Ct unusable,
// start cold) when G is not numerically positive definite.
__device__ __noinline__ bool warm_orthonormalise(const ldsf* ctx) {
    const Mol M = CTX_GET(ctx, M);
    const Shared sh = CTX_GET(ctx, sh);
    constexpr int NB = 32;
    const int n = M.n;
    const int w = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
    glbf* G = M.P;
    glbf* R = M.F;
    glbf* Dg = M.T;
    gemm<false, false>(n, n, n, 1.0, M.Ct, n, M.S, n, 0.0, M.T, n, sh.big);  // C S
    gemm_sym<false, true>(n, n, 1.0, M.T, n, M.Ct, n, G, n, sh.big);         // C S C^T
    if (!chol_factor(G, n, n, R, Dg, sh.big)) return false;
    for (int i0 = 0; i0 < n; i0 += NB) {
        const int nb = n - i0 < NB ? n - i0 : NB;
        glbf* Ci = M.Ct + (size_t)i0 * n;
        for (int r = w; r < nb; r += NWAVE)
            for (int c = lane; c < n; c += WAVE) R[(size_t)r * n + c] = Ci[(size_t)r * n + c];
        __syncthreads();
        if (i0 > 0) gemm<false, false>(nb, n, i0, -1.0, G + (size_t)i0 * n, n, M.Ct, n, 1.0, R, n, sh.big);
        gemm<false, false>(nb, n, nb, 1.0, Dg + (size_t)i0 * NB, nb, R, n, 0.0, Ci, n, sh.big);
    }
    return true;
}

// ---------------------------------------------------------------------------
// Orbitals in ascending energy order for the density products.  The
// orbitals with f > 0 form a prefix of length kocc; G[j] = C_{sidx[j]} (row
// j, for j < kocc, or j < rows when `all_rows`; rows columns) and H[j] = w_j
// G[j] (j < kocc, cols columns)
// with w = f (or f e when `with_e`).  H may alias Ct: it is written only
// after every row of G has been gathered.
// ---------------------------------------------------------------------------
__device__ __noinline__ void gather_occupied(const ldsf* ctx, glbf* G, glbf* H, int rows, int cols, int kocc, bool with_e,
                                             bool all_rows = false) {
    const Mol M = CTX_GET(ctx, M);
    const Shared sh = CTX_GET(ctx, sh);
    const int n = M.n;
    G = uniform(G);
    H = uniform(H);
    rows = uniform(rows);
    cols = uniform(cols);
    kocc = uniform(kocc);
    const int w = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
    for (int j = w; j < (all_rows ? rows : kocc); j += NWAVE) {
        const glbf* src = M.Ct + (size_t)sh.sidx[j] * n;
        for (int c = lane; c < rows; c += WAVE) G[(size_t)j * n + c] = src[c];
    }
    __syncthreads();
    for (int j = w; j < kocc; j += NWAVE) {
        const int o = sh.sidx[j];
        const double f = with_e ? sh.ftot[o] * sh.ev[o] : sh.ftot[o];
        for (int c = lane; c < cols; c += WAVE) H[(size_t)j * n + c] = f * G[(size_t)j * n + c];
    }
    __syncthreads();
}

// ---------------------------------------------------------------------------
// Fock build F = H0 - 1/2 S o (v_i + v_j) (scf/base.py:817-859), its leading
// d x d block
// ---------------------------------------------------------------------------
// Streaming passes over rows run four rows per wave at a time, so that each
// lane has the loads of four rows in flight (one row per wave left a CU's
// waves waiting on memory latency at a fraction of its share of HBM);
// rows past the end are clamped to the last row for the loads and skipped
// for the stores.
// (Of the Fock build's nine loads an iteration, the compiler waits for the first
// four, vin[c] among them, before it issues the others: 20.9 GB/s a workgroup
// with all CUs at work, 30.8 when all nine went out together.)
constexpr int ROWS_PER_WAVE = 4;

__device__ inline void fock_build(const Mol& M, const glbf* vin, int d) {
    const int n = M.n;
    const int w = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
    for (int r0 = w * ROWS_PER_WAVE; r0 < d; r0 += NWAVE * ROWS_PER_WAVE) {
        int rr[ROWS_PER_WAVE];
        double vr[ROWS_PER_WAVE];
#pragma unroll
        for (int u = 0; u < ROWS_PER_WAVE; ++u) {
            rr[u] = r0 + u < d ? r0 + u : d - 1;
            vr[u] = vin[rr[u]];
        }
        for (int c = lane; c < d; c += WAVE) {
            const double vc = vin[c];
            double h[ROWS_PER_WAVE], sv[ROWS_PER_WAVE];
#pragma unroll
            for (int u = 0; u < ROWS_PER_WAVE; ++u) {
                h[u] = M.H0[(size_t)rr[u] * n + c];
                sv[u] = M.S[(size_t)rr[u] * n + c];
            }
#pragma unroll
            for (int u = 0; u < ROWS_PER_WAVE; ++u)
                if (r0 + u < d) M.F[(size_t)rr[u] * n + c] = h[u] - 0.5 * sv[u] * (vr[u] + vc);
        }
    }
    __syncthreads();
}

// ---------------------------------------------------------------------------
// Perturbative occupied-virtual decoupling for intermediate SCF steps of
// closed shells with a clear gap (pseudo-diagonalisation in the sense of
// Stewart, Csaszar and Pulay, J. Comput. Chem. 3, 227 (1982), done with
// matrix-core GEMMs).  The rows of Ct are in ascending energy order, the
// first k doubly occupied.  With A = C^T F C (only its occupied rows and the
// diagonal are formed) and e = diag(A), the first-order amplitudes
// K_ia = A_ia / (e_a - e_i) define the antisymmetric generator
// G = [[0, K], [-K^T, 0]]; the orbitals are rotated by exp(G), which is
// exactly orthogonal:
//   C_occ <- cos(sqrt X) C_occ - sinc(sqrt X) Z
//   C_vir <- C_vir + K^T [sinc(sqrt X) C_occ + phi(X) Z]
// with X = K K^T (k x k), Z = K C_vir (k x n), phi(x) = (cos sqrt x - 1)/x;
// the functions of X are power series evaluated by Horner's rule, truncated
// once the next term is below 1e-17, or 1e-13 in inexact steps (||X||_F
// bounds the spectral norm).  Another pass measures the coupling left and
// rotates again (pass limits and exits: PD_INEXACT_PASSES, PD_EXACT_PASSES).
// (pd_applies: the sizes it takes.)
// Returns 1 when done (rotated, or already decoupled to the tolerance), 0 to
// ask for the Jacobi eigensolve with Ct and F untouched, -1 to ask for it
// after F was used as scratch (the caller rebuilds F).  Jacobi is asked for
// when an amplitude exceeds pd_kmax, a denominator is not positive, k > n/2,
// a series would need more than 9 terms, or (exact calls, loose = 0) the
// last measured coupling is above the tolerance.  On return 1, sh.ev holds the
// diagonal of C F C^T in the rows' order (occupied rows: of the last pass).
// Scratch: T holds C F, then X and Z; P the couplings/amplitudes; F the two
// Horner accumulators (k x n each, k <= n/2).  Rows and columns run to d: n,
// or the real orbitals only (the padding's couplings are exact zeros).
// ---------------------------------------------------------------------------
// Coefficients of the series in X = K K^T used by the rotation: term j of
// cos (0): (-1)^j / (2j)!, sinc (1): (-1)^j / (2j+1)!, phi (2): -(-1)^j / (2j+2)!
struct HornerCoef {
    double v[3][9];
    constexpr HornerCoef() : v() {
        double f = 1.0;  // (2j)!
        for (int j = 0; j <= 8; ++j) {
            if (j > 0) f *= (2.0 * j - 1.0) * (2.0 * j);
            const double sg = (j & 1) ? -1.0 : 1.0;
            v[0][j] = sg / f;
            v[1][j] = sg / (f * (2.0 * j + 1.0));
            v[2][j] = -sg / (f * (2.0 * j + 1.0) * (2.0 * j + 2.0));
        }
    }
};
__constant__ const HornerCoef horner_coef;

constexpr int PD_REFRESH = 4;
__device__ inline bool pd_applies(int n, int k) { return k > 0 && n - k > 0 && 2 * k <= n; }

__device__ __noinline__ int pd_step(const ldsf* ctx, int k, double loose, const glbf* vin, int d, bool refresh) {
    const Mol M = CTX_GET(ctx, M);
    const Shared sh = CTX_GET(ctx, sh);
    const xtb_scf_opts o = karg_load(&CTX_GET(ctx, ka)->o);
    k = uniform(k);
    d = uniform(d);
    loose = uniform_copy(loose);
    vin = uniform(vin);
    const int n = M.n, m = d - k;  // n: leading dimension
    const int w = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
    glbf* Ct = M.Ct;
    glbf* Cv = M.Ct + (size_t)k * n;
    glbf* Kb = M.P;  // k x m, leading dimension m
    // Virtual orbital energies only scale the amplitudes: an error of a few
    // SCF steps in them leaves a second-order coupling, so they are formed
    // (all rows of C F) every PD_REFRESH-th perturbative step only; the
    // others reuse the last values (sh.ev, in the rows' order) and form
    // the occupied rows of C F.  Every 4th step costs no SCF iterations on
    // 500-orbital molecules; never refreshing them costs two.
    const int rows = refresh ? d : k;
    double tm = now_us();
    (void)tm;
    const int npass = loose > 0.0 ? PD_INEXACT_PASSES : PD_EXACT_PASSES;
    for (int pass = 0; pass < npass; ++pass) {
        if (pass > 0) fock_build(M, vin, d);
        // T = C F (rows: all, or the occupied ones) and the diagonal of T C^T,
        // the rows' energies; A_ov = T_occ C_vir^T
        gemm_dot(rows, d, d, Ct, n, M.F, n, M.T, n, Ct, sh.ev, sh.big);
        PD_MARK(sh, 0, tm);
        gemm<false, true>(k, m, d, 1.0, M.T, n, Cv, n, 0.0, Kb, m, sh.big);
        PD_MARK(sh, 1, tm);
        for (int a = d + threadIdx.x; a < n; a += NT) sh.ev[a] = 0.0;  // padding
        __syncthreads();
        double dmax = 0.0;
        for (int i = threadIdx.x; i < n; i += NT) dmax = fmax(dmax, fabs(sh.ev[i]));
        double aov = 0.0, kmax = 0.0, dmin = INFINITY;
        for (int i0 = w * ROWS_PER_WAVE; i0 < k; i0 += NWAVE * ROWS_PER_WAVE) {
            int ii[ROWS_PER_WAVE];
            double ei[ROWS_PER_WAVE];
#pragma unroll
            for (int u = 0; u < ROWS_PER_WAVE; ++u) {
                ii[u] = i0 + u < k ? i0 + u : k - 1;
                ei[u] = sh.ev[ii[u]];
                if (d < n) dmin = fmin(dmin, -ei[u]);  // padding orbitals at 0
            }
            for (int a = lane; a < m; a += WAVE) {
                const double ea = sh.ev[k + a];
                double v[ROWS_PER_WAVE];
#pragma unroll
                for (int u = 0; u < ROWS_PER_WAVE; ++u) v[u] = Kb[(size_t)ii[u] * m + a];
#pragma unroll
                for (int u = 0; u < ROWS_PER_WAVE; ++u) {
                    if (i0 + u >= k) continue;
                    const double den = ea - ei[u];
                    const double amp = v[u] / den;
                    aov = fmax(aov, fabs(v[u]));
                    dmin = fmin(dmin, den);
                    kmax = fmax(kmax, fabs(amp));
                    Kb[(size_t)ii[u] * m + a] = amp;
                }
            }
        }
        double mx[4] = {dmax, aov, kmax, -dmin};
        wg_max_n<4>(mx, sh.red);
        aov = mx[1];
        kmax = mx[2];
        dmin = -mx[3];
        const double tol = fmax(o.jacobi_tol * fmax(mx[0], 1.0), loose > 0.0 ? loose : PD_FINAL_REL * o.x_atol_max);
        if (aov <= tol) return 1;  // decoupled: orbitals stay
        const int fail = pass == 0 ? 0 : -1;
        PD_MARK(sh, 2, tm);
        if (!(dmin > 0.0) || !(kmax <= o.pd_kmax)) return fail;
        // an exact call's last pass only measures: a rotation after it
        // would go unchecked
        if (loose == 0.0 && pass == npass - 1) return fail;
        glbf* X = M.T;
        glbf* Z = M.T + (size_t)k * k;
        gemm_sym<false, true>(k, m, 1.0, Kb, m, Kb, m, X, k, sh.big);
        PD_MARK(sh, 3, tm);
        gemm<false, false>(k, d, m, 1.0, Kb, m, Cv, n, 0.0, Z, n, sh.big);
        PD_MARK(sh, 4, tm);
        double xf = 0.0;
        for (int e = threadIdx.x; e < k * k; e += NT) xf = fma(X[e], X[e], xf);
        xf = sqrt(wg_sum(xf, sh.red));
        // highest power J kept: the first omitted cosine term (the largest of
        // the three series) ||X||^(J+1) / (2J+2)! is below 1e-17 in an exact
        // step and below min(1e-13, 1e-3 loose) in an inexact one.  What is
        // left out perturbs orthonormality by that much; over an SCF run it
        // adds up to ~1e-12, far below the results' tolerances
        const double tolj = loose > 0.0 ? fmin(1e-13, fmax(1e-17, 1e-3 * loose)) : 1e-17;
        int J = 0;
        double term = 0.5 * xf;
        while (term > tolj) {
            ++J;
            term *= xf / ((2.0 * J + 1.0) * (2.0 * J + 2.0));
            if (J > 8) return fail;  // F and Ct untouched in this pass
        }
        const double(&cc)[9] = horner_coef.v[0], (&ss)[9] = horner_coef.v[1], (&ph)[9] = horner_coef.v[2];
        // Horner steps acc <- X acc + a_j C_occ + b_j Z, the update fused into
        // the GEMM epilogue; the two k x n halves of F alternate
        glbf* cur = M.F;
        glbf* nxt = M.F + (size_t)k * n;
        // R = sinc(X) C_occ + phi(X) Z
        wg_axpby_rows(k, d, n, ss[J], Ct, ph[J], Z, cur);
        __syncthreads();
        for (int j = J - 1; j >= 0; --j) {
            PD_MARK(sh, 6, tm);
            gemm_epi(k, d, k, X, k, cur, n, nxt, n, Ct, ss[j], Z, ph[j], sh.big);
            PD_MARK(sh, 5, tm);
            glbf* t = cur;
            cur = nxt;
            nxt = t;
        }
        PD_MARK(sh, 6, tm);
        // C_vir += K^T R
        gemm<true, false>(m, d, k, 1.0, Kb, m, cur, n, 1.0, Cv, n, sh.big);
        PD_MARK(sh, 7, tm);
        // C_occ <- cos(X) C_occ - sinc(X) Z.  The last Horner term is written
        // over C_occ itself: each element of C_occ is read (as E1) and
        // written by the same thread, and no product takes C_occ as an
        // operand, so no copy pass follows
        wg_axpby_rows(k, d, n, cc[J], Ct, -ss[J], Z, J == 0 ? Ct : cur);
        __syncthreads();
        for (int j = J - 1; j >= 0; --j) {
            PD_MARK(sh, 6, tm);
            gemm_epi(k, d, k, X, k, cur, n, j == 0 ? Ct : nxt, n, Ct, cc[j], Z, -ss[j], sh.big);
            PD_MARK(sh, 5, tm);
            glbf* t = cur;
            cur = nxt;
            nxt = t;
        }
        PD_MARK(sh, 6, tm);
#ifdef XTB_PD_TIMERS
        if (threadIdx.x == 0) sh.red[RED_DOUBLES - 12 + 9] += (double)J;
#endif
        // inexact steps: the second-order estimate of what is left
        if (loose > 0.0 && kmax * aov <= tol) return 1;
    }
    // the passes spent: good enough for an inexact step (an exact one has
    // returned from its last, measuring pass)
    return 1;
}

// The padding rows to their place in the whole spectrum, for an eigensolve.
// T is scratch.
__device__ __noinline__ void pad_to_spectrum(const ldsf* ctx, Pad pad) {
    const Mol M = CTX_GET(ctx, M);
    const Shared sh = CTX_GET(ctx, sh);
    pad = uniform_copy(pad);
    const int n = M.n, npad = n - pad.nr;
    const int w = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
    auto from = [&](int u) { return u < pad.p0 ? u : (u < pad.p0 + npad ? u - pad.p0 + pad.nr : u - npad); };
    double e[2];
#pragma unroll
    for (int x = 0; x < 2; ++x) {
        const int u = threadIdx.x + x * NT;
        e[x] = u < n ? sh.ev[from(u)] : 0.0;
    }
    for (int u = w; u < n; u += NWAVE) {
        const glbf* src = M.Ct + (size_t)from(u) * n;
        for (int c = lane; c < n; c += WAVE) M.T[(size_t)u * n + c] = src[c];
    }
    __syncthreads();
#pragma unroll
    for (int x = 0; x < 2; ++x) {
        const int u = threadIdx.x + x * NT;
        if (u < n) sh.ev[u] = e[x];
    }
    wg_axpby((size_t)n * n, 1.0, M.T, 0.0, nullptr, M.Ct);
    __syncthreads();
}

// After a sort: sh.sidx and sh.ev for the order that the next step's rows are
// brought into, the real orbitals ascending, then the padding.  moved: that
// moves a row; kocc: the real orbitals with f > 0, a prefix; p0: see Pad.
struct Behind {
    int p0, kocc;
    bool moved;
};
__device__ __noinline__ Behind pad_behind(const ldsf* ctx, Pad pad) {
    const Shared sh = CTX_GET(ctx, sh);
    pad = uniform_copy(pad);
    const int n = CTX_GET(ctx, M.n);
    const int npad = n - pad.nr, a0 = pad.at, a1 = a0 + npad;
    double red[3] = {0.0, 0.0, 0.0};
    int to[2];
    double e[2];
#pragma unroll
    for (int x = 0; x < 2; ++x) {
        const int o = threadIdx.x + x * NT;
        to[x] = -1;
        if (o >= n) continue;
        e[x] = sh.ev[o];
        const double k = e[x] == e[x] ? e[x] : INFINITY;
        // place among the real orbitals: equal and non-numbers as in wg_sort
        int r = 0;
        if (o >= a0 && o < a1) {
            r = pad.nr + o - a0;
        } else {
            for (int i = 0; i < n; ++i) {
                const double f = sh.ev[i], q = f == f ? f : INFINITY;
                r += (i < a0 || i >= a1) && (q < k || (q == k && i < o));
            }
            if (sh.ftot[o] > 0.0) red[1] = fmax(red[1], (double)(r + 1));
            if (k < 0.0) red[2] = fmax(red[2], (double)(r + 1));
        }
        to[x] = r;
        if (r != o) red[0] = 1.0;
    }
    wg_max_n<3>(red, sh.red);
#pragma unroll
    for (int x = 0; x < 2; ++x)
        if (to[x] >= 0) {
            sh.sidx[to[x]] = threadIdx.x + x * NT;
            sh.ev[to[x]] = e[x];
        }
    __syncthreads();
    return Behind{(int)red[2], (int)red[1], red[0] != 0.0};
}

// ---------------------------------------------------------------------------
// one SCF map v_in -> v_out (scf/base.py:651-675 iterate_potential);
// leaves q, sorted e/occupations and shell/atom charges behind, and in the
// last step (`last`) also P and e_orb (the other steps never store P).
// ---------------------------------------------------------------------------
__device__ __noinline__ int scf_step(ldsf* ctx, const glbf* vin, glbf* vout, int* status, double* ef, double loose,
                                     bool allow_bd, bool sort_rows, bool final_step = false,
                                     int* decoupled = nullptr, bool last = false) {
    const Mol M = CTX_GET(ctx, M);
    const Shared sh = CTX_GET(ctx, sh);
    Pad pad = CTX_GET(ctx, pad);
    int since = CTX_GET(ctx, since);
    const xtb_scf_opts o = karg_load(&CTX_GET(ctx, ka)->o);
    vin = uniform(vin);
    vout = uniform(vout);
    loose = uniform_copy(loose);
    const int n = M.n;
    // Occupation classes for this step's eigensolve.  With integer alpha/beta
    // counts and frontier gaps of at least bd_gap_kt x kT in the previous
    // step's spectrum (sh.skey, ascending; the rows of Ct are in that order),
    // only the coupling between doubly, singly and un-occupied orbitals is
    // removed: that fixes the density of 0/1 occupations, whose Fermi tails
    // at such gaps are below 1/(1 + e^(bd_gap_kt/2)).  The padding orbitals
    // of a padded layout (unit overlap diagonal, zero H0 and potential) are
    // exact eigenvectors at energy 0 with no coupling to any other orbital;
    // they sit in whichever class the sorted spectrum puts them, and the gap
    // test below covers them like any other level.
    int cb_lo = -1, cb_hi = -1;
    if ((allow_bd || final_step) && o.bd_gap_kt > 0.0) {
        const double na = M.nel_a, nb = M.nel_b;
        const int ia = (int)rint(na), ib = (int)rint(nb);
        bool ok = fabs(na - ia) < 1e-12 && fabs(nb - ib) < 1e-12 && ib <= ia;
        // (at kT -> 0 a gap of bd_gap_kt x kT(300 K) is still asked for:
        // the decoupling needs a clear gap to converge, not to be exact)
        const double need = o.bd_gap_kt * fmax(o.kt, 9.5e-4);
        if (ok && ia > 0 && ia < n) ok = sh.skey[ia] - sh.skey[ia - 1] >= need;
        if (ok && ib > 0 && ib < n) ok = sh.skey[ib] - sh.skey[ib - 1] >= need;
        if (ok) { cb_lo = ib; cb_hi = ia; }
    }
    // rows and columns of the products: the real orbitals, or all of them when
    // padding orbitals are among the doubly occupied ones
    const bool trypd = cb_lo >= 0 && cb_lo == cb_hi && o.pd_kmax > 0.0 && pd_applies(n, cb_lo);
    auto unpack = [&]() {
        if (pad.at == pad.p0) return;
        pad_to_spectrum(ctx, pad);
        pad.at = pad.p0;
        if (threadIdx.x == 0) CTX_PUT(ctx, pad, pad);
        __syncthreads();
    };
    int d = pad.nr;
    if (trypd && d < n && pad.p0 < cb_lo) {
        unpack();
        d = n;
    }
    const bool refresh = since == 0 || since >= PD_REFRESH;
    if (trypd) since = refresh ? 1 : since + 1;
    const int d0 = trypd ? d : n;
    // Fock build (scf/base.py:817-859)
    const int w = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
    double t0 = now_us();
    fock_build(M, vin, d0);
    {
        const double t = now_us();
        if (threadIdx.x == 0) {
            sh.tacc[8] += t - t0;
            sh.tacc[9] += 1.0;
        }
        t0 = t;
    }
    int sw = 0;
    bool pd = false, intra = false;
    if (final_step) {
        // Final (exact) step of a gapped closed shell: remove the last
        // occupied-virtual coupling perturbatively (it is second order after
        // that) to the full tolerance.  That fixes the density of the 0/1
        // occupations, the energies and W (rotations inside the occupied
        // block leave C^T f C and C_occ^T A_oo C_occ unchanged); only the
        // orbital energies need the diagonalisation inside the two classes.
        if (trypd) {
            const int r = pd_step(ctx, cb_lo, 0.0, vin, d, refresh);
            intra = r > 0;
            if (r != 0 || d0 < n) fock_build(M, vin, n);  // F may have served as scratch
        }
        if (!intra) cb_lo = cb_hi = -1;
        pd = intra && !o.orbitals;
        if (pd && decoupled) *decoupled = cb_lo;
    } else if (trypd) {
        const int r = pd_step(ctx, cb_lo, loose, vin, d, refresh);
        pd = r > 0;
        if (r < 0 || (r == 0 && d0 < n)) fock_build(M, vin, n);  // F served as scratch
    }
    if (pd) {
        const double dt = now_us() - t0;
        if (threadIdx.x == 0) {
            sh.tacc[2] += dt;
            sh.tacc[3] += dt;
            sh.tacc[6] += 1.0;
        }
    } else {
        unpack();
        // T = F C ; A = C^T T  -> F (with the padding in the last rows A's are
        // F's own zeros)
        const int da = pad.at == pad.nr ? pad.nr : n;
        gemm<false, true>(da, da, da, 1.0, M.F, n, M.Ct, n, 0.0, M.T, n, sh.big);
        gemm_sym<false, false>(da, da, 1.0, M.Ct, n, M.T, n, M.F, n, sh.big);
        double t1 = now_us();
        sw = eig_step(ctx, loose, cb_lo, cb_hi, intra);
        since = 1;  // eigenvalues fresh for the next perturbative step
        double t2 = now_us();
        if (threadIdx.x == 0) {
            sh.tacc[1] += t1 - t0;
            sh.tacc[2] += t2 - t1;
        }
    }
    // an intermediate step's eigensolve that ran out of sweeps only slows
    // the SCF down; the final step's results would be unreliable
    if (sw < 0 && final_step) *status |= XTB_MOL_JACOBI;
    wg_sort(sh.ev, sh.skey, sh.sidx, n);
    // Fermi occupations.  ef[2]: the largest f (1 - f).  Above ~1e-6 some
    // levels lie within ~14 kT of the Fermi level, where the density depends
    // on rotations among near-degenerate orbitals of different occupation:
    // the caller then tightens inexact eigensolves by 2 kT, the bound on
    // |f_i - f_j| / |e_i - e_j| over both channels
    const Filling fl = fill_orbitals(n, M.nao, M.nel_a, M.nel_b, sh.skey, sh.sidx, sh.ftot, sh.red, o.kt,
                                     o.fermi_thresh, o.fermi_maxiter, o.padded != 0, M.occ, M.occ + M.nvec_total);
    if (!fl.ok) *status |= XTB_MOL_FERMI;
    ef[0] = fl.ef[0];
    ef[1] = fl.ef[1];
    ef[2] = fl.soft;
    // P = C diag(f) C^T over the occupied orbitals (F and T are free here).
    // When the rows of Ct are already in ascending order (the usual case once
    // the SCF settles) they are used in place: no gather into F and no copy
    // back, 4 n^2 doubles of traffic less per step
    t0 = now_us();
    bool perm = uniform((int)fl.moved);
    int kocc = uniform(fl.kocc);
    const int held = pad.at == pad.nr ? pad.nr : n;  // rows and columns that move
    int dp = n;                                      // of the density product
    if (!last) {
        dp = pad.nr;
        if (pad.nr < n) {
            const Behind bh = pad_behind(ctx, pad);
            perm = uniform((int)bh.moved);
            kocc = uniform(bh.kocc);
            pad.p0 = uniform(bh.p0);
            pad.at = pad.nr;
        } else
            for (int j = threadIdx.x; j < n; j += NT) sh.ev[j] = sh.skey[j];  // in the sorted rows' order
    }
    if (perm) {
        gather_occupied(ctx, M.F, M.T, last ? n : held, last ? n : dp, kocc, false, sort_rows);
    } else {
        for (int j0 = w * ROWS_PER_WAVE; j0 < kocc; j0 += NWAVE * ROWS_PER_WAVE) {
            int jj[ROWS_PER_WAVE];
            double f[ROWS_PER_WAVE];
#pragma unroll
            for (int u = 0; u < ROWS_PER_WAVE; ++u) {
                jj[u] = j0 + u < kocc ? j0 + u : kocc - 1;
                f[u] = sh.ftot[jj[u]];
            }
            for (int c = lane; c < dp; c += WAVE) {
                double cv[ROWS_PER_WAVE];
#pragma unroll
                for (int u = 0; u < ROWS_PER_WAVE; ++u) cv[u] = M.Ct[(size_t)jj[u] * n + c];
#pragma unroll
                for (int u = 0; u < ROWS_PER_WAVE; ++u)
                    if (j0 + u < kocc) M.T[(size_t)jj[u] * n + c] = f[u] * cv[u];
            }
        }
        __syncthreads();
    }
    if (last) {
        gemm_sym<true, false>(n, kocc, 1.0, perm ? M.F : M.Ct, n, M.T, n, M.P, n, sh.big);
    } else {
        // an intermediate step needs the charges, not P: the Mulliken sums
        // a_i = sum_j P_ij S_ij come from the density product's tiles (P is
        // never stored), into q
        gemm_sym_mull<true, false>(dp, kocc, perm ? M.F : M.Ct, n, M.T, n, M.S, n, M.nao, M.q, sh.big);
    }
#ifdef XTB_PD_TIMERS
    if (threadIdx.x == 0) sh.red[RED_DOUBLES - 12 + 8] += now_us() - t0;
#endif
    if (sort_rows && perm) {
        // the next step starts from the orbitals in ascending energy order
        const int h = last ? n : held;
        if (h == n) wg_axpby((size_t)n * n, 1.0, M.F, 0.0, nullptr, M.Ct);
        else
            for (int r = w; r < h; r += NWAVE)
                for (int c = lane; c < h; c += WAVE) M.Ct[(size_t)r * n + c] = M.F[(size_t)r * n + c];
    }
    const double tm0 = now_us();
    if (threadIdx.x == 0) sh.tacc[1] += tm0 - t0;
    // Mulliken charges and orbital energies (scf/base.py:764-815), one wave
    // per row; the orbital energies only enter the final energy (last step)
    if (!last) {
        for (int i = threadIdx.x; i < n; i += NT) M.q[i] = (i < M.nao) ? M.n0[i] - M.q[i] : 0.0;
    } else {
        const int w = threadIdx.x / WAVE, l = threadIdx.x % WAVE;
        for (int i0 = w * ROWS_PER_WAVE; i0 < n; i0 += NWAVE * ROWS_PER_WAVE) {
            int ii[ROWS_PER_WAVE];
            double sq[ROWS_PER_WAVE], se[ROWS_PER_WAVE];
#pragma unroll
            for (int u = 0; u < ROWS_PER_WAVE; ++u) {
                ii[u] = i0 + u < n ? i0 + u : n - 1;
                sq[u] = 0.0;
                se[u] = 0.0;
            }
            for (int j = l; j < M.nao; j += WAVE) {
                double pv[ROWS_PER_WAVE], sv[ROWS_PER_WAVE], hv[ROWS_PER_WAVE];
#pragma unroll
                for (int u = 0; u < ROWS_PER_WAVE; ++u) {
                    pv[u] = M.P[(size_t)ii[u] * n + j];
                    sv[u] = M.S[(size_t)ii[u] * n + j];
                    hv[u] = M.H0[(size_t)ii[u] * n + j];
                }
#pragma unroll
                for (int u = 0; u < ROWS_PER_WAVE; ++u) {
                    sq[u] = fma(pv[u], sv[u], sq[u]);
                    se[u] = fma(pv[u], hv[u], se[u]);
                }
            }
#pragma unroll
            for (int u = 0; u < ROWS_PER_WAVE; ++u) {
                const double a = wave_sum(sq[u]), e = wave_sum(se[u]);
                const int i = i0 + u;
                if (l == 0 && i < n) {
                    M.q[i] = (i < M.nao) ? M.n0[i] - a : 0.0;
                    M.eorb[i] = (i < M.nao) ? e : 0.0;
                }
            }
        }
    }
    __syncthreads();
    // shell and atom charges
    for (int s = threadIdx.x; s < M.nsh; s += NT) {
        const int o0 = M.sh_ao[s];
        const int nl = 2 * M.us_l[M.sh_us[s]] + 1;
        double acc = 0.0;
        for (int x = 0; x < nl; ++x) acc += M.q[o0 + x];
        sh.qsh[s] = acc;
    }
    __syncthreads();
    for (int a = threadIdx.x; a < M.nat; a += NT) {
        const int s0 = M.atom_sh0[a], ns = M.atom_nsh[a];
        double acc = 0.0;
        for (int x = 0; x < ns; ++x) acc += sh.qsh[s0 + x];
        sh.qat[a] = acc;
    }
    __syncthreads();
    // ES2 (gamma q_sh) + ES3 (hd q_at^2) shell potential, one wave per row
    {
        const int w = threadIdx.x / WAVE, l = threadIdx.x % WAVE;
        const int m = M.nsh;
        for (int s0 = w * ROWS_PER_WAVE; s0 < m; s0 += NWAVE * ROWS_PER_WAVE) {
            int ss[ROWS_PER_WAVE];
            double acc[ROWS_PER_WAVE];
#pragma unroll
            for (int u = 0; u < ROWS_PER_WAVE; ++u) {
                ss[u] = s0 + u < m ? s0 + u : m - 1;
                acc[u] = 0.0;
            }
            for (int t = l; t < m; t += WAVE) {
                const double qt = sh.qsh[t];
                double g[ROWS_PER_WAVE];
#pragma unroll
                for (int u = 0; u < ROWS_PER_WAVE; ++u) g[u] = M.gam[(size_t)ss[u] * m + t];
#pragma unroll
                for (int u = 0; u < ROWS_PER_WAVE; ++u) acc[u] = fma(g[u], qt, acc[u]);
            }
#pragma unroll
            for (int u = 0; u < ROWS_PER_WAVE; ++u) {
                const double v = wave_sum(acc[u]);
                const int s = s0 + u;
                if (l == 0 && s < m) {
                    const int a = M.sh_atom[s];
                    const double hd = M.sp_gam3[M.atom_sp[a]];
                    sh.gq[s] = v;
                    sh.vsh[s] = v + hd * sh.qat[a] * sh.qat[a];
                }
            }
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < n; i += NT) {
        const int s = (i < M.nao) ? M.ao_sh[i] : -1;
        vout[i] = (s >= 0) ? sh.vsh[s] : 0.0;
    }
    if (threadIdx.x == 0) {
        CTX_PUT(ctx, pad, pad);
        CTX_PUT(ctx, since, since);
    }
    __syncthreads();
    const double tm1 = now_us();
    // (P, S) reads of this stage in units of 16 n^2 bytes: the last step
    // reads P, S and H0 (orbital energies); the others form q inside the
    // density product (timed with it) and only add the gamma products here
    if (threadIdx.x == 0) {
        sh.tacc[10] += tm1 - tm0;
        sh.tacc[11] += last ? 1.5 : 0.0;
    }
    return sw < 0 ? 0 : sw;
}

// Inputs and outputs of the fused single point (k_singlepoint) beyond the
// SCF's: positions, and the buffers the integral pass and the gradient fill.
// Defined with the fused kernel (singlepoint.hip); the plain SCF kernel
// never calls them.
__device__ __noinline__ void molecule_integrals(const ldsf* ctx);
__device__ __noinline__ void molecule_forces(const ldsf* ctx);

}  // namespace xtb

// Validation shared by xtb_scf and xtb_singlepoint (host).
static inline int32_t check_scf_args(const xtb_batch* batch, const xtb_scf_opts* opts, const xtb_scf_state* state) {
    if (batch->nmol <= 0 || batch->max_n <= 0) return XTB_EINVAL;
    if (batch->max_n > 1024) return XTB_ETOOBIG;
    if (opts->mixer != 0 && opts->mixer != 1) return XTB_EINVAL;
    if (opts->generations < 1 || opts->generations > (opts->mixer == 1 ? xtb::BROYDEN_MAXR : xtb::MIX_MAXG))
        return XTB_EINVAL;
    if (opts->wg_skip < 0 || opts->wg_skip > 7) return XTB_EINVAL;
    if (opts->jacobi_inner < 1 || opts->jacobi_inner > 20 || opts->eig_inexact < 0.0) return XTB_EINVAL;
    if (!state->F || !state->C || !state->T || !state->P || !state->pot || !state->vnew ||
        !state->q || !state->eorb || !state->emo || !state->occ || !state->hist_x ||
        !state->hist_f || !state->qsh || !state->out || !state->order)
        return XTB_EINVAL;
    return XTB_OK;
}
