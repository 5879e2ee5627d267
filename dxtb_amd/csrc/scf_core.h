// Per-molecule SCF pieces shared by the one-workgroup-per-molecule kernel
// (scf.hip) and the whole-GPU path for one large molecule (large.hip): Fermi
// smearing, the mixers, Cholesky blocks.  Every function here is called by all
// threads of one workgroup; uniform arguments come by value (what comes by
// reference is read from the stack frame, a scratch load, at every use).
#pragma once

#include "common.h"
#include "wg.h"

namespace xtb {

// device wall clock (constant 100 MHz) in microseconds
__device__ inline double now_us() { return (double)wall_clock64() * 0.01; }

// Passes of the perturbative occupied-virtual rotation.  The amplitudes
// divide by the diagonals of the occupied and virtual blocks only, and those
// blocks drift away from diagonal over an SCF run, so the passes converge
// linearly: the largest coupling falls by a factor 0.2 per pass (median;
// 0.35-0.45 at the 90th percentile, 2400 molecules of the serving stream),
// not quadratically.  An inexact SCF step stops after two passes, or once
// the second-order estimate max|K| max|A_ov| is below its tolerance.  The
// final step stops only on a measured coupling below
// max(jacobi_tol max(|e|, 1), PD_FINAL_REL x_atol_max): a coupling d turns
// the orbitals by ~d / gap (gaps >= 60 kT = 0.057 Eh here), so the charges
// and forces move by < 40 d, at most what the SCF's own convergence
// threshold on the potential leaves.  At x_atol_max = 1e-10, 79 % of the
// 2400 molecules meet 1e-11 without a rotation and all within 6
// measurements; 1e-2 x_atol_max needed up to 9 and more, and made that
// launch 17 % longer.  After PD_EXACT_PASSES measurements the step falls
// back to a full eigensolve, which costs as much as ~15 passes on a
// 500-orbital molecule.
constexpr int PD_INEXACT_PASSES = 2;
constexpr int PD_EXACT_PASSES = 7;
constexpr double PD_FINAL_REL = 1e-1;

// ---------------------------------------------------------------------------
// Diagonal blocks of the blocked Cholesky factorisations: one wave, a row per
// lane in registers.  Lane r < 32 holds row r of the block and lane 32 + j
// row j of the identity; the column operations that turn the block into its
// factor L turn the identity into L^-T, so both come out of one pass.  Every
// step works on register 0 and moves the others down by one (chol_steps: CNT
// columns are left behind the pivot at most).
//
// The pass is bound by its serial chain, the pivot's inverse square root and
// then two lane reads and an FMA per column left: 13 us a block as a launch
// of its own.  Factor and inverse through LDS, with the inverse by
// substitution in one lane per column, took 65 us.
// ---------------------------------------------------------------------------
template <int CNT>
__device__ __forceinline__ void chol_steps(double (&x)[32], int c0, int nb, bool& ok, glbf* out, int step) {
    const int lane = threadIdx.x % WAVE;
    for (int c = c0; c < c0 + 8; ++c) {
        const double d = wave_read(x[0], c);
        const bool pos = d > 0.0;
        ok = ok && pos;
        // sqrt(d) and the column over it, each corrected by its residual
        const double inv = pos ? fast_rsq(d) : 1.0;
        double sd = d * inv, v = x[0] * inv;
        sd = pos ? fma(fma(-sd, sd, d), 0.5 * inv, sd) : 1.0;
        v = fma(fma(-v, sd, x[0]), inv, v);
#pragma unroll
        for (int i = 0; i < CNT; ++i) x[i] = fma(-v, wave_read(v, c + 1 + i), x[i + 1]);
        const int r = lane % 32;
        if (r < nb && c < nb && (lane >= 32 || r >= c)) out[(size_t)c * step] = lane >= 32 && r > c ? 0.0 : v;
    }
}

// L (leading dimension ld, lower triangle read) <- its lower Cholesky factor
// in place, the inverse of the factor to Dg (leading dimension nb); nb <= 32.
// Returns false when a pivot is not positive (taken as 1 then: the factor is
// meaningless).
__device__ __noinline__ bool chol_block(glbf* L, int ld, int nb, glbf* Dg) {
    const int lane = threadIdx.x % WAVE, r = lane % 32;
    double x[32];
#pragma unroll
    for (int c = 0; c < 32; ++c) {
        const double a = L[(size_t)(r < nb ? r : nb - 1) * ld + (c < nb ? c : nb - 1)];
        x[c] = lane < 32 && r < nb && c <= r ? a : (r == c ? 1.0 : 0.0);
    }
    bool ok = true;
    glbf* out = lane < 32 ? L + (size_t)r * ld : Dg + r;
    const int step = lane < 32 ? 1 : nb;
    chol_steps<31>(x, 0, nb, ok, out, step);
    chol_steps<23>(x, 8, nb, ok, out, step);
    chol_steps<15>(x, 16, nb, ok, out, step);
    chol_steps<7>(x, 24, nb, ok, out, step);
    return ok;
}

// LDS doubles of the reduction scratch
constexpr int RED_DOUBLES = 192;

// electronic temperatures below this (0.1 K in Hartree) fill the orbitals
// by the aufbau principle instead of Fermi smearing
// (src/dxtb/_src/scf/base.py:888-889)
constexpr double KT_AUFBAU = 3e-7;

// ---------------------------------------------------------------------------
// Fermi smearing of the spin channels (src/dxtb/_src/wavefunction/
// filling.py:201-366): mid-gap start, Newton on the rounded electron count
// (scf/base.py:879), exponent cutoff 50, threshold on |N - sum f|.  Below
// KT_AUFBAU the aufbau occupations of the unrounded count instead
// (filling.py:116-198; base.py:888-889 keeps the initial filling of
// iterator.py:147-189): orbital j (from 0) is full while j + 1 < nel, the
// next one takes nel - ceil(nel) + 1.  Sorted eigenvalues in skey, their
// orbitals in sidx.  Writes the sorted occupations to occ[channel] and
// the orbitals' sums to ftot.
//
// Latency-bound (an exponential and a reduction per Newton step): both
// channels advance together, and equal ones (closed shells) are one: 5.3 us a
// launch at n = 296 (with a sort in the same launch 12.8; one channel after the
// other and a bitonic sort 20).
// ---------------------------------------------------------------------------
struct Filling {
    double ef[2];  // Fermi levels
    double soft;   // largest f (1 - f) of either channel
    int kocc;      // orbitals with f > 0 (a prefix in sorted order)
    bool moved;    // the sort moved an orbital
    bool ok;       // every channel converged
};

template <class F>
__device__ __noinline__ Filling fill_orbitals(int n, int nao, double nel_a, double nel_b, const ldsf* skey,
                                              const ldsi* sidx, F* ftot, ldsf* scratch, double kt, double thr,
                                              int maxiter, bool padded, glbf* occ_a, glbf* occ_b) {
    n = uniform(n);
    nao = uniform(nao);
    nel_a = uniform_copy(nel_a);
    nel_b = uniform_copy(nel_b);
    kt = uniform_copy(kt);
    const double eps = 2.220446049250313e-16;
    const int nch = nel_a == nel_b ? 1 : 2;
    double ef[2] = {0.0, 0.0}, target[2] = {0.0, 0.0};
    bool open[2] = {false, false}, smear[2] = {false, false};
#pragma unroll
    for (int c = 0; c < 2; ++c) {
        double nel = c == 0 ? nel_a : nel_b;
        if (c >= nch || fabs(nel) < eps || kt < KT_AUFBAU) continue;
        nel = rint(nel);
        int homo = (int)ceil(nel - 5e-15) - 1;
        if (homo < 0) homo = 0;
        if (homo > n - 1) homo = n - 1;
        const int lumo = n - 1 <= homo ? homo : homo + 1;
        ef[c] = 0.5 * (skey[homo] + skey[lumo]);
        if (padded && (homo >= nao || lumo >= nao)) ef[c] *= 2.0;  // filling.py:254-264
        target[c] = (double)(homo + 1);
        open[c] = true;
    }
    for (int it = 0; it < maxiter && (open[0] || open[1]); ++it) {
        double acc[4] = {0.0, 0.0, 0.0, 0.0};
        for (int j = threadIdx.x; j < n; j += NT) {
            const double e = skey[j];
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                if (!open[c]) continue;
                const double x = (e - ef[c]) / kt;
                if (x < 50.0) {
                    const double et = exp(x), f = 1.0 / (et + 1.0);
                    acc[2 * c] += f;
                    acc[2 * c + 1] += et * f * f;
                } else {
                    acc[2 * c + 1] += eps * kt;
                }
            }
        }
        wg_sum_n<4>(acc, scratch);
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            if (!open[c]) continue;
            const double diff = target[c] - acc[2 * c];
            if (fabs(diff) <= thr) {
                open[c] = false;
                smear[c] = true;
            } else {
                ef[c] += diff * kt / acc[2 * c + 1];
            }
        }
    }
    const bool ok = !open[0] && !open[1];
    double red[3] = {0.0, 0.0, 0.0};
    for (int j = threadIdx.x; j < n; j += NT) {
        const double e = skey[j];
        double f[2] = {0.0, 0.0};
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            const double nel = c == 0 ? nel_a : nel_b;
            if (c >= nch) {
                f[c] = f[0];
            } else if (smear[c]) {
                const double x = (e - ef[c]) / kt;
                f[c] = x < 50.0 ? 1.0 / (exp(x) + 1.0) : 0.0;
            } else if (kt < KT_AUFBAU && !(fabs(nel) < eps)) {
                const double idx = (double)(j + 1);
                f[c] = idx < nel ? 1.0 : (idx < nel + 1.0 ? nel - ceil(nel) + 1.0 : 0.0);
            }
            red[0] = fmax(red[0], f[c] * (1.0 - f[c]));
        }
        occ_a[j] = f[0];
        occ_b[j] = f[1];
        const int o = sidx[j];
        ftot[o] = f[0] + f[1];
        if (f[0] + f[1] > 0.0) red[1] = (double)(j + 1);
        if (o != j) red[2] = 1.0;
    }
    wg_max_n<3>(red, scratch);
    return Filling{{ef[0], nch == 1 ? ef[0] : ef[1]}, red[0], (int)red[1], red[2] != 0.0, ok};
}

// ---------------------------------------------------------------------------
// Anderson mixing with soft start (scf/mixer/anderson.py:163-317), history in
// a ring buffer of G = generations+1 slots.  Returns the convergence flag of
// the step (mixer/base.py:229-256 on the step's residual).
// ---------------------------------------------------------------------------
// largest history (generations) the mixer takes: its system with the right
// side fits 8 x 8 lanes, and more generations save ~1 % of the iterations
constexpr int MIX_MAXG = 6;

struct Mixer {
    int step, head, G;
    bool soft;  // upstream's soft start; a warm start, already near the fixed point, skips it
};

// what a mixer needs of the options
struct MixOpts {
    double x_atol, x_atol_max, damp, damp_init, diag_offset;
};

// The vectors: n elements; histories hx and hf with `stride` between slots.
__device__ __noinline__ bool anderson(Mixer& mixer, int n, int stride, ldsf* red, MixOpts o, glbf* hx, glbf* hf,
                                      const glbf* xnew, const glbf* xold, glbf* xout, double* resid_inf) {
    n = uniform(n);
    stride = uniform(stride);
    o = uniform_copy(o);
    hx = uniform(hx);
    hf = uniform(hf);
    xnew = uniform(xnew);
    xold = uniform(xold);
    xout = uniform(xout);
    Mixer mx = uniform_copy(mixer);
    const int G = mx.G;
    auto slot = [&](int h) {  // h < G
        const int k = mx.head + h;
        return (size_t)(k < G ? k : k - G) * stride;
    };
    auto X = [&](int h) { return hx + slot(h); };
    auto Fh = [&](int h) { return hf + slot(h); };
    if (mx.step == 0) {
        glbf* x0 = X(0);
        for (int i = threadIdx.x; i < n; i += NT) x0[i] = xold[i];
        __syncthreads();
    }
    mx.step += 1;
    const int gen = G - 1;
    glbf* x0 = X(0);
    glbf* f0 = Fh(0);
    double l2 = 0.0, linf = 0.0;
    for (int i = threadIdx.x; i < n; i += NT) {
        const double f = xnew[i] - x0[i];
        f0[i] = f;
        l2 = fma(f, f, l2);
        linf = fmax(linf, fabs(f));
    }
    l2 = wg_sum(l2, red);
    linf = wg_max(linf, red + NWAVE);
    const bool conv = (sqrt(l2) < o.x_atol) && (linf < o.x_atol_max);
    *resid_inf = linf;
    double theta[MIX_MAXG];
#pragma unroll
    for (int h = 0; h < MIX_MAXG; ++h) theta[h] = 0.0;
    int nn = 0;
    if (mx.step > gen || !mx.soft) nn = (mx.step - 1 < gen) ? mx.step - 1 : gen;  // soft start
    if (nn > 0) {
        // a_hj = (f0 - f_h).(f0 - f_j), b_h = (f0 - f_h).f0 ; h, j = 1..nn.
        // The nt sums (j = nn + 1: b_h) are dealt to the waves, each over all
        // elements: no partial sums to combine
        const int wv = threadIdx.x / WAVE, ln = threadIdx.x % WAVE;
        constexpr int NACC = MIX_MAXG * (MIX_MAXG + 3) / 2, PER = (NACC + NWAVE - 1) / NWAVE;
        ldsf* tot = red;
        const int nt = nn * (nn + 3) / 2;
        const glbf *ph[PER], *pj[PER];
        bool rhs[PER];
        double s[PER];
#pragma unroll
        for (int t = 0; t < PER; ++t) {
            int e = wv + NWAVE * t < nt ? wv + NWAVE * t : nt - 1, h = 1;
            while (e >= nn + 2 - h) e -= nn + 2 - h++;
            ph[t] = Fh(h);
            rhs[t] = h + e > nn;
            pj[t] = rhs[t] ? f0 : Fh(h + e);
            s[t] = 0.0;
        }
#pragma unroll 4
        for (int i = ln; i < n; i += WAVE) {
            const double fi = f0[i];
#pragma unroll
            for (int t = 0; t < PER; ++t) {
                const double a = ph[t][i], b = pj[t][i];
                s[t] = fma(fi - a, rhs[t] ? b : fi - b, s[t]);
            }
        }
#pragma unroll
        for (int t = 0; t < PER; ++t) {
            s[t] = wave_sum(s[t]);
            if (ln == 0 && wv + NWAVE * t < nt) tot[wv + NWAVE * t] = s[t];
        }
        __syncthreads();
        // solve (a * diag(1 + off^2)) theta = b by Gauss-Jordan elimination
        // with partial pivoting: element (r, x) on lane 8 r + x, b in column
        // 7, the same in every wave.  The mixing step takes 15 us a launch at
        // n = 296 (every thread with all sums, reduced one by one, and one
        // thread solving in LDS: 28 us)
        const int r = ln / 8, x = ln % 8;
        double a = 0.0;
        if (r < nn && (x < nn || x == 7)) {
            const int h = x < r ? x : r, j = x == 7 ? nn : (x < r ? r : x);  // h <= j, from 0
            a = tot[h * (2 * nn + 3 - h) / 2 + j - h];
            if (r == x) a *= 1.0 + o.diag_offset * o.diag_offset;
        }
        for (int c = 0; c < nn; ++c) {
            int piv = c;
            double best = fabs(wave_read(a, 9 * c));
            for (int q = c + 1; q < nn; ++q) {
                const double v = fabs(wave_read(a, 8 * q + c));
                if (v > best) {
                    best = v;
                    piv = q;
                }
            }
            a = __shfl(a, 8 * (r == c ? piv : (r == piv ? c : r)) + x, WAVE);
            const double col = __shfl(a, 8 * r + c, WAVE), row = __shfl(a, 8 * c + x, WAVE);
            const double fct = col / wave_read(a, 9 * c);
            if (r != c && x >= c) a -= fct * row;
        }
        a /= __shfl(a, 9 * r, WAVE);  // column 7: theta
#pragma unroll
        for (int h = 0; h < MIX_MAXG; ++h) theta[h] = (h < nn) ? wave_read(a, 8 * h + 7) : 0.0;
        __syncthreads();
    }
    // new slot for the mixed vector = oldest slot
    const int newhead = (mx.head - 1 + G) % G;
    glbf* xn = hx + (size_t)newhead * stride;
    for (int i = threadIdx.x; i < n; i += NT) {
        double xm;
        if (nn > 0) {
            double xb = x0[i], fb = f0[i];
#pragma unroll
            for (int h = 0; h < MIX_MAXG; ++h) {
                if (h < nn) {
                    const double xh = X(h + 1)[i], fh = Fh(h + 1)[i];
                    xb += theta[h] * (xh - x0[i]);
                    fb -= theta[h] * (f0[i] - fh);
                }
            }
            xm = xb + o.damp * fb;
        } else {
            xm = x0[i] + (mx.soft ? o.damp_init : o.damp) * f0[i];
        }
        xout[i] = xm;
        xn[i] = xm;  // slot newhead may alias X(G-1): element-wise read-before-write
    }
    __syncthreads();
    mixer.step = mx.step;
    mixer.head = newhead;
    return conv;
}

// ---------------------------------------------------------------------------
// Limited-memory Broyden root search ("broyden1", good Broyden) on
// g(x) = x - f(x), as upstream's implicit SCF modes run it
// (scf/implicit/default.py, scf/pure/iterator.py:125-147 -> xitorch
// equilibrium, optimize/root/rootsolver.py:42-256 with BroydenFirst,
// _jacobian.py:50-112): inverse Jacobian H = h0 I + sum_k c_k d_k^T with
// h0 = -alpha = 0.5, no line search, x <- x + damp dx with dx = -H g.  After
// each map evaluation (x_prev, g_prev -> x, g): dx = x - x_prev,
// dy = g - g_prev, v = H^T dx, c = dx - H dy, d = v / (dy.v), H += c d^T.
// Converged (TerminationCondition, rootsolver.py:471-492) when the last
// step's |dx| < x_atol and |g| < f_atol.  Upstream keeps every update; here
// at most R = generations (<= BROYDEN_MAXR) are kept and the memory restarts
// from h0 I when full (upstream's "restart" reduction at max_rank = R).
// Storage: c_k in hx slot k, d_k in hf slot k (k < R); x_prev, g_prev in
// slot R.  The first call only records x_prev and g_prev.
// ---------------------------------------------------------------------------
constexpr int BROYDEN_MAXR = 24;

struct Broyden {
    int step, rank, R;
    double dxnorm;  // |dx| of the last step (before damping)
};

// Projections sum_i U_k[i] w_i for k < r, reduced in chunks of 8 and left
// in LDS at red[128 + k] (red holds RED_DOUBLES; wg_sum_n<8> uses the first
// 64).  U_k(i) and w(i) are callables.
template <class UK, class W>
__device__ inline void wg_projections(int r, int n, ldsf* red, UK U, W w, int out0) {
    for (int k0 = 0; k0 < r; k0 += 8) {
        double t[8] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
        for (int i = threadIdx.x; i < n; i += NT) {
            const double wi = w(i);
#pragma unroll
            for (int kk = 0; kk < 8; ++kk)
                if (k0 + kk < r) t[kk] = fma(U(k0 + kk, i), wi, t[kk]);
        }
        wg_sum_n<8>(t, red);
        if (threadIdx.x == 0) {
#pragma unroll
            for (int kk = 0; kk < 8; ++kk)
                if (k0 + kk < r) red[128 + out0 + k0 + kk] = t[kk];
        }
        __syncthreads();
    }
}

__device__ __noinline__ bool broyden(Broyden& bm, int n, int stride, ldsf* red, MixOpts o, double f_atol, glbf* hx,
                                     glbf* hf, const glbf* fx, const glbf* x, glbf* xout, double* resid_inf) {
    static_assert(128 + 2 * BROYDEN_MAXR <= RED_DOUBLES, "projections fit the reduction scratch");
    const int R = bm.R;
    constexpr double h0 = 0.5;  // -alpha, alpha = -0.5 (scf/pure/iterator.py:132)
    auto C = [&](int k) { return hx + (size_t)k * stride; };
    auto D = [&](int k) { return hf + (size_t)k * stride; };
    glbf* xp = C(R);
    glbf* gp = D(R);
    ldsf* proj = red + 128;  // [0, R): first set, [R, 2R): second set
    double g2 = 0.0, ginf = 0.0;
    for (int i = threadIdx.x; i < n; i += NT) {
        const double g = x[i] - fx[i];
        g2 = fma(g, g, g2);
        ginf = fmax(ginf, fabs(g));
    }
    g2 = wg_sum(g2, red);
    ginf = wg_max(ginf, red);
    *resid_inf = ginf;
    if (bm.step > 0) {
        if (bm.dxnorm < o.x_atol && sqrt(g2) < f_atol) {
            // the root search stops before it takes x: its result is the
            // previous input (rootsolver.py:200-215 breaks before x = xnew)
            for (int i = threadIdx.x; i < n; i += NT) xout[i] = xp[i];
            __syncthreads();
            bm.step += 1;
            return true;
        }
        // c_k.dx and d_k.dy over the kept pairs; the new pair goes to slot rr
        // (the memory restarts when full)
        const int r = bm.rank;
        const int rr = r >= R ? 0 : r;
        wg_projections(rr, n, red, [&](int k, int i) { return C(k)[i]; },
                       [&](int i) { return x[i] - xp[i]; }, 0);
        wg_projections(rr, n, red, [&](int k, int i) { return D(k)[i]; },
                       [&](int i) { return (x[i] - fx[i]) - gp[i]; }, R);
        glbf* cn = C(rr);
        glbf* dn = D(rr);
        double dyv = 0.0;
        for (int i = threadIdx.x; i < n; i += NT) {
            const double dx = x[i] - xp[i], dy = (x[i] - fx[i]) - gp[i];
            double v = h0 * dx, hdy = h0 * dy;
            for (int k = 0; k < rr; ++k) {
                v = fma(D(k)[i], proj[k], v);
                hdy = fma(C(k)[i], proj[R + k], hdy);
            }
            cn[i] = dx - hdy;
            dn[i] = v;
            dyv = fma(dy, v, dyv);
        }
        dyv = wg_sum(dyv, red);
        const double sc = 1.0 / dyv;
        for (int i = threadIdx.x; i < n; i += NT) dn[i] *= sc;
        __syncthreads();
        bm.rank = rr + 1;
    } else {
        bm.rank = 0;
    }
    // dx = -H g with the updated memory
    const int rk = bm.rank;
    wg_projections(rk, n, red, [&](int k, int i) { return D(k)[i]; }, [&](int i) { return x[i] - fx[i]; }, 0);
    double dn2 = 0.0;
    for (int i = threadIdx.x; i < n; i += NT) {
        const double xi = x[i], g = xi - fx[i];
        double hg = h0 * g;
        for (int k = 0; k < rk; ++k) hg = fma(C(k)[i], proj[k], hg);
        // x_prev, g_prev <- x, g
        xp[i] = xi;
        gp[i] = g;
        dn2 = fma(hg, hg, dn2);
        xout[i] = xi - o.damp * hg;  // xout may alias x: element-wise read-before-write
    }
    bm.dxnorm = sqrt(wg_sum(dn2, red));
    bm.step += 1;
    return false;
}
}  // namespace xtb
