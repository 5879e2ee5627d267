// Fused single point on gfx950: one workgroup per molecule computes its
// integral pass, runs its SCF (the body of k_scf, scf_kernel.h) and writes
// its analytic gradient, so that a batch is one launch.  A translation unit
// of its own: sharing the SCF's out-of-line device functions with this
// kernel in one code object makes the compiler give those functions more
// conservative register conventions, which grew k_scf's stack frame.
#include "scf_kernel.h"
#include "integral_terms.h"
#include "gradient_terms.h"

namespace xtb {

// One molecule's integral pass by its own workgroup, with the per-element
// code of k_integrals (so the same bits): coordination numbers (CN_PARTS
// lanes per atom), S, H0 and gamma over the shell pairs i <= j, the padding
// orbitals of a padded layout, and the repulsion energy into the molecule's
// record.  The shell pairs are dealt to the threads by class (pp, sp, ss, each
// from a new wave on), so that no wave runs the code of several classes and
// few lanes idle: 68 orbitals 200 -> 83 us, 194 647 -> 435 us (a wave per
// row of shells, every class in every wave).
__device__ __noinline__ void molecule_integrals(const ldsf* ctx) {
    const Mol M = CTX_GET(ctx, M);
    const Shared sh = CTX_GET(ctx, sh);
    kargs* ka = CTX_GET(ctx, ka);
    const xtb_batch b = karg_load(&ka->b);
    const xtb_params par = karg_load(&ka->par);
    const FusedArgs fa = karg_load(&ka->fa);
    double* outs = ka->st.out;
    const int w = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
    for (int a0 = 0; a0 < M.nat; a0 += NT / CN_PARTS) {
        // every lane of a CN_PARTS group takes part in the butterfly
        const int a = a0 + (int)threadIdx.x / CN_PARTS, part = threadIdx.x % CN_PARTS;
        const bool ok = a < M.nat;
        const double v = cn_combine(ok ? cn_part(b, par, fa.pos, M.at0 + a, part) : 0.0);
        if (ok && part == 0) fa.cn[M.at0 + a] = v;
    }
    double* s_alpha = (double*)sh.big;
    double* s_coeff = s_alpha + XTB_MAX_US_LDS * XTB_MAXPRIM;
    for (int i = threadIdx.x; i < par.nus * XTB_MAXPRIM; i += NT) {
        s_alpha[i] = par.us_alpha[i];
        s_coeff[i] = par.us_coeff[i];
    }
    __syncthreads();
    // the molecule's s shells and p shells, in order
    ldsi* ls = (ldsi*)(sh.big + 2 * XTB_MAX_US_LDS * XTB_MAXPRIM);
    ldsi* lp = ls + M.nsh;
    int ns = 0;
    for (int i0 = 0; i0 < M.nsh; i0 += WAVE) {  // (every wave counts, the first one writes)
        const int i = i0 + lane;
        const bool p = i < M.nsh && M.us_l[M.sh_us[i]] != 0;
        const uint64_t mp = __ballot(p), ms = __ballot(i < M.nsh && !p), below = (1ull << lane) - 1;
        if (w == 0 && i < M.nsh) {
            if (p) lp[i0 - ns + __popcll(mp & below)] = i;
            else ls[ns + __popcll(ms & below)] = i;
        }
        ns += __popcll(ms);
    }
    const int np = M.nsh - ns;
    __syncthreads();
    auto pair = [&](auto LI, auto LJ, int i, int j) {
        shell_pair_s_h0_t<decltype(LI)::value, decltype(LJ)::value>(
            b, par, fa.pos, fa.S, fa.H0, M.m, i, j, fa.cn[M.at0 + M.sh_atom[i]], fa.cn[M.at0 + M.sh_atom[j]], s_alpha,
            s_coeff);
        gamma_pair(b, par, fa.pos, fa.gam, M.m, i, j, M.nsh);
    };
    const int n3 = np * (np + 1) / 2, n2 = np * ns, n1 = ns * (ns + 1) / 2;
    const int e2 = (n3 + WAVE - 1) / WAVE * WAVE, e1 = e2 + (n2 + WAVE - 1) / WAVE * WAVE;
    for (int e = threadIdx.x; e < e1 + n1; e += NT) {
        int r, c;
        if (e < e2) {
            if (e >= n3) continue;
            triangle(np, e, r, c);
            pair(IntC<1>{}, IntC<1>{}, lp[r], lp[c]);
        } else if (e < e1) {
            if (e - e2 >= n2) continue;
            const int x = (int)((uint32_t)(e - e2) / (uint32_t)ns), i = ls[e - e2 - x * ns], j = lp[x];
            if (i < j) pair(IntC<0>{}, IntC<1>{}, i, j);
            else pair(IntC<1>{}, IntC<0>{}, j, i);
        } else {
            triangle(ns, e - e1, r, c);
            pair(IntC<0>{}, IntC<0>{}, ls[r], ls[c]);
        }
    }
    if (M.n > M.nao) {
        // padded layout: unit overlap diagonal and zero H0 on the padding
        // orbitals (as k_pad_fill)
        const size_t tot = (size_t)M.n * M.n;
        for (size_t e = threadIdx.x; e < tot; e += NT) {
            const int r = (int)(e / M.n), c = (int)(e % M.n);
            if (r < M.nao && c < M.nao) continue;
            fa.S[M.mat0 + e] = (r == c) ? 1.0 : 0.0;
            fa.H0[M.mat0 + e] = 0.0;
        }
    }
    repulsion_molecule<NT>(b, par, fa.pos, outs, M.m, (double*)sh.red);
    __syncthreads();
}

// One molecule's analytic gradient by its own workgroup, with the per-pair
// code of k_grad_pairs and k_grad_cn but no atomics: each atom pair A < B
// writes its terms to `scr` (the molecule's F buffer, free once W is formed:
// n^2 doubles, and every H, C, N, O atom carries at least two orbitals, so
// n^2 >= 4 nat^2 > 5 nat (nat - 1) / 2), then eight lanes add each atom's pairs
// in a fixed order; so the gradient has the same bits on every run.  Then the
// CN chain rule the same way.  The pairs are dealt to the threads by class
// (both atoms with p shells, one, none), as the shell pairs of the integrals:
// 26 atoms 301 -> 72 us, 77 760 -> 339 us (a wave per atom).  dE/dCN goes to fa.dedcn, dE/dR to fa.grad.
__device__ __noinline__ void molecule_forces(const ldsf* ctx) {
    const Mol M = CTX_GET(ctx, M);
    const Shared sh = CTX_GET(ctx, sh);
    kargs* ka = CTX_GET(ctx, ka);
    const xtb_batch b = karg_load(&ka->b);
    const xtb_params par = karg_load(&ka->par);
    const FusedArgs fa = karg_load(&ka->fa);
    const int w = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
    const int nat = M.nat, n = M.n;
    double* scr = (double*)M.F;
    if (5 * ((size_t)nat * (nat - 1) / 2) > (size_t)n * n) {
        for (int e = threadIdx.x; e < 3 * nat; e += NT) fa.grad[3 * (size_t)M.at0 + e] = NAN;
        return;
    }
    double* s_alpha = (double*)sh.big;
    double* s_coeff = s_alpha + XTB_MAX_US_LDS * XTB_MAXPRIM;
    for (int i = threadIdx.x; i < par.nus * XTB_MAXPRIM; i += NT) {
        s_alpha[i] = par.us_alpha[i];
        s_coeff[i] = par.us_coeff[i];
    }
    __syncthreads();
    auto pidx = [nat](int A, int B) { return (size_t)A * (2 * nat - A - 1) / 2 + (size_t)(B - A - 1); };
    const double* P = (const double*)M.P;
    // atoms with p shells, and those without, in order
    ldsi* lh = (ldsi*)(sh.big + 2 * XTB_MAX_US_LDS * XTB_MAXPRIM);
    ldsi* ll = lh + nat;
    int nh = 0;
    for (int a0 = 0; a0 < nat; a0 += WAVE) {
        const int a = a0 + lane;
        bool p = false;
        if (a < nat)
            for (int s = M.atom_sh0[a]; s < M.atom_sh0[a] + M.atom_nsh[a]; ++s) p = p || M.us_l[M.sh_us[s]] != 0;
        const uint64_t mh = __ballot(p), ml = __ballot(a < nat && !p), below = (1ull << lane) - 1;
        if (w == 0 && a < nat) {
            if (p) lh[nh + __popcll(mh & below)] = a;
            else ll[a0 - nh + __popcll(ml & below)] = a;
        }
        nh += __popcll(mh);
    }
    const int nl = nat - nh;
    __syncthreads();
    const int n3 = nh * (nh - 1) / 2, n2 = nh * nl, n1 = nl * (nl - 1) / 2;
    const int e2 = (n3 + WAVE - 1) / WAVE * WAVE, e1 = e2 + (n2 + WAVE - 1) / WAVE * WAVE;
    for (int t = threadIdx.x; t < e1 + n1; t += NT) {
        int r, c, A, B;
        if (t < e2) {
            if (t >= n3) continue;
            triangle(nh - 1, t, r, c);
            A = lh[r];
            B = lh[c + 1];
        } else if (t < e1) {
            if (t - e2 >= n2) continue;
            const int x = (int)((uint32_t)(t - e2) / (uint32_t)nl), h = lh[x], l = ll[t - e2 - x * nl];
            A = h < l ? h : l;
            B = h < l ? l : h;
        } else {
            triangle(nl - 1, t - e1, r, c);
            A = ll[r];
            B = ll[c + 1];
        }
        double g[3], dA, dB;
        atom_pair_grad(b, par, fa.pos, fa.cn, (const double*)M.gam, (const double*)M.qsh_out, P, (const double*)M.T,
                       (const double*)M.pot, n, M.nsh, M.sh0, M.at0 + A, M.at0 + B, s_alpha, s_coeff, g, dA, dB);
        double* e = scr + 5 * pidx(A, B);
        e[0] = g[0];
        e[1] = g[1];
        e[2] = g[2];
        e[3] = dA;
        e[4] = dB;
    }
    __syncthreads();
    // sums over the eight lanes of an atom (every lane takes part)
    auto over8 = [](double v) {
#pragma unroll
        for (int o = 1; o < 8; o <<= 1) v += __shfl_xor(v, o, WAVE);
        return v;
    };
    const int part = threadIdx.x % 8;
    for (int A0 = 0; A0 < nat; A0 += NT / 8) {
        const int A = A0 + (int)threadIdx.x / 8;
        double g[3] = {0.0, 0.0, 0.0}, d = 0.0;
        for (int B = part; B < nat && A < nat; B += 8) {
            if (B == A) continue;
            const bool low = B < A;
            const double* e = scr + 5 * (low ? pidx(B, A) : pidx(A, B));
            for (int k = 0; k < 3; ++k) g[k] += low ? -e[k] : e[k];
            d += e[low ? 4 : 3];
        }
        for (int k = 0; k < 3; ++k) g[k] = over8(g[k]);
        d = over8(d);
        if (A >= nat || part != 0) continue;
        d += onsite_dedcn(b, par, P, n, M.sh0, M.at0 + A);
        fa.dedcn[M.at0 + A] = d;
        for (int k = 0; k < 3; ++k) fa.grad[3 * (size_t)(M.at0 + A) + k] = g[k];
    }
    __syncthreads();
    for (int t = threadIdx.x; t < nat * (nat - 1) / 2; t += NT) {
        int A, B;
        triangle(nat - 1, t, A, B);
        ++B;
        double g[3] = {0.0, 0.0, 0.0};
        cn_pair_grad(b, par, fa.pos, fa.dedcn, M.at0 + A, M.at0 + B, g);
        double* e = scr + 3 * pidx(A, B);
        e[0] = g[0];
        e[1] = g[1];
        e[2] = g[2];
    }
    __syncthreads();
    for (int A0 = 0; A0 < nat; A0 += NT / 8) {
        const int A = A0 + (int)threadIdx.x / 8;
        double g[3] = {0.0, 0.0, 0.0};
        for (int B = part; B < nat && A < nat; B += 8) {
            if (B == A) continue;
            const bool low = B < A;
            const double* e = scr + 3 * (low ? pidx(B, A) : pidx(A, B));
            for (int k = 0; k < 3; ++k) g[k] += low ? -e[k] : e[k];
        }
        for (int k = 0; k < 3; ++k) g[k] = over8(g[k]);
        if (A >= nat || part != 0) continue;
        for (int k = 0; k < 3; ++k) fa.grad[3 * (size_t)(M.at0 + A) + k] += g[k];
    }
    __syncthreads();
}

__global__ void __launch_bounds__(NT) k_singlepoint(const ScfArgs args) {
    constexpr bool FUSED = true;
#include "scf_body.inc"
}

}  // namespace xtb

using namespace xtb;

extern "C" int32_t xtb_singlepoint(const xtb_batch* batch, const xtb_params* par, const double* positions,
                                   double* S, double* H0, double* cn, double* gamma, const xtb_scf_opts* opts,
                                   const xtb_scf_state* state, double* dedcn, double* grad, void* stream) {
    if (!batch || !par || !positions || !S || !H0 || !cn || !gamma || !opts || !state) return XTB_EINVAL;
    if (opts->want_w && (!dedcn || !grad)) return XTB_EINVAL;
    int rc = check_scf_args(batch, opts, state);
    if (rc != XTB_OK) return rc;
    // the primitives of every unique shell are staged in the eigensolver's
    // LDS region (at least NGEMM_MFMA_LDS doubles)
    if (par->nus > XTB_MAX_US_LDS || 2 * XTB_MAX_US_LDS * XTB_MAXPRIM > NGEMM_MFMA_LDS) return XTB_ETOOBIG;
    int32_t bytes = 0, cap = 0;
    rc = xtb_scf_lds_bytes(batch, &bytes, &cap);
    if (rc != XTB_OK) return rc;
    if (hipFuncSetAttribute((const void*)k_singlepoint, hipFuncAttributeMaxDynamicSharedMemorySize, bytes) !=
        hipSuccess)
        return XTB_EHIP;
    const ScfArgs args{*batch, *par, S, H0, gamma, *opts, *state, {positions, cn, S, H0, gamma, dedcn, grad}, cap};
    hipLaunchKernelGGL(k_singlepoint, dim3(batch->nmol + opts->wg_skip), dim3(NT), bytes, (hipStream_t)stream, args);
    return hipGetLastError() == hipSuccess ? XTB_OK : XTB_EHIP;
}
