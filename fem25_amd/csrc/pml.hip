// Element matrices integrated per omega (gfx950), by sum factorisation at the
// reference's 2 p + 5 points per direction:
//  * PML elements ('A', CM25ISOQ estiff25.f:168-334 with CJACCQ's stretch,
//    cjac.f:399-581)
//  * with quality factors (qp != null) every element in the density-
//    normalised dispersive form: KMDAMP (estiff25.f:511-752) and, for 'A'
//    elements, CMDAMP (estiff25.f:756-961), velocities from VCMPLX.
// Both are the KM25ISOQ bilinear forms with complex coefficients at each
// quadrature point: lambda -> L, mu -> M, rho -> R, derivatives stretched by
// 1/e_x, 1/e_z (ZDAMPFN) inside PML elements:
//   standard:   L = w lambda, M = w mu, R = w rho
//   dispersive: L = w (Vp~^2 - 2 Vs~^2), M = w Vs~^2, R = w.
//
// Every component block of the element matrix is a sum over the points of
// coefficient C(q) times a product of two basis functions or reference
// derivatives.  With N_b = v_bi(xi) v_bj(eta) it is contracted over xi first,
//   G[ai][bi][eta] = sum_xi C f_ai f_bi   (f: v or v'),
// then over eta: N1^2 Q1^2 + N1^4 Q1 products for one C instead of
// N1^4 Q1^2.  A workgroup forms one block of one element (blocks of an
// element touch different values of the operator): its points once, one
// thread each, four coefficients a point.
#pragma once

namespace f25k {

// Blocks: component pairs (1,1), (2,2), (3,3), (1,3), (1,2), (2,3) of the
// operator; 6 and 7 the ky^2 parts of the diagonal blocks, M N N and
// (L + 2 M) N N.  (3,1) is the transpose of (1,3), (2,1) and (3,2) minus the
// transposes of (1,2) and (2,3).
enum { PB_11 = 0, PB_22, PB_33, PB_13, PB_12, PB_23, PB_M, PB_L2, NPB };

template <int NL>
struct PmlSf {
    static constexpr int N1 = NL, Q1 = 2 * NL + 3, Q = Q1 * Q1, NEN = NL * NL, NEE = 3 * NEN;
    // threads: the Q points and the N1^3 items of the last stage in one or two rounds
    static constexpr int NT = NL <= 4 ? 128 : (NL == 5 ? 192 : (NL == 6 ? 256 : 384));
    static constexpr int NG = N1 * N1 * Q1;
    static constexpr size_t lds = (size_t)(4 * Q + 4 * NG) * sizeof(double2) + (2 * N1 * Q1 + NEE) * sizeof(double);
};

// Moduli L, M, density R (all times the quadrature weight and det J), stretch
// ex, ez and the reference derivatives' factors at point (ix, iz) of element e.
struct PmlPoint { double2 L, M, ex, ez; double R, rx, sx, rz, sz; };
__device__ inline PmlPoint pml_at(int e, int ix, int iz, const double *__restrict__ wq, const double *__restrict__ xq,
                                  const int *__restrict__ ieng, const double *__restrict__ xl,
                                  const double *__restrict__ zl, const double *__restrict__ xd,
                                  const double *__restrict__ zd, bool pml, const double *__restrict__ rho,
                                  const double *__restrict__ lam, const double *__restrict__ mu,
                                  const double2 *__restrict__ vps, const double *__restrict__ qp, const double *__restrict__ qs, const PmlPar &par,
                                  int *__restrict__ err) {
    const int *ie = ieng + 4 * e;
    Geo g;
    const int bad = geo_at(xq[ix], xq[iz], ie, xl, zl, g);
    if (bad) *err = 2;
    const double rj = bad ? 1.0 : g.det;
    PmlPoint p;
    p.rx = g.dzdeta / rj; p.sx = -g.dzdxi / rj; p.rz = -g.dxdeta / rj; p.sz = g.dxdxi / rj;
    const double w = wq[ix] * wq[iz] * g.det;
    double r = 0, l = 0, m = 0, xdep = 0, zdep = 0, vel = 0, vsv = 0, qpv = 0, qsv = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int gi = ie[k] - 1;
        r += g.sf[k] * rho[gi];
        l += g.sf[k] * lam[gi];
        m += g.sf[k] * mu[gi];
        if (pml) {
            xdep += g.sf[k] * xd[gi];
            zdep += g.sf[k] * zd[gi];
        }
        const double2 v = vps[gi];
        vel += g.sf[k] * v.x;
        if (qp) {
            vsv += g.sf[k] * v.y;
            qpv += g.sf[k] * qp[gi];
            qsv += g.sf[k] * qs[gi];
        }
    }
    const double2 one = make_double2(1.0, 0.0);
    p.ex = xdep > 2.22e-16 ? zdampfn(xdep, vel, par.xwidth, par.dmax, par.rcoeff, par.fcent, par.omega, par.kappa) : one;
    p.ez = zdep > 2.22e-16 ? zdampfn(zdep, vel, par.zwidth, par.dmax, par.rcoeff, par.fcent, par.omega, par.kappa) : one;
    if (qp) {
        const double2 zp = vcmplx(par.freq, par.freq0, vel, qpv), zs = vcmplx(par.freq, par.freq0, vsv, qsv);
        double2 zp2 = cmul(zp, zp), zs2 = cmul(zs, zs);
        zp2.x *= w; zp2.y *= w; zs2.x *= w; zs2.y *= w;
        p.L = make_double2(zp2.x - 2.0 * zs2.x, zp2.y - 2.0 * zs2.y);
        p.M = zs2;
        p.R = w;
    } else {
        p.L = make_double2(w * l, 0.0);
        p.M = make_double2(w * m, 0.0);
        p.R = w * r;
    }
    return p;
}

__device__ __forceinline__ double2 cadd(double2 a, double2 b) { return make_double2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ double2 cscale(double s, double2 a) { return make_double2(s * a.x, s * a.y); }
__device__ __forceinline__ double2 cimul(double s, double2 a) { return make_double2(-s * a.y, s * a.x); }   // i s a
__device__ __forceinline__ void cfma(double2 &a, double s, double2 b) { a.x = fma(s, b.x, a.x); a.y = fma(s, b.y, a.y); }

// The four coefficients of block kb at a point.  Diagonal blocks: of
// (xi xi), (xi eta) both ways, (eta eta), (N N); (1,3): (xi xi), (xi eta),
// (eta xi), (eta eta); (1,2), (2,3): (xi N), (eta N), (N xi), (N eta).
__device__ inline void pml_coef(int kb, const PmlPoint &p, double k, double w2, double2 *c) {
    const double2 px = cscale(p.rx, p.ex), qx = cscale(p.sx, p.ex), pz = cscale(p.rz, p.ez), qz = cscale(p.sz, p.ez);
    const double2 L2 = cadd(p.L, cscale(2.0, p.M));
    const double2 z = make_double2(0.0, 0.0);
    if (kb <= PB_33) {
        const double2 c1 = kb == PB_11 ? L2 : p.M, c2 = kb == PB_33 ? L2 : p.M;
        c[0] = cadd(cmul(c1, cmul(px, px)), cmul(c2, cmul(pz, pz)));
        c[1] = cadd(cmul(c1, cmul(px, qx)), cmul(c2, cmul(pz, qz)));
        c[2] = cadd(cmul(c1, cmul(qx, qx)), cmul(c2, cmul(qz, qz)));
        c[3] = cscale(k * k, kb == PB_22 ? L2 : p.M);
        c[3].x -= w2 * p.R;
    } else if (kb == PB_13) {
        c[0] = cmul(cadd(p.L, p.M), cmul(px, pz));
        c[1] = cadd(cmul(p.L, cmul(px, qz)), cmul(p.M, cmul(pz, qx)));
        c[2] = cadd(cmul(p.L, cmul(qx, pz)), cmul(p.M, cmul(qz, px)));
        c[3] = cmul(cadd(p.L, p.M), cmul(qx, qz));
    } else if (kb == PB_12) {   // -i ky (L X_a N_b - M N_a X_b)
        c[0] = cimul(-k, cmul(p.L, px));
        c[1] = cimul(-k, cmul(p.L, qx));
        c[2] = cimul(k, cmul(p.M, px));
        c[3] = cimul(k, cmul(p.M, qx));
    } else if (kb == PB_23) {   // i ky (L N_a Z_b - M Z_a N_b)
        c[0] = cimul(-k, cmul(p.M, pz));
        c[1] = cimul(-k, cmul(p.M, qz));
        c[2] = cimul(k, cmul(p.L, pz));
        c[3] = cimul(k, cmul(p.L, qz));
    } else {
        c[0] = c[1] = c[2] = z;
        c[3] = kb == PB_M ? p.M : L2;
    }
}

// (Vp, Vs) at the anchors, the velocities pml_at interpolates
__global__ void k_anchor_vel(int n, const double *__restrict__ rho, const double *__restrict__ lam,
                             const double *__restrict__ mu, double2 *__restrict__ vps) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) vps[i] = make_double2(sqrt((lam[i] + 2.0 * mu[i]) / rho[i]), sqrt(mu[i] / rho[i]));
}

// Positions of the element rows' and columns' values in CSR order, relative
// to the row's start, -1 where a DOF is fixed: pos[slot][row][col].  Built
// once per list of elements; a pair missing from the pattern sets err = 3.
__global__ void k_pml_pos(int nee, const int *__restrict__ order, const int *__restrict__ lm,
                          const int64_t *__restrict__ irptr, const int *__restrict__ jcptr, int *__restrict__ pos,
                          int *__restrict__ err) {
    const int *L = lm + (size_t)order[blockIdx.x] * nee;
    int *o = pos + (size_t)blockIdx.x * nee * nee;
    for (int i = threadIdx.x; i < nee * nee; i += blockDim.x) {
        const int rd = L[i / nee], cd = L[i % nee];
        int v = -1;
        if (rd >= 0 && cd >= 0) {
            const int64_t s = find_col(jcptr, irptr[rd], irptr[rd + 1], cd);
            if (s < 0) *err = 3;
            else v = (int)(s - irptr[rd]);
        }
        o[i] = v;
    }
}

// One block of one element.  SPLIT: the blocks by power of ky of omega
// omf[f0 + blockIdx.z], mats[slot][omega][block][a][b] (block 0..3 without ky and
// with the -omega^2 mass, 4 and 5 per ky, 6 and 7 per ky^2).  Otherwise the
// operator at par, added into CSR order (one launch per colour: no two of its
// elements share a value).
//
// Bound by latency: a few hundred workgroups a colour, each a chain of four
// short stages; the values it adds to are loaded before the last one.
// Measured on MI355X per colour against the direct sums (one workgroup per
// element, geometry per node, a search of the pattern per value): 198 PML
// elements at p4, COMPLEX*8, 445 -> 63 -> about 30 us; 528 dispersive
// elements at p4, COMPLEX*16, 825 -> 136 -> about 65 us (the second step:
// velocities per anchor, loads ahead of the sums, loops over the points not
// unrolled, 122 registers instead of 432).
template <int NL, bool SPLIT, typename CT>
__global__ __launch_bounds__((PmlSf<NL>::NT)) void k_pml_sf(
        int slot0, int nom, int f0, const int *__restrict__ order, const double *__restrict__ omf,
        const double *__restrict__ t1d, const double *__restrict__ wq, const double *__restrict__ xq,
        const int *__restrict__ ieng, const double *__restrict__ xl, const double *__restrict__ zl,
        const double *__restrict__ xd, const double *__restrict__ zd, const char *__restrict__ cdom,
        const double *__restrict__ rho, const double *__restrict__ lam, const double *__restrict__ mu,
        const double2 *__restrict__ vps, const double *__restrict__ qp, const double *__restrict__ qs, PmlPar par, const int *__restrict__ lm,
        const int64_t *__restrict__ irptr, const int *__restrict__ pos, CT *__restrict__ out, int *__restrict__ err) {
    typedef PmlSf<NL> S;
    constexpr int N1 = S::N1, Q1 = S::Q1, Q = S::Q, NEN = S::NEN, NEE = S::NEE, NT = S::NT, NG = S::NG;
    extern __shared__ double sm[];
    double2 *sC = reinterpret_cast<double2 *>(sm);   // [4][Q]
    double2 *sG = sC + 4 * Q;                        // [4][eta][ai][bi]
    double *sv = reinterpret_cast<double *>(sG + 4 * NG), *sd = sv + N1 * Q1;   // v, v' [q][i]
    int64_t *sr = reinterpret_cast<int64_t *>(sd + N1 * Q1);                     // the rows' starts in CSR order
    const int e = order[blockIdx.x], kb = blockIdx.y, tid = threadIdx.x;
    if constexpr (SPLIT) {
        par.omega = omf[f0 + blockIdx.z];
        par.freq = par.omega / (2.0 * M_PI);
        par.kv = kb == PB_12 || kb == PB_23 ? 1.0 : 0.0;
    }
    for (int i = tid; i < N1 * Q1; i += NT) {
        sv[i] = t1d[(i % N1) * Q1 + i / N1];
        sd[i] = t1d[(N1 + i % N1) * Q1 + i / N1];
    }
    if constexpr (!SPLIT)
        for (int i = tid; i < NEE; i += NT) {
            const int d = lm[(size_t)e * NEE + i];
            sr[i] = d >= 0 ? irptr[d] : 0;
        }
    const bool pml = cdom[e] == 'A';
    for (int q = tid; q < Q; q += NT) {
        double2 c[4];
        pml_coef(kb, pml_at(e, q % Q1, q / Q1, wq, xq, ieng, xl, zl, xd, zd, pml, rho, lam, mu, vps, qp, qs, par, err),
                 par.kv, par.omega * par.omega, c);
#pragma unroll
        for (int k = 0; k < 4; ++k) sC[k * Q + q] = c[k];
    }
    __syncthreads();
    // over xi.  g[0]: the sums that go with v_aj v_bj, g[1] v_aj v'_bj,
    // g[2] v'_aj v_bj, g[3] v'_aj v'_bj
    for (int it = tid; it < NG; it += NT) {
        const int bi = it % N1, ai = (it / N1) % N1, qe = it / (N1 * N1);
        double2 g[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) g[k] = make_double2(0.0, 0.0);
        const double2 *C = sC + qe * Q1;
        if (kb <= PB_33) {
#pragma unroll 2
            for (int x = 0; x < Q1; ++x) {
                const double va = sv[x * N1 + ai], vb = sv[x * N1 + bi], da = sd[x * N1 + ai], db = sd[x * N1 + bi];
                cfma(g[0], da * db, C[x]);
                cfma(g[0], va * vb, C[3 * Q + x]);
                cfma(g[1], da * vb, C[Q + x]);
                cfma(g[2], va * db, C[Q + x]);
                cfma(g[3], va * vb, C[2 * Q + x]);
            }
        } else if (kb == PB_13) {
#pragma unroll 2
            for (int x = 0; x < Q1; ++x) {
                const double va = sv[x * N1 + ai], vb = sv[x * N1 + bi], da = sd[x * N1 + ai], db = sd[x * N1 + bi];
                cfma(g[0], da * db, C[x]);
                cfma(g[1], da * vb, C[Q + x]);
                cfma(g[2], va * db, C[2 * Q + x]);
                cfma(g[3], va * vb, C[3 * Q + x]);
            }
        } else if (kb <= PB_23) {
#pragma unroll 2
            for (int x = 0; x < Q1; ++x) {
                const double va = sv[x * N1 + ai], vb = sv[x * N1 + bi], da = sd[x * N1 + ai], db = sd[x * N1 + bi];
                cfma(g[0], da * vb, C[x]);
                cfma(g[0], va * db, C[2 * Q + x]);
                cfma(g[1], va * vb, C[3 * Q + x]);
                cfma(g[2], va * vb, C[Q + x]);
            }
        } else {
            for (int x = 0; x < Q1; ++x) cfma(g[0], sv[x * N1 + ai] * sv[x * N1 + bi], C[3 * Q + x]);
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) sG[k * NG + it] = g[k];
    }
    __syncthreads();
    // over eta: a thread per (aj, ai, bi), the N1 entries of bj
    const int ci = kb == PB_22 || kb == PB_23 ? 1 : (kb == PB_33 ? 2 : 0);
    const int cj = kb == PB_11 ? 0 : (kb == PB_22 || kb == PB_12 ? 1 : 2);
    for (int it = tid; it < N1 * N1 * N1; it += NT) {
        const int bi = it % N1, ai = (it / N1) % N1, aj = it / (N1 * N1), a = aj * N1 + ai;
        const int ra = 3 * a + ci;
        // the values this thread adds to, loaded before the sums (for a fixed
        // row or column the element's first value of the row start: not stored)
        [[maybe_unused]] CT *po[N1], *pt[N1];
        [[maybe_unused]] CT vo[N1], vt[N1];
        [[maybe_unused]] bool ok[N1];
        if constexpr (!SPLIT) {
            const int *P = pos + (size_t)(slot0 + blockIdx.x) * NEE * NEE;
            int p[N1], t[N1];
#pragma unroll
            for (int j = 0; j < N1; ++j) {
                const int cb = 3 * (j * N1 + bi) + cj;
                p[j] = P[ra * NEE + cb];
                t[j] = P[cb * NEE + ra];
            }
#pragma unroll
            for (int j = 0; j < N1; ++j) {
                const int cb = 3 * (j * N1 + bi) + cj;
                ok[j] = p[j] >= 0;
                po[j] = out + sr[ra] + (ok[j] ? p[j] : 0);
                pt[j] = out + sr[cb] + (ok[j] ? t[j] : 0);
                vo[j] = *po[j];
                if (ci != cj) vt[j] = *pt[j];
            }
        }
        double2 s[N1];
#pragma unroll
        for (int j = 0; j < N1; ++j) s[j] = make_double2(0.0, 0.0);
#pragma unroll 1
        for (int y = 0; y < Q1; ++y) {
            const double2 *g = sG + (y * N1 + ai) * N1 + bi;
            const double va = sv[y * N1 + aj], da = sd[y * N1 + aj];
            double2 t0 = cscale(va, g[0]), t1 = cscale(va, g[NG]);
            cfma(t0, da, g[2 * NG]);
            cfma(t1, da, g[3 * NG]);
#pragma unroll
            for (int j = 0; j < N1; ++j) {
                cfma(s[j], sv[y * N1 + j], t0);
                cfma(s[j], sd[y * N1 + j], t1);
            }
        }
        if constexpr (SPLIT) {
            CT *o = out + ((((size_t)(slot0 + blockIdx.x) * nom + f0 + blockIdx.z) * NPB + kb) * NEN + a) * NEN + bi;
#pragma unroll
            for (int j = 0; j < N1; ++j) o[j * N1] = CT{s[j].x, s[j].y};
        } else {
            const double sg = kb == PB_13 ? 1.0 : -1.0;
#pragma unroll
            for (int j = 0; j < N1; ++j) {
                if (!ok[j]) continue;
                vo[j].x += s[j].x;
                vo[j].y += s[j].y;
                *po[j] = vo[j];
                if (ci == cj) continue;
                vt[j].x += sg * s[j].x;
                vt[j].y += sg * s[j].y;
                *pt[j] = vt[j];
            }
        }
    }
}

// ---------------------------------------------------------------------------
// y_b += S_e(omega_b, ky_b) x_b over the elements of one colour whose blocks
// k_pml_sf<SPLIT> holds, after the element product has written y (it stores
// zero rows for PML elements; for a dispersive medium y is zero-filled
// first).  Workgroup (element, group of up to PML_GP pairs of one omega), a
// wave per output component and tile of 16 rows: FP64 MFMA over the element's
// nodes, four at a time, columns eight pairs' real and imaginary parts.  A
// complex block A acts on a pair's columns as Re A (re, im) + Im A (-im, re);
// its ky or ky^2 goes to the column, so one read of a tile serves every pair
// of the omega.  Per component: the diagonal block, its ky^2 part and the two
// couplings; transposed blocks are read transposed.  grp[3 g + 0..2] = (omega
// index, first slot in gpair, count).  Arithmetic in FP64 for every vector
// type.
//
// Bound by latency, then memory: eight blocks an element and omega (80 KB at
// p4) are read once, 330 MB a colour with x and y (70 us at the rate of a
// copy).  Measured on MI355X, 198 elements of one colour at p4, 240 pairs of
// 10 omegas: nine blocks for each power of ky, read per 16 pairs, on the
// vector ALUs 696 us; this form 217 us, and 165 us with the gather's, the
// tiles' and the rows' loads issued together (four waves per SIMD: at 130
// registers one workgroup of six waves fits a CU instead of two).
constexpr int PML_GP = 32;   // pairs of a group

template <int NL>
struct PmlApply {
    static constexpr int NEN = NL * NL, NEE = 3 * NEN, MT = (NEN + 15) / 16, KS = (NEN + 3) / 4, KN = 4 * KS;
    static constexpr int NT = 64 * 3 * MT;
    static constexpr size_t lds = (size_t)3 * KN * PML_GP * sizeof(double2);
};

template <int NL, typename XT>
__global__ __launch_bounds__((PmlApply<NL>::NT)) __attribute__((amdgpu_waves_per_eu(4))) void k_apply_pml(int slot0, int nom, const int *__restrict__ order,
                                                                  const int *__restrict__ lm, const int *__restrict__ grp,
                                                                  const int *__restrict__ gpair, int npair,
                                                                  const double *__restrict__ ky,
                                                                  const double2 *__restrict__ mats,
                                                                  const XT *__restrict__ x, XT *__restrict__ y) {
    typedef PmlApply<NL> S;
    typedef MfmaTraits<double> MF;
    typedef decltype(XT().x) R;
    constexpr int NEN = S::NEN, NEE = S::NEE, MT = S::MT, KS = S::KS, KN = S::KN, GP = PML_GP;
    extern __shared__ double2 xs[];   // [component][node][pair], zero past the last node and pair
    const int e = order[blockIdx.x], g = blockIdx.y, tid = threadIdx.x, lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6), ci = wv / MT, mt = wv % MT;
    const int f = grp[3 * g], first = grp[3 * g + 1], cnt = grp[3 * g + 2];
    const int *L = lm + (size_t)e * NEE;
    // a thread gathers pair tid % GP of rows tid / GP + k NT / GP: its loads
    // are issued together
    constexpr int RS = S::NT / GP, NR = (3 * KN + RS - 1) / RS;
    {
        const int p = tid % GP, r0 = tid / GP;
        const size_t pair = gpair[first + min(p, cnt - 1)];
        int d[NR];
        XT t[NR];
#pragma unroll
        for (int k = 0; k < NR; ++k) d[k] = L[min(r0 + k * RS, NEE - 1)];
#pragma unroll
        for (int k = 0; k < NR; ++k) t[k] = x[(size_t)max(d[k], 0) * npair + pair];
#pragma unroll
        for (int k = 0; k < NR; ++k) {
            const int r = r0 + k * RS;
            const bool in = r < NEE && d[k] >= 0 && p < cnt;
            if (r < 3 * KN)
                xs[((r % 3) * KN + r / 3) * GP + p] =
                    in ? make_double2((double)t[k].x, (double)t[k].y) : make_double2(0.0, 0.0);
        }
    }
    // this wave's four blocks: (block, transposed, input component)
    const int t3 = ci == 1 ? PB_12 : PB_13, c3 = ci == 0 ? 2 : 0;      // 13 x3 | -12^T k x1 | 13^T x1
    const int t4 = ci == 0 ? PB_12 : PB_23, c4 = ci == 1 ? 2 : 1;      // 12 k x2 | 23 k x3 | -23^T k x2
    const int tb[4] = {ci, ci == 1 ? PB_L2 : PB_M, t3, t4}, ic[4] = {ci, ci, c3, c4};
    const bool tr[4] = {false, false, ci != 0, ci == 2};
    const double2 *mb = mats + ((size_t)(slot0 + blockIdx.x) * nom + f) * NPB * NEN * NEN;
    const int m = mt * 16 + (lane & 15), kg = lane >> 4, col = lane & 15, part = col & 1;
    const double2 *ab[4];
    int sb[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        const int mc = min(m, NEN - 1);
        ab[t] = mb + (size_t)tb[t] * NEN * NEN + (tr[t] ? mc : mc * NEN);
        sb[t] = tr[t] ? NEN : 1;
    }
    const int nch = (cnt + 7) / 8;
    // column factors of the couplings, of the ky^2 block, per chunk of pairs
    constexpr int NC = GP / 8;
    double f2[NC], f3[NC], f4[NC];
#pragma unroll
    for (int h = 0; h < NC; ++h) {
        const int p = h * 8 + (col >> 1);
        const double k = p < cnt ? ky[gpair[first + p]] : 0.0;
        f2[h] = k * k;
        f3[h] = ci == 1 ? -k : 1.0;
        f4[h] = ci == 2 ? -k : k;
    }
    typedef typename MF::v4 V4;
    V4 acc[NC];
#pragma unroll
    for (int h = 0; h < NC; ++h) acc[h] = V4{0.0, 0.0, 0.0, 0.0};
    // rows of y this lane adds to, and the blocks' tiles of the first four nodes
    int dr[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int a = mt * 16 + MF::row(kg, i), d = L[3 * min(a, NEN - 1) + ci];
        dr[i] = a < NEN ? d : -1;
    }
    double2 A[4], An[4];
    auto load = [&](int s, double2 *v) {
        const int bc = min(4 * s + kg, NEN - 1);
#pragma unroll
        for (int t = 0; t < 4; ++t) v[t] = ab[t][bc * sb[t]];
    };
    load(0, An);
    __syncthreads();
#pragma unroll 2
    for (int s = 0; s < KS; ++s) {
        const int b = 4 * s + kg;
        const bool in = b < NEN && m < NEN;
#pragma unroll
        for (int t = 0; t < 4; ++t) A[t] = in ? An[t] : make_double2(0.0, 0.0);
        load(min(s + 1, KS - 1), An);   // the next tiles while these multiply
#pragma unroll
        for (int h = 0; h < NC; ++h) {
            if (h >= nch) break;
            const int o = b * GP + h * 8 + (col >> 1);
            const double2 v0 = xs[ic[0] * KN * GP + o], v3 = xs[ic[2] * KN * GP + o], v4 = xs[ic[3] * KN * GP + o];
            // (re, im) and (-im, re) of the column's part
            const double b0 = part ? v0.y : v0.x, d0 = part ? v0.x : -v0.y;
            const double b3 = f3[h] * (part ? v3.y : v3.x), d3 = f3[h] * (part ? v3.x : -v3.y);
            const double b4 = f4[h] * (part ? v4.y : v4.x), d4 = f4[h] * (part ? v4.x : -v4.y);
            acc[h] = MF::mma(A[0].x, b0, acc[h]);
            acc[h] = MF::mma(A[0].y, d0, acc[h]);
            acc[h] = MF::mma(A[1].x, f2[h] * b0, acc[h]);
            acc[h] = MF::mma(A[1].y, f2[h] * d0, acc[h]);
            acc[h] = MF::mma(A[2].x, b3, acc[h]);
            acc[h] = MF::mma(A[2].y, d3, acc[h]);
            acc[h] = MF::mma(A[3].x, b4, acc[h]);
            acc[h] = MF::mma(A[3].y, d4, acc[h]);
        }
    }
    R *yp = reinterpret_cast<R *>(y) + part;
    R yv[NC][4];
    size_t po[NC];
#pragma unroll
    for (int h = 0; h < NC; ++h) {
        po[h] = gpair[first + min(h * 8 + (col >> 1), cnt - 1)];
#pragma unroll
        for (int i = 0; i < 4; ++i) yv[h][i] = yp[((size_t)max(dr[i], 0) * npair + po[h]) * 2];
    }
#pragma unroll
    for (int h = 0; h < NC; ++h)
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (dr[i] >= 0 && h * 8 + (col >> 1) < cnt)
                yp[((size_t)dr[i] * npair + po[h]) * 2] = (R)((double)yv[h][i] + acc[h][i]);
}

}  // namespace f25k
