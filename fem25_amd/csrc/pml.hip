// Element matrices integrated per omega (gfx950): PML elements and, in a
// dispersive medium, every element (CM25ISOQ, KMDAMP, CMDAMP; the moduli and
// the stretch as described in kernels.hip), by sum factorisation at the
// reference's 2 p + 5 points per direction.
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
// omf[blockIdx.z], mats[slot][omega][block][a][b] (block 0..3 without ky and
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
        int slot0, int nom, const int *__restrict__ order, const double *__restrict__ omf,
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
        par.omega = omf[blockIdx.z];
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
            CT *o = out + ((((size_t)(slot0 + blockIdx.x) * nom + blockIdx.z) * NPB + kb) * NEN + a) * NEN + bi;
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

}  // namespace f25k
