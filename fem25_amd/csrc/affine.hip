// Kernels for parallelogram elements (gfx950): the adjoint gradient by sum
// factorisation at the NL-point Gauss-Legendre rule.
//
// An element whose bilinear map is affine has a constant Jacobian, so every
// integrand of the element operator and of its model derivatives is a
// polynomial: GLL basis functions or their derivatives (degree at most p per
// direction, twice) times a bilinear coefficient, 2 p + 1 in all, which the
// (p + 1)-point Gauss rule integrates exactly.  The reference's 2 p + 5
// point rule (asmble.f90:110-112) gives the same integrals: the results
// differ by rounding only, at (p + 1)^2 instead of (2 p + 5)^2 points.
//
// With u_2 = i w the operator (kernels.hip, top) is real in (u_1, w, u_3):
//   div = X_1 + Z_3 + k w,  a12 = X_w - k u_1,  a23 = Z_w - k u_3,
//   a13 = Z_1 + X_3         (X, Z: x and z derivatives, k = ky)
// so a complex vector is two independent real problems, (Re u_1, Im u_2,
// Re u_3) and (Im u_1, Re u_2, Im u_3), the second with -k in place of k
// (its w is -Re u_2; the sign goes to k).  A lane owns one eta point of one
// real problem: its first pass contracts the element's values along eta with
// the lane's own 1-D values, everything along xi is then lane-local with
// wave-uniform coefficients.
#pragma once

namespace f25k {

// record of an element (k_aff_rec): rx, sx, rz, sz (d xi/dx, d eta/dx,
// d xi/dz, d eta/dz), det J, rho, lambda, mu at the four corners, 1 for a
// PML element
constexpr int AFR = 20;

// 1-D table (af_table on the host): v_j(q) [NL][NL], v'_j(q) [NL][NL], then
// w h_0, w h_1, h_0, h_1, w at the points (h_0, h_1 the hat functions)
template <int NL>
struct AfTab {
    static constexpr int V = 0, D = NL * NL, HW0 = 2 * NL * NL, HW1 = HW0 + NL, H0 = HW1 + NL, H1 = H0 + NL,
                         W = H1 + NL, SIZE = W + NL;
};

// Lanes of a wave: PP real problems (PW complex vectors) times NL eta points
// (60, 64, 60, 60, 56 lanes at p2..p6), lane = eta * PP + problem.
template <int NL>
struct AfShape {
    static constexpr int NEN = NL * NL, NEE = 3 * NEN;
    static constexpr int PP = (64 / NL) & ~1, PW = PP / 2, LN = PP * NL;
    static constexpr int NW = 4;                             // waves of a workgroup
    // the gradient's LDS per wave: element values of both fields for PW triples
    static constexpr int GS = 2 * NEE * PW;
    static constexpr size_t lds_grad = (size_t)NW * GS * 16 + 2 * NL * NL * 8;
};

__global__ void k_aff_rec(int nelem, const int *__restrict__ ieng, const double *__restrict__ xl,
                          const double *__restrict__ zl, const double *__restrict__ rho,
                          const double *__restrict__ lam, const double *__restrict__ mu,
                          const char *__restrict__ cdom, double *__restrict__ rec) {
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= nelem) return;
    double *o = rec + (size_t)e * AFR;
    int a[4];
    for (int k = 0; k < 4; ++k) a[k] = ieng[4 * e + k] - 1;
    const double xx = 0.25 * ((xl[a[1]] - xl[a[0]]) + (xl[a[2]] - xl[a[3]]));
    const double xe = 0.25 * ((xl[a[3]] - xl[a[0]]) + (xl[a[2]] - xl[a[1]]));
    const double zx = 0.25 * ((zl[a[1]] - zl[a[0]]) + (zl[a[2]] - zl[a[3]]));
    const double ze = 0.25 * ((zl[a[3]] - zl[a[0]]) + (zl[a[2]] - zl[a[1]]));
    const double det = xx * ze - xe * zx;
    o[0] = ze / det; o[1] = -zx / det; o[2] = -xe / det; o[3] = xx / det; o[4] = det;
    for (int k = 0; k < 4; ++k) { o[5 + k] = rho[a[k]]; o[9 + k] = lam[a[k]]; o[13 + k] = mu[a[k]]; }
    o[17] = cdom[e] == 'A' ? 1.0 : 0.0;
    o[18] = o[19] = 0.0;
}

// 16 bytes per lane from global memory straight into LDS (l: the wave's base,
// lane i's value lands at l + 16 i); complete after dma_wait.
__device__ __forceinline__ void dma16(const void *g, void *l) {
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)g,
                                     (__attribute__((address_space(3))) void *)l, 16, 0, 0);
}
__device__ __forceinline__ void dma_wait() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }
// the wave's own LDS accesses so far are complete, and stay before what follows
__device__ __forceinline__ void lds_wait() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

// Gathers one element's values of the wave's V vectors into its LDS region,
// [vector][NEE] values of 16 bytes: lane i takes element values i, i + 64, ...
// of each vector, so a load is a wave-uniform base (the vector) and a lane
// offset (the DOF) kept over the whole batch.  Fixed DOFs are not loaded:
// their values are set to zero once (zero).
template <int NEE, int V>
struct AfGather {
    static constexpr int K = (NEE + 63) / 64;
    int off[K];   // DOF of the lane's element value, -1: none
    __device__ __forceinline__ void init(int lane, const int *lm) {
#pragma unroll
        for (int k = 0; k < K; ++k) off[k] = lane + 64 * k < NEE ? lm[lane + 64 * k] : -1;
    }
    __device__ __forceinline__ void zero(int lane, double2 *dst) {
#pragma unroll
        for (int k = 0; k < K; ++k)
            if (lane + 64 * k < NEE && off[k] < 0)
                for (int v = 0; v < V; ++v) dst[v * NEE + lane + 64 * k] = make_double2(0.0, 0.0);
        lds_wait();
    }
    // base(v): the vector's values by DOF
    template <typename F>
    __device__ __forceinline__ void get(double2 *dst, F base) {
#pragma unroll
        for (int k = 0; k < K; ++k)
            if (off[k] >= 0)
#pragma unroll
                for (int v = 0; v < V; ++v) dma16(base(v) + off[k], dst + v * NEE + 64 * k);
    }
};

// First pass of one component: T1[i] = sum_j v_j(eta) a_ji, T2[i] the same
// with v'_j; a: LDS, node (j, i) at a[(j NL + i) * STEP].  x holds column 0 on
// entry and column 0 of the next component (an) on return: each column is
// read while the one before it is summed.
template <int NL, int STEP>
__device__ __forceinline__ void af_first(const double *a, const double *an, const double *v, const double *d,
                                         double *x, double *T1, double *T2) {
#pragma unroll
    for (int i = 0; i < NL; ++i) {
        double n[NL];
        const double *p = i + 1 < NL ? a + (i + 1) * STEP : an;
#pragma unroll
        for (int j = 0; j < NL; ++j) n[j] = p[j * NL * STEP];
        double t1 = v[0] * x[0], t2 = d[0] * x[0];
#pragma unroll
        for (int j = 1; j < NL; ++j) {
            t1 = fma(v[j], x[j], t1);
            t2 = fma(d[j], x[j], t2);
        }
        T1[i] = t1;
        T2[i] = t2;
        // formed here, not where they are used: the compiler would keep the
        // loaded values, NL^2 a component, instead of 2 NL sums
        asm volatile("" : "+v"(T1[i]), "+v"(T2[i]));
#pragma unroll
        for (int j = 0; j < NL; ++j) x[j] = n[j];
    }
}

// Value and reference derivatives at xi point q (vq, dq: its 1-D values).
template <int NL>
__device__ __forceinline__ void af_point(const double *T1, const double *T2, const double *vq, const double *dq,
                                         double &U, double &Xi, double &Et) {
    U = vq[0] * T1[0];
    Xi = dq[0] * T1[0];
    Et = vq[0] * T2[0];
#pragma unroll
    for (int i = 1; i < NL; ++i) {
        U = fma(vq[i], T1[i], U);
        Xi = fma(dq[i], T1[i], Xi);
        Et = fma(vq[i], T2[i], Et);
    }
}

// ---------------------------------------------------------------------------
// Gradient densities of parallelogram elements, projected on the corners:
// part[e][corner][lambda, mu, rho] as k_grad_sf leaves it.  One workgroup per
// element; its waves take chunks of PW triples in turn.  The densities
//   l: div_l div_u, m: 2 (X1 X1' + Z3 Z3' + k^2 w w') + a12 a12' + a23 a23' + a13 a13',
//   r: -omega^2 (u1 u1' + w w' + u3 u3')
// of a point are added into six sums per lane (two hats along xi); the hats
// along eta and the weights come once at the end.  RECT: every element's
// sides lie along x and z (sx = rz = 0), and T2 carries sz.
//
// Bound by latency at two waves per SIMD (T1, T2 of both fields are 12 NL doubles
// a lane, 168 of the 256 registers at p6).  Measured on MI355X: 200x100 p4, 128 triples
// 9.30 -> 1.62 ms (FP64 pipe about half busy, 4.5 GB from HBM of 3.9 GB read
// once); 121x59 p6, 45 triples 2.99 -> 0.56 ms.  On the way: slots numbered
// across vectors (index arithmetic per load) 2.03 ms at p4, one column at a
// time in the first pass (each waited for its LDS reads) 1.82; the point
// loop unrolled spills (p6 1.03 ms against 0.56), its 1-D values loaded one
// point ahead 1.67 ms.
template <int NL, bool RECT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void k_grad_af(
        const int *__restrict__ elems, const double *__restrict__ rec, const double *__restrict__ tab,
        const int *__restrict__ lm, int ntrip, int64_t ndof, const double *__restrict__ omega,
        const double *__restrict__ ky, const double2 *__restrict__ u, const double2 *__restrict__ l,
        double *__restrict__ part) {
    typedef AfShape<NL> S;
    typedef AfTab<NL> TB;
    constexpr int NEE = S::NEE, PP = S::PP, PW = S::PW, LN = S::LN;
    extern __shared__ double sm[];
    __shared__ double red[S::NW][12];
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int nw = blockDim.x >> 6;
    double2 *sw = reinterpret_cast<double2 *>(sm) + wv * S::GS;
    double *st = sm + S::NW * S::GS * 2;
    const int e = elems[blockIdx.x];
    const double *rc = rec + (size_t)e * AFR;
    if (rc[17] != 0.0) {   // PML elements are outside the gradient
        if (threadIdx.x < 12) part[(size_t)e * 12 + threadIdx.x] = 0.0;
        return;
    }
    for (int i = threadIdx.x; i < 2 * NL * NL; i += blockDim.x) st[i] = tab[i];
    __syncthreads();
    const int nch = (ntrip + PW - 1) / PW;
    typedef AfGather<NEE, 2 * PW> G;
    G ga;
    ga.init(lane, lm + (size_t)e * NEE);
    ga.zero(lane, sw);
    // vectors 0 .. PW - 1: u of the chunk's triples, then l
    auto base = [&](int t0) {
        return [=](int v) -> const double2 * {
            return (v >= PW ? l : u) + (size_t)min(t0 + v % PW, ntrip - 1) * ndof;
        };
    };
    if (wv < nch) ga.get(sw, base(wv * PW));
    const int le = min(lane, LN - 1), eta = le / PP, tr = (le % PP) >> 1, im = le & 1;
    const double rx = rc[0], sxx = rc[1], rz = rc[2], sz = rc[3];
    double g[6];
#pragma unroll
    for (int k = 0; k < 6; ++k) g[k] = 0.0;
    auto trip = [&](int ch) { return min(ch * PW + tr, ntrip - 1); };
    double omn = omega[trip(wv)], kyn = ky[trip(wv)];   // of the next chunk, loaded ahead with its values
    for (int ch = wv; ch < nch; ch += nw) {
        const int t = ch * PW + tr;
        const bool live = lane < LN && t < ntrip;
        const double w2 = -omn * omn, kv = im ? -kyn : kyn;
        dma_wait();
        double T1[2][3][NL], T2[2][3][NL];
        {
            double v[NL], d[NL];
#pragma unroll
            for (int j = 0; j < NL; ++j) { v[j] = st[eta * NL + j]; d[j] = (RECT ? sz : 1.0) * st[NL * NL + eta * NL + j]; }
            const double *a = reinterpret_cast<const double *>(sw + tr * NEE);
            auto at = [&](int k) {   // component k % 3 of field k / 3
                return a + (k / 3) * (2 * PW * NEE) + 2 * (k % 3) + (k % 3 == 1 ? 1 - im : im);
            };
            double x[NL];
#pragma unroll
            for (int j = 0; j < NL; ++j) x[j] = at(0)[j * NL * 6];
#pragma unroll
            for (int k = 0; k < 6; ++k)
                af_first<NL, 6>(at(k), at(k < 5 ? k + 1 : 0), v, d, x, T1[k / 3][k % 3], T2[k / 3][k % 3]);
        }
        lds_wait();
        if (ch + nw < nch) {
            ga.get(sw, base((ch + nw) * PW));
            omn = omega[trip(ch + nw)];
            kyn = ky[trip(ch + nw)];
        }
        double s[6];
#pragma unroll
        for (int k = 0; k < 6; ++k) s[k] = 0.0;
#pragma unroll 1
        for (int q = 0; q < NL; ++q) {
            const double *vq = tab + TB::V + q * NL, *dq = tab + TB::D + q * NL;
            const double a0 = tab[TB::HW0 + q], a1 = tab[TB::HW1 + q];
            double U[2][3], X0[2], Z2[2], div[2], a12[2], a23[2], a13[2];
#pragma unroll
            for (int f = 0; f < 2; ++f) {
                double X[3], Z[3];
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    double Xi, Et;
                    af_point<NL>(T1[f][c], T2[f][c], vq, dq, U[f][c], Xi, Et);
                    X[c] = RECT ? rx * Xi : rx * Xi + sxx * Et;
                    Z[c] = RECT ? Et : rz * Xi + sz * Et;
                }
                X0[f] = X[0];
                Z2[f] = Z[2];
                div[f] = X[0] + Z[2] + kv * U[f][1];
                a12[f] = X[1] - kv * U[f][0];
                a23[f] = Z[1] - kv * U[f][2];
                a13[f] = Z[0] + X[2];
            }
            const double uw = U[0][1] * U[1][1];
            const double dl = div[0] * div[1];
            const double dm = fma(2.0, fma(X0[0], X0[1], fma(Z2[0], Z2[1], kv * kv * uw)),
                                  fma(a12[0], a12[1], fma(a23[0], a23[1], a13[0] * a13[1])));
            const double dr = fma(U[0][0], U[1][0], fma(U[0][2], U[1][2], uw));
            s[0] = fma(a0, dl, s[0]); s[1] = fma(a1, dl, s[1]);
            s[2] = fma(a0, dm, s[2]); s[3] = fma(a1, dm, s[3]);
            s[4] = fma(a0, dr, s[4]); s[5] = fma(a1, dr, s[5]);
        }
        if (live) {
#pragma unroll
            for (int k = 0; k < 4; ++k) g[k] += s[k];
            g[4] = fma(w2, s[4], g[4]);
            g[5] = fma(w2, s[5], g[5]);
        }
    }
    // corners (-,-), (+,-), (+,+), (-,+)
    const double h0 = tab[TB::H0 + eta], h1 = tab[TB::H1 + eta], we = tab[TB::W + eta] * rc[4];
    double o[12];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        o[k] = we * h0 * g[2 * k];
        o[3 + k] = we * h0 * g[2 * k + 1];
        o[6 + k] = we * h1 * g[2 * k + 1];
        o[9 + k] = we * h1 * g[2 * k];
    }
#pragma unroll
    for (int k = 0; k < 12; ++k)
        for (int d = 32; d > 0; d >>= 1) o[k] += __shfl_xor(o[k], d);
    if (lane == 0)
#pragma unroll
        for (int k = 0; k < 12; ++k) red[wv][k] = o[k];
    __syncthreads();
    if (threadIdx.x < 12) {
        double t = 0.0;
        for (int w = 0; w < nw; ++w) t += red[w][threadIdx.x];
        part[(size_t)e * 12 + threadIdx.x] = t;
    }
}

}  // namespace f25k
