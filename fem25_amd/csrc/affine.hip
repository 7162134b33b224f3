// Kernels for parallelogram elements (gfx950): the batched product and the
// adjoint gradient by sum factorisation at the NL-point Gauss-Legendre rule.
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
// coefficients common to the wave.  In the product those reach the FMAs as
// DPP operands: the 16 values of a xi point (v_i, v'_i and the weighted hats)
// lie across each row of 16 lanes, one register pair a point.  (As scalar registers the
// tables of p6 do not fit: hoisted out of the loops they spilled, 3,700 vector
// instructions per chunk of the product instead of 1,900; loaded per point
// each load is waited for.)
#pragma once

namespace f25k {

// record of an element (k_aff_rec): rx, sx, rz, sz (d xi/dx, d eta/dx,
// d xi/dz, d eta/dz), det J, rho, lambda, mu at the four corners, 1 for a
// PML element
constexpr int AFR = 20;

// offsets in the 1-D table (af_table on the host): rows of 16 values per
// point, v_j, v'_j, then w h_0 and w h_1 at HW0, HW1 (h_0, h_1 the hat
// functions); after the rows h_0, h_1, w
template <int NL>
struct AfTab {
    static constexpr int HW0 = 14, HW1 = 15, H0 = 16 * NL, H1 = 17 * NL, W = 18 * NL;
};

// Lanes of a wave: PP real problems (PW complex vectors) times NL eta points
// (60, 64, 60, 60, 56 lanes at p2..p6), lane = eta * PP + problem.
template <int NL>
struct AfShape {
    static constexpr int NEN = NL * NL, NEE = 3 * NEN;
    static constexpr int PP = (64 / NL) & ~1, PW = PP / 2, LN = PP * NL;
    static constexpr int NW = 4;                             // waves of a workgroup
    // the product's LDS per wave: element values of PW vectors, the exchange
    // of one component's sums, the addresses the element's rows are read from
    // and written to
    static constexpr int XS = NEE * PW, ES = 2 * NL * 64;
    static constexpr size_t lds_apply = (size_t)NW * (XS * 16 + ES * 8 + NEE * 16) + 16 * NL * 8;
    // the gradient's LDS per wave: element values of both fields for PW triples
    // (VS values a vector: not a multiple of 256 bytes, or the triples' reads
    // meet in one bank)
    static constexpr int VS = NEE % 16 ? NEE : NEE + 1, GS = 2 * VS * PW;
    static constexpr size_t lds_grad(int nw) { return (size_t)nw * GS * 16 + 16 * NL * 8; }
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

// 16 or 4 bytes per lane from global memory straight into LDS (l: the wave's
// base, lane i's value lands at l + 16 i or l + 4 i); complete after dma_wait.
__device__ __forceinline__ void dma16(const void *g, void *l) {
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)g,
                                     (__attribute__((address_space(3))) void *)l, 16, 0, 0);
}
__device__ __forceinline__ void dma4(const void *g, void *l) {
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)g,
                                     (__attribute__((address_space(3))) void *)l, 4, 0, 0);
}
__device__ __forceinline__ void dma_wait() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }
// the wave's own LDS accesses so far are complete, and stay before what follows
__device__ __forceinline__ void lds_wait() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

// Gathers one element's values of the wave's V vectors into its LDS region,
// [vector][VS] values of 16 bytes: lane i takes element values i, i + 64, ...
// of each vector, so a load is a wave-uniform base (the vector) and a lane
// offset (the DOF) kept over the whole batch.  Fixed DOFs are not loaded:
// their values are set to zero once (zero).
template <int NEE, int V, int VS>
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
                for (int v = 0; v < V; ++v) dst[v * VS + lane + 64 * k] = make_double2(0.0, 0.0);
        lds_wait();
    }
    // base(v): the vector's values by DOF, null for a vector that is not there
    template <typename F>
    __device__ __forceinline__ void get(double2 *dst, F base) {
#pragma unroll
        for (int v = 0; v < V; ++v) {
            const double2 *b = base(v);
            if (b)
#pragma unroll
                for (int k = 0; k < K; ++k)
                    if (off[k] >= 0) dma16(b + off[k], dst + v * VS + 64 * k);
        }
    }
};

// First pass of one component: T1[i] = sum_j v_j(eta) a_ji, T2[i] the same
// with v'_j; a: LDS, node (j, i) at a[(j NL + i) * STEP].  x holds column 0 on
// entry and column 0 of the next component (an) on return: each column is
// read while the one before it is summed.
template <int NL, int STEP, typename R>
__device__ __forceinline__ void af_first(const R *a, const R *an, const double *v, const double *d,
                                         double *x, double *T1, double *T2) {
#pragma unroll
    for (int i = 0; i < NL; ++i) {
        double n[NL];
        const R *p = i + 1 < NL ? a + (i + 1) * STEP : an;
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

// acc += (value J of the row of 16 lanes in cq) * op, in program order: the
// statement order below keeps the live values within the registers up to p5
// (at p6 all but 36 bytes a lane of them), which the compiler's own order of an
// unrolled point loop does not
template <int J>
__device__ __forceinline__ void fb(double &acc, double cq, double op) {
    asm volatile("v_fmac_f64_dpp %0, %1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf"
                 : "+v"(acc)
                 : "v"(cq), "v"(op), "i"(J));
}

// Values and reference derivatives of three components at the xi point of cq.
template <int NL, int... I>
__device__ __forceinline__ void af_point(const double (*T1)[NL], const double (*T2)[NL], double cq, double *U, double *Xi,
                                         double *Et, std::integer_sequence<int, I...>) {
#pragma unroll
    for (int c = 0; c < 3; ++c) U[c] = Xi[c] = Et[c] = 0.0;
    ((fb<I>(U[0], cq, T1[0][I]), fb<I>(U[1], cq, T1[1][I]), fb<I>(U[2], cq, T1[2][I]),
      fb<NL + I>(Xi[0], cq, T1[0][I]), fb<NL + I>(Xi[1], cq, T1[1][I]), fb<NL + I>(Xi[2], cq, T1[2][I]),
      fb<I>(Et[0], cq, T2[0][I]), fb<I>(Et[1], cq, T2[1][I]), fb<I>(Et[2], cq, T2[2][I])),
     ...);
}

// The same for one component with scalar 1-D values (vq, dq: uniform).
template <int NL>
__device__ __forceinline__ void af_point_s(const double *T1, const double *T2, const double *vq, const double *dq,
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

// Projection of one component's fluxes at the xi point of cq on the node columns.
template <int NL, int... I>
__device__ __forceinline__ void af_project(double *P1, double *P2, double cq, double A, double B, double N,
                                           std::integer_sequence<int, I...>) {
    ((fb<I>(P1[I], cq, N), fb<I>(P2[I], cq, B)), ...);
    (fb<NL + I>(P1[I], cq, A), ...);
}

// Rows of one node column from its sums at the eta point of cq.
template <int NL, int... J>
__device__ __forceinline__ void af_rows(double *Y, double cq, double p1, double p2, std::integer_sequence<int, J...>) {
    (fb<J>(Y[J], cq, p1), ...);
    (fb<NL + J>(Y[J], cq, p2), ...);
}

// ---------------------------------------------------------------------------
// y_b = S(omega_b, ky_b) x_b over the parallelogram elements of one colour.
// A wave takes PW pairs of one element at a time and walks the element's
// chunks of pairs part, part + nsplit, ... of nch; four waves of consecutive
// numbers form a workgroup and share only the 1-D table.  Per chunk: the
// first pass from LDS, then per xi point the fields, the fluxes (density and
// moduli bilinear in the corners) and their projection back along xi; the
// last contraction, over eta, runs across lanes: one component's sums at a
// time go through LDS and each lane forms the NL rows of one xi node column.
// The next chunk's values stream into LDS meanwhile.  A fixed DOF reads the
// zero value of its LDS slot.  The rows of y a lane adds to are read from and
// written to addresses kept in LDS: zpad (npair zeros) for a node touched
// first and for a fixed DOF, sink (npair values) for the stores of a fixed
// DOF, so that none of them is a branch (they were a quarter of the
// instructions).  PML elements only store zeros where they touch a node
// first.  lm, lm_out: the DOFs read and written, as in k_apply_v (below 2^27,
// so that a slot's DOF and pair pack into one register).
//
// Bound by memory at p4 and by FP64 issue and memory together at p6: four
// colours read x 1.56 (p4) and 1.36 (p6) times and read y back for the nodes
// they share, 7.3 GB a product at 200x100 p4, 128 pairs (4.2 TB/s without
// the point loop, where a large copy runs at 4.66).  Measured on MI355X
// against the block product of k_apply_v: 200x100 p4, 128 pairs 2.25 -> 1.93
// ms; 160x80 p6, 192 pairs 6.92 -> 4.2; 40x20 p4, one pair 135 -> 68 us.  On
// the way, at p4 / p6: scalar tables 2.17 / 5.81; loads waited for after the
// stores 2.13 / 4.84; the three components' rows kept and stored together
// 2.33 / 5.80; row addresses computed per row 2.05 / 4.75; the rows' values
// loaded before the point loop 2.05 / 7.1 (registers).  complex64 vectors
// through registers into LDS, widened on the way, instead of two pieces a
// value straight into it: 120x60 p6 spills, 128 pairs 2.03 ms against 1.60
// (p4, p5 within 2%).
template <int NL, typename XT, bool RECT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void k_apply_af(
        const int *__restrict__ order, int nel, int nsplit, int nch, const double *__restrict__ rec,
        const double *__restrict__ tab, const int *__restrict__ lm, const int *__restrict__ lm_out,
        const unsigned long long *__restrict__ first, int npair, const double *__restrict__ omega,
        const double *__restrict__ ky, const XT *__restrict__ x, XT *__restrict__ y, const XT *__restrict__ zpad,
        XT *__restrict__ sink) {
    typedef AfShape<NL> S;
    typedef AfTab<NL> TB;
    typedef decltype(XT().x) R;
    constexpr int NEE = S::NEE, PP = S::PP, PW = S::PW, LN = S::LN, ES = S::ES;
    // complex128 values lie whole in LDS, complex64 as real parts, then
    // imaginary parts (two pieces of 4 bytes; widened as they are read)
    constexpr bool WIDE = sizeof(XT) == 16;
    constexpr int NG = (S::XS + 63) / 64, STEP = WIDE ? 2 : 1, IM = WIDE ? 1 : S::XS;
    extern __shared__ double sm[];
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    double2 *sx = reinterpret_cast<double2 *>(sm) + wv * S::XS;
    R *sv = reinterpret_cast<R *>(sx);
    double *sb = sm + S::NW * S::XS * 2 + wv * ES;
    uint64_t *sr = reinterpret_cast<uint64_t *>(sm + S::NW * (S::XS * 2 + ES)) + wv * 2 * NEE;   // read, then written
    double *st = sm + S::NW * (S::XS * 2 + ES + 2 * NEE);
    for (int i = threadIdx.x; i < 16 * NL; i += 256) st[i] = tab[i];
    __syncthreads();
    const int wx = blockIdx.x * S::NW + wv, ei = wx / nsplit, part = wx % nsplit;
    if (ei >= nel) return;
    const int e = order[ei];
    const double *rc = rec + (size_t)e * AFR;
    const unsigned long long fmask = first[e];
    const int *L = lm + (size_t)e * NEE, *LO = lm_out + (size_t)e * NEE;
    if (rc[17] != 0.0) {
        for (int ch = part; ch < nch; ch += nsplit)
            for (int s = lane; s < S::XS; s += 64) {
                const int d = s / PW, pair = ch * PW + s % PW, dof = LO[d];
                if (dof >= 0 && pair < npair && ((fmask >> (d / 3)) & 1ull)) y[(size_t)dof * npair + pair] = XT{0, 0};
            }
        return;
    }
    // gather slot s = lane + 64 r: element value s / PW of pair s % PW.  Every
    // DOF is loaded before the first is used (one latency, not one per slot)
    constexpr int NO = (NEE + 63) / 64;
    int dp[NG], ds[NO];
#pragma unroll
    for (int r = 0; r < NG; ++r) dp[r] = L[min((lane + 64 * r) / PW, NEE - 1)];
#pragma unroll
    for (int r = 0; r < NO; ++r) ds[r] = LO[min(lane + 64 * r, NEE - 1)];
#pragma unroll
    for (int r = 0; r < NG; ++r) {
        const int s = lane + 64 * r;
        if (s < S::XS && dp[r] < 0) sv[s * STEP] = sv[s * STEP + IM] = 0;
        dp[r] = s < S::XS && dp[r] >= 0 ? dp[r] * 16 + s % PW : -1;
    }
#pragma unroll
    for (int r = 0; r < NO; ++r) {
        const int i = lane + 64 * r;
        XT *row = ds[r] >= 0 ? y + (size_t)ds[r] * npair : sink;
        if (i < NEE) {
            sr[i] = reinterpret_cast<uint64_t>(ds[r] >= 0 && !((fmask >> (i / 3)) & 1ull) ? row : zpad);
            sr[NEE + i] = reinterpret_cast<uint64_t>(row);
        }
    }
    auto get = [&](int p0) {
#pragma unroll
        for (int r = 0; r < NG; ++r)
            if (dp[r] >= 0) {
                const XT *src = x + ((size_t)(dp[r] >> 4) * npair + min(p0 + (dp[r] & 15), npair - 1));
                if constexpr (WIDE) dma16(src, sx + 64 * r);
                else {
                    dma4(src, sv + 64 * r);
                    dma4(reinterpret_cast<const R *>(src) + 1, sv + IM + 64 * r);
                }
            }
    };
    lds_wait();
    get(part * PW);
    const int le = min(lane, LN - 1), eta = le / PP, pr = (le % PP) >> 1, im = le & 1;
    const double *stl = st + (lane & 15);   // the lane's values of the table's rows
    const auto seq = std::make_integer_sequence<int, NL>();
    auto pairof = [&](int ch) { return min(ch * PW + pr, npair - 1); };
    double omn = omega[pairof(part)], kyn = ky[pairof(part)];   // of the next chunk, loaded ahead with its values
    // geometry and the corner values at the lane's eta point, times w det J
    const double rx = rc[0], sxx = rc[1], rz = rc[2], sz = rc[3];
    const double h0 = tab[TB::H0 + eta], h1 = tab[TB::H1 + eta], we = tab[TB::W + eta] * rc[4];
    const double rL = (rc[5] * h0 + rc[8] * h1) * we, rR = (rc[6] * h0 + rc[7] * h1) * we;
    const double lL = (rc[9] * h0 + rc[12] * h1) * we, lR = (rc[10] * h0 + rc[11] * h1) * we;
    const double mL = (rc[13] * h0 + rc[16] * h1) * we, mR = (rc[14] * h0 + rc[15] * h1) * we;
    dma_wait();
    for (int ch = part; ch < nch; ch += nsplit) {
        const int pair = ch * PW + pr;
        const bool live = lane < LN && pair < npair;
        const double w2 = -omn * omn, kv = im ? -kyn : kyn;
        double T1[3][NL], T2[3][NL];
        {
            double v[NL], d[NL], c0[NL];
#pragma unroll
            for (int j = 0; j < NL; ++j) { v[j] = st[eta * 16 + j]; d[j] = (RECT ? sz : 1.0) * st[eta * 16 + NL + j]; }
            const R *a = sv + STEP * pr;
            auto at = [&](int c) { return a + c * PW * STEP + (c == 1 ? 1 - im : im) * IM; };
#pragma unroll
            for (int j = 0; j < NL; ++j) c0[j] = at(0)[j * NL * 3 * PW * STEP];
#pragma unroll
            for (int c = 0; c < 3; ++c) af_first<NL, 3 * PW * STEP>(at(c), at(c < 2 ? c + 1 : 0), v, d, c0, T1[c], T2[c]);
        }
        lds_wait();
        if (ch + nsplit < nch) {
            get((ch + nsplit) * PW);
            omn = omega[pairof(ch + nsplit)];
            kyn = ky[pairof(ch + nsplit)];
        }
        const double rL2 = rL * w2, rR2 = rR * w2;
        double P1[3][NL], P2[3][NL];
#pragma unroll
        for (int c = 0; c < 3; ++c)
#pragma unroll
            for (int i = 0; i < NL; ++i) P1[c][i] = P2[c][i] = 0.0;
#pragma unroll
        for (int q = 0; q < NL; ++q) {
            const double cq = stl[q * 16];
            double U[3], Xi[3], Et[3], X[3], Z[3], lq = 0.0, mq = 0.0, rq = 0.0;
            fb<TB::HW0>(lq, cq, lL); fb<TB::HW0>(mq, cq, mL); fb<TB::HW0>(rq, cq, rL2);
            fb<TB::HW1>(lq, cq, lR); fb<TB::HW1>(mq, cq, mR); fb<TB::HW1>(rq, cq, rR2);
            af_point<NL>(T1, T2, cq, U, Xi, Et, seq);
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                X[c] = RECT ? rx * Xi[c] : rx * Xi[c] + sxx * Et[c];
                Z[c] = RECT ? Et[c] : rz * Xi[c] + sz * Et[c];
            }
            const double ld = lq * (X[0] + Z[2] + kv * U[1]), m2 = 2.0 * mq;
            const double FX0 = fma(m2, X[0], ld), FZ2 = fma(m2, Z[2], ld), F13 = mq * (Z[0] + X[2]);
            const double FX1 = mq * (X[1] - kv * U[0]), FZ1 = mq * (Z[1] - kv * U[2]);
            const double FX[3] = {FX0, FX1, F13}, FZ[3] = {F13, FZ1, FZ2};
            const double FN[3] = {rq * U[0] - kv * FX1, fma(kv, ld, fma(kv * kv, m2, rq) * U[1]), rq * U[2] - kv * FZ1};
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                const double A = RECT ? rx * FX[c] : rx * FX[c] + rz * FZ[c];
                const double B = RECT ? sz * FZ[c] : sxx * FX[c] + sz * FZ[c];
                af_project<NL>(P1[c], P2[c], cq, A, B, FN[c], seq);
            }
        }
        double cr[NL];
#pragma unroll
        for (int q = 0; q < NL; ++q) cr[q] = stl[q * 16];
        // the rows this lane adds to: node column i = eta, rows j; bytes from
        // a row's address to the lane's value of components 1, 3 and of 2
        const uint64_t po = (uint64_t)min(pair, npair - 1) * sizeof(XT);
        const uint64_t oc[2] = {po + im * sizeof(R), po + (1 - im) * sizeof(R)};
        const uint64_t *se = sr + 3 * eta;
        R yv[3][NL];
#pragma unroll
        for (int c = 0; c < 3; ++c)
#pragma unroll
            for (int j = 0; j < NL; ++j) yv[c][j] = *(const __attribute__((address_space(1))) R *)(se[j * NL * 3 + c] + oc[c == 1]);
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            lds_wait();   // the previous component's sums are read
#pragma unroll
            for (int i = 0; i < NL; ++i) {
                sb[(2 * i) * 64 + lane] = P1[c][i];
                sb[(2 * i + 1) * 64 + lane] = P2[c][i];
            }
            lds_wait();
            double Y[NL];
#pragma unroll
            for (int j = 0; j < NL; ++j) Y[j] = 0.0;
            const double *b = sb + 2 * eta * 64 + le % PP;
#pragma unroll
            for (int q = 0; q < NL; ++q) {
                const double p1 = b[q * PP], p2 = b[64 + q * PP];
                af_rows<NL>(Y, cr[q], p1, p2, seq);
            }
            if (c == 0) {
                // every load so far (the rows' values, the next chunk's) is
                // awaited here, before the first store: a later wait for any
                // of them would wait for the stores before it too
                dma_wait();
#pragma unroll
                for (int k = 0; k < 3 * NL; ++k) asm volatile("" : "+v"(yv[k / NL][k % NL]));
            }
            if (live)
#pragma unroll
                for (int j = 0; j < NL; ++j)
                    *(__attribute__((address_space(1))) R *)(se[NEE + j * NL * 3 + c] + oc[c == 1]) = (R)((double)yv[c][j] + Y[j]);
        }
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
// a lane, 168 of the 256 registers at p6, where 12 to 16 bytes a lane spill), at
// p6 and many triples by memory too (400x200, 192 triples: 101 GB read, each
// value 1.9 times, 2 GB written by the spills, 22.8 ms).  Measured on MI355X: 200x100 p4, 128 triples
// 9.30 -> 1.62 ms (FP64 pipe about half busy, 4.5 GB from HBM of 3.9 GB read
// once); 121x59 p6, 45 triples 2.99 -> 0.56 ms.  On the way: slots numbered
// across vectors (index arithmetic per load) 2.03 ms at p4, one column at a
// time in the first pass (each waited for its LDS reads) 1.82; the point
// loop unrolled spills (p6 1.03 ms against 0.56), its 1-D values loaded one
// point ahead 1.67 ms, or as DPP operands in program order 1.71 (p6 0.65):
// here the scalar loads of a rolled loop cost less than that order.  LDS and
// loads follow the triples there are: one triple at 120x60, p4 149 -> 97 us,
// p6 191 -> 118; vectors a multiple of 256 bytes apart (p3) met in one bank:
// 128 triples at 120x60 738 -> 392 us.
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
    double *st = sm + nw * S::GS * 2;
    const int e = elems[blockIdx.x];
    const double *rc = rec + (size_t)e * AFR;
    if (rc[17] != 0.0) {   // PML elements are outside the gradient
        if (threadIdx.x < 12) part[(size_t)e * 12 + threadIdx.x] = 0.0;
        return;
    }
    for (int i = threadIdx.x; i < 16 * NL; i += blockDim.x) st[i] = tab[i];
    __syncthreads();
    const int nch = (ntrip + PW - 1) / PW;
    typedef AfGather<NEE, 2 * PW, S::VS> G;
    G ga;
    ga.init(lane, lm + (size_t)e * NEE);
    ga.zero(lane, sw);
    // vectors 0 .. PW - 1: u of the chunk's triples, then l
    auto base = [&](int t0) {
        return [=](int v) -> const double2 * {
            return t0 + v % PW < ntrip ? (v >= PW ? l : u) + (size_t)(t0 + v % PW) * ndof : nullptr;
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
            for (int j = 0; j < NL; ++j) { v[j] = st[eta * 16 + j]; d[j] = (RECT ? sz : 1.0) * st[eta * 16 + NL + j]; }
            const double *a = reinterpret_cast<const double *>(sw + tr * S::VS);
            auto at = [&](int k) {   // component k % 3 of field k / 3
                return a + (k / 3) * (2 * PW * S::VS) + 2 * (k % 3) + (k % 3 == 1 ? 1 - im : im);
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
            const double *vq = tab + 16 * q, *dq = vq + NL;
            const double a0 = tab[16 * q + TB::HW0], a1 = tab[16 * q + TB::HW1];
            double U[2][3], X0[2], Z2[2], div[2], a12[2], a23[2], a13[2];
#pragma unroll
            for (int f = 0; f < 2; ++f) {
                double X[3], Z[3];
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    double Xi, Et;
                    af_point_s<NL>(T1[f][c], T2[f][c], vq, dq, U[f][c], Xi, Et);
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
