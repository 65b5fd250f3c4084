// Far fields of a surface current on a Raviart-Thomas space: the reference's
//     potential(op, points, coeffs, X; quadstrat = SingleNumQStrat(10))
// (src/postproc.jl:138-150,174-211, farfieldlocal! :273-288) for the far-field
// operators of src/maxwell/farfield.jl:1-120:
//     MWFarField3D                     amplitude (y x (K J)) x y        :61-63
//     MWDoubleLayerFarField3D          amplitude  y x (K J)             :65-67
//     MWDoubleLayerRotatedFarField3D   amplitude  y x ((K J) x n)       :98-100
//     MWFarField3DDropConstant         coeff      (y x (K J)) x y,  K = expm1(.)  :69-75
// with K(y, x) = exp(gamma y.x) (:59) and J(x) = sum_n coeffs[n] f_n(x) the
// current at the rule point x (the rule is a Dunavant triangle rule of the
// SingleNumQStrat degree, src/postproc/farfield.jl:3-7).
//
// The reference loops point -> cell -> rule point -> shape and scatters into ff;
// here the sum is regrouped as ff(y) = amplitude I(y, S(y)) with
//     S(y) = sum over all rule points x of K(y, x) w J(x),
// which is linear in the current.  On the cells' scale the phase is small, and S is a sum
// over (direction, cell) pairs of a short series that the rule's symmetry leaves
// (k_ff_cells, k_ff_partial_cells).  Otherwise (the drop-constant kernel, cells of more than
// half a wavelength) the current is formed once per rule point (k_ff_current) and S is a
// dense sum over (direction, point) pairs (k_ff_partial: directions on lanes, points staged
// through LDS and broadcast to every lane).  Chunks of cells or points over the grid's
// second dimension are summed in a fixed order (k_ff_finish).  Everything is FP64.
#include <algorithm>
#include <cmath>
#include <complex>
#include <mutex>

#include "bh_device.h"
#include "bh_internal.h"

namespace bh {

namespace {

constexpr int kFFThreads = 256;    // directions per workgroup, and points per LDS tile
constexpr int kFFPoint = 9;        // doubles per staged point: x[3], Re wJ[3], Im wJ[3]
constexpr int kFFBlocks = 4096;    // target workgroups of k_ff_partial
constexpr int kFFLanes = 64;       // directions per workgroup of k_ff_partial_cells: one wave, so that few
                                   // directions leave few idle lanes
constexpr int kFFWaves = 16384;    // target workgroups of k_ff_partial_cells

// One thread per (cell, rule point): the absolute position x and the weighted
// current w J(x), J = sum_r a_r (x - v_r) / (2 A) with a_r = sum over the
// element-to-dof slots (dof, c) of (cell, r) of c coeffs[dof] (the RT shape
// values of src/bases/local/rtlocal.jl and the assemblydata scatter of
// postproc.jl:200-205).  rotated: w J x n (the rotated double layer's J x n).
__global__ void k_ff_current(const double *__restrict__ geo, const double *__restrict__ qp, int Q, int64_t nf,
                             const int32_t *__restrict__ e2d, const double *__restrict__ e2c, int kmax,
                             const double *__restrict__ coeffs, int rotated, double *__restrict__ pts)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nf * Q) return;
    const int64_t c = i / Q;
    const double *g = geo + c * kGeo;
    const double *q = qp + i * 4;
    const double x[3] = {q[0] + g[kGeoC], q[1] + g[kGeoC + 1], q[2] + g[kGeoC + 2]};
    const double s = q[3] / (2.0 * g[kGeoA]);
    double jr[3] = {0.0, 0.0, 0.0}, ji[3] = {0.0, 0.0, 0.0};
    for (int r = 0; r < 3; ++r) {
        double ar = 0.0, ai = 0.0;
        for (int k = 0; k < kmax; ++k) {
            const int64_t at = (c * 3 + r) * kmax + k;
            const int dof = e2d[at];
            if (dof < 0) continue;
            ar += e2c[at] * coeffs[2 * (int64_t)dof];
            ai += e2c[at] * coeffs[2 * (int64_t)dof + 1];
        }
        for (int d = 0; d < 3; ++d) {
            const double f = (x[d] - g[3 * r + d]) * s;
            jr[d] += ar * f;
            ji[d] += ai * f;
        }
    }
    if (rotated) {
        const double *nn = g + kGeoN;
        const double tr[3] = {jr[1] * nn[2] - jr[2] * nn[1], jr[2] * nn[0] - jr[0] * nn[2], jr[0] * nn[1] - jr[1] * nn[0]};
        const double ti[3] = {ji[1] * nn[2] - ji[2] * nn[1], ji[2] * nn[0] - ji[0] * nn[2], ji[0] * nn[1] - ji[1] * nn[0]};
        for (int d = 0; d < 3; ++d) { jr[d] = tr[d]; ji[d] = ti[d]; }
    }
    double *o = pts + i * kFFPoint;
    for (int d = 0; d < 3; ++d) {
        o[d] = x[d];
        o[3 + d] = jr[d];
        o[6 + d] = ji[d];
    }
}

// Partial sums S_chunk(y) = sum over the chunk's points of K(y, x) w J(x).
// Grid: x = direction blocks of kFFThreads lanes, y = chunks of `per` points.
// Every lane takes part in the LDS staging and the barriers, also the lanes past
// the last direction.  K = exp(gamma t) or, with expm1, exp(gamma t) - 1 formed as
// (e^a - 1) - 2 e^a sin^2(b/2) + i e^a sin(b) for gamma t = a + i b, so that small
// phases keep their relative accuracy.
__global__ __launch_bounds__(kFFThreads) void k_ff_partial(const double *__restrict__ pts, int64_t M, int64_t per,
                                                           const double *__restrict__ dirs, int64_t P, double gr,
                                                           double gi, int expm1_kernel, double *__restrict__ part)
{
    __shared__ double tile[kFFThreads * kFFPoint];
    const int64_t p = (int64_t)blockIdx.x * kFFThreads + threadIdx.x;
    const bool live = p < P;
    const double y0 = live ? dirs[3 * p] : 0.0, y1 = live ? dirs[3 * p + 1] : 0.0, y2 = live ? dirs[3 * p + 2] : 0.0;
    const int64_t c0 = (int64_t)blockIdx.y * per;
    const int64_t c1 = c0 + per < M ? c0 + per : M;
    double sr[3] = {0.0, 0.0, 0.0}, si[3] = {0.0, 0.0, 0.0};
    for (int64_t t0 = c0; t0 < c1; t0 += kFFThreads) {
        const int cnt = (int)(c1 - t0 < kFFThreads ? c1 - t0 : kFFThreads);
        __syncthreads();
        for (int e = threadIdx.x; e < cnt * kFFPoint; e += kFFThreads) tile[e] = pts[t0 * kFFPoint + e];
        __syncthreads();
        if (!live) continue;
        for (int j = 0; j < cnt; ++j) {
            const double *s = tile + j * kFFPoint;
            const double t = y0 * s[0] + y1 * s[1] + y2 * s[2];
            double sn, cs;
            double kr, ki;
            if (!expm1_kernel) {
                sincos(gi * t, &sn, &cs);
                if (gr != 0.0) {
                    const double ea = exp(gr * t);
                    kr = ea * cs;
                    ki = ea * sn;
                } else {
                    kr = cs;
                    ki = sn;
                }
            } else {
                const double b = gi * t;
                const double h = sin(0.5 * b);
                const double em = expm1(gr * t);
                kr = em - 2.0 * (em + 1.0) * h * h;
                ki = (em + 1.0) * sin(b);
            }
            for (int d = 0; d < 3; ++d) {
                sr[d] += kr * s[3 + d] - ki * s[6 + d];
                si[d] += kr * s[6 + d] + ki * s[3 + d];
            }
        }
    }
    if (!live) return;
    double *o = part + ((int64_t)blockIdx.y * P + p) * 6;
    for (int d = 0; d < 3; ++d) {
        o[d] = sr[d];
        o[3 + d] = si[d];
    }
}

// ---------------------------------------------------------------- cell-factored kernels
// With c the centroid and d_i = v_i - c the vertices relative to it (d_1 + d_2 + d_3 = 0),
// a rule point is x = c + sum_i l_i d_i and gamma y.x = gamma y.c + sum_i l_i z_i,
// z_i = gamma y.d_i.  The current of a cell is linear, J = s (x - c) + a1 d_1 + a2 d_2, so a
// direction needs of a cell only
//     F(z) = sum_q w_q exp(sum_i l_iq z_i)   and   sum_q w_q l_iq exp(.) = dF/dz_i.
// The Dunavant rules are symmetric under the permutations of the vertices: F is a symmetric
// function of z_1, z_2, z_3 whose sum is zero, i.e. a series in E2 = z1 z2 + z2 z3 + z3 z1
// and E3 = z1 z2 z3 alone,
//     F = sum_n 1/n! sum_{2j+3k=n} c_jk E2^j E3^k,
// and along d_1, d_2 (d_3 = -d_1 - d_2) the gradient is
//     sum_i d_i dF/dz_i = -(z1 - z3)(F_E2 + z2 F_E3) d_1 - (z2 - z3)(F_E2 + z1 F_E3) d_2.
// The coefficients c_jk belong to the rule, not to the cell.  Degree 10 takes 14 terms
// where the sum over the points takes 25 points with a sine and a cosine each.

constexpr int kFFMaxDegree = 28;
constexpr int ff_kmax(int D) { return D / 3; }
constexpr int ff_jmax(int D, int k) { return (D - 3 * k) / 2; }
constexpr int ff_terms(int D)
{
    int t = 0;
    for (int k = 0; k <= ff_kmax(D); ++k) t += ff_jmax(D, k) + 1;
    return t;
}
constexpr int kFFCell = 22;   // doubles per cell: c[3], d1[3], d2[3], p1[3], p2[3], a1, a2, s (complex), one unused

// One thread per cell: its record for k_ff_partial_cells.  With a_r = sum over the
// element-to-dof slots (dof, c) of (cell, r) of c coeffs[dof] (the assemblydata scatter of
// postproc.jl:200-205) and the RT shapes (x - v_r) / (2 A) (src/bases/local/rtlocal.jl), the
// current times the area is s (x - c) + a1 d_1 + a2 d_2 with s = (a_1 + a_2 + a_3) / 2,
// a1 = (a_3 - a_1) / 2, a2 = (a_3 - a_2) / 2.  p1, p2: the vectors that carry the sum,
// d_1 and d_2, or d_1 x n and d_2 x n for the rotated double layer's J x n.
__global__ void k_ff_cells(const double *__restrict__ geo, int64_t nf, const int32_t *__restrict__ e2d,
                           const double *__restrict__ e2c, int kmax, const double *__restrict__ coeffs, int rotated,
                           double *__restrict__ rec)
{
    const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= nf) return;
    const double *g = geo + c * kGeo;
    double ar[3], ai[3];
    for (int r = 0; r < 3; ++r) {
        ar[r] = ai[r] = 0.0;
        for (int k = 0; k < kmax; ++k) {
            const int64_t at = (c * 3 + r) * kmax + k;
            const int dof = e2d[at];
            if (dof < 0) continue;
            ar[r] += e2c[at] * coeffs[2 * (int64_t)dof];
            ai[r] += e2c[at] * coeffs[2 * (int64_t)dof + 1];
        }
    }
    double *o = rec + c * kFFCell;
    double d[2][3];
    for (int k = 0; k < 3; ++k) {   // from the edges: the centroid's rounding stays out of the short vectors
        o[k] = g[kGeoC + k];
        const double e = g[k] - g[3 + k], f = g[k] - g[6 + k], h = g[3 + k] - g[6 + k];
        d[0][k] = (e + f) / 3.0;
        d[1][k] = (h - e) / 3.0;
    }
    for (int v = 0; v < 2; ++v) {
        double p[3] = {d[v][0], d[v][1], d[v][2]};
        if (rotated) cross3(p, d[v], g + kGeoN);
        for (int k = 0; k < 3; ++k) {
            o[3 + 3 * v + k] = d[v][k];
            o[9 + 3 * v + k] = p[k];
        }
    }
    o[15] = 0.5 * (ar[2] - ar[0]);
    o[16] = 0.5 * (ai[2] - ai[0]);
    o[17] = 0.5 * (ar[2] - ar[1]);
    o[18] = 0.5 * (ai[2] - ai[1]);
    o[19] = 0.5 * (ar[0] + ar[1] + ar[2]);
    o[20] = 0.5 * (ai[0] + ai[1] + ai[2]);
    o[21] = 0.0;
}

// Partial sums S_chunk(y) = sum over the chunk's cells of sum_q w K(y, x_q) J(x_q),
// K = exp(gamma y.x).  A lane holds one direction; the cells of a chunk are the same for
// every lane, so their records and the coefficients are scalar loads and nothing is staged.
// z_i enters as t_i = sigma y.d_i, real: lossless (LOSSY = false, gamma = i g) sigma = g and
// the powers of i are in the coefficients' signs, so that a power E3^k carries i^k: even k
// real, odd k imaginary.  Otherwise sigma = |gamma| and the coefficients are complex,
// times (gamma / |gamma|)^n; (ur, ui) = |gamma| / gamma then turns dF/dt into dF/dz.
// coef: for each k, j ascending, c_jk / n! (LOSSY: re, im), the parity sign included.
// Bound by FP64 VALU issue: 118 FP64 instructions per (direction, cell) lossless at
// degree 10, 35 of them sincos_f64.  Measured on the MI355X, 65,341 directions x 26,664
// cells, 25-point rule (degree 10): 7.8 ms, against 56.0 ms for the sum over the points with
// Taylor sines and cosines; 2701 x 2002, lossy: 116 us (degree 20) against 628 us with sincos and
// exp at each point.
template <int D, bool LOSSY>
__global__ __launch_bounds__(kFFLanes) void k_ff_partial_cells(const double *__restrict__ rec, int64_t nf,
                                                               int64_t per_cells, const double *__restrict__ dirs,
                                                               int64_t P, double gr, double gi, double sigma, double ur,
                                                               double ui, const double *__restrict__ coef,
                                                               double *__restrict__ part)
{
    constexpr int NK = ff_kmax(D) + 1, W = LOSSY ? 2 : 1;
    const int64_t p = (int64_t)blockIdx.x * kFFLanes + threadIdx.x;
    const int64_t pc = p < P ? p : P - 1;
    const double y0 = dirs[3 * pc], y1 = dirs[3 * pc + 1], y2 = dirs[3 * pc + 2];
    const int64_t c0 = (int64_t)blockIdx.y * per_cells;
    const int64_t c1 = c0 + per_cells < nf ? c0 + per_cells : nf;
    double sr[3] = {0.0, 0.0, 0.0}, si[3] = {0.0, 0.0, 0.0};
    for (int64_t c = c0; c < c1; ++c) {
        const double *s = rec + c * kFFCell;
        const double tc = y0 * s[0] + y1 * s[1] + y2 * s[2];
        const double t1 = sigma * (y0 * s[3] + y1 * s[4] + y2 * s[5]);
        const double t2 = sigma * (y0 * s[6] + y1 * s[7] + y2 * s[8]);
        const double t3 = -(t1 + t2);
        const double e3 = t1 * t2 * t3, e2 = -(t1 * t1 + t2 * (t1 + t2));
        // f[k] = sum_j c_jk E2^j and its derivative in E2
        double f[NK][W], h[NK][W];
        {
            int at = 0;
#pragma unroll
            for (int k = 0; k < NK; ++k) {
                const int J = ff_jmax(D, k);
#pragma unroll
                for (int w = 0; w < W; ++w) {
                    f[k][w] = coef[(at + J) * W + w];
                    h[k][w] = 0.0;
                }
#pragma unroll
                for (int j = J - 1; j >= 0; --j)
#pragma unroll
                    for (int w = 0; w < W; ++w) {
                        h[k][w] = j == J - 1 ? f[k][w] : h[k][w] * e2 + f[k][w];
                        f[k][w] = f[k][w] * e2 + coef[(at + j) * W + w];
                    }
                at += J + 1;
            }
        }
        double Fr, Fi, Ar, Ai, Br, Bi;   // F, F_E2, F_E3
        if constexpr (LOSSY) {
            Fr = f[NK - 1][0]; Fi = f[NK - 1][1];
            Ar = h[NK - 1][0]; Ai = h[NK - 1][1];
            Br = (NK - 1) * f[NK - 1][0]; Bi = (NK - 1) * f[NK - 1][1];
#pragma unroll
            for (int k = NK - 2; k >= 0; --k) {
                Fr = Fr * e3 + f[k][0]; Fi = Fi * e3 + f[k][1];
                Ar = Ar * e3 + h[k][0]; Ai = Ai * e3 + h[k][1];
                if (k > 0) { Br = Br * e3 + k * f[k][0]; Bi = Bi * e3 + k * f[k][1]; }
            }
        } else {
            // even k: real; odd k: imaginary, one factor E3 taken out
            constexpr int KE = (NK - 1) / 2 * 2, KO = (NK - 2) / 2 * 2 + 1;   // largest even and odd k
            static_assert(NK >= 3, "the degrees in use reach E3^2");
            const double w2 = e3 * e3;
            double fe = f[KE][0], he = h[KE][0], be = KE * f[KE][0];
#pragma unroll
            for (int k = KE - 2; k >= 0; k -= 2) {
                fe = fe * w2 + f[k][0];
                he = he * w2 + h[k][0];
                if (k > 0) be = be * w2 + k * f[k][0];
            }
            double fo = f[KO][0], ho = h[KO][0], bo = KO * f[KO][0];
#pragma unroll
            for (int k = KO - 2; k >= 1; k -= 2) {
                fo = fo * w2 + f[k][0];
                ho = ho * w2 + h[k][0];
                bo = bo * w2 + k * f[k][0];
            }
            Fr = fe; Fi = e3 * fo;
            Ar = he; Ai = e3 * ho;
            Br = e3 * be; Bi = bo;
        }
        const double w1 = t3 - t1, w2_ = t3 - t2;
        double q1r = w1 * (Ar + t2 * Br), q1i = w1 * (Ai + t2 * Bi);
        double q2r = w2_ * (Ar + t1 * Br), q2i = w2_ * (Ai + t1 * Bi);
        if constexpr (LOSSY) {   // times |gamma| / gamma
            const double a = q1r, b = q2r;
            q1r = ur * a - ui * q1i; q1i = ur * q1i + ui * a;
            q2r = ur * b - ui * q2i; q2i = ur * q2i + ui * b;
        } else {                 // times 1 / i
            const double a = q1r, b = q2r;
            q1r = q1i; q1i = -a;
            q2r = q2i; q2i = -b;
        }
        const double g1r = s[15] * Fr - s[16] * Fi + s[19] * q1r - s[20] * q1i;
        const double g1i = s[15] * Fi + s[16] * Fr + s[19] * q1i + s[20] * q1r;
        const double g2r = s[17] * Fr - s[18] * Fi + s[19] * q2r - s[20] * q2i;
        const double g2i = s[17] * Fi + s[18] * Fr + s[19] * q2i + s[20] * q2r;
        double en, ec;
        sincos_f64(gi * tc, &en, &ec);
        if constexpr (LOSSY) {
            const double ea = exp(gr * tc);
            en *= ea;
            ec *= ea;
        }
        const double h1r = ec * g1r - en * g1i, h1i = ec * g1i + en * g1r;
        const double h2r = ec * g2r - en * g2i, h2i = ec * g2i + en * g2r;
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            sr[d] += s[9 + d] * h1r + s[12 + d] * h2r;
            si[d] += s[9 + d] * h1i + s[12 + d] * h2i;
        }
    }
    if (p >= P) return;
    double *o = part + ((int64_t)blockIdx.y * P + p) * 6;
    for (int d = 0; d < 3; ++d) {
        o[d] = sr[d];
        o[3 + d] = si[d];
    }
}

// The coefficients of F for a triangle rule, up to degree kFFMaxDegree: c[n][k] with
// 2j + 3k = n, and bound[n] >= max |sum_q w_q (l.t)^n| over |t_i| <= 1.  With t = (1, tau,
// -1 - tau), E2 = -(1 + tau + tau^2) and E3 = -tau (1 + tau), the lowest power of tau in
// E2^j E3^k is k, so the degree-n part follows power by power.
struct FFSeries {
    bool ok = false;
    long double c[kFFMaxDegree + 1][kFFMaxDegree / 3 + 1] = {};
    double bound[kFFMaxDegree + 1] = {};
};

const FFSeries &ff_series(int degree)
{
    static FFSeries table[kMaxTriDegree + 1];
    static std::mutex mu;
    std::lock_guard<std::mutex> g(mu);
    FFSeries &S = table[degree];
    if (S.ok) return S;
    double u[kMaxTriPts], v[kMaxTriPts], w[kMaxTriPts];
    const int Q = triangle_rule(degree, u, v, w);
    for (int n = 0; n <= kFFMaxDegree; ++n) {
        // coefficients of 1, tau, tau^2, ... of sum_q 2 w_q (alpha + beta tau)^n, only as many as are solved for
        const int K = n / 3;
        long double r[kFFMaxDegree / 3 + 1] = {};
        double bd = 0.0;
        for (int q = 0; q < Q; ++q) {
            const long double l3 = 1.0L - u[q] - v[q], al = u[q] - l3, be = v[q] - l3;
            for (int m = 0; m <= K; ++m) {
                long double t = 2.0L * w[q];
                for (int i = 0; i < n - m; ++i) t *= al;
                for (int i = 0; i < m; ++i) t *= be * (n - i) / (i + 1);
                r[m] += t;
            }
            const double hi = std::max({u[q], v[q], (double)l3}), lo = std::min({u[q], v[q], (double)l3});
            bd += std::fabs(2.0 * w[q]) * std::pow(hi - lo, n);
        }
        S.bound[n] = bd;
        for (int k = n & 1; k <= K; k += 2) {
            const int j = (n - 3 * k) / 2;
            // (1 + tau + tau^2)^j (1 + tau)^k up to tau^(K - k)
            long double e[kFFMaxDegree / 3 + 1] = {1.0L};
            for (int i = 0; i < j + k; ++i)
                for (int m = K - k; m >= 1; --m) e[m] += e[m - 1] + (i < j && m >= 2 ? e[m - 2] : 0.0L);
            const long double sg = (j + k) & 1 ? -1.0L : 1.0L, a = sg * r[k];
            S.c[n][k] = a;
            for (int m = 0; m <= K - k; ++m) r[k + m] -= sg * a * e[m];
        }
    }
    S.ok = true;
    return S;
}

// Smallest of the degrees in use whose series leaves out less than 1e-17 for phases
// |gamma y.d_i| <= theta (0: none).  The gradient's terms end one power earlier, so the
// power theta^D / D! decides; the bounds of the powers fall from there on.
int ff_degree(const FFSeries &S, double theta)
{
    if (!std::isfinite(theta)) return 0;
    for (int D : {6, 10, 14, 20, 28}) {
        double r = S.bound[D];
        for (int j = 1; j <= D; ++j) r *= theta / j;
        if (r <= 1e-17 && theta < D) return D;
    }
    return 0;
}

// ff(y) = amplitude I(y, S), S = sum of the chunk partials in chunk order;
// I = (y x S) x y (single layer, drop-constant) or y x S (double layers; the
// rotated one's J x n was taken in k_ff_current).  Output: 3 complex per point.
// Eight lanes per direction share the chunks (a small call has hundreds of chunks, and one
// lane's chain over them took 62 us at 2701 directions and 372 chunks; 17 us now); the
// order of the sum is fixed by the chunk count.
__global__ __launch_bounds__(256) void k_ff_finish(const double *__restrict__ part, int64_t nchunk,
                                                   const double *__restrict__ dirs, int64_t P, int transverse,
                                                   double ar, double ai, double *__restrict__ ff)
{
    const int64_t p = (int64_t)blockIdx.x * 32 + (threadIdx.x >> 3);
    const int64_t pc = p < P ? p : P - 1;
    double s[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    for (int64_t k = threadIdx.x & 7; k < nchunk; k += 8) {
        const double *q = part + (k * P + pc) * 6;
        for (int d = 0; d < 6; ++d) s[d] += q[d];
    }
#pragma unroll
    for (int off = 1; off < 8; off <<= 1)
        for (int d = 0; d < 6; ++d) s[d] += __shfl_xor(s[d], off, 64);
    if (p >= P || (threadIdx.x & 7)) return;
    const double y[3] = {dirs[3 * p], dirs[3 * p + 1], dirs[3 * p + 2]};
    double v[6];
    for (int h = 0; h < 2; ++h) {   // real and imaginary parts separately (y is real)
        const double *a = s + 3 * h;
        const double c[3] = {y[1] * a[2] - y[2] * a[1], y[2] * a[0] - y[0] * a[2], y[0] * a[1] - y[1] * a[0]};
        if (transverse) {
            v[3 * h + 0] = c[1] * y[2] - c[2] * y[1];
            v[3 * h + 1] = c[2] * y[0] - c[0] * y[2];
            v[3 * h + 2] = c[0] * y[1] - c[1] * y[0];
        } else {
            for (int d = 0; d < 3; ++d) v[3 * h + d] = c[d];
        }
    }
    double *o = ff + p * 6;
    for (int d = 0; d < 3; ++d) {
        o[2 * d] = ar * v[d] - ai * v[3 + d];
        o[2 * d + 1] = ar * v[3 + d] + ai * v[d];
    }
}

void check_ff_launch(const char *what)
{
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) BH_FAIL(BH_ERR_HIP, "launch of %s failed: %s", what, hipGetErrorString(e));
}

}  // namespace

}  // namespace bh

using namespace bh;

extern "C" int bh_farfield(bh_ctx *ctx, int kind, const double *gamma, const double *amplitude, const bh_space *X,
                           const double *coeffs, int64_t npoints, const double *points, int rule, double *ff)
{
    BH_API_BEGIN
    BH_REQUIRE(ctx && X && gamma && amplitude, "NULL argument");
    BH_REQUIRE(kind == BH_FF_SINGLELAYER || kind == BH_FF_DOUBLELAYER || kind == BH_FF_DOUBLELAYER_ROTATED ||
                   kind == BH_FF_DROPCONSTANT,
               "unknown far-field kind %d", kind);
    BH_REQUIRE(rule >= 1, "SingleNumQStrat: triangle rule degree %d must be at least 1", rule);
    if (rule > kMaxTriDegree)
        BH_FAIL(BH_ERR_UNSUPPORTED, "SingleNumQStrat: no triangle rule of degree %d on the GPU path (1..%d)", rule,
                kMaxTriDegree);
    BH_REQUIRE(npoints >= 0, "npoints < 0");
    BH_REQUIRE(std::isfinite(gamma[0]) && std::isfinite(gamma[1]), "gamma is not finite");
    if (npoints == 0) return BH_OK;
    BH_REQUIRE(points && ff, "points or ff is NULL");
    bh_space *sp = const_cast<bh_space *>(X);
    BH_REQUIRE(sp->ndofs == 0 || coeffs, "coeffs is NULL");
    Mesh &m = *sp->mesh;
    hipStream_t s = ctx->stream;
    const int64_t P = npoints;
    const bool transverse = kind == BH_FF_SINGLELAYER || kind == BH_FF_DROPCONSTANT;
    const bool rotated = kind == BH_FF_DOUBLELAYER_ROTATED;
    // Cell-factored path: every kind but the drop-constant one (whose small phases keep their
    // relative accuracy through expm1 at each point), where a series degree covers the largest
    // in-cell phase, theta = |gamma| max|y| max|v - c|, and the phase at the centroids stays
    // where sincos_f64's reduction is exact.
    const double ga = std::hypot(gamma[0], gamma[1]);
    const FFSeries &S = ff_series(rule);
    int D = 0;
    if (kind != BH_FF_DROPCONSTANT && m.nf > 0) {
        double y2 = 0.0;
        for (int64_t p = 0; p < P; ++p) {
            const double *y = points + 3 * p;
            y2 = std::max(y2, y[0] * y[0] + y[1] * y[1] + y[2] * y[2]);
        }
        const double ymax = std::sqrt(y2) * (1.0 + 1e-12);
        if (ga * ymax * m.cmax < 1e5) D = ff_degree(S, ga * ymax * m.rho);
    }
    PoolBuf<double> dcoef(*ctx, 2 * sp->ndofs + 2), ddir(*ctx, 3 * P), dff(*ctx, 6 * P);
    if (sp->ndofs) dcoef.upload(coeffs, 2 * sp->ndofs, s);
    ddir.upload(points, 3 * P, s);
    // partial sums take 48 bytes per (chunk, direction); keep them under 1 GiB
    const int64_t cap = std::max<int64_t>(1, ((int64_t)1 << 30) / (48 * P));
    const int64_t nblk = (P + (D ? kFFLanes : kFFThreads) - 1) / (D ? kFFLanes : kFFThreads);
    int64_t nchunk = ((D ? kFFWaves : kFFBlocks) + nblk - 1) / nblk;
    PoolBuf<double> dpart, dwork, dser;
    if (D) {
        const bool lossy = gamma[0] != 0.0;
        nchunk = std::max<int64_t>(1, std::min({nchunk, m.nf, cap}));
        const int64_t per = (m.nf + nchunk - 1) / nchunk;
        nchunk = (m.nf + per - 1) / per;
        BH_REQUIRE(nblk <= 0x7fffffff && nchunk <= 65535, "too many far-field directions");
        // c_jk / n! times (gamma / |gamma|)^n, k by k; lossless: gamma = i g, t = g y.d, so i^n without
        // the i that an odd power of E3 carries
        double ser[2 * ff_terms(kFFMaxDegree)];
        const std::complex<double> u = ga > 0.0 ? std::complex<double>(gamma[0], gamma[1]) / ga : 1.0;
        int at = 0;
        for (int k = 0; k <= ff_kmax(D); ++k)
            for (int j = 0; j <= ff_jmax(D, k); ++j) {
                const int n = 2 * j + 3 * k;
                long double f = S.c[n][k];
                for (int i = 2; i <= n; ++i) f /= i;
                if (lossy) {
                    std::complex<double> z = (double)f;
                    for (int i = 0; i < n; ++i) z *= u;
                    ser[at++] = z.real();
                    ser[at++] = z.imag();
                } else {
                    ser[at++] = (double)(((n - (k & 1)) / 2) & 1 ? -f : f);
                }
            }
        dpart.alloc(*ctx, nchunk * P * 6);
        dwork.alloc(*ctx, m.nf * kFFCell);
        dser.alloc(*ctx, at);
        dser.upload(ser, at, s);
        {
            ProfScope prof(*ctx, "k_ff_cells", (double)m.nf);
            k_ff_cells<<<(unsigned)((m.nf + 255) / 256), 256, 0, s>>>(m.d_geo.p, m.nf, sp->d_e2d.p, sp->d_e2c.p, sp->kmax,
                                                                    dcoef.p, rotated, dwork.p);
            check_ff_launch("k_ff_cells");
        }
        ProfScope prof(*ctx, "k_ff_partial_cells", (double)m.nf * (double)P);
        const dim3 grid((unsigned)nblk, (unsigned)nchunk);
        const double sigma = lossy ? ga : gamma[1], ur = u.real(), ui = -u.imag();
#define BH_FF_CELLS(DEG)                                                                                              \
    do {                                                                                                              \
        if (lossy) k_ff_partial_cells<DEG, true><<<grid, kFFLanes, 0, s>>>(dwork.p, m.nf, per, ddir.p, P, gamma[0],  \
                                                                           gamma[1], sigma, ur, ui, dser.p, dpart.p); \
        else k_ff_partial_cells<DEG, false><<<grid, kFFLanes, 0, s>>>(dwork.p, m.nf, per, ddir.p, P, 0.0, gamma[1],  \
                                                                      sigma, 0.0, 0.0, dser.p, dpart.p);             \
    } while (0)
        switch (D) {
        case 6: BH_FF_CELLS(6); break;
        case 10: BH_FF_CELLS(10); break;
        case 14: BH_FF_CELLS(14); break;
        case 20: BH_FF_CELLS(20); break;
        default: BH_FF_CELLS(28); break;
        }
#undef BH_FF_CELLS
        check_ff_launch("k_ff_partial_cells");
    } else {
        int Q = 0;
        const double *qp = (const double *)quad_points(m, rule, &Q, false, s);
        const int64_t M = m.nf * Q;
        const int64_t tiles = (M + kFFThreads - 1) / kFFThreads;
        nchunk = std::max<int64_t>(1, std::min({nchunk, tiles, cap}));
        BH_REQUIRE(nblk <= 0x7fffffff && nchunk <= 65535, "too many far-field directions");
        const int64_t per_tiles = (tiles + nchunk - 1) / nchunk;          // whole tiles per chunk
        dpart.alloc(*ctx, nchunk * P * 6);
        dwork.alloc(*ctx, M * kFFPoint + 1);
        if (M > 0) {
            ProfScope prof(*ctx, "k_ff_current", (double)M);
            k_ff_current<<<(unsigned)((M + 255) / 256), 256, 0, s>>>(m.d_geo.p, qp, Q, m.nf, sp->d_e2d.p, sp->d_e2c.p,
                                                                   sp->kmax, dcoef.p, rotated, dwork.p);
            check_ff_launch("k_ff_current");
        }
        ProfScope prof(*ctx, "k_ff_partial", (double)M * (double)P);
        k_ff_partial<<<dim3((unsigned)nblk, (unsigned)nchunk), kFFThreads, 0, s>>>(
            dwork.p, M, per_tiles * kFFThreads, ddir.p, P, gamma[0], gamma[1], kind == BH_FF_DROPCONSTANT, dpart.p);
        check_ff_launch("k_ff_partial");
    }
    {
        ProfScope prof(*ctx, "k_ff_finish", (double)P);
        k_ff_finish<<<(unsigned)((P + 31) / 32), 256, 0, s>>>(dpart.p, nchunk, ddir.p, P, transverse, amplitude[0],
                                                             amplitude[1], dff.p);
        check_ff_launch("k_ff_finish");
    }
    BH_CHECK_HIP(hipMemcpyAsync(ff, dff.p, sizeof(double) * 6 * P, hipMemcpyDeviceToHost, s));
    BH_CHECK_HIP(hipStreamSynchronize(s));
    for (PoolBuf<double> *b : {&dcoef, &ddir, &dff, &dpart, &dwork, &dser}) b->done();
    BH_API_END
}
