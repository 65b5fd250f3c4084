// Plane-wave right-hand side: b[m] = sum over the shapes (c, r, a) of dof m of
// a * sum_p w_p f_r(x_p) . T E(x_p), E(x) = amplitude exp(-gamma d.x) pol
// (src/excitation.jl:38-115, src/maxwell/mwexc.jl:36-42), with the traces of
// excitation.jl:168-180: TangTraceMW (n x E) x n, which tested with a tangential f
// equals f . E, and CrossTraceMW n x E, n the cell's normal.
#include <algorithm>
#include <cmath>
#include <vector>

#include "bh_device.h"
#include "bh_internal.h"

namespace bh {

struct PlaneWave {
    double d[3], pr[3], pi[3], gr, gi, ar, ai;
};

// 32 lanes to a dof, each a point of one of its shapes at a time (two cells of 16 points at the
// default degree 8), summed by a shuffle tree.  Bound by the latency of one evaluation: a thread
// per dof went through its 32 points one after the other, 22 us at 702 dofs; now 4.
constexpr int kPwLanes = 32;

__global__ __launch_bounds__(256) void k_planewave(const double *__restrict__ geo, const double *__restrict__ qp, int Q,
                                                   const int *__restrict__ ptr, const int *__restrict__ cell,
                                                   const int *__restrict__ ref, const double *__restrict__ coef,
                                                   int ndofs, PlaneWave pw, int trace, double *__restrict__ b)
{
    const int m = (int)(((long long)blockIdx.x * 256 + threadIdx.x) / kPwLanes), lane = threadIdx.x % kPwLanes;
    if (m >= ndofs) return;   // whole groups of lanes
    double sr = 0.0, si = 0.0;
    const int k0 = ptr[m], items = (ptr[m + 1] - k0) * Q;
    for (int it = lane; it < items; it += kPwLanes) {
        const int k = k0 + it / Q, p = it % Q;
        const int c = cell[k], r = ref[k];
        const double *g = geo + (size_t)c * kGeo;
        const double inv2A = 1.0 / (2.0 * g[kGeoA]);
        // the polarisation as seen by f: pol itself, or n x pol for the cross trace
        double pr[3], pi[3];
        if (trace == BH_TRACE_CROSS) {
            const double *nrm = g + kGeoN;
            cross3(pr, nrm, pw.pr);
            cross3(pi, nrm, pw.pi);
        } else {
            for (int k2 = 0; k2 < 3; ++k2) { pr[k2] = pw.pr[k2]; pi[k2] = pw.pi[k2]; }
        }
        const double *q = qp + ((size_t)c * Q + p) * 4;
        const double x[3] = {q[0] + g[kGeoC], q[1] + g[kGeoC + 1], q[2] + g[kGeoC + 2]};
        const double f[3] = {(x[0] - g[3 * r]) * inv2A, (x[1] - g[3 * r + 1]) * inv2A, (x[2] - g[3 * r + 2]) * inv2A};
        const double t = pw.d[0] * x[0] + pw.d[1] * x[1] + pw.d[2] * x[2];
        double s, co;
        sincos(pw.gi * t, &s, &co);
        const double ea = pw.gr == 0.0 ? 1.0 : exp(-pw.gr * t);
        // phase = amplitude * exp(-gamma t)
        const double er = ea * co, ei = -ea * s;
        const double phr = pw.ar * er - pw.ai * ei, phi = pw.ar * ei + pw.ai * er;
        const double er2 = f[0] * pr[0] + f[1] * pr[1] + f[2] * pr[2];
        const double ei2 = f[0] * pi[0] + f[1] * pi[1] + f[2] * pi[2];
        const double w = q[3] * coef[k];
        sr += w * (er2 * phr - ei2 * phi);
        si += w * (er2 * phi + ei2 * phr);
    }
#pragma unroll
    for (int off = kPwLanes / 2; off >= 1; off >>= 1) {
        sr += __shfl_xor(sr, off, 64);
        si += __shfl_xor(si, off, 64);
    }
    if (lane == 0) {
        b[2 * (size_t)m] = sr;
        b[2 * (size_t)m + 1] = si;
    }
}

}  // namespace bh

using namespace bh;

extern "C" int bh_assemble_planewave(bh_ctx *ctx, const bh_space *X, const double *direction, const double *pol_re,
                                     const double *pol_im, const double *gamma, const double *amplitude, int rule,
                                     int accumulate, double *b)
{
    return bh_assemble_excitation(ctx, X, BH_TRACE_TANGENTIAL, direction, pol_re, pol_im, gamma, amplitude, rule,
                                  accumulate, b);
}

extern "C" int bh_assemble_excitation(bh_ctx *ctx, const bh_space *X, int trace, const double *direction,
                                      const double *pol_re, const double *pol_im, const double *gamma,
                                      const double *amplitude, int rule, int accumulate, double *b)
{
    BH_API_BEGIN
    BH_REQUIRE(ctx && X && direction && pol_re && pol_im && gamma && amplitude, "NULL argument");
    BH_REQUIRE(trace == BH_TRACE_TANGENTIAL || trace == BH_TRACE_CROSS, "trace must be BH_TRACE_TANGENTIAL or "
               "BH_TRACE_CROSS");
    const int64_t n = X->ndofs;
    if (n == 0) return BH_OK;
    BH_REQUIRE(b != nullptr, "b is NULL");
    bh_space *sp = const_cast<bh_space *>(X);
    Mesh &m = *sp->mesh;
    int Q = 0;
    const double *qp = (const double *)quad_points(m, rule, &Q, false, ctx->stream);
    PlaneWave pw{};
    for (int k = 0; k < 3; ++k) { pw.d[k] = direction[k]; pw.pr[k] = pol_re[k]; pw.pi[k] = pol_im[k]; }
    pw.gr = gamma[0]; pw.gi = gamma[1]; pw.ar = amplitude[0]; pw.ai = amplitude[1];
    // the result's buffer comes from the pool, which keeps buffers of 1 MiB or more
    PoolBuf<double> db(*ctx, std::max<size_t>(2 * (size_t)n, size_t(1) << 17));
    const long long lanes = (long long)n * kPwLanes;
    BH_REQUIRE((lanes + 255) / 256 < (1LL << 31), "too many dofs for one launch");
    k_planewave<<<(unsigned)((lanes + 255) / 256), 256, 0, ctx->stream>>>(m.d_geo.p, qp, Q, sp->d_ptr.p, sp->d_cell.p,
                                                                        sp->d_ref.p, sp->d_coeff.p, (int)n, pw, trace,
                                                                        db.p);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) BH_FAIL(BH_ERR_HIP, "launch of k_planewave failed: %s", hipGetErrorString(e));
    std::vector<double> part(accumulate ? 2 * n : 0);   // what b holds is added here
    BH_CHECK_HIP(hipMemcpyAsync(accumulate ? part.data() : b, db.p, sizeof(double) * 2 * n, hipMemcpyDeviceToHost,
                                ctx->stream));
    BH_CHECK_HIP(hipStreamSynchronize(ctx->stream));
    db.done();
    for (size_t i = 0; i < part.size(); ++i) b[i] += part[i];
    BH_API_END
}
