// Order dispatch of the DGSEM stage pipeline and the kernels that do not depend on the
// polynomial order (residual reduction, time-step scan, conservation-sum finalisation).
// The order-templated kernels live in hg_kernels.h and are instantiated per order by
// hg_inst.hip.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "hg_device.h"

namespace hg {

namespace {

__device__ inline double nan_max(double a, double b) { return (b > a || b != b) ? b : a; }

// max|QDot| per equation over n residual partials (4 doubles each), by one workgroup of 1024
// lanes: partials first + t, stepping by stride, every lane keeping four partials' loads in
// flight, then wavefront shuffles and LDS; the four maxima go to out[stride_out c].  The maximum does
// not depend on the order (NaN wins every compare), so the result is exact whatever the grid.
__device__ __forceinline__ void max_partials(const double *part, int n, int first, int stride, double *out,
                                             int stride_out) {
    __shared__ double s[16][4];
    const int t = threadIdx.x;
    const double2 *p2 = (const double2 *)part;
    double m[4] = {0.0, 0.0, 0.0, 0.0};
    int b = first + t;
    for (; b + 3 * stride < n; b += 4 * stride) {
        double2 v[8];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            v[2 * u] = p2[(int64_t)(b + u * stride) * 2];
            v[2 * u + 1] = p2[(int64_t)(b + u * stride) * 2 + 1];
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            m[0] = nan_max(m[0], v[2 * u].x); m[1] = nan_max(m[1], v[2 * u].y);
            m[2] = nan_max(m[2], v[2 * u + 1].x); m[3] = nan_max(m[3], v[2 * u + 1].y);
        }
    }
    for (; b < n; b += stride) {
        const double2 a = p2[(int64_t)b * 2], c = p2[(int64_t)b * 2 + 1];
        m[0] = nan_max(m[0], a.x); m[1] = nan_max(m[1], a.y); m[2] = nan_max(m[2], c.x); m[3] = nan_max(m[3], c.y);
    }
#pragma unroll
    for (int c = 0; c < 4; ++c)
        for (int off = 32; off > 0; off >>= 1) m[c] = nan_max(m[c], __shfl_xor(m[c], off, 64));
    if ((t & 63) == 0) {
#pragma unroll
        for (int c = 0; c < 4; ++c) s[t >> 6][c] = m[c];
    }
    __syncthreads();
    if (t < 4) {
        double v = s[0][t];
        for (int w = 1; w < 16; ++w) v = nan_max(v, s[w][t]);
        out[t * stride_out] = v;
    }
}

// Workgroup g of the grid reduces its share of the partials to out + 4 g.
__global__ __launch_bounds__(1024) void k_resid_final(const double *part, int nb, double *out, int stride_out) {
    max_partials(part, nb, blockIdx.x * 1024, 1024 * gridDim.x, out + blockIdx.x * 4, stride_out);
}

// TimeIntegrator_EstimateTimeStep (DGTimeIntegrator.f90:462-511), second half: the running
// maxima of |u| and a advance in element order starting from the values saved by the
// previous call, and dt is the minimum over elements of cfl*dx/(umax+amax)/(N+1) taken
// with the maxima as they stood at that element.  Maxima and minima are exact in any order.  One
// workgroup takes 4096 elements at a time, four consecutive ones per lane: the lane's running
// maxima, a shuffle scan over the wavefront, one over the wavefronts.  (A chunk per lane, with one
// lane combining 1024 of them, took 69 us at 16.5 k elements and 190 us at 65 k; this takes 12 and 30.)
__global__ __launch_bounds__(1024) void k_dt_scan(int K, const double *umax, const double *amax, const double *dx,
                                                  double coef, double N1, double dt_max, double *state, double *dt_out,
                                                  const double *n1e) {
    __shared__ double su[2][16], sa[2][16], sd[16];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    double ru = state[0], ra = state[1], dt = dt_max;   // the maxima before this round's elements
    for (int e0 = 0, round = 0; e0 < K; e0 += 4096, round ^= 1) {
        const int b = e0 + 4 * t;
        double u[4], a[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            u[c] = b + c < K ? umax[b + c] : 0.0;
            a[c] = b + c < K ? amax[b + c] : 0.0;
        }
#pragma unroll
        for (int c = 1; c < 4; ++c) { u[c] = fmax(u[c], u[c - 1]); a[c] = fmax(a[c], a[c - 1]); }
        double pu = u[3], pa = a[3];   // inclusive over the wavefront's lanes so far
        for (int off = 1; off < 64; off <<= 1) {
            const double vu = __shfl_up(pu, off, 64), va = __shfl_up(pa, off, 64);
            if (lane >= off) { pu = fmax(pu, vu); pa = fmax(pa, va); }
        }
        if (lane == 63) { su[round][wave] = pu; sa[round][wave] = pa; }
        double lu = __shfl_up(pu, 1, 64), la = __shfl_up(pa, 1, 64);   // the lanes before this one
        if (lane == 0) { lu = 0.0; la = 0.0; }
        __syncthreads();   // the other half of su, sa is the next round's
        double tu = 0.0, ta = 0.0;
        for (int w = 0; w < 16; ++w) {
            if (w == wave) { lu = fmax(lu, tu); la = fmax(la, ta); }
            tu = fmax(tu, su[round][w]); ta = fmax(ta, sa[round][w]);
        }
        lu = fmax(lu, ru); la = fmax(la, ra);
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            if (b + c >= K) continue;
            const double de = coef * dx[b + c] / (fmax(lu, u[c]) + fmax(la, a[c])) / (n1e ? n1e[b + c] : N1);
            dt = fmin(dt, de);
        }
        ru = fmax(ru, tu); ra = fmax(ra, ta);
    }
    for (int off = 32; off > 0; off >>= 1) dt = fmin(dt, __shfl_xor(dt, off, 64));
    if (lane == 0) sd[wave] = dt;
    __syncthreads();
    if (t == 0) {
        for (int w = 1; w < 16; ++w) dt = fmin(dt, sd[w]);
        *dt_out = dt;
        state[0] = ru; state[1] = ra;
    }
}

// The four sums of nb partials: every lane a strided share, then a fixed tree, so a mesh always
// adds in the same order.  (One lane per sum took 270 us over 2.4 k partials.)
__global__ __launch_bounds__(1024) void k_cons_final(const double *partial, int nb, double *out) {
    __shared__ double s[16][4];
    const int t = threadIdx.x;
    const double2 *p2 = (const double2 *)partial;
    double v[4] = {0.0, 0.0, 0.0, 0.0};
    for (int b = t; b < nb; b += 1024) {
        const double2 x = p2[(int64_t)b * 2], y = p2[(int64_t)b * 2 + 1];
        v[0] += x.x; v[1] += x.y; v[2] += y.x; v[3] += y.y;
    }
#pragma unroll
    for (int c = 0; c < 4; ++c)
        for (int off = 32; off > 0; off >>= 1) v[c] += __shfl_xor(v[c], off, 64);
    if ((t & 63) == 0) {
#pragma unroll
        for (int c = 0; c < 4; ++c) s[t >> 6][c] = v[c];
    }
    __syncthreads();
    if (t < 4) {
        double acc = s[0][t];
        for (int w = 1; w < 16; ++w) acc += s[w][t];
        out[t] = acc;
    }
}

// Surface monitors of one zone (QuadMesh_Integrals.incf:67-346): one workgroup; each lane sums a
// strided share of the zone's face nodes from the stored element-side Q traces (the energy slot
// shifted back by Eref in the FP32 form) and, for Navier-Stokes, the stored viscous face-flux
// traces, whose momentum components are the stress tensor (mu (f1, f2, g2) = tau_xx, tau_xy,
// tau_yy, ViscousFluxes.f90:416-461) or its product with the normal (VT_NORMAL); then a fixed-order reduction.
template <typename TR>
__global__ __launch_bounds__(1024) void k_surface_integrals(const int *slots, int nslots, int P, const TR *tr,
                                                            const TR *vtr, int vt, const int4 *face, const double *egeo,
                                                            const double *w, double gm1, double Eref,
                                                            const double *mu_a, double mu, double *out) {
    __shared__ double s[16][9];
    const int t = threadIdx.x;
    double acc[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
    for (int x = t; x < nslots * P; x += 1024) {
        const int slot = slots[x / P], k = x % P;
        const int4 fr = face[slot];
        const int gi = (fr.x & FF_CURVED) ? ((fr.x & FF_SELFREV) ? P - 1 - k : k) : 0;
        const int wi = (fr.x & FF_SELFREV) ? P - 1 - k : k;
        const double *geo = egeo + 3 * ((int64_t)fr.z + gi);
        const double nx = geo[0], ny = geo[1], dS = geo[2], wq = w[wi];
        const TR *q = tr + ((int64_t)slot * P + k) * 4;
        const double r = q[0], ru = q[1], rv = q[2], E = (double)q[3] + Eref;
        const double p = gm1 * (E - 0.5 * (ru * ru + rv * rv) / r);
        const double un = ru * nx + rv * ny;
        acc[0] += wq * dS;
        acc[1] += p * dS * wq;
        acc[2] += r * dS * wq;
        acc[3] += p * wq * nx * dS;
        acc[4] += p * wq * ny * dS;
        acc[5] += wq * un * dS;
        acc[6] += wq * un * dS / r;
        if (vtr) {
            const TR *v = vtr + ((int64_t)slot * P + k) * vt;
            // the traces carry mu + mu_a of the (boundary) face; the monitor's stress has mu
            const double sc = mu_a ? mu / (mu + mu_a[slot >> 2]) : 1.0;
            if (vt == VT_NORMAL) {
                acc[7] += wq * (v[0] * sc) * dS;
                acc[8] += wq * (v[1] * sc) * dS;
            } else {
                const double txx = v[0] * sc, txy = v[1] * sc, tyy = v[3] * sc;
                acc[7] += wq * (txx * nx + txy * ny) * dS;
                acc[8] += wq * (txy * nx + tyy * ny) * dS;
            }
        }
    }
#pragma unroll
    for (int c = 0; c < 9; ++c)
        for (int off = 32; off > 0; off >>= 1) acc[c] += __shfl_xor(acc[c], off, 64);
    if ((t & 63) == 0) {
#pragma unroll
        for (int c = 0; c < 9; ++c) s[t >> 6][c] = acc[c];
    }
    __syncthreads();
    if (t < 9) {
        double v = s[0][t];
        for (int wv = 1; wv < 16; ++wv) v += s[wv][t];
        out[t] = v;
    }
}

// Probe_Update (IO/Monitors.f90:739-846), one wavefront per probe: B = l_xi^T A l_eta with
// (A l_eta)(i) = sum_j A(i,j) l_eta(j) (BilinearForm, MatrixOperations.f90:185-209) for each
// conservative variable of Q (or of QDot for rhot .. rhoet), lane (i, eq) a row's sum and lane eq the
// sum over i; then the tracked variable.  (One lane per probe: 4 P^2 dependent loads, 21 us at P = 6
// for any number of probes; this takes 4.)
__global__ __launch_bounds__(64) void k_probes(const double *Q, const double *QDot, const int2 *ev, const double *l,
                                               int n, int P, double gm1, double gamma, double *out) {
    __shared__ double row[64], b4[4];
    const int k = blockIdx.x, t = threadIdx.x, i = t >> 2, eq = t & 3;
    const int2 x = ev[k];
    const double *lx = l + (int64_t)k * 2 * P, *ly = lx + P;
    const double *A = ((x.y >= 4 && x.y <= 7) ? QDot : Q) + (int64_t)x.x * P * P * 4;
    if (i < P) {
        double r = 0.0;
        for (int j = 0; j < P; ++j) r += A[(i + P * j) * 4 + eq] * ly[j];
        row[t] = r;
    }
    __syncthreads();
    if (t < 4) {
        double b = 0.0;
        for (int c = 0; c < P; ++c) b += lx[c] * row[4 * c + t];
        b4[t] = b;
    }
    __syncthreads();
    if (t != 0) return;
    const double v[4] = {b4[0], b4[1], b4[2], b4[3]};
    double o;
    switch (x.y) {
    case 8: o = v[1] / v[0]; break;
    case 9: o = v[2] / v[0]; break;
    case 10: o = gm1 * (v[3] - 0.5 * (v[1] * v[1] + v[2] * v[2]) / v[0]); break;
    case 11: o = sqrt(v[1] * v[1] + v[2] * v[2]) / v[0] / sqrt(gamma); break;
    default: o = v[x.y & 3]; break;
    }
    out[k] = o;
}

__global__ __launch_bounds__(256) void k_copy(const double2 *src, double2 *dst, int n) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) dst[i] = src[i];
}

__global__ __launch_bounds__(256) void k_store_values(const double *src, int n, int stride, double *dst) {
    for (int i = threadIdx.x; i < n; i += 256) dst[i] = src[(int64_t)i * stride];
}

// Residual of each case of a batch (one workgroup): the maxima of its tiles' partials.
__global__ __launch_bounds__(1024) void k_batch_resid(const double *part, const int2 *ranges, double *const *out) {
    const int2 r = ranges[blockIdx.x];
    max_partials(part + (int64_t)r.x * 4, r.y - r.x, 0, 1024, out[blockIdx.x], kResidStride);
}

}  // namespace

bool supported_order(int N) { return N >= 1 && N <= 12; }

#define HG_DISPATCH_P(P_, CALL)          \
    switch (P_) {                        \
    case 2: return CALL(2);              \
    case 3: return CALL(3);              \
    case 4: return CALL(4);              \
    case 5: return CALL(5);              \
    case 6: return CALL(6);              \
    case 7: return CALL(7);              \
    case 8: return CALL(8);              \
    case 9: return CALL(9);              \
    case 10: return CALL(10);            \
    case 11: return CALL(11);            \
    case 12: return CALL(12);            \
    case 13: return CALL(13);            \
    default: return hipErrorInvalidValue; \
    }

hipError_t launch_art_visc(int P, bool mixed, const StageArgs &a, const double *evol, const double *w, double *mu_a,
                           hipStream_t st) {
#define HG_CALL(PV) art_visc_p<PV>(mixed, a, evol, w, mu_a, st)
    HG_DISPATCH_P(P, HG_CALL)
#undef HG_CALL
}

hipError_t launch_prolong(int P, bool mixed, const StageArgs &a, hipStream_t st) {
#define HG_CALL(PV) prolong_p<PV>(mixed, a, st)
    HG_DISPATCH_P(P, HG_CALL)
#undef HG_CALL
}

template <int PHYS>
static hipError_t launch_stage_phys(int P, int tile, bool mixed, const StageArgs &a, hipStream_t st) {
#define HG_CALL(PV) stage_phys_p<PV, PHYS>(tile, mixed, a, st)
    HG_DISPATCH_P(P, HG_CALL)
#undef HG_CALL
}

hipError_t launch_stage(int P, int tile, bool mixed, const StageArgs &a, hipStream_t st) {
    if (!a.ph.ns) return launch_stage_phys<0>(P, tile, mixed, a, st);
    if (a.ph.viscous == 2) return launch_stage_phys<2>(P, tile, mixed, a, st);
    return launch_stage_phys<1>(P, tile, mixed, a, st);
}

hipError_t launch_gradient(int P, int tile, bool mixed, const StageArgs &a, hipStream_t st) {
#define HG_CALL(PV) gradient_p<PV>(tile, mixed, a, st)
    HG_DISPATCH_P(P, HG_CALL)
#undef HG_CALL
}

hipError_t launch_resid_final(const double *part, int nb, double *out, hipStream_t st, double *scratch) {
    // one workgroup up to 8 partials per lane; beyond, a first pass of up to kResidGroups
    // workgroups into scratch, then one workgroup over their maxima (one workgroup over 64 k
    // partials took 37 us, two launches take 9, one over 3.3 k partials 4.5)
    const int groups = std::min(kResidGroups, (nb + 1023) / 1024);
    if (groups <= 8 || !scratch) {
        hipLaunchKernelGGL(k_resid_final, dim3(1), dim3(1024), 0, st, part, nb, out, kResidStride);
        return hipGetLastError();
    }
    hipLaunchKernelGGL(k_resid_final, dim3(groups), dim3(1024), 0, st, part, nb, scratch, 1);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_resid_final, dim3(1), dim3(1024), 0, st, scratch, groups, out, kResidStride);
    return hipGetLastError();
}

int tile_threads(int P, int tile) {
#define HG_CALL(PV) tile_threads_p<PV>(tile)
    switch (P) {
    case 2: return HG_CALL(2);
    case 3: return HG_CALL(3);
    case 4: return HG_CALL(4);
    case 5: return HG_CALL(5);
    case 6: return HG_CALL(6);
    case 7: return HG_CALL(7);
    case 8: return HG_CALL(8);
    case 9: return HG_CALL(9);
    case 10: return HG_CALL(10);
    case 11: return HG_CALL(11);
    case 12: return HG_CALL(12);
    case 13: return HG_CALL(13);
    default: return 0;
    }
#undef HG_CALL
}

int tile_elems(int P, int tile) {
#define HG_CALL(PV) tile_elems_p<PV>(tile)
    switch (P) {
    case 2: return HG_CALL(2);
    case 3: return HG_CALL(3);
    case 4: return HG_CALL(4);
    case 5: return HG_CALL(5);
    case 6: return HG_CALL(6);
    case 7: return HG_CALL(7);
    case 8: return HG_CALL(8);
    case 9: return HG_CALL(9);
    case 10: return HG_CALL(10);
    case 11: return HG_CALL(11);
    case 12: return HG_CALL(12);
    case 13: return HG_CALL(13);
    default: return 0;
    }
#undef HG_CALL
}

int stage_blocks(int P, int tile, int K) {
#define HG_CALL(PV) stage_blocks_p<PV>(tile, K)
    switch (P) {
    case 2: return HG_CALL(2);
    case 3: return HG_CALL(3);
    case 4: return HG_CALL(4);
    case 5: return HG_CALL(5);
    case 6: return HG_CALL(6);
    case 7: return HG_CALL(7);
    case 8: return HG_CALL(8);
    case 9: return HG_CALL(9);
    case 10: return HG_CALL(10);
    case 11: return HG_CALL(11);
    case 12: return HG_CALL(12);
    case 13: return HG_CALL(13);
    default: return 0;
    }
#undef HG_CALL
}

hipError_t launch_dt_elem(int P, const double *Q, int K, double gamma, double gm1, double *umax, double *amax,
                          hipStream_t st) {
#define HG_CALL(PV) dt_elem_p<PV>(Q, K, gamma, gm1, umax, amax, st)
    HG_DISPATCH_P(P, HG_CALL)
#undef HG_CALL
}

hipError_t launch_dt_scan(int K, const double *umax, const double *amax, const double *dx, double coef, double N1,
                          double dt_max, double *state, double *dt_out, hipStream_t st, const double *n1e) {
    hipLaunchKernelGGL(k_dt_scan, dim3(1), dim3(1024), 0, st, K, umax, amax, dx, coef, N1, dt_max, state, dt_out,
                       n1e);
    return hipGetLastError();
}

static hipError_t cons_partial(int P, const double *Q, const double *jac, const double *w, int K, int mode,
                               double gamma, double gm1, double *partial,
                               int nbk, hipStream_t st) {
#define HG_CALL(PV) (cons_blocks_p<PV>(K) > nbk ? hipErrorInvalidValue : cons_partial_p<PV>(Q, jac, w, K, mode, gamma, gm1, partial, st))
    HG_DISPATCH_P(P, HG_CALL)
#undef HG_CALL
}

static int cons_blocks(int P, int K) {
#define HG_CALL(PV) cons_blocks_p<PV>(K)
    switch (P) {
    case 2: return HG_CALL(2);
    case 3: return HG_CALL(3);
    case 4: return HG_CALL(4);
    case 5: return HG_CALL(5);
    case 6: return HG_CALL(6);
    case 7: return HG_CALL(7);
    case 8: return HG_CALL(8);
    case 9: return HG_CALL(9);
    case 10: return HG_CALL(10);
    case 11: return HG_CALL(11);
    case 12: return HG_CALL(12);
    case 13: return HG_CALL(13);
    default: return 0;
    }
#undef HG_CALL
}

hipError_t launch_cons_sums(int P, const double *Q, const double *jac, const double *w, int K, double *partial,
                            int nbk, double *out, hipStream_t st) {
    hipError_t e = cons_partial(P, Q, jac, w, K, 0, 0.0, 0.0, partial, nbk, st);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_cons_final, dim3(1), dim3(1024), 0, st, partial, cons_blocks(P, K), out);
    return hipGetLastError();
}

hipError_t launch_volume_integrals(int P, const double *Q, const double *jac, const double *w, int K, double gamma,
                                   double gm1, double *partial, int nbk, double *out, hipStream_t st) {
    hipError_t e = cons_partial(P, Q, jac, w, K, 1, gamma, gm1, partial, nbk, st);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_cons_final, dim3(1), dim3(1024), 0, st, partial, cons_blocks(P, K), out);
    return hipGetLastError();
}

hipError_t launch_surface_integrals(bool mixed, const int *slots, int nslots, int P, const void *tr, const void *vtr, int vt,
                                    const int4 *face, const double *egeo, const double *w, double gm1, double Eref,
                                    const double *mu_a, double mu, double *out, hipStream_t st) {
    if (mixed)
        hipLaunchKernelGGL((k_surface_integrals<float>), dim3(1), dim3(1024), 0, st, slots, nslots, P,
                           (const float *)tr, (const float *)vtr, vt, face, egeo, w, gm1, Eref, mu_a, mu, out);
    else
        hipLaunchKernelGGL((k_surface_integrals<double>), dim3(1), dim3(1024), 0, st, slots, nslots, P,
                           (const double *)tr, (const double *)vtr, vt, face, egeo, w, gm1, Eref, mu_a, mu, out);
    return hipGetLastError();
}

hipError_t launch_copy(const void *src, void *dst, size_t bytes, hipStream_t st) {
    const int n = (int)(bytes / 16);
    hipLaunchKernelGGL(k_copy, dim3((n + 255) / 256), dim3(256), 0, st, (const double2 *)src, (double2 *)dst, n);
    return hipGetLastError();
}

hipError_t launch_store_values(const double *src, int n, int stride, double *dst, hipStream_t st) {
    hipLaunchKernelGGL(k_store_values, dim3(1), dim3(256), 0, st, src, n, stride, dst);
    return hipGetLastError();
}

hipError_t launch_probes(const double *Q, const double *QDot, const int2 *ev, const double *l, int n, int P,
                         double gm1, double gamma, double *out, hipStream_t st) {
    hipLaunchKernelGGL(k_probes, dim3(n), dim3(64), 0, st, Q, QDot, ev, l, n, P, gm1, gamma, out);
    return hipGetLastError();
}

}  // namespace hg

namespace hg {

hipError_t launch_batch_stage(int variant, int rs, int tile, const BatchArgs &b, int block, hipStream_t st) {
#define HG_RS(V)                                                    \
    switch (rs) {                                                   \
    case -1: return batch_stage_v##V##_rs0(tile, b, block, st);     \
    case 0: return batch_stage_v##V##_rs1(tile, b, block, st);      \
    case 1: return batch_stage_v##V##_rs2(tile, b, block, st);      \
    case 2: return batch_stage_v##V##_rs3(tile, b, block, st);      \
    case 3: return batch_stage_v##V##_rs4(tile, b, block, st);      \
    default: return hipErrorInvalidValue;                           \
    }
    switch (variant) {
    case 0: HG_RS(0)
    case 1: HG_RS(1)
    case 2: HG_RS(2)
    case 3: HG_RS(3)
    case 4: HG_RS(4)
    case 5: HG_RS(5)
    default: return hipErrorInvalidValue;
    }
#undef HG_RS
}

hipError_t launch_batch_gradient(int variant, int tile, const BatchArgs &b, int block, hipStream_t st) {
    switch (variant) {
    case 2: return batch_gradient_v2(tile, b, block, st);
    case 3: return batch_gradient_v3(tile, b, block, st);
    case 4: return batch_gradient_v4(tile, b, block, st);
    case 5: return batch_gradient_v5(tile, b, block, st);
    default: return hipErrorInvalidValue;
    }
}

hipError_t launch_batch_stage_p(int variant, int rs, int P, int tile, const BatchArgs &b, hipStream_t st) {
#define HG_RS(V)                                                        \
    switch (rs) {                                                       \
    case -1: return batch_stage_v##V##_rs0_p(P, tile, b, st);           \
    case 0: return batch_stage_v##V##_rs1_p(P, tile, b, st);            \
    case 1: return batch_stage_v##V##_rs2_p(P, tile, b, st);            \
    case 2: return batch_stage_v##V##_rs3_p(P, tile, b, st);            \
    case 3: return batch_stage_v##V##_rs4_p(P, tile, b, st);            \
    default: return hipErrorInvalidValue;                               \
    }
    switch (variant) {
    case 0: HG_RS(0)
    case 1: HG_RS(1)
    case 2: HG_RS(2)
    case 3: HG_RS(3)
    case 4: HG_RS(4)
    case 5: HG_RS(5)
    default: return hipErrorInvalidValue;
    }
#undef HG_RS
}

hipError_t launch_batch_gradient_p(int variant, int P, int tile, const BatchArgs &b, hipStream_t st) {
    switch (variant) {
    case 2: return batch_gradient_v2_p(P, tile, b, st);
    case 3: return batch_gradient_v3_p(P, tile, b, st);
    case 4: return batch_gradient_v4_p(P, tile, b, st);
    case 5: return batch_gradient_v5_p(P, tile, b, st);
    default: return hipErrorInvalidValue;
    }
}

hipError_t launch_batch_resid(const double *part, const int2 *ranges, double *const *out, int ncases, hipStream_t st) {
    hipLaunchKernelGGL(k_batch_resid, dim3(ncases), dim3(1024), 0, st, part, ranges, out);
    return hipGetLastError();
}

}  // namespace hg
