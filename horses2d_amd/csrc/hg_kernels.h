// Stage, gradient and trace kernels of the DGSEM residual + low-storage RK for gfx950.
//
// Data layout in HBM (uniform polynomial order P = N+1 per handle):
//   Q, G      : FP64, reference layout  Q[(e*P*P + i + P*j)*4 + eq]
//   traces    : [(e*4 + f)*P + k][4]  element-local face orientation, FP64 or FP32
//   viscous flux traces: [(e*4 + f)*P + k][vt], FP64 or FP32: mu times each side's viscous
//               flux at its face nodes, in FP64 its normal component (the gradient itself is never
//               stored: the nodal gradient is recomputed inside each stage)
//   metric    : five planes of e*P*P+n: Ja11, Ja12, Ja21, Ja22, 1/jac (FP64 or FP32; the FP32
//               form stores one record per element when the metric is element-constant, the FP64
//               form one per line of nodes when every element is straight-sided); the
//               divisions by the Jacobian (DGSpatialDiscretizationMethods.f90:226-233) are
//               multiplications by its reciprocal (a last-bit difference, not bit-exact)
//
// Tiling: a workgroup owns EPB whole elements (one lane per node, one lane per face node);
// two tile shapes per order are compiled (the widest that fits one wavefront, and the widest
// that fits four) and the faster is chosen per handle at creation.  Every global load a lane
// needs is issued before the first barrier so that its latency overlaps with the other
// lanes' loads; the element state is staged in LDS for the tensor-product contractions.
//
// Each element computes the Riemann fluxes of its own four faces: the neighbor reads the
// same trace values and evaluates the identical expression, so both sides see
// bit-identical fluxes (the reference's FL = F, FR = -F), and the face lifts are subtracted
// in ascending global edge order (DGSpatialDiscretizationMethods.f90:196-220).
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

#include "hg_device.h"
#include "hg_physics.h"

namespace hg {

template <typename T>
__device__ inline T ld(const void *p, int64_t i) { return ((const T *)p)[i]; }

// Per equation, the maximum of |q| over a wavefront's lanes, every lane active.  Lane l returns that of
// value wave_max4_value(l).  Magnitudes compare as the unsigned integers of their bits, where a NaN is
// above infinity.  Two steps within the quads halve the values
// a lane carries, so each of the other four exchanges one value instead of four: 10 cross-lane moves
// of 32 bits against the 48 of a shuffle tree per value, which made the last stage of a step 10 %
// longer than the others (148 against 135 us on an ensemble of 16 M unknowns, 235 against 214 us on
// the 256 x 256 interior-penalty mesh).
__device__ __forceinline__ int wave_max4_value(int l) { return 2 * (l & 1) + ((l >> 1) & 1); }

template <int CTRL>
__device__ __forceinline__ uint64_t dpp_move(uint64_t v) {
    const int lo = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)v, CTRL, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)(v >> 32), CTRL, 0xf, 0xf, false);
    return ((uint64_t)(uint32_t)hi << 32) | (uint32_t)lo;
}

__device__ __forceinline__ uint64_t wave_max4(const double *q) {
    uint64_t v[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) v[c] = (uint64_t)__double_as_longlong(fabs(q[c]));
    const int l = threadIdx.x;
    constexpr int QUAD_XOR1 = 0xB1, QUAD_XOR2 = 0x4E, ROW_ROR4 = 0x124, ROW_ROR8 = 0x128;
    const bool odd = l & 1, up = l & 2;
    // even lanes keep values 0, 1 and hand over 2, 3
    const uint64_t r0 = dpp_move<QUAD_XOR1>(odd ? v[0] : v[2]), r1 = dpp_move<QUAD_XOR1>(odd ? v[1] : v[3]);
    const uint64_t p0 = max(odd ? v[2] : v[0], r0), p1 = max(odd ? v[3] : v[1], r1);
    uint64_t m = max(up ? p1 : p0, dpp_move<QUAD_XOR2>(up ? p0 : p1));
    m = max(m, dpp_move<ROW_ROR4>(m));
    m = max(m, dpp_move<ROW_ROR8>(m));
    m = max(m, (uint64_t)__shfl_xor((unsigned long long)m, 16, 64));
    return max(m, (uint64_t)__shfl_xor((unsigned long long)m, 32, 64));
}

// Tile handled by workgroup b of nb.  The dispatcher hands consecutive workgroups to the eight
// XCDs in turn; this gives each XCD a contiguous range of tiles (a band of the mesh), so that
// the traces a tile reads from its neighbours were mostly written through the same XCD's L2.
// A bijection of [0, nb): every tile is processed once, wherever it runs.
__device__ __forceinline__ int xcd_tile(int b, int nb) {
    const int x = b & 7, q = b >> 3, per = nb >> 3, rem = nb & 7;
    return x * per + (x < rem ? x : rem) + q;
}

// LDS layout of an element's nodes: node (i, j) is entry i + RS j of ES entries per element, an
// entry being 16 bytes of each plane (Quads below).  The pads spread the rows (P = 4 and 8, whose
// rows of 64 and 128 B otherwise share banks) or the elements of a tile (P = 3, 6, 7) over the
// banks.  The row and column reads of a wide tile's FP64 contraction, and its trace reads, timed
// alone (one 32-byte entry per node without pads -> this layout): P = 3 29 -> 16 and 23 -> 16 us,
// P = 4 38 -> 25 and 37 -> 21, P = 5 38 -> 30 and 31 -> 23, P = 6 53 -> 38 and 28 -> 20,
// P = 7 45 -> 40 and 29 -> 23, P = 8 92 -> 45 and 72 -> 22, P = 9 71 -> 53 and 31 -> 23; pads at
// the other orders gain nothing.
template <int P>
struct Layout {
    static constexpr int RS = P + ((P == 4 || P == 8) ? 1 : 0);
    static constexpr int ES = P * RS + ((P == 3 || P == 6) ? 3 : P == 7 ? 7 : P == 8 ? -1 : 0);
    // entry of node n (= i + P j) of the tile's element s
    __device__ static constexpr int at(int s, int n) { return s * ES + n + (RS - P) * (n / P); }
};

template <int P, int EPB_>
struct Tile {
    static constexpr int PP = P * P;
    static constexpr int EPB = EPB_;
    static constexpr int NF = EPB * 4 * P;
    static constexpr int NN = EPB * PP;
    static constexpr int NL = EPB * Layout<P>::ES;   // entries of a node array in LDS
    static constexpr int TPB = (((NN > NF ? NN : NF) + 63) / 64) * 64;
};

// Arrays of NL four-value entries in LDS.  FP64: two planes of 16-byte halves (entry x of plane h
// holds values 2 h, 2 h + 1), so that neighbouring entries are 16 bytes apart for every ds_read_b128
// instead of 32, where half of the banks were visited twice; FP32: one plane of float4.
template <typename R, int NL>
struct Quads {
    static constexpr int SIZE = 4 * NL;   // values of R
    __device__ static __forceinline__ void get(const R *A, int x, R *v) {
        if constexpr (sizeof(R) == 8) {
            const double2 a = *(const double2 *)(A + 2 * x), b = *(const double2 *)(A + 2 * NL + 2 * x);
            v[0] = a.x; v[1] = a.y; v[2] = b.x; v[3] = b.y;
        } else {
            const float4 a = *(const float4 *)(A + 4 * x);
            v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
        }
    }
    __device__ static __forceinline__ void put(R *A, int x, const R *v) {
        if constexpr (sizeof(R) == 8) {
            *(double2 *)(A + 2 * x) = make_double2(v[0], v[1]);
            *(double2 *)(A + 2 * NL + 2 * x) = make_double2(v[2], v[3]);
        } else {
            *(float4 *)(A + 4 * x) = make_float4(v[0], v[1], v[2], v[3]);
        }
    }
    // values 2 h and 2 h + 1 of entry x
    __device__ static __forceinline__ void get_half(const R *A, int x, int h, R &a, R &b) {
        if constexpr (sizeof(R) == 8) {
            const double2 v = *(const double2 *)(A + 2 * NL * h + 2 * x);
            a = v.x; b = v.y;
        } else {
            const float2 v = *(const float2 *)(A + 4 * x + 2 * h);
            a = v.x; b = v.y;
        }
    }
};

// Trace of a face from the staged element state (DGSpatialDiscretizationMethods.f90:1520-1574):
// X is an array of NL entries (Quads), x0 the element's first.  Accumulated in FP64 with explicit
// fma in l order so that every kernel that forms a trace (prolongation, stage epilogue) produces
// the same bits; A = T accumulates in the tile's own type (the FP32 form's gradient traces, which
// only the kernel that forms them ever evaluates).
template <int P, int NL, int UNROLL = P, typename T, typename A>
__device__ __forceinline__ void face_trace(const T *X, int x0, const A *sLb, int f, int k, A *out) {
    const A *lb = (f == 0 || f == 3) ? sLb : sLb + P;
    // nodes (k, l) of a horizontal face or (l, k) of a vertical one: a base and a stride, so
    // the loop body has no face-dependent branch
    constexpr int RS = Layout<P>::RS;
    const bool horiz = (f == 0 || f == 2);
    const int base = x0 + (horiz ? k : RS * k), step = horiz ? RS : 1;
#pragma unroll
    for (int c = 0; c < 4; ++c) out[c] = A(0);
#pragma unroll UNROLL
    for (int l = 0; l < P; ++l) {
        T v[4];
        Quads<T, NL>::get(X, base + step * l, v);
#pragma unroll
        for (int c = 0; c < 4; ++c) out[c] = fma((A)v[c], lb[l], out[c]);
    }
}

// The same together with the derivative along the line at its end, sum of q(l) lbd(l) (lbd: lb D or lb
// hatD, one row per side), from the same reads.
template <int P, int NL, int UNROLL = P>
__device__ __forceinline__ void face_trace_slope(const double *X, int x0, const double *sLb, const double *sLbd, int f,
                                                 int k, double *out, double *nd) {
    const int side = (f == 0 || f == 3) ? 0 : P;
    constexpr int RS = Layout<P>::RS;
    const bool horiz = (f == 0 || f == 2);
    const int base = x0 + (horiz ? k : RS * k), step = horiz ? RS : 1;
#pragma unroll
    for (int c = 0; c < 4; ++c) out[c] = nd[c] = 0.0;
#pragma unroll UNROLL
    for (int l = 0; l < P; ++l) {
        double v[4];
        Quads<double, NL>::get(X, base + step * l, v);
        const double b = sLb[side + l], d = sLbd[side + l];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            out[c] = fma(v[c], b, out[c]);
            nd[c] = fma(v[c], d, nd[c]);
        }
    }
}

// Derivative along a face at its node k from the face's Q traces (an array of NF entries, f0 the face's
// first), M the transposed D or hatD.
template <int P, int NF, int UNROLL = P>
__device__ __forceinline__ void face_tangent(const double *T, int f0, const double *M, int k, double *td) {
#pragma unroll
    for (int c = 0; c < 4; ++c) td[c] = 0.0;
#pragma unroll UNROLL
    for (int l = 0; l < P; ++l) {
        double v[4];
        Quads<double, NF>::get(T, f0 + l, v);
        const double d = M[l * P + k];
#pragma unroll
        for (int c = 0; c < 4; ++c) td[c] = fma(v[c], d, td[c]);
    }
}

// The same for an eight-value array (two Quads arrays one after the other): one pass over the nodes.
template <int P, int NL, int UNROLL = P, typename T, typename A>
__device__ __forceinline__ void face_trace8(const T *X, int x0, const A *sLb, int f, int k, A *out) {
    const A *lb = (f == 0 || f == 3) ? sLb : sLb + P;
    constexpr int RS = Layout<P>::RS;
    const bool horiz = (f == 0 || f == 2);
    const int base = x0 + (horiz ? k : RS * k), step = horiz ? RS : 1;
#pragma unroll
    for (int c = 0; c < 8; ++c) out[c] = A(0);
#pragma unroll UNROLL
    for (int l = 0; l < P; ++l) {
        T v[8];
        Quads<T, NL>::get(X, base + step * l, v);
        Quads<T, NL>::get(X + Quads<T, NL>::SIZE, base + step * l, v + 4);
#pragma unroll
        for (int c = 0; c < 8; ++c) out[c] = fma((A)v[c], lb[l], out[c]);
    }
}

// Tile choices: 0 = widest tile within one wavefront, 1 = widest within four wavefronts whose
// Euler FP64 LDS tile (state, two contravariant fluxes, face fluxes: 96 ES + 128 P bytes per
// element) stays within 31 KB, so that five workgroups fit a CU's LDS (the batched kernels' LDS
// is the largest tile over all orders).  P = 4: 12 elements, three full wavefronts, where 13 fit.
template <int P>
struct Tiles {
    static constexpr int a64 = 64 / (P * P), b64 = 64 / (4 * P);
    static constexpr int a256 = 256 / (P * P), b256 = 256 / (4 * P);
    static constexpr int lds_fit = (31 * 1024) / (96 * Layout<P>::ES + 128 * P);
    static constexpr int lds_cap = P == 4 ? 12 : lds_fit;
    static constexpr int small = (a64 < b64 ? a64 : b64) > 0 ? (a64 < b64 ? a64 : b64) : 1;
    static constexpr int wide = (a256 < b256 ? a256 : b256) > 0 ? (a256 < b256 ? a256 : b256) : 1;
    static constexpr int large = (wide < lds_cap ? wide : lds_cap) > 0 ? (wide < lds_cap ? wide : lds_cap) : 1;
};

// The state of node g: each lane reads its own node's 32 bytes, so no lane waits for another's
// before it has its own.
__device__ __forceinline__ void load_node(const double *Q, int64_t g, double *q) {
    const double2 *p = (const double2 *)(Q + g * 4);
    const double2 a = p[0], b = p[1];
    q[0] = a.x; q[1] = a.y; q[2] = b.x; q[3] = b.y;
}

// The state slot the compute type sees (energy shifted in the FP32 form).
template <typename R>
__device__ __forceinline__ R qslot(const PhysParams &pp, double v, int c) {
    return (R)(c == 3 ? slot_energy<R>(pp, v) : v);
}

// The compute-type copy of a node's state that the FP32 form's gradient contractions read.
template <int NL, typename R>
__device__ __forceinline__ void put_slots(const PhysParams &pp, R *sQf, int x, const double *q) {
    R v[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) v[c] = qslot<R>(pp, q[c], c);
    Quads<R, NL>::put(sQf, x, v);
}

// ------------------------------------------------------------------ prolongation
template <int P, int EPB, typename TR>
__global__ __launch_bounds__((Tile<P, EPB>::TPB)) void k_prolong(StageArgs a) {
    using T = Tile<P, EPB>;
    __shared__ __align__(16) double sQ[T::NL * 4];
    __shared__ double sLb[2 * P];
    const int t = threadIdx.x, e0 = blockIdx.x * EPB;
    if (t < 2 * P) sLb[t] = a.lb[t];
    if (t < T::NN && e0 + t / T::PP < a.K) {
        double q[4];
        load_node(a.Q, (int64_t)e0 * T::PP + t, q);
        Quads<double, T::NL>::put(sQ, Layout<P>::at(t / T::PP, t % T::PP), q);
    }
    __syncthreads();
    if (t < T::NF) {
        const int s = t / (4 * P), f = (t / P) % 4, k = t % P, e = e0 + s;
        if (e < a.K) {
            double tq[4];
            face_trace<P, T::NL>(sQ, s * Layout<P>::ES, sLb, f, k, tq);
            tq[3] = slot_energy<TR>(a.ph, tq[3]);
            TR *o = (TR *)a.tr_out + ((int64_t)(e * 4 + f) * P + k) * 4;
#pragma unroll
            for (int c = 0; c < 4; ++c) o[c] = (TR)tq[c];
        }
    }
}

// ------------------------------------------------------------------ gradient helpers
// Both the trace kernel (k_gradient) and the stage kernel evaluate the element gradient with
// these functions, so the gradient a stage recomputes for its own element is the one whose
// face traces its neighbours read.

// The state a boundary face node's ghost state starts from: its zone's record (8 doubles per
// zone, the state in the first four), or, on a face flagged FF_FSTATE, the node's own value of
// the zone's boundary-state function (slot = (element*4 + face)*P + node).
__device__ __forceinline__ const double *zone_state(const StageArgs &a, int flags, int y, int64_t slot) {
    return (flags & FF_FSTATE) ? a.fstate + slot * 4 : a.zone + 8 * y;
}

// BR1 solution flux at a face node: uStar n dS in both directions (DGViscous_BR1.f90:313-328;
// boundary faces use the ghost state's uSB, DGViscousMethods.f90:786-917).  FP64: six values per face
// node, uStar dS and (nx, ny), which the lift multiplies by lw n; FP32, whose sums keep the order (uStar
// dS) nx lw: (uStar dS) nx and (uStar dS) ny, formed once here, as two Quads arrays.
// zd: the boundary's zone state (zone_state); NF: face nodes of the tile, t: this one.
template <typename R>
constexpr int br1_width() { return sizeof(R) == 8 ? 6 : 8; }

template <int NF, typename R>
__device__ __forceinline__ void put_br1_flux(R *Fu, int t, const R *f, R nx, R ny) {
    if constexpr (sizeof(R) == 8) {
        R *out = Fu + t * 6;
#pragma unroll
        for (int c = 0; c < 4; ++c) out[c] = f[c];
        out[4] = nx; out[5] = ny;
    } else {
        R fx[4], fy[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) { fx[c] = f[c] * nx; fy[c] = f[c] * ny; }
        Quads<R, NF>::put(Fu, t, fx);
        Quads<R, NF>::put(Fu + 4 * NF, t, fy);
    }
}

template <int NF, typename R, bool XB>
__device__ __forceinline__ void br1_face_flux(const StageArgs &a, const Phys<R> &ph, int flags, const double *zd,
                                              const R *qs, const R *qo, R nx, R ny, R dS, R *Fu, int t) {
    const int kind = flags & 15;
    R us[4];
    if (kind <= FK_PERIODIC) {
#pragma unroll
        for (int c = 0; c < 4; ++c) us[c] = R(0.5) * (qs[c] + qo[c]);
        if (kind == FK_INT_R) {
#pragma unroll
            for (int c = 0; c < 4; ++c) us[c] = -us[c];
        }
    } else if (kind == FK_MORTAR) {
        // projected and signed by the mortar kernel (load_face put it in qo)
        if (flags & FF_MCURVED) {
            // a curved mortar edge: qo holds uStar dS nx already; the y terms follow separately
            put_br1_flux<NF>(Fu, t, qo, R(1), R(0));
            return;
        }
#pragma unroll
        for (int c = 0; c < 4; ++c) us[c] = qo[c];
    } else {
        R uB[4];
        int neu;
        ghost_state<R, XB>(kind, flags, zd, a.ph, ph, qs, nx, ny, uB, us, neu);
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) us[c] = us[c] * dS;
    put_br1_flux<NF>(Fu, t, us, nx, ny);
}

// BR1 gradient at node (i, j): ( -Vector_StdVolumeGreen(Q) + sum_faces Vector_StdFace(uStar) ) / jac
// (DGViscous_BR1.f90:48-111, DGWeakIntegrals.f90:503-622), faces lifted in edge-id order.
// q: the tile's state in the compute type (Quads; energy slot shifted in the FP32 form), Ja: its
// metric (Quads: Ja11, Ja21, Ja12, Ja22), x0 the element's first entry in both, Fu: the tile's uStar
// fluxes (see br1_face_flux), f0 the element's first face node, sHat: hatD transposed (hatD(i, l) at [l*P + i]).
// Faces whose bit 8 + f is set in ord are curved p-non-conforming or subdivided edges, whose
// lift terms come per direction from the mortar kernel (uStar dS n projected direction by
// direction): the face lane stores the x terms with the "normal" (1, 0), and mortar_y_lift adds
// the y terms afterwards.
template <int P, int NL, int NF, typename R, int UNROLL = P>
__device__ __forceinline__ void br1_node_gradient(const R *q, const R *Ja, int x0, const R *sHat, const R *Fu, int f0,
                                                  const R *sLbw, int ord, int i, int j, R ijac, R *dq,
                                                  bool affine = false, R j11 = R(0), R j12 = R(0), R j21 = R(0),
                                                  R j22 = R(0)) {
    bool done = false;
    if constexpr (sizeof(R) == 8) {
        if (affine) {   // the metric out of the sums
            R dxi[4] = {0, 0, 0, 0}, deta[4] = {0, 0, 0, 0};
            // half unrolled up to P = 9, where the full loop spills a few registers
            constexpr int HALF = UNROLL > 2 && P <= 9 ? (P + 1) / 2 : UNROLL;
#pragma unroll HALF
            for (int l = 0; l < P; ++l) {
                const R hi = sHat[l * P + i], hj = sHat[l * P + j];
                R vx[4], vy[4];
                Quads<R, NL>::get(q, x0 + l + Layout<P>::RS * j, vx);
                Quads<R, NL>::get(q, x0 + i + Layout<P>::RS * l, vy);
#pragma unroll
                for (int c = 0; c < 4; ++c) { dxi[c] += vx[c] * hi; deta[c] += vy[c] * hj; }
            }
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                dq[c] = -(dxi[c] * j11 + deta[c] * j12);
                dq[4 + c] = -(dxi[c] * j21 + deta[c] * j22);
            }
            done = true;
        }
    }
    if (!done) {
        // Every accumulator receives its xi terms (l = 0..P-1) then its eta terms; each state value
        // is read once and used for both directions, and the metric-weighted derivative entry
        // Ja * hatD is formed once per node for all four variables.
        constexpr int RS = Layout<P>::RS;
        using V = Quads<R, NL>;
        R acc[8];
#pragma unroll
        for (int c = 0; c < 8; ++c) acc[c] = R(0);
#pragma unroll UNROLL
        for (int l = 0; l < P; ++l) {
            const int m = x0 + l + RS * j;
            const R h = sHat[l * P + i];
            R j11, j21, v[4];
            V::get_half(Ja, m, 0, j11, j21);
            V::get(q, m, v);
            const R w0 = j11 * h, w2 = j21 * h;
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                acc[c] += v[c] * w0;
                acc[4 + c] += v[c] * w2;
            }
        }
#pragma unroll UNROLL
        for (int l = 0; l < P; ++l) {
            const int m = x0 + i + RS * l;
            const R h = sHat[l * P + j];
            R j12, j22, v[4];
            V::get_half(Ja, m, 1, j12, j22);
            V::get(q, m, v);
            const R w1 = j12 * h, w3 = j22 * h;
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                acc[c] += v[c] * w1;
                acc[4 + c] += v[c] * w3;
            }
        }
#pragma unroll
        for (int c = 0; c < 8; ++c) dq[c] = -acc[c];
    }
#pragma unroll
    for (int o = 0; o < 4; ++o) {
        const int f = (ord >> (2 * o)) & 3;
        const int xf = f0 + f * P + ((f == 0 || f == 2) ? i : j);
        const R lw = (f == 0) ? sLbw[j] : (f == 1) ? sLbw[P + i] : (f == 2) ? sLbw[P + j] : sLbw[i];
        if constexpr (sizeof(R) == 8) {
            const R *F = Fu + xf * 6;
            const R wx = F[4] * lw, wy = F[5] * lw;
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                dq[c] += F[c] * wx;
                dq[4 + c] += F[c] * wy;
            }
        } else {
            R ux[4], uy[4];
            Quads<R, NF>::get(Fu, xf, ux);
            Quads<R, NF>::get(Fu + 4 * NF, xf, uy);
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                dq[c] += ux[c] * lw;
                dq[4 + c] += uy[c] * lw;
            }
        }
    }
#pragma unroll
    for (int c = 0; c < 8; ++c) dq[c] = dq[c] * ijac;
}

// The y-direction lift terms of an element's curved mortar faces (bit 8 + f of ord), added to
// the gradient br1_node_gradient formed: (uStar dS ny projected) lw / jac from mu8 (the element's
// [(f*P + k)*8] block of StageArgs::mustar).  FP64 only (meshes with mortar edges run in it).
template <int P, typename R>
__device__ __forceinline__ void mortar_y_lift(const double *mu8, const R *sLbw, int ord, int i, int j, R ijac, R *dq) {
    if constexpr (sizeof(R) == 8) {
#pragma unroll 1
        for (int f = 0; f < 4; ++f) {
            if (!((ord >> (8 + f)) & 1)) continue;
            const R lw = (f == 0) ? sLbw[j] : (f == 1) ? sLbw[P + i] : (f == 2) ? sLbw[P + j] : sLbw[i];
            const double *M = mu8 + (f * P + ((f == 0 || f == 2) ? i : j)) * 8;
#pragma unroll
            for (int c = 0; c < 4; ++c) dq[4 + c] += (R)(M[4 + c] * lw) * ijac;
        }
    }
}

// Interior (broken) gradient of the IP method (QuadElement_QuadProcedures.incf:42-88); q as above.
// sD: D transposed (D(i, l) at [l*P + i]).
template <int P, int NL, typename R, int UNROLL = P>
__device__ __forceinline__ void ip_node_gradient(const R *q, int x0, const R *sD, int i, int j, R j11, R j12, R j21,
                                                 R j22, R ijac, R *dq) {
    // l outermost (each accumulator still sums l = 0..P-1 in order): few nodes' values live
    R dxi[4] = {R(0), R(0), R(0), R(0)}, deta[4] = {R(0), R(0), R(0), R(0)};
#pragma unroll UNROLL
    for (int l = 0; l < P; ++l) {
        const R di = sD[l * P + i], dj = sD[l * P + j];
        R qx[4], qy[4];
        Quads<R, NL>::get(q, x0 + l + Layout<P>::RS * j, qx);
        Quads<R, NL>::get(q, x0 + i + Layout<P>::RS * l, qy);
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            dxi[c] += di * qx[c];
            deta[c] += dj * qy[c];
        }
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        dq[c] = (dxi[c] * j11 + deta[c] * j12) * ijac;
        dq[4 + c] = (dxi[c] * j21 + deta[c] * j22) * ijac;
    }
}

// Metric of node g, node n (= i + P j) of element e.  METRIC_NODE: five planes of nodes; METRIC_ELEM
// (FP32 form): five planes of elements.  METRIC_LINE (FP64 form, straight-sided elements): the
// derivatives of the bilinear map along eta depend on i alone and those along xi on j alone, so two
// values per line of nodes replace 40 B per node, and the Jacobian and its reciprocal are formed here in
// the host's operations, hence the same bits.  128 x 128 elements at N = 6: the Euler stage
// 37.7 -> 33.2 us, the BR1 gradient kernel 27.0 -> 23.5 us.  Parallelograms: one reciprocal per element
// behind the lines (128 x 128, N = 6, Navier-Stokes: 178.6 -> 176.5 us a step without the divisions).
template <int P, typename R>
__device__ __forceinline__ void load_metric(const StageArgs &a, int e, int n, int64_t g, R &j11, R &j12, R &j21, R &j22,
                                            R &ijac) {
    if constexpr (sizeof(R) == 8) {
        if (a.metric_kind == METRIC_LINE) {
            const double2 *L = (const double2 *)a.metric;
            const double2 e11 = L[(int64_t)e * P + n % P], e12 = L[(int64_t)(a.K + e) * P + n / P];
            j11 = e11.x; j21 = e11.y; j12 = e12.x; j22 = e12.y;
            if (a.affine) {
                ijac = ((const double *)a.metric)[4 * (int64_t)a.K * P + e];
                return;
            }
            double jac;
            {
#pragma clang fp contract(off)
                jac = j22 * j11 - j21 * j12;
            }
            ijac = 1.0 / jac;
            return;
        }
    }
    const bool el = sizeof(R) == 4 && a.metric_kind == METRIC_ELEM;
    const int64_t i = el ? (int64_t)e : g, st = el ? (int64_t)a.K : a.nodes;
    j11 = ld<R>(a.metric, i); j12 = ld<R>(a.metric, st + i);
    j21 = ld<R>(a.metric, 2 * st + i); j22 = ld<R>(a.metric, 3 * st + i);
    ijac = ld<R>(a.metric, 4 * st + i);
}

// Viscosity of a face: mu + edge % mu_a, the edge's artificial viscosity being the mean of its
// elements' (ComputeEdgeViscosity, DGArtificialDissipation.f90:340-363; boundary and periodic
// faces: the own element's).  Without artificial dissipation, mu.
template <typename R>
__device__ __forceinline__ R face_mu(const StageArgs &a, const Phys<R> &ph, int fe, int4 fr) {
    if (!a.mu_a) return ph.mu;
    const double ma = (fr.x & 15) <= FK_INT_R ? (a.mu_a[fe] + a.mu_a[fr.y >> 2]) / 2.0 : a.mu_a[fe];
    return (R)(a.ph.mu + ma);
}

// Edge viscosity of the Laplacian dissipation (JumpsBasedEdgeViscosity,
// DGArtificialDissipation.f90:340-363): the mean of the two elements' (boundary and periodic
// faces: the own element's).
__device__ __forceinline__ double face_lap(const StageArgs &a, int fe, int4 fr) {
    return (fr.x & 15) <= FK_INT_R ? (a.lap[fe] + a.lap[fr.y >> 2]) / 2.0 : a.lap[fe] / 1.0;
}

// Face-node geometry and the neighbour's Q trace (periodic and interior faces).
template <int P, typename R, typename TR>
__device__ __forceinline__ void load_face(const StageArgs &a, int fe, int ff, int fk, int4 &fr, R &nx, R &ny, R &dS,
                                          R *qo, int64_t &nslot) {
    fr = a.face[fe * 4 + ff];
    const bool curved = fr.x & FF_CURVED, selfrev = fr.x & FF_SELFREV, rev = fr.x & FF_REV;
    const int gi = curved ? (selfrev ? P - 1 - fk : fk) : 0;
    const double *geo = a.egeo + 3 * ((int64_t)fr.z + gi);
    nx = (R)geo[0]; ny = (R)geo[1]; dS = (R)geo[2];
    nslot = (int64_t)fr.y * P + (rev ? P - 1 - fk : fk);
    if ((fr.x & 15) <= FK_PERIODIC) {
        const TR *nbt = (const TR *)a.tr_in + nslot * 4;
#pragma unroll
        for (int c = 0; c < 4; ++c) qo[c] = (R)nbt[c];
    } else if ((fr.x & 15) == FK_MORTAR && a.mustar) {
        // p-non-conforming edge: this side's projected uStar in place of a neighbour trace
        const double *u = a.mustar + ((int64_t)(fe * 4 + ff) * P + fk) * 8;
#pragma unroll
        for (int c = 0; c < 4; ++c) qo[c] = (R)u[c];
    }
}

// Values of a stored viscous flux trace that a stage keeps.
template <typename R>
constexpr int vis_width() { return sizeof(R) == 8 ? VT_NORMAL : VT_FLUX; }

// One side's viscous flux trace of a face node.  FP64: its components along (nx, ny); opposite: stored
// along the opposite normal (the partner of a periodic face).
template <typename R, typename TR>
__device__ __forceinline__ void load_viscous_trace(const StageArgs &a, int64_t slot, R nx, R ny, bool opposite, R *v) {
    if constexpr (sizeof(R) == 4) {
        const TR *o = (const TR *)a.dtr + slot * VT_FLUX;
#pragma unroll
        for (int c = 0; c < VT_FLUX; ++c) v[c] = (R)o[c];
    } else if (a.vt == VT_NORMAL) {
        const TR *o = (const TR *)a.dtr + slot * VT_NORMAL;
#pragma unroll
        for (int c = 0; c < VT_NORMAL; ++c) v[c] = opposite ? -o[c] : o[c];
    } else {
        const TR *o = (const TR *)a.dtr + slot * VT_FLUX;
        v[0] = o[0] * nx + o[1] * ny;
        v[1] = o[1] * nx + o[3] * ny;
        v[2] = o[2] * nx + o[4] * ny;
    }
}

// mu (f, g) of one side of a face node from its viscous flux trace (FP32 form).
template <typename R>
__device__ __forceinline__ void viscous_trace_flux(const R *v, R *f, R *g) {
    f[0] = R(0); f[1] = v[0]; f[2] = v[1]; f[3] = v[2];
    g[0] = R(0); g[1] = v[1]; g[2] = v[3]; g[3] = v[4];
}

// Own Q trace of a face node as the previous stage (or the prolongation) stored it: the values
// the neighbour reads, in the compute type.
template <int P, typename R, typename TR>
__device__ __forceinline__ void stored_trace(const StageArgs &a, int fe, int ff, int fk, R *qs) {
    const TR *o = (const TR *)a.tr_in + ((int64_t)(fe * 4 + ff) * P + fk) * 4;
#pragma unroll
    for (int c = 0; c < 4; ++c) qs[c] = (R)o[c];
}

// mu times this side's viscous flux at a face node from its Q trace and gradient trace
// (ViscousFluxes.f90:39-80, adiabatic walls :279-318), stored at the face node's slot of the traces.
// mdq: where a p-non-conforming face keeps its gradient trace for the mortar kernel (or null).
template <typename R, typename TR>
__device__ __forceinline__ void put_viscous_trace(const StageArgs &a, const Phys<R> &ph, int flags, const R *qs,
                                                  const R *ds, int64_t slot, R nx, R ny, R muf, double *mdq) {
    if (mdq) {
#pragma unroll
        for (int c = 0; c < 8; ++c) mdq[c] = (double)ds[c];
    }
    R fv[4], gv[4];
    if (is_adiabatic(flags)) adiabatic_flux(ph, qs, ds, fv, gv);
    else viscous_flux(ph, qs, ds, fv, gv);
    if (sizeof(R) == 8 && a.vt == VT_NORMAL) {
        TR *o = (TR *)a.dtr_out + slot * VT_NORMAL;
#pragma unroll
        for (int c = 0; c < VT_NORMAL; ++c) o[c] = (TR)(muf * (fv[c + 1] * nx + gv[c + 1] * ny));
    } else {
        TR *o = (TR *)a.dtr_out + slot * VT_FLUX;
        o[0] = (TR)(muf * fv[1]); o[1] = (TR)(muf * fv[2]); o[2] = (TR)(muf * fv[3]);
        o[3] = (TR)(muf * gv[2]); o[4] = (TR)(muf * gv[3]);
    }
}

// This side's viscous flux at a face node from its Q trace qs and the element's nodal gradient
// tile (two Quads arrays, x0 the element's first entry).  The gradient trace is accumulated in FP64 in
// the FP64 form and in FP32 in the FP32 form (lbR: lb in the compute type).
template <int P, int NL, typename R, typename TR, int UNROLL = P>
__device__ __forceinline__ void viscous_face_trace(const StageArgs &a, const Phys<R> &ph, int flags, const R *qs,
                                                   const R *sDQ, int x0, const double *sLb, const R *lbR, int ff,
                                                   int fk, int64_t slot, R nx, R ny, R muf, double *mdq) {
    R ds[8];
    if constexpr (sizeof(R) == 4) {
        face_trace8<P, NL, UNROLL>(sDQ, x0, lbR, ff, fk, ds);
    } else {
        face_trace8<P, NL, UNROLL>(sDQ, x0, sLb, ff, fk, ds);
    }
    put_viscous_trace<R, TR>(a, ph, flags, qs, ds, slot, nx, ny, muf, mdq);
}

// Jacobian times the physical gradient, constant metric.
__device__ __forceinline__ void affine_gradient(const double *dxi, const double *deta, double j11, double j12, double j21,
                                                double j22, double *ds) {
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        ds[c] = dxi[c] * j11 + deta[c] * j12;
        ds[4 + c] = dxi[c] * j21 + deta[c] * j22;
    }
}

// ------------------------------------------------------------------ gradient trace kernel
// Evaluates the element gradient (BR1 or IP), its traces on the element's four faces and, from
// them and the Q traces, this side's viscous flux at every face node, which both elements of
// the face read in their stage kernels.  The gradient at the nodes is not stored: each stage
// kernel recomputes it for its own element.
template <int P, int EPB, bool BR1, typename R>
struct GradSmem {
    using T = Tile<P, EPB>;
    struct Inputs {
        alignas(16) double sQ[sizeof(R) == 4 ? 2 : T::NL * 4];   // FP64 form: the state
        alignas(16) R sQf[sizeof(R) == 4 ? T::NL * 4 : 1];        // FP32 form: the compute-type state
        // the metric; parallelograms, FP64: the faces' Q traces
        alignas(16) R sJa[sizeof(R) == 8 ? (T::NL > T::NF ? T::NL : T::NF) * 4 : BR1 ? T::NL * 4 : 1];
    };
    // the state and the metric are dead once every node's gradient is formed: the gradient
    // tile takes their place
    union {
        Inputs in;
        alignas(16) R sDQ[T::NL * 8];
    } u;
    alignas(16) double sLb[2 * P];
    alignas(16) R sFu[BR1 ? T::NF * br1_width<R>() : 1];
    alignas(16) R sHat[BR1 ? T::PP : 1];
    alignas(16) R sLbw[4 * P];   // lbw, then lb in the compute type
    alignas(16) R sD[BR1 ? 1 : T::PP];
    // parallelograms, FP64: lb M per side (M: hatD or D) and lb lbw of the sides; the face
    // fluxes at the ends of their faces, [(s*4 + f)*2 + end]
    alignas(16) R sLbd[sizeof(R) == 8 ? 2 * P + 4 : 1];
    alignas(16) R sEnd[BR1 && sizeof(R) == 8 ? EPB * 8 * 4 : 1];
};

// gradient_body for parallelograms in FP64, whose metric is constant to rounding.  The physical gradient is then a constant
// combination of the reference derivatives, and so its trace of theirs: along the face from the Q trace,
// across it from the nodes of one line, each P terms.  A BR1 lift enters as the own and the opposite
// face's value at this node and the two adjacent faces' values at this face's corners.  8 P fused
// multiply-adds per variable and face node in place of 2 P (BR1: 4 P) per node and then 2 P per face node.
// Bounded by latency and memory, no longer by LDS: 128 x 128, N = 6 24.6 -> 22.7 us, 61 x 53, N = 10
// 16.6 -> 12.9 us.
template <int P, int EPB, bool BR1, bool XB>
__device__ __forceinline__ void gradient_affine(const StageArgs &a, const int e0, GradSmem<P, EPB, BR1, double> &S) {
    using T = Tile<P, EPB>;
    constexpr int NL = T::NL, NF = T::NF, NE = 8 * EPB;
    // Rolled with the boundary kinds compiled in: unrolled, the interior penalty's kernel takes 96 registers
    // at P = 3, 194 at 8 and 296 at 13 instead of 82 to 90, which cost the form whose gradient runs every
    // stage (artificial viscosity) up to a tenth of a step (80 x 80 elements, N = 6: 144.6 -> 136.0 us a step;
    // 48 x 48, N = 11: 174.2 -> 158.2).
    constexpr int UNROLL = !BR1 && XB ? 1 : P;
    using FaceV = Quads<double, NF>;
    const int t = threadIdx.x, TPB = blockDim.x;
    const Phys<double> ph(a.ph);
    double *sQ = S.u.in.sQ, *sT = S.u.in.sJa, *sFu = S.sFu, *sM = BR1 ? S.sHat : S.sD;
    if (t < 2 * P) {
        S.sLb[t] = a.lb[t];
        S.sLbd[t] = a.lb[(BR1 ? 2 : 4) * P + t];
        if (BR1) S.sLbw[t] = a.lbw[t];
    }
    if (BR1 && t < 4) S.sLbd[2 * P + t] = a.lb[6 * P + t];
    for (int x = t; x < T::PP; x += TPB) sM[x] = (BR1 ? a.hatD : a.D)[(x % P) * P + x / P];
    const int s = t / T::PP, n = t % T::PP;
    if (t < T::NN && e0 + s < a.K) {
        double qg[4];
        load_node(a.Q, (int64_t)e0 * T::PP + t, qg);
        Quads<double, NL>::put(sQ, Layout<P>::at(s, n), qg);
    }
    const int fs = t / (4 * P), ff = (t / P) % 4, fk = t % P, fe = e0 + fs;
    const bool face_active = t < NF && fe < a.K;
    int4 fr = make_int4(0, 0, 0, 0);
    double nx = 0.0, ny = 0.0, qs[4] = {0.0, 0.0, 0.0, 0.0}, j11 = 0.0, j12 = 0.0, j21 = 0.0, j22 = 0.0, ijac = 1.0;
    if (face_active) {
        stored_trace<P, double, double>(a, fe, ff, fk, qs);
        const int fi = (ff & 1) ? (ff == 1 ? P - 1 : 0) : fk, fj = (ff & 1) ? fk : (ff == 2 ? P - 1 : 0);
        load_metric<P, double>(a, fe, fi + P * fj, 0, j11, j12, j21, j22, ijac);   // of the nearest node
        FaceV::put(sT, t, qs);
        double dS, qo[4] = {0.0, 0.0, 0.0, 0.0};
        int64_t nslot;
        load_face<P, double, double>(a, fe, ff, fk, fr, nx, ny, dS, qo, nslot);
        if constexpr (BR1)
            br1_face_flux<NF, double, XB>(a, ph, fr.x, zone_state(a, fr.x, fr.y, (int64_t)(fe * 4 + ff) * P + fk), qs,
                                          qo, nx, ny, dS, sFu, t);
    }
    __syncthreads();
    double ds[8];
    if (face_active) {
        const bool horiz = ff == 0 || ff == 2;
        double qt[4], nd[4], td[4];
        face_trace_slope<P, NL, UNROLL>(sQ, fs * Layout<P>::ES, S.sLb, S.sLbd, ff, fk, qt, nd);
        face_tangent<P, NF, UNROLL>(sT, (fs * 4 + ff) * P, sM, fk, td);
        affine_gradient(horiz ? td : nd, horiz ? nd : td, j11, j12, j21, j22, ds);
    }
    if constexpr (BR1) {
        // by lanes that have no face node, where the tile has enough
        constexpr int NF64 = (NF + 63) / 64 * 64, OFF = NF64 + NE <= T::TPB ? NF64 : NF + NE <= T::TPB ? NF : 0;
        const int x = t - OFF;
        if (x >= 0 && x < NE && e0 + x / 8 < a.K) {
            const double *lb = S.sLb + (x & 1) * P, *F = sFu + (x >> 1) * P * 6;
            double v[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int l = 0; l < P; ++l)
#pragma unroll
                for (int c = 0; c < 4; ++c) v[c] = fma(F[l * 6 + c], lb[l], v[c]);
            Quads<double, NE>::put(S.sEnd, x, v);
        }
        __syncthreads();
        if (face_active) {
#pragma unroll
            for (int c = 0; c < 8; ++c) ds[c] = -ds[c];
            const int side = (ff == 0 || ff == 3) ? 0 : 1;
#pragma unroll
            for (int o = 0; o < 4; ++o) {
                // the own face, the opposite one, the adjacent ones at their sides 0 and 1
                const int gf = o < 2 ? (ff ^ (2 * o)) : (ff & 1) ? (o == 2 ? 0 : 2) : (o == 2 ? 3 : 1);
                const double lw = o < 2 ? S.sLbd[2 * P + 2 * side + (side ^ o)] : S.sLbw[(o - 2) * P + fk];
                const int xf = (fs * 4 + gf) * P;
                double F[4];
                if (o < 2) {
#pragma unroll
                    for (int c = 0; c < 4; ++c) F[c] = sFu[(xf + fk) * 6 + c];
                } else {
                    Quads<double, NE>::get(S.sEnd, (fs * 4 + gf) * 2 + side, F);
                }
                const double wx = sFu[xf * 6 + 4] * lw, wy = sFu[xf * 6 + 5] * lw;
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    ds[c] += F[c] * wx;
                    ds[4 + c] += F[c] * wy;
                }
            }
        }
    }
    if (face_active) {
#pragma unroll
        for (int c = 0; c < 8; ++c) ds[c] *= ijac;
        const double muf = XB ? face_mu<double>(a, ph, fe, fr) : ph.mu;
        const int64_t slot = (int64_t)(fe * 4 + ff) * P + fk;
        double *mdq = ((fr.x & 15) == FK_MORTAR && a.mdq) ? a.mdq + slot * 8 : nullptr;
        put_viscous_trace<double, double>(a, ph, fr.x, qs, ds, slot, nx, ny, muf, mdq);
    }
}

// One element tile [e0, e0+EPB) of the gradient; any workgroup size >= Tile<P, EPB>::TPB.
// XB: the Euler-wall, Dirichlet and pressure boundary kinds are compiled in.
template <int P, int EPB, bool BR1, typename R, typename TR, bool XB = false>
__device__ __forceinline__ void gradient_body(const StageArgs &a, const int e0, GradSmem<P, EPB, BR1, R> &S) {
    using T = Tile<P, EPB>;
    constexpr int PP = T::PP, NN = T::NN, NF = T::NF;
    const int TPB = blockDim.x;
    if constexpr (sizeof(R) == 8) {
        if (a.affine) {
            gradient_affine<P, EPB, BR1, XB>(a, e0, S);
            return;
        }
    }
    double *sQ = S.u.in.sQ, *sLb = S.sLb;
    R *sDQ = S.u.sDQ, *sJa = S.u.in.sJa, *sFu = S.sFu, *sHat = S.sHat, *sLbw = S.sLbw, *sD = S.sD;
    const int t = threadIdx.x;
    const Phys<R> ph(a.ph);
    if (t < 2 * P) { sLb[t] = a.lb[t]; sLbw[t] = (R)a.lbw[t]; sLbw[2 * P + t] = (R)a.lb[t]; }
    for (int x = t; x < PP; x += TPB) {
        if (BR1) sHat[x] = (R)a.hatD[(x % P) * P + x / P];
        else sD[x] = (R)a.D[(x % P) * P + x / P];
    }
    const int64_t nb0 = (int64_t)e0 * PP;
    constexpr bool COPY = sizeof(R) == 4;
    constexpr int NL = T::NL;
    const R *sQr;
    if constexpr (COPY) sQr = S.u.in.sQf; else sQr = (const R *)sQ;
    // ---- hoisted global loads
    const int s = t / PP, n = t % PP, e = e0 + s, x0 = s * Layout<P>::ES, xn = Layout<P>::at(s, n);
    const bool node_active = (t < NN) && (e < a.K);
    R ijac = R(1), j11 = R(0), j12 = R(0), j21 = R(0), j22 = R(0);
    int ord = 0;
    if (node_active) {
        const int64_t g = nb0 + s * PP + n;
        double qg[4];
        load_node(a.Q, g, qg);
        load_metric<P, R>(a, e, n, g, j11, j12, j21, j22, ijac);
        if constexpr (COPY) put_slots<NL, R>(a.ph, S.u.in.sQf, xn, qg);
        else Quads<double, NL>::put(sQ, xn, qg);
        if (BR1) {
            ord = a.forder[e];
            const R jv[4] = {j11, j21, j12, j22};
            Quads<R, NL>::put(sJa, xn, jv);
        }
    }
    const int fs = t / (4 * P), ff = (t / P) % 4, fk = t % P, fe = e0 + fs;
    const bool face_active = (t < NF) && (fe < a.K);
    int4 fr = make_int4(0, 0, 0, 0);
    R nx = R(0), ny = R(0), dS = R(0), qo[4] = {R(0), R(0), R(0), R(0)};
    int64_t nslot = 0;
    R qs[4] = {R(0), R(0), R(0), R(0)};
    if (face_active) {
        load_face<P, R, TR>(a, fe, ff, fk, fr, nx, ny, dS, qo, nslot);
        stored_trace<P, R, TR>(a, fe, ff, fk, qs);
    }
    if (BR1 && face_active)
        br1_face_flux<NF, R, XB>(a, ph, fr.x, zone_state(a, fr.x, fr.y, (int64_t)(fe * 4 + ff) * P + fk), qs, qo, nx,
                                 ny, dS, sFu, t);
    __syncthreads();
    R dq[8];
    if (node_active) {
        const int i = n % P, j = n / P;
        if (BR1) {
            br1_node_gradient<P, NL, NF, R>(sQr, sJa, x0, sHat, sFu, s * 4 * P, sLbw, ord, i, j, ijac, dq);
            if (ord >> 8) mortar_y_lift<P, R>(a.mustar + (int64_t)e * 4 * P * 8, sLbw, ord, i, j, ijac, dq);
        }
        else ip_node_gradient<P, NL, R>(sQr, x0, sD, i, j, j11, j12, j21, j22, ijac, dq);
    }
    __syncthreads();   // every lane is done with the state and the metric
    if (node_active) {
        Quads<R, NL>::put(sDQ, xn, dq);
        Quads<R, NL>::put(sDQ + 4 * NL, xn, dq + 4);
    }
    __syncthreads();
    if (face_active) {
        const R muf = XB ? face_mu<R>(a, ph, fe, fr) : ph.mu;
        const int64_t slot = (int64_t)(fe * 4 + ff) * P + fk;
        double *mdq = ((fr.x & 15) == FK_MORTAR && a.mdq) ? a.mdq + slot * 8 : nullptr;
        viscous_face_trace<P, NL, R, TR>(a, ph, fr.x, qs, sDQ, fs * Layout<P>::ES, sLb, sLbw + 2 * P, ff, fk, slot, nx,
                                         ny, muf, mdq);
    }
}

template <int P, int EPB, bool BR1, typename R, typename TR, bool XB = false>
__global__ __launch_bounds__((Tile<P, EPB>::TPB)) void k_gradient(StageArgs a) {
    __shared__ GradSmem<P, EPB, BR1, R> S;
    gradient_body<P, EPB, BR1, R, TR, XB>(a, xcd_tile(blockIdx.x, gridDim.x) * EPB, S);
}

// ------------------------------------------------------------------ the stage kernel
template <int P, int EPB, bool NS, bool IP, typename R>
struct StageSmem {
    using T = Tile<P, EPB>;
    alignas(16) double sQ[T::NL * 4];
    alignas(16) double sLb[2 * P];
    struct Fluxes {
        alignas(16) R sCF[T::NL * 4];          // BR1: the metric Ja during the gradient phase
        alignas(16) R sCG[T::NL * 4];          // NS, FP32: the compute-type state until the node phase
    };
    // IP: the epilogue's gradient tile takes the place of the contravariant fluxes
    union {
        Fluxes f;
        alignas(16) R sDQ[IP ? T::NL * 8 : 1];
    } u;
    // the face fluxes (BR1: uStar fluxes during the gradient phase); once every wavefront has
    // lifted them, the residual maxima
    union {
        alignas(16) R sF[NS && !IP ? T::NF * br1_width<R>() : T::NF * 4];
        uint64_t sRes[4][4];
    };
    // IP gradient-face terms.  FP32: the face phase's contravariant fluxes, then (same arrays) the
    // U / V lift coefficients.  FP64: the flux along the face in sU, then V there, while U, whose
    // weight is the face flux's, is added to sF: the fifth of the LDS this saves lets four workgroups
    // instead of three share a CU (P = 4 to 7; 101 x 77, N = 5: 28.5 -> 25.6 us a stage).
    alignas(16) R sU[IP ? T::NF * 4 : NS ? 1 : 0];
    alignas(16) R sV[IP && sizeof(R) == 4 ? T::NF * 4 : NS ? 1 : 0];
    alignas(16) R sHat[T::PP];          // transposed, as sD: a wavefront's reads are consecutive
    alignas(16) R sD[NS ? T::PP : 0];   // IP gradient; BR1: the Laplacian dissipation's interior gradient
    // Euler in FP64 reads lbw from memory and holds nothing it does not need: LDS is allocated in 1280
    // bytes, and at P = 6 to 8 it is at 25 of these that five workgroups share a CU's 160 KB (64 cases
    // of N = 3 to 8 in one launch: 3197 -> 2758 us a step; 128 x 128, N = 7: 38.4 -> 37.3 us a stage)
    // lbw; IP in FP32: lb (epilogue) behind it
    alignas(16) R sLbw[IP && sizeof(R) == 4 ? 4 * P : NS || sizeof(R) == 4 ? 2 * P : 0];
    alignas(16) R sDlbw[NS ? 2 * P : 0];
};

// Wavefronts per SIMD the stage kernel's register allocation has to leave room for: in FP64, as many as
// the wide tiles' LDS allows, four of the Navier-Stokes form with one solver and five of the Euler form.
// Some kernels meet that with scratch: 12 to 20 bytes a lane of Euler at P = 5 and 7 and of the batch
// kernels over all orders (the wavefront is worth more: 64 cases of N = 3 to 8 in one launch, with the
// LDS that goes with it, 3197 -> 2758 us a step), 8 to 20 of interior penalty at P = 7 and 11, 136 of the
// narrow tile of P = 4 with Lax-Friedrichs.
// The exact solver takes 141 registers of BR1 and 173 of interior penalty: three wavefronts (168), or
// four with 60 to 160 bytes of scratch a lane, which pay from P = 5 and 8 on (2 M nodes, us a step at three
// and four: BR1 P = 4 694 and 710, P = 10 618 and 573; interior penalty P = 3 971 and 1026, P = 4 672 and
// 704, P = 9 694 and 678, P = 12 751 and 714).  With the boundary kinds, and with the solver chosen at
// run time, interior penalty takes 172 where three wavefronts leave 168 (P = 4 946 -> 715, P = 12 1258 ->
// 763).  Euler: the 129 registers with the boundary kinds to 128 (P = 10 455 -> 410), FP32's 74 to 72
// (P = 12 335 -> 321) but at P = 8, where the two that spill cost more (301 and 308).
constexpr int stage_waves(bool ns, bool ip, int rs, bool xbf, bool fp64, int P) {
    if (rs == 2 && !ns) return fp64 ? 4 : P == 8 ? 1 : 7;
    if (rs == 2 && fp64) return xbf || P < (ip ? 8 : 5) ? 3 : 4;
    if (rs < 0 && fp64 && ip) return 3;
    return !fp64 || rs < 0 || rs == 2 || xbf ? 1 : ns ? 4 : 5;
}

// One element tile [e0, e0+EPB) of a stage; any workgroup size >= Tile<P, EPB>::TPB (at most
// 256).  rslot is the residual partial this tile writes; cq, cg are the stage's RK factors.
// Navier-Stokes: the element's nodal gradient is recomputed here from the LDS tile and the Q
// traces (it stays in registers); the viscous fluxes of both sides of a face are read from
// what the gradient kernel stored.  The own Q traces are read from the stored traces as well.
// Interior penalty: the gradient is element-local, so the RK update's epilogue also forms the
// next stage's viscous face-flux traces from the updated tile (the work of k_gradient, with
// the same device functions and the same bits), and no gradient kernel runs between stages.
// XBF: the Euler-wall, Dirichlet and pressure boundary kinds and artificial dissipation are
// compiled in (always with the run-time solver choice, RS = -1).
template <int P, int EPB, bool NS, bool IP, int RS, typename R, typename TR, bool XBF = false>
__device__ __forceinline__ void stage_body(const StageArgs &a, const int e0, const int64_t rslot, const double cq,
                                           const double cg, StageSmem<P, EPB, NS, IP, R> &S) {
    using T = Tile<P, EPB>;
    constexpr bool XB = RS < 0 || XBF;
    constexpr int PP = T::PP, NN = T::NN, NF = T::NF;
    constexpr bool BR1 = NS && !IP;
    // The contraction and trace loops, whose sums are the same either way.  Unrolled, their LDS reads
    // overlap (2 to 5 % of a step at every order); the kernels with every solver or boundary kind
    // compiled in, and FP32 interior penalty, are where the registers this takes cost a wavefront per SIMD
    // (256 x 256, N = 7, mixed: 78 registers and 543 us a step at 2, 81 and 575 us unrolled).
    constexpr int UNROLL = (XB || RS == 2) ? 1 : (IP && sizeof(R) == 4) ? 2 : P;
    constexpr bool LBW_MEM = !NS && sizeof(R) == 8;
    const int TPB = blockDim.x;
    double *sQ = S.sQ, *sLb = S.sLb;
    R *sCF = S.u.f.sCF, *sCG = S.u.f.sCG, *sF = S.sF, *sU = S.sU, *sV = S.sV;
    R *sHat = S.sHat, *sD = S.sD, *sLbw = S.sLbw, *sDlbw = S.sDlbw;
    const int t = threadIdx.x;
    const Phys<R> ph(a.ph);
    const bool ipgrad = IP && a.ph.ip_gradflux;
    const bool affine = NS && sizeof(R) == 8 && a.affine;   // constant metric
    if (a.resid_max && !a.do_resid && e0 == 0 && t < 4) a.resid_max[t * kResidStride] = 0.0;
    if (t < 2 * P) {
        sLb[t] = a.lb[t];
        if (!LBW_MEM) sLbw[t] = (R)a.lbw[t];
        if (NS) sDlbw[t] = (R)a.dlbw[t];
        if (IP && sizeof(R) == 4) sLbw[2 * P + t] = (R)a.lb[t];
    }
    for (int x = t; x < PP; x += TPB) {
        const int xt = (x % P) * P + x / P;
        sHat[x] = (R)a.hatD[xt];
        if (IP || (BR1 && XB)) sD[x] = (R)a.D[xt];
    }
    const int64_t nb0 = (int64_t)e0 * PP;
    // NS in FP32: a compute-type copy of the state for the gradient contractions, in sCG (each
    // node lane reads its own entry once more before the node phase overwrites it)
    constexpr bool COPY = NS && sizeof(R) == 4;
    constexpr int NL = T::NL;
    using NodeV = Quads<R, NL>;    // node arrays
    using FaceV = Quads<R, NF>;    // face-node arrays
    const R *sQr;
    if constexpr (COPY) sQr = sCG; else sQr = (const R *)sQ;

    // ---- hoisted global loads: node lane
    const int s = t / PP, n = t % PP, e = e0 + s, x0 = s * Layout<P>::ES, xn = Layout<P>::at(s, n);
    const bool node_active = (t < NN) && (e < a.K);
    const int64_t g = nb0 + s * PP + n;
    R j11 = R(0), j12 = R(0), j21 = R(0), j22 = R(0), ijac = R(1);
    int ord = 0;
    // the own node's state: staged in LDS for the gradient contractions (Navier-Stokes) and for
    // the update; the Euler form takes its flux from the registers, so nothing there waits for
    // another lane until the fluxes are formed
    double qg[4];
    if (node_active) {
        load_node(a.Q, g, qg);
        load_metric<P, R>(a, e, n, g, j11, j12, j21, j22, ijac);
        ord = a.forder[e];
        Quads<double, NL>::put(sQ, xn, qg);
        if constexpr (COPY) put_slots<NL, R>(a.ph, sCG, xn, qg);
        if (BR1 && !affine) {
            const R jv[4] = {j11, j21, j12, j22};
            NodeV::put(sCF, xn, jv);
        }
    }
    // ---- hoisted global loads: face lane
    const int fs = t / (4 * P), ff = (t / P) % 4, fk = t % P, fe = e0 + fs;
    const bool face_active = (t < NF) && (fe < a.K);
    int4 fr = make_int4(0, 0, 0, 0);
    R nx = R(0), ny = R(0), dS = R(0), qo[4] = {R(0), R(0), R(0), R(0)};
    int64_t nslot = 0;
    R qs[4] = {R(0), R(0), R(0), R(0)};
    if (face_active) {
        load_face<P, R, TR>(a, fe, ff, fk, fr, nx, ny, dS, qo, nslot);
        stored_trace<P, R, TR>(a, fe, ff, fk, qs);
    }
    if (BR1 && face_active)
        br1_face_flux<NF, R, XB>(a, ph, fr.x, zone_state(a, fr.x, fr.y, (int64_t)(fe * 4 + ff) * P + fk), qs, qo, nx,
                                 ny, dS, sF, t);
    if (NS) __syncthreads();

    // ---- own nodal gradient (Navier-Stokes), kept in registers for the node phase
    R dq[NS ? 8 : 1];
    // BR1 with the Laplacian dissipation: the element's interior gradient as well (its volume
    // flux, DGArtificialDissipation.f90:207-222); interior penalty: that is dq itself
    constexpr bool LAPG = BR1 && XB;
    R dqi[LAPG ? 8 : 1];
    if (NS && node_active) {
        const int i = n % P, j = n / P;
        if (BR1) {
            br1_node_gradient<P, NL, NF, R, UNROLL>(sQr, sCF, x0, sHat, sF, s * 4 * P, sLbw, ord, i, j, ijac, dq, affine,
                                                    j11, j12, j21, j22);
            if (ord >> 8) mortar_y_lift<P, R>(a.mustar + (int64_t)e * 4 * P * 8, sLbw, ord, i, j, ijac, dq);
        }
        else ip_node_gradient<P, NL, R, UNROLL>(sQr, x0, sD, i, j, j11, j12, j21, j22, ijac, dq);
        if (LAPG && a.lap) ip_node_gradient<P, NL, R, UNROLL>(sQr, x0, sD, i, j, j11, j12, j21, j22, ijac, dqi);
    }
    // the neighbour's viscous flux trace, issued before the barrier and consumed in the face phase
    constexpr int VW = NS ? vis_width<R>() : 1;
    R vn[VW];
    R invh = R(0);
    if (NS && face_active) {
        if ((fr.x & 15) <= FK_PERIODIC) {
            load_viscous_trace<R, TR>(a, nslot, nx, ny, (fr.x & 15) == FK_PERIODIC, vn);
            if (XB && a.mu_a && (fr.x & 15) == FK_PERIODIC) {
                // a periodic face is a boundary edge of each side, whose viscosity (its own
                // element's mu_a) both sides' fluxes take; the partner stored its trace with its own
                const double ms = a.ph.mu + a.mu_a[fe], mp = a.ph.mu + a.mu_a[fr.y >> 2];
                const R sc = (R)(ms / mp);
#pragma unroll
                for (int c = 0; c < VW; ++c) vn[c] = vn[c] * sc;
            }
        }
        if (IP) invh = (R)a.einvh[fr.w];
    }
    // the node phase overwrites sCF (the metric, BR1) and sCG (the FP32 state copy)
    if (BR1 || COPY) __syncthreads();

    // ---- node phase: contravariant fluxes (DGSpatial_QDotVolumeLoop, DGWeakIntegrals.f90:111-171)
    if (node_active) {
        R q[4], f[4], gg[4];
        if constexpr (COPY) {
            NodeV::get(sQr, xn, q);
        } else {
            if (NS) Quads<double, NL>::get(sQ, xn, qg);
#pragma unroll
            for (int c = 0; c < 4; ++c) q[c] = qslot<R>(a.ph, qg[c], c);
        }
        inviscid_flux(ph, q, f, gg);
        if (NS) {
            R fv[4], gv[4];
            viscous_flux(ph, q, dq, fv, gv);
            // e % mu_a (DGViscous_BR1.f90:307, DGViscous_IP.f90:84)
            const R mue = (XB && a.mu_a) ? (R)(a.ph.mu + a.mu_a[e]) : ph.mu;
            // Laplacian dissipation: F = Fi - Fv - Fa, Fa = mu_e times the interior gradient
            R fa[4] = {R(0), R(0), R(0), R(0)}, ga[4] = {R(0), R(0), R(0), R(0)};
            if (XB && a.lap) {
                const R lm = (R)a.lap[e];
                const R *di = LAPG ? dqi : dq;
#pragma unroll
                for (int c = 0; c < 4; ++c) { fa[c] = lm * di[c]; ga[c] = lm * di[4 + c]; }
            }
#pragma unroll
            for (int c = 0; c < 4; ++c) { f[c] = (f[c] - mue * fv[c]) - fa[c]; gg[c] = (gg[c] - mue * gv[c]) - ga[c]; }
        }
        R cf[4], cg4[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            cf[c] = f[c] * j11 + gg[c] * j21;
            cg4[c] = f[c] * j12 + gg[c] * j22;
        }
        NodeV::put(sCF, xn, cf);
        NodeV::put(sCG, xn, cg4);
    }

    // ---- face phase: Riemann fluxes of the element's own four faces
    constexpr bool FOLD = IP && sizeof(R) == 8;
    R vown[FOLD ? 4 : 1];   // FP64: V of the own face node
    auto put_gradient_flux = [&](const R *fc, const R *gc) {
        if constexpr (FOLD) {
            const bool horiz = ff == 0 || ff == 2;
            R along[4];
#pragma unroll
            for (int c = 0; c < 4; ++c) { along[c] = horiz ? fc[c] : gc[c]; vown[c] = horiz ? gc[c] : fc[c]; }
            FaceV::put(sU, t, along);
        } else {
            FaceV::put(sU, t, fc);
            FaceV::put(sV, t, gc);
        }
    };
    if (face_active) {
        const int kind = fr.x & 15;
        if (kind == FK_MORTAR) {
            // p-non-conforming edge: (Fi - Fv) dS projected to this side by the mortar kernel
            const double *mf = a.mflux + ((int64_t)(fe * 4 + ff) * P + fk) * 4;
            const R F[4] = {(R)mf[0], (R)mf[1], (R)mf[2], (R)mf[3]};
            FaceV::put(sF, t, F);
            if (ipgrad) {
                // this side's IP gradient flux, projected and times dS by the mortar kernel, in
                // contravariant components (DGWeakIntegrals.f90:268-495)
                const double *mg = a.mgrad + ((int64_t)(fe * 4 + ff) * P + fk) * 8;
                const R *fm = (const R *)a.fmet + ((int64_t)(fe * 4 + ff) * P + fk) * 5;
                R fc[4], gc[4];
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    const R gx = (R)mg[c], gy = (R)mg[4 + c];
                    fc[c] = (gx * fm[0] + gy * fm[1]) * fm[4];
                    gc[c] = (gx * fm[2] + gy * fm[3]) * fm[4];
                }
                put_gradient_flux(fc, gc);
            }
        } else {
            R vs[VW];   // own viscous flux trace
            if (NS) load_viscous_trace<R, TR>(a, (int64_t)(fe * 4 + ff) * P + fk, nx, ny, false, vs);
            int rs = a.ph.riemann;
            R uSB[4] = {R(0), R(0), R(0), R(0)};
            int neumann = 0, prescribed = 0;
            if (kind > FK_PERIODIC) {
                prescribed = ghost_state<R, XB>(kind, fr.x, zone_state(a, fr.x, fr.y, (int64_t)(fe * 4 + ff) * P + fk),
                                                a.ph, ph, qs, nx, ny, qo, uSB, neumann);
                const int zr = (fr.x >> FF_RS_SHIFT) & 15;
                if (zr) rs = zr - 1;
            }
            R Fi[4];
            if (XB && prescribed) {
                // WEAK_PRESCRIBED (DGSpatialDiscretizationMethods.f90:1194-1198): the inviscid
                // normal flux of the boundary's state
                R fp[4], gp[4];
                inviscid_flux(ph, qo, fp, gp);
#pragma unroll
                for (int c = 0; c < 4; ++c) Fi[c] = fp[c] * nx + gp[c] * ny;
            } else if (kind == FK_INT_R) riemann<RS, R>(rs, ph, qo, qs, nx, ny, Fi);
            else riemann<RS, R>(rs, ph, qs, qo, nx, ny, Fi);
            R F[4];
            if (!NS) {
#pragma unroll
                for (int c = 0; c < 4; ++c) F[c] = Fi[c] * dS;
            } else {
                R Fv[4] = {R(0), R(0), R(0), R(0)};
                R Fa[4] = {R(0), R(0), R(0), R(0)};   // Laplacian dissipation: -mu Area (QL - QR)
                R G8[8] = {R(0), R(0), R(0), R(0), R(0), R(0), R(0), R(0)};
                const R muf = XB ? face_mu<R>(a, ph, fe, fr) : ph.mu;
                const R lapA = (XB && a.lap) ? (R)(face_lap(a, fe, fr) * a.earea[fr.w]) : R(0);
                const R pen = IP ? ph.sigma0 * muf * (R)(P - 1) * (R)(P - 1) * invh : R(0);
                if (kind <= FK_PERIODIC) {
                    const R *uL = (kind == FK_INT_R) ? qo : qs, *uR = (kind == FK_INT_R) ? qs : qo;
                    if constexpr (sizeof(R) == 8) {
#pragma unroll
                        for (int c = 0; c < VW; ++c) Fv[c + 1] = R(0.5) * (vs[c] + vn[c]);
                    } else {
                        const R *vL = (kind == FK_INT_R) ? vn : vs, *vR = (kind == FK_INT_R) ? vs : vn;
                        R fL[4], gL[4], fR[4], gR[4];
                        viscous_trace_flux(vL, fL, gL);
                        viscous_trace_flux(vR, fR, gR);
#pragma unroll
                        for (int c = 0; c < 4; ++c) {
                            R acc = R(0);
                            acc = acc + R(0.5) * (fL[c] + fR[c]) * nx;
                            acc = acc + R(0.5) * (gL[c] + gR[c]) * ny;
                            Fv[c] = acc;
                        }
                    }
                    if (IP) {
#pragma unroll
                        for (int c = 0; c < 4; ++c) Fv[c] = Fv[c] - pen * (uL[c] - uR[c]);
                    }
                    if (XB && a.lap) {
#pragma unroll
                        for (int c = 0; c < 4; ++c) Fa[c] = -(lapA * (uL[c] - uR[c]));
                    }
                    if (ipgrad) {
                        // IP_GradientRiemannSolver (DGViscous_IP.f90:216-249): this side's share
                        R fgr[8], f4[4], g4[4];
#pragma unroll
                        for (int c = 0; c < 4; ++c) { fgr[c] = (uL[c] - uR[c]) * nx; fgr[4 + c] = (uL[c] - uR[c]) * ny; }
                        const R *own = (kind == FK_INT_R) ? uR : uL;
                        viscous_flux(ph, own, fgr, f4, g4);
                        const R cf = (kind == FK_INT_R ? -R(0.5) : R(0.5)) * ph.ip_eps * muf;
#pragma unroll
                        for (int c = 0; c < 4; ++c) { G8[c] = cf * f4[c] * dS; G8[4 + c] = cf * g4[c] * dS; }
                    }
                } else if (!neumann) {
                    const bool adiab = is_adiabatic(fr.x);
                    // adiabatic or not, as the gradient kernel chose
                    if constexpr (sizeof(R) == 8) {
#pragma unroll
                        for (int c = 0; c < VW; ++c) Fv[c + 1] = vs[c];
                    } else {
                        R fv4[4], gv4[4];
                        viscous_trace_flux(vs, fv4, gv4);
#pragma unroll
                        for (int c = 0; c < 4; ++c) {
                            R acc = R(0);
                            acc = acc + fv4[c] * nx;
                            acc = acc + gv4[c] * ny;
                            Fv[c] = acc;
                        }
                    }
                    if (IP) {
#pragma unroll
                        for (int c = 0; c < 4; ++c) Fv[c] = Fv[c] - pen * (qs[c] - uSB[c]);
                    }
                    if (XB && a.lap) {
#pragma unroll
                        for (int c = 0; c < 4; ++c) Fa[c] = -(lapA * (qs[c] - uSB[c]));
                    }
                    if (ipgrad) {
                        R fgr[8], f4[4], g4[4];
#pragma unroll
                        for (int c = 0; c < 4; ++c) { fgr[c] = (qs[c] - uSB[c]) * nx; fgr[4 + c] = (qs[c] - uSB[c]) * ny; }
                        if (adiab) adiabatic_flux(ph, qs, fgr, f4, g4);
                        else viscous_flux(ph, qs, fgr, f4, g4);
                        const R cf = ph.ip_eps * muf;
#pragma unroll
                        for (int c = 0; c < 4; ++c) { G8[c] = cf * f4[c] * dS; G8[4 + c] = cf * g4[c] * dS; }
                    }
                }
                if (kind <= FK_INT_R) {
#pragma unroll
                    for (int c = 0; c < 4; ++c) F[c] = ((Fi[c] - Fv[c]) - Fa[c]) * dS;
                } else {
#pragma unroll
                    for (int c = 0; c < 4; ++c) F[c] = ((Fi[c] * dS - Fv[c] * dS) - Fa[c] * dS);
                }
                if (ipgrad) {
                    // contravariant gradient-flux components at the face (DGWeakIntegrals.f90:268-495)
                    const R *fm = (const R *)a.fmet + ((int64_t)(fe * 4 + ff) * P + fk) * 5;
                    R fc[4], gc[4];
#pragma unroll
                    for (int c = 0; c < 4; ++c) {
                        fc[c] = (G8[c] * fm[0] + G8[4 + c] * fm[1]) * fm[4];   // fm[4] = 1/jac at the face node
                        gc[c] = (G8[c] * fm[2] + G8[4 + c] * fm[3]) * fm[4];
                    }
                    put_gradient_flux(fc, gc);
                }
            }
            if (kind == FK_INT_R) {
#pragma unroll
                for (int c = 0; c < 4; ++c) F[c] = -F[c];
            }
            FaceV::put(sF, t, F);
        }
    }
    __syncthreads();

    // ---- IP gradient face terms: U (lbw coefficient) and V (dlbw coefficient) per face node;
    // horizontal faces: U = hatD . Fc, V = Gc ; vertical faces: U = hatD . Gc, V = Fc
    if (ipgrad) {
        R u2[4], v2[4];
        if (face_active) {
            const bool horiz = (ff == 0 || ff == 2);
            const R *src = FOLD || horiz ? sU : sV;
            const int xf = (fs * 4 + ff) * P;
#pragma unroll
            for (int c = 0; c < 4; ++c) u2[c] = R(0);
#pragma unroll
            for (int l = 0; l < P; ++l) {
                const R h = sHat[l * P + fk];
                R v[4];
                FaceV::get(src, xf + l, v);
#pragma unroll
                for (int c = 0; c < 4; ++c) u2[c] += h * v[c];
            }
            if constexpr (FOLD) {
                FaceV::get(sF, t, v2);
#pragma unroll
                for (int c = 0; c < 4; ++c) u2[c] += v2[c];
            } else {
                FaceV::get(horiz ? sV : sU, xf + fk, v2);
            }
        }
        __syncthreads();   // every face has read its fluxes: U and V take their place
        if (face_active) {
            FaceV::put(FOLD ? sF : sU, t, u2);
            FaceV::put(FOLD ? sU : sV, t, FOLD ? vown : v2);
        }
        __syncthreads();
    }

    // ---- node phase 2: volume contraction, ordered face lifts, /jac, RK update
    double qd[4] = {0.0, 0.0, 0.0, 0.0};
    double gold[4] = {0.0, 0.0, 0.0, 0.0};
    if (node_active && a.mode == 0 && !a.first_stage) {
        const double2 *gp = (const double2 *)(a.G + g * 4);
        const double2 g01 = gp[0], g23 = gp[1];
        gold[0] = g01.x; gold[1] = g01.y; gold[2] = g23.x; gold[3] = g23.y;
    }
    if (node_active) {
        const int i = n % P, j = n / P;
        R acc[4] = {R(0), R(0), R(0), R(0)};
#pragma unroll UNROLL
        for (int l = 0; l < P; ++l) {
            const R hi = sHat[l * P + i], hj = sHat[l * P + j];
            R cF[4], cG[4];
            NodeV::get(sCF, x0 + l + Layout<P>::RS * j, cF);
            NodeV::get(sCG, x0 + i + Layout<P>::RS * l, cG);
#pragma unroll
            for (int c = 0; c < 4; ++c) acc[c] = acc[c] + hi * cF[c] + hj * cG[c];
        }
#pragma unroll
        for (int o = 0; o < 4; ++o) {
            const int f = (ord >> (2 * o)) & 3;
            const int idx = (f == 0 || f == 2) ? i : j;
            const int oth = (f == 0 || f == 2) ? j : i;
            const int side = (f == 0 || f == 3) ? 0 : P;
            const R lw = LBW_MEM ? (R)a.lbw[side + oth] : sLbw[side + oth];
            const int xf = (s * 4 + f) * P + idx;
            R Ff[4];
            FaceV::get(sF, xf, Ff);
#pragma unroll
            for (int c = 0; c < 4; ++c) acc[c] = acc[c] - Ff[c] * lw;
            if (FOLD && ipgrad) {
                const R dlw = sDlbw[side + oth];
                R Vf[4];
                FaceV::get(sU, xf, Vf);
#pragma unroll
                for (int c = 0; c < 4; ++c) acc[c] = acc[c] - Vf[c] * dlw;
            } else if (ipgrad) {
                const R dlw = sDlbw[side + oth];
                R Uf[4], Vf[4];
                FaceV::get(sU, xf, Uf);
                FaceV::get(sV, xf, Vf);
#pragma unroll
                for (int c = 0; c < 4; ++c) acc[c] = acc[c] - (Uf[c] * lw + Vf[c] * dlw);
            }
        }
#pragma unroll
        for (int c = 0; c < 4; ++c) qd[c] = (double)(acc[c] * ijac);   // QDot / jac
        if (a.mode == 1) {
            double2 *o = (double2 *)(a.QDot + g * 4);
            o[0] = make_double2(qd[0], qd[1]);
            o[1] = make_double2(qd[2], qd[3]);
        } else {
            double gv[4];
            if (a.first_stage) {
#pragma unroll
                for (int c = 0; c < 4; ++c) gv[c] = cq * qd[c];
            } else {
#pragma unroll
                for (int c = 0; c < 4; ++c) gv[c] = fma(a.am, gold[c], cq * qd[c]);
            }
            // the last stage's register is read by nobody: the next step's first stage starts it anew
            if (!a.do_resid) {
                double2 *go = (double2 *)(a.G + g * 4);
                go[0] = make_double2(gv[0], gv[1]);
                go[1] = make_double2(gv[2], gv[3]);
            }
            double qn[4];
            Quads<double, NL>::get(sQ, xn, qn);
#pragma unroll
            for (int c = 0; c < 4; ++c) qn[c] = fma(cg, gv[c], qn[c]);
            double2 *qo2 = (double2 *)(a.Q + g * 4);
            qo2[0] = make_double2(qn[0], qn[1]);
            qo2[1] = make_double2(qn[2], qn[3]);
            Quads<double, NL>::put(sQ, xn, qn);
        }
    }
    __syncthreads();
    // max|QDot| per equation: across the wavefront, then across the workgroup's wavefronts; one
    // partial per workgroup (reduced by k_resid_final), or one atomic maximum
    if (a.do_resid) {
        const uint64_t m = wave_max4(qd);   // zeros where the lane has no node
        if ((t & 63) < 4) S.sRes[t >> 6][t & 3] = m;
        __syncthreads();
    }
    if (a.do_resid && t < 4) {
        uint64_t v = S.sRes[0][t];
        for (int w = 1; w < TPB / 64; ++w) v = max(v, S.sRes[w][t]);
        const int c = wave_max4_value(t);
        // few workgroups: straight into the handle's four maxima, cleared by the step's first stage
        if (a.resid_max) atomicMax((unsigned long long *)(a.resid_max + c * kResidStride), (unsigned long long)v);
        else a.resid_part[rslot * 4 + c] = __longlong_as_double((long long)v);
    }
    if (a.mode == 0) {
        R qn[4];   // the next stage's own Q trace in the compute type (IP epilogue)
        constexpr bool SLOPE = IP && sizeof(R) == 8;
        double nd[4] = {0.0, 0.0, 0.0, 0.0};
        if (face_active) {
            double tq[4];
            if (SLOPE && affine)
                face_trace_slope<P, NL, UNROLL>(sQ, fs * Layout<P>::ES, sLb, a.lb + 4 * P, ff, fk, tq, nd);
            else face_trace<P, NL, UNROLL>(sQ, fs * Layout<P>::ES, sLb, ff, fk, tq);
            tq[3] = slot_energy<TR>(a.ph, tq[3]);
            TR *o = (TR *)a.tr_out + ((int64_t)(fe * 4 + ff) * P + fk) * 4;
#pragma unroll
            for (int c = 0; c < 4; ++c) o[c] = (TR)tq[c];
#pragma unroll
            for (int c = 0; c < 4; ++c) qn[c] = (R)(TR)tq[c];
        }
        if constexpr (IP) {
          if constexpr (SLOPE) {
            if (affine && (!XB || a.ip_epi)) {
                // the gradient's trace from the face's Q trace and the line across it, as gradient_affine
                if (face_active) FaceV::put(sU, t, qn);
                __syncthreads();
                if (face_active) {
                    const bool horiz = ff == 0 || ff == 2;
                    double td[4], ds[8], m11, m12, m21, m22, mij;
                    const int fi = horiz ? fk : (ff == 1 ? P - 1 : 0), fj = horiz ? (ff == 2 ? P - 1 : 0) : fk;
                    load_metric<P, double>(a, fe, fi + P * fj, 0, m11, m12, m21, m22, mij);
                    face_tangent<P, NF, UNROLL>(sU, (fs * 4 + ff) * P, sD, fk, td);
                    affine_gradient(horiz ? td : nd, horiz ? nd : td, m11, m12, m21, m22, ds);
#pragma unroll
                    for (int c = 0; c < 8; ++c) ds[c] *= mij;
                    const int64_t slot = (int64_t)(fe * 4 + ff) * P + fk;
                    double *mdq = ((fr.x & 15) == FK_MORTAR && a.mdq) ? a.mdq + slot * 8 : nullptr;
                    put_viscous_trace<double, double>(a, ph, fr.x, qn, ds, slot, nx, ny, ph.mu, mdq);
                }
                return;
            }
          }
          if (!XB || a.ip_epi) {   // uniform: the launch's flag
            // the updated state in the compute type (FP32: a fresh copy, the node phase
            // overwrote the first one), the broken gradient, its traces and this side's
            // viscous flux: what k_gradient evaluates for the updated state
            const R *sQn;
            if constexpr (COPY) {
                if (node_active) {
                    double qu[4];
                    Quads<double, NL>::get(sQ, xn, qu);
                    put_slots<NL, R>(a.ph, sCG, xn, qu);
                }
                __syncthreads();
                sQn = sCG;
            } else {
                sQn = (const R *)sQ;
            }
            R dq[8];
            if (node_active) {
                // the metric again from memory: keeping it live from the node phase costs the
                // FP64 kernel a wavefront per SIMD
                R m11, m12, m21, m22, mij;
                load_metric<P, R>(a, e, n, g, m11, m12, m21, m22, mij);
                ip_node_gradient<P, NL, R, UNROLL>(sQn, x0, sD, n % P, n / P, m11, m12, m21, m22, mij, dq);
            }
            __syncthreads();   // the state copy and the fluxes' space are free
            R *sDQ = S.u.sDQ;
            if (node_active) {
                NodeV::put(sDQ, xn, dq);
                NodeV::put(sDQ + 4 * NL, xn, dq + 4);
            }
            __syncthreads();
            if (face_active) {
                const int64_t slot = (int64_t)(fe * 4 + ff) * P + fk;
                double *mdq = ((fr.x & 15) == FK_MORTAR && a.mdq) ? a.mdq + slot * 8 : nullptr;
                viscous_face_trace<P, NL, R, TR, UNROLL>(a, ph, fr.x, qn, sDQ, fs * Layout<P>::ES, sLb, sLbw + 2 * P, ff,
                                                         fk, slot, nx, ny, ph.mu, mdq);
            }
          }
        }
    }
}

template <int P, int EPB, bool NS, bool IP, int RS, typename R, typename TR, bool XBF = false>
__global__ __launch_bounds__((Tile<P, EPB>::TPB))
    __attribute__((amdgpu_waves_per_eu(stage_waves(NS, IP, RS, XBF, sizeof(R) == 8, P)))) void k_stage(StageArgs a) {
    __shared__ StageSmem<P, EPB, NS, IP, R> S;
    double cq = a.cq, cg = a.cg;
    if (a.dt_dev) {   // graph replay: the step size lives in device memory
        const double d = *a.dt_dev;
        if (a.dt_cq) cq *= d;
        if (a.dt_cg) cg *= d;
    }
    const int b = xcd_tile(blockIdx.x, gridDim.x);
    stage_body<P, EPB, NS, IP, RS, R, TR, XBF>(a, b * EPB, b, cq, cg, S);
}

// ------------------------------------------------------------------ time step and sums
template <int P>
__global__ __launch_bounds__(256) void k_dt_elem(const double *Q, int K, double gamma, double gm1, double *umax,
                                                 double *amax) {
    constexpr int PP = P * P, EPB = 256 / PP > 0 ? 256 / PP : 1;
    __shared__ double su[256], sa[256];
    const int t = threadIdx.x, s = t / PP, n = t % PP, e = blockIdx.x * EPB + s;
    double u = 0.0, aa = 0.0;
    if (t < EPB * PP && e < K) {
        const double *q = Q + ((int64_t)e * PP + n) * 4;
        u = sqrt(q[1] * q[1] + q[2] * q[2]) / q[0];
        const double ur = q[1] / q[0], vr = q[2] / q[0];
        aa = sqrt(gamma * gm1 * (q[3] / q[0] - 0.5 * (ur * ur) - 0.5 * (vr * vr)));
    }
    su[t] = u; sa[t] = aa;
    __syncthreads();
    // P lanes each a column's maximum, then one lane theirs (2 P dependent reads instead of P^2)
    const bool col = t < EPB * PP && e < K && n < P;
    if (col) {
        for (int x = n + P; x < PP; x += P) { u = fmax(u, su[s * PP + x]); aa = fmax(aa, sa[s * PP + x]); }
        su[t] = u; sa[t] = aa;   // entries below P, which no lane reads above
    }
    __syncthreads();
    if (col && n == 0) {
        double mu = 0.0, ma = 0.0;
        for (int x = 0; x < P; ++x) { mu = fmax(mu, su[s * PP + x]); ma = fmax(ma, sa[s * PP + x]); }
        umax[e] = mu; amax[e] = ma;
    }
}

// mode 0: sum_e sum_ij w_i w_j J Q (four conserved variables); mode 1: the volume monitors
// sum w_i w_j J ("One") and sum w_i w_j J (p / rho^gamma - 1)^2 ("dSnorm" squared),
// QuadMesh_Integrals.incf:22-65.
template <int P>
__global__ __launch_bounds__(256) void k_cons_partial(const double *Q, const double *jac, const double *w, int K,
                                                      int mode, double gamma, double gm1, double *partial) {
    constexpr int PP = P * P, EPB = 256 / PP > 0 ? 256 / PP : 1;
    __shared__ double sv[256][4];
    const int t = threadIdx.x, s = t / PP, n = t % PP, e = blockIdx.x * EPB + s;
    double v[4] = {0, 0, 0, 0};
    if (t < EPB * PP && e < K) {
        const int i = n % P, j = n / P;
        const int64_t g = (int64_t)e * PP + n;
        const double c = w[i] * w[j] * jac[g];
        if (mode == 0) {
            for (int k = 0; k < 4; ++k) v[k] = c * Q[g * 4 + k];
        } else {
            const double *q = Q + g * 4;
            const double p = gm1 * (q[3] - 0.5 * (q[1] * q[1] + q[2] * q[2]) / q[0]);
            const double d = p / pow(q[0], gamma) - 1.0;
            v[0] = c;
            v[1] = c * (d * d);
        }
    }
    for (int k = 0; k < 4; ++k) sv[t][k] = v[k];
    __syncthreads();
    for (int wd = 128; wd > 0; wd >>= 1) {
        if (t < wd)
            for (int k = 0; k < 4; ++k) sv[t][k] += sv[t + wd][k];
        __syncthreads();
    }
    if (t < 4) partial[blockIdx.x * 4 + t] = sv[0][t];
}

// ------------------------------------------------------------------ per-order launchers
template <int P, int EPB>
inline int tile_blocks(int K) { return (K + EPB - 1) / EPB; }

// PHYS: 0 Euler, 1 Navier-Stokes BR1, 2 Navier-Stokes IP.
template <int P, int EPB, int PHYS, int RS, bool XBF = false>
hipError_t stage_launch(bool mixed, const StageArgs &a, hipStream_t st) {
    constexpr int TPB = Tile<P, EPB>::TPB;
    constexpr bool NS = PHYS >= 1, IP = PHYS == 2;
    const int nb = tile_blocks<P, EPB>(a.K);
    if (mixed) hipLaunchKernelGGL((k_stage<P, EPB, NS, IP, RS, float, float, XBF>), dim3(nb), dim3(TPB), 0, st, a);
    else hipLaunchKernelGGL((k_stage<P, EPB, NS, IP, RS, double, double, XBF>), dim3(nb), dim3(TPB), 0, st, a);
    return hipGetLastError();
}

template <int P, int EPB, int PHYS>
hipError_t stage_tile(bool mixed, const StageArgs &a, hipStream_t st) {
    switch (a.ph.rs_kernel) {
    case 0: return stage_launch<P, EPB, PHYS, 0>(mixed, a, st);
    case 1: return stage_launch<P, EPB, PHYS, 1>(mixed, a, st);
    case 2: return stage_launch<P, EPB, PHYS, 2>(mixed, a, st);
    case 3: return stage_launch<P, EPB, PHYS, 3>(mixed, a, st);
    default: return hipErrorInvalidValue;
    }
}

template <int P, int EPB>
hipError_t gradient_tile(bool mixed, const StageArgs &a, hipStream_t st) {
    constexpr int TPB = Tile<P, EPB>::TPB;
    const int nb = tile_blocks<P, EPB>(a.K);
    const bool br1 = a.ph.viscous == 1;
    // BR1 lifts the boundary's uSB (the boundary kinds must be compiled in); with artificial
    // dissipation every viscous trace takes the face's mu + mu_a
    if (a.ph.xbc && (br1 || a.ph.ad)) {
        if (mixed) {
            if (br1) hipLaunchKernelGGL((k_gradient<P, EPB, true, float, float, true>), dim3(nb), dim3(TPB), 0, st, a);
            else hipLaunchKernelGGL((k_gradient<P, EPB, false, float, float, true>), dim3(nb), dim3(TPB), 0, st, a);
        } else {
            if (br1) hipLaunchKernelGGL((k_gradient<P, EPB, true, double, double, true>), dim3(nb), dim3(TPB), 0, st, a);
            else hipLaunchKernelGGL((k_gradient<P, EPB, false, double, double, true>), dim3(nb), dim3(TPB), 0, st, a);
        }
        return hipGetLastError();
    }
    if (mixed) {
        if (br1) hipLaunchKernelGGL((k_gradient<P, EPB, true, float, float>), dim3(nb), dim3(TPB), 0, st, a);
        else hipLaunchKernelGGL((k_gradient<P, EPB, false, float, float>), dim3(nb), dim3(TPB), 0, st, a);
    } else {
        if (br1) hipLaunchKernelGGL((k_gradient<P, EPB, true, double, double>), dim3(nb), dim3(TPB), 0, st, a);
        else hipLaunchKernelGGL((k_gradient<P, EPB, false, double, double>), dim3(nb), dim3(TPB), 0, st, a);
    }
    return hipGetLastError();
}

// The run-time-solver form (rs_kernel = -1) is compiled for the wide tile only.
template <int P, int PHYS>
hipError_t stage_phys_p(int tile, bool mixed, const StageArgs &a, hipStream_t st) {
    if (a.ph.rs_kernel < 0) return stage_launch<P, Tiles<P>::large, PHYS, -1>(mixed, a, st);
    if (a.ph.xbc) {   // one solver, the boundary kinds and artificial dissipation compiled in (wide tile)
        constexpr int EPB = Tiles<P>::large;
        switch (a.ph.rs_kernel) {
        case 0: return stage_launch<P, EPB, PHYS, 0, true>(mixed, a, st);
        case 1: return stage_launch<P, EPB, PHYS, 1, true>(mixed, a, st);
        case 2: return stage_launch<P, EPB, PHYS, 2, true>(mixed, a, st);
        case 3: return stage_launch<P, EPB, PHYS, 3, true>(mixed, a, st);
        default: return hipErrorInvalidValue;
        }
    }
    return tile == 0 ? stage_tile<P, Tiles<P>::small, PHYS>(mixed, a, st)
                     : stage_tile<P, Tiles<P>::large, PHYS>(mixed, a, st);
}

template <int P>
int tile_threads_p(int tile) {
    return tile == 0 ? Tile<P, Tiles<P>::small>::TPB : Tile<P, Tiles<P>::large>::TPB;
}

template <int P>
int tile_elems_p(int tile) {
    return tile == 0 ? Tiles<P>::small : Tiles<P>::large;
}

template <int P>
int stage_blocks_p(int tile, int K) {
    return tile == 0 ? tile_blocks<P, Tiles<P>::small>(K) : tile_blocks<P, Tiles<P>::large>(K);
}

template <int P>
hipError_t gradient_p(int tile, bool mixed, const StageArgs &a, hipStream_t st) {
    return tile == 0 ? gradient_tile<P, Tiles<P>::small>(mixed, a, st)
                     : gradient_tile<P, Tiles<P>::large>(mixed, a, st);
}

template <int P>
hipError_t prolong_p(bool mixed, const StageArgs &a, hipStream_t st) {
    constexpr int EPB = Tiles<P>::large, TPB = Tile<P, EPB>::TPB;
    const int nb = tile_blocks<P, EPB>(a.K);
    if (mixed) hipLaunchKernelGGL((k_prolong<P, EPB, float>), dim3(nb), dim3(TPB), 0, st, a);
    else hipLaunchKernelGGL((k_prolong<P, EPB, double>), dim3(nb), dim3(TPB), 0, st, a);
    return hipGetLastError();
}

template <int P>
hipError_t dt_elem_p(const double *Q, int K, double gamma, double gm1, double *umax, double *amax, hipStream_t st) {
    constexpr int EPB = 256 / (P * P) > 0 ? 256 / (P * P) : 1;
    hipLaunchKernelGGL((k_dt_elem<P>), dim3((K + EPB - 1) / EPB), dim3(256), 0, st, Q, K, gamma, gm1, umax, amax);
    return hipGetLastError();
}

template <int P>
int cons_blocks_p(int K) {
    constexpr int EPB = 256 / (P * P) > 0 ? 256 / (P * P) : 1;
    return (K + EPB - 1) / EPB;
}

template <int P>
hipError_t cons_partial_p(const double *Q, const double *jac, const double *w, int K, int mode, double gamma,
                          double gm1, double *partial, hipStream_t st) {
    hipLaunchKernelGGL((k_cons_partial<P>), dim3(cons_blocks_p<P>(K)), dim3(256), 0, st, Q, jac, w, K, mode, gamma,
                       gm1, partial);
    return hipGetLastError();
}

// ------------------------------------------------------------------ artificial viscosity
// Jumps-based artificial viscosity of each element (JumpsBasedElementViscosity,
// DGArtificialDissipation.f90:277-338), from the stage's Q traces: per
// face sum_k w_k (2 (qL - qR) / (qL + qR))^2 dS for rho and rho E (Edge_ComputeJumps and its
// variants, QuadElement_EdgeProcedures.incf:1348-1619: curved interior faces per-node dS, the
// others dS of the edge's first node; boundary faces the boundary state uSB), normalised by the
// four faces' area, through the smooth switch, times Ceps sqrt(Volume)/(N+1).  FP64 in both
// forms (the FP32 form's traces, energy shifted back).
template <int P, typename TR>
__global__ __launch_bounds__(256) void k_art_visc(StageArgs a, const double *evol, const double *w, double *mu_a) {
    // one lane per face node (EPB elements of 4P lanes per workgroup); the first lane of each
    // element sums its 4P terms face by face in node order, then applies the switch
    constexpr int FN = 4 * P, EPB = 256 / FN;
    __shared__ double sj[EPB * FN][3];
    const int t = threadIdx.x, s = t / FN, l = t % FN, e = blockIdx.x * EPB + s;
    const bool act = (t < EPB * FN) && (e < a.K);
    if (act) {
        const Phys<double> ph(a.ph);
        const double es = sizeof(TR) == 4 ? a.ph.Eref : 0.0;
        const int f = l / P, k = l % P;
        const int4 fr = a.face[e * 4 + f];
        const int kind = fr.x & 15;
        const bool curved = fr.x & FF_CURVED, selfrev = fr.x & FF_SELFREV, rev = fr.x & FF_REV;
        const TR *o = (const TR *)a.tr_in + ((int64_t)(e * 4 + f) * P + k) * 4;
        const double qs[4] = {(double)o[0], (double)o[1], (double)o[2], (double)o[3] + es};
        const int gi = curved ? (selfrev ? P - 1 - k : k) : 0;
        const double *geo = a.egeo + 3 * ((int64_t)fr.z + gi);
        double qo[4], dS = geo[2];
        if (kind <= FK_PERIODIC) {
            const TR *nb = (const TR *)a.tr_in + ((int64_t)fr.y * P + (rev ? P - 1 - k : k)) * 4;
            qo[0] = (double)nb[0]; qo[1] = (double)nb[1]; qo[2] = (double)nb[2]; qo[3] = (double)nb[3] + es;
            if (kind == FK_PERIODIC) dS = a.egeo[3 * (int64_t)fr.z + 2];
        } else {
            double uB[4];
            int neu;
            ghost_state<double, true>(kind, fr.x, zone_state(a, fr.x, fr.y, (int64_t)(e * 4 + f) * P + k), a.ph, ph, qs,
                                      geo[0], geo[1], uB, qo, neu);
            dS = a.egeo[3 * (int64_t)fr.z + 2];
        }
        const double nr = 2.0 * (qs[0] - qo[0]) / (qs[0] + qo[0]);
        const double ne = 2.0 * (qs[3] - qo[3]) / (qs[3] + qo[3]);
        sj[t][0] = w[k] * nr * nr * dS;
        sj[t][1] = w[k] * ne * ne * dS;
        sj[t][2] = w[k] * geo[2];
    }
    __syncthreads();
    if (!act || l != 0) return;
    double gr = 0.0, ge = 0.0, area = 0.0;
    for (int f = 0; f < 4; ++f) {
        double jr = 0.0, je = 0.0, ar = 0.0;
        for (int k = 0; k < P; ++k) {
            const double *v = sj[s * FN + f * P + k];
            jr = jr + v[0];
            je = je + v[1];
            ar = ar + v[2];
        }
        gr = gr + jr;
        ge = ge + je;
        area = area + ar;
    }
    double gk = (gr > ge ? gr : ge) / area;
    const double kw = 5.0, s0 = log10(1.0 / pow((double)P, 4.0)) + 1.0;
    double G;
    if (!(gk > 1.0e-8)) {
        G = 0.0;
    } else {
        gk = log10(gk);
        if (gk < s0 - kw) G = 0.0;
        else if (gk < s0 + kw) G = 0.5 * sin(0.5 * 3.141592653589793 * (gk - s0) / kw) + 0.5;
        else G = 1.0;
    }
    mu_a[e] = a.ph.ad_ceps * (sqrt(evol[e]) / (double)P) * G;
}

template <int P>
hipError_t art_visc_p(bool mixed, const StageArgs &a, const double *evol, const double *w, double *mu_a,
                      hipStream_t st) {
    constexpr int EPB = 256 / (4 * P);
    const int nb = (a.K + EPB - 1) / EPB;
    if (mixed) hipLaunchKernelGGL((k_art_visc<P, float>), dim3(nb), dim3(256), 0, st, a, evol, w, mu_a);
    else hipLaunchKernelGGL((k_art_visc<P, double>), dim3(nb), dim3(256), 0, st, a, evol, w, mu_a);
    return hipGetLastError();
}

#define HG_INSTANTIATE_STAGE(PV, PHYS) \
    template hipError_t stage_phys_p<PV, PHYS>(int, bool, const StageArgs &, hipStream_t);

#define HG_INSTANTIATE_ORDER(PV)                                                                              \
    template int stage_blocks_p<PV>(int, int);                                                                \
    template int tile_threads_p<PV>(int);                                                                     \
    template int tile_elems_p<PV>(int);                                                                       \
    template hipError_t gradient_p<PV>(int, bool, const StageArgs &, hipStream_t);                            \
    template hipError_t prolong_p<PV>(bool, const StageArgs &, hipStream_t);                                  \
    template hipError_t art_visc_p<PV>(bool, const StageArgs &, const double *, const double *, double *,     \
                                       hipStream_t);                                                          \
    template hipError_t dt_elem_p<PV>(const double *, int, double, double, double *, double *, hipStream_t);  \
    template int cons_blocks_p<PV>(int);                                                                      \
    template hipError_t cons_partial_p<PV>(const double *, const double *, const double *, int, int, double,  \
                                           double, double *, hipStream_t);

}  // namespace hg
