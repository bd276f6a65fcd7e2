// kernels_flux_fused.hip -- flux residual of interior, wall and outer points,
// one pass over each point's walk, in FP64 or in the mixed form.
//
// The reference walks each of a point's direction lists separately and
// recomputes, for every list an edge (i,k) belongs to, the same limited
// reconstruction at both ends (interior_flux_dGxpos.f90:92-104).  An
// interior neighbour belongs to exactly one list per axis, so each edge is
// reconstructed three times.  This kernel walks each point's walk once (conn
// with a membership bit per direction list, then the list entries that are
// not an in-order subsequence of conn), reconstructs each end
// once, evaluates the exponentials and error functions of each axis once
// per end, and forms the directional fluxes of that edge from them.  The
// mathematics is the reference's, the rounding is not that of the list-by-list
// kernel, which keeps the reference's expressions: the FP64 form has its own
// (edge_end, erf_exp.h: refined quotients and roots, erf and exp from one table
// step), multiply-adds of an expression are fused (-ffp-contract=on), and the
// least-squares solve is applied edge by edge, through the Cramer weights of
// each list (sum_j (G_k - G_i)*(c . (dels, delt, deln)) instead of the 3x3 solve
// of the accumulated sums).
//
// A point is handled by a group of lanes, kFluxGroup = 4 of them unless the
// points are few (flux_small), each taking every fourth neighbour, and the
// group sums its partial residuals at the end, in an order that does not
// depend on the number of lanes.  Per lane this is the same work as one lane
// per point, but a resident wave holds 64 / kFluxGroup points instead of 64:
// the neighbour data of all points in flight on one XCD then fits its 4 MB L2.
// With one lane per point at the 8 resident waves per CU the FP64 kernel's
// registers allow, each point's q, qm and dq were fetched from HBM about 19
// times per launch.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "device_common.h"
#include "device_state.h"
#include "erf_exp.h"
#include "kernels.h"
#include "qlskum_math.h"



namespace mfcfd {

namespace {

constexpr int kFluxGroup = 4;

// quantities of one reconstructed end state shared by every flux of the edge;
// b_scale: B = b_scale*exp(-S*S) (FP64), or sqrt(pi*beta) (FP32)
template <typename T>
struct EndState {
    T rho, pr, ut[3], sqrt_beta, b_scale, e5;
};

template <typename T>
__device__ __forceinline__ void rotate_end(EndState<T>& e, const Frame<T>& f, T u1, T u2, T u3) {
    e.ut[0] = f.t1[0] * u1 + f.t1[1] * u2 + f.t1[2] * u3;
    e.ut[1] = f.t2[0] * u1 + f.t2[1] * u2 + f.t2[2] * u3;
    e.ut[2] = f.n[0] * u1 + f.n[1] * u2 + f.n[2] * u3;
    const T u_sqr = e.ut[0] * e.ut[0] + e.ut[1] * e.ut[1] + e.ut[2] * e.ut[2];
    e.e5 = T(2.5) * e.pr + T(0.5) * e.rho * u_sqr;
}

// The limited reconstruction at one end of an edge (limiters.f90:18-40), its
// primitive variables (qvariables_to_primitive_variables.f90:16-30) and what
// the fluxes take from them.
__device__ __forceinline__ EndState<float> edge_end(const float q[5], const float* dq, const float* qm, float epsi2,
                                                    float delx, float dely, float delz, const Frame<float>& f,
                                                    float pi) {
    float prim[5];
    reconstruct_end<float>(q, dq, qm, epsi2, delx, dely, delz, prim);
    EndState<float> e;
    e.rho = prim[0];
    e.pr = prim[4];
    const float beta = ddiv(0.5f * e.rho, e.pr);
    e.sqrt_beta = dsqrt_fast(beta);
    e.b_scale = dsqrt_fast(pi * beta);
    rotate_end(e, f, prim[1], prim[2], prim[3]);
    return e;
}

// FP64: the same quantities with fewer divisions and roots.
//   limiter   num/den with the common factor del_neg taken out of both;
//   beta      is -q5/2 itself (the reference gets it back as 0.5*rho/p), and
//             1/beta, sqrt(beta) and 1/sqrt(beta) come from one root;
//   rho       exp(q1 + beta*u*u - 2.5*log(beta)) as exp(q1 + beta*u*u) *
//             beta^(-5/2), with no logarithm.
// Against the reference's expressions in 64-bit-mantissa arithmetic, over
// states of Mach 0 to 3, the flux residual's error is that of the same
// expressions in doubles or up to 1% less.
__device__ __forceinline__ EndState<double> edge_end(const double q[5], const double* dq, const double* qm,
                                                     double epsi2, double delx, double dely, double delz,
                                                     const Frame<double>& f, double pi) {
    double qt[5];
#pragma unroll
    for (int r = 0; r < 5; ++r) {
        const double dn = -0.5 * (delx * dq[3 * r] + dely * dq[3 * r + 1] + delz * dq[3 * r + 2]);
        const double dp = (dn > 0.0 ? qm[2 * r] : qm[2 * r + 1]) - q[r];
        const double a = fma(dp, dp, epsi2), dn2 = 2.0 * dn;
        const double ratio = div_refined(fma(dn2, dp, a), fma(dn, dn2 + dp, a));
        // a NaN ratio or a NaN dn gives 1
        const double phi = __builtin_fabs(dn) > kLimiterThreshold ? __builtin_fmin(ratio, 1.0) : 1.0;
        qt[r] = fma(phi, dn, q[r]);
    }
    EndState<double> e;
    const double beta = -0.5 * qt[4];
    const RootOf y = root_of(beta);
    // y^2 and y^5 with what their roundings drop (l2, l5) and the root's own
    // correction y.e added at the end
    const double y2 = y.y * y.y, l2 = fma(y.y, y.y, -y2);
    const double temp = 0.5 * (y2 + fma(y2, y.e, l2));   // 0.5/beta
    const double u1 = qt[1] * temp, u2 = qt[2] * temp, u3 = qt[3] * temp;
    const double y4 = y2 * y2, y5 = y4 * y.y;
    const double l4 = fma(2.0 * y2, l2, fma(y2, y2, -y4));
    const double l5 = fma(y4, y.y, -y5) + fma(l4, y.y, 2.5 * y.e * y5);
    e.rho = exp_series(fma(beta, fma(u3, u3, fma(u2, u2, u1 * u1)), qt[0])) * (y5 + l5);
    e.pr = e.rho * temp;
    e.sqrt_beta = sqrt_of(y);
    e.b_scale = rsqrt_of(y, 0.28209479177387814);   // 0.5/sqrt(pi)
    rotate_end(e, f, u1, u2, u3);
    return e;
}

// S = u_a*sqrt(beta), B = 0.5*exp(-S*S)/sqrt(pi*beta), erf(S)
template <int A, typename T>
__device__ __forceinline__ void axis_terms(const EndState<T>& e, T& B, T& er) {
    const T S = e.ut[A] * e.sqrt_beta;
    T ex;
    if constexpr (sizeof(T) == 8) {
        erf_exp(S, er, ex);
        B = e.b_scale * ex;
    } else {
        ex = dexp(-S * S);
        B = ddiv(T(0.5) * ex, e.b_scale);
        er = derf_e(S, ex);
    }
}

// split_fluxes.f90 flux_G{x,y,z}{p,n}; sg = +1 or -1
template <int A, typename T>
__device__ __forceinline__ void half_flux(const EndState<T>& e, T sg, T B, T er, T G[5]) {
    const T ua = e.ut[A];
    const T Aa = T(0.5) * (T(1) + sg * er);
    const T temp1 = (ua * Aa + sg * B);
    G[0] = e.rho * temp1;
    G[1] = e.rho * e.ut[0] * temp1;
    G[2] = e.rho * e.ut[1] * temp1;
    G[3] = e.rho * e.ut[2] * temp1;
    G[1 + A] = e.pr * Aa + e.rho * ua * temp1;
    const T tail = (e.e5 + T(0.5) * e.pr) * B;
    G[4] = (e.e5 + e.pr) * ua * Aa + sg * tail;
}

// octant_fluxes.f90 flux_Gw{x,y}{p,n} (sn = -1) / flux_Go{x,y}{p,n} (sn = +1)
template <int A, typename T>
__device__ __forceinline__ void octant_flux(const EndState<T>& e, T sg, T sn, T Ba, T era, T B3, T er3,
                                            T G[5]) {
    const T ua = e.ut[A];
    const T Aa = T(0.5) * (T(1) + sg * era);
    const T A3 = T(0.5) * (T(1) + sn * er3);
    const T temp1 = (ua * Aa + sg * Ba);
    G[0] = e.rho * temp1 * A3;
    if (A == 0) {
        G[1] = (e.pr * Aa + e.rho * e.ut[0] * temp1) * A3;
        G[2] = e.rho * e.ut[1] * temp1 * A3;
    } else {
        G[1] = e.rho * e.ut[0] * temp1 * A3;
        G[2] = (e.pr * Aa + e.rho * e.ut[1] * temp1) * A3;
    }
    G[3] = e.rho * temp1 * (e.ut[2] * A3 + sn * B3);
    const T tb = (e.e5 + T(0.5) * e.pr) * Ba;
    const T temp3 = (e.e5 + e.pr) * ua * Aa + sg * tb;
    const T tn = T(0.5) * e.rho * e.ut[2] * B3 * temp1;
    G[4] = temp3 * A3 + sn * tn;
}

// flux differences in T, Cramer-weighted sums in FP64
template <typename T>
__device__ __forceinline__ void accumulate(double acc[5], const T Gi[5], const T Gk[5], double w) {
#pragma unroll
    for (int r = 0; r < 5; ++r) acc[r] = acc[r] + (double)(Gk[r] - Gi[r]) * w;
}

__device__ __forceinline__ double cramer_weight(const double* cf, int d, double wgt, double dels,
                                                double delt, double deln) {
    return wgt * (cf[3 * d] * dels + cf[3 * d + 1] * delt + cf[3 * d + 2] * deln);
}

// Half-range fluxes along axis A for the lists of that axis the entry is in:
// ab bit 0 = list 2A (positive half), bit 1 = list 2A+1.  An interior
// neighbour of conn is in exactly one of the two (generate_connectivity.f90:
// 72-106 splits with <= 0 and > 0); a spilled entry may be in either.
template <int A, typename T>
__device__ __forceinline__ void half_axis(const EndState<T>& ei, const EndState<T>& ek, unsigned ab, T Bi, T eri,
                                          T Bk, T erk, const double* cf, double wgt, double dels, double delt,
                                          double deln, double acc[5]) {
    T Gi[5], Gk[5];
    const bool pos = ab & 1u;
    const T sg = pos ? T(1) : T(-1);
    half_flux<A>(ei, sg, Bi, eri, Gi);
    half_flux<A>(ek, sg, Bk, erk, Gk);
    accumulate(acc, Gi, Gk, cramer_weight(cf, 2 * A + (pos ? 0 : 1), wgt, dels, delt, deln));
    if (ab == 3u) {
        half_flux<A>(ei, T(-1), Bi, eri, Gi);
        half_flux<A>(ek, T(-1), Bk, erk, Gk);
        accumulate(acc, Gi, Gk, cramer_weight(cf, 2 * A + 1, wgt, dels, delt, deln));
    }
}

// interior points on this kernel have every walk entry in exactly one list
// per axis (checked at bind)
template <int A, typename T>
__device__ __forceinline__ void interior_axis(const EndState<T>& ei, const EndState<T>& ek, unsigned bits,
                                              const double* cf, double wgt, double dels, double delt,
                                              double deln, double acc[5]) {
    const bool pos = (bits >> (2 * A)) & 1u;
    const T sg = pos ? T(1) : T(-1);
    T Bi, eri, Bk, erk, Gi[5], Gk[5];
    axis_terms<A>(ei, Bi, eri);
    axis_terms<A>(ek, Bk, erk);
    half_flux<A>(ei, sg, Bi, eri, Gi);
    half_flux<A>(ek, sg, Bk, erk, Gk);
    accumulate(acc, Gi, Gk, cramer_weight(cf, 2 * A + (pos ? 0 : 1), wgt, dels, delt, deln));
}

// x and y half-range lists of an interior point on the general path
template <typename T>
__device__ __forceinline__ void half_axes_xy(const EndState<T>& ei, const EndState<T>& ek, unsigned bits,
                                             const double* cf, double wgt, double dels, double delt, double deln,
                                             double acc[5]) {
    T Bi, eri, Bk, erk;
    const unsigned abx = bits & 3u, aby = (bits >> 2) & 3u;
    if (abx) {
        axis_terms<0>(ei, Bi, eri);
        axis_terms<0>(ek, Bk, erk);
        half_axis<0>(ei, ek, abx, Bi, eri, Bk, erk, cf, wgt, dels, delt, deln, acc);
    }
    if (aby) {
        axis_terms<1>(ei, Bi, eri);
        axis_terms<1>(ek, Bk, erk);
        half_axis<1>(ei, ek, aby, Bi, eri, Bk, erk, cf, wgt, dels, delt, deln, acc);
    }
}

// Quarter-range fluxes along tangent axis A of a wall point (sn = -1, Gw)
// or an outer point (sn = +1, Go).  Their x/y lists split with <= 0 and
// >= 0 (generate_connectivity.f90:148-170, 216-238): a neighbour with a zero
// offset sits in both.
template <int A, typename T>
__device__ __forceinline__ void octant_axis(const EndState<T>& ei, const EndState<T>& ek, unsigned bits, T sn,
                                            T B3i, T er3i, T B3k, T er3k, const double* cf, double wgt,
                                            double dels, double delt, double deln, double acc[5]) {
    const unsigned ab = (bits >> (2 * A)) & 3u;
    if (!ab) return;
    T Bi, eri, Bk, erk, Gi[5], Gk[5];
    axis_terms<A>(ei, Bi, eri);
    axis_terms<A>(ek, Bk, erk);
    const bool pos = ab & 1u;
    const T sg = pos ? T(1) : T(-1);
    octant_flux<A>(ei, sg, sn, Bi, eri, B3i, er3i, Gi);
    octant_flux<A>(ek, sg, sn, Bk, erk, B3k, er3k, Gk);
    accumulate(acc, Gi, Gk, cramer_weight(cf, 2 * A + (pos ? 0 : 1), wgt, dels, delt, deln));
    if (ab == 3u) {
        octant_flux<A>(ei, T(-1), sn, Bi, eri, B3i, er3i, Gi);
        octant_flux<A>(ek, T(-1), sn, Bk, erk, B3k, er3k, Gk);
        accumulate(acc, Gi, Gk, cramer_weight(cf, 2 * A + 1, wgt, dels, delt, deln));
    }
}

// CLASS 0: interior points whose walk is conn with every entry in exactly
// one list per axis (6 half-range lists).  CLASS 1: every other point, told
// apart by status: wall points take the Gw octant lists in x and y, the
// half-range z- list over conn and the factor 2 of flux_residual.f90:50;
// outer points the Go octant lists and the half-range z+ list (:54-66);
// interior points whose lists the 22-column spill altered the six
// half-range lists, each walk entry in the lists its bits name (:68-81).
// T: arithmetic of the reconstruction and fluxes (double: the FP64 form;
// float: the mixed form, reading the FP32 q, qm, dq); geometry, Cramer
// weights and the sums stay FP64.
// WAVES: minimum waves per SIMD the kernel is compiled for (its register
// cap); the launch picks one of the compiled variants and a block size
// G: lanes that share the point (lane: this one's number among them)
template <int CLASS, bool UW, typename T, int G>
__device__ __forceinline__ void flux_point(const DevGeom& g, const DevState& s, const FlowParams& fp, int i,
                                           int lane) {
    const QArrays<T> qa = qarrays<T>(s);
    const Frame<double> f = load_frame(g.frame, i);
    const Frame<T> ft = frame_as<T>(f);
    const T pi = T(fp.pi);
    const double4 pi4 = g.pos[i];
    // the point's own reconstruction inputs are re-read for every neighbour:
    // the four lanes of a group read the same addresses, which costs the
    // gather little, and holding them would cost registers and resident
    // waves (FP32: 116 instead of 139 VGPRs, 4 instead of 3 waves per SIMD)
    const T* qip = qa.qp(i);
    const T* dqi = qa.dqp(i);
    const T* qmi = qa.qmp(i);
    const T epsi2_i = T(limiter_epsi2(fp.vl_const, pi4.w));
    const double* cf = g.coef + 18 * (long long)i;
    const int nb = g.nwalk[i];
    const unsigned* wk = g.walk + kWalkCols * (long long)i;
    const int st_i = CLASS == 1 ? g.status[i] : 0;
    const T sn = st_i == 2 ? T(1) : T(-1);
    double acc[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
    for (int base = 0; base < nb; base += G) {
        const int j = base + lane;
        // the entry's own sum over its lists first: it is what add_terms moves
        double sum[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
        const unsigned e = j < nb ? wk[j] : 0u;
        const unsigned bits = e & ((1u << kWalkMaskBits) - 1u);
        if (bits != 0u) {
            const int k = (int)(e >> kWalkMaskBits);
            const double4 pk = g.pos[k];
            const double delx = pk.x - pi4.x;
            const double dely = pk.y - pi4.y;
            const double delz = pk.z - pi4.z;
            const double dels = delx * f.t1[0] + dely * f.t1[1] + delz * f.t1[2];
            const double delt = delx * f.t2[0] + dely * f.t2[1] + delz * f.t2[2];
            const double deln = delx * f.n[0] + dely * f.n[1] + delz * f.n[2];
            const double wgt = wls_weight<UW>(dels, delt, deln, fp.power);
            T qi[5], qk[5];
#pragma unroll
            for (int r = 0; r < 5; ++r) qi[r] = qip[r];
            const EndState<T> ei = edge_end(qi, dqi, qmi, epsi2_i, T(delx), T(dely), T(delz), ft, pi);
#pragma unroll
            for (int r = 0; r < 5; ++r) qk[r] = qa.qp(k)[r];
            const EndState<T> ek = edge_end(qk, qa.dqp(k), qa.qmp(k), T(limiter_epsi2(fp.vl_const, pk.w)), T(delx),
                                            T(dely), T(delz), ft, pi);
            if (CLASS == 0) {
                interior_axis<0>(ei, ek, bits, cf, wgt, dels, delt, deln, sum);
                interior_axis<1>(ei, ek, bits, cf, wgt, dels, delt, deln, sum);
                interior_axis<2>(ei, ek, bits, cf, wgt, dels, delt, deln, sum);
            } else {
                T B3i, er3i, B3k, er3k;
                axis_terms<2>(ei, B3i, er3i);
                axis_terms<2>(ek, B3k, er3k);
                if (st_i == 0) {
                    half_axes_xy(ei, ek, bits, cf, wgt, dels, delt, deln, sum);
                } else {
                    octant_axis<0>(ei, ek, bits, sn, B3i, er3i, B3k, er3k, cf, wgt, dels, delt, deln, sum);
                    octant_axis<1>(ei, ek, bits, sn, B3i, er3i, B3k, er3k, cf, wgt, dels, delt, deln, sum);
                }
                const unsigned abz = (bits >> (2 * 2)) & 3u;
                if (abz) half_axis<2>(ei, ek, abz, B3i, er3i, B3k, er3k, cf, wgt, dels, delt, deln, sum);
            }
        }
#pragma unroll
        for (int r = 0; r < 5; ++r) acc[r] = add_terms<G>(acc[r], sum[r]);
    }
#pragma unroll
    for (int r = 0; r < 5; ++r) acc[r] = group_sum<4>(acc[r]);
    if (lane == 0) {
#pragma unroll
        for (int r = 0; r < 5; ++r) s.flux_res[5 * (long long)i + r] = st_i == 1 ? 2.0 * acc[r] : acc[r];
    }
}

template <int CLASS, bool UW, typename T, int WAVES>
__global__ void __launch_bounds__(kBlock, WAVES) k_flux_fused(DevGeom g, DevState s, FlowParams fp, const int* idx,
                                                             int count) {
    if constexpr (sizeof(T) == 8) load_erf_nodes();
    const unsigned t = (unsigned)xcd_index();
    const int m = (int)(t / kFluxGroup);
    if (m >= count) return;  // whole groups: blocks hold a multiple of kFluxGroup lanes
    flux_point<CLASS, UW, T, kFluxGroup>(g, s, fp, idx[m], (int)(t % kFluxGroup));
}

// blocks of the general class in k_flux_small, a whole number per XCD
__host__ __device__ inline int small_blocks(int points, int lanes) {
    const int blocks = (int)(((long long)points * lanes + kBlock - 1) / kBlock);
    return (blocks + kXcds - 1) / kXcds * kXcds;
}

// Both classes of a cloud that does not fill the chip in one launch, GG lanes
// per point of the general class, whose points take longer and come first,
// and GI per point of the interior one, from the next block on.
// (FP64: two waves per SIMD; capped at three it spills 23 registers, and the
// 250,000-point iteration takes 479 instead of 426 us.)
template <bool UW, typename T, int GG, int GI>
__global__ void __launch_bounds__(kBlock, sizeof(T) == 4 && GI == kFluxGroup ? 3 : 2)
    k_flux_small(DevGeom g, DevState s, FlowParams fp, const int* general, int n_general, const int* interior,
                 int n_interior) {
    if constexpr (sizeof(T) == 8) load_erf_nodes();
    const int first = small_blocks(n_general, GG), b = (int)blockIdx.x;
    if (b < first) {
        const int t = xcd_block(b, first) * kBlock + (int)threadIdx.x, m = t / GG;
        if (m < n_general) flux_point<1, UW, T, GG>(g, s, fp, general[m], t % GG);   // whole groups
    } else {
        const int t = xcd_block(b - first, (int)gridDim.x - first) * kBlock + (int)threadIdx.x, m = t / GI;
        if (m < n_interior) flux_point<0, UW, T, GI>(g, s, fp, interior[m], t % GI);
    }
}

template <bool UW, typename T, int GG, int GI>
void launch_small(const DevGeom& g, const DevState& s, const FlowParams& p, const TypeLists& tl, int parts,
                  hipStream_t st) {
    const int ng = parts & 2 ? tl.n_fused_wall : 0, ni = parts & 1 ? tl.n_fused_interior : 0;
    const int blocks = small_blocks(ng, GG) + grid_for((long long)ni * GI, kBlock);
    if (blocks > 0)
        hipLaunchKernelGGL((k_flux_small<UW, T, GG, GI>), dim3(blocks), dim3(kBlock), 0, st, g, s, p, tl.fused_wall,
                           ng, tl.fused_interior, ni);
}

template <int CLASS, typename T>
void launch_class(const DevGeom& g, const DevState& s, const FlowParams& p, const int* idx, int count,
                  const KernelShape& ks, hipStream_t st) {
    if (count <= 0) return;
    int block = ks.block > 0 && ks.block <= kBlock ? ks.block : kBlock;
    block -= block % kFluxGroup;
    const dim3 grid(grid_for((long long)count * kFluxGroup, block)), blk(block);
    // the reservation counts the FP64 kernels' own table
    constexpr int own = sizeof(T) == 8 ? kErfNodes * (int)sizeof(double2) : 0;
    const int lds = ks.lds > own ? ks.lds - own : 0;
    if (p.power != 0.0) {
        hipLaunchKernelGGL((k_flux_fused<CLASS, false, T, 2>), grid, blk, lds, st, g, s, p, idx, count);
        return;
    }
    // caps of three waves and more are the FP32 variants'; the FP64 kernels spill
    // under them (2M points, interior class: 2.88 ms with three and 5.09 with four
    // against 1.95 with two) and run with two instead
    if constexpr (sizeof(T) == 4) {
        const auto launch = [&](auto waves) {
            hipLaunchKernelGGL((k_flux_fused<CLASS, true, T, decltype(waves)::value>), grid, blk, lds, st, g, s, p, idx,
                               count);
        };
        switch (ks.waves) {
            case 3: return launch(std::integral_constant<int, 3>{});
            case 4: return launch(std::integral_constant<int, 4>{});
            case 5: return launch(std::integral_constant<int, 5>{});
            case 6: return launch(std::integral_constant<int, 6>{});
            default: break;
        }
    }
    if (ks.waves == 1)
        hipLaunchKernelGGL((k_flux_fused<CLASS, true, T, 1>), grid, blk, lds, st, g, s, p, idx, count);
    else
        hipLaunchKernelGGL((k_flux_fused<CLASS, true, T, 2>), grid, blk, lds, st, g, s, p, idx, count);
}

}  // namespace

// Whether one launch takes both classes.  The general class, an eighth of the
// points, leaves the chip mostly idle by itself up to some 100,000 points, and
// in one launch it fills what the interior class leaves free.  The larger
// registers of the two kernels then hold for both (FP32: three waves per SIMD
// instead of the interior class's four), so the gain shrinks with the size.  An
// explicit iteration in us, a launch per class -> one launch:
//                       FP64            mixed
//       1,209 points     87 ->   33      89 ->  31
//      20,000           106 ->   62     105 ->  49
//      50,000           137 ->  107     122 ->  84
//     100,000           200 ->  178     174 -> 138
//     170,000           290 ->  266     241 -> 217
//     350,000           579 ->  545     458 -> 430
//     500,000           816 ->  784     622 -> 610
//     600,000           977 ->  949     746 -> 745  (best class shapes 735)
//     750,000          1230 -> 1189     943 -> 937  (921)
// The line, at 450,000 interior points, is where the mixed form's gain ends; it
// serves both forms, and FP64 leaves 3% beyond it.  Below it no shape of a launch
// per class is faster.  With weighted least squares at 150,000 points 246 -> 233
// and 199 -> 183, at 170,000 (one launch 263 and 205) a launch each.
bool flux_joint(const TypeLists& tl, double power) {
    const int ng = tl.n_fused_wall, ni = tl.n_fused_interior;
    return ng <= (power != 0.0 ? 20000 : 100000) && ni <= 450000;
}

// The joint launch, and the lanes that share a point in it; false: each class
// takes a launch.  Four lanes take a point's 25 neighbours in seven steps, each
// a chain of dependent loads and arithmetic, and with few points the steps are
// what counts: 32 lanes take one step, 16 two.  They cost nothing while the chip
// has room, about a third more than four lanes once it is full (the lanes beyond
// 25 idle, terms are moved between lanes).  An iteration in us, FP64 / mixed, on
// both sides of each line (general + interior lanes):
//   general points 20,000   15,145 (100,000 in all)  16+4   178 / 138   4+4   172 / 145
//                           22,592 (150,000)         16+4   245 / 194   4+4   240 / 199
//   interior points 24,000  22,937 (27,000)          16+16   70 /  58   16+4   73 /  62
//                           28,090 (33,000)          16+16   82 /  64   16+4   81 /  62
//   general points 4,000     3,252 (20,000)          32+16   62 /  49   16+16  59 /  49
//                            4,063 (27,000)          32+16   74 /  59   16+16  70 /  58
//   interior points 4,000    3,777 (6,057)           32+32   39 /  34   32+16  41 /  34
//                           16,748 (20,000)          32+32   64 /  50   32+16  62 /  49
// and weighted, interior points 24,000: 23,760  16+16  69 / 62   16+4  67 / 57,
// 29,040  84 / 74 and 73 / 60.
template <typename T>
static bool flux_small(const DevGeom& g, const DevState& s, const FlowParams& p, const TypeLists& tl,
                       hipStream_t st, int parts) {
    if (!flux_joint(tl, p.power)) return false;
    const int ng = tl.n_fused_wall, ni = tl.n_fused_interior;
    if (p.power != 0.0) {
        // weighted least squares: the two that cover most sizes
        if (ni > 24000) launch_small<false, T, 16, 4>(g, s, p, tl, parts, st);
        else launch_small<false, T, 16, 16>(g, s, p, tl, parts, st);
    } else if (ng > 20000) {
        launch_small<true, T, 4, 4>(g, s, p, tl, parts, st);
    } else if (ni > 24000) {
        launch_small<true, T, 16, 4>(g, s, p, tl, parts, st);
    } else if (ng > 4000) {
        launch_small<true, T, 16, 16>(g, s, p, tl, parts, st);
    } else if (ni > 4000) {
        launch_small<true, T, 32, 16>(g, s, p, tl, parts, st);
    } else {
        launch_small<true, T, 32, 32>(g, s, p, tl, parts, st);
    }
    return true;
}

template <typename T>
static void launch_flux(const DevGeom& g, const DevState& s, const FlowParams& p, const TypeLists& tl,
                        hipStream_t st, int parts, const LaunchShapes& ls) {
    if (flux_small<T>(g, s, p, tl, st, parts)) return;
    if (parts & 1) launch_class<0, T>(g, s, p, tl.fused_interior, tl.n_fused_interior, ls.flux_interior, st);
    if (parts & 2) launch_class<1, T>(g, s, p, tl.fused_wall, tl.n_fused_wall, ls.flux_wall, st);
}

void launch_flux_fused(const DevGeom& g, const DevState& s, const FlowParams& p, const TypeLists& tl,
                       hipStream_t st, int parts, bool mixed, const LaunchShapes& ls) {
    if (mixed) launch_flux<float>(g, s, p, tl, st, parts, ls);
    else launch_flux<double>(g, s, p, tl, st, parts, ls);
}

}  // namespace mfcfd
