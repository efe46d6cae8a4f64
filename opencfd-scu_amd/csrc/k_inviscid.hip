// k_inviscid.hip - fused inviscid sweep per direction (gfx950).
//
// One pass per direction replaces the reference's split kernel
// (split_Jac3d_Stager_Warming_ker, src/OCFD_split.cu:145-198) and its ten
// derivative launches (OCFD_d?1 / OCFD_d?2, src/OCFD_Schemes_Choose.cu:88-765,
// each launching one P or M kernel per variable with an atomicAdd into du,
// src/OCFD_Schemes.cu:293-381):
//
//   phase 1  load rho,u,v,w,T and the direction's cofactors for a tile of
//            nodes (+4 ghost nodes each side along the sweep), compute the
//            sound speed and the Steger-Warming f+/f- of all 5 variables,
//            stage them in LDS (they never touch HBM);
//   phase 2  one thread per half node: P and M reconstructions of all 5
//            variables with the reference's boundary closures;
//   phase 3  one thread per node: du += -(hP(i+1/2)-hP(i-1/2))/h, then += the
//            M term, in the reference's order (x P, x M, y P, ...), with no
//            atomics; on small grids each direction into its own five fields.
//            The reference multiplies every term by the node's Ajac; here the
//            RK stage multiplies their sum once, so the sweeps do not read it.
//
// S (double or float) is the type of the primitives, the split fluxes, the
// reconstructions and du; the WENO weight arithmetic and the Jacobian factor
// with the accumulation into du are always double.
#include <type_traits>

#include "mlp_dev.h"
#include "ocfd_dev.h"
#include "ocfd_kernels.h"

namespace {

// sqrt(x) and 1/sqrt(x) together.  FP64: two coupled Newton steps from the
// hardware's estimate (5e-8) and a last correction of each: 15 instructions,
// where a square root and a division of their own, with the scaling that only
// subnormal and huge arguments need, take 30.  Largest errors over 2e6
// arguments of e^-40..e^40: root 1.1e-16, reciprocal 1.7e-16, as of the square
// root and division (du and the state come out the same distance from 80-bit
// arithmetic with either).  x = 0 gives NaN in both (ROOT0: the root is 0).  FP32:
// the hardware's instructions, 1 ulp each; without ROOT0 the root is x times the
// reciprocal root (two roundings), at x = 0 NaN and infinity.
template <bool ROOT0, typename R>
__device__ __forceinline__ void sqrt_pair(R x, R& root, R& inv) {
    if constexpr (std::is_same<R, float>::value) {
        if constexpr (ROOT0) {
            root = __builtin_amdgcn_sqrtf(x);
        } else {
            inv = __builtin_amdgcn_rsqf(x);
            root = x * inv;
        }
    } else {
        double y = __builtin_amdgcn_rsq(x);
        if (ROOT0) y = x == 0.0 ? 0.0 : y;
        double g = x * y, h = 0.5 * y;
        double e = fma(-h, g, 0.5);
        g = fma(g, e, g);
        h = fma(h, e, h);
        e = fma(-h, g, 0.5);
        g = fma(g, e, g);
        h = fma(h, e, h);
        root = fma(fma(-g, g, x), h, g);
        inv = h + h;
        inv = fma(fma(-root, inv, 1.0), inv, inv);
    }
}

// Steger-Warming split of one node (src/OCFD_split.cu:92-142), the reference's
// sums over the three waves with u -+ c n formed in one fused operation from
// c/|A| and the waves' energies |u -+ c n|^2/2 + W c^2 formed once for both
// sides: about 100 instructions a node against 165.  Summed instead as f_i =
// u_i f0 + n_i c (l3 - l2), 85 instructions, the energy of a low-Mach flow
// cancels: du's error against 80-bit arithmetic was up to 8 % (ramp 14 %) above
// the reference's sums' in a component, while a step took 1 % less (1024x256x128
// 19.75 ms, now 19.95; y sweep of 512x128x64 147.8 us, 148.3).  Written with n
// normalised first or with W c^2 apart it rounds no better in the state and
// the z sweep loses its fifth wave (1083 -> 1127 us).  l = (E +- |E|)/2 with the
// factor rho/(2 gamma) in it.
template <typename R>
__device__ __forceinline__ void sw_split(R tmp0d, R u, R v, R w, R cc, R A1, R A2, R A3, const Consts& c,
                                         R* fp, R* fm) {
    R ss, rs;
    sqrt_pair<false>(A1 * A1 + A2 * A2 + A3 * A3, ss, rs);
    const R E1 = A1 * u + A2 * v + A3 * w;
    const R E2 = E1 - cc * ss, E3 = E1 + cc * ss;
    const R eps = R(c.epsl_sw);
    R a1, a2, a3;
    if (eps == R(0)) {
        // sqrt(x*x) == |x| in binary floating point with round-to-nearest
        // (no underflow of x*x): the same values without three square roots
        a1 = fabs(E1); a2 = fabs(E2); a3 = fabs(E3);
    } else {
        a1 = sqrt(E1 * E1 + eps * eps); a2 = sqrt(E2 * E2 + eps * eps); a3 = sqrt(E3 * E3 + eps * eps);
    }
    const R k2 = u * u + v * v + w * w, ccr = cc * rs;
    // u -+ c n
    const R um = fma(-ccr, A1, u), up = fma(ccr, A1, u), vm = fma(-ccr, A2, v), vp = fma(ccr, A2, v),
            wm = fma(-ccr, A3, w), wp = fma(ccr, A3, w);
    const R vv = (R(c.gamma) - R(1.0)) * k2, W2 = R(c.split_c3) * cc * cc;
    const R Km = fma(R(0.50), um * um + vm * vm + wm * wm, W2), Kp = fma(R(0.50), up * up + vp * vp + wp * wp, W2);
    const R C1 = R(c.split_c1), q = R(0.50) * tmp0d;
    auto side = [&](R l1, R l2, R l3, R* f) {
        const R a = C1 * l1;
        f[0] = fma(C1, l1, l2) + l3;
        f[1] = fma(l3, up, fma(l2, um, a * u));
        f[2] = fma(l3, vp, fma(l2, vm, a * v));
        f[3] = fma(l3, wp, fma(l2, wm, a * w));
        f[4] = fma(l3, Kp, fma(l2, Km, l1 * vv));
    };
    side((E1 + a1) * q, (E2 + a2) * q, (E3 + a3) * q, fp);
    side((E1 - a1) * q, (E2 - a2) * q, (E3 - a3) * q, fm);
}

// What the split of a node reads, and f+ and f- of it along direction DIR.
template <typename S> struct NodeIn { S d, u, v, w, T, a[3]; };
template <int DIR, typename S>
__device__ __forceinline__ NodeIn<S> load_node(const SweepArgsT<S>& A, int i, int j, int k) {
    const long long q = gidx(A.g, i, j, k);
    return {A.d[q], A.u[q], A.v[q], A.w[q], A.T[q],
            {S(A.M[3 * DIR][q]), S(A.M[3 * DIR + 1][q]), S(A.M[3 * DIR + 2][q])}};
}
template <typename S>
__device__ __forceinline__ void split_node(const SweepArgsT<S>& A, const NodeIn<S>& n, S* fp, S* fm) {
    S root, inv;
    sqrt_pair<true>(n.T, root, inv);
    const S cc = root * S(A.c.rama);  // sound_speed_kernel, src/commen_kernel.cu:144-153
    sw_split<S>(n.d * S(A.c.tmp0), n.u, n.v, n.w, cc, n.a[0], n.a[1], n.a[2], A.c, fp, fm);
}
template <int DIR, typename S>
__device__ __forceinline__ void split_node(const SweepArgsT<S>& A, int i, int j, int k, S* fp, S* fm) {
    split_node<S>(A, load_node<DIR>(A, i, j, k), fp, fm);
}

// The direction's part of du's variable m at node i along it, added to pre if
// ACC: P then M, in the reference's order, the sum in double.  face(v, 0 / 1):
// value v (P of variable v < 5, M of v - 5) at the node's left / right face.
template <int DIR, bool ACC, typename S, typename F>
__device__ __forceinline__ S du_of(const SweepArgsT<S>& A, int i, int m, double pre, F&& face) {
    const int n_dir = DIR == 0 ? A.g.nx : DIR == 1 ? A.g.ny : A.g.nz;
    const bool zp = A.nrp[DIR] && i == 0, zm = A.nrm[DIR] && i == n_dir - 1;
    const double rh = 1.0 / A.h[DIR];
    const double dP = zp ? 0.0 : double(face(m, 1) - face(m, 0));
    const double dM = zm ? 0.0 : double(face(5 + m, 1) - face(5 + m, 0));
    return S(fma(-dM, rh, ACC ? fma(-dP, rh, pre) : -dP * rh));
}
// du_of for the five variables of a node (linear index q).  PARTS: into the
// direction's own group of du, else into the one du.  ACC: added to pre, the
// earlier directions' part; else written, streamed (nothing reads it before the
// next sweep or the RK stage).
template <int DIR, bool PARTS, bool ACC, typename S, typename F>
__device__ __forceinline__ void put_du(const SweepArgsT<S>& A, int i, long long q, const double* pre, F&& face) {
#pragma unroll
    for (int m = 0; m < 5; m++) {
        S* o = &A.du[((PARTS ? 5 * DIR : 0) + m) * A.fs + q];
        const S r = du_of<DIR, ACC>(A, i, m, ACC ? pre[m] : 0.0, face);
        if constexpr (ACC) *o = r;
        else __builtin_nontemporal_store(r, o);
    }
}
// P and M half-node values of all five variables at face j+1/2 (c = j+1, r =
// j-n, the reference's coords and coords+start-end): the closure/scheme case
// of the P side (OCFD_bound_scheme_kernel_p, src/OCFD_bound_Scheme.cu:739-819)
// and of the M side (OCFD_bound_scheme_kernel_m, 855-944; hybrid_auto:
// src/OCFD_Schemes_hybrid_auto.cu:911-919, 1008-1016) is decided once per
// face, then each case loops over the variables (ld(v, k) = f+ of variable v
// (v < 5) or f- of variable v-5 at stencil node k, k = 0..7 for nodes
// j-3..j+4).
template <typename R, typename W, int SCH, typename LD>
__device__ __forceinline__ void face_all_p(LD&& ld, int c, int r, int bl, int br, int hy, R tvlim, R tvmax, R* hp) {
    constexpr int kaP = Ext<SCH, 0>::ka, kbP = Ext<SCH, 0>::kb;
    // P: 0..3 left closures (c), 4..6 right closures, 7 scheme, 8 WENO7, 9 WENO5
    int pc;
    if (bl && c <= -kaP) pc = c;
    else if (br && r >= -kbP) pc = r == -1 ? 4 : r == -2 ? 5 : 6;
    else if (SCH == OCFD_HYBRIDAUTO) pc = hy == 1 ? 7 : hy == 2 ? 8 : 9;
    else pc = 7;
    if (pc == 7) {
#pragma unroll
        for (int m = 0; m < 5; m++) {
            R g[8];
#pragma unroll
            for (int k = 0; k < 8; k++) g[k] = ld(m, k);
            if (SCH == OCFD_WENO7) hp[m] = weno7_up<R, W>(g);
            else if (SCH == OCFD_UP7 || SCH == OCFD_HYBRIDAUTO) hp[m] = up7_up(g);
            else if (SCH == OCFD_WENO5) hp[m] = weno5_up<R, W>(g + 1);
            else if (SCH == OCFD_NND2) hp[m] = nnd2_up(g + 2);
            else if (SCH == OCFD_WENO7_SYMBO) hp[m] = symbo_up<R, W>(g, 0, tvlim, tvmax);
            else if (SCH == OCFD_WENO7_SYMBO_LIM) hp[m] = symbo_up<R, W>(g, 1, tvlim, tvmax);
            else if (SCH == OCFD_OMP6_HR) hp[m] = omp6_up(0, g);
            else if (SCH == OCFD_OMP6_LD) hp[m] = omp6_up(1, g);
            else hp[m] = omp6_up(2, g);
        }
    } else if (pc == 8) {
#pragma unroll
        for (int m = 0; m < 5; m++) {
            R g[8];
#pragma unroll
            for (int k = 0; k < 7; k++) g[k] = ld(m, k);
            hp[m] = weno7_up<R, W>(g);
        }
    } else if (pc == 9 || pc == 3 || pc == 6) {
#pragma unroll
        for (int m = 0; m < 5; m++) {
            R g[8];
#pragma unroll
            for (int k = 1; k < 6; k++) g[k] = ld(m, k);
            hp[m] = weno5_up<R, W>(g + 1);
        }
    } else {
#pragma unroll
        for (int m = 0; m < 5; m++) {
            R g[8];
#pragma unroll
            for (int k = 0; k < 8; k++) g[k] = ld(m, k);
            if (pc == 0) hp[m] = g[4];
            else if (pc == 1) hp[m] = weno5_up_left<R, W>(g + 1);
            else if (pc == 2) hp[m] = weno5_up_leftplus<R, W>(g + 1);
            else if (pc == 4) hp[m] = g[3] + R(0.5) * d_minmod2(g[3] - g[2], g[3] - g[2]);
            else hp[m] = weno5_up_rightplus<R, W>(g + 1);
        }
    }
}
// M half-node values (ld(5+m, k) = f- of variable m at node j-3+k).
template <typename R, typename W, int SCH, typename LD>
__device__ __forceinline__ void face_all_m(LD&& ld, int c, int r, int bl, int br, int hy, R* hm) {
    constexpr int kaM = Ext<SCH, 1>::ka, kbM = Ext<SCH, 1>::kb;
    // M: 0..2 left closures (c), 3..6 right closures, 7 scheme, 8 WENO7, 9 WENO5
    int mc;
    if (bl && c < -kaM) mc = c < 2 ? c : 2;  // c >= 2: plain WENO5
    else if (br && r >= -kbM - 1) mc = r == -1 ? 3 : r == -2 ? 4 : r == -3 ? 5 : 6;
    else if (SCH == OCFD_HYBRIDAUTO) mc = hy == 1 ? 7 : hy == 2 ? 8 : 9;
    else mc = 7;
    if (mc == 7) {
#pragma unroll
        for (int m = 0; m < 5; m++) {
            R g[8];
#pragma unroll
            for (int k = 0; k < 8; k++) g[k] = ld(5 + m, k);
            if (SCH == OCFD_WENO7) hm[m] = weno7_dn<R, W>(g + 1);
            else if (SCH == OCFD_UP7 || SCH == OCFD_HYBRIDAUTO) hm[m] = up7_dn(g);
            else if (SCH == OCFD_WENO5) hm[m] = weno5_dn<R, W>(g + 2);
            else if (SCH == OCFD_NND2) hm[m] = nnd2_dn(g + 3);
            else if (SCH == OCFD_WENO7_SYMBO || SCH == OCFD_WENO7_SYMBO_LIM) hm[m] = symbo_dn<R, W>(g);
            else if (SCH == OCFD_OMP6_HR) hm[m] = omp6_dn(0, g);
            else if (SCH == OCFD_OMP6_LD) hm[m] = omp6_dn(1, g);
            else hm[m] = omp6_dn(2, g);
        }
    } else if (mc == 8) {
#pragma unroll
        for (int m = 0; m < 5; m++) {
            R g[8];
#pragma unroll
            for (int k = 1; k < 8; k++) g[k] = ld(5 + m, k);
            hm[m] = weno7_dn<R, W>(g + 1);
        }
    } else if (mc == 9 || mc == 2 || mc == 6) {
#pragma unroll
        for (int m = 0; m < 5; m++) {
            R g[8];
#pragma unroll
            for (int k = 2; k < 7; k++) g[k] = ld(5 + m, k);
            hm[m] = weno5_dn<R, W>(g + 2);
        }
    } else {
#pragma unroll
        for (int m = 0; m < 5; m++) {
            R g[8];
#pragma unroll
            for (int k = 0; k < 8; k++) g[k] = ld(5 + m, k);
            if (mc == 0) hm[m] = weno5_dn_left<R, W>(g + 2);
            else if (mc == 1) hm[m] = weno5_dn_leftplus<R, W>(g + 2);
            else if (mc == 3) hm[m] = g[3];
            else if (mc == 4) hm[m] = g[4] - R(0.5) * d_minmod2(g[4] - g[3], g[4] - g[3]);
            else hm[m] = weno5_dn_rightplus<R, W>(g + 2);
        }
    }
}
template <typename R, typename W, int SCH, typename LD>
__device__ __forceinline__ void face_all(LD&& ld, int c, int r, int bl, int br, int hy, R tvlim, R tvmax, R* hp,
                                         R* hm) {
    face_all_p<R, W, SCH>(ld, c, r, bl, br, hy, tvlim, tvmax, hp);
    face_all_m<R, W, SCH>(ld, c, r, bl, br, hy, hm);
}

// The closure/scheme case of a face's P value (0..3 left closures by c, 4..6
// right closures, 7 the scheme, 8 WENO7, 9 WENO5) and M value (0..2 left
// closures, 3..6 right closures, 7 the scheme, 8 WENO7, 9 WENO5): the
// selection of face_all_p / face_all_m.
template <int SCH>
__device__ __forceinline__ int case_p(int c, int r, int bl, int br, int hy) {
    constexpr int kaP = Ext<SCH, 0>::ka, kbP = Ext<SCH, 0>::kb;
    if (bl && c <= -kaP) return c;
    if (br && r >= -kbP) return r == -1 ? 4 : r == -2 ? 5 : 6;
    if (SCH == OCFD_HYBRIDAUTO) return hy == 1 ? 7 : hy == 2 ? 8 : 9;
    return 7;
}
template <int SCH>
__device__ __forceinline__ int case_m(int c, int r, int bl, int br, int hy) {
    constexpr int kaM = Ext<SCH, 1>::ka, kbM = Ext<SCH, 1>::kb;
    if (bl && c < -kaM) return c < 2 ? c : 2;
    if (br && r >= -kbM - 1) return r == -1 ? 3 : r == -2 ? 4 : r == -3 ? 5 : 6;
    if (SCH == OCFD_HYBRIDAUTO) return hy == 1 ? 7 : hy == 2 ? 8 : 9;
    return 7;
}
// One P value (case pc) or M value (case mc) of hybrid_auto from the stencil
// g[0..7] of nodes j-3..j+4: the formulas of face_all_p / face_all_m case by
// case.
template <typename R, typename W>
__device__ __forceinline__ R recon_p_hybrid(int pc, const R* g) {
    switch (pc) {
        case 0: return g[4];
        case 1: return weno5_up_left<R, W>(g + 1);
        case 2: return weno5_up_leftplus<R, W>(g + 1);
        case 4: return g[3] + R(0.5) * d_minmod2(g[3] - g[2], g[3] - g[2]);
        case 5: return weno5_up_rightplus<R, W>(g + 1);
        case 7: return up7_up(g);
        case 8: return weno7_up<R, W>(g);
        default: return weno5_up<R, W>(g + 1);  // 3, 6, 9
    }
}
template <typename R, typename W>
__device__ __forceinline__ R recon_m_hybrid(int mc, const R* g) {
    switch (mc) {
        case 0: return weno5_dn_left<R, W>(g + 2);
        case 1: return weno5_dn_leftplus<R, W>(g + 2);
        case 3: return g[3];
        case 4: return g[4] - R(0.5) * d_minmod2(g[4] - g[3], g[4] - g[3]);
        case 5: return weno5_dn_rightplus<R, W>(g + 2);
        case 7: return up7_dn(g);
        case 8: return weno7_dn<R, W>(g + 1);
        default: return weno5_dn<R, W>(g + 2);  // 2, 6, 9
    }
}

// hybrid_auto sends most faces to UP7 and a few (at shocks, and closures near
// DIF_BOUND faces) to WENO7 / WENO5.  A wave whose lanes each ran their own
// face's ten reconstructions would run the WENO code ten times over for a
// single WENO face while the other lanes wait.  Instead the UP7 faces are
// computed by their own lanes and the ten P and M values of the other
// ("special") faces are spread over the wave, one value per lane: up to six
// special faces per wave in one pass; a wave with more takes the per-face
// path.  Same formulas, so the same values.  Used in the x sweep, which is
// VALU-bound (91 % VALU busy on the 1024x384x256 swept ramp; 2.40 -> 2.23 ms
// per launch); the tiles, at 48-60 % VALU busy, measured the same or 2 %
// slower with it and keep the per-face path.
constexpr int COMPACT_MAX = 6;  // special faces per wave spread in one pass (10 values each)
// The lane of the n-th special face of the wave (n-th set bit of mask).
__device__ __forceinline__ int nth_lane(unsigned long long mask, int n) {
    for (int t = 0; t < n; t++) mask &= mask - 1;
    return mask ? __builtin_ctzll(mask) : 0;
}

// Orders the LDS accesses of one wave (its own LDS operations execute in
// order; this keeps the compiler from moving them).
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// x sweep.  A wave owns XR row segments of XS output nodes: its 64 lanes are the
// XS + 8 nodes of each segment (4 ghost nodes each side), then its XS + 1 faces,
// then its XS nodes.  One segment of 56 nodes, or two of 24 (two rows) where
// that leaves fewer lanes idle: 64 nodes are 3 x 24 on half as many waves per
// row (67 % of the lanes at work against 50 %), 61 nodes 64 % against 48 %.  The
// waves of a block share nothing and wait only for themselves.
template <int XR> struct XSeg { static constexpr int L = 64 / XR, XS = L - 8; };

// LEARN (first RK stage with the learned sensor, hybrid_auto): before phase
// 1 the wave of a row runs the learned sensor on its 64 nodes s0-4..s0+59
// (features, two BF16-MFMA layers, the flag rule; mlp_dev.h), writes the
// flags and probabilities of the nodes its faces use (s0-1..s0+55) and takes
// each face's flag from the lane of its node instead of loading it.
//
// bx, by, bz: segment, group of WAVES * XR rows, plane; sh: the block's LDS (640
// values per wave).
template <int SCH, int XR, int WAVES, bool PARTS, typename S, bool LEARN>
__device__ __forceinline__ void sweep_x(const SweepArgsT<S>& A, int bx, int by, int bz, S* sh) {
    constexpr int L = XSeg<XR>::L, XS = XSeg<XR>::XS;
    const Geo& g = A.g;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int pos = lane % L, s0 = bx * XS, k2 = bz;
    const int j = (by * WAVES + wv) * XR + lane / L;  // the lane's row
    const int n_dir = g.nx;
    const bool row = j < g.ny;
    S* w = sh + wv * 640;  // value v of lane n at w[64 v + n]

    const int jf = s0 - 1 + pos;  // the lane's face jf+1/2
    const bool fvalid = pos <= XS && jf <= n_dir - 1 && row;
    int hy = 0;
    if constexpr (LEARN) {
        static_assert(SCH == OCFD_HYBRIDAUTO && XR == 1, "the learned sensor selects hybrid_auto's schemes");
        __shared__ unsigned short sXm[WAVES][64 * mlp::LS];
        mlp::FeatIn<S> F;
        F.g = g;
        F.d = A.d; F.u = A.u; F.v = A.v; F.w = A.w; F.T = A.T;
        for (int m = 0; m < M_COUNT; m++) F.M[m] = A.M[m];
        F.p00 = A.c.p00;
        F.rama = A.c.rama;
        mlp::Lane W;
        mlp::lane_weights_packed(A.mlp.P, lane, W);
        const int sn = s0 - 4 + lane;  // this lane's node
        const int ic = sn < -1 ? -1 : (sn > n_dir - 1 ? n_dir - 1 : sn);
        const int jr = row ? j : g.ny - 1;
        float f[mlp::NF];
        mlp::features(F, ic, jr, k2, f);
        const float prob = mlp::wave_prob(f, sXm[wv], W, lane);
        const long long qn = gidx(g, ic, jr, k2);
        const int fl = mlp::flag_rule(prob, mlp::jameson_kp(F, qn, A.c.hy_i1, A.c.hy_i2), A.mlp.lo, A.mlp.hi);
        if (lane >= 3 && lane <= 3 + XS && sn == ic && row) {
            A.flag[0][qn] = (int8_t)fl;
            if (sn >= 0) {
                A.flag[1][qn] = (int8_t)fl;
                A.flag[2][qn] = (int8_t)fl;
            }
            if (A.mlp.prob) A.mlp.prob[qn] = prob;
        }
        hy = __shfl(fl, (lane + 3) & 63);  // face jf+1/2 has the flag of node jf = s0-4 + (lane+3)
    } else {
        if (SCH == OCFD_HYBRIDAUTO && fvalid) hy = A.flag[0][gidx(g, jf, j, k2)];
    }

    // ---- phase 1: split of the lane's node into LDS
    {
        const int sn = s0 - 4 + pos;
        S fp[5], fm[5];
        if (sn <= n_dir + 3 && row) {
            split_node<0>(A, sn, j, k2, fp, fm);
        } else {
#pragma unroll
            for (int m = 0; m < 5; m++) { fp[m] = S(0); fm[m] = S(0); }
        }
#pragma unroll
        for (int m = 0; m < 5; m++) {
            w[64 * m + lane] = fp[m];
            w[64 * (5 + m) + lane] = fm[m];
        }
    }
    wave_sync();

    // ---- phase 2: the lane's face (its stencil nodes are those of lanes
    // lane..lane+7 of its segment)
    S hp[5], hm[5];
#pragma unroll
    for (int m = 0; m < 5; m++) { hp[m] = S(0); hm[m] = S(0); }
    const int c = jf + 1, r = jf - n_dir;
    if constexpr (SCH == OCFD_HYBRIDAUTO) {
        int pc = 7, mc = 7;
        if (fvalid) {
            pc = case_p<SCH>(c, r, A.bl[0], A.br[0], hy);
            mc = case_m<SCH>(c, r, A.bl[0], A.br[0], hy);
        }
        const bool special = fvalid && (pc != 7 || mc != 7);
        if (fvalid && !special) {
#pragma unroll
            for (int m = 0; m < 5; m++) {
                S gp[8], gm[8];
#pragma unroll
                for (int k = 0; k < 8; k++) {
                    gp[k] = w[64 * m + lane + k];
                    gm[k] = w[64 * (5 + m) + lane + k];
                }
                hp[m] = up7_up(gp);
                hm[m] = up7_dn(gm);
            }
        }
        const unsigned long long smask = __ballot(special);
        const int nspec = __popcll(smask);
        const bool spread = nspec <= COMPACT_MAX;
        // job of this lane: value v (P of variable v < 5, M of variable v-5)
        // of the special face held by lane fl
        const bool job = spread && lane < 10 * nspec;
        const int fl = nth_lane(smask, job ? lane / 10 : 0), v = lane % 10;
        const int pcj = __shfl(pc, fl), mcj = __shfl(mc, fl);
        S res = S(0);
        if (job) {
            S gg[8];
#pragma unroll
            for (int k = 0; k < 8; k++) gg[k] = w[64 * v + fl + k];
            res = v < 5 ? recon_p_hybrid<S, double>(pcj, gg) : recon_m_hybrid<S, double>(mcj, gg);
        }
        if (special && !spread)
            face_all<S, double, SCH>([&](int vv, int k) { return w[64 * vv + lane + k]; }, c, r, A.bl[0], A.br[0], hy,
                                     S(A.c.tv_lim), S(A.c.tv_max), hp, hm);
        wave_sync();
        if (!(special && spread)) {
#pragma unroll
            for (int m = 0; m < 5; m++) {
                w[64 * m + lane] = hp[m];
                w[64 * (5 + m) + lane] = hm[m];
            }
        }
        if (job) w[64 * v + fl] = res;
    } else {
        if (fvalid)
            face_all<S, double, SCH>([&](int v, int k) { return w[64 * v + lane + k]; }, c, r, A.bl[0], A.br[0], hy,
                                     S(A.c.tv_lim), S(A.c.tv_max), hp, hm);
        wave_sync();
#pragma unroll
        for (int m = 0; m < 5; m++) {
            w[64 * m + lane] = hp[m];
            w[64 * (5 + m) + lane] = hm[m];
        }
    }
    wave_sync();

    // ---- phase 3: du at the lane's node i (faces i-1/2 and i+1/2 of lanes
    // lane and lane+1)
    const int i = s0 + pos;
    if (pos < XS && i < n_dir && row)
        put_du<0, PARTS, false>(A, i, gidx(g, i, j, k2), nullptr, [&](int v, int right) { return w[64 * v + lane + right]; });
}

// Half-node values of one direction over a tile of TX x TR nodes in x and R (1:
// y, 2: z), at index k2 of the third direction: the flux split of the tile and
// its halo along DIR (0 or R) into LDS, then the faces' P and M values over
// them, value v of face f of line a at sh[tile_at(v, f, a, TX|TR + 1)].  Lines
// of x keep their nodes together, lines of R their x neighbours: both as memory
// has them.
template <bool ALONG, int NA> __device__ __forceinline__ int tile_at(int v, int n, int a, int len) {
    return ALONG ? (v * NA + a) * len + n : (v * len + n) * NA + a;
}
template <int DIR, int R, int SCH, int TX, int TR, typename S>
__device__ __forceinline__ void tile_faces(const SweepArgsT<S>& A, int x0, int r0, int k2, S* sh) {
    constexpr bool ALONG = DIR == 0;
    static_assert((R == 1 || R == 2) && (DIR == 0 || DIR == R), "x or R");
    constexpr int NS = ALONG ? TX : TR, NA = ALONG ? TR : TX, NN = NS + 8, NF = NS + 1;
    static_assert(NF * NA <= 256, "a face per thread");
    const Geo& g = A.g;
    const int tid = threadIdx.x;
    const int a0 = ALONG ? r0 : x0, s0 = ALONG ? x0 : r0;
    const int n_dir = DIR == 0 ? g.nx : DIR == 1 ? g.ny : g.nz, n_a = !ALONG ? g.nx : R == 1 ? g.ny : g.nz;
    // (x, y, z) of position s of line a
    auto ix = [&](int s, int a) { return ALONG ? s : a; };
    auto iy = [&](int s, int a) { return R == 1 ? (ALONG ? a : s) : k2; };
    auto iz = [&](int s, int a) { return R == 2 ? (ALONG ? a : s) : k2; };
    // item idx of a tile of lines of len: its position and line
    auto pos = [](int idx, int len) { return ALONG ? idx % len : idx / NA; };
    auto line = [](int idx, int len) { return ALONG ? idx / len : idx % NA; };

    // this thread's face, j+1/2 of line a0 + al; its hybrid flag is fetched
    // first, so that its latency hides behind phase 1
    const int al = line(tid, NF), fl = pos(tid, NF), j = s0 - 1 + fl;
    const bool valid = tid < NF * NA && j <= n_dir - 1 && a0 + al < n_a;
    int hy = 0;
    if (SCH == OCFD_HYBRIDAUTO && valid) hy = A.flag[DIR][gidx(g, ix(j, a0 + al), iy(j, a0 + al), iz(j, a0 + al))];

    // ---- phase 1: split of NN x NA nodes into LDS.  FP64 issues the loads of a
    // thread's both nodes before the first split (1024x256x128 ramp: x and y
    // 1800 -> 1745 us, z 1086 -> 1077; 512x128x64: y 149 -> 146, z 142 -> 139); in FP32,
    // which would lose waves to their registers, node after node is faster (x
    // and y 180 us against 187, z 93 against 97).  The loads of y issued before
    // the faces of x cost FP64 its fifth wave or spills (1770-1950 us).
    constexpr int NT = NN * NA;
    static_assert(NT <= 512, "at most two nodes per thread");
    auto put = [&](int n, int a, bool ok, auto&& split) {
        S fp[5], fm[5];
        if (ok) {
            split(fp, fm);
        } else {
#pragma unroll
            for (int m = 0; m < 5; m++) { fp[m] = S(0); fm[m] = S(0); }
        }
#pragma unroll
        for (int m = 0; m < 5; m++) {
            sh[tile_at<ALONG, NA>(m, n, a, NN)] = fp[m];
            sh[tile_at<ALONG, NA>(5 + m, n, a, NN)] = fm[m];
        }
    };
    if constexpr (sizeof(S) == 8) {
        NodeIn<S> in[2];
        bool ok[2];
#pragma unroll
        for (int p = 0; p < 2; p++) {
            const int idx = tid + 256 * p, s = s0 - 4 + pos(idx, NN), ac = a0 + line(idx, NN);
            ok[p] = idx < NT && s <= n_dir + 3 && ac < n_a;
            if (ok[p]) in[p] = load_node<DIR>(A, ix(s, ac), iy(s, ac), iz(s, ac));
        }
#pragma unroll
        for (int p = 0; p < 2; p++) {
            const int idx = tid + 256 * p;
            if (idx < NT) put(pos(idx, NN), line(idx, NN), ok[p], [&](S* fp, S* fm) { split_node<S>(A, in[p], fp, fm); });
        }
    } else {
        for (int idx = tid; idx < NT; idx += 256) {
            const int a = line(idx, NN), n = pos(idx, NN);
            const int s = s0 - 4 + n, ac = a0 + a;
            put(n, a, s <= n_dir + 3 && ac < n_a,
                [&](S* fp, S* fm) { split_node<DIR>(A, ix(s, ac), iy(s, ac), iz(s, ac), fp, fm); });
        }
    }
    __syncthreads();

    // ---- phase 2: the thread's face
    S hp[5], hm[5];
#pragma unroll
    for (int m = 0; m < 5; m++) { hp[m] = S(0); hm[m] = S(0); }
    if (valid)
        face_all<S, double, SCH>([&](int v, int k) { return sh[tile_at<ALONG, NA>(v, fl + k, al, NN)]; }, j + 1, j - n_dir,
                                 A.bl[DIR], A.br[DIR], hy, S(A.c.tv_lim), S(A.c.tv_max), hp, hm);
    __syncthreads();
    if (tid < NF * NA) {
#pragma unroll
        for (int m = 0; m < 5; m++) {  // tile_at of the face
            sh[m * NF * NA + tid] = hp[m];
            sh[(5 + m) * NF * NA + tid] = hm[m];
        }
    }
    __syncthreads();
}

// Sweep along R of a tile, and before it (XTOO) along x, whose part of du stays
// in registers: idx = x + TX r is a thread's output node in both.  ACC: added
// to du.
template <int R, int SCH, int TX, int TR, bool XTOO, bool ACC, bool PARTS, typename S>
__device__ __forceinline__ void sweep_tile(const SweepArgsT<S>& A, int bx, int by, int bz, S* sh) {
    constexpr int NPT = (TX * TR + 255) / 256;
    const Geo& g = A.g;
    const int x0 = bx * TX, r0 = by * TR, n_r = R == 1 ? g.ny : g.nz;
    double part[NPT][5];
    auto nodes = [&](auto&& f) {
#pragma unroll
        for (int t = 0; t < NPT; t++) {
            const int idx = threadIdx.x + 256 * t;
            const int i = x0 + idx % TX, r = r0 + idx / TX;
            if (idx < TX * TR && i < g.nx && r < n_r) f(t, idx, i, r, R == 1 ? gidx(g, i, r, bz) : gidx(g, i, bz, r));
        }
    };
    if constexpr (XTOO) {
        tile_faces<0, R, SCH, TX, TR>(A, x0, r0, bz, sh);
        nodes([&](int t, int idx, int i, int, long long) {
            auto face = [&](int v, int right) { return sh[tile_at<true, TR>(v, idx % TX + right, idx / TX, TX + 1)]; };
#pragma unroll
            for (int m = 0; m < 5; m++) part[t][m] = double(du_of<0, false>(A, i, m, 0.0, face));
        });
        __syncthreads();
    } else if constexpr (ACC) {
        // fetched before the faces, so that its latency hides behind them
        nodes([&](int t, int, int, int, long long q) {
#pragma unroll
            for (int m = 0; m < 5; m++) part[t][m] = double(A.du[m * A.fs + q]);
        });
    }
    tile_faces<R, R, SCH, TX, TR>(A, x0, r0, bz, sh);
    nodes([&](int t, int idx, int, int r, long long q) {
        put_du<R, PARTS, XTOO || ACC>(A, r, q, part[t],
                                      [&](int v, int right) { return sh[v * (TR + 1) * TX + idx + right * TX]; });
    });
}


// ---------------------------------------------------------------------------
// Characteristic-space reconstruction (CHARTERIC = 1):
// OCFD_weno7_SYMBO_character_P/M_kernel and
// OCFD_HybridAuto_character_P/M_Jameson_kernel (src/OCFD_flux_charteric.cu:
// 754-908, 1000-1268).  Same three phases as the physical sweeps, on one
// tile shape for all directions; per face j+1/2 in phase 2:
//   * the face state (means of u, v, w, c and the cofactor row over nodes j
//     and j+1) gives the left and right eigenvector matrices L and R
//     (get_para_charteric_*, flux_charteric_ptoc/ctop_kernel, :321-752);
//   * the eight f+ vectors of the stencil are projected with L, the five
//     characteristic variables reconstructed with the closures of the
//     physical path, and R maps the result back; the same for f-.  A hybrid
//     face with flag 1 (UP7) stays in physical space.
// The face state, L and R are FP64 on both paths.  Phase 3 follows
// put_du_character_p/m_kernel (:16-119): with a closure on one face only, the
// boundary node of that face takes a physical-space difference of the split
// flux (OCFD_bound_character_kernel_p/m, :121-319) instead of the face
// difference, the non-reflecting zero applies only there, and the low-side
// M difference is not taken in y (the reference's test compares the y flag
// with the z value).
// ---------------------------------------------------------------------------
struct CharFace {
    double L[25], R[25];
};
__device__ __forceinline__ void char_face(double u0, double v0, double w0, double c0, double a10, double a20,
                                          double a30, double u1, double v1, double w1, double c1, double a11,
                                          double a21, double a31, double gamma, CharFace& F) {
    const double u = (u0 + u1) * 0.5, v = (v0 + v1) * 0.5, w = (w0 + w1) * 0.5, c = (c0 + c1) * 0.5;
    const double a1 = (a10 + a11) * 0.5, a2 = (a20 + a21) * 0.5, a3 = (a30 + a31) * 0.5;
    double ss = sqrt(a1 * a1 + a2 * a2 + a3 * a3);
    const double n1 = a1 / ss, n2 = a2 / ss, n3 = a3 / ss;
    double l1, l2, l3;
    if (fabs(n3) <= fabs(n2)) {
        ss = sqrt(n1 * n1 + n2 * n2);
        l1 = -n2 / ss; l2 = n1 / ss; l3 = 0.0;
    } else {
        ss = sqrt(n1 * n1 + n3 * n3);
        l1 = -n3 / ss; l2 = 0.0; l3 = n1 / ss;
    }
    const double m1 = n2 * l3 - n3 * l2, m2 = n3 * l1 - n1 * l3, m3 = n1 * l2 - n2 * l1;
    const double KK = (gamma - 1.0) / (c * c);
    const double X1 = 1.0 / (2.0 * c);
    const double un = u * n1 + v * n2 + w * n3;
    const double v2 = (u * u + v * v + w * w) * 0.5;
    double* L = F.L;
    L[0] = 1.0 - KK * v2; L[1] = KK * u; L[2] = KK * v; L[3] = KK * w; L[4] = -KK;
    L[5] = -(u * l1 + v * l2 + w * l3); L[6] = l1; L[7] = l2; L[8] = l3; L[9] = 0.0;
    L[10] = -(u * m1 + v * m2 + w * m3); L[11] = m1; L[12] = m2; L[13] = m3; L[14] = 0.0;
    L[15] = KK * v2 * 0.5 + X1 * un;
    L[16] = -X1 * n1 - KK * u * 0.5; L[17] = -X1 * n2 - KK * v * 0.5; L[18] = -X1 * n3 - KK * w * 0.5;
    L[19] = KK * 0.5;
    L[20] = L[15] - 2 * X1 * un;
    L[21] = 2 * X1 * n1 + L[16]; L[22] = 2 * X1 * n2 + L[17]; L[23] = 2 * X1 * n3 + L[18]; L[24] = L[19];
    const double H = v2 + 1.0 / KK;
    double* R = F.R;
    R[0] = 1.0; R[1] = 0.0; R[2] = 0.0; R[3] = 1.0; R[4] = 1.0;
    R[5] = u; R[6] = l1; R[7] = m1; R[8] = u - c * n1; R[9] = 2 * u - R[8];
    R[10] = v; R[11] = l2; R[12] = m2; R[13] = v - c * n2; R[14] = 2 * v - R[13];
    R[15] = w; R[16] = l3; R[17] = m3; R[18] = w - c * n3; R[19] = 2 * w - R[18];
    R[20] = v2; R[21] = u * l1 + v * l2 + w * l3; R[22] = u * m1 + v * m2 + w * m3;
    R[23] = H - c * un; R[24] = 2 * H - R[23];
}
__device__ __forceinline__ void mv5(const double* M, const double* x, double* y) {
#pragma unroll
    for (int i = 0; i < 5; i++)
        y[i] = M[5 * i] * x[0] + M[5 * i + 1] * x[1] + M[5 * i + 2] * x[2] + M[5 * i + 3] * x[3] + M[5 * i + 4] * x[4];
}

template <int DIR> struct CharTile { static constexpr int NS = 24, NA = 8; };
template <> struct CharTile<0> { static constexpr int NS = 56, NA = 4; };

// bx, by, bz: tile along and across the sweep, third index; sh and shb: the
// block's LDS.
template <int DIR, int SCH, bool ACC, typename S>
__device__ __forceinline__ void sweep_char(const SweepArgsT<S>& A, int bx, int by, int bz, S* sh,
                                           S (*shb)[10][8]) {
    constexpr int NS = CharTile<DIR>::NS, NA = CharTile<DIR>::NA, NN = NS + 8, NF = NS + 1;
    static_assert(NN * NA == 256 && NF * NA <= 256 && (DIR != 0 || (NA == 4 && NF <= 64)),
                  "one node and at most one face per thread; x: one row per wave");
    // shb: boundary differences [low/high][P 0..4, M 5..9][column]
    const Geo& g = A.g;
    const int tid = threadIdx.x;
    const int s0 = (DIR == 0 ? bx : by) * NS, a0 = (DIR == 0 ? by : bx) * NA, k2 = bz;
    const int bl = A.bl[DIR], br = A.br[DIR];
    const int n_dir = DIR == 0 ? g.nx : DIR == 1 ? g.ny : g.nz;
    const int n_acr = DIR == 0 ? g.ny : g.nx;
    auto lin = [&](int s, int a) -> long long {
        return DIR == 0 ? gidx(g, s, a, k2) : DIR == 1 ? gidx(g, a, s, k2) : gidx(g, a, k2, s);
    };
    // lanes run along x: along the sweep for x, across it for y and z
    auto at = [](int v, int n, int a) { return DIR == 0 ? (v * NA + a) * NN + n : (v * NN + n) * NA + a; };
    auto fat = [](int v, int f, int a) { return DIR == 0 ? (v * NA + a) * NF + f : (v * NF + f) * NA + a; };
    const int fyc = bl && br ? 3 : bl ? 1 : br ? 2 : 0;  // closures: both, low, high, none

    // ---- phase 1: split into LDS
    {
        const int n = DIR == 0 ? tid % NN : tid / NA, a = DIR == 0 ? tid / NN : tid % NA;
        const int s = s0 - 4 + n, ac = a0 + a;
        S fp[5], fm[5];
        if (s <= n_dir + 3 && ac < n_acr) {
            split_node<DIR>(A, DIR == 0 ? s : ac, DIR == 0 ? ac : DIR == 1 ? s : k2, DIR == 2 ? s : k2, fp, fm);
        } else {
#pragma unroll
            for (int m = 0; m < 5; m++) { fp[m] = S(0); fm[m] = S(0); }
        }
#pragma unroll
        for (int m = 0; m < 5; m++) {
            sh[at(m, n, a)] = fp[m];
            sh[at(5 + m, n, a)] = fm[m];
        }
    }
    __syncthreads();

    // ---- phase 2: one face per thread
    S hp[5], hm[5];
    // x: wave a handles row a (lane = face along the row); y, z: lanes across
    const bool fthread = DIR == 0 ? (tid & 63) < NF : tid < NF * NA;
    const int f_loc = DIR == 0 ? tid & 63 : tid / NA, a_loc = DIR == 0 ? tid >> 6 : tid % NA;
    const int j = s0 - 1 + f_loc, ac = a0 + a_loc;
    const bool fvalid = fthread && j <= n_dir - 1 && ac < n_acr;
    if (fvalid) {
        auto ld = [&](int v, int k) { return sh[at(v, f_loc + k, a_loc)]; };
        int hy = 0;
        if (SCH == OCFD_HYBRIDAUTO) hy = A.flag[DIR][lin(j, ac)];
        const int c = j + 1, r = j - n_dir;
        if (SCH == OCFD_HYBRIDAUTO && hy == 1) {
            face_all<S, double, SCH>(ld, c, r, bl, br, hy, S(A.c.tv_lim), S(A.c.tv_max), hp, hm);
        } else {
            const long long q0 = lin(j, ac), q1 = lin(j + 1, ac);
            const double rama = A.c.rama;
            const double *m1 = A.M[3 * DIR], *m2 = A.M[3 * DIR + 1], *m3 = A.M[3 * DIR + 2];
            CharFace F;
            char_face(double(A.u[q0]), double(A.v[q0]), double(A.w[q0]), sqrt(double(A.T[q0])) * rama, m1[q0],
                      m2[q0], m3[q0], double(A.u[q1]), double(A.v[q1]), double(A.w[q1]),
                      sqrt(double(A.T[q1])) * rama, m1[q1], m2[q1], m3[q1], A.c.gamma, F);
            S cs[5][8];
            double x[5], y[5], hc[5];
            S hcs[5];
#pragma unroll
            for (int k = 0; k < 8; k++) {
#pragma unroll
                for (int m = 0; m < 5; m++) x[m] = double(ld(m, k));
                mv5(F.L, x, y);
#pragma unroll
                for (int m = 0; m < 5; m++) cs[m][k] = S(y[m]);
            }
            face_all_p<S, double, SCH>([&](int v, int k) { return cs[v][k]; }, c, r, bl, br, hy,
                                       S(A.c.tv_lim), S(A.c.tv_max), hcs);
#pragma unroll
            for (int m = 0; m < 5; m++) hc[m] = double(hcs[m]);
            mv5(F.R, hc, y);
#pragma unroll
            for (int m = 0; m < 5; m++) hp[m] = S(y[m]);
#pragma unroll
            for (int k = 0; k < 8; k++) {
#pragma unroll
                for (int m = 0; m < 5; m++) x[m] = double(ld(5 + m, k));
                mv5(F.L, x, y);
#pragma unroll
                for (int m = 0; m < 5; m++) cs[m][k] = S(y[m]);
            }
            face_all_m<S, double, SCH>([&](int v, int k) { return cs[v - 5][k]; }, c, r, bl, br, hy, hcs);
#pragma unroll
            for (int m = 0; m < 5; m++) hc[m] = double(hcs[m]);
            mv5(F.R, hc, y);
#pragma unroll
            for (int m = 0; m < 5; m++) hm[m] = S(y[m]);
        }
        // physical-space differences of the boundary nodes (node j-3+k at k)
        if (j == 0 && fyc == 1) {
#pragma unroll
            for (int m = 0; m < 5; m++) {
                shb[0][m][a_loc] = ld(m, 4) - ld(m, 3);
                const S f0 = ld(5 + m, 3), f1 = ld(5 + m, 4), f2 = ld(5 + m, 5);
                shb[0][5 + m][a_loc] =
                    (f1 - S(0.5) * d_minmod2(f2 - f1, f1 - f0)) - (f0 - S(0.5) * d_minmod2(f1 - f0, f1 - f0));
            }
        }
        if (j == n_dir - 1 && fyc == 2) {
#pragma unroll
            for (int m = 0; m < 5; m++) {
                const S a = ld(m, 3), b = ld(m, 2), cc = ld(m, 1);
                shb[1][m][a_loc] = (a + S(0.5) * d_minmod2(a - b, a - b)) - (b + S(0.5) * d_minmod2(a - b, b - cc));
                shb[1][5 + m][a_loc] = ld(5 + m, 3) - ld(5 + m, 2);
            }
        }
    }
    __syncthreads();
    if (fthread) {
#pragma unroll
        for (int m = 0; m < 5; m++) {
            sh[fat(m, f_loc, a_loc)] = fvalid ? hp[m] : S(0);
            sh[fat(5 + m, f_loc, a_loc)] = fvalid ? hm[m] : S(0);
        }
    }
    __syncthreads();

    // ---- phase 3: du at nodes, P then M
    if (DIR == 0 ? (tid & 63) < NS : tid < NS * NA) {
        const int n = DIR == 0 ? tid & 63 : tid / NA, a = DIR == 0 ? tid >> 6 : tid % NA;
        const int i = s0 + n, ai = a0 + a;
        if (i < n_dir && ai < n_acr) {
            const long long q = lin(i, ai);
            const double rh = 1.0 / A.h[DIR];
            const bool lowP = fyc == 1 && i == 0, highP = fyc == 2 && i == n_dir - 1;
            const bool highM = fyc == 2 && i == n_dir - 1, lowM = fyc == 1 && i == 0 && DIR != 1;
#pragma unroll
            for (int m = 0; m < 5; m++) {
                double tP, tM;
                if (lowP) tP = A.nrp[DIR] ? 0.0 : -double(shb[0][m][a]) * rh;
                else if (highP) tP = -double(shb[1][m][a]) * rh;
                else tP = -double(sh[fat(m, n + 1, a)] - sh[fat(m, n, a)]) * rh;
                if (highM) tM = A.nrm[DIR] ? 0.0 : -double(shb[1][5 + m][a]) * rh;
                else if (lowM) tM = -double(shb[0][5 + m][a]) * rh;
                else tM = -double(sh[fat(5 + m, n + 1, a)] - sh[fat(5 + m, n, a)]) * rh;
                S* o = &A.du[m * A.fs + q];
                if constexpr (ACC) *o = S((double(*o) + tP) + tM);
                else __builtin_nontemporal_store(S(tP + tM), o);
            }
        }
    }
}

// y/z tile shapes (output nodes x columns).  FP64: 14 nodes x 16 columns
// (128-byte row segments): on the 1024x384x256 swept ramp the y sweep 3.58-3.74
// -> 3.43-3.53 ms and the z sweep 3.91-4.00 -> 3.53-3.58 ms against 28 x 8 (12 x
// 16 in between; 56 x 4, 4.4 and 6.2 ms), although it splits 1.57 nodes per
// output node against 1.29.
template <typename S> struct YZ { static constexpr int NS = 14, NA = 16; };
template <> struct YZ<float> { static constexpr int NS = 15, NA = 16; };

// ---------------------------------------------------------------------------
// Larger grids: x and y in one launch (k_sweep_tile with XTOO), z after it; or
// x, y and z by themselves, x writing du, the others adding to it.  A wave of
// the x sweep is a block of its own.
//
// x and y together move 128 B a point in FP64 instead of 248 (the primitives
// once, du written and not read back), yet take as long as the two alone where
// these run at the copy rate (1024x256x128 ramp 1.79 ms, 1.77 apart): barriers,
// LDS (busy 72 % of the cycles on the 1024x384x256 ramp) and VALU (65 %) bound the
// tile (profiles/ramp1024x384x256_sweep30_sweep_counters.md).  What they leave to
// the gradient kernel on the other stream is the gain, measured when the launch
// came: a step of 1024x256x128 19.88 -> 19.55 ms, 640x192x96 5.18 -> 5.00,
// 256x128x128 WENO7 3.08 -> 3.00 (x + y 465 -> 431 us), mixed 512x128x64 1.69 ->
// 1.61, mixed 131x99x80 0.648 -> 0.626.
// Two neighbouring faces a thread, which read 40 LDS values a face for 70,
// need 104-122 VGPRs for 76 and were slower (276 -> 310 us at 512x128x64), and so
// were more threads a block; x lines spread free of bank conflicts (18 % of the
// LDS cycles), and hybrid_auto's special faces given out over the wave as in
// sweep_x, changed nothing.
// ---------------------------------------------------------------------------
template <int SCH, int XR, typename S, bool LEARN>
__global__ void __launch_bounds__(64) k_sweep_x(SweepArgsT<S> A) {
    __shared__ S sh[640];
    const Blk B = xcd_block();
    sweep_x<SCH, XR, 1, false, S, LEARN>(A, B.x, B.y, B.z, sh);
}
template <int DIR, int SCH, bool XTOO, typename S>
__global__ void __launch_bounds__(256) k_sweep_tile(SweepArgsT<S> A) {
    constexpr int NS = YZ<S>::NS, NA = YZ<S>::NA;
    constexpr int LR = (NS + 8) * NA, LX = XTOO ? (NA + 8) * NS : 0;
    __shared__ S sh[10 * (LR > LX ? LR : LX)];
    const Blk B = xcd_block();
    sweep_tile<DIR, SCH, NA, NS, XTOO, !XTOO, false, S>(A, B.x, B.y, B.z, sh);
}
// hybrid_auto is held to 3 waves per SIMD (168 VGPRs, 8 spilled): at 2 the
// kernel is latency-bound (203x93x45, one launch: x 139 -> 111 us; y and z,
// which were at 3, 79 -> 77 and 62 -> 60; at 4 waves 124, 90, 69).  The SYMBO
// forms need 256 and would spill half of them.
template <int DIR, int SCH, typename S>
__global__ void __launch_bounds__(256, SCH == OCFD_HYBRIDAUTO ? 3 : 2) k_char(SweepArgsT<S> A) {
    using C = CharTile<DIR>;
    __shared__ S sh[10 * (C::NS + 8) * C::NA];
    __shared__ S shb[2][10][8];
    const Blk B = xcd_block();
    sweep_char<DIR, SCH, DIR != 0, S>(A, B.x, B.y, B.z, sh, shb);
}

// ---------------------------------------------------------------------------
// The three sweeps in one launch, each direction writing its part of du to
// its own five fields, which the RK stage adds: the sweeps then
// depend on nothing but the stage's state.  For small grids (sweeps_merged):
// a launch of theirs is as long as its slowest block, and three of them with
// their gaps are replaced by one (64^3: 24 + 21 + 21 us -> 48 us, 45 now, 20x16x12: 9 +
// 10 + 10 -> 10).  On larger ones it gains less than the stage pays for reading
// three parts (256x128x128: 712 -> 670 us, the stage 234 -> 297;
// 1024x256x128: 2.96 -> 2.92 ms and 2.02 -> 2.60).  Blocks in the order x, y, z;
// cutting the domain into boxes whose x, y and z blocks follow one another, for
// the Infinity Cache, was slower at every size (64^3 51-59 us, 256x128x128
// 720-860).  The SYMBO schemes are held to 4 waves per SIMD (128 VGPRs, 2
// spilled) where they would take 3: 97x61x53, 91 -> 84 us; k_sweep_tile, which
// would spill 18, is not (256x128x128: 249 us, held 299).
// ---------------------------------------------------------------------------
struct SweepGrid {
    int nt[3][3];  // tiles of a direction along x, y, z
    int run[3];    // its blocks, a multiple of 8
};
// Tile of block b of a direction: the blocks an XCD gets (every eighth) are
// neighbours, as in xcd_block(); false: a padding block.
__device__ __forceinline__ bool run_tile(unsigned b, int run, const int* nt, Blk& t) {
    const int q = (int)(b & 7u) * (run >> 3) + (int)(b >> 3);
    if (q >= nt[0] * nt[1] * nt[2]) return false;
    t.x = q % nt[0];
    t.y = (q / nt[0]) % nt[1];
    t.z = q / (nt[0] * nt[1]);
    return true;
}
constexpr int XWAVES = 4;  // waves of an x block here
template <int SCH, int XR, typename S>
__global__ void __launch_bounds__(256, SCH == OCFD_WENO7_SYMBO || SCH == OCFD_WENO7_SYMBO_LIM ? 4 : 1) k_sweeps(SweepArgsT<S> A, SweepGrid G) {
    constexpr int NS = YZ<S>::NS, NA = YZ<S>::NA;
    constexpr int LDS_YZ = 10 * (NS + 8) * NA, LDS_X = 640 * XWAVES;
    __shared__ S sh[LDS_YZ > LDS_X ? LDS_YZ : LDS_X];
    unsigned b = blockIdx.x;
    Blk t;
    if (b < (unsigned)G.run[0]) {
        if (run_tile(b, G.run[0], G.nt[0], t)) sweep_x<SCH, XR, XWAVES, true, S, false>(A, t.x, t.y, t.z, sh);
        return;
    }
    b -= G.run[0];
    if (b < (unsigned)G.run[1]) {
        if (run_tile(b, G.run[1], G.nt[1], t)) sweep_tile<1, SCH, NA, NS, false, false, true, S>(A, t.x, t.y, t.z, sh);
        return;
    }
    b -= G.run[1];
    if (run_tile(b, G.run[2], G.nt[2], t)) sweep_tile<2, SCH, NA, NS, false, false, true, S>(A, t.x, t.y, t.z, sh);
}

int tiles(int n, int t) { return (n + t - 1) / t; }
// Two segments per wave where a row's waves then come to less than half.
bool two_segments(const Geo& g) { return tiles(g.nx, XSeg<2>::XS) < 2 * tiles(g.nx, XSeg<1>::XS); }

// first: 0 for all three directions, 1 for y and z.
template <int SCH, typename S>
void launch_merged(const SweepArgsT<S>& a, int first, hipStream_t st) {
    const Geo& g = a.g;
    constexpr int NS = YZ<S>::NS, NA = YZ<S>::NA;
    const bool two = two_segments(g);
    const int xs = two ? XSeg<2>::XS : XSeg<1>::XS, rows = XWAVES * (two ? 2 : 1);
    const SweepGrid z{};
    SweepGrid G = z;
    const int nt[3][3] = {{tiles(g.nx, xs), tiles(g.ny, rows), g.nz},
                          {tiles(g.nx, NA), tiles(g.ny, NS), g.nz},
                          {tiles(g.nx, NA), tiles(g.nz, NS), g.ny}};
    unsigned nb = 0;
    for (int d = first; d < 3; d++) {
        for (int q = 0; q < 3; q++) G.nt[d][q] = nt[d][q];
        G.run[d] = tiles(nt[d][0] * nt[d][1] * nt[d][2], 8) * 8;
        nb += G.run[d];
    }
    if (two) hipLaunchKernelGGL((k_sweeps<SCH, 2, S>), dim3(nb), dim3(256), 0, st, a, G);
    else hipLaunchKernelGGL((k_sweeps<SCH, 1, S>), dim3(nb), dim3(256), 0, st, a, G);
}

// -1: no kernel for this scheme and direction.
template <int SCH, typename S>
int launch_scheme(int dir, const SweepArgsT<S>& a, hipStream_t st) {
    const Geo& g = a.g;
    constexpr int NS = YZ<S>::NS, NA = YZ<S>::NA;
    if (dir == SWEEP_XY) {
        hipLaunchKernelGGL((k_sweep_tile<1, SCH, true, S>), dim3(tiles(g.nx, NA), tiles(g.ny, NS), g.nz), dim3(256), 0, st,
                           a);
        return 0;
    }
    if (dir == SWEEP_ALL || dir == SWEEP_YZ) {
        launch_merged<SCH>(a, dir == SWEEP_YZ, st);
        return 0;
    }
    if (dir == 2) {
        hipLaunchKernelGGL((k_sweep_tile<2, SCH, false, S>), dim3(tiles(g.nx, NA), tiles(g.nz, NS), g.ny), dim3(256), 0, st,
                           a);
        return 0;
    }
    if constexpr (SCH == OCFD_HYBRIDAUTO) {  // the one scheme for which x and y may be apart (sweeps_xy)
        if (dir == 1) {
            hipLaunchKernelGGL((k_sweep_tile<1, SCH, false, S>), dim3(tiles(g.nx, NA), tiles(g.ny, NS), g.nz), dim3(256), 0,
                               st, a);
            return 0;
        }
        if (dir == 0) {
            const bool two = !a.mlp.P && two_segments(g);
            const dim3 grid = two ? dim3(tiles(g.nx, XSeg<2>::XS), tiles(g.ny, 2), g.nz)
                                  : dim3(tiles(g.nx, XSeg<1>::XS), g.ny, g.nz);
            if (a.mlp.P) hipLaunchKernelGGL((k_sweep_x<SCH, 1, S, true>), grid, dim3(64), 0, st, a);
            else if (two) hipLaunchKernelGGL((k_sweep_x<SCH, 2, S, false>), grid, dim3(64), 0, st, a);
            else hipLaunchKernelGGL((k_sweep_x<SCH, 1, S, false>), grid, dim3(64), 0, st, a);
            return 0;
        }
    }
    return -1;
}
template <int SCH, typename S>
void launch_char_scheme(int dir, const SweepArgsT<S>& a, hipStream_t st) {
    const Geo& g = a.g;
    if (dir == 0)
        hipLaunchKernelGGL((k_char<0, SCH, S>), dim3(tiles(g.nx, CharTile<0>::NS), tiles(g.ny, CharTile<0>::NA), g.nz),
                           dim3(256), 0, st, a);
    else if (dir == 1)
        hipLaunchKernelGGL((k_char<1, SCH, S>), dim3(tiles(g.nx, CharTile<1>::NA), tiles(g.ny, CharTile<1>::NS), g.nz),
                           dim3(256), 0, st, a);
    else
        hipLaunchKernelGGL((k_char<2, SCH, S>), dim3(tiles(g.nx, CharTile<2>::NA), tiles(g.nz, CharTile<2>::NS), g.ny),
                           dim3(256), 0, st, a);
}

}  // namespace

// Points up to which the three sweeps of a stage run in one launch, on one
// stream with the rest of the stage: 20x16x12 140 -> 63 us a step, 64^3
// 296 -> 244, 61x47x39 161 -> 114, 97x61x53 540 -> 510; above, 131x99x80 mixed
// 660 -> 667, 256x128x128 3168 -> 3300.
bool sweeps_merged(const Geo& g) { return (long long)g.nx * g.ny * g.nz <= 500000; }

// Whether x and y of a larger grid are one launch.  They are for every scheme
// but one: a step of 131x99x80 to 512x256x128, FP64 and mixed, is shorter by 3-7 %
// with UP7, 4-7 with NND2, 2-4 with WENO5, 1-4 with WENO7.  hybrid_auto in FP64
// keeps them apart between 1.5 and 10 million points: with shocks in the flow
// the x sweep by itself spreads its few WENO faces over the wave, which the
// tiles do not (ramps, ms a step apart and together: 2.1 M points 1.402 and 1.421,
// 4.2 M 2.68 and 2.74, 8.4 M 5.01 and 5.03); a launch and its tail less count
// for more below (1.0 M 0.894 and 0.868, still 1.091 and 1.039 at 1.51 M), du's
// bytes above (12.6 M 7.45 and 7.26, 16.8 M 9.99 and 9.67).  The flow is not
// known here: without shocks together is shorter there too (box, 4.2 M 2.37 and
// 2.29).
template <typename S> bool sweeps_xy(int scheme, const Geo& g) {
    const long long n = (long long)g.nx * g.ny * g.nz;
    return scheme != OCFD_HYBRIDAUTO || sizeof(S) == 4 || n < 1500000 || n > 10000000;
}
template bool sweeps_xy<double>(int, const Geo&);
template bool sweeps_xy<float>(int, const Geo&);

template <typename S>
int launch_sweep(int scheme, int dir, const SweepArgsT<S>& a, hipStream_t st) {
    switch (scheme) {
    case OCFD_UP7: return launch_scheme<OCFD_UP7>(dir, a, st);
    case OCFD_WENO5: return launch_scheme<OCFD_WENO5>(dir, a, st);
    case OCFD_WENO7: return launch_scheme<OCFD_WENO7>(dir, a, st);
    case OCFD_WENO7_SYMBO: return launch_scheme<OCFD_WENO7_SYMBO>(dir, a, st);
    case OCFD_WENO7_SYMBO_LIM: return launch_scheme<OCFD_WENO7_SYMBO_LIM>(dir, a, st);
    case OCFD_NND2: return launch_scheme<OCFD_NND2>(dir, a, st);
    case OCFD_OMP6_HR: return launch_scheme<OCFD_OMP6_HR>(dir, a, st);
    case OCFD_OMP6_LD: return launch_scheme<OCFD_OMP6_LD>(dir, a, st);
    case OCFD_OMP6_CD8: return launch_scheme<OCFD_OMP6_CD8>(dir, a, st);
    case OCFD_HYBRIDAUTO: return launch_scheme<OCFD_HYBRIDAUTO>(dir, a, st);
    }
    return -1;
}
template int launch_sweep<double>(int, int, const SweepArgsT<double>&, hipStream_t);
template int launch_sweep<float>(int, int, const SweepArgsT<float>&, hipStream_t);

template <typename S>
int launch_sweep_char(int scheme, int dir, const SweepArgsT<S>& a, hipStream_t st) {
    switch (scheme) {
    case OCFD_WENO7_SYMBO: launch_char_scheme<OCFD_WENO7_SYMBO>(dir, a, st); break;
    case OCFD_WENO7_SYMBO_LIM: launch_char_scheme<OCFD_WENO7_SYMBO_LIM>(dir, a, st); break;
    case OCFD_HYBRIDAUTO: launch_char_scheme<OCFD_HYBRIDAUTO>(dir, a, st); break;
    default: return -1;
    }
    return 0;
}
template int launch_sweep_char<double>(int, int, const SweepArgsT<double>&, hipStream_t);
template int launch_sweep_char<float>(int, int, const SweepArgsT<float>&, hipStream_t);
