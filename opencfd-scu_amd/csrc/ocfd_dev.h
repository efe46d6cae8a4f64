// ocfd_dev.h - device-side definitions shared by the gfx950 kernels.
//
// Layout: every field (primitives, pressure, metrics, conserved state, RHS,
// viscous fluxes) is one padded box of (nx+8) x (ny+8) x (nz+8) doubles with
// the reference's LAP=4 ghost layers (head/cuda_utility.h:16-27), x fastest.
// The row pitch ldx is a multiple of 16 doubles and the base pointer is offset
// so that interior x=0 of every row is 128-byte aligned.  Because all fields
// share one layout, a grid point has the same linear index in every array.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <type_traits>

#define OCFD_LAPD 4

struct Geo {
    int nx, ny, nz;       // interior sizes
    int ldx, ldy;         // row pitch (elements), rows per plane (ny+8)
    long long sz;         // plane stride = ldx*ldy
    long long off0;       // linear index of interior (0,0,0)
    double hx, hy, hz;
};

// Linear index of interior point (i,j,k); ghosts are i<0 or i>=nx etc.
__host__ __device__ __forceinline__ long long gidx(const Geo& g, int i, int j, int k) {
    return g.off0 + (long long)i + (long long)g.ldx * ((long long)j + (long long)g.ldy * (long long)k);
}

// XCD-aware tile order.  Workgroups are dispatched round-robin over the 8
// XCDs (each with its own L2), so consecutive block indices land on
// different L2s and neighbouring tiles - which share 128-byte lines and halo
// rows - would each fetch them from HBM.  xcd_block() maps the hardware block
// index to a logical tile index such that every XCD walks one contiguous run
// of tiles (x fastest): neighbours then share that XCD's L2.  It is a
// permutation of [0, nblocks) whatever the hardware mapping is.
struct Blk { int x, y, z; };
__device__ __forceinline__ Blk xcd_block() {
    const unsigned gx = gridDim.x, gy = gridDim.y;
    const unsigned nb = gx * gy * gridDim.z;
    const unsigned b = blockIdx.x + gx * (blockIdx.y + gy * blockIdx.z);
#ifdef OCFD_NO_XCD_REMAP
    const unsigned t = b;  // hardware order (for comparison builds)
    (void)nb;
#else
    const unsigned q = nb >> 3, r = nb & 7u, x = b & 7u, s = b >> 3;
    const unsigned t = (x < r ? x * (q + 1) : r * (q + 1) + (x - r) * q) + s;
#endif
    Blk o;
    o.x = (int)(t % gx);
    o.y = (int)((t / gx) % gy);
    o.z = (int)(t / (gx * gy));
    return o;
}

// Raw buffer access to a range of one array (a z plane of a field): the base
// is a scalar resource and the lane's address one 32-bit byte offset, where a
// plain pointer costs two registers and a 64-bit add per access.  Loads past
// the range return 0 and stores past it are dropped, so lanes without a point
// take the offset BUF_NONE instead of a branch.
constexpr unsigned BUF_NONE = 0x80000000u;  // past every range: a plane holds at most 2^31 / 16 elements
enum { BUF_PLAIN = 0, BUF_STREAM = 2 };     // cache policy: BUF_STREAM = non-temporal
template <typename T> struct Buf {
    __amdgpu_buffer_rsrc_t r;
    __device__ __forceinline__ Buf(const T* base, long long elems)
        : r(__builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(base), 0, (int)(elems * (long long)sizeof(T)), 0x00020000)) {}
    template <int AUX = BUF_PLAIN> __device__ __forceinline__ T ld(unsigned off) const {
        if constexpr (sizeof(T) == 8) return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b64(r, (int)off, 0, AUX));
        else return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b32(r, (int)off, 0, AUX));
    }
    template <int AUX = BUF_PLAIN> __device__ __forceinline__ void st(unsigned off, T v) const {
        if constexpr (sizeof(T) == 8) {
            typedef unsigned u2 __attribute__((ext_vector_type(2)));
            __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u2, v), r, (int)off, 0, AUX);
        } else {
            __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), r, (int)off, 0, AUX);
        }
    }
};

// The same value, opaque to the optimiser.  Taken anew in each step of a march,
// a field stride keeps the addresses of a step's planes (a group's base plus a
// multiple of the stride, scalar adds) from being hoisted out of the loop,
// where two dozen of them overflow the scalar registers.
__device__ __forceinline__ long long opaque(long long v) {
    asm volatile("" : "+s"(v));
    return v;
}

// The 10 metric fields kept on the device (cofactors and Ajac,
// src/OCFD_Comput_Jacobian3d.cu:285-295).
enum { M_KX = 0, M_KY, M_KZ, M_IX, M_IY, M_IZ, M_SX, M_SY, M_SZ, M_JAC, M_COUNT };

struct Consts {
    double gamma, ama, cv, cp, tsb, amu_c0, tmp0, split_c1, split_c3, vis_c;
    double epsl_sw, p00;                     // p00 = 1/(gamma*Ma^2)
    double rama;                             // 1/Ma
    double hy_i1, hy_i2;                     // HY_DP_INTV
    double tv_lim, tv_max;                   // WENO_TV_Limiter / WENO_TV_MAX
};

// --------------------------------------------------------------------------
// Half-node reconstructions (device restatement of src/OCFD_Schemes.cu and
// src/OCFD_bound_Scheme.cu).  s points at the first node the reference kernel
// gathers; expressions keep the reference operand order.
// --------------------------------------------------------------------------
template <typename R> __device__ __forceinline__ R d_sgn1(R x) { return x >= R(0) ? R(1) : R(-1); }
template <typename R> __device__ __forceinline__ R d_minmod2(R a, R b) {
    return R(0.5) * (d_sgn1(a) + d_sgn1(b)) * fmin(fabs(a), fabs(b));
}
template <typename R> __device__ __forceinline__ R d_minmod4(R a, R b, R c, R d) {
    R m = R(0.5) * (d_sgn1(a) + d_sgn1(b));
    m = m * fabs(R(0.5) * (d_sgn1(a) + d_sgn1(c)));
    m = m * fabs(R(0.5) * (d_sgn1(a) + d_sgn1(d)));
    return m * fmin(fmin(a, b), fmin(c, d));
}

// num / den of weights and weighted values, den > 0 and far from the ends of
// the range: reciprocal by two Newton steps from the hardware's estimate and
// one product (6 instructions; the IEEE division with its scaling, 12).
// The quotients here are corrections to a nodal value, so their last ulp is
// far below the ulp of the result.
__device__ __forceinline__ double weight_div(double num, double den) {
    double y = __builtin_amdgcn_rcp(den);
    y = fma(fma(-den, y, 1.0), y, y);
    y = fma(fma(-den, y, 1.0), y, y);
    return num * y;
}

// WENO7 upwind (P) half-node value from nodes s[0..6] (src/OCFD_Schemes.cu:616-663).
// R: type of the stencil values and smoothness indicators; W: type of the
// epsilon/weight arithmetic (the mixed-precision path keeps W = double).
//
// The reference's sums over the stencil values, regrouped over the
// differences the four sub-stencils share: e_i = s_{i+1} - s_i, D_i = e_i -
// e_{i-1}, T_k = D_{k+2} - D_{k+1}.  Its a (first derivative at node 3), b =
// 6 beta and c = 6 T are
//   a = 6 e2 + 3 D2 + 2 T0, 3 (e2 + e3) - T1, 3 (e2 + e3) - T2, 6 e3 - 3 D4 + 2 T3
//   beta = D2 + T0, D3, D4, D4 - T3   (its stencil 2 takes the node i+1)
// its indicator 960 a^2 + 1040 b^2 + 1043 c^2 + 80 a c is 480 (a (2 a + T) +
// 78 beta^2 + 78.225 T^2), and its candidates q_k are 12 s3 + delta_k.  The
// weights do not change when epsilon and the indicators are divided by 480.
// 88 instructions per value against about 130; cancellation happens in the
// differences, which are exact for neighbouring values, and the weighted part
// is a correction to s3: the error against 64-bit (and on the FP32 path
// against FP64) values is no larger.
template <typename R, typename W = R> __device__ __forceinline__ R weno7_up(const R* s) {
    const R e0 = s[1] - s[0], e1 = s[2] - s[1], e2 = s[3] - s[2], e3 = s[4] - s[3], e4 = s[5] - s[4], e5 = s[6] - s[5];
    const R D1 = e1 - e0, D2 = e2 - e1, D3 = e3 - e2, D4 = e4 - e3, D5 = e5 - e4;
    const R T0 = D2 - D1, T1 = D3 - D2, T2 = D4 - D3, T3 = D5 - D4;
    const R m3 = R(3) * (e2 + e3);
    const W e = W(3.456e-4 / 480.0);
    auto ind = [&](R a, R be, R T) {  // epsilon + indicator, squared
        W q;
        if constexpr (std::is_same<R, W>::value)
            q = fma(a, fma(R(2), a, T), fma(R(78) * be, be, fma(R(78.225) * T, T, e)));
        else
            q = e + W(fma(a, fma(R(2), a, T), fma(R(78) * be, be, R(78.225) * T * T)));
        return q * q;
    };
    const W q0 = ind(fma(R(2), T0, fma(R(3), D2, R(6) * e2)), D2 + T0, T0);
    const W q1 = ind(m3 - T1, D3, T1);
    const W q2 = ind(m3 - T2, D4, T2);
    const W q3 = ind(fma(R(2), T3, fma(R(-3), D4, R(6) * e3)), D4 - T3, T3);
    const W q01 = q0 * q1, q23 = q2 * q3;
    const W w0 = q1 * q23, w1 = W(12) * q0 * q23, w2 = W(18) * q01 * q3, w3 = W(4) * q01 * q2;
    const W d0 = W(fma(R(13), e2, fma(R(-10), e1, R(3) * e0)));
    const W d1 = W(fma(R(3), e3, fma(R(4), e2, -e1)));
    const W d2 = W(fma(R(6), e3, e2 - e4));
    const W d3 = W(fma(R(9), e3, fma(R(-4), e4, e5)));
    const W num = fma(w3, d3, fma(w2, d2, fma(w1, d1, w0 * d0)));
    return R(W(s[3]) + weight_div(num, W(12) * ((w0 + w1) + (w2 + w3))));
}
// WENO7 M side: the same reconstruction on the mirrored stencil
// (src/OCFD_Schemes.cu:692-741); s[0..6].
template <typename R, typename W = R> __device__ __forceinline__ R weno7_dn(const R* s) {
    R m[7] = {s[6], s[5], s[4], s[3], s[2], s[1], s[0]};
    return weno7_up<R, W>(m);
}

// UP7 (src/OCFD_Schemes.cu:865-931), its coefficients already divided by 420.
template <typename R> __device__ __forceinline__ R up7_up(const R* s) {
    return R(-3.0 / 420.0) * s[0] + R(25.0 / 420.0) * s[1] + R(-101.0 / 420.0) * s[2] + R(319.0 / 420.0) * s[3] +
           R(214.0 / 420.0) * s[4] + R(-38.0 / 420.0) * s[5] + R(4.0 / 420.0) * s[6];
}
template <typename R> __device__ __forceinline__ R up7_dn(const R* s) {  // s[1..7]
    return R(-3.0 / 420.0) * s[7] + R(25.0 / 420.0) * s[6] + R(-101.0 / 420.0) * s[5] + R(319.0 / 420.0) * s[4] +
           R(214.0 / 420.0) * s[3] + R(-38.0 / 420.0) * s[2] + R(4.0 / 420.0) * s[1];
}

// WENO5 Jiang-Shu (src/OCFD_Schemes.cu:1118-1210) and the one-sided subsets
// used by the closures (src/OCFD_bound_Scheme.cu:557-735).
template <typename R> __device__ __forceinline__ R w5_beta_l(const R* s) {  // stencil s0..s2 (leftmost)
    R t = s[0] - R(2) * s[1] + s[2], u = s[0] - R(4) * s[1] + R(3) * s[2];
    R S = R(13) * t * t; S += R(3) * u * u; return S;
}
template <typename R> __device__ __forceinline__ R w5_beta_c(const R* s) {  // s1..s3
    R t = s[1] - R(2) * s[2] + s[3], u = s[1] - s[3];
    R S = R(13) * t * t; S += R(3) * u * u; return S;
}
template <typename R> __device__ __forceinline__ R w5_beta_r(const R* s) {  // s2..s4
    R t = s[2] - R(2) * s[3] + s[4], u = R(3) * s[2] - R(4) * s[3] + s[4];
    R S = R(13) * t * t; S += R(3) * u * u; return S;
}
template <typename R, typename W = R> __device__ __forceinline__ R weno5_up(const R* s) {
    const W e = W(12.0) * W(1e-6);  // 12.0*ep with ep = 1e-6, as the reference writes it
    const W S0 = w5_beta_r(s), S1 = w5_beta_c(s), S2 = w5_beta_l(s);
    R q03 = R(2) * s[2] + R(5) * s[3] - s[4];
    R q13 = -s[1] + R(5) * s[2] + R(2) * s[3];
    R q23 = R(2) * s[0] - R(7) * s[1] + R(11) * s[2];
    W a0 = W(3) * ((e + S1) * (e + S1)) * ((e + S2) * (e + S2));
    W a1 = W(6) * ((e + S0) * (e + S0)) * ((e + S2) * (e + S2));
    W a2 = ((e + S0) * (e + S0)) * ((e + S1) * (e + S1));
    return R((a0 * W(q03) + a1 * W(q13) + a2 * W(q23)) / (W(6) * (a0 + a1 + a2)));
}
template <typename R, typename W = R> __device__ __forceinline__ R weno5_dn(const R* s) {
    R m[5] = {s[4], s[3], s[2], s[1], s[0]};
    return weno5_up<R, W>(m);
}
template <typename R, typename W = R> __device__ __forceinline__ R weno5_up_left(const R* s) {  // OCFD_weno5_kernel_P_left
    const W e = W(12.0) * W(1e-6);  // 12.0*ep with ep = 1e-6, as the reference writes it
    const W S0 = w5_beta_r(s);
    W a0 = W(1) / ((e + S0) * (e + S0));
    return R(a0 * W(R(2) * s[2] + R(5) * s[3] - s[4]) / (W(6) * a0));
}
template <typename R, typename W = R> __device__ __forceinline__ R weno5_up_leftplus(const R* s) {
    const W e = W(12.0) * W(1e-6);  // 12.0*ep with ep = 1e-6, as the reference writes it
    const W S0 = w5_beta_r(s), S1 = w5_beta_c(s);
    W a0 = W(3) / ((e + S0) * (e + S0));
    W a1 = W(6) / ((e + S1) * (e + S1));
    R q03 = R(2) * s[2] + R(5) * s[3] - s[4];
    R q13 = -s[1] + R(5) * s[2] + R(2) * s[3];
    return R((a0 * W(q03) + a1 * W(q13)) / (W(6) * (a0 + a1)));
}
template <typename R, typename W = R> __device__ __forceinline__ R weno5_up_rightplus(const R* s) {
    const W e = W(12.0) * W(1e-6);  // 12.0*ep with ep = 1e-6, as the reference writes it
    const W S1 = w5_beta_c(s), S2 = w5_beta_l(s);
    W a1 = W(6) / ((e + S1) * (e + S1));
    W a2 = W(1) / ((e + S2) * (e + S2));
    R q13 = -s[1] + R(5) * s[2] + R(2) * s[3];
    R q23 = R(2) * s[0] - R(7) * s[1] + R(11) * s[2];
    return R((a1 * W(q13) + a2 * W(q23)) / (W(6) * (a1 + a2)));
}
template <typename R, typename W = R> __device__ __forceinline__ R weno5_dn_left(const R* s) {  // OCFD_weno5_kernel_M_left
    R m[5] = {s[4], s[3], s[2], s[1], s[0]};
    const W e = W(12.0) * W(1e-6);  // 12.0*ep with ep = 1e-6, as the reference writes it
    const W S2 = w5_beta_l(m);
    W a2 = W(1) / ((e + S2) * (e + S2));
    return R(a2 * W(R(2) * m[0] - R(7) * m[1] + R(11) * m[2]) / (W(6) * a2));
}
template <typename R, typename W = R> __device__ __forceinline__ R weno5_dn_leftplus(const R* s) {
    R m[5] = {s[4], s[3], s[2], s[1], s[0]};
    return weno5_up_rightplus<R, W>(m);
}
template <typename R, typename W = R> __device__ __forceinline__ R weno5_dn_rightplus(const R* s) {
    R m[5] = {s[4], s[3], s[2], s[1], s[0]};
    return weno5_up_leftplus<R, W>(m);
}

// WENO7-SYMBO (src/OCFD_Schemes.cu:391-589); P side with optional TV
// limiter; the M side never takes the linear branch (TVmin stays 0).
// Regrouped over shared differences like weno7_up: its indicators 720 t^2 +
// 780 b^2 + 781 c^2 are 720 (a^2 + 39 beta^2 + 39.05 T^2), with a, beta, T of
// stencils 0..3 as there and, for stencil 4, a = 26 e4 - 31 e5 + 11 e6, beta =
// D5 - 2 T4.
template <typename R, typename W = R> __device__ __forceinline__ R symbo_core(const R* s, bool linear) {
    const R e0 = s[1] - s[0], e1 = s[2] - s[1], e2 = s[3] - s[2], e3 = s[4] - s[3], e4 = s[5] - s[4], e5 = s[6] - s[5],
            e6 = s[7] - s[6];
    W w0, w1, w2, w3, w4;
    if (linear) {
        w0 = W(0.0401954833730); w1 = W(0.2493800006710); w2 = W(0.4802686256260);
        w3 = W(0.2009775476730); w4 = W(0.0291783426580);
    } else {
        const R D1 = e1 - e0, D2 = e2 - e1, D3 = e3 - e2, D4 = e4 - e3, D5 = e5 - e4, D6 = e6 - e5;
        const R T0 = D2 - D1, T1 = D3 - D2, T2 = D4 - D3, T3 = D5 - D4, T4 = D6 - D5;
        const R m3 = R(3) * (e2 + e3);
        const W e = W(2.592e-6 / 720.0);
        auto ind = [&](R a, R be, R T) {  // epsilon + indicator
            if constexpr (std::is_same<R, W>::value) return fma(a, a, fma(R(39) * be, be, fma(R(39.05) * T, T, e)));
            else return e + W(fma(a, a, fma(R(39) * be, be, R(39.05) * T * T)));
        };
        const W q0 = ind(fma(R(2), T0, fma(R(3), D2, R(6) * e2)), D2 + T0, T0);
        const W q1 = ind(m3 - T1, D3, T1);
        const W q2 = ind(m3 - T2, D4, T2);
        const W q3 = ind(fma(R(2), T3, fma(R(-3), D4, R(6) * e3)), D4 - T3, T3);
        W q4 = ind(fma(R(11), e6, fma(R(-31), e5, R(26) * e4)), fma(R(-2), T4, D5), T4);
        q4 = fmax(fmax(fmax(q0, q1), fmax(q2, q3)), q4);
        const W q01 = q0 * q1, q34 = q3 * q4, q234 = q2 * q34, q012 = q01 * q2;
        w0 = W(0.0401954833730) * q1 * q234;
        w1 = W(0.2493800006710) * q0 * q234;
        w2 = W(0.4802686256260) * q01 * q34;
        w3 = W(0.2009775476730) * q012 * q4;
        w4 = W(0.0291783426580) * q012 * q3;
    }
    const W d0 = W(fma(R(13), e2, fma(R(-10), e1, R(3) * e0)));
    const W d1 = W(fma(R(3), e3, fma(R(4), e2, -e1)));
    const W d2 = W(fma(R(6), e3, e2 - e4));
    const W d3 = W(fma(R(9), e3, fma(R(-4), e4, e5)));
    const W d4 = W(fma(R(12), e3, fma(R(-13), e4, fma(R(10), e5, R(-3) * e6))));
    const W num = fma(w4, d4, fma(w3, d3, fma(w2, d2, fma(w1, d1, w0 * d0))));
    return R(W(s[3]) + weight_div(num, W(12) * (((w0 + w1) + (w2 + w3)) + w4)));
}
template <typename R, typename W = R> __device__ __forceinline__ R symbo_up(const R* s, int lmt, R tvlim, R tvmax) {
    bool lin = false;
    if (lmt) {
        R a0 = fabs(s[1] - s[0]) + fabs(s[2] - s[1]) + fabs(s[3] - s[2]);
        R a1 = fabs(s[2] - s[1]) + fabs(s[3] - s[2]) + fabs(s[4] - s[3]);
        R a2 = fabs(s[3] - s[2]) + fabs(s[4] - s[3]) + fabs(s[5] - s[4]);
        R a3 = fabs(s[4] - s[3]) + fabs(s[5] - s[4]) + fabs(s[6] - s[5]);
        R a4 = fabs(s[5] - s[4]) + fabs(s[6] - s[5]) + fabs(s[7] - s[6]);
        R tvmin = fmin(fmin(fmin(a0, a1), fmin(a2, a3)), a4);
        R tvmx = fmax(fmax(fmax(a0, a1), fmax(a2, a3)), a4);
        lin = (tvmx < tvlim * tvmin) && (tvmx < tvmax);
    } else {
        lin = (R(1) < tvlim * R(0)) && (R(1) < tvmax);
    }
    return symbo_core<R, W>(s, lin);
}
template <typename R, typename W = R> __device__ __forceinline__ R symbo_dn(const R* s) {
    R m[8] = {s[7], s[6], s[5], s[4], s[3], s[2], s[1], s[0]};
    return symbo_core<R, W>(m, false);
}

// OMP6 (src/OCFD_Schemes.cu:936-1092).  The M limiter is kept as in the
// reference (it is not the mirror image of the P limiter).
template <typename R> __device__ __forceinline__ void omp6_mn(int fl, R& mid, R& m) {
    R mm, nn;
    if (fl == 1) { mm = R(0.001); nn = R(0); }
    else if (fl == 2) { mm = R(0); nn = R(-1.0 / 140.0); }
    else { mm = R(0.015); nn = R(0); }
    mid = R(0.5) * (mm + nn);
    m = R(0.5) * (mm - nn);
}
template <typename R> __device__ __forceinline__ R omp6_lin(const R* s, R mid, R m) {
    return (R(60) * mid * s[7] + (R(1) - R(60) * m - R(360) * mid) * s[6] +
            (R(-8) + R(360) * m + R(900) * mid) * s[5] + (R(37) - R(900) * m - R(1200) * mid) * s[4] +
            (R(37) + R(1200) * m + R(900) * mid) * s[3] + (R(-8) - R(900) * m - R(360) * mid) * s[2] +
            (R(1) + R(360) * m + R(60) * mid) * s[1] - R(60) * m * s[0]) / R(60);
}
template <typename R> __device__ __forceinline__ R omp6_up(int fl, const R* s) {
    R mid, m, n;
    omp6_mn(fl, mid, m);
    mid = omp6_lin(s, mid, m);
    m = s[3] + d_minmod2(s[4] - s[3], s[3] - s[2]);
    if ((mid - s[3]) * (mid - m) >= R(1e-10)) {
        m = s[2] + s[4] - R(2) * s[3];
        n = s[3] + s[5] - R(2) * s[4];
        R t = R(0.5) * (s[3] + s[4]) - R(0.5) * d_minmod4(R(4) * m - n, R(4) * n - m, n, m);
        R nb = s[1] + s[3] - R(2) * s[2];
        R t1 = s[3] + R(0.5) * (s[3] - s[2]) + R(4) * d_minmod4(R(4) * nb - m, R(4) * m - nb, m, nb) / R(3);
        R lo = fmax(fmin(fmin(s[3], s[4]), t), fmin(fmin(s[3], s[3] + R(4) * (s[3] - s[2])), t1));
        R hi = fmin(fmax(s[4], fmax(s[3], t)), fmax(fmax(s[3], s[3] + R(4) * (s[3] - s[2])), t1));
        mid = mid + d_minmod2(hi - mid, lo - mid);
    }
    return mid;
}
template <typename R> __device__ __forceinline__ R omp6_dn(int fl, const R* s) {
    R mid, m, n;
    omp6_mn(fl, mid, m);
    R rv[8] = {s[7], s[6], s[5], s[4], s[3], s[2], s[1], s[0]};
    mid = omp6_lin(rv, mid, m);
    m = s[4] + d_minmod2(s[3] - s[4], s[4] - s[5]);
    if ((mid - s[4]) * (mid - m) >= R(1e-10)) {
        m = s[5] + s[3] - R(2) * s[4];
        n = s[4] + s[2] - R(2) * s[3];
        R t = R(0.5) * (s[4] + s[3]) - R(0.5) * d_minmod4(R(4) * m - n, R(4) * n - m, n, m);
        R nb = s[6] + s[4] - R(2) * s[5];
        R t1 = s[4] + R(0.5) * (s[4] - s[3]) + R(4) * d_minmod4(R(4) * nb - m, R(4) * m - nb, m, nb) / R(3);
        R lo = fmax(fmin(fmin(s[5], s[3]), t), fmin(fmin(s[4], s[4] + R(4) * (s[4] - s[5])), t1));
        R hi = fmin(fmax(s[3], fmax(s[4], t)), fmax(fmax(s[4], s[4] + R(4) * (s[4] - s[5])), t1));
        mid = mid + d_minmod2(hi - mid, lo - mid);
    }
    return mid;
}

// NND2 (src/OCFD_Schemes.cu:800-837); s = &stencil[1].
template <typename R> __device__ __forceinline__ R nnd2_up(const R* s) {
    return s[1] + R(0.5) * d_minmod2(s[2] - s[1], s[1] - s[0]);
}
template <typename R> __device__ __forceinline__ R nnd2_dn(const R* s) {
    return s[1] + R(0.5) * d_minmod2(s[0] - s[1], s[1] - s[2]);
}

// Stencil extents (ia1, ib1) of each scheme's kernels.
template <int SCH, int SIDE> struct Ext {
    static constexpr int ka = (SCH == 303) ? -3 : (SCH == 302 || SCH == 306) ? -2 : (SIDE == 0 ? -3 : -4);
    static constexpr int kb = (SCH == 303) ? 3 : (SCH == 302 || SCH == 306) ? 2 : (SIDE == 0 ? 4 : 3);
};
