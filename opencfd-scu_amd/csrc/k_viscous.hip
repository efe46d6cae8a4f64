// k_viscous.hip - viscous terms (gfx950).
//
// Restates du_vis_Jacobian3d (src/OCFD_Stream.cu:307-335) in two kernels:
//
//   k_visc_gf  : the 12 derivatives of u,v,w,T along xi/eta/zeta (CD6/CD8 with
//                the D0 closures: du_viscous_Jacobian3d_init,
//                src/OCFD_NS_Jacobian3d.cu:58-77; OCFD_CD6/CD8_kernel,
//                src/OCFD_Schemes.cu:96-156; OCFD_D0bound_scheme_kernel,
//                src/OCFD_bound_Scheme.cu:79-186) and, at the same point, the
//                contravariant viscous fluxes Ev1..4 of all three directions
//                (vis_flux_ker, src/OCFD_NS_Jacobian3d.cu:80-281).  The
//                gradients never leave registers.
//   k_visc_div : d(Ev)/dxi + d(Ev)/deta + d(Ev)/dzeta (OCFD_d?0 of Ev +
//                YF_Pe_XF, src/OCFD_NS_Jacobian3d.cu:304-440,
//                src/commen_kernel.cu:158-169), no atomics, and with it the
//                RK stage of the point; or, for callers that want the
//                right-hand side in memory, the divergence alone.
//   k_qcrit    : the Q criterion of the analysis events (same derivatives).
//
// S (double or float) is the type of u,v,w,T, mu, the derivatives, the
// fluxes, du and dv; the Jacobian factor of the divergence and its sums are
// double.
//
// Both use 2.5-D blocking: a block owns a TX x TY tile of (x,y) columns and
// marches through a chunk of z planes (chunk_planes).  x and y neighbours come from the
// current plane staged in LDS with its 4-point halo; z neighbours come from a
// 9-plane queue each thread keeps in registers for its own column.
#include <type_traits>

#include "ocfd_dev.h"
#include "ocfd_kernels.h"

namespace {

constexpr int TX = 32, TY = 8;  // columns per block
// z planes per block where a launch fills the chip anyway (chunk_planes).
// FP64, 1024x384x256: the gradient kernel 16 / 24 / 32 / 64 planes 4.57 / 4.55 /
// 4.46 / 4.74 ms; FP32: 8 is the fastest alone, 16 the faster step beside the
// sweeps.
template <typename S> struct KZ_ { static constexpr int v = 32; };
template <> struct KZ_<float> { static constexpr int v = 16; };

// Central derivative at interior index i (0..n-1) from s[0..8] = values at
// i-4..i+4 (OCFD_CD6/CD8_kernel + D0 closures + put_d0_kernel).  rh = 1/h; the
// reference's divisions by 12, 60, 840 and h are multiplications by the
// reciprocals here (a difference of an ulp or two per derivative).  CL =
// false compiles the interior formula alone, for callers that know that no
// closure is in reach.
template <int SV, typename R, bool CL = true>
__device__ __forceinline__ R cd9(const R* s, int i, int n, int bl, int br, R rh) {
    const R* c = s + 4;
    R tmp;
    if (CL && bl && i <= 3) {
        if (i == 0) tmp = (c[1] - c[0]);
        else if (i == 1) tmp = (c[1] - c[-1]) * R(0.5);
        else if (i == 2) tmp = (c[-2] - R(8) * c[-1] + R(8) * c[1] - c[2]) * R(1.0 / 12.0);
        else tmp = (c[3] - c[-3] - R(9) * (c[2] - c[-2]) + R(45) * (c[1] - c[-1])) * R(1.0 / 60.0);
    } else if (CL && br && i >= n - 4) {
        const int t1 = i - n;
        if (t1 == -1) tmp = (c[0] - c[-1]);
        else if (t1 == -2) tmp = (c[1] - c[-1]) * R(0.5);
        else if (t1 == -3) tmp = (c[-2] - R(8) * c[-1] + R(8) * c[1] - c[2]) * R(1.0 / 12.0);
        else tmp = (c[3] - c[-3] - R(9) * (c[2] - c[-2]) + R(45) * (c[1] - c[-1])) * R(1.0 / 60.0);
    } else if (SV == OCFD_CD6) {
        tmp = (R(45) * (c[1] - c[-1]) - R(9) * (c[2] - c[-2]) + (c[3] - c[-3])) * R(1.0 / 60.0);
    } else {
        tmp = (R(672) * (c[1] - c[-1]) - R(168) * (c[2] - c[-2]) + R(32) * (c[3] - c[-3]) - R(3) * (c[4] - c[-4])) *
              R(1.0 / 840.0);
    }
    return tmp * rh;
}

// Tile bookkeeping shared by both kernels.
struct Tile25 {
    int i0, j0, i, j, kbeg, kend;
    bool own;
};
__device__ __forceinline__ Tile25 tile_of(const Geo& g, int kz) {
    Tile25 t;
    const Blk B = xcd_block();
    t.i0 = B.x * TX;
    t.j0 = B.y * TY;
    t.i = t.i0 + threadIdx.x;
    t.j = t.j0 + threadIdx.y;
    t.kbeg = B.z * kz;
    t.kend = min(t.kbeg + kz, g.nz);
    t.own = t.i < g.nx && t.j < g.ny;
    return t;
}

// Gradients of u, v, w, T at (t.i, t.j, k) from the plane tile pl (the
// current plane with its x and y strips, row pitch PW) and the thread's z
// queue q, and at the same point the viscous fluxes Ev1..4 of the three
// directions (vis_flux_s_ker / vis_flux_e_ker / vis_flus_ev_ker) from the
// point's metrics met.  oo: the point's byte offset in a plane (BUF_NONE: no
// point, nothing is written).  CL = false: no derivative of the block's plane
// reaches a closure (the caller decides per block and plane), and the body is
// straight-line code.
template <int SV, typename S, int PW, bool CL>
__device__ __forceinline__ void gf_point(const ViscArgsT<S>& A, const Tile25& t, int k, long long fs, unsigned oo,
                                         const S* met,
                                         const S (*pl)[PW * (TY + 8)],
                                         const S (*q)[9], int tx, int ty, S rhx, S rhy, S rhz) {
    const Geo& g = A.g;
    S gr[4][3];
#pragma unroll
    for (int f = 0; f < 4; f++) {
        S s[9];
#pragma unroll
        for (int m = 0; m < 9; m++) s[m] = pl[f][(ty + 4) * PW + tx + m];
        gr[f][0] = cd9<SV, S, CL>(s, t.i, g.nx, A.bnd[0], A.bnd[1], rhx);
#pragma unroll
        for (int m = 0; m < 9; m++) s[m] = pl[f][(ty + m) * PW + tx + 4];
        gr[f][1] = cd9<SV, S, CL>(s, t.j, g.ny, A.bnd[2], A.bnd[3], rhy);
        gr[f][2] = cd9<SV, S, CL>(q[f], k, g.nz, A.bnd[4], A.bnd[5], rhz);
    }
    const S Akx = met[M_KX], Aky = met[M_KY], Akz = met[M_KZ];
    const S Aix = met[M_IX], Aiy = met[M_IY], Aiz = met[M_IZ];
    const S Asx = met[M_SX], Asy = met[M_SY], Asz = met[M_SZ];
    const S Aj1 = met[M_JAC];
    // Sutherland's law at the point (get_Amu_kernal, src/commen_kernel.cu:
    // 122-131) from its T (the centre of the z queue), in FP64 as the RK stage
    // and the boundary kernels form it: the same value as a viscosity field
    // written after each stage, without its 8 B/pt store and reload
    const double Tp = double(q[3][4]);
    const S Amu = S(A.c.amu_c0 * sqrt(Tp * Tp * Tp) / (A.c.tsb + Tp));
    // vis_flux_s_ker / vis_flux_e_ker / vis_flus_ev_ker
    const S uk = gr[0][0], ui = gr[0][1], us = gr[0][2];
    const S vk = gr[1][0], vi = gr[1][1], vs = gr[1][2];
    const S wk = gr[2][0], wi = gr[2][1], ws = gr[2][2];
    const S Tk = gr[3][0], Ti = gr[3][1], Ts = gr[3][2];
    const S ux = uk * Akx + ui * Aix + us * Asx;
    const S vx = vk * Akx + vi * Aix + vs * Asx;
    const S wx = wk * Akx + wi * Aix + ws * Asx;
    const S uy = uk * Aky + ui * Aiy + us * Asy;
    const S vy = vk * Aky + vi * Aiy + vs * Asy;
    const S wy = wk * Aky + wi * Aiy + ws * Asy;
    const S uz = uk * Akz + ui * Aiz + us * Asz;
    const S vz = vk * Akz + vi * Aiz + vs * Asz;
    const S wz = wk * Akz + wi * Aiz + ws * Asz;
    const S div = ux + vy + wz;
    const S two3 = S(2.0 / 3.0);
    const S s11 = (S(2) * ux - two3 * div) * Amu;
    const S s22 = (S(2) * vy - two3 * div) * Amu;
    const S s33 = (S(2) * wz - two3 * div) * Amu;
    const S s12 = (uy + vx) * Amu;
    const S s13 = (uz + wx) * Amu;
    const S s23 = (vz + wy) * Amu;
    const S Amuk = Amu * S(A.c.vis_c);
    const S Tx = Tk * Akx + Ti * Aix + Ts * Asx;
    const S Ty = Tk * Aky + Ti * Aiy + Ts * Asy;
    const S Tz = Tk * Akz + Ti * Aiz + Ts * Asz;
    const S u = q[0][4], v = q[1][4], w = q[2][4];
    const S E1 = u * s11 + v * s12 + w * s13 + Amuk * Tx;
    const S E2 = u * s12 + v * s22 + w * s23 + Amuk * Ty;
    const S E3 = u * s13 + v * s23 + w * s33 + Amuk * Tz;
    const S ax[3] = {Akx, Aix, Asx}, ay[3] = {Aky, Aiy, Asy}, az[3] = {Akz, Aiz, Asz};
#pragma unroll
    for (int d = 0; d < 3; d++) {
        const S akx = ax[d] * Aj1, aky = ay[d] * Aj1, akz = az[d] * Aj1;
        // written once here and read by another kernel: streamed
        auto put = [&](int m, S v) {
            Buf<S>(A.ev + (long long)(k + 4) * g.sz + (4 * d + m) * fs, g.sz).template st<BUF_STREAM>(oo, v);
        };
        put(0, akx * s11 + aky * s12 + akz * s13);
        put(1, akx * s12 + aky * s22 + akz * s23);
        put(2, akx * s13 + aky * s23 + akz * s33);
        put(3, akx * E1 + aky * E2 + akz * E3);
    }
}

// Whether a central-derivative closure is in reach of the block's plane k:
// the same for every thread of the block.
template <typename S>
__device__ __forceinline__ bool near_closure(const ViscArgsT<S>& A, const Tile25& t, int k) {
    const Geo& g = A.g;
    return (A.bnd[0] && t.i0 <= 3) || (A.bnd[1] && t.i0 + TX > g.nx - 4) || (A.bnd[2] && t.j0 <= 3) ||
           (A.bnd[3] && t.j0 + TY > g.ny - 4) || (A.bnd[4] && k <= 3) || (A.bnd[5] && k >= g.nz - 4);
}

// Gradients and viscous fluxes of a plane, marching in z.  The next plane's
// strips and queue values and the point's metrics are in flight while a plane
// is computed.  Bound by HBM (512x128x64 5.7 TB/s of traffic) and by latency
// behind it: what moved it is when loads are issued.  Raw buffer accesses took
// the FP64 kernel from 233 VGPRs to 204 (still 2 waves per SIMD) and the FP32
// kernel from 3 waves to 4, and made the ring of strips fetched five planes
// ahead pointless: 1024x256x128 1.58 -> 1.54 ms, 512x128x64 193 -> 182 us, mixed
// 120 -> 117 us (1024x384x256 1 %, though it fetches 178.5 B/pt for 152.5: a
// strip's second reader finds it evicted more often).  Dropped: metrics loaded
// after the derivatives to fit 3 waves (182 -> 241 us, mixed 117 -> 167), a plane
// ahead (194, 141), 32x16 tiles (210, 126).
template <int SV, typename S>
__global__ void __launch_bounds__(TX * TY, sizeof(S) == 8 ? 2 : 4) k_visc_gf(ViscArgsT<S> A, int kz) {
    constexpr int NT = TX * TY;
    constexpr int PW = TX + 8, PN = PW * (TY + 8);
    static_assert(NT >= 8 * TX, "y strips: one position per thread");
    const Geo& g = A.g;
    const Tile25 t = tile_of(g, kz);
    const int tx = threadIdx.x, ty = threadIdx.y, tid = ty * TX + tx;
    const S rhx = S(1.0 / g.hx), rhy = S(1.0 / g.hy), rhz = S(1.0 / g.hz);
    __shared__ S pl[4][PN];
    // byte offset of (i, j) in a plane, up to the ghost layers
    auto off = [&](int i, int j) {
        return i < g.nx + 4 && j < g.ny + 4 ? (unsigned)((i + 4) + g.ldx * (j + 4)) * (unsigned)sizeof(S) : BUF_NONE;
    };
    const unsigned oo = t.own ? off(t.i, t.j) : BUF_NONE;
    const unsigned od = t.own ? oo / (unsigned)sizeof(S) * 8u : BUF_NONE;  // in the FP64 metric fields
    // the thread's own tile position: from the queue when owned, else from
    // memory (x/y ghosts inside the tile)
    const unsigned oc = t.own ? BUF_NONE : off(t.i, t.j);
    // halo strips a derivative reads: 4 + 4 columns beside the tile's rows
    // (the first 8 * TY threads) and 4 + 4 rows beside its columns (the first
    // 8 * TX threads); the corners are never read
    const int xc = tid & 7, xr = tid >> 3;
    const bool xs = tid < 8 * TY, ys = tid < 8 * TX;
    const int yr = tid / TX;
    const unsigned ox = xs ? off(xc < 4 ? t.i0 - 4 + xc : t.i0 + TX + xc - 4, t.j0 + xr) : BUF_NONE;
    const unsigned oy = ys ? off(t.i0 + tx, yr < 4 ? t.j0 - 4 + yr : t.j0 + TY + yr - 4) : BUF_NONE;
    const int px = (xr + 4) * PW + (xc < 4 ? xc : TX + xc), py = (yr < 4 ? yr : TY + yr) * PW + tx + 4;
    const int pc = (ty + 4) * PW + tx + 4;
    // plane k of u, v, w, T (consecutive fields)
    long long fs = A.fs;
    auto bs = [&](int f, int k) { return Buf<S>(A.u + (long long)(k + 4) * g.sz + f * fs, g.sz); };
    S xv[4] = {}, yv[4] = {}, cv[4];
    auto load_strips = [&](int k) {
        if (ys)
#pragma unroll
            for (int f = 0; f < 4; f++) yv[f] = bs(f, k).ld(oy);
        if (xs)
#pragma unroll
            for (int f = 0; f < 4; f++) xv[f] = bs(f, k).ld(ox);
    };
    auto load_own = [&](int k) {
#pragma unroll
        for (int f = 0; f < 4; f++) cv[f] = bs(f, k).ld(oc);
    };
    // z queue of the own column: q[f][m] = field f at plane k-4+m
    S q[4][9], nq[4];
#pragma unroll
    for (int m = 0; m < 8; m++)
#pragma unroll
        for (int f = 0; f < 4; f++) q[f][m] = bs(f, t.kbeg - 4 + m).ld(oo);
#pragma unroll
    for (int f = 0; f < 4; f++) nq[f] = bs(f, t.kbeg + 4).ld(oo);
    load_strips(t.kbeg);
    load_own(t.kbeg);
    for (int k = t.kbeg; k < t.kend; k++) {
        fs = opaque(fs);
#pragma unroll
        for (int f = 0; f < 4; f++) {
            q[f][8] = nq[f];
            pl[f][pc] = t.own ? q[f][4] : cv[f];
            if (ys) pl[f][py] = yv[f];
            if (xs) pl[f][px] = xv[f];
        }
        // the point's metrics: read once, streamed; in flight across the
        // barrier and the derivatives
        S met[M_COUNT];
#pragma unroll
        for (int m = 0; m < M_COUNT; m++)
            met[m] = S(Buf<double>(A.M[0] + (long long)(k + 4) * g.sz + m * fs, g.sz).template ld<BUF_STREAM>(od));
        __syncthreads();
        if (k + 1 < t.kend) {
#pragma unroll
            for (int f = 0; f < 4; f++) nq[f] = bs(f, k + 5).ld(oo);
            load_own(k + 1);
            load_strips(k + 1);
        }
        if (near_closure(A, t, k)) gf_point<SV, S, PW, true>(A, t, k, fs, oo, met, pl, q, tx, ty, rhx, rhy, rhz);
        else gf_point<SV, S, PW, false>(A, t, k, fs, oo, met, pl, q, tx, ty, rhx, rhy, rhz);
#pragma unroll
        for (int f = 0; f < 4; f++)
#pragma unroll
            for (int m = 0; m < 8; m++) q[f][m] = q[f][m + 1];
        __syncthreads();
    }
}

// prim->cons of one point (pri_to_cons_kernel, src/commen_kernel.cu:32-64).
__device__ __forceinline__ void p2c5(double d, double u, double v, double w, double T, double cv, double* f) {
    f[0] = d;
    f[1] = u * d;
    f[2] = v * d;
    f[3] = w * d;
    f[4] = d * ((u * u + v * v + w * w) * 0.5 + cv * T);
}

// The divergence of Ev (Ev_x needs x neighbours, Ev_y y neighbours, Ev_z z
// neighbours; periodic neighbours are read where they are, so the Ev ghost
// layers are never filled and stay 0) and, with KRK = 1..3, the RK stage of
// the point that it completes: the viscous terms never go to memory.  KRK = 0
// leaves them in memory (dv) for the callers that want them there.
//
// The stage as OCFD_time_advance_ker1/2/3 (src/OCFD_time.cu:44-94) with
// cons->prim + p (cons_to_pri_kernel, src/commen_kernel.cu:77-109).  f is written
// in every stage and read by the next: formed again from the primitives, which
// would save 40 B/pt of writes in stages 1 and 2, it goes through four
// divisions, a difference and back, and the error of the state after 10 to 40
// steps against 80-bit arithmetic grows by 9 % (energy up to 28 %).
// PARTS: groups of du to add (1, or 3 where each sweep writes its own).
// G.faces: f of the six faces from the primitives as OCFD_bc leaves it
// (src/OCFD_boundary.cu:40-91), for runs whose boundary condition changes
// nothing else; G.ghost[dir]: the point's copy in the periodic ghost layers.
//
// Bound by HBM.  The strips of the next plane are in flight while a plane is
// computed.  All accesses are raw buffer accesses (Buf): with plain pointers
// the 40 addresses of a point took the kernel to 255 VGPRs and spills (FP32:
// slower than the separate kernels, 252 us against 215 on 512x128x64); with
// them it needs 203, FP32 125 (223, and 128 with 12 spilled, where it adds three
// parts of du).  Divergence and stage as one launch against
// three (two of two flux components, then the stage): 1024x256x128 2.42 -> 2.17
// ms, 512x128x64 296 -> 251 us, mixed 215 -> 172 us, 640x192x96 mixed 567 -> 510
// us.
constexpr int NTD = TX * TY;
template <int SV, typename S, int KRK, int PARTS>
__global__ void __launch_bounds__(NTD, sizeof(S) == 8 ? 2 : 4) k_visc_div(ViscArgsT<S> A, StageArgsT<S> G, int kz) {
    static_assert(TY == 8, "one y-halo value per thread: 8 halo rows of TX columns");
    // FP64, at 2 waves per SIMD, has registers to fetch the point's values a
    // plane ahead (512x128x64, then without f in stages 1 and 2: 252 -> 232 us
    // against loads after the derivatives at 3 waves); FP32 fetches them before the derivatives and keeps 4 waves
    // (172 us; a plane ahead 179 at 3 waves, 192 at 4)
    constexpr bool AHEAD = sizeof(S) == 8;
    constexpr int XW = TX + 8, NC = 4;
    const Geo& g = A.g;
    const Tile25 t = tile_of(g, kz);
    const int tx = threadIdx.x, ty = threadIdx.y, tid = ty * TX + tx;
    const S rhx = S(1.0 / g.hx), rhy = S(1.0 / g.hy), rhz = S(1.0 / g.hz);
    __shared__ S ex[NC][TY * XW];
    __shared__ S ey[NC][(TY + 8) * TX];
    long long fs = A.fs;
    // byte offset of (i, j) in a plane; i and j up to the ghost layers,
    // wrapped where the direction is periodic
    auto off = [&](int i, int j) { return (unsigned)((i + 4) + g.ldx * (j + 4)) * (unsigned)sizeof(S); };
    auto wrap = [](int i, int n, int per) { return per ? (i < 0 ? i + n : i >= n ? i - n : i) : i; };
    auto off_x = [&](int i, int j) { return i < g.nx + 4 && j < g.ny ? off(wrap(i, g.nx, A.per[0]), j) : BUF_NONE; };
    auto off_y = [&](int i, int j) { return i < g.nx && j < g.ny + 4 ? off(i, wrap(j, g.ny, A.per[1])) : BUF_NONE; };
    // halo: x strips of 4 + 4 columns (the first 8 * TY threads), y strips of
    // 4 + 4 rows (one value per thread)
    const int hc = tid & 7, hr = (tid >> 3) & (TY - 1);
    const bool xh = tid < 8 * TY;
    const unsigned oo = t.own ? off(t.i, t.j) : BUF_NONE;
    const unsigned od = t.own ? oo / (unsigned)sizeof(S) * 8u : BUF_NONE;  // in the FP64 fields
    const unsigned ox = off_x(t.i, t.j), oy = off_y(t.i, t.j);
    const unsigned oxh = xh ? off_x(hc < 4 ? t.i0 - 4 + hc : t.i0 + TX + hc - 4, t.j0 + hr) : BUF_NONE;
    const unsigned oyh = off_y(t.i, ty < 4 ? t.j0 - 4 + ty : t.j0 + TY + ty - 4);
    const int lx = ty * XW + tx + 4, lxh = hr * XW + (hc < 4 ? hc : TX + hc);
    const int ly = (ty + 4) * TX + tx, lyh = (ty < 4 ? ty : TY + ty) * TX + tx;
    auto zwrap = [&](int k) { return A.per[2] ? (k < 0 ? k + g.nz : k >= g.nz ? k - g.nz : k) : k; };
    // plane k of field m of a group
    auto bs = [&](const S* base, int m, int k) { return Buf<S>(base + (long long)(k + 4) * g.sz + m * fs, g.sz); };
    auto bd = [&](const double* base, int m, int k) { return Buf<double>(base + (long long)(k + 4) * g.sz + m * fs, g.sz); };

    S xv[NC], yv[NC], xhv[NC] = {}, yhv[NC], q[NC][9], nq[NC];
    auto load_strips = [&](int k) {
#pragma unroll
        for (int f = 0; f < NC; f++) xv[f] = bs(A.ev, f, k).ld(ox);
#pragma unroll
        for (int f = 0; f < NC; f++) yv[f] = bs(A.ev, 4 + f, k).ld(oy);
#pragma unroll
        for (int f = 0; f < NC; f++) yhv[f] = bs(A.ev, 4 + f, k).ld(oyh);
        if (xh)
#pragma unroll
            for (int f = 0; f < NC; f++) xhv[f] = bs(A.ev, f, k).ld(oxh);
    };
    // the stage's own values of the point: du, Ajac, the base state fn and
    // the state f before the stage (as loaded: nothing waits for them before
    // the point is formed)
    S sr[PARTS][5];
    double sj = 0.0, sn[5], so[5];
    auto load_point = [&](int k) {
        if (!KRK) return;
#pragma unroll
        for (int p = 0; p < PARTS; p++)
#pragma unroll
            for (int m = 0; m < 5; m++) sr[p][m] = bs(G.du, 5 * p + m, k).template ld<BUF_STREAM>(oo);
        sj = bd(G.jac, 0, k).template ld<BUF_STREAM>(od);
#pragma unroll
        for (int m = 0; m < 5; m++) sn[m] = bd(G.fn, m, k).template ld<BUF_STREAM>(od);
        if (KRK == 1) return;
#pragma unroll
        for (int m = 0; m < 5; m++) so[m] = bd(G.f, m, k).template ld<BUF_STREAM>(od);
    };
#pragma unroll
    for (int m = 0; m < 8; m++)
#pragma unroll
        for (int f = 0; f < NC; f++) q[f][m] = bs(A.ev, 8 + f, zwrap(t.kbeg - 4 + m)).ld(oo);
    auto load_next = [&](int k) {
#pragma unroll
        for (int f = 0; f < NC; f++) nq[f] = bs(A.ev, 8 + f, zwrap(k)).ld(oo);
    };
    load_next(t.kbeg + 4);
    load_strips(t.kbeg);
    if (AHEAD) load_point(t.kbeg);
    for (int k = t.kbeg; k < t.kend; k++) {
        fs = opaque(fs);
#pragma unroll
        for (int f = 0; f < NC; f++) {
            q[f][8] = nq[f];
            ex[f][lx] = xv[f];
            ey[f][ly] = yv[f];
            ey[f][lyh] = yhv[f];
            if (xh) ex[f][lxh] = xhv[f];
        }
        __syncthreads();
        if (k + 1 < t.kend) {
            load_next(k + 5);
            load_strips(k + 1);
        }
        // CL = false: no closure in reach of the block's plane (straight-line
        // code).  The sums are double; the node's Ajac, by which the reference
        // multiplies each of these terms, is applied to the whole right-hand
        // side by the RK stage.
        double dv[NC];
        auto derivs = [&](auto cl) {
            constexpr bool CL = decltype(cl)::value;
#pragma unroll
            for (int m = 0; m < NC; m++) {
                S s[9];
#pragma unroll
                for (int r = 0; r < 9; r++) s[r] = ex[m][ty * XW + tx + r];
                const S vx = cd9<SV, S, CL>(s, t.i, g.nx, A.bnd[0], A.bnd[1], rhx);
#pragma unroll
                for (int r = 0; r < 9; r++) s[r] = ey[m][(ty + r) * TX + tx];
                const S vy = cd9<SV, S, CL>(s, t.j, g.ny, A.bnd[2], A.bnd[3], rhy);
                const S vz = cd9<SV, S, CL>(q[m], k, g.nz, A.bnd[4], A.bnd[5], rhz);
                dv[m] = (double(vx) + double(vy)) + double(vz);
            }
        };
        if (!AHEAD) load_point(k);
        if (near_closure(A, t, k)) derivs(std::true_type{});
        else derivs(std::false_type{});
        if (!KRK) {
#pragma unroll
            for (int m = 0; m < NC; m++) bs(A.dv, m, k).st(oo, S(dv[m]));
        } else {
            const double dt = G.dt;
            double fv[5];
#pragma unroll
            for (int m = 0; m < 5; m++) {
                double r = double(sr[0][m]);
#pragma unroll
                for (int p = 1; p < PARTS; p++) r += double(sr[p][m]);
                if (m) r += dv[m - 1];
                r *= sj;
                if (KRK == 1) fv[m] = sn[m] + dt * r;
                else if (KRK == 2) fv[m] = 3.0 / 4.0 * sn[m] + 1.0 / 4.0 * (so[m] + dt * r);
                else fv[m] = 1.0 / 3.0 * sn[m] + 2.0 / 3.0 * (so[m] + dt * r);
            }
            const double d1 = fv[0], u1 = fv[1] / d1, v1 = fv[2] / d1, w1 = fv[3] / d1;
            const double T2 = (fv[4] - 0.5 * d1 * (u1 * u1 + v1 * v1 + w1 * w1)) / (d1 * G.c.cv);
            const S pr[5] = {S(d1), S(u1), S(v1), S(w1), S(T2)};
#pragma unroll
            for (int m = 0; m < 5; m++) bs(G.d, m, k).st(oo, pr[m]);
            if (KRK == 3) bs(G.P, 0, k).template st<BUF_STREAM>(oo, S(T2 * d1 / (G.c.gamma * G.c.ama * G.c.ama)));
            if (KRK == 3 && G.flap)
#pragma unroll
                for (int m = 0; m < 5; m++) bd(G.flap, m, k).template st<BUF_STREAM>(od, fv[m]);
            if (G.faces && (t.i == 0 || t.i == g.nx - 1 || t.j == 0 || t.j == g.ny - 1 || k == 0 || k == g.nz - 1))
                p2c5(double(pr[0]), double(pr[1]), double(pr[2]), double(pr[3]), double(pr[4]), G.c.cv, fv);
#pragma unroll
            for (int m = 0; m < 5; m++) bd(G.f, m, k).template st<BUF_STREAM>(od, fv[m]);
            auto copy_to = [&](int kk, unsigned o) {
#pragma unroll
                for (int m = 0; m < 5; m++) bs(G.d, m, kk).st(o, pr[m]);
            };
            if (G.ghost[0] && t.own && (t.i < 4 || t.i >= g.nx - 4)) copy_to(k, off(t.i < 4 ? t.i + g.nx : t.i - g.nx, t.j));
            if (G.ghost[1] && t.own && (t.j < 4 || t.j >= g.ny - 4)) copy_to(k, off(t.i, t.j < 4 ? t.j + g.ny : t.j - g.ny));
            if (G.ghost[2] && (k < 4 || k >= g.nz - 4)) copy_to(k < 4 ? k + g.nz : k - g.nz, oo);
        }
        if (AHEAD && k + 1 < t.kend) load_point(k + 1);
#pragma unroll
        for (int f = 0; f < NC; f++)
#pragma unroll
            for (int m = 0; m < 8; m++) q[f][m] = q[f][m + 1];
        __syncthreads();
    }
}

// Q criterion of the velocity (get_Q / get_Q_kernal, src/OCFD_ana.cu:
// 299-420): the nine derivatives of u, v, w along xi/eta/zeta with the
// viscous scheme and its D0 closures (OCFD_dx0/dy0/dz0), the Cartesian
// gradient from the cofactors, Q = (ux vy + ux wz + vy wz - uy vx - uz wx
// - vz wy) Ajac^2.  A diagnostic run once: one thread per point, stencils read
// straight from memory, FP64 arithmetic on both paths.
template <int SV, typename S>
__global__ void __launch_bounds__(256) k_qcrit(ViscArgsT<S> A, double* __restrict__ qout) {
    const Geo& g = A.g;
    const int i = blockIdx.x * 64 + threadIdx.x, j = blockIdx.y * 4 + threadIdx.y, k = blockIdx.z;
    if (i >= g.nx || j >= g.ny) return;
    const long long qi = gidx(g, i, j, k);
    const double rhx = 1.0 / g.hx, rhy = 1.0 / g.hy, rhz = 1.0 / g.hz;
    const S* src[3] = {A.u, A.v, A.w};
    double gr[3][3];
#pragma unroll
    for (int f = 0; f < 3; f++) {
        double s[9];
#pragma unroll
        for (int m = 0; m < 9; m++) s[m] = double(src[f][qi + (m - 4)]);
        gr[f][0] = cd9<SV>(s, i, g.nx, A.bnd[0], A.bnd[1], rhx);
#pragma unroll
        for (int m = 0; m < 9; m++) s[m] = double(src[f][qi + (long long)(m - 4) * g.ldx]);
        gr[f][1] = cd9<SV>(s, j, g.ny, A.bnd[2], A.bnd[3], rhy);
#pragma unroll
        for (int m = 0; m < 9; m++) s[m] = double(src[f][qi + (long long)(m - 4) * g.sz]);
        gr[f][2] = cd9<SV>(s, k, g.nz, A.bnd[4], A.bnd[5], rhz);
    }
    const double Akx = A.M[M_KX][qi], Aky = A.M[M_KY][qi], Akz = A.M[M_KZ][qi];
    const double Aix = A.M[M_IX][qi], Aiy = A.M[M_IY][qi], Aiz = A.M[M_IZ][qi];
    const double Asx = A.M[M_SX][qi], Asy = A.M[M_SY][qi], Asz = A.M[M_SZ][qi];
    const double ux = gr[0][0] * Akx + gr[0][1] * Aix + gr[0][2] * Asx;
    const double vx = gr[1][0] * Akx + gr[1][1] * Aix + gr[1][2] * Asx;
    const double wx = gr[2][0] * Akx + gr[2][1] * Aix + gr[2][2] * Asx;
    const double uy = gr[0][0] * Aky + gr[0][1] * Aiy + gr[0][2] * Asy;
    const double vy = gr[1][0] * Aky + gr[1][1] * Aiy + gr[1][2] * Asy;
    const double wy = gr[2][0] * Aky + gr[2][1] * Aiy + gr[2][2] * Asy;
    const double uz = gr[0][0] * Akz + gr[0][1] * Aiz + gr[0][2] * Asz;
    const double vz = gr[1][0] * Akz + gr[1][1] * Aiz + gr[1][2] * Asz;
    const double wz = gr[2][0] * Akz + gr[2][1] * Aiz + gr[2][2] * Asz;
    const double aj = A.M[M_JAC][qi];
    qout[qi] = (ux * vy + ux * wz + vy * wz - uy * vx - uz * wx - vz * wy) * aj * aj;
}

// z planes per block.  A launch that does not fill the chip is bound by the
// longest march: its planes are spread over as many blocks as the GPU holds
// at once (2 per CU of the FP64 kernels, 4 of the FP32 ones), each block paying the
// 8 planes of its z queue again from L2.  Measured when it came, a gradient
// launch, against the fixed chunks: 64^3 82 -> 17.5 us, 61x47x39 84 -> 13.2,
// 203x93x45 142 -> 53.5 (now 15.8, 11.1 and 48; the divergence, then two components a
// launch, 38 -> 9.0, 38.5 -> 7.8, 55 -> 21.2 each); 512x128x64, which 32 planes fill
// exactly, keeps them (16: 196 -> 204 us).  Larger launches take the fixed chunk,
// where the extra z reads are what counts.
template <typename S>
int chunk_planes(const Geo& g, int cols) {
    constexpr int RES = 256 * (sizeof(S) == 8 ? 2 : 4), MOST = 32;
    if (cols <= RES) {
        const int nch = RES / cols, kz = (g.nz + nch - 1) / nch;
        if (kz <= MOST) return kz;
    }
    return KZ_<S>::v;
}

template <typename S>
dim3 grid25(const Geo& g, int& kz) {
    const int gx = (g.nx + TX - 1) / TX, gy = (g.ny + TY - 1) / TY;
    kz = chunk_planes<S>(g, gx * gy);
    return dim3(gx, gy, (g.nz + kz - 1) / kz);
}

}  // namespace

template <typename S>
void launch_visc_gf(const ViscArgsT<S>& a, hipStream_t st) {
    int kz;
    const dim3 grid = grid25<S>(a.g, kz), blk(TX, TY);
    if (a.svis == OCFD_CD6) hipLaunchKernelGGL((k_visc_gf<OCFD_CD6, S>), grid, blk, 0, st, a, kz);
    else hipLaunchKernelGGL((k_visc_gf<OCFD_CD8, S>), grid, blk, 0, st, a, kz);
}
namespace {
template <int SV, typename S>
void launch_div(const ViscArgsT<S>& a, const StageArgsT<S>& st_, int krk, hipStream_t st) {
    int kz;
    const dim3 grid = grid25<S>(a.g, kz), blk(TX, TY);
    auto go = [&](auto k, auto parts) {
        hipLaunchKernelGGL((k_visc_div<SV, S, decltype(k)::value, decltype(parts)::value>), grid, blk, 0, st, a, st_, kz);
    };
    auto stage = [&](auto parts) {
        if (krk == 1) go(std::integral_constant<int, 1>{}, parts);
        else if (krk == 2) go(std::integral_constant<int, 2>{}, parts);
        else go(std::integral_constant<int, 3>{}, parts);
    };
    if (krk == 0) go(std::integral_constant<int, 0>{}, std::integral_constant<int, 1>{});
    else if (st_.parts == 3) stage(std::integral_constant<int, 3>{});
    else stage(std::integral_constant<int, 1>{});
}
}  // namespace
template <typename S>
void launch_visc_div(const ViscArgsT<S>& a, hipStream_t st) {
    const StageArgsT<S> none{};
    if (a.svis == OCFD_CD6) launch_div<OCFD_CD6>(a, none, 0, st);
    else launch_div<OCFD_CD8>(a, none, 0, st);
}
template <typename S>
void launch_visc_stage(const ViscArgsT<S>& a, const StageArgsT<S>& s, hipStream_t st) {
    if (a.svis == OCFD_CD6) launch_div<OCFD_CD6>(a, s, s.krk, st);
    else launch_div<OCFD_CD8>(a, s, s.krk, st);
}
template <typename S>
void launch_qcrit(const ViscArgsT<S>& a, double* q, hipStream_t st) {
    const dim3 grid((a.g.nx + 63) / 64, (a.g.ny + 3) / 4, a.g.nz);
    if (a.svis == OCFD_CD6) hipLaunchKernelGGL((k_qcrit<OCFD_CD6, S>), grid, dim3(64, 4), 0, st, a, q);
    else hipLaunchKernelGGL((k_qcrit<OCFD_CD8, S>), grid, dim3(64, 4), 0, st, a, q);
}
template void launch_qcrit<double>(const ViscArgsT<double>&, double*, hipStream_t);
template void launch_qcrit<float>(const ViscArgsT<float>&, double*, hipStream_t);
template void launch_visc_gf<double>(const ViscArgsT<double>&, hipStream_t);
template void launch_visc_gf<float>(const ViscArgsT<float>&, hipStream_t);
template void launch_visc_div<double>(const ViscArgsT<double>&, hipStream_t);
template void launch_visc_div<float>(const ViscArgsT<float>&, hipStream_t);
template void launch_visc_stage<double>(const ViscArgsT<double>&, const StageArgsT<double>&, hipStream_t);
template void launch_visc_stage<float>(const ViscArgsT<float>&, const StageArgsT<float>&, hipStream_t);
