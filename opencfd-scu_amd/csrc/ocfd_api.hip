// ocfd_api.hip - host side of libocfd_hip.so: the context, device memory, the
// time loop and the C ABI declared in include/ocfd.h.
//
// The step sequence restates NS_solver_real (src/OCFD_NS_Solver.cu:39-177)
// with du_comput (src/OCFD_Stream.cu:28-54) at STREAM=0 and one rank:
//   swap f/fn; for KRK=1..3 { [sensor at KRK=1]; periodic fill of the
//   primitives; x/y/z inviscid sweeps; viscous gradients, fluxes, periodic
//   fill of the fluxes, divergence; RK stage + cons->prim + mu; IBC; face
//   refresh }; Istep++; tt+=dt; filter.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <string>
#include <type_traits>
#include <vector>

#include "ocfd_kernels.h"

namespace {

thread_local std::string g_err;

int fail(int code, const std::string& msg) {
    g_err = msg;
    return code;
}

#define HIPCK(expr)                                                                       \
    do {                                                                                  \
        hipError_t e_ = (expr);                                                           \
        if (e_ != hipSuccess)                                                             \
            return fail(OCFD_ERR_HIP, std::string(#expr) + ": " + hipGetErrorString(e_)); \
    } while (0)

struct ProfRec {
    const char* name;
    hipEvent_t a, b;
};

}  // namespace

struct ocfd_ctx {
    ocfd_config cfg;
    int device = 0;
    hipStream_t st = nullptr;
    // second stream: the viscous gradients and fluxes (and, where a right-hand
    // side is asked for by itself, their divergence into dv) run beside the
    // inviscid sweeps, with which they share inputs only; joined before the
    // RK stage
    hipStream_t st2 = nullptr;
    hipEvent_t ev_fork = nullptr, ev_join = nullptr;
    bool serial = false;  // OCFD_SERIAL=1: one stream (per-kernel timing with an external profiler)
    bool bc108_split = false;  // OCFD_BC108_SPLIT=1: IBC 108 and the face refresh in three launches
    bool graphs = true;        // OCFD_GRAPH=0: no HIP graph replay of steps
    // pinned staging buffer of the device-to-host downloads (grown on demand)
    void* pin = nullptr;
    size_t pin_bytes = 0;
    hipEvent_t pin_ev[3] = {};  // one per slot of a download in pieces
    Geo g;
    Consts c;
    long long fs = 0;  // elements per field
    // device memory
    std::vector<void*> allocs;
    // primitives, viscosity, right-hand side and viscous fluxes: double on
    // the plain path; float (the s* pointers) on the mixed path
    bool mixed = false;
    double *d = nullptr, *u = nullptr, *v = nullptr, *w = nullptr, *T = nullptr, *P = nullptr;
    // du: the inviscid part, or with du_parts = 3 (small grids, sweeps_merged)
    // 3 x 5 fields, one group written by each sweep; dv: the viscous part of
    // du[1..4], allocated by the first call that wants a right-hand side in
    // memory (need_dv: a step's stage forms it in registers).
    int du_parts = 1;
    double *du = nullptr, *amu = nullptr, *ev = nullptr, *dv = nullptr;
    float *sd = nullptr, *su = nullptr, *sv = nullptr, *sw = nullptr, *sT = nullptr, *sP = nullptr;
    float *sdu = nullptr, *samu = nullptr, *sev = nullptr, *sdv = nullptr;
    // always double: metrics, conserved state, filter input, scratch
    double* M[M_COUNT] = {};
    double *f = nullptr, *fn = nullptr, *flap = nullptr;
    double* grad = nullptr;  // 12 fields of scratch (metric set-up, precision conversions)
    int8_t* flag[3] = {};
    double *ub1 = nullptr, *fxd = nullptr, *gzd = nullptr;
    float* mlp_params = nullptr;  // learned sensor (null: the plain sensor)
    float* mlp_store = nullptr;   // device copy of the parameters
    float* mlp_packed = nullptr;  // and the inference kernels' packed form of them
    float* mlp_prob = nullptr;    // its probability per node (LAP layout)
    float mlp_lo = 0.2f, mlp_hi = 0.8f;
    bool mlp_fused = true;        // learned sensor in the x sweep (else its own pass)
    double* diag_part = nullptr;  // 2 * diag_sum_blocks partial sums
    int* diag_scan = nullptr;     // 2 * DIAG_SCAN_BLOCKS counts
    double* b124 = nullptr;       // IBC 124 tables: inlet [5][nz][ny], upper [5][ny][nx], coeff [3][ny][nx], udist [ny][nx]
    std::vector<double> in124_host, up124_host;  // caller tables (flow-inlet-section.dat, flow-outboundary.dat)
    bool v_dist_need = false;     // IBC 124 wall disturbance present
    double* avg = nullptr;        // time averages of d,u,v,w,T (analysis style 101)
    int avg_n = 0;                // samples in them (Istep_average)
    double avg_tt = 0.0;          // their accumulated time (tt_average)
    // host state
    std::vector<double> coord_x, coord_z;  // mesh x, z (interior, for IBC 108 set-up)
    std::vector<double> coord_top_x;       // x along the top row at k=0
    std::vector<double> mesh;              // x, y, z (interior, 3 arrays) as loaded
    std::vector<double> inlet;             // [4][ny]
    bool have_inlet = false, have_grid = false, have_flow = false, inited = false;
    double TM[OCFD_MTMAX] = {}, fait[OCFD_MTMAX] = {};
    int x_begin = 0;
    int istep = 0;
    double tt = 0.0;
    int fpara[OCFD_MAX_FILTERS][11];
    bool filter_dir[3] = {false, false, false};
    // profiling
    // the last right-hand side's viscous part is still only in Ev (finish_rhs)
    bool div_pending = false;
    bool prof = false;
    std::vector<ProfRec> recs;
    std::vector<hipEvent_t> pool;
    std::vector<std::pair<std::string, std::pair<int, double>>> acc;
    hipEvent_t step_a = nullptr, step_b = nullptr;
    double last_step_ms = 0.0;
};

namespace {

// The arrays whose type follows the precision of the context.
template <typename S>
struct View {
    S *d, *u, *v, *w, *T, *P, *amu, *du, *ev, *dv;
};
template <typename S> View<S> view(ocfd_ctx* x);
template <> View<double> view<double>(ocfd_ctx* x) {
    return {x->d, x->u, x->v, x->w, x->T, x->P, x->amu, x->du, x->ev, x->dv};
}
template <> View<float> view<float>(ocfd_ctx* x) {
    return {x->sd, x->su, x->sv, x->sw, x->sT, x->sP, x->samu, x->sdu, x->sev, x->sdv};
}

hipEvent_t get_event(ocfd_ctx* x) {
    if (!x->pool.empty()) {
        hipEvent_t e = x->pool.back();
        x->pool.pop_back();
        return e;
    }
    hipEvent_t e;
    if (hipEventCreate(&e) != hipSuccess) return nullptr;
    return e;
}

// Run a launch bracketed by events when profiling.
template <typename F>
int timed(ocfd_ctx* x, const char* name, F&& fn) {
    if (!x->prof) {
        fn();
    } else {
        hipEvent_t a = get_event(x), b = get_event(x);
        if (!a || !b) return fail(OCFD_ERR_HIP, std::string(name) + ": hipEventCreate failed");
        HIPCK(hipEventRecord(a, x->st));
        fn();
        HIPCK(hipEventRecord(b, x->st));
        x->recs.push_back({name, a, b});
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(OCFD_ERR_HIP, std::string(name) + ": " + hipGetErrorString(e));
    return 0;
}

int flush_prof(ocfd_ctx* x) {
    if (x->recs.empty()) return 0;
    HIPCK(hipStreamSynchronize(x->st));
    for (auto& r : x->recs) {
        float ms = 0.f;
        HIPCK(hipEventElapsedTime(&ms, r.a, r.b));
        bool found = false;
        for (auto& e : x->acc)
            if (e.first == r.name) {
                e.second.first += 1;
                e.second.second += ms;
                found = true;
                break;
            }
        if (!found) x->acc.push_back({r.name, {1, (double)ms}});
        x->pool.push_back(r.a);
        x->pool.push_back(r.b);
    }
    x->recs.clear();
    return 0;
}

#define TRY(expr)             \
    do {                      \
        int rc_ = (expr);     \
        if (rc_) return rc_;  \
    } while (0)

double* alloc_fields(ocfd_ctx* x, int n, int& rc) {
    // 16 doubles of slack so that the base can be shifted by 12 elements:
    // element 0 of a row then sits 96 bytes past a 128-byte boundary and the
    // interior (x index 4) is 128-byte aligned.
    size_t bytes = ((size_t)x->fs * n + 16) * sizeof(double);
    void* p = nullptr;
    if (hipMalloc(&p, bytes) != hipSuccess) {
        rc = fail(OCFD_ERR_HIP, "hipMalloc failed (" + std::to_string(bytes) + " bytes)");
        return nullptr;
    }
    if (hipMemsetAsync(p, 0, bytes, x->st) != hipSuccess) {
        rc = fail(OCFD_ERR_HIP, "hipMemsetAsync failed");
        return nullptr;
    }
    x->allocs.push_back(p);
    return (double*)p + 12;
}

float* alloc_fields_f32(ocfd_ctx* x, int n, int& rc) {
    // same element layout as alloc_fields; shifting the base by 28 elements
    // puts the interior (x index 4) of every row on a 128-byte boundary (the
    // mixed path rounds the row pitch to 32 elements)
    size_t bytes = ((size_t)x->fs * n + 32) * sizeof(float);
    void* p = nullptr;
    if (hipMalloc(&p, bytes) != hipSuccess) {
        rc = fail(OCFD_ERR_HIP, "hipMalloc failed (" + std::to_string(bytes) + " bytes)");
        return nullptr;
    }
    x->allocs.push_back(p);
    if (hipMemsetAsync(p, 0, bytes, x->st) != hipSuccess) {
        rc = fail(OCFD_ERR_HIP, "hipMemsetAsync failed");
        return nullptr;
    }
    return (float*)p + 28;
}

int8_t* alloc_bytes(ocfd_ctx* x, size_t n, int& rc) {
    void* p = nullptr;
    if (hipMalloc(&p, n + 256) != hipSuccess) {
        rc = fail(OCFD_ERR_HIP, "hipMalloc failed");
        return nullptr;
    }
    x->allocs.push_back(p);
    if (hipMemsetAsync(p, 0, n + 256, x->st) != hipSuccess) {
        rc = fail(OCFD_ERR_HIP, "hipMemsetAsync failed");
        return nullptr;
    }
    return (int8_t*)p + 96;
}

// The device of a context for the allocations of a call that may come from a
// thread whose current device is another one.
struct OnDevice {
    int prev = -1;
    explicit OnDevice(int d) {
        if (hipGetDevice(&prev) != hipSuccess || prev == d || hipSetDevice(d) != hipSuccess) prev = -1;
    }
    ~OnDevice() {
        if (prev >= 0) (void)hipSetDevice(prev);
    }
};

// The buffer dv: 4 fields beside the 56 (mixed: 32 and 24 FP32) of a context,
// which a run that only steps never reads.
int need_dv(ocfd_ctx* x) {
    if (x->dv || x->sdv) return 0;
    OnDevice on(x->device);
    int rc = 0;
    if (x->mixed) x->sdv = alloc_fields_f32(x, 4, rc);
    else x->dv = alloc_fields(x, 4, rc);
    return rc;
}

bool supported_scheme(int s) { return (s >= OCFD_UP7 && s <= OCFD_HYBRIDAUTO); }

// Host copy of an interior array (nx*ny*nz, x fastest) into a padded field.
int upload_interior(ocfd_ctx* x, double* dst, const double* src, double ghost_value) {
    const Geo& g = x->g;
    std::vector<double> h((size_t)x->fs, ghost_value);
    for (int k = 0; k < g.nz; k++)
        for (int j = 0; j < g.ny; j++)
            std::memcpy(&h[(size_t)(gidx(g, 0, j, k) + 12)], src + ((size_t)k * g.ny + j) * g.nx,
                        sizeof(double) * g.nx);
    HIPCK(hipMemcpyAsync(dst - 12, h.data(), sizeof(double) * x->fs, hipMemcpyHostToDevice, x->st));
    HIPCK(hipStreamSynchronize(x->st));
    return 0;
}

// The pinned staging buffer, grown to at least `bytes`.
int ensure_pin(ocfd_ctx* x, size_t bytes) {
    if (bytes <= x->pin_bytes) return 0;
    HIPCK(hipStreamSynchronize(x->st));
    if (x->pin) (void)hipHostFree(x->pin);
    x->pin = nullptr;
    x->pin_bytes = 0;
    if (hipHostMalloc(&x->pin, bytes, hipHostMallocDefault) != hipSuccess) {
        x->pin = nullptr;
        return fail(OCFD_ERR_HIP, "hipHostMalloc failed (" + std::to_string(bytes) + " bytes)");
    }
    x->pin_bytes = bytes;
    return 0;
}

// Device-to-host copy of `bytes` at src, ordered after the work on the
// context's stream, through a pinned staging buffer; returns the staged
// host copy (valid until the next call).  A plain hipMemcpy into pageable
// memory takes the runtime's own staging path instead, and after such a copy
// a context created later in the same process was measured to lose the
// overlap of its two streams (mixed path on the 512x128x64 ramp: 2.13 ->
// 2.37 ms/step).
const void* d2h(ocfd_ctx* x, const void* src, size_t bytes, int& rc) {
    if ((rc = ensure_pin(x, bytes))) return nullptr;
    if (hipMemcpyAsync(x->pin, src, bytes, hipMemcpyDeviceToHost, x->st) != hipSuccess ||
        hipStreamSynchronize(x->st) != hipSuccess) {
        rc = fail(OCFD_ERR_HIP, "device-to-host copy failed");
        return nullptr;
    }
    return x->pin;
}
#define D2H(ptr, x, src, bytes)                       \
    do {                                              \
        int rc_ = 0;                                  \
        ptr = d2h((x), (src), (bytes), rc_);          \
        if (rc_) return rc_;                          \
    } while (0)

// nf arrays of interior values to host arrays, widened from S: pack(dst) launches
// what writes them to dst without ghost layers, one after another, so that the
// host copies long runs instead of rows.  Up to DIRECT bytes it writes straight
// into the pinned buffer (no copy of its own: a 20x16x12 state 5 copies and
// waits -> 1), above that the packed values come over in pieces of PIECE bytes,
// three in flight, while the host copies the one before.
template <typename S, typename F>
int download_packed(ocfd_ctx* x, double* const* out, int nf, F&& pack) {
    constexpr size_t DIRECT = 1u << 20, PIECE = 16u << 20;
    constexpr int SLOTS = 3;
    const size_t n = (size_t)x->g.nx * x->g.ny * x->g.nz;
    const size_t total = n * nf, bytes = total * sizeof(S);
    auto unpack = [&](const S* p, size_t first, size_t count) {
        while (count) {
            const size_t o = first % n, m = std::min(count, n - o);
            double* d = out[first / n] + o;
            if constexpr (std::is_same<S, double>::value) std::memcpy(d, p, m * sizeof(double));
            else
                for (size_t q = 0; q < m; q++) d[q] = double(p[q]);
            p += m;
            first += m;
            count -= m;
        }
    };
    if (bytes <= DIRECT) {
        TRY(ensure_pin(x, bytes));
        TRY(timed(x, "pack", [&] { pack((S*)x->pin); }));
        HIPCK(hipStreamSynchronize(x->st));
        unpack((const S*)x->pin, 0, total);
        return 0;
    }
    // packed into the scratch fields after the first (which ocfd_get_q fills)
    S* const dev = (S*)(x->grad + x->fs);
    const size_t piece = PIECE / sizeof(S), np = (total + piece - 1) / piece;
    TRY(ensure_pin(x, std::min(bytes, SLOTS * PIECE)));
    {
        OnDevice on(x->device);  // an event can be recorded on streams of its own device only
        for (auto& e : x->pin_ev)
            if (!e) HIPCK(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    }
    TRY(timed(x, "pack", [&] { pack(dev); }));
    auto slot = [&](size_t c) { return (S*)x->pin + (c % SLOTS) * piece; };
    auto count = [&](size_t c) { return std::min(piece, total - c * piece); };
    auto fetch = [&](size_t c) -> int {
        HIPCK(hipMemcpyAsync(slot(c), dev + c * piece, count(c) * sizeof(S), hipMemcpyDeviceToHost, x->st));
        HIPCK(hipEventRecord(x->pin_ev[c % SLOTS], x->st));
        return 0;
    };
    for (size_t c = 0; c < np && c < SLOTS; c++) TRY(fetch(c));
    for (size_t c = 0; c < np; c++) {
        HIPCK(hipEventSynchronize(x->pin_ev[c % SLOTS]));
        unpack(slot(c), c * piece, count(c));
        if (c + SLOTS < np) TRY(fetch(c + SLOTS));
    }
    return 0;
}

// The interiors of nf fields (null destinations are left out) to host arrays.
// A single FP64 field of up to SMALL bytes comes over as it is, with its ghost
// layers: there a copy costs less than a launch that writes to host memory
// (8x8x8 14.8 us packed, 10.9 so; 20x16x12 15.2, 14.5; 48x40x32, 600 KiB, 33, 52).
template <typename S>
int download_fields(ocfd_ctx* x, const S* const* src, double* const* dst, int nf) {
    PackArgsT<S> a;
    double* out[PACK_FIELDS];
    a.g = x->g;
    a.nf = 0;
    for (int q = 0; q < nf; q++)
        if (dst[q]) {
            out[a.nf] = dst[q];
            a.src[a.nf++] = src[q];
        }
    if (!a.nf) return 0;
    constexpr size_t SMALL = 128u << 10;
    if constexpr (std::is_same<S, double>::value)
        if (const size_t bytes = sizeof(double) * (size_t)x->fs; a.nf == 1 && bytes <= SMALL) {
            const Geo& g = x->g;
            const void* hv;
            D2H(hv, x, a.src[0] - 12, bytes);
            const double* h = (const double*)hv + 12;
            for (int k = 0; k < g.nz; k++)
                for (int j = 0; j < g.ny; j++)
                    std::memcpy(out[0] + ((size_t)k * g.ny + j) * g.nx, h + gidx(g, 0, j, k), sizeof(double) * g.nx);
            return 0;
        }
    return download_packed<S>(x, out, a.nf, [&](S* d) {
        a.dst = d;
        launch_pack(a, x->st);
    });
}
template <typename S>
int download_any(ocfd_ctx* x, const S* src, double* dst) {
    return download_fields(x, &src, &dst, 1);
}

// IPERIODIC as a mask (bit 0: x, 1: y, 2: z).
int periodic_dirs(const ocfd_ctx* x) {
    int m = 0;
    for (int dir = 0; dir < 3; dir++)
        if (x->cfg.iperiodic[dir]) m |= 1 << dir;
    return m;
}
template <typename T>
int fill_periodic(ocfd_ctx* x, T* base, int nf, const char* name) {
    if (const int dirs = periodic_dirs(x))
        TRY(timed(x, name, [&] { launch_fill(x->g, base, nf, x->fs, dirs, x->st); }));
    return 0;
}

template <typename S>
int fill_prims(ocfd_ctx* x) {
    // d,u,v,w,T are allocated as one group of 5 contiguous fields
    return fill_periodic(x, view<S>(x).d, 5, "fill_prims");
}

// Field of any storage type <-> interior host array, through the double
// scratch field for float fields.
template <typename S>
int upload_any(ocfd_ctx* x, S* dst, const double* src, double ghost_value) {
    if constexpr (std::is_same<S, double>::value) {
        return upload_interior(x, dst, src, ghost_value);
    } else {
        TRY(upload_interior(x, x->grad, src, ghost_value));
        TRY(timed(x, "convert", [&] { launch_convert(dst, x->grad, x->fs, x->st); }));
        HIPCK(hipStreamSynchronize(x->st));
        return 0;
    }
}
template <typename S>
BCArgsT<S> bc_args(ocfd_ctx* x) {
    BCArgsT<S> a;
    const View<S> V = view<S>(x);
    a.g = x->g;
    a.c = x->c;
    a.d = V.d; a.u = V.u; a.v = V.v; a.w = V.w; a.T = V.T; a.amu = V.amu; a.f = x->f;
    a.fs = x->fs;
    a.ub1 = x->ub1; a.fx = x->fxd; a.gz = x->gzd;
    a.x_begin = x->x_begin;
    a.ht = 1.0;
    a.epsl = x->cfg.bc_rpara[1];
    a.tw = x->cfg.bc_rpara[0];
    a.wall_not_normal = x->cfg.bc_npara[3];
    // the viscosity follows the primitives the boundary condition changes:
    // x = 0, y = 0 and y = ny-1 for IBC 108; x = 0, z = 0 and z = nz-1 for 124
    a.mu_faces = x->cfg.ibc == 108 ? 0x0d : x->cfg.ibc == 124 ? 0x31 : 0;
    a.in124 = a.up124 = a.coeff124 = a.udist124 = nullptr;
    a.sin_aoa = a.cos_aoa = 0.0;
    if (x->cfg.ibc == 124 && x->b124) {
        const Geo& g = x->g;
        const long long nyz = (long long)g.ny * g.nz, nxy = (long long)g.nx * g.ny;
        a.in124 = x->b124;
        a.up124 = x->cfg.bc_npara[2] == 1 ? x->b124 + 5 * nyz : nullptr;
        a.coeff124 = x->v_dist_need ? x->b124 + 5 * nyz + 5 * nxy : nullptr;
        a.udist124 = x->b124 + 5 * nyz + 8 * nxy;
        const double aoa = x->cfg.bc_rpara[0] * 3.141592653589793 / 180;
        a.sin_aoa = std::sin(aoa);
        a.cos_aoa = std::cos(aoa);
        a.tw = x->cfg.bc_rpara[1];
    }
    return a;
}

// OCFD_bc (src/OCFD_boundary.cu:18-92) followed by the viscosity of the
// faces it may change.
template <typename S>
int apply_bc(ocfd_ctx* x) {
    BCArgsT<S> a = bc_args<S>(x);
    if (x->cfg.ibc == 108) {
        double ht = 0.0;
        const double beta = x->cfg.bc_rpara[4];
        if (beta > 0.) {
            for (int m = 0; m < x->cfg.bc_npara[1] && m < OCFD_MTMAX; m++)
                ht = ht + x->TM[m] * std::sin((m + 1) * beta * x->tt);
        } else {
            ht = 1.;
        }
        a.ht = ht;
        // IBC 108 and the face refresh in one launch (OCFD_BC108_SPLIT=1 at
        // ocfd_create: the three separate launches, the same values)
        if (!x->bc108_split) {
            TRY(timed(x, "bc108", [&] { launch_bc108_faces(a, x->st); }));
            return 0;
        }
        TRY(timed(x, "bc108", [&] { launch_bc108(a, x->st); }));
    } else if (x->cfg.ibc == 124) {
        // bc_user_Liftbody3d (src/OCFD_boundary_Liftbody3D.cu:221-229): the
        // wall-disturbance time factor has no phase here
        double ht = 0.0;
        const double beta = x->cfg.bc_rpara[4];
        if (beta > 0.) {
            for (int m = 0; m < x->cfg.bc_npara[4] && m < OCFD_MTMAX; m++)
                ht = ht + x->TM[m] * std::sin((m + 1) * beta * x->tt);
        } else {
            ht = 1.;
        }
        a.ht = ht;
        TRY(timed(x, "bc124", [&] { launch_bc124_faces(a, x->cfg.bc_npara[0] == 1, x->st); }));
        return 0;
    } else {
        a.amu = nullptr;  // no face changes primitives: mu is already current
    }
    TRY(timed(x, "face_refresh", [&] { launch_face_refresh(a, x->st); }));
    return 0;
}

template <typename S>
MlpSensorArgsT<S> mlp_args(ocfd_ctx* x) {
    const View<S> V = view<S>(x);
    MlpSensorArgsT<S> a;
    a.g = x->g;
    a.c = x->c;
    a.d = V.d; a.u = V.u; a.v = V.v; a.w = V.w; a.T = V.T;
    for (int m = 0; m < M_COUNT; m++) a.M[m] = x->M[m];
    a.params = x->mlp_packed;
    a.lo = x->mlp_lo;
    a.hi = x->mlp_hi;
    a.fx = x->flag[0]; a.fy = x->flag[1]; a.fz = x->flag[2];
    a.prob = x->mlp_prob;
    return a;
}

template <typename S>
ViscArgsT<S> visc_args(ocfd_ctx* x) {
    const View<S> V = view<S>(x);
    ViscArgsT<S> va;
    va.g = x->g;
    va.c = x->c;
    va.svis = x->cfg.scheme_vis;
    for (int q = 0; q < 6; q++) va.bnd[q] = x->cfg.dif_bound[q];
    for (int q = 0; q < 3; q++) va.per[q] = x->cfg.iperiodic[q];
    va.u = V.u; va.v = V.v; va.w = V.w; va.T = V.T; va.amu = V.amu;
    for (int m = 0; m < M_COUNT; m++) va.M[m] = x->M[m];
    va.ev = V.ev; va.dv = V.dv; va.fs = x->fs;
    return va;
}

// The right-hand side of a stage: the inviscid part into du, the viscous
// fluxes into Ev and, unless the caller's stage takes their divergence itself
// (fused: launch_visc_stage), the viscous part into dv.  ghosts: the
// periodic ghost layers of the primitives already hold the stage's state.
template <typename S>
int rhs(ocfd_ctx* x, int krk, bool fused = false, bool ghosts = false) {
    const ocfd_config& C = x->cfg;
    if (!fused) TRY(need_dv(x));
    const View<S> V = view<S>(x);
    // hybrid_auto flags, once per step at the first stage: the plain sensor
    // before the periodic fill, as du_comput orders it (it reads the ghost
    // layers the previous stage's fill left); the learned sensor, which has
    // no counterpart in the reference, after the fill, from the filled ghost
    // layers, either in its own pass over all nodes or by the x sweep for
    // the nodes of its rows (i >= -1, j, k >= 0) and here for the ghost
    // planes j = -1 and k = -1 that only the y and z sweeps read (the
    // default; ocfd_set_sensor_fused chooses).  Both forms run the same
    // arithmetic (mlp_dev.h) and give the same flags.  With CHARTERIC = 1,
    // whose sweeps are other kernels, the separate pass.
    const bool learned = C.scheme_invis == OCFD_HYBRIDAUTO && krk == 1 && x->mlp_params;
    const bool fuse_learned = learned && x->mlp_fused && !C.charteric;
    if (C.scheme_invis == OCFD_HYBRIDAUTO && krk == 1 && !learned)
        TRY(timed(x, "sensor", [&] { launch_sensor(x->g, x->c, V.d, V.T, x->flag[0], x->flag[1], x->flag[2], x->st); }));
    if (!ghosts) TRY(fill_prims<S>(x));
    const MlpSensorArgsT<S> ma = mlp_args<S>(x);
    if (learned) {
        if (!fuse_learned) {
            TRY(timed(x, "sensor_mlp", [&] { launch_mlp_sensor(ma, 0, x->st); }));
        } else {
            TRY(timed(x, "sensor_mlp_planes", [&] { launch_mlp_sensor(ma, 1, x->st); }));
            TRY(timed(x, "sensor_mlp_planes", [&] { launch_mlp_sensor(ma, 2, x->st); }));
        }
    }
    const ViscArgsT<S> va = visc_args<S>(x);
    // the viscous terms read the primitives and metrics and write only Ev
    // and dv: on the second stream they overlap the sweeps (which write only
    // du).  Kernel timing runs everything in order on one stream.
    // Small grids (the merged sweeps) stay on one stream too: there the events
    // of a fork and a join cost more than the overlap gives (20x16x12: 104 -> 72
    // us a step, 61x47x39 130 -> 115, 64^3 275 -> 269, 97x61x53 528 either way).
    const bool overlap = !x->prof && !x->serial && x->du_parts == 1;
    if (overlap) {
        HIPCK(hipEventRecord(x->ev_fork, x->st));
        HIPCK(hipStreamWaitEvent(x->st2, x->ev_fork, 0));
        launch_visc_gf(va, x->st2);
        if (!fused) launch_visc_div(va, x->st2);
        HIPCK(hipGetLastError());
        HIPCK(hipEventRecord(x->ev_join, x->st2));
    }
    SweepArgsT<S> a;
    a.g = x->g;
    a.c = x->c;
    a.d = V.d; a.u = V.u; a.v = V.v; a.w = V.w; a.T = V.T;
    for (int m = 0; m < M_COUNT; m++) a.M[m] = x->M[m];
    a.du = V.du;
    a.fs = x->fs;
    const double h[3] = {x->g.hx, x->g.hy, x->g.hz};
    for (int dir = 0; dir < 3; dir++) {
        a.flag[dir] = x->flag[dir];
        a.h[dir] = h[dir];
        a.bl[dir] = C.dif_bound[2 * dir]; a.br[dir] = C.dif_bound[2 * dir + 1];
        a.nrp[dir] = C.non_ref[2 * dir]; a.nrm[dir] = C.non_ref[2 * dir + 1];
    }
    a.mlp.P = nullptr;
    a.mlp.lo = ma.lo; a.mlp.hi = ma.hi;
    a.mlp.prob = ma.prob;
    static const char* names[3] = {"sweep_x", "sweep_y", "sweep_z"};
    int lrc = 0;
    auto sweep = [&](int dir, const char* name) -> int {
        a.mlp.P = fuse_learned && dir == 0 ? ma.params : nullptr;
        return timed(x, a.mlp.P ? "sweep_x_learned" : name, [&] {
            lrc = C.charteric ? launch_sweep_char(C.scheme_invis, dir, a, x->st) : launch_sweep(C.scheme_invis, dir, a, x->st);
        });
    };
    if (x->du_parts == 3) {
        // the learned sensor's x sweep writes the flags that y and z read
        if (fuse_learned) TRY(sweep(0, names[0]));
        if (!lrc) TRY(sweep(fuse_learned ? SWEEP_YZ : SWEEP_ALL, "sweeps"));
    } else if (C.charteric || fuse_learned || !sweeps_xy<S>(C.scheme_invis, x->g)) {
        for (int dir = 0; dir < 3 && !lrc; dir++) TRY(sweep(dir, names[dir]));
    } else {
        TRY(sweep(SWEEP_XY, "sweep_xy"));
        if (!lrc) TRY(sweep(2, names[2]));
    }
    if (lrc) return fail(OCFD_ERR_UNSUPPORTED, "scheme not supported");
    if (overlap) {
        HIPCK(hipStreamWaitEvent(x->st, x->ev_join, 0));
    } else {
        TRY(timed(x, "visc_flux", [&] { launch_visc_gf(va, x->st); }));
        if (!fused) TRY(timed(x, "visc_div", [&] { launch_visc_div(va, x->st); }));
    }
    x->div_pending = fused;
    return 0;
}

// The viscous part of the last right-hand side, where its stage took it from
// Ev without leaving it in memory (Ev still holds that stage's fluxes).
template <typename S>
int finish_rhs_t(ocfd_ctx* x) {
    const ViscArgsT<S> va = visc_args<S>(x);
    TRY(timed(x, "visc_div", [&] { launch_visc_div(va, x->st); }));
    x->div_pending = false;
    return 0;
}
int finish_rhs(ocfd_ctx* x) {
    TRY(need_dv(x));
    if (!x->div_pending) return 0;
    return x->mixed ? finish_rhs_t<float>(x) : finish_rhs_t<double>(x);
}

bool filter_due(ocfd_ctx* x, int istep) {
    for (int m = 0; m < x->cfg.nfilter; m++)
        if (x->fpara[m][0] > 0 && istep % x->fpara[m][0] == 0) return true;
    return false;
}

// filtering (src/OCFD_filtering.cu:75-183) with the launch geometry of
// filter_{x,y,z}3d_shock (src/OCFD_filtering.cu:418-606): the x and y launches
// cover ib <= i < ie-1 in their direction; the z launch runs the y kernel and
// covers jb <= j < min(je-1, jb + 6*ceil((je-jb)/8)).
template <typename S>
int do_filter(ocfd_ctx* x) {
    if (!filter_due(x, x->istep)) return 0;
    const View<S> V = view<S>(x);
    int dirs = 0;
    for (int dir = 0; dir < 3; dir++)
        if (x->filter_dir[dir]) dirs |= 1 << dir;
    dirs &= periodic_dirs(x);
    if (dirs) {
        TRY(timed(x, "fill_filter", [&] { launch_fill(x->g, V.P, 1, x->fs, dirs, x->st); }));
        TRY(timed(x, "fill_filter", [&] { launch_fill(x->g, x->flap, 5, x->fs, dirs, x->st); }));
    }
    for (int m = 0; m < x->cfg.nfilter; m++) {
        if (!(x->tt <= x->cfg.filter_rpara[m][2])) continue;
        const int* p = x->fpara[m];
        if (p[0] <= 0 || x->istep % p[0] != 0) continue;
        if (p[10] != 2) continue;
        FilterArgsT<S> a;
        a.g = x->g; a.P = V.P; a.flap = x->flap; a.f = x->f; a.fs = x->fs;
        a.s0 = x->cfg.filter_rpara[m][0];
        a.rth = x->cfg.filter_rpara[m][1];
        const int ib = p[4], ie = p[5], jb = p[6], je = p[7], kb = p[8], ke = p[9];
        if (p[1] == 1) {
            a.dir = 0;
            a.lo[0] = ib; a.hi[0] = ie - 1; a.lo[1] = jb; a.hi[1] = je; a.lo[2] = kb; a.hi[2] = ke;
            TRY(timed(x, "filter", [&] { launch_filter(a, x->st); }));
        }
        if (p[2] == 1) {
            a.dir = 1;
            a.lo[0] = ib; a.hi[0] = ie; a.lo[1] = jb; a.hi[1] = je - 1; a.lo[2] = kb; a.hi[2] = ke;
            TRY(timed(x, "filter", [&] { launch_filter(a, x->st); }));
        }
        if (p[3] == 1) {
            a.dir = 1;
            int yend = jb + 6 * ((je - jb + 7) / 8);
            if (yend > je - 1) yend = je - 1;
            a.lo[0] = ib; a.hi[0] = ie; a.lo[1] = jb; a.hi[1] = yend; a.lo[2] = kb; a.hi[2] = ke;
            TRY(timed(x, "filter", [&] { launch_filter(a, x->st); }));
        }
    }
    return 0;
}

template <typename S>
StageArgsT<S> stage_args(ocfd_ctx* x, int krk, bool write_flap) {
    const View<S> V = view<S>(x);
    StageArgsT<S> sa;
    sa.g = x->g; sa.c = x->c; sa.krk = krk; sa.dt = x->cfg.dt;
    sa.f = x->f; sa.fn = x->fn; sa.du = V.du; sa.parts = x->du_parts; sa.dv = V.dv; sa.jac = x->M[M_JAC];
    sa.flap = write_flap ? x->flap : nullptr;
    sa.d = V.d; sa.u = V.u; sa.v = V.v; sa.w = V.w; sa.T = V.T; sa.amu = V.amu;
    // the pressure is read only after a step (filter, get_pressure, analysis):
    // the first two stages skip it
    sa.P = krk == 3 ? V.P : nullptr;
    sa.fs = x->fs;
    sa.faces = 0;
    for (int q = 0; q < 3; q++) sa.ghost[q] = 0;
    return sa;
}

template <typename S>
int one_step_t(ocfd_ctx* x) {
    std::swap(x->f, x->fn);
    const bool fdue = x->flap && filter_due(x, x->istep + 1);
    // without a boundary condition nothing changes the primitives between a
    // stage and the next right-hand side: the stage refreshes f on the faces
    // and, before stages 2 and 3, writes the periodic ghost layers itself (at
    // stage 1 the plain sensor still reads the layers of the stage before)
    const bool plain = x->cfg.ibc == 0;
    for (int krk = 1; krk <= 3; krk++) {
        StageArgsT<S> sa = stage_args<S>(x, krk, krk == 3 && fdue);
        sa.faces = plain;
        for (int q = 0; q < 3; q++) sa.ghost[q] = plain && krk < 3 && x->cfg.iperiodic[q];
        TRY(rhs<S>(x, krk, true, plain && krk > 1));
        TRY(timed(x, "visc_stage", [&] { launch_visc_stage(visc_args<S>(x), sa, x->st); }));
        if (!plain) TRY(apply_bc<S>(x));
    }
    x->istep++;
    x->tt += x->cfg.dt;
    TRY(do_filter<S>(x));
    return 0;
}

// Precision dispatch of the templated drivers.
int one_step(ocfd_ctx* x) { return x->mixed ? one_step_t<float>(x) : one_step_t<double>(x); }
int rhs_any(ocfd_ctx* x, int krk) { return x->mixed ? rhs<float>(x, krk) : rhs<double>(x, krk); }
int apply_bc_any(ocfd_ctx* x) { return x->mixed ? apply_bc<float>(x) : apply_bc<double>(x); }
int do_filter_any(ocfd_ctx* x) { return x->mixed ? do_filter<float>(x) : do_filter<double>(x); }

// IBC 108 set-up, bc_user_Compression_conner_init (src/OCFD_boundary_init.c:
// 376-516), with glibc rand() from its default seed as in the reference.
int ibc108_init(ocfd_ctx* x) {
    const ocfd_config& C = x->cfg;
    const Geo& g = x->g;
    const int nx = g.nx, ny = g.ny, nz = g.nz;
    if (!x->have_inlet) {
        // INLET_BOUNDARY = 1 reads the profile from flow1d-inlet.dat
        // (src/OCFD_boundary_init.c:376-395); without it the inlet would be
        // all zero (d = 0) and the run would turn to NaN
        if (C.bc_npara[2] == 1)
            return fail(OCFD_ERR_STATE, "IBC 108 with INLET_BOUNDARY = 1 needs the inlet profile "
                                        "(ocfd_set_inlet_profile / flow1d-inlet.dat) before ocfd_init");
        x->inlet.assign(4 * ny, 0.0);
        for (int j = 0; j < ny; j++) {
            x->inlet[j] = 1.; x->inlet[ny + j] = 1.; x->inlet[2 * ny + j] = 0.; x->inlet[3 * ny + j] = 1.;
        }
    }
    const int MZMAX = C.bc_npara[0], MTMAX = C.bc_npara[1];
    const double XDB = C.bc_rpara[2], XDE = C.bc_rpara[3], XUB = C.bc_rpara[6], SLZ = C.bc_rpara[7];
    x->x_begin = 0;
    for (int i = 0; i < nx; i++)
        if (x->coord_top_x[i] <= XUB) x->x_begin = i;
    std::vector<double> fx(nx), gz(nz);
    srand(1);
    const int MZ1 = std::abs(MZMAX);
    std::vector<double> faiz(MZ1 + 1), zl(MZ1 + 1);
    double ztmp = 0.;
    for (int k = 0; k < MZ1; k++) {
        faiz[k] = rand() / (double)RAND_MAX;
        zl[k] = (k == 0) ? 1. : zl[k - 1] / 1.25;
        ztmp = ztmp + zl[k];
    }
    for (int k = 0; k < MZ1; k++) zl[k] = zl[k] / ztmp;
    const double PI = 3.141592653589793;
    for (int i = 0; i < nx; i++) {
        const double xa = x->coord_x[i];
        if (xa >= XDB && xa <= XDE) {
            const double seta = 10. * PI * (xa - XDB) / (XDB - XDE);
            fx[i] = 4. / std::sqrt(27.) * std::sin(seta) * (1. - std::cos(seta));
        } else {
            fx[i] = 0.;
        }
    }
    for (int k = 0; k < nz; k++) {
        gz[k] = 0.;
        const double seta = x->coord_z[k] / SLZ;
        if (MZMAX > 0) {
            for (int m = 0; m < MZMAX; m++) gz[k] = gz[k] + zl[m] * std::sin(2. * PI * (m + 1) * (seta + faiz[m]));
        } else if (MZMAX == 0) {
            gz[k] = 1.;
        } else {
            gz[k] = std::sin(-2. * PI * MZMAX * seta);
        }
    }
    double Ttmp = 0.;
    for (int k = 0; k < MTMAX && k < OCFD_MTMAX; k++) {
        x->fait[k] = rand() / (double)RAND_MAX;
        x->TM[0] = 1.;
        if (k > 0) x->TM[k] = x->TM[k - 1] / 1.25;
        Ttmp = Ttmp + x->TM[k];
    }
    for (int k = 0; k < MTMAX && k < OCFD_MTMAX; k++) x->TM[k] = x->TM[k] / Ttmp;
    int rc = 0;
    if (!x->ub1) {
        x->ub1 = (double*)alloc_bytes(x, sizeof(double) * (4 * ny + nx + nz), rc);
        if (rc) return rc;
        x->fxd = x->ub1 + 4 * ny;
        x->gzd = x->fxd + nx;
    }
    HIPCK(hipMemcpyAsync(x->ub1, x->inlet.data(), sizeof(double) * 4 * ny, hipMemcpyHostToDevice, x->st));
    HIPCK(hipMemcpyAsync(x->fxd, fx.data(), sizeof(double) * nx, hipMemcpyHostToDevice, x->st));
    HIPCK(hipMemcpyAsync(x->gzd, gz.data(), sizeof(double) * nz, hipMemcpyHostToDevice, x->st));
    HIPCK(hipStreamSynchronize(x->st));
    return 0;
}

// bc_user_Liftbody3d_init (src/OCFD_boundary_init.c:95-318) with the
// parameters of bc_parameter (:50-71): the inlet table from the caller (the
// reference's flow-inlet-section.dat) when IF_WITHLEADING = 1, else from the
// loaded flow at i = 0; the upper table from the caller when
// IFLAG_UPPERBOUNDARY = 1; the wall disturbance (a multi-wave blowing/suction
// pattern along y when MZMAX != 0, else seeded noise on the wall points whose
// x lies in [WALL_DIS_BEGIN, WALL_DIS_END], along the mesh line normal to the
// wall) and the upper disturbance of u; the time factors TM.  The reference
// seeds rand() with the clock, so no two of its runs agree; glibc rand() from
// its default seed is used here, which makes runs repeatable.
template <typename S>
int ibc124_init(ocfd_ctx* x) {
    const ocfd_config& C = x->cfg;
    const Geo& g = x->g;
    const int nx = g.nx, ny = g.ny, nz = g.nz;
    const long long nyz = (long long)ny * nz, nxy = (long long)nx * ny;
    const int withleading = C.bc_npara[1], upper_mode = C.bc_npara[2], MZMAX = C.bc_npara[3], MTMAX = C.bc_npara[4];
    const double EPSL_WALL = C.bc_rpara[2], EPSL_UPPER = C.bc_rpara[3];
    const double DB = C.bc_rpara[5], DE = C.bc_rpara[6];
    const double PI = 3.141592653589793;
    if (x->mesh.size() != 3 * (size_t)nx * ny * nz) return fail(OCFD_ERR_STATE, "IBC 124 needs the mesh coordinates");
    std::vector<double> tab((size_t)(5 * nyz + 9 * nxy), 0.0);
    double* in = tab.data();
    double* up = in + 5 * nyz;
    double* coeff = up + 5 * nxy;
    double* udist = coeff + 3 * nxy;
    if (withleading == 1) {
        if (x->in124_host.size() != (size_t)(5 * nyz))
            return fail(OCFD_ERR_STATE, "IBC 124 with IF_WITHLEADING = 1 needs the inlet table (ocfd_set_bc_tables)");
        std::copy(x->in124_host.begin(), x->in124_host.end(), in);
    } else {
        const View<S> V = view<S>(x);
        const S* f[5] = {V.d, V.u, V.v, V.w, V.T};
        for (int m = 0; m < 5; m++) {
            const void* hv;
            D2H(hv, x, f[m], sizeof(S) * (size_t)x->fs);
            const S* h = (const S*)hv;
            for (int k = 0; k < nz; k++)
                for (int j = 0; j < ny; j++) in[m * nyz + (long long)k * ny + j] = double(h[(size_t)gidx(g, 0, j, k)]);
        }
    }
    if (upper_mode == 1) {
        if (x->up124_host.size() != (size_t)(5 * nxy))
            return fail(OCFD_ERR_STATE, "IBC 124 with IFLAG_UPPERBOUNDARY = 1 needs the upper table (ocfd_set_bc_tables)");
        std::copy(x->up124_host.begin(), x->up124_host.end(), up);
    }
    const double* X = x->mesh.data();
    const double* Y = X + (size_t)nx * ny * nz;
    const double* Z = Y + (size_t)nx * ny * nz;
    auto at = [&](int i, int j, int k) { return ((size_t)k * ny + j) * nx + i; };
    srand(1);
    bool need = false;
    if (MZMAX != 0) {
        // get_xy_blow_suction_multiwave (:320-372) along x at j = k = 0 and y
        need = true;
        const int MZ1 = std::abs(MZMAX);
        std::vector<double> faiz(MZ1 + 1), zl(MZ1 + 1), fx(nx), gz(ny);
        double ztmp = 0.;
        for (int k = 0; k < MZ1; k++) {
            faiz[k] = rand() / (double)RAND_MAX;
            zl[k] = (k == 0) ? 1. : zl[k - 1] / 1.25;
            ztmp = ztmp + zl[k];
        }
        for (int k = 0; k < MZ1; k++) zl[k] = zl[k] / ztmp;
        for (int i = 0; i < nx; i++) {
            const double xa = X[at(i, 0, 0)];
            if (xa >= DB && xa <= DE) {
                const double seta = 10. * PI * (xa - DB) / (DB - DE);
                fx[i] = 4. / std::sqrt(27.) * std::sin(seta) * (1. - std::cos(seta));
            } else {
                fx[i] = 0.;
            }
        }
        for (int j = 0; j < ny; j++) {
            gz[j] = 0.;
            const double seta = ((double)j) / ny;
            if (MZMAX > 0) {
                for (int m = 0; m < MZMAX; m++) gz[j] = gz[j] + zl[m] * std::sin(2. * PI * (m + 1) * (seta + faiz[m]));
            } else {
                gz[j] = std::sin(-2. * PI * MZMAX * seta);
            }
        }
        for (int j = 0; j < ny; j++)
            for (int i = 0; i < nx; i++) {
                const double vdw = fx[i] * gz[j];
                const size_t o = (size_t)j * nx + i;
                coeff[o] = 0;
                coeff[nxy + o] = EPSL_WALL * vdw * std::sin(2 * PI / ny * j);
                coeff[2 * nxy + o] = EPSL_WALL * vdw * std::cos(2 * PI / ny * j);
            }
    } else {
        std::vector<double> tv(nxy), tu(nxy);
        for (int j = 0; j < ny; j++)
            for (int i = 0; i < nx; i++) {
                double r = (rand() / (double)RAND_MAX - 0.5) * 2.0;
                tv[(size_t)j * nx + i] = EPSL_WALL * r;
                r = (rand() / (double)RAND_MAX - 0.5) * 2.0;
                tu[(size_t)j * nx + i] = EPSL_UPPER * r;
            }
        for (int j = 0; j < ny; j++)
            for (int i = 0; i < nx; i++) {
                const size_t o = (size_t)j * nx + i;
                const double xw = X[at(i, j, 0)];
                double vdw = 0.0;
                if (xw >= DB && xw <= DE) {
                    need = true;
                    vdw = tv[o];
                }
                udist[o] = tu[o];
                const double xn = X[at(i, j, 1)] - X[at(i, j, 0)], yn = Y[at(i, j, 1)] - Y[at(i, j, 0)];
                const double zn = Z[at(i, j, 1)] - Z[at(i, j, 0)];
                const double sn = std::sqrt(xn * xn + yn * yn + zn * zn);
                coeff[o] = vdw * xn / sn;
                coeff[nxy + o] = vdw * yn / sn;
                coeff[2 * nxy + o] = vdw * zn / sn;
            }
    }
    x->v_dist_need = need;
    // get_fait_multifrequancy (:501-517)
    double Ttmp = 0.;
    for (int k = 0; k < MTMAX && k < OCFD_MTMAX; k++) {
        x->fait[k] = rand() / (double)RAND_MAX;
        x->TM[0] = 1.;
        if (k > 0) x->TM[k] = x->TM[k - 1] / 1.25;
        Ttmp = Ttmp + x->TM[k];
    }
    for (int k = 0; k < MTMAX && k < OCFD_MTMAX; k++) x->TM[k] = x->TM[k] / Ttmp;
    int rc = 0;
    if (!x->b124) {
        x->b124 = (double*)alloc_bytes(x, sizeof(double) * tab.size(), rc);
        if (rc) return rc;
    }
    HIPCK(hipMemcpyAsync(x->b124, tab.data(), sizeof(double) * tab.size(), hipMemcpyHostToDevice, x->st));
    HIPCK(hipStreamSynchronize(x->st));
    return 0;
}

// Metrics of the symmetry planes of IBC 124 (boundary_Jac3d_Liftbody_Ajac,
// src/OCFD_Comput_Jacobian3d.cu:619-662): y ghosts mirrored, with the sign of
// a vector's y component (and of the y row of the cofactors) flipped.
int ibc124_mirror_metrics(ocfd_ctx* x) {
    if (x->cfg.ibc != 124 || x->cfg.bc_npara[0] != 1) return 0;
    // M order: Akx Aky Akz Aix Aiy Aiz Asx Asy Asz Ajac
    const double sign[M_COUNT] = {1, -1, 1, -1, 1, -1, 1, -1, 1, 1};
    for (int m = 0; m < M_COUNT; m++)
        TRY(timed(x, "mirror", [&] { launch_mirror_y(x->g, x->M[m], sign[m], x->st); }));
    return 0;
}

// ocfd_init body: pri_to_cons over the interior (src/OCFD_init.cu:99-110),
// the IBC 108 set-up, then the NS_solver_real prologue
// (src/OCFD_NS_Solver.cu:46-54): ghost fill, BC, viscosity everywhere.
template <typename S>
int init_fields(ocfd_ctx* x) {
    BCArgsT<S> a = bc_args<S>(x);
    TRY(timed(x, "prim2cons", [&] { launch_p2c_all(a, x->st); }));
    if (x->cfg.ibc == 108) TRY(ibc108_init(x));
    if (x->cfg.ibc == 124) TRY(ibc124_init<S>(x));
    TRY(fill_prims<S>(x));
    TRY(apply_bc<S>(x));
    a = bc_args<S>(x);
    TRY(timed(x, "amu", [&] { launch_amu_all(a, x->st); }));
    return 0;
}

// ---------------------------------------------------------------------------
// Scratch of ocfd_diagnostics_noalloc: one file-scope device array, which
// every GPU the library runs on holds at its own address until the process
// ends.  In host code `scratch` is only a stand-in for the symbol: its device
// address is fetched once per device (noalloc_setup, called by ocfd_create
// with the device current) and only that address is used afterwards.
// Layout in doubles: [0,4) results {sum E, sum T, NaN count, negative count},
// then the partial sums of E and of T (diag_sum_blocks each), then the
// 2*DIAG_SCAN_BLOCKS int counts.
// ---------------------------------------------------------------------------
constexpr long long NOALLOC_DOUBLES = OCFD_NOALLOC_SCRATCH_BYTES / 8;
static __device__ __align__(256) double scratch[NOALLOC_DOUBLES];

constexpr int NOALLOC_MAX_DEVICES = 64;
std::mutex g_scratch_mu;
double* g_scratch_dev[NOALLOC_MAX_DEVICES] = {};

int noalloc_setup(int device) {
    if (device < 0 || device >= NOALLOC_MAX_DEVICES) return fail(OCFD_ERR_ARG, "device index out of range");
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (g_scratch_dev[device]) return 0;
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p)
        return fail(OCFD_ERR_HIP, std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
    g_scratch_dev[device] = static_cast<double*>(p);
    return 0;
}

long long noalloc_doubles_needed(const Geo& g) {
    return 4 + 2LL * diag_sum_blocks(g) + DIAG_SCAN_BLOCKS;  // the counts: 2 ints per scan block
}

}  // namespace

// ===========================================================================
// C ABI
// ===========================================================================
extern "C" {

const char* ocfd_last_error(void) { return g_err.c_str(); }

int ocfd_create(const ocfd_config* cfg, int device, ocfd_ctx** out) {
    if (!cfg || !out) return fail(OCFD_ERR_ARG, "null argument");
    *out = nullptr;
    const ocfd_config& C = *cfg;
    if (C.nx < 8 || C.ny < 8 || C.nz < 8) return fail(OCFD_ERR_CONFIG, "GRID_3D: each size must be >= 8");
    if ((C.npx0 > 1) || (C.npy0 > 1) || (C.npz0 > 1))
        return fail(OCFD_ERR_UNSUPPORTED, "PARALLEL_3D must be 1 1 1 (one GPU)");
    if (C.stream_mode != 0) return fail(OCFD_ERR_UNSUPPORTED, "STREAM=1 needs multiple ranks; use STREAM=0");
    // src/OCFD_Schemes_Choose.cu:103-145: the characteristic kernels exist for
    // WENO7_SYMBO(_LIM) and hybrid_auto only (the reference prints a message
    // and leaves the inviscid term out for the others)
    if (C.charteric != 0 && C.charteric != 1) return fail(OCFD_ERR_CONFIG, "CHARTERIC must be 0 or 1");
    if (C.charteric == 1 && C.scheme_invis != OCFD_WENO7_SYMBO && C.scheme_invis != OCFD_WENO7_SYMBO_LIM &&
        C.scheme_invis != OCFD_HYBRIDAUTO)
        return fail(OCFD_ERR_UNSUPPORTED, "CHARTERIC=1 needs WENO7_SYMBO, WENO7_SYMBO_LIM or SCHEME_HYBRIDAUTO");
    if (!supported_scheme(C.scheme_invis)) return fail(OCFD_ERR_CONFIG, "SCHEME_INVIS not recognised");
    if (C.scheme_vis != OCFD_CD6 && C.scheme_vis != OCFD_CD8) return fail(OCFD_ERR_CONFIG, "SCHEME_VIS not recognised");
    if (C.scheme_invis == OCFD_HYBRIDAUTO && C.hy_style != 2)
        return fail(OCFD_ERR_UNSUPPORTED, "hybrid_auto: only HY_STYLE = 2 (Jameson sensor) is supported");
    if (C.ibc != 0 && C.ibc != 108 && C.ibc != 124)
        return fail(OCFD_ERR_UNSUPPORTED, "IBC: only 0, 108 and 124 are supported");
    // INIT_STAT = 0 runs the reference's built-in test geometry and a
    // different boundary routine (bc_user_Liftbody3d_simple), not provided
    if (C.ibc == 124 && C.init_stat != 1) return fail(OCFD_ERR_UNSUPPORTED, "IBC 124 needs INIT_STAT = 1");
    // the wall-disturbance time tables TM/fait hold OCFD_MTMAX modes
    // (MTMAX is BC_NPARA[1] for IBC 108, BC_NPARA[4] for IBC 124; the
    // reference sizes them to MTMAX)
    if ((C.ibc == 108 && C.bc_npara[1] > OCFD_MTMAX) || (C.ibc == 124 && C.bc_npara[4] > OCFD_MTMAX))
        return fail(OCFD_ERR_CONFIG, "MTMAX (BC_NPARA) above " + std::to_string(OCFD_MTMAX) + " is not supported");
    if (C.precision != OCFD_PREC_FP64 && C.precision != OCFD_PREC_MIXED)
        return fail(OCFD_ERR_CONFIG, "PRECISION: FP64 or MIXED");
    const long long npts = (long long)(C.nx + 8) * (C.ny + 8) * (C.nz + 8);
    if (npts > (1LL << 31)) return fail(OCFD_ERR_CONFIG, "grid too large for one context");

    ocfd_ctx* x = new ocfd_ctx();
    x->cfg = C;
    x->device = device;
    if (hipSetDevice(device) != hipSuccess) {
        delete x;
        return fail(OCFD_ERR_HIP, "hipSetDevice failed");
    }
    if (const int rc = noalloc_setup(device)) {
        delete x;
        return rc;
    }
    if (hipStreamCreateWithFlags(&x->st, hipStreamNonBlocking) != hipSuccess ||
        hipStreamCreateWithFlags(&x->st2, hipStreamNonBlocking) != hipSuccess ||
        hipEventCreateWithFlags(&x->ev_fork, hipEventDisableTiming) != hipSuccess ||
        hipEventCreateWithFlags(&x->ev_join, hipEventDisableTiming) != hipSuccess) {
        ocfd_destroy(x);
        return fail(OCFD_ERR_HIP, "hipStreamCreate / hipEventCreate failed");
    }
    if (const char* e = std::getenv("OCFD_SERIAL")) x->serial = std::atoi(e) != 0;
    if (const char* e = std::getenv("OCFD_BC108_SPLIT")) x->bc108_split = std::atoi(e) != 0;
    if (const char* e = std::getenv("OCFD_GRAPH")) x->graphs = std::atoi(e) != 0;
    Geo& g = x->g;
    g.nx = C.nx; g.ny = C.ny; g.nz = C.nz;
    // row pitch: 128-byte rows in FP64; 32 elements (128 bytes) in FP32 too
    // on the mixed path
    const int pitch = C.precision == OCFD_PREC_MIXED ? 32 : 16;
    g.ldx = ((C.nx + 8) + pitch - 1) / pitch * pitch;
    g.ldy = C.ny + 8;
    g.sz = (long long)g.ldx * g.ldy;
    g.off0 = 4 + (long long)g.ldx * (4 + (long long)g.ldy * 4);
    // src/OCFD_init.cu:29-31
    g.hx = 1.0 / (C.nx - 1.0);
    g.hy = 1.0 / (C.ny - 1.0);
    g.hz = 1.0 / (C.nz - 1.0);
    x->fs = g.sz * (C.nz + 8) + 32;  // a multiple of 32 elements: every field of a group stays aligned
    // opencfd_para_init, src/OCFD_init.cu:381-410
    Consts& c = x->c;
    const double gm = C.gamma, Ma = C.ama;
    const double Tref = C.t_ref <= 0 ? 288.150 : C.t_ref;
    c.gamma = gm; c.ama = Ma;
    c.cv = 1.0 / (gm * (gm - 1.0) * Ma * Ma);
    c.cp = 1.0 / ((gm - 1.0) * Ma * Ma);
    c.tsb = 110.4 / Tref;
    c.amu_c0 = 1.0 / C.re * (1.0 + 110.4 / Tref);
    c.tmp0 = 1.0 / (2.0 * gm);
    c.split_c1 = 2.0 * (gm - 1.0);
    c.split_c3 = (3.0 - gm) / (2.0 * (gm - 1.0));
    c.vis_c = c.cp / C.pr;
    c.epsl_sw = C.epsl_sw;
    c.p00 = 1.0 / (gm * Ma * Ma);
    c.rama = 1.0 / Ma;
    c.hy_i1 = C.hy_dp_intv[0];
    c.hy_i2 = C.hy_dp_intv[1];
    c.tv_lim = 5.0;  // src/parameters.c:75-76
    c.tv_max = 0.2;

    x->mixed = C.precision == OCFD_PREC_MIXED;
    // the characteristic sweeps run one direction at a time
    x->du_parts = !C.charteric && sweeps_merged(g) ? 3 : 1;
    int rc = 0;
    double* met = alloc_fields(x, M_COUNT, rc);
    double* fa = rc ? nullptr : alloc_fields(x, 5, rc);
    double* fb = rc ? nullptr : alloc_fields(x, 5, rc);
    double* gr = rc ? nullptr : alloc_fields(x, 12, rc);
    if (!rc && C.nfilter > 0) x->flap = alloc_fields(x, 5, rc);
    if (!x->mixed) {
        double* prim = rc ? nullptr : alloc_fields(x, 6, rc);  // d,u,v,w,T,P
        double* dua = rc ? nullptr : alloc_fields(x, 5 * x->du_parts, rc);
        double* am = rc ? nullptr : alloc_fields(x, 1, rc);
        double* ev = rc ? nullptr : alloc_fields(x, 12, rc);
        if (!rc) {
            x->d = prim; x->u = prim + x->fs; x->v = prim + 2 * x->fs; x->w = prim + 3 * x->fs;
            x->T = prim + 4 * x->fs; x->P = prim + 5 * x->fs;
            x->du = dua; x->amu = am; x->ev = ev;
        }
    } else {
        float* prim = rc ? nullptr : alloc_fields_f32(x, 6, rc);
        float* dua = rc ? nullptr : alloc_fields_f32(x, 5 * x->du_parts, rc);
        float* am = rc ? nullptr : alloc_fields_f32(x, 1, rc);
        float* ev = rc ? nullptr : alloc_fields_f32(x, 12, rc);
        if (!rc) {
            x->sd = prim; x->su = prim + x->fs; x->sv = prim + 2 * x->fs; x->sw = prim + 3 * x->fs;
            x->sT = prim + 4 * x->fs; x->sP = prim + 5 * x->fs;
            x->sdu = dua; x->samu = am; x->sev = ev;
        }
    }
    for (int dd = 0; dd < 3 && !rc; dd++) x->flag[dd] = alloc_bytes(x, (size_t)x->fs, rc);
    if (rc) {
        ocfd_destroy(x);
        return rc;
    }
    for (int m = 0; m < M_COUNT; m++) x->M[m] = met + m * x->fs;
    x->f = fa; x->fn = fb; x->grad = gr;
    // metrics start at 1.0 everywhere (src/OCFD_Comput_Jacobian3d.cu:34-48)
    launch_set(g, met - 12, x->fs * M_COUNT + 16, 1.0, x->st);
    // set_para_filtering clamps at one rank (src/OCFD_filtering.cu:20-73)
    for (int k = 0; k < C.nfilter && k < OCFD_MAX_FILTERS; k++) {
        int* p = x->fpara[k];
        for (int q = 0; q < 11; q++) p[q] = C.filter_npara[k][q];
        if (p[1] == 1) x->filter_dir[0] = true;
        if (p[2] == 1) x->filter_dir[1] = true;
        if (p[3] == 1) x->filter_dir[2] = true;
        if (!C.iperiodic[0]) { p[4] = std::max(p[4], 6); p[5] = std::min(p[5], C.nx - 5); }
        if (!C.iperiodic[1]) { p[6] = std::max(p[6], 6); p[7] = std::min(p[7], C.ny - 5); }
        if (!C.iperiodic[2]) { p[8] = std::max(p[8], 6); p[9] = std::min(p[9], C.nz - 5); }
        // keep every read inside the 4 ghost layers even for ranges given
        // beyond the grid (the reference would read out of its arrays)
        p[4] = std::max(p[4], 0); p[5] = std::min(p[5], C.nx);
        p[6] = std::max(p[6], 0); p[7] = std::min(p[7], C.ny);
        p[8] = std::max(p[8], 0); p[9] = std::min(p[9], C.nz);
    }
    if (hipEventCreate(&x->step_a) != hipSuccess || hipEventCreate(&x->step_b) != hipSuccess ||
        hipStreamSynchronize(x->st) != hipSuccess) {
        ocfd_destroy(x);
        return fail(OCFD_ERR_HIP, "initial fill failed");
    }
    *out = x;
    return 0;
}

int ocfd_destroy(ocfd_ctx* x) {
    if (!x) return 0;
    // teardown: errors are not actionable here and are ignored
    if (x->st) (void)hipStreamSynchronize(x->st);
    for (auto& r : x->recs) { (void)hipEventDestroy(r.a); (void)hipEventDestroy(r.b); }
    for (auto e : x->pool) (void)hipEventDestroy(e);
    if (x->step_a) (void)hipEventDestroy(x->step_a);
    if (x->step_b) (void)hipEventDestroy(x->step_b);
    if (x->st2) (void)hipStreamSynchronize(x->st2);
    for (void* p : x->allocs) (void)hipFree(p);
    if (x->pin) (void)hipHostFree(x->pin);
    for (auto e : x->pin_ev)
        if (e) (void)hipEventDestroy(e);
    if (x->ev_fork) (void)hipEventDestroy(x->ev_fork);
    if (x->ev_join) (void)hipEventDestroy(x->ev_join);
    if (x->st2) (void)hipStreamDestroy(x->st2);
    if (x->st) (void)hipStreamDestroy(x->st);
    delete x;
    return 0;
}

int ocfd_load_mesh(ocfd_ctx* x, const double* X, const double* Y, const double* Z) {
    if (!x || !X || !Y || !Z) return fail(OCFD_ERR_ARG, "null argument");
    const Geo& g = x->g;
    const ocfd_config& C = x->cfg;
    // coordinates go into three scratch fields of the gradient buffer:
    // ghosts keep 1.0, periodic faces get the unshifted wrapped values
    // (src/OCFD_Comput_Jacobian3d.cu:120-146)
    double* crd = x->grad + 9 * x->fs;  // fields 9,10,11
    const double* src[3] = {X, Y, Z};
    for (int q = 0; q < 3; q++) TRY(upload_interior(x, crd + q * x->fs, src[q], 1.0));
    TRY(fill_periodic(x, crd, 3, "metric_fill"));
    if (C.ibc == 124 && C.bc_npara[0] == 1) {
        // boundary_Jac3d_Axx (src/OCFD_Comput_Jacobian3d.cu:592-617): the
        // coordinates of the symmetry planes' ghosts, y odd
        for (int q = 0; q < 3; q++)
            TRY(timed(x, "mirror", [&] { launch_mirror_y(g, crd + q * x->fs, q == 1 ? -1.0 : 1.0, x->st); }));
    }
    // 9 derivatives into gradient fields 0..8: xi xj xk yi yj yk zi zj zk
    for (int q = 0; q < 3; q++)
        for (int dir = 0; dir < 3; dir++)
            TRY(timed(x, "metric_deriv", [&] {
                launch_metric_deriv(g, crd + q * x->fs, dir, C.jac_bound[dir], x->grad + (3 * q + dir) * x->fs, x->st);
            }));
    TRY(timed(x, "cofactors", [&] { launch_cofactors(g, x->grad, x->fs, x->M, x->st); }));
    TRY(fill_periodic(x, x->M[0], M_COUNT, "metric_fill"));
    TRY(ibc124_mirror_metrics(x));
    HIPCK(hipStreamSynchronize(x->st));
    // host copies for the IBC 108 set-up and the Jacobi writer
    const size_t nxy = (size_t)g.nx * g.ny;
    const size_t nall = nxy * g.nz;
    x->mesh.resize(3 * nall);
    std::memcpy(x->mesh.data(), X, sizeof(double) * nall);
    std::memcpy(x->mesh.data() + nall, Y, sizeof(double) * nall);
    std::memcpy(x->mesh.data() + 2 * nall, Z, sizeof(double) * nall);
    x->coord_x.assign(X, X + g.nx);                         // x at (i, 0, 0)
    x->coord_top_x.assign(X + (size_t)(g.ny - 1) * g.nx, X + (size_t)(g.ny - 1) * g.nx + g.nx);
    x->coord_z.resize(g.nz);
    for (int k = 0; k < g.nz; k++) x->coord_z[k] = Z[(size_t)k * nxy];
    x->have_grid = true;
    return 0;
}

int ocfd_load_jacobi(ocfd_ctx* x, const double* a13) {
    if (!x || !a13) return fail(OCFD_ERR_ARG, "null argument");
    const Geo& g = x->g;
    const size_t n = (size_t)g.nx * g.ny * g.nz;
    // file order Axx Ayy Azz Akx Aky Akz Aix Aiy Aiz Asx Asy Asz Ajac
    for (int m = 0; m < M_COUNT; m++) TRY(upload_interior(x, x->M[m], a13 + (3 + m) * n, 1.0));
    TRY(fill_periodic(x, x->M[0], M_COUNT, "metric_fill"));
    TRY(ibc124_mirror_metrics(x));  // src/OCFD_init.cu:116-122
    HIPCK(hipStreamSynchronize(x->st));
    const double* X = a13;
    const double* Z = a13 + 2 * n;
    const size_t nxy = (size_t)g.nx * g.ny;
    x->mesh.assign(a13, a13 + 3 * n);
    x->coord_x.assign(X, X + g.nx);
    x->coord_top_x.assign(X + (size_t)(g.ny - 1) * g.nx, X + (size_t)(g.ny - 1) * g.nx + g.nx);
    x->coord_z.resize(g.nz);
    for (int k = 0; k < g.nz; k++) x->coord_z[k] = Z[(size_t)k * nxy];
    x->have_grid = true;
    return 0;
}

int ocfd_load_flow(ocfd_ctx* x, const double* d, const double* u, const double* v, const double* w,
                   const double* T, int istep, double tt) {
    if (!x || !d || !u || !v || !w || !T) return fail(OCFD_ERR_ARG, "null argument");
    const double* src[5] = {d, u, v, w, T};
    if (x->mixed) {
        float* dst[5] = {x->sd, x->su, x->sv, x->sw, x->sT};
        for (int q = 0; q < 5; q++) TRY(upload_any(x, dst[q], src[q], 0.0));
    } else {
        double* dst[5] = {x->d, x->u, x->v, x->w, x->T};
        for (int q = 0; q < 5; q++) TRY(upload_any(x, dst[q], src[q], 0.0));
    }
    x->istep = istep;
    x->tt = tt;
    x->have_flow = true;
    return 0;
}

int ocfd_set_inlet_profile(ocfd_ctx* x, const double* prof) {
    if (!x || !prof) return fail(OCFD_ERR_ARG, "null argument");
    x->inlet.assign(prof, prof + 4 * x->g.ny);
    x->have_inlet = true;
    return 0;
}

int ocfd_set_bc_tables(ocfd_ctx* x, const double* inlet5, const double* upper5) {
    if (!x) return fail(OCFD_ERR_ARG, "null context");
    const long long nyz = (long long)x->g.ny * x->g.nz, nxy = (long long)x->g.nx * x->g.ny;
    if (inlet5) x->in124_host.assign(inlet5, inlet5 + 5 * nyz);
    if (upper5) x->up124_host.assign(upper5, upper5 + 5 * nxy);
    return 0;
}

int ocfd_init(ocfd_ctx* x) {
    if (!x) return fail(OCFD_ERR_ARG, "null context");
    if (!x->have_grid || !x->have_flow) return fail(OCFD_ERR_STATE, "load the grid and the flow before ocfd_init");
    TRY(x->mixed ? init_fields<float>(x) : init_fields<double>(x));
    HIPCK(hipStreamSynchronize(x->st));
    x->inited = true;
    return 0;
}

int ocfd_rhs(ocfd_ctx* x, int krk) {
    if (!x || !x->inited) return fail(OCFD_ERR_STATE, "context not initialised");
    TRY(rhs_any(x, krk));
    TRY(flush_prof(x));
    return 0;
}

// Whether a step's launches have the same arguments every step, so that a
// HIP graph of two steps (after which f and fn are back in place) can be
// replayed: no filter (due every N steps), no time-dependent wall
// disturbance (its factor ht follows tt), no kernel timing.
bool steps_replayable(const ocfd_ctx* x) {
    const ocfd_config& C = x->cfg;
    if (!x->graphs || x->prof || x->serial || C.nfilter > 0) return false;
    if ((C.ibc == 108 || C.ibc == 124) && C.bc_rpara[4] > 0.) return false;
    return true;
}

// Steps [0, n) with n >= 4 as replays of one captured graph of two steps:
// the capture runs the host side of two steps (swaps, counters) and records
// their launches, the first replay executes them, each further replay
// advances the counters as two steps do.  Returns the steps done (even).
// If the capture, its instantiation or the first replay fails, the host
// state (f/fn, step counter, time) is put back as it was, graphs are turned
// off for this context and done = 0, so the caller runs the steps eagerly.
int step_graph(ocfd_ctx* x, int n, int& done) {
    done = 0;
    double* const f0 = x->f;
    double* const fn0 = x->fn;
    const int istep0 = x->istep;
    const double tt0 = x->tt;
    auto give_up = [&] {
        x->f = f0;
        x->fn = fn0;
        x->istep = istep0;
        x->tt = tt0;
        x->graphs = false;
        (void)hipGetLastError();
        return 0;
    };
    hipGraph_t gr = nullptr;
    hipGraphExec_t ge = nullptr;
    if (hipStreamBeginCapture(x->st, hipStreamCaptureModeRelaxed) != hipSuccess) return give_up();
    int rc = one_step(x);
    if (!rc) rc = one_step(x);
    const hipError_t ec = hipStreamEndCapture(x->st, &gr);
    if (rc || ec != hipSuccess) {
        if (gr) (void)hipGraphDestroy(gr);
        return give_up();
    }
    if (hipGraphInstantiate(&ge, gr, nullptr, nullptr, 0) != hipSuccess) {
        (void)hipGraphDestroy(gr);
        return give_up();
    }
    hipError_t e = hipSuccess;
    for (; done + 2 <= n; done += 2) {
        const int istep_before = x->istep;
        const double tt_before = x->tt;
        if (done > 0) {  // the host side of two more steps (the swaps cancel)
            x->istep += 2;
            x->tt += x->cfg.dt;
            x->tt += x->cfg.dt;
        }
        e = hipGraphLaunch(ge, x->st);
        if (e != hipSuccess) {
            x->istep = istep_before;
            x->tt = tt_before;
            break;
        }
    }
    (void)hipStreamSynchronize(x->st);
    (void)hipGraphExecDestroy(ge);
    (void)hipGraphDestroy(gr);
    if (e != hipSuccess) {
        if (done == 0) return give_up();
        return fail(OCFD_ERR_HIP, std::string("hipGraphLaunch: ") + hipGetErrorString(e));
    }
    return 0;
}

int ocfd_step(ocfd_ctx* x, int nsteps) {
    if (!x || !x->inited) return fail(OCFD_ERR_STATE, "context not initialised");
    HIPCK(hipEventRecord(x->step_a, x->st));
    int s = 0;
    if (nsteps >= 4 && steps_replayable(x)) TRY(step_graph(x, nsteps, s));
    for (; s < nsteps; s++) TRY(one_step(x));
    HIPCK(hipEventRecord(x->step_b, x->st));
    HIPCK(hipEventSynchronize(x->step_b));
    float ms = 0.f;
    HIPCK(hipEventElapsedTime(&ms, x->step_a, x->step_b));
    x->last_step_ms = ms;
    TRY(flush_prof(x));
    return 0;
}

int ocfd_sync(ocfd_ctx* x) {
    if (!x) return fail(OCFD_ERR_ARG, "null context");
    HIPCK(hipStreamSynchronize(x->st));
    return 0;
}

double ocfd_last_step_ms(ocfd_ctx* x) { return x ? x->last_step_ms : 0.0; }

int ocfd_get_flow(ocfd_ctx* x, double* d, double* u, double* v, double* w, double* T, int* istep, double* tt) {
    if (!x) return fail(OCFD_ERR_ARG, "null context");
    double* dst[5] = {d, u, v, w, T};
    if (x->mixed) {
        // the stored FP32 primitives: like the reference's they lag the
        // filter, which changes only f at the end of a step
        const float* src[5] = {x->sd, x->su, x->sv, x->sw, x->sT};
        TRY(download_fields(x, src, dst, 5));
    } else {
        const double* src[5] = {x->d, x->u, x->v, x->w, x->T};
        TRY(download_fields(x, src, dst, 5));
    }
    if (istep) *istep = x->istep;
    if (tt) *tt = x->tt;
    return 0;
}

int ocfd_get_state(ocfd_ctx* x, double* f5) {
    if (!x || !f5) return fail(OCFD_ERR_ARG, "null argument");
    const size_t n = (size_t)x->g.nx * x->g.ny * x->g.nz;
    const double* src[5];
    double* dst[5];
    for (int m = 0; m < 5; m++) {
        src[m] = x->f + m * x->fs;
        dst[m] = f5 + m * n;
    }
    return download_fields(x, src, dst, 5);
}

int ocfd_get_du(ocfd_ctx* x, double* du5) {
    if (!x || !du5) return fail(OCFD_ERR_ARG, "null argument");
    TRY(finish_rhs(x));
    const size_t n = (size_t)x->g.nx * x->g.ny * x->g.nz;
    double* out[5];
    for (int m = 0; m < 5; m++) out[m] = du5 + m * n;
    return download_packed<double>(x, out, 5, [&](double* d) {
        if (x->mixed) launch_pack_du(stage_args<float>(x, 1, false), d, x->st);
        else launch_pack_du(stage_args<double>(x, 1, false), d, x->st);
    });
}

int ocfd_get_pressure(ocfd_ctx* x, double* p) {
    if (!x || !p) return fail(OCFD_ERR_ARG, "null argument");
    return x->mixed ? download_any(x, (const float*)x->sP, p) : download_any(x, (const double*)x->P, p);
}

int ocfd_get_amu(ocfd_ctx* x, double* a) {
    if (!x || !a) return fail(OCFD_ERR_ARG, "null argument");
    // the time step does not keep the viscosity field (the gradient kernel
    // forms mu from T): get_Amu's kernel fills it from the current T first
    if (x->mixed) {
        const BCArgsT<float> b = bc_args<float>(x);
        TRY(timed(x, "amu", [&] { launch_amu_all(b, x->st); }));
        return download_any(x, (const float*)x->samu, a);
    }
    const BCArgsT<double> b = bc_args<double>(x);
    TRY(timed(x, "amu", [&] { launch_amu_all(b, x->st); }));
    return download_any(x, (const double*)x->amu, a);
}

int ocfd_get_metrics(ocfd_ctx* x, double* a13) {
    if (!x || !a13) return fail(OCFD_ERR_ARG, "null argument");
    const size_t n = (size_t)x->g.nx * x->g.ny * x->g.nz;
    if (x->mesh.size() == 3 * n) std::memcpy(a13, x->mesh.data(), sizeof(double) * 3 * n);
    else std::memset(a13, 0, sizeof(double) * 3 * n);
    const double* src[M_COUNT];
    double* dst[M_COUNT];
    for (int m = 0; m < M_COUNT; m++) {
        src[m] = x->M[m];
        dst[m] = a13 + (3 + m) * n;
    }
    return download_fields(x, src, dst, M_COUNT);
}

int ocfd_diagnostics(ocfd_ctx* x, double* mean_energy, double* mean_T, long long* n_nan_T, long long* n_neg_T) {
    if (!x || !x->inited) return fail(OCFD_ERR_STATE, "context not initialised");
    const Geo& g = x->g;
    const int nb = diag_sum_blocks(g);
    int rc = 0;
    if (!x->diag_part) {
        x->diag_part = (double*)alloc_bytes(x, sizeof(double) * 2 * nb, rc);
        if (rc) return rc;
        x->diag_scan = (int*)alloc_bytes(x, sizeof(int) * 2 * DIAG_SCAN_BLOCKS, rc);
        if (rc) return rc;
    }
    const double* E = x->f + 4 * x->fs;
    if (x->mixed)
        TRY(timed(x, "diag", [&] { launch_diag(g, E, x->sT, x->diag_part, x->diag_part + nb, x->diag_scan, x->st); }));
    else
        TRY(timed(x, "diag", [&] { launch_diag(g, E, x->T, x->diag_part, x->diag_part + nb, x->diag_scan, x->st); }));
    std::vector<double> part((size_t)2 * nb);
    std::vector<int> cnt((size_t)2 * DIAG_SCAN_BLOCKS);
    const void* hv;
    D2H(hv, x, x->diag_part, sizeof(double) * 2 * nb);
    std::memcpy(part.data(), hv, sizeof(double) * 2 * nb);
    D2H(hv, x, x->diag_scan, sizeof(int) * 2 * DIAG_SCAN_BLOCKS);
    std::memcpy(cnt.data(), hv, sizeof(int) * 2 * DIAG_SCAN_BLOCKS);
    double se = 0.0, st = 0.0;
    for (int b = 0; b < nb; b++) { se += part[b]; st += part[nb + b]; }
    long long nn = 0, ng = 0;
    for (int b = 0; b < DIAG_SCAN_BLOCKS; b++) { nn += cnt[2 * b]; ng += cnt[2 * b + 1]; }
    const double npts = (double)g.nx * g.ny * g.nz;  // ana_residual divides by the global point count
    if (mean_energy) *mean_energy = se / npts;
    if (mean_T) *mean_T = st / npts;
    if (n_nan_T) *n_nan_T = nn;
    if (n_neg_T) *n_neg_T = ng;
    return 0;
}

int ocfd_diagnostics_noalloc(ocfd_ctx* x, double* mean_energy, double* mean_T, long long* n_nan_T,
                             long long* n_neg_T) {
    if (!x) return fail(OCFD_ERR_ARG, "null context");
    const Geo& g = x->g;
    const long long need = noalloc_doubles_needed(g);
    if (need > NOALLOC_DOUBLES)
        return fail(OCFD_ERR_UNSUPPORTED,
                    "ocfd_diagnostics_noalloc: this grid needs " + std::to_string(need * 8) +
                        " bytes of scratch, above the " + std::to_string(NOALLOC_DOUBLES * 8) +
                        " bytes of OCFD_NOALLOC_SCRATCH_BYTES (use ocfd_diagnostics)");
    if (!x->inited) return fail(OCFD_ERR_STATE, "context not initialised");
    double* s = g_scratch_dev[x->device];
    if (!s) return fail(OCFD_ERR_STATE, "scratch address not set up for this device");
    const long long nb = diag_sum_blocks(g);
    double* partE = s + 4;
    double* partT = partE + nb;
    int* scan = reinterpret_cast<int*>(partT + nb);
    const double* E = x->f + 4 * x->fs;
    // every partial, count and result slot is written by these launches:
    // nothing left by an earlier call is read
    if (x->mixed) launch_diag(g, E, x->sT, partE, partT, scan, x->st);
    else launch_diag(g, E, x->T, partE, partT, scan, x->st);
    launch_diag_final(partE, partT, nb, scan, s, x->st);
    HIPCK(hipGetLastError());
    double out[4];
    HIPCK(hipMemcpyAsync(out, s, sizeof(out), hipMemcpyDeviceToHost, x->st));
    HIPCK(hipStreamSynchronize(x->st));
    long long cnt[2];
    std::memcpy(cnt, out + 2, sizeof(cnt));
    const double npts = (double)g.nx * g.ny * g.nz;
    if (mean_energy) *mean_energy = out[0] / npts;
    if (mean_T) *mean_T = out[1] / npts;
    if (n_nan_T) *n_nan_T = cnt[0];
    if (n_neg_T) *n_neg_T = cnt[1];
    return 0;
}

int ocfd_set_sensor(ocfd_ctx* x, const float* params, float lo, float hi) {
    if (!x) return fail(OCFD_ERR_ARG, "null context");
    if (!params) {
        x->mlp_params = nullptr;  // the buffers stay allocated for a later call
        return 0;
    }
    if (!(lo >= 0.f && hi <= 1.f && lo <= hi)) return fail(OCFD_ERR_ARG, "confidence band needs 0 <= lo <= hi <= 1");
    int rc = 0;
    if (!x->mlp_prob) {
        float* pb = alloc_fields_f32(x, 1, rc);
        if (rc) return rc;
        float* pp = (float*)alloc_bytes(x, sizeof(float) * MLP_NPARAM, rc);
        if (rc) return rc;
        float* pk = (float*)alloc_bytes(x, sizeof(float) * MLP_PACKED_FLOATS, rc);
        if (rc) return rc;
        x->mlp_prob = pb;
        x->mlp_store = pp;
        x->mlp_packed = pk;
    }
    HIPCK(hipMemcpyAsync(x->mlp_store, params, sizeof(float) * MLP_NPARAM, hipMemcpyHostToDevice, x->st));
    launch_mlp_pack(x->mlp_store, x->mlp_packed, x->st);
    HIPCK(hipGetLastError());
    HIPCK(hipStreamSynchronize(x->st));
    x->mlp_params = x->mlp_store;
    x->mlp_lo = lo;
    x->mlp_hi = hi;
    return 0;
}

int ocfd_set_sensor_fused(ocfd_ctx* x, int on) {
    if (!x) return fail(OCFD_ERR_ARG, "null context");
    x->mlp_fused = on != 0;
    return 0;
}

int ocfd_get_sensor_prob(ocfd_ctx* x, float* prob) {
    if (!x || !prob) return fail(OCFD_ERR_ARG, "null argument");
    if (!x->mlp_prob) return fail(OCFD_ERR_STATE, "the learned sensor has not been set");
    const Geo& g = x->g;
    const void* hv;
    D2H(hv, x, x->mlp_prob, sizeof(float) * x->fs);
    const float* h = (const float*)hv;
    for (int k = 0; k < g.nz; k++)
        for (int j = 0; j < g.ny; j++)
            std::memcpy(prob + ((size_t)k * g.ny + j) * g.nx, &h[(size_t)gidx(g, 0, j, k)], sizeof(float) * g.nx);
    return 0;
}

int ocfd_write_jacobi(ocfd_ctx* x, const char* path) {
    if (!x || !path) return fail(OCFD_ERR_ARG, "null argument");
    if (!x->have_grid) return fail(OCFD_ERR_STATE, "load the grid before writing OCFD3d-Jacobi.dat");
    const Geo& g = x->g;
    std::vector<double> a((size_t)13 * g.nx * g.ny * g.nz);
    TRY(ocfd_get_metrics(x, a.data()));
    return ocfd_write_records(path, g.nx, g.ny, g.nz, 13, a.data());
}

int ocfd_get_hybrid_flags(ocfd_ctx* x, int8_t* fx, int8_t* fy, int8_t* fz) {
    if (!x) return fail(OCFD_ERR_ARG, "null context");
    const Geo& g = x->g;
    int8_t* outs[3] = {fx, fy, fz};
    for (int dd = 0; dd < 3; dd++) {
        if (!outs[dd]) continue;
        const void* hv;
        D2H(hv, x, x->flag[dd], (size_t)x->fs);
        const int8_t* h = (const int8_t*)hv;
        const int ex = g.nx + (dd == 0), ey = g.ny + (dd == 1), ez = g.nz + (dd == 2);
        for (int k = 0; k < ez; k++)
            for (int j = 0; j < ey; j++)
                for (int i = 0; i < ex; i++)
                    outs[dd][(size_t)i + (size_t)ex * ((size_t)j + (size_t)ey * k)] =
                        h[(size_t)gidx(g, i - (dd == 0), j - (dd == 1), k - (dd == 2))];
    }
    return 0;
}

// ---------------------------------------------------------------------------
// Analysis events (OCFD_ana, src/OCFD_ana.cu:588-619).
// ---------------------------------------------------------------------------
}  // extern "C"

namespace {

// Whole LAP box of a field (index = gidx) as doubles.
template <typename S>
int download_box(ocfd_ctx* x, const S* src, std::vector<double>& out) {
    const void* hv;
    D2H(hv, x, src, sizeof(S) * (size_t)x->fs);
    const S* h = (const S*)hv;
    out.assign(h, h + x->fs);
    return 0;
}
int download_box_any(ocfd_ctx* x, int field, std::vector<double>& out) {
    // field: 0..4 = d,u,v,w,T
    if (x->mixed) {
        float* f[5] = {x->sd, x->su, x->sv, x->sw, x->sT};
        return download_box(x, f[field], out);
    }
    double* f[5] = {x->d, x->u, x->v, x->w, x->T};
    return download_box(x, f[field], out);
}

// ana_NAN_and_NT (src/OCFD_ana.cu:105-222): T over the LAP box.  The device
// scan counts; the locations are printed from a host copy only when there is
// something to print.
int ana_nan_nt(ocfd_ctx* x) {
    const Geo& g = x->g;
    long long nnan = 0, nneg = 0;
    TRY(ocfd_diagnostics(x, nullptr, nullptr, &nnan, &nneg));
    std::printf("It is analyzing NAN......\n");
    if (nnan || nneg) {
        std::vector<double> T;
        TRY(download_box_any(x, 4, T));
        bool first = true;
        for (int k = -4; k < g.nz + 4 && nnan && first; k++)
            for (int j = -4; j < g.ny + 4 && first; j++)
                for (int i = -4; i < g.nx + 4 && first; i++)
                    if (std::isnan(T[(size_t)gidx(g, i, j, k)])) {
                        std::printf("NAN occured in Global ID(%d , %d , %d)\n\n", i, j, k);
                        first = false;
                    }
        for (int k = -4; k < g.nz + 4 && nneg; k++)
            for (int j = -4; j < g.ny + 4; j++)
                for (int i = -4; i < g.nx + 4; i++)
                    if (T[(size_t)gidx(g, i, j, k)] < 0)
                        std::printf("Negative T occured in Global ID(%d , %d , %d)\n\n", i, j, k);
    }
    if (nneg > 10) {
        std::printf("Negative T points %lld > %d\n", nneg, 10);
        return fail(OCFD_ERR_NUMERIC, "negative T at " + std::to_string(nneg) + " points");
    }
    if (nnan) {
        std::printf("NAN occured , program Abort\n");
        return fail(OCFD_ERR_NUMERIC, "NaN in T");
    }
    return 0;
}

// ana_time_average (src/OCFD_ana.cu:256-298) with the averaged-file read of
// read_file (src/OCFD_IO.c:94-151) at the first call and OCFD_save(1, ...)
// (src/OCFD_IO.c:156-214) every KSTEP_SAVE steps.
int ana_time_average(ocfd_ctx* x) {
    const Geo& g = x->g;
    const size_t n = (size_t)g.nx * g.ny * g.nz;
    std::printf("It is averaging......\n");
    if (!x->avg) {
        int rc = 0;
        double* a = alloc_fields(x, 5, rc);  // zeroed: init_time_average
        if (rc) return rc;
        x->avg = a;
        x->avg_n = 0;
        x->avg_tt = 0.0;
        const char* name = "opencfd.average";
        FILE* fh = std::fopen(name, "rb");
        if (!fh) {
            std::printf("Average file: %s is not exit\n\n", name);
        } else {
            std::fclose(fh);
            std::printf("read average_data begin\n");
            std::vector<double> h(5 * n);
            int is = 0;
            double t = 0.0;
            TRY(ocfd_read_flow_file(name, g.nx, g.ny, g.nz, h.data(), h.data() + n, h.data() + 2 * n,
                                    h.data() + 3 * n, h.data() + 4 * n, &is, &t));
            x->avg_n = is;
            x->avg_tt = t;
            std::printf("Istep_average=%d , tt_average=%lf\n", is, t);
            for (int m = 0; m < 5; m++) TRY(upload_interior(x, x->avg + m * x->fs, h.data() + m * n, 0.0));
            std::printf("read average_data ok\n");
        }
    }
    if (x->mixed)
        TRY(timed(x, "time_avg", [&] {
            launch_time_avg(g, x->sd, x->su, x->sv, x->sw, x->sT, x->avg, x->fs, x->avg_n, x->st);
        }));
    else
        TRY(timed(x, "time_avg", [&] {
            launch_time_avg(g, x->d, x->u, x->v, x->w, x->T, x->avg, x->fs, x->avg_n, x->st);
        }));
    x->avg_n += 1;
    x->avg_tt += x->cfg.dt;
    if (x->cfg.kstep_save > 0 && x->istep % x->cfg.kstep_save == 0) {
        std::vector<double> h(5 * n);
        for (int m = 0; m < 5; m++) TRY(download_any(x, (const double*)(x->avg + m * x->fs), h.data() + m * n));
        char name[64];
        std::snprintf(name, sizeof name, "OCFD%08d.average", x->avg_n);
        std::printf("write data file: %s\n", name);
        TRY(ocfd_write_flow_file(name, g.nx, g.ny, g.nz, h.data(), h.data() + n, h.data() + 2 * n, h.data() + 3 * n,
                                 h.data() + 4 * n, x->avg_n, x->avg_tt));
    }
    return 0;
}

bool is_hybrid(const ocfd_ctx* x) { return x->cfg.scheme_invis == OCFD_HYBRIDAUTO && x->flag[0]; }

// HybridAuto_scheme_IO (src/OCFD_Schemes_hybrid_auto.cu:706-744) through
// write_2d_XY (src/OCFD_IO_mpi.c:63-125) at k = NZ/2: each line is the flag
// at flat index (k, j, i+1) of the direction's face array read with the
// interior row length of that array, and the pressure at node (i+1, j, k).
// The reference prints an array that style 2 never writes (pPP_d); the
// pressure p00*d*T that the style-2 sensor reads is printed instead.
int ana_scheme_io(ocfd_ctx* x) {
    if (!is_hybrid(x)) return fail(OCFD_ERR_STATE, "analysis style 102 needs SCHEME_HYBRIDAUTO");
    const Geo& g = x->g;
    const int nx = g.nx, ny = g.ny, nz = g.nz, K = nz / 2;
    std::vector<int8_t> fl[3] = {std::vector<int8_t>((size_t)(nx + 1) * ny * nz),
                                 std::vector<int8_t>((size_t)nx * (ny + 1) * nz),
                                 std::vector<int8_t>((size_t)nx * ny * (nz + 1))};
    TRY(ocfd_get_hybrid_flags(x, fl[0].data(), fl[1].data(), fl[2].data()));
    std::vector<double> d, T;
    TRY(download_box_any(x, 0, d));
    TRY(download_box_any(x, 4, T));
    const double p00 = x->c.p00;
    const char dn[3] = {'x', 'y', 'z'};
    for (int dd = 0; dd < 3; dd++) {
        const size_t rowlen = dd == 0 ? nx + 1 : nx, rows = dd == 1 ? ny + 1 : ny;
        char name[64];
        std::snprintf(name, sizeof name, "Scheme_%c%08d.dat", dn[dd], x->istep);
        FILE* fh = std::fopen(name, "w");
        if (!fh) return fail(OCFD_ERR_IO, std::string("cannot write ") + name);
        std::fprintf(fh, "variables=scheme\n");
        std::fprintf(fh, "zone i=%d, j=%d\n", nx, ny);
        for (int j = 0; j < ny; j++)
            for (int i = 0; i < nx; i++) {
                const int flag = fl[dd][((size_t)K * rows + j) * rowlen + i + 1];
                const size_t q = (size_t)gidx(g, i + 1, j, K);
                std::fprintf(fh, "%08d%15.6lf\n", flag, p00 * d[q] * T[q]);
            }
        std::fclose(fh);
    }
    return 0;
}

// get_Q (src/OCFD_ana.cu:384-458): Q.dat as nz records of the interior, and
// Q%02d%02d%02d.dat (rank 0 0 0) as text x y z Q.  The reference's kernel
// writes the LAP positions of an array allocated without ghost layers; the
// values it means, Q at the interior points, are what is written here.
int ana_q(ocfd_ctx* x) {
    const Geo& g = x->g;
    const size_t n = (size_t)g.nx * g.ny * g.nz;
    std::vector<double> q(n);
    TRY(ocfd_get_q(x, q.data()));
    TRY(ocfd_write_records("Q.dat", g.nx, g.ny, g.nz, 1, q.data()));
    FILE* fh = std::fopen("Q000000.dat", "w");
    if (!fh) return fail(OCFD_ERR_IO, "cannot write Q000000.dat");
    std::fprintf(fh, "variables=x,y,z,Q\n");
    std::fprintf(fh, "zone i=%d ,j=%d ,k=%d\n", g.nx, g.ny, g.nz);
    const bool have = x->mesh.size() == 3 * n;
    for (size_t p = 0; p < n; p++)
        std::fprintf(fh, "%15.6f%15.6f%15.6f%15.6f\n", have ? x->mesh[p] : 0.0, have ? x->mesh[n + p] : 0.0,
                     have ? x->mesh[2 * n + p] : 0.0, q[p]);
    std::fclose(fh);
    return 0;
}

// ana_saveplaneXY/YZ/XZ (src/OCFD_ana.cu:459-586) with write_2d_XYa/YZa/XZa
// (src/OCFD_IO_mpi.c:128-260): per listed plane a header record {Istep, tt}
// appended to Savedata-XY%03d.dat (YZ, XZ), then for each plane of the band
// one record per variable d,u,v,w,T.  ANA_NPARA& = count, band width, first
// plane of each band (0-based global indices).
int ana_planes(ocfd_ctx* x, int style, int id) {
    const ocfd_config& C = x->cfg;
    const Geo& g = x->g;
    if (id < 0 || id >= C.nana) return fail(OCFD_ERR_ARG, "analysis event id out of range");
    const int* np = C.ana_npara[id];
    const int count = np[0], band = np[1];
    if (count < 0 || count + 2 > OCFD_ANA_NPARA || band < 0)
        return fail(OCFD_ERR_CONFIG, "ANA_NPARA: bad plane count or band width");
    const int dir = style == 104 ? 2 : style == 105 ? 0 : 1;  // the fixed index: z, x, y
    const int nfix = dir == 0 ? g.nx : dir == 1 ? g.ny : g.nz;
    for (int p = 0; p < count; p++)
        if (np[p + 2] < 0 || np[p + 2] + band > nfix) return fail(OCFD_ERR_CONFIG, "ANA_NPARA: plane outside the grid");
    const size_t n = (size_t)g.nx * g.ny * g.nz;
    std::vector<double> h(5 * n);
    int is = 0;
    double t = 0.0;
    TRY(ocfd_get_flow(x, h.data(), h.data() + n, h.data() + 2 * n, h.data() + 3 * n, h.data() + 4 * n, &is, &t));
    const char* tag = style == 104 ? "XY" : style == 105 ? "YZ" : "XZ";
    for (int p = 0; p < count; p++) {
        std::printf("Save data ...., %d, %lf, %d\n", x->istep, x->tt, p);
        char name[64];
        std::snprintf(name, sizeof name, "Savedata-%s%03d.dat", tag, p);
        FILE* fh = std::fopen(name, "ab");
        if (!fh) return fail(OCFD_ERR_IO, std::string("cannot write ") + name);
        const int32_t hb = (int32_t)(sizeof(double) + sizeof(int));
        const int32_t is32 = x->istep;
        std::fwrite(&hb, 4, 1, fh);
        std::fwrite(&is32, 4, 1, fh);
        std::fwrite(&x->tt, 8, 1, fh);
        std::fwrite(&hb, 4, 1, fh);
        std::vector<double> plane;
        for (int s = np[p + 2]; s < np[p + 2] + band; s++)
            for (int m = 0; m < 5; m++) {
                const double* f = h.data() + m * n;
                plane.clear();
                if (dir == 2) {  // XY: x fastest, then y
                    plane.assign(f + (size_t)s * g.nx * g.ny, f + (size_t)(s + 1) * g.nx * g.ny);
                } else if (dir == 0) {  // YZ: y fastest, then z
                    for (int k = 0; k < g.nz; k++)
                        for (int j = 0; j < g.ny; j++) plane.push_back(f[((size_t)k * g.ny + j) * g.nx + s]);
                } else {  // XZ: x fastest, then z
                    for (int k = 0; k < g.nz; k++)
                        for (int i = 0; i < g.nx; i++) plane.push_back(f[((size_t)k * g.ny + s) * g.nx + i]);
                }
                const int32_t nb = (int32_t)(plane.size() * sizeof(double));
                std::fwrite(&nb, 4, 1, fh);
                std::fwrite(plane.data(), sizeof(double), plane.size(), fh);
                std::fwrite(&nb, 4, 1, fh);
            }
        std::fclose(fh);
    }
    return 0;
}

}  // namespace

extern "C" {

int ocfd_get_q(ocfd_ctx* x, double* q) {
    if (!x || !q) return fail(OCFD_ERR_ARG, "null argument");
    if (!x->inited) return fail(OCFD_ERR_STATE, "context not initialised");
    const ocfd_config& C = x->cfg;
    double* out = x->grad;  // first scratch field
    if (x->mixed) {
        ViscArgsT<float> va;
        va.g = x->g; va.c = x->c; va.svis = C.scheme_vis;
        for (int m = 0; m < 6; m++) va.bnd[m] = C.dif_bound[m];
        va.u = x->su; va.v = x->sv; va.w = x->sw; va.T = x->sT; va.amu = x->samu;
        for (int m = 0; m < M_COUNT; m++) va.M[m] = x->M[m];
        va.ev = x->sev; va.dv = x->sdv; va.fs = x->fs;
        TRY(timed(x, "qcrit", [&] { launch_qcrit(va, out, x->st); }));
    } else {
        ViscArgsT<double> va;
        va.g = x->g; va.c = x->c; va.svis = C.scheme_vis;
        for (int m = 0; m < 6; m++) va.bnd[m] = C.dif_bound[m];
        va.u = x->u; va.v = x->v; va.w = x->w; va.T = x->T; va.amu = x->amu;
        for (int m = 0; m < M_COUNT; m++) va.M[m] = x->M[m];
        va.ev = x->ev; va.dv = x->dv; va.fs = x->fs;
        TRY(timed(x, "qcrit", [&] { launch_qcrit(va, out, x->st); }));
    }
    return download_any(x, (const double*)out, q);
}

int ocfd_get_time_average(ocfd_ctx* x, double* d, double* u, double* v, double* w, double* T, int* nsamples,
                          double* tt_avg) {
    if (!x) return fail(OCFD_ERR_ARG, "null context");
    if (!x->avg) return fail(OCFD_ERR_STATE, "no time average yet (analysis style 101)");
    double* outs[5] = {d, u, v, w, T};
    for (int m = 0; m < 5; m++)
        if (outs[m]) TRY(download_any(x, (const double*)(x->avg + m * x->fs), outs[m]));
    if (nsamples) *nsamples = x->avg_n;
    if (tt_avg) *tt_avg = x->avg_tt;
    return 0;
}

// HybridAuto_scheme_Proportion (src/OCFD_Schemes_hybrid_auto.cu:747-830):
// counts of 1, 2 and anything else over each face array, divided by the
// product of the two other global sizes and then by N + NP0 (NP0 = 1).
int ocfd_hybrid_proportions(ocfd_ctx* x, double* frac9) {
    if (!x || !frac9) return fail(OCFD_ERR_ARG, "null argument");
    if (!is_hybrid(x)) return fail(OCFD_ERR_STATE, "hybrid proportions need SCHEME_HYBRIDAUTO");
    const Geo& g = x->g;
    const size_t sz[3] = {(size_t)(g.nx + 1) * g.ny * g.nz, (size_t)g.nx * (g.ny + 1) * g.nz,
                          (size_t)g.nx * g.ny * (g.nz + 1)};
    std::vector<int8_t> fl[3] = {std::vector<int8_t>(sz[0]), std::vector<int8_t>(sz[1]), std::vector<int8_t>(sz[2])};
    TRY(ocfd_get_hybrid_flags(x, fl[0].data(), fl[1].data(), fl[2].data()));
    const double other[3] = {(double)g.ny * g.nz, (double)g.nx * g.nz, (double)g.nx * g.ny};
    const double len[3] = {(double)g.nx + 1, (double)g.ny + 1, (double)g.nz + 1};
    for (int dd = 0; dd < 3; dd++) {
        double t1 = 0.0, t2 = 0.0, t3 = 0.0;
        for (int8_t f : fl[dd]) {
            if (f == 1) t1 += 1.0;
            else if (f == 2) t2 += 1.0;
            else t3 += 1.0;
        }
        frac9[3 * dd] = t1 / other[dd] / len[dd];
        frac9[3 * dd + 1] = t2 / other[dd] / len[dd];
        frac9[3 * dd + 2] = t3 / other[dd] / len[dd];
    }
    return 0;
}

int ocfd_analysis(ocfd_ctx* x, int style, int id) {
    if (!x) return fail(OCFD_ERR_ARG, "null context");
    if (!x->inited) return fail(OCFD_ERR_STATE, "context not initialised");
    switch (style) {
        case 100: return ana_nan_nt(x);
        case 101: return ana_time_average(x);
        case 102: return ana_scheme_io(x);
        case 103: return ana_q(x);
        case 104:
        case 105:
        case 106: return ana_planes(x, style, id);
        case 107: {
            if (!is_hybrid(x)) return 0;
            double fr[9];
            TRY(ocfd_hybrid_proportions(x, fr));
            const char* dn[3] = {"X", "Y", "Z"};
            for (int dd = 0; dd < 3; dd++)
                std::printf("The first type scheme of Hybrid schemes in direction %s is %lf%%, second is %lf%%, "
                            "third is %lf%%\n",
                            dn[dd], fr[3 * dd], fr[3 * dd + 1], fr[3 * dd + 2]);
            return 0;
        }
        default: return 0;
    }
}

// ---------------------------------------------------------------------------
// Learned-sensor trainer: training samples, parameters and Adam moments on one
// device.  No counterpart in the reference.
// ---------------------------------------------------------------------------
struct ocfd_mlp {
    int device = 0;
    hipStream_t st = nullptr;
    long long cap = 0, n = 0;
    float *X = nullptr, *y = nullptr;   // [cap][24], [cap]
    float *P = nullptr, *m1 = nullptr, *m2 = nullptr, *grad = nullptr;
    float *part = nullptr;              // partial gradient sums of one batch
    size_t part_cap = 0;                // floats
    float *prob = nullptr;              // probabilities of one ocfd_mlp_predict call
    int prob_cap = 0;
    int* idx = nullptr;                 // sample order of one epoch
    float* loss = nullptr;              // one value per batch of an epoch
    long long loss_cap = 0;
    int adam_t = 0;
    std::vector<void*> allocs;
};

namespace {
int mlp_alloc(ocfd_mlp* m, void** p, size_t bytes) {
    void* q = nullptr;  // *p keeps what it had if this fails
    if (hipMalloc(&q, bytes) != hipSuccess) return fail(OCFD_ERR_HIP, "hipMalloc failed (" + std::to_string(bytes) + " bytes)");
    m->allocs.push_back(q);
    *p = q;
    return 0;
}
int mlp_ensure_batch(ocfd_mlp* m, int nb) {
    const size_t n = mlp_part_floats(nb);
    if (n <= m->part_cap) return 0;
    TRY(mlp_alloc(m, (void**)&m->part, sizeof(float) * n));
    m->part_cap = n;
    return 0;
}
// splitmix64: the seeded sample order of the training epochs
uint64_t splitmix(uint64_t& s) {
    uint64_t z = (s += 0x9E3779B97F4A7C15ULL);
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
    return z ^ (z >> 31);
}
}  // namespace

int ocfd_mlp_create(int device, long long capacity, ocfd_mlp** out) {
    if (!out || capacity <= 0) return fail(OCFD_ERR_ARG, "bad argument");
    *out = nullptr;
    ocfd_mlp* m = new ocfd_mlp();
    m->device = device;
    m->cap = capacity;
    int rc = 0;
    if (hipSetDevice(device) != hipSuccess || hipStreamCreateWithFlags(&m->st, hipStreamNonBlocking) != hipSuccess) {
        delete m;
        return fail(OCFD_ERR_HIP, "hipSetDevice / hipStreamCreate failed");
    }
    rc = mlp_alloc(m, (void**)&m->X, sizeof(float) * 24 * (size_t)capacity);
    if (!rc) rc = mlp_alloc(m, (void**)&m->y, sizeof(float) * (size_t)capacity);
    if (!rc) rc = mlp_alloc(m, (void**)&m->idx, sizeof(int) * (size_t)capacity);
    if (!rc) rc = mlp_alloc(m, (void**)&m->P, sizeof(float) * MLP_NPARAM);
    if (!rc) rc = mlp_alloc(m, (void**)&m->m1, sizeof(float) * MLP_NPARAM);
    if (!rc) rc = mlp_alloc(m, (void**)&m->m2, sizeof(float) * MLP_NPARAM);
    if (!rc) rc = mlp_alloc(m, (void**)&m->grad, sizeof(float) * (MLP_NPARAM + 1));
    if (rc) {
        ocfd_mlp_destroy(m);
        return rc;
    }
    // seeded He-style initial weights (uniform with the variance of the
    // normal He initialisation), zero biases, zero Adam moments
    std::vector<float> p(MLP_NPARAM, 0.f);
    uint64_t s = 0x5EED5EEDULL;
    auto uni = [&](float bound) { return (float)((splitmix(s) >> 11) * (1.0 / 9007199254740992.0) * 2.0 - 1.0) * bound; };
    for (int i = 0; i < 768; i++) p[i] = uni(std::sqrt(3.f * 2.f / 24.f));
    for (int i = 800; i < 1824; i++) p[i] = uni(std::sqrt(3.f * 2.f / 32.f));
    for (int i = 1856; i < 1888; i++) p[i] = uni(std::sqrt(3.f / 32.f));
    if (hipMemcpy(m->P, p.data(), sizeof(float) * MLP_NPARAM, hipMemcpyHostToDevice) != hipSuccess ||
        hipMemset(m->m1, 0, sizeof(float) * MLP_NPARAM) != hipSuccess ||
        hipMemset(m->m2, 0, sizeof(float) * MLP_NPARAM) != hipSuccess) {
        ocfd_mlp_destroy(m);
        return fail(OCFD_ERR_HIP, "trainer initialisation failed");
    }
    *out = m;
    return 0;
}

int ocfd_mlp_destroy(ocfd_mlp* m) {
    if (!m) return 0;
    if (m->st) (void)hipStreamSynchronize(m->st);
    for (void* p : m->allocs) (void)hipFree(p);
    if (m->st) (void)hipStreamDestroy(m->st);
    delete m;
    return 0;
}

int ocfd_mlp_set_params(ocfd_mlp* m, const float* params) {
    if (!m || !params) return fail(OCFD_ERR_ARG, "null argument");
    HIPCK(hipMemcpy(m->P, params, sizeof(float) * MLP_NPARAM, hipMemcpyHostToDevice));
    HIPCK(hipMemset(m->m1, 0, sizeof(float) * MLP_NPARAM));
    HIPCK(hipMemset(m->m2, 0, sizeof(float) * MLP_NPARAM));
    m->adam_t = 0;
    return 0;
}

int ocfd_mlp_get_params(ocfd_mlp* m, float* params) {
    if (!m || !params) return fail(OCFD_ERR_ARG, "null argument");
    HIPCK(hipStreamSynchronize(m->st));
    HIPCK(hipMemcpy(params, m->P, sizeof(float) * MLP_NPARAM, hipMemcpyDeviceToHost));
    return 0;
}

long long ocfd_mlp_sample_count(ocfd_mlp* m) { return m ? m->n : 0; }

int ocfd_mlp_clear(ocfd_mlp* m) {
    if (!m) return fail(OCFD_ERR_ARG, "null argument");
    m->n = 0;
    return 0;
}

int ocfd_mlp_put_samples(ocfd_mlp* m, const float* X, const float* y, long long n) {
    if (!m || !X || !y || n < 0) return fail(OCFD_ERR_ARG, "bad argument");
    if (m->n + n > m->cap) return fail(OCFD_ERR_ARG, "trainer capacity exceeded");
    HIPCK(hipMemcpy(m->X + 24 * m->n, X, sizeof(float) * 24 * (size_t)n, hipMemcpyHostToDevice));
    HIPCK(hipMemcpy(m->y + m->n, y, sizeof(float) * (size_t)n, hipMemcpyHostToDevice));
    m->n += n;
    return 0;
}

int ocfd_mlp_get_samples(ocfd_mlp* m, long long first, long long n, float* X, float* y) {
    if (!m || first < 0 || n < 0 || first + n > m->n) return fail(OCFD_ERR_ARG, "bad range");
    HIPCK(hipStreamSynchronize(m->st));
    if (X) HIPCK(hipMemcpy(X, m->X + 24 * first, sizeof(float) * 24 * (size_t)n, hipMemcpyDeviceToHost));
    if (y) HIPCK(hipMemcpy(y, m->y + first, sizeof(float) * (size_t)n, hipMemcpyDeviceToHost));
    return 0;
}

int ocfd_mlp_collect(ocfd_mlp* m, ocfd_ctx* x, int stride) {
    if (!m || !x || stride < 1) return fail(OCFD_ERR_ARG, "bad argument");
    if (!x->inited) return fail(OCFD_ERR_STATE, "context not initialised");
    if (m->device != x->device) return fail(OCFD_ERR_ARG, "trainer and context are on different devices");
    const long long n = mlp_collect_count(x->g, stride);
    if (m->n + n > m->cap) return fail(OCFD_ERR_ARG, "trainer capacity exceeded");
    float* X = m->X + 24 * m->n;
    float* y = m->y + m->n;
    if (x->mixed) {
        const MlpSensorArgsT<float> a = mlp_args<float>(x);
        TRY(timed(x, "mlp_collect", [&] { launch_mlp_collect(a, stride, X, y, x->st); }));
    } else {
        const MlpSensorArgsT<double> a = mlp_args<double>(x);
        TRY(timed(x, "mlp_collect", [&] { launch_mlp_collect(a, stride, X, y, x->st); }));
    }
    HIPCK(hipStreamSynchronize(x->st));
    m->n += n;
    return 0;
}

int ocfd_mlp_grad(ocfd_mlp* m, long long first, int n, float wpos, float* grads, float* loss) {
    if (!m || n <= 0 || first < 0 || first + n > m->n) return fail(OCFD_ERR_ARG, "bad range");
    TRY(mlp_ensure_batch(m, n));
    launch_mlp_step(m->P, m->X + 24 * first, m->y + first, nullptr, n, wpos, m->part, m->grad, m->m1, m->m2, 0, 0.f,
                    m->grad + MLP_NPARAM, m->st);
    HIPCK(hipGetLastError());
    HIPCK(hipStreamSynchronize(m->st));
    if (grads) HIPCK(hipMemcpy(grads, m->grad, sizeof(float) * MLP_NPARAM, hipMemcpyDeviceToHost));
    if (loss) HIPCK(hipMemcpy(loss, m->grad + MLP_NPARAM, sizeof(float), hipMemcpyDeviceToHost));
    return 0;
}

int ocfd_mlp_train(ocfd_mlp* m, int epochs, int batch, float lr, float wpos, unsigned long long seed,
                   float* epoch_loss) {
    if (!m || epochs <= 0 || batch <= 0) return fail(OCFD_ERR_ARG, "bad argument");
    if (m->n < batch) return fail(OCFD_ERR_STATE, "fewer samples than one batch");
    TRY(mlp_ensure_batch(m, batch));
    const long long nbat = m->n / batch;  // the remainder of an epoch's order is left out
    if (nbat > m->loss_cap) {
        TRY(mlp_alloc(m, (void**)&m->loss, sizeof(float) * (size_t)nbat));
        m->loss_cap = nbat;
    }
    std::vector<int> order((size_t)m->n);
    std::vector<float> lh((size_t)nbat);
    uint64_t s = seed;
    for (int e = 0; e < epochs; e++) {
        for (long long i = 0; i < m->n; i++) order[(size_t)i] = (int)i;
        for (long long i = m->n - 1; i > 0; i--) std::swap(order[(size_t)i], order[(size_t)(splitmix(s) % (uint64_t)(i + 1))]);
        HIPCK(hipMemcpyAsync(m->idx, order.data(), sizeof(int) * (size_t)m->n, hipMemcpyHostToDevice, m->st));
        for (long long b = 0; b < nbat; b++) {
            m->adam_t++;
            launch_mlp_step(m->P, m->X, m->y, m->idx + b * batch, batch, wpos, m->part, nullptr, m->m1, m->m2,
                            m->adam_t, lr, m->loss + b, m->st);
        }
        HIPCK(hipGetLastError());
        HIPCK(hipStreamSynchronize(m->st));  // the order buffer is rewritten next epoch
        if (epoch_loss) {
            HIPCK(hipMemcpy(lh.data(), m->loss, sizeof(float) * (size_t)nbat, hipMemcpyDeviceToHost));
            double t = 0.0;
            for (long long b = 0; b < nbat; b++) t += lh[(size_t)b];
            epoch_loss[e] = (float)(t / (double)nbat);
        }
    }
    return 0;
}

int ocfd_mlp_predict(ocfd_mlp* m, long long first, int n, float* prob) {
    // FP32 forward on stored samples (the training arithmetic), for checks
    if (!m || !prob || n <= 0 || first < 0 || first + n > m->n) return fail(OCFD_ERR_ARG, "bad range");
    if (n > m->prob_cap) {
        TRY(mlp_alloc(m, (void**)&m->prob, sizeof(float) * (size_t)n));
        m->prob_cap = n;
    }
    launch_mlp_predict(m->P, m->X + 24 * first, n, m->prob, m->st);
    HIPCK(hipGetLastError());
    HIPCK(hipStreamSynchronize(m->st));
    HIPCK(hipMemcpy(prob, m->prob, sizeof(float) * (size_t)n, hipMemcpyDeviceToHost));
    return 0;
}

int ocfd_set_sensor_from(ocfd_ctx* x, ocfd_mlp* m, float lo, float hi) {
    if (!x || !m) return fail(OCFD_ERR_ARG, "null argument");
    std::vector<float> p(MLP_NPARAM);
    TRY(ocfd_mlp_get_params(m, p.data()));
    return ocfd_set_sensor(x, p.data(), lo, hi);
}

int ocfd_profile_enable(ocfd_ctx* x, int on) {
    if (!x) return fail(OCFD_ERR_ARG, "null context");
    TRY(flush_prof(x));
    x->prof = on != 0;
    return 0;
}
int ocfd_profile_reset(ocfd_ctx* x) {
    if (!x) return fail(OCFD_ERR_ARG, "null context");
    TRY(flush_prof(x));
    x->acc.clear();
    return 0;
}
int ocfd_profile_count(ocfd_ctx* x) {
    if (!x) return 0;
    flush_prof(x);
    return (int)x->acc.size();
}
int ocfd_profile_entry(ocfd_ctx* x, int i, char* name, int* launches, double* total_ms) {
    if (!x || i < 0 || i >= (int)x->acc.size()) return fail(OCFD_ERR_ARG, "bad profile index");
    if (name) {
        std::strncpy(name, x->acc[i].first.c_str(), 63);
        name[63] = 0;
    }
    if (launches) *launches = x->acc[i].second.first;
    if (total_ms) *total_ms = x->acc[i].second.second;
    return 0;
}

}  // extern "C"

// ===========================================================================
// Reference-named entry points on one process-wide context.  They keep the
// signatures of the reference's extern "C" functions so that its control
// flow (opencfd.c: read_parameters, opencfd_mem_init_all, init,
// NS_solver_real) drives this library unchanged.  Errors print the message
// and exit(1), as CUDA_CALL/MPI_Abort do in the reference.
// ===========================================================================
namespace {
ocfd_ctx* g_ctx = nullptr;
ocfd_config g_cfg;
bool g_cfg_ok = false;

void die(const char* where, int rc) {
    std::fprintf(stderr, "%s failed (status %d): %s\n", where, rc, g_err.c_str());
    std::exit(1);
}
#define SHIM(expr)                     \
    do {                               \
        int rc_ = (expr);              \
        if (rc_) die(__func__, rc_);   \
    } while (0)

bool file_exists(const char* p) {
    FILE* fh = std::fopen(p, "rb");
    if (!fh) return false;
    std::fclose(fh);
    return true;
}
}  // namespace

extern "C" {

ocfd_ctx* ocfd_global_ctx(void) { return g_ctx; }

void read_parameters(void) {
    int rc = ocfd_read_config("opencfd-scu.in", &g_cfg);
    if (rc == OCFD_ERR_IO) {
        std::printf("opencfd-scu.in is not find!\n");
        std::exit(-1);
    }
    if (rc) {
        std::printf("SCHEMES CHOOSE IS WRONG\n");
        std::exit(0);
    }
    g_cfg_ok = true;
    std::printf("Mesh(Nx,Ny,Nz): (%d,%d,%d)\n", g_cfg.nx, g_cfg.ny, g_cfg.nz);
    std::printf("Re=%f , Ma=%f , Gamma=%f , dt=%f\n", g_cfg.re, g_cfg.ama, g_cfg.gamma, g_cfg.dt);
}

void opencfd_mem_init_all(void) {
    if (!g_cfg_ok) read_parameters();
    int dev = 0;
    if (const char* s = std::getenv("LOCAL_RANK")) dev = std::atoi(s);
    SHIM(ocfd_create(&g_cfg, dev, &g_ctx));
}

void init(void) {
    if (!g_ctx) opencfd_mem_init_all();
    const Geo& g = g_ctx->g;
    const size_t n = (size_t)g.nx * g.ny * g.nz;
    if (g_cfg.init_stat == 0) die("init (INIT_STAT=0 uses the reference's built-in cylinder mesh; not supported)", OCFD_ERR_UNSUPPORTED);
    if (file_exists("OCFD3d-Jacobi.dat")) {
        std::vector<double> a((size_t)13 * n);
        SHIM(ocfd_read_records("OCFD3d-Jacobi.dat", g.nx, g.ny, g.nz, 13, a.data()));
        SHIM(ocfd_load_jacobi(g_ctx, a.data()));
    } else {
        std::vector<double> a((size_t)3 * n);
        SHIM(ocfd_read_records("OCFD3d-Mesh.dat", g.nx, g.ny, g.nz, 3, a.data()));
        SHIM(ocfd_load_mesh(g_ctx, a.data(), a.data() + n, a.data() + 2 * n));
    }
    // src/OCFD_IO.c:37-91: Opencfd.msg holds the restart step
    char name[64] = "opencfd.dat";
    if (FILE* fh = std::fopen("Opencfd.msg", "rb")) {
        int32_t s = -1;
        if (std::fread(&s, 4, 1, fh) == 1 && s >= 0) std::snprintf(name, sizeof name, "OCFD%08d.dat", s);
        std::fclose(fh);
    } else {
        std::printf("Opencfd.msg is not exist, read initial file : opencfd.dat ......\n");
    }
    std::printf("read initial data file: %s \n\n", name);
    std::vector<double> p((size_t)5 * n);
    int istep = 0;
    double tt = 0;
    SHIM(ocfd_read_flow_file(name, g.nx, g.ny, g.nz, p.data(), p.data() + n, p.data() + 2 * n, p.data() + 3 * n,
                             p.data() + 4 * n, &istep, &tt));
    std::printf("Istep=%d , tt=%lf\n", istep, tt);
    SHIM(ocfd_load_flow(g_ctx, p.data(), p.data() + n, p.data() + 2 * n, p.data() + 3 * n, p.data() + 4 * n, istep,
                        tt));
    if (g_cfg.ibc == 108 && g_cfg.bc_npara[2] == 1) {
        // flow1d-inlet.dat: one header line, then ny rows of y d u v T
        FILE* fh = std::fopen("flow1d-inlet.dat", "r");
        if (!fh) die("init (flow1d-inlet.dat)", OCFD_ERR_IO);
        char line[512];
        if (!std::fgets(line, sizeof line, fh)) die("init (flow1d-inlet.dat)", OCFD_ERR_IO);
        std::vector<double> prof((size_t)4 * g.ny);
        for (int j = 0; j < g.ny; j++) {
            double y, a, b, c2, d;
            if (std::fscanf(fh, "%lf%lf%lf%lf%lf", &y, &a, &b, &c2, &d) != 5) die("init (flow1d-inlet.dat)", OCFD_ERR_IO);
            prof[j] = a; prof[g.ny + j] = b; prof[2 * g.ny + j] = c2; prof[3 * g.ny + j] = d;
        }
        std::fclose(fh);
        SHIM(ocfd_set_inlet_profile(g_ctx, prof.data()));
    }
    if (g_cfg.ibc == 124) {
        // bc_user_Liftbody3d_init (src/OCFD_boundary_init.c:118-201): five
        // records of NZ*NY (inlet) / NY*NX (upper) values
        std::vector<double> in, up;
        if (g_cfg.bc_npara[1] == 1) {
            std::printf("read inlet boundary data: flow-inlet-section.dat\n");
            in.resize((size_t)5 * g.ny * g.nz);
            SHIM(ocfd_read_records("flow-inlet-section.dat", g.ny, g.nz, 1, 5, in.data()));
        }
        if (g_cfg.bc_npara[2] == 1) {
            std::printf("read upper boundary data: flow-outboundary.dat\n");
            up.resize((size_t)5 * g.nx * g.ny);
            SHIM(ocfd_read_records("flow-outboundary.dat", g.nx, g.ny, 1, 5, up.data()));
        }
        SHIM(ocfd_set_bc_tables(g_ctx, in.empty() ? nullptr : in.data(), up.empty() ? nullptr : up.data()));
    }
    SHIM(ocfd_init(g_ctx));
    std::printf("init ok\n\n");
}

void NS_solver_real(void) {
    if (!g_ctx) die("NS_solver_real (call init first)", OCFD_ERR_STATE);
    const ocfd_config& C = g_cfg;
    const Geo& g = g_ctx->g;
    const size_t n = (size_t)g.nx * g.ny * g.nz;
    double total = 0.0, window = 0.0;
    do {
        SHIM(ocfd_step(g_ctx, 1));
        total += g_ctx->last_step_ms;
        window += g_ctx->last_step_ms;
        // src/OCFD_NS_Solver.cu:99-101 (a zero Kstep is skipped: the reference
        // would divide by it)
        for (int i = 0; i < C.nana; i++)
            if (C.ana_event[i][1] > 0 && g_ctx->istep % C.ana_event[i][1] == 0) OCFD_ana(C.ana_event[i][0], i);
        if (C.kstep_show > 0 && g_ctx->istep % C.kstep_show == 0) {
            // src/OCFD_NS_Solver.cu:124-152: mean total energy (NaN => the
            // NaN / negative-T check, which aborts) and mean T
            double E0 = 0.0, T0 = 0.0;
            long long nnan = 0, nneg = 0;
            SHIM(ocfd_diagnostics(g_ctx, &E0, &T0, &nnan, &nneg));
            if (std::isnan(E0)) {
                if (nneg > 10) {
                    std::printf("Negative T points %lld > %d\n", nneg, 10);
                    std::exit(1);
                }
                if (nnan) {
                    std::printf("NAN occured , program Abort\n");
                    std::exit(1);
                }
            }
            std::printf("%lf of %lf ( %d ) , using %lf\n", g_ctx->tt, C.end_time, g_ctx->istep, total * 1e-3);
            std::printf("%d steps GPU time %lf\n", C.kstep_show, window * 1e-3);
            std::printf("Averaged Total Energy is %lf\n", E0);
            std::printf("Averaged Total T is %lf\n\n", T0);
            window = 0.0;
        }
        if (C.kstep_save > 0 && g_ctx->istep % C.kstep_save == 0) {
            std::vector<double> p((size_t)5 * n);
            int is = 0;
            double t = 0;
            SHIM(ocfd_get_flow(g_ctx, p.data(), p.data() + n, p.data() + 2 * n, p.data() + 3 * n, p.data() + 4 * n, &is,
                               &t));
            char name[64];
            std::snprintf(name, sizeof name, "OCFD%08d.dat", is);
            std::printf("write data file: %s\n", name);
            SHIM(ocfd_write_flow_file(name, g.nx, g.ny, g.nz, p.data(), p.data() + n, p.data() + 2 * n,
                                      p.data() + 3 * n, p.data() + 4 * n, is, t));
        }
        if (C.end_time <= 0.0) break;
    } while (g_ctx->tt < C.end_time);
    std::printf("OK! opencfd is finished\nTotal GPU time %lf\n", total * 1e-3);
}

void OCFD_ana(int style, int ID) {
    if (!g_ctx) die("OCFD_ana (call init first)", OCFD_ERR_STATE);
    const int rc = ocfd_analysis(g_ctx, style, ID);
    if (rc == OCFD_ERR_NUMERIC) std::exit(1);  // MPI_Abort, src/OCFD_ana.cu:212-221
    if (rc) die(__func__, rc);
    if (style == 103) std::exit(0);  // get_Q ends the run, src/OCFD_ana.cu:456
}

void du_comput(int KRK) { SHIM(rhs_any(g_ctx, KRK)); }

void OCFD_time_advance(int KRK) {
    ocfd_ctx* x = g_ctx;
    SHIM(finish_rhs(x));
    const bool flap = KRK == 3 && x->flap && filter_due(x, x->istep + 1);
    if (x->mixed) {
        const StageArgsT<float> sa = stage_args<float>(x, KRK, flap);
        SHIM(timed(x, "stage", [&] { launch_stage(sa, x->st); }));
    } else {
        const StageArgsT<double> sa = stage_args<double>(x, KRK, flap);
        SHIM(timed(x, "stage", [&] { launch_stage(sa, x->st); }));
    }
}

void get_duvwT(void) {
    ocfd_ctx* x = g_ctx;
    // get_duvwT also computes the pressure
    if (x->mixed) {
        StageArgsT<float> sa = stage_args<float>(x, 1, false);
        sa.P = x->sP;
        SHIM(timed(x, "c2p", [&] { launch_c2p_all(sa, x->st); }));
    } else {
        StageArgsT<double> sa = stage_args<double>(x, 1, false);
        sa.P = x->P;
        SHIM(timed(x, "c2p", [&] { launch_c2p_all(sa, x->st); }));
    }
}

void get_Amu(void) {
    ocfd_ctx* x = g_ctx;
    if (x->mixed) {
        const BCArgsT<float> a = bc_args<float>(x);
        SHIM(timed(x, "amu", [&] { launch_amu_all(a, x->st); }));
    } else {
        const BCArgsT<double> a = bc_args<double>(x);
        SHIM(timed(x, "amu", [&] { launch_amu_all(a, x->st); }));
    }
}

void OCFD_bc(void) { SHIM(apply_bc_any(g_ctx)); }

void filtering(double* pf, double* pf0, double* pp) {
    (void)pf; (void)pf0; (void)pp;
    SHIM(do_filter_any(g_ctx));
}

void opencfd_mem_finalize_all(void) {
    ocfd_destroy(g_ctx);
    g_ctx = nullptr;
}

}  // extern "C"
