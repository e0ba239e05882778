// Operator face of libmcb (include/mcb_ops.h): one HIP kernel per reference
// kernel of src/kernels.cuh, on the reference's SoA layout. Thread per cell,
// 64-wide rows along x (one wave64 per row segment) instead of the reference's
// 8x8x8 blocks, so every population plane is read and written in 256-byte
// runs; the boundary kernels run over the faces. The per-cell arithmetic lives in lattice.hpp and is shared with the
// fused step kernels.
#include "bubble.hpp"
#include "common.hpp"

namespace mcb {
namespace {

constexpr int OBX = 64, OBY = 4;

struct OpArgs {
    Geo geo;
    Phys phys;
    int mode;        // mcb_bc_mode
    int tau_g_one;
};

__device__ __forceinline__ bool is_interior(int i, int j, int k, const Geo& g) {
    return !(i == 0 || i == g.nx - 1 || j == 0 || j == g.ny - 1 || k == 0 || k == g.nz - 1);
}

// Cell coordinates of this thread; false when outside the lattice or, in
// REFERENCE mode with interior_only, on a face (lbm.cu:14 and its copies).
__device__ __forceinline__ bool cell_of(const OpArgs& a, bool interior_only, int& i, int& j, int& k) {
    i = blockIdx.x * OBX + threadIdx.x;
    j = blockIdx.y * OBY + threadIdx.y;
    k = blockIdx.z;
    if (i >= a.geo.nx || j >= a.geo.ny || k >= a.geo.nz) return false;
    if (interior_only && a.mode == MCB_BC_REFERENCE && !is_interior(i, j, k, a.geo)) return false;
    return true;
}

__device__ __forceinline__ long long lin(int i, int j, int k, const Geo& g) {
    return (long long)k * g.nxy + (long long)j * g.nx + i;
}

// Element access at an offset from a wave-uniform pointer. The kernels of the
// loop read and write up to 51 values per cell, and 64-bit addresses per lane
// cost as many instructions as their arithmetic (gradCalc on 64x64x256: 8.2 us,
// bound by them). Below 2^30 cells (Off = unsigned) an access is a scalar base
// and a 32-bit byte offset; larger lattices keep 64-bit offsets.
template <class Off> __device__ __forceinline__ float get(const float* base, Off o) {
    if constexpr (sizeof(Off) == 4) return ld32(base, o);
    else return base[o];
}
template <class Off> __device__ __forceinline__ void put(float* base, Off o, float v) {
    if constexpr (sizeof(Off) == 4) st32(base, o, v);
    else base[o] = v;
}

// A cell's offset and those of its neighbours x + SIGN c_l, periodic.
template <class Off> struct Here {
    Off xs[3], ys[3], zs[3];
    __device__ __forceinline__ Here(int i, int j, int k, const Geo& g)
        : xs{(Off)shift<-1>(i, g.nx), (Off)i, (Off)shift<1>(i, g.nx)},
          ys{(Off)shift<-1>(j, g.ny) * (Off)g.nx, (Off)j * (Off)g.nx, (Off)shift<1>(j, g.ny) * (Off)g.nx},
          zs{(Off)shift<-1>(k, g.nz) * (Off)g.nxy, (Off)k * (Off)g.nxy, (Off)shift<1>(k, g.nz) * (Off)g.nxy} {}
    __device__ __forceinline__ Off me() const { return zs[1] + ys[1] + xs[1]; }
    template <int L, int SIGN = 1> __device__ __forceinline__ Off nb() const {
        return zs[1 + SIGN * CZ[L]] + ys[1 + SIGN * CY[L]] + xs[1 + SIGN * CX[L]];
    }
};

// ------------------------------------------------------------------ init.cu

__global__ __launch_bounds__(256) void k_initTensor(float* pxx, float* pyy, float* pzz, float* pxy, float* pxz,
                                                    float* pyz, float* rho, OpArgs a) {
    int i, j, k;
    if (!cell_of(a, false, i, j, k)) return;
    const long long x = lin(i, j, k, a.geo);
    const float val = 1.0f;
    pxx[x] = val; pyy[x] = val; pzz[x] = val;
    pxy[x] = val; pxz[x] = val; pyz[x] = val;
    rho[x] = val;
}

struct BubbleArgs {
    int n;
    float b[4 * MCB_OPS_MAX_BUBBLES];
    float width;
};

// bubble_phi_cell: the same bits as the host initialisation.
__global__ __launch_bounds__(256) void k_initPhase(float* phi, OpArgs a, BubbleArgs bb) {
    int i, j, k;
    if (!cell_of(a, true, i, j, k)) return;
    static_assert(sizeof(mcb_bubble) == 4 * sizeof(float), "bubble record = cx, cy, cz, r");
    phi[lin(i, j, k, a.geo)] = bubble_phi_cell(i, j, k, a.geo.nx, a.geo.ny, a.geo.nz, a.mode == MCB_BC_PERIODIC,
                                               reinterpret_cast<const mcb_bubble*>(bb.b), bb.n, bb.width);
}

__global__ __launch_bounds__(256) void k_initDist(const float* rho, const float* phi, float* f, float* g, OpArgs a) {
    int i, j, k;
    if (!cell_of(a, false, i, j, k)) return;
    const long long x = lin(i, j, k, a.geo);
    const float r = rho[x], ph = phi[x];
    for_links([&](auto lc) {
        constexpr int l = decltype(lc)::value;
        f[x + l * a.geo.plane] = a.phys.w[WC[l]] * r;
    });
    for_links([&](auto lc) {
        constexpr int l = decltype(lc)::value;
        g[x + l * a.geo.plane] = a.phys.w[WC[l]] * ph;
    });
}

// ------------------------------------------------------------------- lbm.cu

template <class Off> __global__ __launch_bounds__(256) void k_phiCalc(float* phi, const float* g, OpArgs a) {
    int i, j, k;
    if (!cell_of(a, true, i, j, k)) return;
    const Off x = Here<Off>(i, j, k, a.geo).me();
    float sum = 0.0f;
    for_links([&](auto lc) { sum += get(g + decltype(lc)::value * a.geo.plane, x); });
    put(phi, x, sum);
}

template <class Off>
__global__ __launch_bounds__(256) void k_gradCalc(const float* phi, float* normx, float* normy, float* normz,
                                                  float* indicator, OpArgs a) {
    int i, j, k;
    if (!cell_of(a, true, i, j, k)) return;
    const Derived d(a.phys);
    const Here<Off> h(i, j, k, a.geo);
    float nx, ny, nz, ind;
    grad_normal([&](auto lc) { return get(phi, h.template nb<decltype(lc)::value>()); }, d, nx, ny, nz, ind);
    const Off x = h.me();
    put(normx, x, nx);
    put(normy, x, ny);
    put(normz, x, nz);
    put(indicator, x, ind);
}

template <class Off>
__global__ __launch_bounds__(256) void k_curvatureCalc(float* curvature, const float* indicator, const float* normx,
                                                       const float* normy, const float* normz, float* ffx, float* ffy,
                                                       float* ffz, OpArgs a) {
    int i, j, k;
    if (!cell_of(a, true, i, j, k)) return;
    const Derived d(a.phys);
    const Here<Off> h(i, j, k, a.geo);
    const Off x = h.me();
    float curv, fx, fy, fz;
    curvature_force(
        [&](auto lc, float& ax, float& ay, float& az) {
            constexpr int l = decltype(lc)::value;
            const Off o = h.template nb<l>();
            if constexpr (CX[l] != 0) ax = get(normx, o);
            if constexpr (CY[l] != 0) ay = get(normy, o);
            if constexpr (CZ[l] != 0) az = get(normz, o);
        },
        a.phys, d, get(normx, x), get(normy, x), get(normz, x), get(indicator, x), curv, fx, fy, fz);
    put(curvature, x, curv);
    put(ffx, x, fx);
    put(ffy, x, fy);
    put(ffz, x, fz);
}

template <class Off>
__global__ __launch_bounds__(256) void k_momentiCalc(float* ux, float* uy, float* uz, float* rho, const float* ffx,
                                                     const float* ffy, const float* ffz, const float* f, float* pxx,
                                                     float* pyy, float* pzz, float* pxy, float* pxz, float* pyz,
                                                     OpArgs a) {
    int i, j, k;
    if (!cell_of(a, true, i, j, k)) return;
    const Off x = Here<Off>(i, j, k, a.geo).me();
    float fv[Q];
    for_links([&](auto lc) {
        constexpr int l = decltype(lc)::value;
        fv[l] = get(f + l * a.geo.plane, x);
    });
    const Moments m = moments<true>(fv, a.phys, get(ffx, x), get(ffy, x), get(ffz, x));
    put(pxx, x, m.pxx);
    put(pyy, x, m.pyy);
    put(pzz, x, m.pzz);
    put(pxy, x, m.pxy);
    put(pxz, x, m.pxz);
    put(pyz, x, m.pyz);
    put(ux, x, m.ux);
    put(uy, x, m.uy);
    put(uz, x, m.uz);
    put(rho, x, m.rho);
}

template <class Off>
__global__ __launch_bounds__(256) void k_collisionFluid(float* f, const float* ux, const float* uy, const float* uz,
                                                        const float* ffx, const float* ffy, const float* ffz,
                                                        const float* rho, const float* pxx, const float* pyy,
                                                        const float* pzz, const float* pxy, const float* pxz,
                                                        const float* pyz, OpArgs a) {
    int i, j, k;
    if (!cell_of(a, true, i, j, k)) return;
    const Derived d(a.phys);
    const Here<Off> h(i, j, k, a.geo);
    const Off x = h.me();
    Moments m;
    m.rho = get(rho, x);
    m.ux = get(ux, x);
    m.uy = get(uy, x);
    m.uz = get(uz, x);
    m.pxx = get(pxx, x);
    m.pyy = get(pyy, x);
    m.pzz = get(pzz, x);
    m.pxy = get(pxy, x);
    m.pxz = get(pxz, x);
    m.pyz = get(pyz, x);
    const FluidCell c = fluid_cell<true>(m, get(ffx, x), get(ffy, x), get(ffz, x));
    for_links([&](auto lc) {
        constexpr int l = decltype(lc)::value;
        put(f + l * a.geo.plane, h.template nb<l>(), fluid_post<l, true>(c, a.phys, d));
    });
}

template <class Off>
__global__ __launch_bounds__(256) void k_collisionPhase(float* g, const float* ux, const float* uy, const float* uz,
                                                        const float* phi, const float* normx, const float* normy,
                                                        const float* normz, OpArgs a) {
    int i, j, k;
    if (!cell_of(a, true, i, j, k)) return;
    const Derived d(a.phys);
    const Off x = Here<Off>(i, j, k, a.geo).me();
    const PhaseCell c = phase_cell(a.phys, get(phi, x), get(ux, x), get(uy, x), get(uz, x), get(normx, x),
                                   get(normy, x), get(normz, x));
    if (a.tau_g_one) {
        for_links([&](auto lc) {
            constexpr int l = decltype(lc)::value;
            put(g + l * a.geo.plane, x, phase_post<l>(c, a.phys));
        });
    } else {
        float pre[Q];
        for_links([&](auto lc) {
            constexpr int l = decltype(lc)::value;
            pre[l] = get(g + l * a.geo.plane, x);
        });
        for_links([&](auto lc) {
            constexpr int l = decltype(lc)::value;
            put(g + l * a.geo.plane, x, phase_post_bgk<l>(c, a.phys, d, pre[l]));
        });
    }
}

template <class Off> __global__ __launch_bounds__(256) void k_streamingCalc(const float* g, float* g_out, OpArgs a) {
    int i, j, k;
    if (!cell_of(a, false, i, j, k)) return;
    const Here<Off> h(i, j, k, a.geo);
    float v[Q];
    for_links([&](auto lc) {
        constexpr int l = decltype(lc)::value;
        v[l] = get(g + l * a.geo.plane, h.template nb<l, -1>());
    });
    for_links([&](auto lc) {
        constexpr int l = decltype(lc)::value;
        put(g_out + l * a.geo.plane, h.me(), v[l]);
    });
}

// Cell e of the lattice's faces: the two z faces, then the two y faces and the
// two x faces without the cells of those before, x (or y) fastest. Launched
// over the faces only: with a thread per cell of the lattice nearly every wave
// held a face lane or two (x = 0, x = nx - 1) and walked through all links for
// them (fgBoundary on 64x64x256: 27.6 us for 7% of the cells).
__host__ __device__ __forceinline__ long long face_cells(const Geo& g) {
    return 2LL * g.nxy + 2LL * g.nx * (g.nz - 2) + 2LL * (g.ny - 2) * (g.nz - 2);
}
__device__ __forceinline__ bool face_of(long long e, const Geo& g, int& i, int& j, int& k) {
    if (e < 2LL * g.nxy) {
        const unsigned r = (unsigned)(e % g.nxy);
        k = e < g.nxy ? 0 : g.nz - 1;
        j = (int)(r / (unsigned)g.nx);
        i = (int)(r % (unsigned)g.nx);
        return true;
    }
    e -= 2LL * g.nxy;
    const long long ny_face = (long long)g.nx * (g.nz - 2), nx_face = (long long)(g.ny - 2) * (g.nz - 2);
    if (e < 2 * ny_face) {
        const unsigned r = (unsigned)(e % ny_face);
        j = e < ny_face ? 0 : g.ny - 1;
        k = 1 + (int)(r / (unsigned)g.nx);
        i = (int)(r % (unsigned)g.nx);
        return true;
    }
    e -= 2 * ny_face;
    if (e < 2 * nx_face) {
        const unsigned r = (unsigned)(e % nx_face);
        i = e < nx_face ? 0 : g.nx - 1;
        k = 1 + (int)(r / (unsigned)(g.ny - 2));
        j = 1 + (int)(r % (unsigned)(g.ny - 2));
        return true;
    }
    return false;
}

__global__ __launch_bounds__(256) void k_fgBoundary(float* f, const float* rho, float* g, const float* phi, OpArgs a) {
    int i, j, k;
    if (!face_of((long long)blockIdx.x * 256 + threadIdx.x, a.geo, i, j, k)) return;
    const long long x = lin(i, j, k, a.geo);
    const float r = rho[x], ph = phi[x];
    auto inside = [&](int ni, int nj, int nk) {
        return ni >= 0 && ni < a.geo.nx && nj >= 0 && nj < a.geo.ny && nk >= 0 && nk < a.geo.nz;
    };
    for_links([&](auto lc) {
        constexpr int l = decltype(lc)::value;
        const int ni = i + CX[l], nj = j + CY[l], nk = k + CZ[l];
        if (!inside(ni, nj, nk)) return;
        const long long o = lin(ni, nj, nk, a.geo) + l * a.geo.plane;
        f[o] = r * a.phys.w[WC[l]];
        g[o] = ph * a.phys.w[WC[l]];
    });
}

// Zero-gradient phi on the six faces. Serial order z, y, x (each reading the
// previous result) leaves every face node equal to the interior node at the
// clamped coordinates, which a single pass can write without a race: face
// nodes only read interior nodes.
__global__ __launch_bounds__(256) void k_boundaryConditions(float* phi, OpArgs a) {
    int i, j, k;
    if (!face_of((long long)blockIdx.x * 256 + threadIdx.x, a.geo, i, j, k)) return;
    const int ci = min(max(i, 1), a.geo.nx - 2);
    const int cj = min(max(j, 1), a.geo.ny - 2);
    const int ck = min(max(k, 1), a.geo.nz - 2);
    phi[lin(i, j, k, a.geo)] = phi[lin(ci, cj, ck, a.geo)];
}

__global__ __launch_bounds__(256) void k_movingWallBC(float* f, const float* rho, OpArgs a) {
    // The reference maps (i, k) onto a 3-D launch and covers k < 8*ceil(NY/8);
    // one thread per (i, k) here, same stores.
    const int i = blockIdx.x * OBX + threadIdx.x;
    const int k = blockIdx.y * OBY + threadIdx.y;
    const int kmax = min(a.geo.nz, ((a.geo.ny + 7) / 8) * 8);
    if (i >= a.geo.nx || k >= kmax) return;
    const float U_wall = 0.03f;
    const long long xb = lin(i, 0, k, a.geo), xt = lin(i, a.geo.ny - 1, k, a.geo);
    const float rb = rho[xb], rt = rho[xt];
    for_links([&](auto lc) {
        constexpr int l = decltype(lc)::value;
        const float cu = ((float)CX[l] * (-U_wall)) / CSSQ;
        f[xb + l * a.geo.plane] = rb * a.phys.w[WC[l]] * (1.0f + cu);
    });
    for_links([&](auto lc) {
        constexpr int l = decltype(lc)::value;
        const float cu = ((float)CX[l] * U_wall) / CSSQ;
        f[xt + l * a.geo.plane] = rt * a.phys.w[WC[l]] * (1.0f + cu);
    });
}

// ------------------------------------------------------------ launch helpers

mcb_status check_common(int NX, int NY, int NZ, const mcb_op_consts* c) {
    if (!c) return MCB_ERR_INVALID_ARG;
    if (NX < 3 || NY < 3 || NZ < 3) return MCB_ERR_INVALID_ARG;
    if ((long long)NX * NY * NZ >= (1LL << 31)) return MCB_ERR_INVALID_ARG;
    if (NZ > 65535) return MCB_ERR_INVALID_ARG;
    if (c->bc_mode != MCB_BC_PERIODIC && c->bc_mode != MCB_BC_REFERENCE) return MCB_ERR_INVALID_ARG;
    return MCB_OK;
}

OpArgs make_args(int NX, int NY, int NZ, const mcb_op_consts* c) {
    OpArgs a;
    a.geo.nx = NX; a.geo.ny = NY; a.geo.nz = NZ;
    a.geo.nxy = NX * NY;
    a.geo.n = (long long)NX * NY * NZ;
    a.geo.plane = a.geo.n;   // the reference layout has no padding
    a.phys = phys_from_consts(*c);
    a.mode = c->bc_mode;
    a.tau_g_one = c->tau_g_is_one;
    return a;
}

dim3 grid_of(const Geo& g) { return dim3((g.nx + OBX - 1) / OBX, (g.ny + OBY - 1) / OBY, g.nz); }
const dim3 kBlock(OBX, OBY, 1);

dim3 face_grid(const Geo& g) { return dim3((unsigned)((face_cells(g) + 255) / 256)); }

// Launches kernel K<Off> over the cells with the offset type the lattice needs.
#define MCB_LAUNCH_CELLS(K, ...)                                                                            \
    do {                                                                                                    \
        if (a.geo.n < (1LL << 30)) hipLaunchKernelGGL(K<unsigned>, grid_of(a.geo), kBlock, 0, s, __VA_ARGS__); \
        else hipLaunchKernelGGL(K<long long>, grid_of(a.geo), kBlock, 0, s, __VA_ARGS__);                   \
    } while (0)

mcb_status launched() { return hip_status(hipGetLastError()); }

template <class... P> bool any_null(P... p) { return ((p == nullptr) || ...); }

}  // namespace
}  // namespace mcb

using namespace mcb;

#define MCB_OP_PROLOGUE(...)                                          \
    mcb_status st_ = check_common(NX, NY, NZ, c);                     \
    if (st_ != MCB_OK) return st_;                                    \
    if (any_null(__VA_ARGS__)) return MCB_ERR_INVALID_ARG;            \
    const OpArgs a = make_args(NX, NY, NZ, c);                        \
    hipStream_t s = static_cast<hipStream_t>(stream)

extern "C" {

mcb_status mcb_initTensor(float* pxx, float* pyy, float* pzz, float* pxy, float* pxz, float* pyz, float* rho,
                          int NX, int NY, int NZ, const mcb_op_consts* c, void* stream) {
    MCB_OP_PROLOGUE(pxx, pyy, pzz, pxy, pxz, pyz, rho);
    hipLaunchKernelGGL(k_initTensor, grid_of(a.geo), kBlock, 0, s, pxx, pyy, pzz, pxy, pxz, pyz, rho, a);
    return launched();
}

mcb_status mcb_initPhase(float* phi, int NX, int NY, int NZ, const mcb_op_consts* c, void* stream) {
    MCB_OP_PROLOGUE(phi);
    if (c->n_bubbles < 1 || c->n_bubbles > MCB_OPS_MAX_BUBBLES || !(c->width > 0.0f)) return MCB_ERR_INVALID_ARG;
    BubbleArgs bb;
    bb.n = c->n_bubbles;
    for (int q = 0; q < 4 * MCB_OPS_MAX_BUBBLES; ++q) bb.b[q] = c->bubbles[q];
    bb.width = c->width;
    hipLaunchKernelGGL(k_initPhase, grid_of(a.geo), kBlock, 0, s, phi, a, bb);
    return launched();
}

mcb_status mcb_initDist(const float* rho, const float* phi, float* f, float* g, int NX, int NY, int NZ,
                        const mcb_op_consts* c, void* stream) {
    MCB_OP_PROLOGUE(rho, phi, f, g);
    hipLaunchKernelGGL(k_initDist, grid_of(a.geo), kBlock, 0, s, rho, phi, f, g, a);
    return launched();
}

mcb_status mcb_phiCalc(float* phi, const float* g, int NX, int NY, int NZ, const mcb_op_consts* c, void* stream) {
    MCB_OP_PROLOGUE(phi, g);
    MCB_LAUNCH_CELLS(k_phiCalc, phi, g, a);
    return launched();
}

mcb_status mcb_gradCalc(const float* phi, float* normx, float* normy, float* normz, float* indicator, int NX, int NY,
                        int NZ, const mcb_op_consts* c, void* stream) {
    MCB_OP_PROLOGUE(phi, normx, normy, normz, indicator);
    MCB_LAUNCH_CELLS(k_gradCalc, phi, normx, normy, normz, indicator, a);
    return launched();
}

mcb_status mcb_curvatureCalc(float* curvature, const float* indicator, const float* normx, const float* normy,
                             const float* normz, float* ffx, float* ffy, float* ffz, int NX, int NY, int NZ,
                             const mcb_op_consts* c, void* stream) {
    MCB_OP_PROLOGUE(curvature, indicator, normx, normy, normz, ffx, ffy, ffz);
    MCB_LAUNCH_CELLS(k_curvatureCalc, curvature, indicator, normx, normy, normz, ffx,
                       ffy, ffz, a);
    return launched();
}

mcb_status mcb_momentiCalc(float* ux, float* uy, float* uz, float* rho, const float* ffx, const float* ffy,
                           const float* ffz, const float* f, float* pxx, float* pyy, float* pzz, float* pxy,
                           float* pxz, float* pyz, int NX, int NY, int NZ, const mcb_op_consts* c, void* stream) {
    MCB_OP_PROLOGUE(ux, uy, uz, rho, ffx, ffy, ffz, f, pxx, pyy, pzz, pxy, pxz, pyz);
    MCB_LAUNCH_CELLS(k_momentiCalc, ux, uy, uz, rho, ffx, ffy, ffz, f, pxx, pyy, pzz,
                       pxy, pxz, pyz, a);
    return launched();
}

mcb_status mcb_collisionFluid(float* f, const float* ux, const float* uy, const float* uz, const float* ffx,
                              const float* ffy, const float* ffz, const float* rho, const float* pxx, const float* pyy,
                              const float* pzz, const float* pxy, const float* pxz, const float* pyz, int NX, int NY,
                              int NZ, const mcb_op_consts* c, void* stream) {
    MCB_OP_PROLOGUE(f, ux, uy, uz, ffx, ffy, ffz, rho, pxx, pyy, pzz, pxy, pxz, pyz);
    MCB_LAUNCH_CELLS(k_collisionFluid, f, ux, uy, uz, ffx, ffy, ffz, rho, pxx, pyy,
                       pzz, pxy, pxz, pyz, a);
    return launched();
}

mcb_status mcb_collisionPhase(float* g, const float* ux, const float* uy, const float* uz, const float* phi,
                              const float* normx, const float* normy, const float* normz, int NX, int NY, int NZ,
                              const mcb_op_consts* c, void* stream) {
    MCB_OP_PROLOGUE(g, ux, uy, uz, phi, normx, normy, normz);
    MCB_LAUNCH_CELLS(k_collisionPhase, g, ux, uy, uz, phi, normx, normy, normz, a);
    return launched();
}

mcb_status mcb_streamingCalc(const float* g, float* g_out, int NX, int NY, int NZ, const mcb_op_consts* c,
                             void* stream) {
    MCB_OP_PROLOGUE(g, g_out);
    if (g == g_out) return MCB_ERR_INVALID_ARG;
    MCB_LAUNCH_CELLS(k_streamingCalc, g, g_out, a);
    return launched();
}

mcb_status mcb_fgBoundary(float* f, const float* rho, float* g, const float* phi, int NX, int NY, int NZ,
                          const mcb_op_consts* c, void* stream) {
    MCB_OP_PROLOGUE(f, rho, g, phi);
    hipLaunchKernelGGL(k_fgBoundary, face_grid(a.geo), dim3(256), 0, s, f, rho, g, phi, a);
    return launched();
}

mcb_status mcb_boundaryConditions(float* phi, int NX, int NY, int NZ, const mcb_op_consts* c, void* stream) {
    MCB_OP_PROLOGUE(phi);
    hipLaunchKernelGGL(k_boundaryConditions, face_grid(a.geo), dim3(256), 0, s, phi, a);
    return launched();
}

mcb_status mcb_movingWallBC(float* f, const float* rho, int NX, int NY, int NZ, const mcb_op_consts* c,
                            void* stream) {
    MCB_OP_PROLOGUE(f, rho);
    const int kmax = std::min(NZ, ((NY + 7) / 8) * 8);
    dim3 grid((NX + OBX - 1) / OBX, (kmax + OBY - 1) / OBY, 1);
    hipLaunchKernelGGL(k_movingWallBC, grid, kBlock, 0, s, f, rho, a);
    return launched();
}

}  // extern "C"
