// Definitions of the Launch<T> members; included by kernels_f64.hip and kernels_f32.hip.
#pragma once
#include "kernels.inl"
#include "gradient.inl"
#include "launch.h"

namespace mflbm {

namespace {
inline unsigned blocks(int64_t n, int b = 256) { return (unsigned)((n + b - 1) / b); }

// Threads of periodic_phi.
int64_t periodic_threads(const Dims& d, int kper, int jper) {
    return (kper ? (int64_t)d.nx * d.ny : 0) + (jper ? (int64_t)d.nx * d.nz : 0) + (kper && jper ? d.nx : 0);
}

// Workgroups of the open boundaries and the periodic copies.
template <typename T>
void boundary_groups(BoundaryArgs<T>& B, const Dims& d, int threads) {
    // inlet and outlet on separate threads when both are set and their planes are apart
    B.split = B.in_bc && B.out_bc && d.nz >= 6;
    B.nbc = B.in_bc || B.out_bc ? (int)blocks((int64_t)(B.split ? 2 : 1) * d.nx * d.ny, threads) : 0;
    B.npair = (int)blocks(B.npairs, threads * dev::PAIRS);
    B.blocks = (B.nbc + B.npair + 7) / 8 * 8;
}

template <typename T>
__global__ __launch_bounds__(256) void k_pack_solid_normals(const T* __restrict__ x, const T* __restrict__ y,
                                                            const T* __restrict__ z, const int32_t* __restrict__ wet,
                                                            int n, T* __restrict__ dst) {
    const int w = blockIdx.x * 256 + threadIdx.x;
    if (w >= n) return;
    const int c = wet[w];
    dst[w] = x[c];
    dst[(int64_t)n + w] = y[c];
    dst[2 * (int64_t)n + w] = z[c];
}

template <typename T>
__global__ __launch_bounds__(256) void k_to_real(const double* __restrict__ src, T* __restrict__ dst, int64_t n) {
    const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (t < n) dst[t] = (T)src[t];
}
}  // namespace

namespace {
template <typename T, int THREADS>
void launch_collide(const Sparse<T>& S, T* phi, const Dims& d, const StepConst<T>& P, bool odd, const PhiGhosts<T>* ghosts,
                    hipStream_t s) {
    unsigned grid = blocks(S.nf, THREADS);
    PhiGhosts<T> G{};
    if (ghosts) {
        G = *ghosts;
        G.rest = (int)((blocks(dev::ghost_phi_threads(G, d), THREADS) + 7) / 8 * 8);
        grid += G.rest;
    }
    if (P.mrt == 2) {
        if (odd) dev::k_collide<T, true, true, THREADS><<<grid, THREADS, 0, s>>>(S, phi, d, P, G);
        else dev::k_collide<T, false, true, THREADS><<<grid, THREADS, 0, s>>>(S, phi, d, P, G);
    } else {  // collision models 1, 3, 4
        if (odd) dev::k_collide<T, true, false, THREADS><<<grid, THREADS, 0, s>>>(S, phi, d, P, G);
        else dev::k_collide<T, false, false, THREADS><<<grid, THREADS, 0, s>>>(S, phi, d, P, G);
    }
}
}  // namespace

template <typename T>
void Launch<T>::collide(const Sparse<T>& S, T* phi, const Dims& d, const StepConst<T>& P, bool odd,
                        const PhiGhosts<T>* ghosts, hipStream_t s) {
    if (S.nf <= 0) return;
    // One wave to a workgroup where workgroups of 256 nodes would leave half of the 256 CUs without
    // one.  us, odd / even, 256 and 64 threads: 32^3 FP64 8.5 / 5.9 and 6.3 / 5.0, 40^3 FP32 6.8 / 4.6
    // and 6.4 / 4.5; 48^3 level; 64^3 FP32 14.1 / 7.1 and 14.7 / 7.4, 256^3 FP64 1127 / 752 and 1138 /
    // 770 (128 threads: 1128 / 758).
    if (S.nf < 128 * 256) launch_collide<T, 64>(S, phi, d, P, odd, ghosts, s);
    else launch_collide<T, 256>(S, phi, d, P, odd, ghosts, s);
}

template <typename T>
void Launch<T>::boundary(const Sparse<T>& S, const Fields<T>& F, const StepConst<T>& P, BoundaryArgs<T> B, bool after_odd,
                         hipStream_t s) {
    boundary_groups(B, F.d, 256);
    const unsigned grid = (unsigned)(B.nbc + B.npair) + blocks(periodic_threads(F.d, B.kper, B.jper));
    if (grid == 0) return;
    if (after_odd) dev::k_boundary<T, true><<<grid, 256, 0, s>>>(S, F, P, B);
    else dev::k_boundary<T, false><<<grid, 256, 0, s>>>(S, F, P, B);
}

template <typename T>
void Launch<T>::porous_plate(const Sparse<T>& S, const Dims& d, const StepConst<T>& P, const int32_t* pmap, int zp,
                             int blocked, bool after_odd, hipStream_t s) {
    const int n = d.nx * d.ny;
    if (after_odd) dev::k_porous_plate<T, true><<<blocks(n), 256, 0, s>>>(S, d, P, pmap, zp, blocked);
    else dev::k_porous_plate<T, false><<<blocks(n), 256, 0, s>>>(S, d, P, pmap, zp, blocked);
}

template <typename T>
void Launch<T>::conv_init(const Fields<T>& F, T rho_ref, T* conv, hipStream_t s) {
    dev::k_conv_init<T><<<blocks((int64_t)F.d.X1 * F.d.Y1), 256, 0, s>>>(F, rho_ref, conv);
}

template <typename T>
void Launch<T>::phi_extrap(const Fields<T>& F, const NodeLists& L, hipStream_t s, bool inner) {
    if (L.n_solid_bnd > 0)
        dev::k_phi_extrap<T><<<blocks(L.n_solid_bnd), 256, 0, s>>>(F, L.solid_bnd, L.n_solid_bnd, inner);
}

template <typename T>
void Launch<T>::normals(const Fields<T>& F, const StepConst<T>& P, const NodeLists& L, hipStream_t s) {
    if (L.n_fluid_ext > 0) dev::k_normals<T><<<blocks(L.n_fluid_ext), 256, 0, s>>>(F, P, L.fluid_ext, L.n_fluid_ext);
}

template <typename T>
void Launch<T>::normal_extrap(const Fields<T>& F, const NodeLists& L, hipStream_t s) {
    if (L.n_solid_bnd > 0) dev::k_normal_extrap<T><<<blocks(L.n_solid_bnd), 256, 0, s>>>(F, L.solid_bnd, L.n_solid_bnd);
}

template <typename T>
void Launch<T>::curvature(const Fields<T>& F, const StepConst<T>& P, const NodeLists& L, T* aux, hipStream_t s) {
    if (L.n_fluid > 0) dev::k_curvature<T><<<blocks(L.n_fluid), 256, 0, s>>>(F, P, L.fluid, L.n_fluid, aux);
}

namespace {
unsigned boxes(const Dims& d, bool force, const int (&t)[3], int (&tiles)[3]) {
    const int n[3] = {d.nx, d.ny, d.nz};
    // normals over [-1, n+2]^3, forces over [1, n]^3
    for (int a = 0; a < 3; ++a) tiles[a] = (n[a] + (force ? 0 : 4) + t[a] - 1) / t[a];
    return (unsigned)(tiles[0] * tiles[1] * tiles[2]);
}

// Calls f with the box shapes of a domain: the small ones where a CU would have less than one box
// of k_grad_force.  us, normals / force, large and small boxes: 32^3 FP64 6.6 / 6.8 and 5.6 / 6.2, 40^3
// FP64 7.0 / 7.2 and 6.2 / 7.4, FP32 6.3 / 5.7 and 5.6 / 5.6; beyond, 54^3 FP64 7.5 / 9.1 and 8.9 / 9.8,
// FP32 6.2 / 6.7 and 7.0 / 7.1 (the halos of small boxes are more than half of what they load).
template <typename T, class Fn>
void with_boxes(const Dims& d, Fn&& f) {
    int t[3];
    if (boxes(d, true, GradTiles<T>::F, t) < 256) f(SmallGradTiles{});
    else f(GradTiles<T>{});
}

// Sets the box counts of one of the two kernels; returns its grid.
template <typename T, class Shape>
unsigned box_grid(GradArgs<T>& A, bool force) {
    int t[3];
    const unsigned n = boxes(A.d, force, force ? Shape::F : Shape::N, t);
    A.tiles_x = t[0]; A.tiles_y = t[1]; A.tiles_z = t[2];
    return n;
}
}  // namespace

template <typename T>
int Launch<T>::tile_boxes(const Dims& d, bool force, int* columns) {
    int n = 0;
    with_boxes<T>(d, [&](auto shape) {
        using S = decltype(shape);
        int t[3];
        n = (int)boxes(d, force, force ? S::F : S::N, t);
        if (columns) *columns = (S::F[0] + 4) * (S::F[1] + 4);
    });
    return n;
}

template <typename T>
void Launch<T>::tile_counts(const GradArgs<T>& A, TileDesc* ndesc, TileDesc* fdesc, hipStream_t s) {
    with_boxes<T>(A.d, [&](auto shape) {
        using S = decltype(shape);
        GradArgs<T> B = A;
        const unsigned gn = box_grid<T, S>(B, false);
        dev::k_tile_lists<T, S::N[0], S::N[1], S::N[2], false, false><<<gn, 64, 0, s>>>(B, ndesc, TileFill{});
        const unsigned gf = box_grid<T, S>(B, true);
        dev::k_tile_lists<T, S::F[0], S::F[1], S::F[2], true, false><<<gf, 64, 0, s>>>(B, fdesc, TileFill{});
    });
}

template <typename T>
void Launch<T>::tile_fill(const GradArgs<T>& A, const TileFill& out, hipStream_t s) {
    with_boxes<T>(A.d, [&](auto shape) {
        using S = decltype(shape);
        GradArgs<T> B = A;
        const unsigned gn = box_grid<T, S>(B, false);
        dev::k_tile_lists<T, S::N[0], S::N[1], S::N[2], false, true>
            <<<gn, 64, 0, s>>>(B, const_cast<TileDesc*>(A.lists.ndesc), out);
        const unsigned gf = box_grid<T, S>(B, true);
        dev::k_tile_lists<T, S::F[0], S::F[1], S::F[2], true, true>
            <<<gf, 64, 0, s>>>(B, const_cast<TileDesc*>(A.lists.fdesc), out);
    });
}

template <typename T>
void Launch<T>::gradient_boundary(const GradArgs<T>& A, const Sparse<T>& S, const Fields<T>& F, const StepConst<T>& P,
                                  BoundaryArgs<T> B, bool after_odd, hipStream_t s) {
    with_boxes<T>(A.d, [&](auto shape) {
        using H = decltype(shape);
        constexpr int NX = H::N[0], NY = H::N[1], NZ = H::N[2];
        constexpr int FX = H::F[0], FY = H::F[1], FZ = H::F[2], threads = (FX + 4) * (FY + 4);
        GradArgs<T> G = A;
        const unsigned gn = box_grid<T, H>(G, false);
        dev::k_grad_normals<T, NX, NY, NZ><<<gn, (NX + 4) * (NY + 4), 0, s>>>(G, P);
        const unsigned gf = box_grid<T, H>(G, true);
        boundary_groups(B, F.d, threads);
        if (B.blocks == 0) dev::k_grad_force<T, FX, FY, FZ, 0><<<gf, threads, 0, s>>>(G, P, S, F, B);
        else if (after_odd) dev::k_grad_force<T, FX, FY, FZ, 1><<<gf + B.blocks, threads, 0, s>>>(G, P, S, F, B);
        else dev::k_grad_force<T, FX, FY, FZ, 2><<<gf + B.blocks, threads, 0, s>>>(G, P, S, F, B);
    });
}

template <typename T>
void Launch<T>::gradient(const GradArgs<T>& A, const StepConst<T>& P, hipStream_t s) {
    if (A.shape == GRAD_SHAPE_TILES) {
        gradient_boundary(A, Sparse<T>{}, Fields<T>{}, P, BoundaryArgs<T>{}, false, s);
        return;
    }
    const int chunks = (A.d.nz + A.kchunk - 1) / A.kchunk;
    const unsigned grid = (unsigned)(A.tiles_x * A.tiles_y * chunks);
    static_assert(GRAD_NSHAPES == 5, "one case per shape");
    switch (A.shape) {
#define MFLBM_GRAD_SHAPE(n)                                                                                  \
    case n:                                                                                                  \
        dev::k_gradient<T, GRAD_SHAPES[n].tx, GRAD_SHAPES[n].ty, GRAD_SHAPES[n].threads>                     \
            <<<grid, GRAD_SHAPES[n].threads, 0, s>>>(A, P);                                                  \
        break;
        MFLBM_GRAD_SHAPE(0)
        MFLBM_GRAD_SHAPE(1)
        MFLBM_GRAD_SHAPE(2)
        MFLBM_GRAD_SHAPE(3)
        MFLBM_GRAD_SHAPE(4)
#undef MFLBM_GRAD_SHAPE
        default: break;
    }
}

template <typename T>
void Launch<T>::velocity_change(const Sparse<T>& S, const StepConst<T>& P, double* prev, double* part, double* out,
                                hipStream_t s) {
    const int nb = (int)blocks(S.nf);
    if (nb > 0) dev::k_velocity_change<T><<<nb, 256, 0, s>>>(S, P, prev, part);
    dev::k_sum_pairs<T><<<1, 256, 0, s>>>(part, nb, out);
}

template <typename T>
void Launch<T>::aux_refresh(const Fields<T>& F, const StepConst<T>& P, const NodeLists& L, T* aux, hipStream_t s) {
    if (L.n_fluid > 0) dev::k_aux_refresh<T><<<blocks(L.n_fluid), 256, 0, s>>>(F, P, L.fluid, L.n_fluid, aux);
}

template <typename T>
void Launch<T>::cells(const Sparse<T>& S, T* dense, const Dims& d, const int32_t* ext_node, const int32_t* ext_off,
                      int n_ext, bool to_dense, hipStream_t s) {
    if (to_dense) {
        if (S.nf > 0) dev::k_fluid_cells<T, true><<<blocks(S.nf), 256, 0, s>>>(S, dense, d);
        if (n_ext > 0) dev::k_extra_cells<T, true><<<blocks(n_ext), 256, 0, s>>>(S, dense, d, ext_node, ext_off);
    } else {
        if (S.nf > 0) dev::k_fluid_cells<T, false><<<blocks(S.nf), 256, 0, s>>>(S, dense, d);
        if (n_ext > 0) dev::k_extra_cells<T, false><<<blocks(n_ext), 256, 0, s>>>(S, dense, d, ext_node, ext_off);
    }
}

template <typename T>
void Launch<T>::init_phi(const Fields<T>& F, int option, double z0, double phi_inlet, int open_z, double sa_target,
                         uint64_t seed, hipStream_t s) {
    dev::k_init_phi<T><<<blocks(F.d.S4), 256, 0, s>>>(F, option, z0, phi_inlet, open_z, sa_target, seed);
}

template <typename T>
void Launch<T>::init_eq(const Fields<T>& F, const double* rho, const double* u, const double* v, const double* w,
                        bool relaxed, double rho_ref, hipStream_t s) {
    if (relaxed) dev::k_init_eq<T, true><<<blocks(F.d.S1), 256, 0, s>>>(F, rho, u, v, w, rho_ref);
    else dev::k_init_eq<T, false><<<blocks(F.d.S1), 256, 0, s>>>(F, rho, u, v, w, rho_ref);
}

template <typename T>
void Launch<T>::macro(const Sparse<T>& S, const StepConst<T>& P, const Dims& d, double* rho, double* u, double* v,
                      double* w, hipStream_t s) {
    if (S.nf > 0) dev::k_macro<T><<<blocks(S.nf), 256, 0, s>>>(S, P, d, rho, u, v, w);
}

template <typename T>
void Launch<T>::monitor(const Sparse<T>& S, const StepConst<T>& P, const T* phi, const Dims& d, const int32_t* zstart,
                        int nsplit, double* part, double* out, hipStream_t s) {
    dim3 grid(nsplit, d.nz);
    dev::k_monitor_partial<T><<<grid, 256, 0, s>>>(S, P, phi, d, zstart, part);
    dev::k_monitor_combine<T><<<blocks((int64_t)d.nz * dev::MON_VALUES, 64), 64, 0, s>>>(part, nsplit, d.nz, out);
}

template <typename T>
void Launch<T>::pack_solid_normals(const T* x, const T* y, const T* z, const int32_t* wet, int n, T* dst, hipStream_t s) {
    if (n > 0) k_pack_solid_normals<T><<<blocks(n), 256, 0, s>>>(x, y, z, wet, n, dst);
}

template <typename T>
void Launch<T>::to_real(const double* src, T* dst, int64_t n, hipStream_t s) {
    k_to_real<T><<<blocks(n), 256, 0, s>>>(src, dst, n);
}

}  // namespace mflbm
