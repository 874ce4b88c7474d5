// Host-side launchers of the step kernels, one explicit instantiation per precision
// (kernels_f64.hip, kernels_f32.hip).  All launches are asynchronous on `s`.
#pragma once
#include <hip/hip_runtime.h>
#include "lattice.h"

namespace mflbm {

template <typename T>
struct Launch {
    // ghosts: the ghost phi to write as well (its `rest` is set here), or null
    static void collide(const Sparse<T>& S, T* phi, const Dims& d, const StepConst<T>& P, bool odd, const PhiGhosts<T>* ghosts,
                        hipStream_t s);
    // Periodic copies and open boundaries of one step; B without nbc, npair, blocks and split.
    static void boundary(const Sparse<T>& S, const Fields<T>& F, const StepConst<T>& P, BoundaryArgs<T> B, bool after_odd,
                         hipStream_t s);
    static void porous_plate(const Sparse<T>& S, const Dims& d, const StepConst<T>& P, const int32_t* pmap, int zp,
                             int blocked, bool after_odd, hipStream_t s);
    static void conv_init(const Fields<T>& F, T rho_ref, T* conv, hipStream_t s);
    // inner: only of the nodes [1, nx] x [1, ny] x [0, nz+1]
    static void phi_extrap(const Fields<T>& F, const NodeLists& L, hipStream_t s, bool inner = false);
    static void normals(const Fields<T>& F, const StepConst<T>& P, const NodeLists& L, hipStream_t s);
    static void normal_extrap(const Fields<T>& F, const NodeLists& L, hipStream_t s);
    static void curvature(const Fields<T>& F, const StepConst<T>& P, const NodeLists& L, T* aux, hipStream_t s);
    static void gradient(const GradArgs<T>& A, const StepConst<T>& P, hipStream_t s);
    // The two-pass chain with, in its second launch, the populations' part of boundary().
    static void gradient_boundary(const GradArgs<T>& A, const Sparse<T>& S, const Fields<T>& F, const StepConst<T>& P,
                                  BoundaryArgs<T> B, bool after_odd, hipStream_t s);
    // Boxes of the two-pass chain's kernels, and its work lists: first their sizes (na and nb of
    // the descriptors), then, with the descriptors complete, the lists.
    // boxes of one of the kernels; columns: loaded columns of a box of k_grad_force
    static int tile_boxes(const Dims& d, bool force, int* columns = nullptr);
    static void tile_counts(const GradArgs<T>& A, TileDesc* ndesc, TileDesc* fdesc, hipStream_t s);
    static void tile_fill(const GradArgs<T>& A, const TileFill& out, hipStream_t s);
    static void aux_refresh(const Fields<T>& F, const StepConst<T>& P, const NodeLists& L, T* aux, hipStream_t s);
    static void cells(const Sparse<T>& S, T* dense, const Dims& d, const int32_t* ext_node, const int32_t* ext_off,
                      int n_ext, bool to_dense, hipStream_t s);
    static void init_phi(const Fields<T>& F, int option, double z0, double phi_inlet, int open_z, double sa_target,
                         uint64_t seed, hipStream_t s);
    static void init_eq(const Fields<T>& F, const double* rho, const double* u, const double* v, const double* w,
                        bool relaxed, double rho_ref, hipStream_t s);
    static void macro(const Sparse<T>& S, const StepConst<T>& P, const Dims& d, double* rho, double* u, double* v,
                      double* w, hipStream_t s);
    // relative velocity change since the last call; part: 2 * ceil(nf / 256) doubles, out: 2
    static void velocity_change(const Sparse<T>& S, const StepConst<T>& P, double* prev, double* part, double* out,
                                hipStream_t s);
    static void monitor(const Sparse<T>& S, const StepConst<T>& P, const T* phi, const Dims& d, const int32_t* zstart,
                        int nsplit, double* part, double* out, hipStream_t s);
    static void to_real(const double* src, T* dst, int64_t n, hipStream_t s);
    // dst[c * n + w] = component c of the solid normal at S4 node wet[w].
    static void pack_solid_normals(const T* x, const T* y, const T* z, const int32_t* wet, int n, T* dst, hipStream_t s);
};

extern template struct Launch<double>;
extern template struct Launch<float>;

}  // namespace mflbm
