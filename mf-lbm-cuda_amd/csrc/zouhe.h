// Open-boundary column functions: Zou-He pressure inlet (k = 1) and outlet (k = nz) for
// one (i, j) column (src/main_iteration_GPU.cu:1085-1241 inlet, 1363-1524 outlet), the
// velocity inlet, the convective outlet and the porous plate.
//
// Written against accessors so the same bodies serve the device kernel and the host-side pass
// that records which population slots the boundary touches:
//   f.rd(a, b, c, e), f.rw(a, b, c, e) -> the cell of slot e at node (a, b, c), loaded: get(g)
//       the population of colour g, set(g, v) replaces it, put() stores both (rw cells only)
//   wall(a, b, c)    -> int  solid flag
//   ph(a, b, c)      -> T&   order parameter
//   (porous plate) f(a, b, c, e, g) -> T&
// A column loads every cell before it stores the first, so that a thread waits for memory
// twice (the plane map, then the cells) rather than once per colour and store: boundary updates
// of a step 13.6 -> 7.7 us at 32^3 FP64, 14.0 -> 8.4 at 64^3 FP32, 42.8 -> 40.0 at 256^3 FP64,
// where the cells' bytes set the time.
// The sums follow the slot order of each reference variant; the orders differ between the
// before-odd and after-odd kernels and so does the rounding.  No branch depends on a
// population value, so a recording pass sees every access.
#pragma once
#include "lattice.h"

namespace mflbm {

// PHI = false leaves out the ghost planes of phi, which a caller may fill separately: inlet_phi
// for either inlet, four copies of phi(i, j, nz) for the Zou-He outlet, convective_phi.
template <typename T, class Phi>
MFLBM_HD void inlet_phi(const StepConst<T>& P, int i, int j, int w, Phi&& ph) {
    T& p0 = ph(i, j, 0);
    const T pv = P.phi_inlet * (1 - w) + p0 * w;
    p0 = pv;
    ph(i, j, -1) = pv;
    ph(i, j, -2) = pv;
    ph(i, j, -3) = pv;
}

// phi_nz: phi(i, j, nz) of this step
template <typename T, class Phi, class CP>
MFLBM_HD void convective_phi(const StepConst<T>& P, int i, int j, int nz, int w, T phi_nz, Phi&& ph, CP&& cphi) {
    const T u = P.uin_avg, tmp = T(1.0) / (T(1.0) + u);
    T& pg = ph(i, j, nz + 1);
    const T pv = ((cphi() + u * phi_nz) * tmp) * (1 - w) + pg * w;
    pg = pv;
    cphi() = pv;
    ph(i, j, nz + 2) = pv;
    ph(i, j, nz + 3) = pv;
    ph(i, j, nz + 4) = pv;
}

template <typename T, bool AFTER_ODD, bool PHI = true, class Acc, class Wall, class Phi>
MFLBM_HD void zou_he_column(const StepConst<T>& P, int i, int j, int nz, int do_in, int do_out, Acc&& f, Wall&& wall,
                            Phi&& ph) {
    const T c3 = T(0.333333333333333333), c6 = T(0.166666666666666667);
    if (do_in) {
        const int w = wall(i, j, 1);
        T rT[2];
        rT[1] = P.rho_in;
        rT[0] = P.rho_in * P.sa_inject;
        rT[1] = rT[1] - rT[0];
        if (!AFTER_ODD) {
            auto f0 = f.rd(i, j, 1, 0), f1 = f.rd(i - 1, j, 1, 1), f2 = f.rd(i + 1, j, 1, 2), f3 = f.rd(i, j - 1, 1, 3),
                 f4 = f.rd(i, j + 1, 1, 4), f7 = f.rd(i - 1, j - 1, 1, 7), f8 = f.rd(i + 1, j - 1, 1, 8),
                 f9 = f.rd(i - 1, j + 1, 1, 9), f10 = f.rd(i + 1, j + 1, 1, 10), f6 = f.rd(i, j, 2, 6),
                 f14 = f.rd(i + 1, j, 2, 14), f13 = f.rd(i - 1, j, 2, 13), f18 = f.rd(i, j + 1, 2, 18),
                 f17 = f.rd(i, j - 1, 2, 17);
            auto d5 = f.rw(i, j, 0, 5), d11 = f.rw(i - 1, j, 0, 11), d12 = f.rw(i + 1, j, 0, 12), d15 = f.rw(i, j - 1, 0, 15),
                 d16 = f.rw(i, j + 1, 0, 16);
            for (int g = 0; g < 2; ++g) {
                const T tt = (rT[g] - (f0.get(g) + f1.get(g) + f2.get(g) + f3.get(g) + f4.get(g) + f7.get(g) + f8.get(g) +
                                       f9.get(g) + f10.get(g) +
                                       T(2.0) * (f6.get(g) + f14.get(g) + f13.get(g) + f18.get(g) + f17.get(g)))) *
                             P.relaxation;
                const T tnx = T(0.5) * (f1.get(g) + f7.get(g) + f9.get(g) - (f2.get(g) + f8.get(g) + f10.get(g)));
                const T tny = T(0.5) * (f3.get(g) + f7.get(g) + f8.get(g) - (f4.get(g) + f10.get(g) + f9.get(g)));
                d5.set(g, (f6.get(g) + c3 * tt) * (1 - w) + d5.get(g) * w);
                d11.set(g, (f14.get(g) + c6 * tt - tnx) * (1 - w) + d11.get(g) * w);
                d12.set(g, (f13.get(g) + c6 * tt + tnx) * (1 - w) + d12.get(g) * w);
                d15.set(g, (f18.get(g) + c6 * tt - tny) * (1 - w) + d15.get(g) * w);
                d16.set(g, (f17.get(g) + c6 * tt + tny) * (1 - w) + d16.get(g) * w);
            }
            d5.put(); d11.put(); d12.put(); d15.put(); d16.put();
        } else {
            auto f0 = f.rd(i, j, 1, 0), f1 = f.rd(i, j, 1, 1), f2 = f.rd(i, j, 1, 2), f3 = f.rd(i, j, 1, 3),
                 f4 = f.rd(i, j, 1, 4), f5 = f.rd(i, j, 1, 5), f7 = f.rd(i, j, 1, 7), f8 = f.rd(i, j, 1, 8),
                 f9 = f.rd(i, j, 1, 9), f10 = f.rd(i, j, 1, 10), f11 = f.rd(i, j, 1, 11), f12 = f.rd(i, j, 1, 12),
                 f15 = f.rd(i, j, 1, 15), f16 = f.rd(i, j, 1, 16);
            auto d6 = f.rw(i, j, 1, 6), d13 = f.rw(i, j, 1, 13), d14 = f.rw(i, j, 1, 14), d17 = f.rw(i, j, 1, 17),
                 d18 = f.rw(i, j, 1, 18);
            for (int g = 0; g < 2; ++g) {
                const T tt = (rT[g] - (f0.get(g) + f2.get(g) + f1.get(g) + f4.get(g) + f3.get(g) + f8.get(g) + f7.get(g) +
                                       f10.get(g) + f9.get(g) +
                                       T(2.0) * (f5.get(g) + f11.get(g) + f12.get(g) + f15.get(g) + f16.get(g)))) *
                             P.relaxation;
                const T tnx = T(0.5) * (f2.get(g) + f8.get(g) + f10.get(g) - (f1.get(g) + f7.get(g) + f9.get(g)));
                const T tny = T(0.5) * (f4.get(g) + f9.get(g) + f10.get(g) - (f3.get(g) + f8.get(g) + f7.get(g)));
                d6.set(g, (f5.get(g) + c3 * tt) * (1 - w) + d6.get(g) * w);
                d13.set(g, (f12.get(g) + c6 * tt + tnx) * (1 - w) + d13.get(g) * w);
                d14.set(g, (f11.get(g) + c6 * tt - tnx) * (1 - w) + d14.get(g) * w);
                d17.set(g, (f16.get(g) + c6 * tt + tny) * (1 - w) + d17.get(g) * w);
                d18.set(g, (f15.get(g) + c6 * tt - tny) * (1 - w) + d18.get(g) * w);
            }
            d6.put(); d13.put(); d14.put(); d17.put(); d18.put();
        }
        if (PHI) inlet_phi<T>(P, i, j, w, ph);
    }
    if (do_out) {
        const int w = wall(i, j, nz);
        const T phv = ph(i, j, nz);
        if (!AFTER_ODD) {
            auto f0 = f.rd(i, j, nz, 0), f1 = f.rd(i - 1, j, nz, 1), f2 = f.rd(i + 1, j, nz, 2), f3 = f.rd(i, j - 1, nz, 3),
                 f4 = f.rd(i, j + 1, nz, 4), f7 = f.rd(i - 1, j - 1, nz, 7), f8 = f.rd(i + 1, j - 1, nz, 8),
                 f9 = f.rd(i - 1, j + 1, nz, 9), f10 = f.rd(i + 1, j + 1, nz, 10), f5 = f.rd(i, j, nz - 1, 5),
                 f11 = f.rd(i - 1, j, nz - 1, 11), f12 = f.rd(i + 1, j, nz - 1, 12), f15 = f.rd(i, j - 1, nz - 1, 15),
                 f16 = f.rd(i, j + 1, nz - 1, 16);
            auto d6 = f.rw(i, j, nz + 1, 6), d13 = f.rw(i - 1, j, nz + 1, 13), d14 = f.rw(i + 1, j, nz + 1, 14),
                 d17 = f.rw(i, j - 1, nz + 1, 17), d18 = f.rw(i, j + 1, nz + 1, 18);
            T t1 = f0.get(0) + f1.get(0) + f2.get(0) + f3.get(0) + f4.get(0) + f7.get(0) + f8.get(0) + f9.get(0) + f10.get(0) +
                   T(2.0) * (f5.get(0) + f11.get(0) + f12.get(0) + f15.get(0) + f16.get(0)) + f0.get(1) + f1.get(1) +
                   f2.get(1) + f3.get(1) + f4.get(1) + f7.get(1) + f8.get(1) + f9.get(1) + f10.get(1) +
                   T(2.0) * (f5.get(1) + f11.get(1) + f12.get(1) + f15.get(1) + f16.get(1)) - P.rho_out;
            const T t2 = t1 * T(0.5) * (T(1.0) - phv);
            t1 = t1 - t2;
            const T tt2[2] = {t1, t2};
            for (int g = 0; g < 2; ++g) {
                const T tt = tt2[g];
                const T tnx = T(0.5) * (f1.get(g) + f7.get(g) + f9.get(g) - (f2.get(g) + f8.get(g) + f10.get(g)));
                const T tny = T(0.5) * (f3.get(g) + f7.get(g) + f8.get(g) - (f4.get(g) + f10.get(g) + f9.get(g)));
                d6.set(g, (f5.get(g) - c3 * tt) * (1 - w) + d6.get(g) * w);
                d13.set(g, (f12.get(g) - c6 * tt - tnx) * (1 - w) + d13.get(g) * w);
                d14.set(g, (f11.get(g) - c6 * tt + tnx) * (1 - w) + d14.get(g) * w);
                d17.set(g, (f16.get(g) - c6 * tt - tny) * (1 - w) + d17.get(g) * w);
                d18.set(g, (f15.get(g) - c6 * tt + tny) * (1 - w) + d18.get(g) * w);
            }
            d6.put(); d13.put(); d14.put(); d17.put(); d18.put();
        } else {
            auto f0 = f.rd(i, j, nz, 0), f1 = f.rd(i, j, nz, 1), f2 = f.rd(i, j, nz, 2), f3 = f.rd(i, j, nz, 3),
                 f4 = f.rd(i, j, nz, 4), f6 = f.rd(i, j, nz, 6), f7 = f.rd(i, j, nz, 7), f8 = f.rd(i, j, nz, 8),
                 f9 = f.rd(i, j, nz, 9), f10 = f.rd(i, j, nz, 10), f13 = f.rd(i, j, nz, 13), f14 = f.rd(i, j, nz, 14),
                 f17 = f.rd(i, j, nz, 17), f18 = f.rd(i, j, nz, 18);
            auto d5 = f.rw(i, j, nz, 5), d11 = f.rw(i, j, nz, 11), d12 = f.rw(i, j, nz, 12), d15 = f.rw(i, j, nz, 15),
                 d16 = f.rw(i, j, nz, 16);
            T t1 = f0.get(0) + f2.get(0) + f1.get(0) + f4.get(0) + f3.get(0) + f8.get(0) + f7.get(0) + f10.get(0) + f9.get(0) +
                   T(2.0) * (f6.get(0) + f14.get(0) + f13.get(0) + f18.get(0) + f17.get(0)) + f0.get(1) + f2.get(1) +
                   f1.get(1) + f4.get(1) + f3.get(1) + f8.get(1) + f7.get(1) + f10.get(1) + f9.get(1) +
                   T(2.0) * (f6.get(1) + f14.get(1) + f13.get(1) + f18.get(1) + f17.get(1)) - P.rho_out;
            const T t2 = t1 * T(0.5) * (T(1.0) - phv);
            t1 = t1 - t2;
            const T tt2[2] = {t1, t2};
            for (int g = 0; g < 2; ++g) {
                const T tt = tt2[g];
                const T tnx = T(0.5) * (f2.get(g) + f8.get(g) + f10.get(g) - (f1.get(g) + f7.get(g) + f9.get(g)));
                const T tny = T(0.5) * (f4.get(g) + f10.get(g) + f9.get(g) - (f3.get(g) + f7.get(g) + f8.get(g)));
                d5.set(g, (f6.get(g) - c3 * tt) * (1 - w) + d5.get(g) * w);
                d11.set(g, (f14.get(g) - c6 * tt + tnx) * (1 - w) + d11.get(g) * w);
                d12.set(g, (f13.get(g) - c6 * tt - tnx) * (1 - w) + d12.get(g) * w);
                d15.set(g, (f18.get(g) - c6 * tt + tny) * (1 - w) + d15.get(g) * w);
                d16.set(g, (f17.get(g) - c6 * tt - tny) * (1 - w) + d16.get(g) * w);
            }
            d5.put(); d11.put(); d12.put(); d15.put(); d16.put();
        }
        if (PHI)
            for (int m = 1; m <= 4; ++m) ph(i, j, nz + m) = phv;
    }
}

// Velocity inlet at k = 1 by bounce-back with the injected momentum of the column's inlet
// velocity w_in, split between the colours by the injected saturation
// (src/main_iteration_GPU.cu:1008-1077, inlet_bounce_back_velocity_BC_{before,after}_odd).
template <typename T, bool AFTER_ODD, bool PHI = true, class Acc, class Wall, class Phi>
MFLBM_HD void velocity_inlet_column(const StepConst<T>& P, int i, int j, T w_in, Acc&& f, Wall&& wall, Phi&& ph) {
    const int w = wall(i, j, 1);
    T t2 = w_in * P.relaxation;
    const T t1 = t2 * P.sa_inject;  // fluid 1
    t2 = t2 - t1;                   // fluid 2
    const T a1 = T(6.0) * (T(1.0) / T(18.0)), a2 = T(6.0) * (T(1.0) / T(36.0));
    if (!AFTER_ODD) {
        auto f6 = f.rd(i, j, 1, 6), f14 = f.rd(i, j, 1, 14), f13 = f.rd(i, j, 1, 13), f18 = f.rd(i, j, 1, 18),
             f17 = f.rd(i, j, 1, 17);
        auto d5 = f.rw(i, j, 0, 5), d11 = f.rw(i - 1, j, 0, 11), d12 = f.rw(i + 1, j, 0, 12), d15 = f.rw(i, j - 1, 0, 15),
             d16 = f.rw(i, j + 1, 0, 16);
        for (int g = 0; g < 2; ++g) {
            const T tg = g == 0 ? t1 : t2;
            d5.set(g, (f6.get(g) + a1 * tg) * (1 - w) + d5.get(g) * w);
            d11.set(g, (f14.get(g) + a2 * tg) * (1 - w) + d11.get(g) * w);
            d12.set(g, (f13.get(g) + a2 * tg) * (1 - w) + d12.get(g) * w);
            d15.set(g, (f18.get(g) + a2 * tg) * (1 - w) + d15.get(g) * w);
            d16.set(g, (f17.get(g) + a2 * tg) * (1 - w) + d16.get(g) * w);
        }
        d5.put(); d11.put(); d12.put(); d15.put(); d16.put();
    } else {
        auto f5 = f.rd(i, j, 0, 5), f12 = f.rd(i + 1, j, 0, 12), f11 = f.rd(i - 1, j, 0, 11), f16 = f.rd(i, j + 1, 0, 16),
             f15 = f.rd(i, j - 1, 0, 15);
        auto d6 = f.rw(i, j, 1, 6), d13 = f.rw(i, j, 1, 13), d14 = f.rw(i, j, 1, 14), d17 = f.rw(i, j, 1, 17),
             d18 = f.rw(i, j, 1, 18);
        for (int g = 0; g < 2; ++g) {
            const T tg = g == 0 ? t1 : t2;
            d6.set(g, (f5.get(g) + a1 * tg) * (1 - w) + d6.get(g) * w);
            d13.set(g, (f12.get(g) + a2 * tg) * (1 - w) + d13.get(g) * w);
            d14.set(g, (f11.get(g) + a2 * tg) * (1 - w) + d14.get(g) * w);
            d17.set(g, (f16.get(g) + a2 * tg) * (1 - w) + d17.get(g) * w);
            d18.set(g, (f15.get(g) + a2 * tg) * (1 - w) + d18.get(g) * w);
        }
        d6.put(); d13.put(); d14.put(); d17.put(); d18.put();
    }
    if (PHI) inlet_phi<T>(P, i, j, w, ph);
}

// Convective outlet at k = nz: the unknown populations and the ghost phi follow
// d/dt + u d/dz = 0 with u = P.uin_avg, from the values stored for the column at the last
// step (cs(e, g) populations, cphi() phi), which are then replaced
// (src/main_iteration_GPU.cu:1245-1357, outlet_convective_BC_{before,after}_odd).
template <typename T, bool AFTER_ODD, bool PHI = true, class Acc, class Wall, class Phi, class CS, class CP>
MFLBM_HD void convective_outlet_column(const StepConst<T>& P, int i, int j, int nz, Acc&& f, Wall&& wall, Phi&& ph,
                                       CS&& cs, CP&& cphi) {
    const T u = P.uin_avg;
    const T tmp = T(1.0) / (T(1.0) + u);
    const int w = wall(i, j, nz);
    if (!AFTER_ODD) {
        auto f6 = f.rd(i, j, nz, 6), f13 = f.rd(i - 1, j, nz, 13), f14 = f.rd(i + 1, j, nz, 14), f17 = f.rd(i, j - 1, nz, 17),
             f18 = f.rd(i, j + 1, nz, 18);
        auto d6 = f.rw(i, j, nz + 1, 6), d13 = f.rw(i - 1, j, nz + 1, 13), d14 = f.rw(i + 1, j, nz + 1, 14),
             d17 = f.rw(i, j - 1, nz + 1, 17), d18 = f.rw(i, j + 1, nz + 1, 18);
        for (int g = 0; g < 2; ++g) {
            d6.set(g, ((cs(6, g) + u * f6.get(g)) * tmp) * (1 - w) + d6.get(g) * w);
            d13.set(g, ((cs(13, g) + u * f13.get(g)) * tmp) * (1 - w) + d13.get(g) * w);
            d14.set(g, ((cs(14, g) + u * f14.get(g)) * tmp) * (1 - w) + d14.get(g) * w);
            d17.set(g, ((cs(17, g) + u * f17.get(g)) * tmp) * (1 - w) + d17.get(g) * w);
            d18.set(g, ((cs(18, g) + u * f18.get(g)) * tmp) * (1 - w) + d18.get(g) * w);
        }
        d6.put(); d13.put(); d14.put(); d17.put(); d18.put();
        for (int g = 0; g < 2; ++g) {
            cs(6, g) = d6.get(g);
            cs(13, g) = d13.get(g);
            cs(14, g) = d14.get(g);
            cs(17, g) = d17.get(g);
            cs(18, g) = d18.get(g);
        }
    } else {
        auto f5 = f.rd(i, j, nz - 1, 5), f11 = f.rd(i, j, nz - 1, 11), f12 = f.rd(i, j, nz - 1, 12),
             f15 = f.rd(i, j, nz - 1, 15), f16 = f.rd(i, j, nz - 1, 16);
        auto d5 = f.rw(i, j, nz, 5), d11 = f.rw(i, j, nz, 11), d12 = f.rw(i, j, nz, 12), d15 = f.rw(i, j, nz, 15),
             d16 = f.rw(i, j, nz, 16);
        for (int g = 0; g < 2; ++g) {
            d5.set(g, ((cs(6, g) + u * f5.get(g)) * tmp) * (1 - w) + d5.get(g) * w);
            d11.set(g, ((cs(14, g) + u * f11.get(g)) * tmp) * (1 - w) + d11.get(g) * w);
            d12.set(g, ((cs(13, g) + u * f12.get(g)) * tmp) * (1 - w) + d12.get(g) * w);
            d15.set(g, ((cs(18, g) + u * f15.get(g)) * tmp) * (1 - w) + d15.get(g) * w);
            d16.set(g, ((cs(17, g) + u * f16.get(g)) * tmp) * (1 - w) + d16.get(g) * w);
        }
        d5.put(); d11.put(); d12.put(); d15.put(); d16.put();
        for (int g = 0; g < 2; ++g) {
            cs(6, g) = d5.get(g);
            cs(14, g) = d11.get(g);
            cs(13, g) = d12.get(g);
            cs(18, g) = d15.get(g);
            cs(17, g) = d16.get(g);
        }
    }
    if (PHI) convective_phi<T>(P, i, j, nz, w, ph(i, j, nz), ph, cphi);
}

// Recording accessor of the host passes: note(a, b, c, e) for every cell.
template <class Note>
struct CellRecorder {
    Note note;
    struct Cell {
        double get(int) const { return 0.0; }
        void set(int, double) {}
        void put() {}
    };
    Cell rd(int a, int b, int c, int e) { note(a, b, c, e, false); return {}; }
    Cell rw(int a, int b, int c, int e) { note(a, b, c, e, true); return {}; }
};
template <class Note>
CellRecorder(Note) -> CellRecorder<Note>;

// Porous plate at k = zp that lets one colour through and reflects the other, `blocked`
// (0 = fluid 1, 1 = fluid 2) (src/main_iteration_GPU.cu:1744-1882, porous_plate_BC_*).
template <bool AFTER_ODD, class Acc>
MFLBM_HD void porous_plate_column(int i, int j, int zp, int blocked, Acc&& f) {
    const int b = blocked, c = 1 - blocked;
    if (!AFTER_ODD) {
        f(i, j, zp, 6, b) = f(i, j, zp - 1, 5, b);
        f(i - 1, j, zp, 13, b) = f(i, j, zp - 1, 12, b);
        f(i + 1, j, zp, 14, b) = f(i, j, zp - 1, 11, b);
        f(i, j - 1, zp, 17, b) = f(i, j, zp - 1, 16, b);
        f(i, j + 1, zp, 18, b) = f(i, j, zp - 1, 15, b);
        f(i, j, zp, 5, b) = f(i, j, zp + 1, 6, b);
        f(i + 1, j, zp, 12, b) = f(i, j, zp + 1, 13, b);
        f(i - 1, j, zp, 11, b) = f(i, j, zp + 1, 14, b);
        f(i, j + 1, zp, 16, b) = f(i, j, zp + 1, 17, b);
        f(i, j - 1, zp, 15, b) = f(i, j, zp + 1, 18, b);
        const int up[5] = {6, 13, 14, 17, 18}, dn[5] = {5, 12, 11, 16, 15};
        for (int m = 0; m < 5; ++m) f(i, j, zp, up[m], c) = f(i, j, zp + 1, up[m], c);
        for (int m = 0; m < 5; ++m) f(i, j, zp, dn[m], c) = f(i, j, zp - 1, dn[m], c);
    } else {
        f(i, j, zp - 1, 5, b) = f(i, j, zp, 6, b);
        f(i, j, zp - 1, 12, b) = f(i - 1, j, zp, 13, b);
        f(i, j, zp - 1, 11, b) = f(i + 1, j, zp, 14, b);
        f(i, j, zp - 1, 16, b) = f(i, j - 1, zp, 17, b);
        f(i, j, zp - 1, 15, b) = f(i, j + 1, zp, 18, b);
        f(i, j, zp + 1, 6, b) = f(i, j, zp, 5, b);
        f(i, j, zp + 1, 13, b) = f(i + 1, j, zp, 12, b);
        f(i, j, zp + 1, 14, b) = f(i - 1, j, zp, 11, b);
        f(i, j, zp + 1, 17, b) = f(i, j + 1, zp, 16, b);
        f(i, j, zp + 1, 18, b) = f(i, j - 1, zp, 15, b);
        const int up[5] = {6, 13, 14, 17, 18}, dn[5] = {5, 12, 11, 16, 15};
        for (int m = 0; m < 5; ++m) f(i, j, zp - 1, dn[m], c) = f(i, j, zp, dn[m], c);
        for (int m = 0; m < 5; ++m) f(i, j, zp + 1, up[m], c) = f(i, j, zp, up[m], c);
    }
}

// Population slots the periodic ghost copies move, in the reference's kernel order
// (Z faces, Y faces, ZY edges; src/main_iteration_GPU.cu:1529-1689).  cb(dst_node,
// src_node, slot) receives s1 node indices; a later call for the same destination
// overrides an earlier one, as the later reference kernel overwrites it.
template <class CB>
inline void periodic_pdf_copies(const Dims& d, int kper, int jper, bool odd, CB&& cb) {
    const int nx = d.nx, ny = d.ny, nz = d.nz;
    if (kper) {
        const int up[5] = {6, 14, 13, 18, 17}, dn[5] = {5, 11, 12, 15, 16};
        for (int j = 1; j <= ny; ++j)
            for (int i = 1; i <= nx; ++i)
                for (int m = 0; m < 5; ++m) {
                    if (!odd) {
                        cb(i1(d, i, j, nz + 1), i1(d, i, j, 1), up[m]);
                        cb(i1(d, i, j, 0), i1(d, i, j, nz), dn[m]);
                    } else {
                        cb(i1(d, i, j, 1), i1(d, i, j, nz + 1), up[m]);
                        cb(i1(d, i, j, nz), i1(d, i, j, 0), dn[m]);
                    }
                }
    }
    if (jper) {
        const int up[5] = {4, 10, 9, 16, 18}, dn[5] = {3, 7, 8, 15, 17};
        for (int k = 1; k <= nz; ++k)
            for (int i = 1; i <= nx; ++i)
                for (int m = 0; m < 5; ++m) {
                    if (!odd) {
                        cb(i1(d, i, ny + 1, k), i1(d, i, 1, k), up[m]);
                        cb(i1(d, i, 0, k), i1(d, i, ny, k), dn[m]);
                    } else {
                        cb(i1(d, i, 1, k), i1(d, i, ny + 1, k), up[m]);
                        cb(i1(d, i, ny, k), i1(d, i, 0, k), dn[m]);
                    }
                }
    }
    if (kper && jper) {
        for (int i = 1; i <= nx; ++i) {
            if (!odd) {
                cb(i1(d, i, ny + 1, nz + 1), i1(d, i, 1, 1), 18);
                cb(i1(d, i, ny + 1, 0), i1(d, i, 1, nz), 16);
                cb(i1(d, i, 0, nz + 1), i1(d, i, ny, 1), 17);
                cb(i1(d, i, 0, 0), i1(d, i, ny, nz), 15);
            } else {
                cb(i1(d, i, 1, 1), i1(d, i, ny + 1, nz + 1), 18);
                cb(i1(d, i, 1, nz), i1(d, i, ny + 1, 0), 16);
                cb(i1(d, i, ny, 1), i1(d, i, 0, nz + 1), 17);
                cb(i1(d, i, ny, nz), i1(d, i, 0, 0), 15);
            }
        }
    }
}

}  // namespace mflbm
