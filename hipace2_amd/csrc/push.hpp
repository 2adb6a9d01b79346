// Plasma push arithmetic shared by the push kernel and its adjoint: the dual number of the
// second-order Taylor sub-step, the momentum right-hand side and the particle boundary
// parameters. Templates on the number type, so the adjoint instantiates the same
// expressions with forward-mode tangents.
#pragma once
#include <hip/hip_runtime.h>

namespace hpq {

// Forward-mode dual number for the second-order Taylor step (src/utils/DualNumbers.H:13-43).
// A factor or term that does not depend on the parameter stays a plain number instead of a dual
// number with derivative zero: the products with that zero, which no compiler may drop, only
// ever added a zero.
template <class R>
struct Dual {
    R v, e;
    __host__ __device__ Dual(R a) : v(a), e(0) {}
    __host__ __device__ Dual(R a, R b) : v(a), e(b) {}
};
template <class R>
__host__ __device__ __forceinline__ Dual<R> operator+(const Dual<R>& a, const Dual<R>& b) { return {a.v + b.v, a.e + b.e}; }
template <class R>
__host__ __device__ __forceinline__ Dual<R> operator-(const Dual<R>& a, const Dual<R>& b) { return {a.v - b.v, a.e - b.e}; }
template <class R>
__host__ __device__ __forceinline__ Dual<R> operator*(const Dual<R>& a, const Dual<R>& b) {
    return {a.v * b.v, a.e * b.v + a.v * b.e};
}
template <class R, class S>
__host__ __device__ __forceinline__ Dual<R> operator+(const Dual<R>& a, const S& b) { return {a.v + b, a.e}; }
template <class R, class S>
__host__ __device__ __forceinline__ Dual<R> operator-(const Dual<R>& a, const S& b) { return {a.v - b, a.e}; }
template <class R, class S>
__host__ __device__ __forceinline__ Dual<R> operator*(const Dual<R>& a, const S& b) { return {a.v * b, a.e * b}; }

// PlasmaMomentumPush, src/particles/pusher/PushPlasmaParticles.H:37-75 (no laser terms). T: the
// number type of the particle, F of the fields at it, S of the constants.
template <class T, class F, class S>
__host__ __device__ __forceinline__ void momentum_rhs(const T& ux, const T& uy, const T& psi_inv, const F& ExmBy,
                                                      const F& EypBx, const F& Ez, const F& Bx_c, const F& By_c,
                                                      const F& Bz, S ci, S qmc, T& dux, T& duy, T& dpsi) {
    const S half = S(0.5), cc = ci * ci, qc = qmc * ci;
    const T gamma_psi = (psi_inv * half) * psi_inv * (ux * ux * cc + S(1.0) + uy * uy * cc) + half;
    dux = (gamma_psi * ExmBy + By_c + (uy * Bz) * psi_inv) * qmc;
    duy = (gamma_psi * EypBx - Bx_c - (ux * Bz) * psi_inv) * qmc;
    dpsi = ((ux * ExmBy + uy * EypBx) * ci * psi_inv - Ez) * qc;
}

struct BC {
    int type;
    double plo0, plo1, phi0, phi1;
};

}  // namespace hpq
