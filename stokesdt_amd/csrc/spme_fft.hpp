// The SPME transforms' shared pieces: the influence multiply and the launches
// of the two-stage kernels (fft_kernels.hpp, one source file per precision).
#pragma once
#include <cmath>
#include "sdt_internal.hpp"

namespace sdt {

// raises a kernel's dynamic LDS limit once per kernel and size: later
// launches (and graph captures of them) make no attribute call
void allow_lds(const void* fn, size_t bytes);

// The RPY influence tensor at one wave vector (src/mob/spme.cc:201-310,
// spme.h:114-123), applied to the NC components of one right-hand side.
// Mono (NC = 3): B = lm2 (1 - k^2/3)(I - k k^T / k^2). Poly (NC = 6, spreads
// of f and a^2 f): the reference's three mesh round trips (flags 1, 2, 2)
// reduce to two outputs
//   U = G (F f - k^2/6 F[a^2 f]),  W = -k^2/6 G F f,  G = lm2 (I - k k^T / k^2)
// interpolated as interp(U) + a_i^2 interp(W).
// lm2 = 6 pi e^{-k^2 / 4 xi^2} / k^2 (1 + k^2/4xi^2 + k^4/8xi^4) |b|^2; the
// exponential and |b|^2 are products over the dimensions, so they come as one
// factor per mesh index (influence_factors) and f is the product of three.
// Wave vectors come as integers m (k = 2 pi m / L): |m|^2 and the direction
// m / |m| are then free of the rounding of 2 pi / L, which would enter every
// mode with the same sign.
template <typename T>
struct Influence {
    T c, ck, cq;   // 6 pi / dk^2, dk^2 and dk^2 / xi^2 for dk = 2 pi / L
    __device__ __forceinline__ Influence(double box, double xi) {
        const double dk = 2.0 * M_PI / box;
        c = (T)(6.0 * M_PI / (dk * dk));
        ck = (T)(dk * dk);
        cq = (T)(dk * dk / (xi * xi));
    }
    template <int NC>
    __device__ __forceinline__ void apply(int mx, int my, int mz, T f, cplx<T>* g) const {
        const int n = mx * mx + my * my + mz * mz;
        const T tn = (T)n, in = n > 0 ? T(1) / tn : T(0);
        const T x = (T)mx, y = (T)my, z = (T)mz;
        const T q = tn * cq;
        const T m2 = c * f * in * (T(1) + q * (T(0.25) + q * T(0.125)));
        // (I - m m^T / |m|^2) v, scaled by s
        auto project = [&](cplx<T>* v, T s) __attribute__((always_inline)) {
            const T dr = (x * v[0].x + y * v[1].x + z * v[2].x) * in;
            const T di = (x * v[0].y + y * v[1].y + z * v[2].y) * in;
            v[0] = cplx<T>{s * (v[0].x - x * dr), s * (v[0].y - x * di)};
            v[1] = cplx<T>{s * (v[1].x - y * dr), s * (v[1].y - y * di)};
            v[2] = cplx<T>{s * (v[2].x - z * dr), s * (v[2].y - z * di)};
        };
        if constexpr (NC == 3) {
            project(g, m2 * (T(1) - tn * (ck / T(3))));
        } else {
            const T r = -tn * (ck / T(6));
            cplx<T> w[3];
#pragma unroll
            for (int i = 0; i < 3; i++) {
                w[i] = cplx<T>{r * g[i].x, r * g[i].y};
                g[i] = cplx<T>{g[i].x + r * g[3 + i].x, g[i].y + r * g[3 + i].y};
            }
            project(g, m2);
            project(w, m2);
#pragma unroll
            for (int i = 0; i < 3; i++) g[3 + i] = w[i];
        }
    }
};

// Launches of the two-stage transforms; tw: K roots of unity (cos, sin), fac:
// the influence factors per mesh index
template <typename T>
struct Fft2Launch {
    static bool has(int K);          // K has a two-stage kernel
    static bool plane_fits(int K);   // and the fused x + y plane fits LDS
    static bool has_xy(int K);       // and separate x and y passes
    static void plane(int K, bool fwd, int nmesh, T* real, cplx<T>* spec, const double* tw,
                      hipStream_t s);
    static void xy(int K, bool fwd, int nmesh, T* real, cplx<T>* spec, const double* tw,
                   hipStream_t s);
    // ntmax, lnpmax: at most that many threads and 2^lnpmax pencils per
    // component in a workgroup
    static void z(int K, int NC, int b, cplx<T>* spec, const double* tw, const double* fac,
                  int ntmax, int lnpmax, double box, double xi, hipStream_t s);
};

}  // namespace sdt
