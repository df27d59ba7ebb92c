// Two-stage transforms K = R1 R2 with the mesh side known at compile time:
// the fused x + y plane passes, the separate x and y passes and the z pass
// with the influence multiply. Included by one source file per precision.
//
// What bounds them is HBM (a copy reaches 5.0 TB/s on this card): each pass
// reads and writes its data once. The general radix chain of fft_lds.hpp that
// they replace took a trip through LDS with run-time index arithmetic per
// radix (four for K = 90 = 2 3 3 5) and reached a third of that. Measured,
// TB/s forward plane / z / inverse plane, before -> after:
//   K =  90 FP32, 300 meshes  1.7 / 2.1 / 1.7 -> 5.2 / 4.7 / 4.4
//   K =  90 FP64,  48 meshes  1.7 / 1.9 / 1.7 -> 5.7 / 4.8 / 4.7
//   K = 128 FP32, 300 meshes  5.0 / 3.5 / 4.3 -> 5.1 / 4.4 / 5.5
//   K = 128 FP64, 300 meshes  2.8 / 3.0 / 2.3 -> 4.9 / 4.7 / 4.9
//   K = 180 FP32,  48 meshes  1.8 / 2.2 / 1.7 -> 3.7 / 4.2 / 3.6 (one
//     workgroup per CU: its phases are not overlapped)
// separate x and y passes (both, in bytes moved):
//   K = 216 FP32,  24 meshes  2.1 / 2.2 / 2.1 -> 4.0 / 3.9 / 3.9
//   K = 256 FP64,  18 meshes  2.4 / 1.7 / 2.4 -> 3.9 / 2.4 / 3.9
//
// A stage holds one butterfly in registers. With first radix A and last radix
// B (K = A B), butterfly j < B of stage 1 takes elements j + B u (u < A),
// applies w_K^(j u) and leaves its outputs in LDS as row j of a pencil's
// B x A array; butterfly j < A of stage 2 takes column j and holds the
// results j + A u (u < B). Rows are padded to an odd length and pencils to an
// odd stride, so both accesses and the pencil-wise ones spread over the banks.
// The first stage reads global memory and the last one writes it directly:
// a pencil passes through LDS once per pair of stages. Twiddles w_K^(j u),
// j < R2, u < R1, are one table in LDS that serves either stage order.
#pragma once
#include "fft_lds.hpp"
#include "spme_fft.hpp"

namespace sdt {

constexpr int fft_odd(int n) { return n | 1; }

template <int R1, int R2>
struct Fft2 {
    static constexpr int K = R1 * R2, H = K / 2, Kh = H + 1;
    // first radix R1: R2 rows of R1; first radix R2: R1 rows of R2
    static constexpr int RA = fft_odd(R1), PSA = fft_odd(R2 * RA);
    static constexpr int RB = fft_odd(R2), PSB = fft_odd(R1 * RB);
    static constexpr int TWN = R2 * RA;        // twiddle table [R2][RA]
    // position of element e of a pencil after the stages with last radix L,
    // first radix F (row e / F, column e % F)
    static constexpr __device__ __forceinline__ int posa(int e) { return (e / R1) * RA + e % R1; }
    static constexpr __device__ __forceinline__ int posb(int e) { return (e / R2) * RB + e % R2; }
};

// The twiddle table in two steps, so that a workgroup's first data loads are
// issued between them: fetch() starts the table's loads, store() waits for
// those alone (they are the older ones) and writes them to LDS. CT: entries a
// thread fetches ahead, of at most ceil(K / blockDim).
template <typename T, int R1, int R2, int CT>
struct Twiddles {
    typedef Fft2<R1, R2> F;
    double2 w[CT];
    static __device__ __forceinline__ int entry(int i) { return (i / R1) * (i % R1); }   // < K
    __device__ __forceinline__ void fetch(const double* __restrict__ tw_g) {
        const double2* g = reinterpret_cast<const double2*>(tw_g);
#pragma unroll
        for (int c = 0; c < CT; c++)
            w[c] = g[entry(min((int)(threadIdx.x + c * blockDim.x), F::K - 1))];
    }
    __device__ __forceinline__ void store(cplx<T>* tw, const double* __restrict__ tw_g) const {
#pragma unroll
        for (int c = 0; c < CT; c++) {
            const int i = threadIdx.x + c * blockDim.x;
            if (i < F::K) tw[(i / R1) * F::RA + i % R1] = cplx<T>{(T)w[c].x, (T)w[c].y};
        }
        for (int i = threadIdx.x + CT * blockDim.x; i < F::K; i += blockDim.x) {
            const int e = entry(i);
            tw[(i / R1) * F::RA + i % R1] = cplx<T>{(T)tw_g[2 * e], (T)tw_g[2 * e + 1]};
        }
    }
};

// ------------------------------------------------ fused x + y plane -------
// One workgroup per z-plane of one mesh. Forward: x (two real rows per
// complex transform, first radix R2, last R1), then the split into the rows'
// half spectra on the way into the first stage along y (first radix R1, last
// R2). The inverse mirrors it. One LDS buffer; the split and the merge read
// one pencil layout and write the other, with a butterfly per thread in
// registers across the barrier.
template <typename T, int R1, int R2>
struct PlaneShape {
    typedef Fft2<R1, R2> F;
    static constexpr int items = F::Kh * R2;   // butterflies of the split / merge
    static constexpr int MAXB = items > 1024 ? 2 : 1;
    static constexpr int NT = ((items + MAXB - 1) / MAXB + 63) / 64 * 64;
    static constexpr int PENF = F::H * F::PSB > F::Kh * F::PSA ? F::H * F::PSB : F::Kh * F::PSA;
    static constexpr size_t lds_fwd = (size_t)(F::TWN + PENF) * sizeof(cplx<T>);
    static constexpr size_t lds_inv = (size_t)(F::TWN + F::Kh * F::PSA) * sizeof(cplx<T>);
};

template <typename T, int R1, int R2>
__global__ void __launch_bounds__((PlaneShape<T, R1, R2>::NT))
fft2_plane_fwd_kernel(const T* __restrict__ real, cplx<T>* __restrict__ spec,
                      const double* __restrict__ tw_g) {
    typedef Fft2<R1, R2> F;
    typedef PlaneShape<T, R1, R2> S;
    constexpr int K = F::K, H = F::H, Kh = F::Kh, NT = S::NT;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    cplx<T>* tw = reinterpret_cast<cplx<T>*>(smem_raw);
    cplx<T>* buf = tw + F::TWN;
    const size_t plane = blockIdx.x;
    const T* src = real + plane * K * K;
    {
        Twiddles<T, R1, R2, (K + NT - 1) / NT> t;
        t.fetch(tw_g);
        t.store(tw, tw_g);
    }
    __syncthreads();
    for (int it = threadIdx.x; it < H * R1; it += NT) {
        const int p = it / R1, j = it % R1;
        const T* ra = src + (size_t)(2 * p) * K + j;
        cplx<T> a[R2];
#pragma unroll
        for (int u = 0; u < R2; u++) a[u] = cplx<T>{ra[R1 * u], ra[K + R1 * u]};
        small_dft<T, R2, -1>(a);
#pragma unroll
        for (int u = 1; u < R2; u++) a[u] = cmul(a[u], tw[u * F::RA + j]);
        cplx<T>* o = buf + p * F::PSB + j * F::RB;
#pragma unroll
        for (int u = 0; u < R2; u++) o[u] = a[u];
    }
    __syncthreads();
    for (int it = threadIdx.x; it < H * R2; it += NT) {
        const int p = it / R2, j = it % R2;
        cplx<T>* o = buf + p * F::PSB + j;
        cplx<T> a[R1];
#pragma unroll
        for (int u = 0; u < R1; u++) a[u] = o[u * F::RB];
        small_dft<T, R1, -1>(a);
#pragma unroll
        for (int u = 0; u < R1; u++) o[u * F::RB] = a[u];
    }
    __syncthreads();
    {
        cplx<T> a[S::MAXB][R1];
#pragma unroll
        for (int v = 0; v < S::MAXB; v++) {
            const int it = threadIdx.x + v * NT;
            if (it >= Kh * R2) continue;
            const int j = it / Kh, kx = it % Kh;
            const int pk = F::posb(kx), pm = F::posb(kx == 0 ? 0 : K - kx);
            const T h = T(0.5);
#pragma unroll
            for (int u = 0; u < R1; u++) {
                // row y of the pair Z = A + i B: A when y is even, else B
                const int y = j + R2 * u;
                const cplx<T>* z = buf + (y >> 1) * F::PSB;
                const cplx<T> zk = z[pk], zm = z[pm];
                a[v][u] = (y & 1) ? cplx<T>{h * (zk.y + zm.y), h * (zm.x - zk.x)}
                                  : cplx<T>{h * (zk.x + zm.x), h * (zk.y - zm.y)};
            }
            small_dft<T, R1, -1>(a[v]);
#pragma unroll
            for (int u = 1; u < R1; u++) a[v][u] = cmul(a[v][u], tw[j * F::RA + u]);
        }
        __syncthreads();
#pragma unroll
        for (int v = 0; v < S::MAXB; v++) {
            const int it = threadIdx.x + v * NT;
            if (it >= Kh * R2) continue;
            const int j = it / Kh, kx = it % Kh;
            cplx<T>* o = buf + kx * F::PSA + j * F::RA;
#pragma unroll
            for (int u = 0; u < R1; u++) o[u] = a[v][u];
        }
        __syncthreads();
    }
    cplx<T>* dst = spec + plane * K * Kh;
    for (int it = threadIdx.x; it < Kh * R1; it += NT) {
        const int j = it / Kh, kx = it % Kh;
        const cplx<T>* o = buf + kx * F::PSA + j;
        cplx<T> a[R2];
#pragma unroll
        for (int u = 0; u < R2; u++) a[u] = o[u * F::RA];
        small_dft<T, R2, -1>(a);
#pragma unroll
        for (int u = 0; u < R2; u++) dst[(j + R1 * u) * Kh + kx] = a[u];
    }
}

template <typename T, int R1, int R2>
__global__ void __launch_bounds__((PlaneShape<T, R1, R2>::NT))
fft2_plane_inv_kernel(const cplx<T>* __restrict__ spec, T* __restrict__ real,
                      const double* __restrict__ tw_g) {
    typedef Fft2<R1, R2> F;
    typedef PlaneShape<T, R1, R2> S;
    constexpr int K = F::K, H = F::H, Kh = F::Kh, NT = S::NT;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    cplx<T>* tw = reinterpret_cast<cplx<T>*>(smem_raw);
    cplx<T>* buf = tw + F::TWN;
    const size_t plane = blockIdx.x;
    const cplx<T>* src = spec + plane * K * Kh;
    {
        Twiddles<T, R1, R2, (K + NT - 1) / NT> t;
        t.fetch(tw_g);
        t.store(tw, tw_g);
    }
    __syncthreads();
    for (int it = threadIdx.x; it < Kh * R2; it += NT) {
        const int j = it / Kh, kx = it % Kh;
        cplx<T> a[R1];
#pragma unroll
        for (int u = 0; u < R1; u++) a[u] = src[(j + R2 * u) * Kh + kx];
        small_dft<T, R1, +1>(a);
#pragma unroll
        for (int u = 1; u < R1; u++) a[u] = cmulc(a[u], tw[j * F::RA + u]);
        cplx<T>* o = buf + kx * F::PSA + j * F::RA;
#pragma unroll
        for (int u = 0; u < R1; u++) o[u] = a[u];
    }
    __syncthreads();
    for (int it = threadIdx.x; it < Kh * R1; it += NT) {
        const int j = it / Kh, kx = it % Kh;
        cplx<T>* o = buf + kx * F::PSA + j;
        cplx<T> a[R2];
#pragma unroll
        for (int u = 0; u < R2; u++) a[u] = o[u * F::RA];
        small_dft<T, R2, +1>(a);
#pragma unroll
        for (int u = 0; u < R2; u++) o[u * F::RA] = a[u];
    }
    __syncthreads();
    {
        cplx<T> a[S::MAXB][R1];
#pragma unroll
        for (int v = 0; v < S::MAXB; v++) {
            const int it = threadIdx.x + v * NT;
            if (it >= H * R2) continue;
            const int j = it / H, p = it % H;
            const int p0 = F::posa(2 * p), p1 = F::posa(2 * p + 1);
#pragma unroll
            for (int u = 0; u < R1; u++) {
                // Z = A + i B of the half spectra A, B of rows 2p, 2p + 1
                const int e = j + R2 * u;
                const bool lo = e <= H;
                const cplx<T>* o = buf + (lo ? e : K - e) * F::PSA;
                cplx<T> A = o[p0], B = o[p1];
                if (e == 0 || e == H) { A.y = T(0); B.y = T(0); }
                a[v][u] = lo ? cplx<T>{A.x - B.y, A.y + B.x} : cplx<T>{A.x + B.y, B.x - A.y};
            }
            small_dft<T, R1, +1>(a[v]);
#pragma unroll
            for (int u = 1; u < R1; u++) a[v][u] = cmulc(a[v][u], tw[j * F::RA + u]);
        }
        __syncthreads();
#pragma unroll
        for (int v = 0; v < S::MAXB; v++) {
            const int it = threadIdx.x + v * NT;
            if (it >= H * R2) continue;
            const int j = it / H, p = it % H;
            cplx<T>* o = buf + p * F::PSA + j * F::RA;
#pragma unroll
            for (int u = 0; u < R1; u++) o[u] = a[v][u];
        }
        __syncthreads();
    }
    T* dst = real + plane * K * K;
    for (int it = threadIdx.x; it < H * R1; it += NT) {
        const int p = it / R1, j = it % R1;
        const cplx<T>* o = buf + p * F::PSA + j;
        cplx<T> a[R2];
#pragma unroll
        for (int u = 0; u < R2; u++) a[u] = o[u * F::RA];
        small_dft<T, R2, +1>(a);
        T* ra = dst + (size_t)(2 * p) * K + j;
#pragma unroll
        for (int u = 0; u < R2; u++) {
            ra[R1 * u] = a[u].x;
            ra[K + R1 * u] = a[u].y;
        }
    }
}

// ------------------------------------------------ separate x, y passes ----
// Where a plane does not fit LDS. The same stages and operations as the fused
// plane kernels (the same bits). npen pencils per workgroup (x: pairs of rows, y: consecutive
// kx of one plane).
constexpr int kXYThreads = 256;

template <typename T, int R1, int R2>
__global__ void __launch_bounds__(kXYThreads)
fft2_x_r2c_kernel(long long npair, const T* __restrict__ real, cplx<T>* __restrict__ spec,
                  const double* __restrict__ tw_g, int npen) {
    typedef Fft2<R1, R2> F;
    constexpr int K = F::K, Kh = F::Kh;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    cplx<T>* tw = reinterpret_cast<cplx<T>*>(smem_raw);
    cplx<T>* buf = tw + F::TWN;
    const long long p0 = (long long)blockIdx.x * npen;
    const int np = (int)min((long long)npen, npair - p0);
    const T* src = real + p0 * 2 * K;
    auto load1 = [&](int it, cplx<T>* a) __attribute__((always_inline)) {
        const int p = it / R1, j = it % R1;
        const T* ra = src + (size_t)(2 * p) * K + j;
#pragma unroll
        for (int u = 0; u < R2; u++) a[u] = cplx<T>{ra[R1 * u], ra[K + R1 * u]};
    };
    {
        Twiddles<T, R1, R2, (K + kXYThreads - 1) / kXYThreads> t;
        t.fetch(tw_g);
        cplx<T> a[R2];
        int it = threadIdx.x;
        if (it < np * R1) load1(it, a);
        t.store(tw, tw_g);
        __syncthreads();
        while (it < np * R1) {
            const int p = it / R1, j = it % R1;
            small_dft<T, R2, -1>(a);
#pragma unroll
            for (int u = 1; u < R2; u++) a[u] = cmul(a[u], tw[u * F::RA + j]);
            cplx<T>* o = buf + p * F::PSB + j * F::RB;
#pragma unroll
            for (int u = 0; u < R2; u++) o[u] = a[u];
            it += kXYThreads;
            if (it < np * R1) load1(it, a);
        }
    }
    __syncthreads();
    for (int it = threadIdx.x; it < np * R2; it += kXYThreads) {
        const int p = it / R2, j = it % R2;
        cplx<T>* o = buf + p * F::PSB + j;
        cplx<T> a[R1];
#pragma unroll
        for (int u = 0; u < R1; u++) a[u] = o[u * F::RB];
        small_dft<T, R1, -1>(a);
#pragma unroll
        for (int u = 0; u < R1; u++) o[u * F::RB] = a[u];
    }
    __syncthreads();
    cplx<T>* dst = spec + p0 * 2 * Kh;
    for (int it = threadIdx.x; it < np * Kh; it += kXYThreads) {
        const int p = it / Kh, k = it % Kh;
        const cplx<T>* z = buf + p * F::PSB;
        const cplx<T> zk = z[F::posb(k)], zm = z[F::posb(k == 0 ? 0 : K - k)];
        const T h = T(0.5);
        cplx<T>* o = dst + (size_t)(2 * p) * Kh + k;
        o[0] = cplx<T>{h * (zk.x + zm.x), h * (zk.y - zm.y)};
        o[Kh] = cplx<T>{h * (zk.y + zm.y), h * (zm.x - zk.x)};
    }
}

template <typename T, int R1, int R2>
__global__ void __launch_bounds__(kXYThreads)
fft2_x_c2r_kernel(long long npair, const cplx<T>* __restrict__ spec, T* __restrict__ real,
                  const double* __restrict__ tw_g, int npen) {
    typedef Fft2<R1, R2> F;
    constexpr int K = F::K, H = F::H, Kh = F::Kh;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    cplx<T>* tw = reinterpret_cast<cplx<T>*>(smem_raw);
    cplx<T>* buf = tw + F::TWN;
    const long long p0 = (long long)blockIdx.x * npen;
    const int np = (int)min((long long)npen, npair - p0);
    const cplx<T>* src = spec + p0 * 2 * Kh;
    // Z = A + i B of the half spectra A, B of a row pair, element e at row
    // e % R2, column e / R2 of the pencil: a butterfly's own row, in place.
    // The loads of a thread (XB at a time) are in flight together.
    constexpr int XB = 4;
    Twiddles<T, R1, R2, (K + kXYThreads - 1) / kXYThreads> t;
    t.fetch(tw_g);
    for (int i0 = threadIdx.x; i0 < np * Kh; i0 += XB * kXYThreads) {
        cplx<T> A[XB], B[XB];
#pragma unroll
        for (int v = 0; v < XB; v++) {
            const int i = min(i0 + v * kXYThreads, np * Kh - 1);
            const int p = i / Kh, k = i % Kh;
            const cplx<T>* s = src + (size_t)(2 * p) * Kh + k;
            A[v] = s[0];
            B[v] = s[Kh];
        }
#pragma unroll
        for (int v = 0; v < XB; v++) {
            const int i = i0 + v * kXYThreads;
            const int p = i / Kh, k = i % Kh;
            if (i >= np * Kh) continue;
            if (k == 0 || k == H) { A[v].y = T(0); B[v].y = T(0); }
            cplx<T>* o = buf + p * F::PSA;
            o[(k % R2) * F::RA + k / R2] = cplx<T>{A[v].x - B[v].y, A[v].y + B[v].x};
            if (k > 0 && k < H) {
                const int e = K - k;
                o[(e % R2) * F::RA + e / R2] = cplx<T>{A[v].x + B[v].y, B[v].x - A[v].y};
            }
        }
    }
    t.store(tw, tw_g);
    __syncthreads();
    for (int it = threadIdx.x; it < np * R2; it += kXYThreads) {
        const int p = it / R2, j = it % R2;
        cplx<T>* o = buf + p * F::PSA + j * F::RA;
        cplx<T> a[R1];
#pragma unroll
        for (int u = 0; u < R1; u++) a[u] = o[u];
        small_dft<T, R1, +1>(a);
        o[0] = a[0];
#pragma unroll
        for (int u = 1; u < R1; u++) o[u] = cmulc(a[u], tw[j * F::RA + u]);
    }
    __syncthreads();
    T* dst = real + p0 * 2 * K;
    for (int it = threadIdx.x; it < np * R1; it += kXYThreads) {
        const int p = it / R1, j = it % R1;
        const cplx<T>* o = buf + p * F::PSA + j;
        cplx<T> a[R2];
#pragma unroll
        for (int u = 0; u < R2; u++) a[u] = o[u * F::RA];
        small_dft<T, R2, +1>(a);
        T* ra = dst + (size_t)(2 * p) * K + j;
#pragma unroll
        for (int u = 0; u < R2; u++) {
            ra[R1 * u] = a[u].x;
            ra[K + R1 * u] = a[u].y;
        }
    }
}

template <typename T, int R1, int R2, int SIGN>
__global__ void __launch_bounds__(kXYThreads)
fft2_y_kernel(cplx<T>* __restrict__ spec, const double* __restrict__ tw_g, int lnp) {
    typedef Fft2<R1, R2> F;
    constexpr int K = F::K, Kh = F::Kh;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    cplx<T>* tw = reinterpret_cast<cplx<T>*>(smem_raw);
    cplx<T>* buf = tw + F::TWN;
    const int NP = 1 << lnp;
    const int nkb = (Kh + NP - 1) >> lnp;
    // neighbouring chunks share cache lines (rows are not whole lines): keep
    // them on one XCD
    const unsigned lid = xcd_logical_id(blockIdx.x, gridDim.x);
    const int kx0 = (int)(lid % nkb) << lnp;
    cplx<T>* base = spec + (size_t)(lid / nkb) * K * Kh + kx0;
    const int nv = min(NP, Kh - kx0);
    auto load1 = [&](int it, cplx<T>* a) __attribute__((always_inline)) {
        const int l = min(it & (NP - 1), nv - 1), j = it >> lnp;
#pragma unroll
        for (int u = 0; u < R1; u++) a[u] = base[(size_t)(j + R2 * u) * Kh + l];
    };
    {
        Twiddles<T, R1, R2, (K + kXYThreads - 1) / kXYThreads> t;
        t.fetch(tw_g);
        cplx<T> a[R1];
        int it = threadIdx.x;
        if (it < NP * R2) load1(it, a);
        t.store(tw, tw_g);
        __syncthreads();
        while (it < NP * R2) {
            const int l = it & (NP - 1), j = it >> lnp;
            small_dft<T, R1, SIGN>(a);
#pragma unroll
            for (int u = 1; u < R1; u++)
                a[u] = SIGN < 0 ? cmul(a[u], tw[j * F::RA + u]) : cmulc(a[u], tw[j * F::RA + u]);
            cplx<T>* o = buf + l * F::PSA + j * F::RA;
#pragma unroll
            for (int u = 0; u < R1; u++) o[u] = a[u];
            it += kXYThreads;
            if (it < NP * R2) load1(it, a);
        }
    }
    __syncthreads();
    for (int it = threadIdx.x; it < NP * R1; it += kXYThreads) {
        const int l = it & (NP - 1), j = it >> lnp;
        if (l >= nv) continue;
        const cplx<T>* o = buf + l * F::PSA + j;
        cplx<T> a[R2];
#pragma unroll
        for (int u = 0; u < R2; u++) a[u] = o[u * F::RA];
        small_dft<T, R2, SIGN>(a);
#pragma unroll
        for (int u = 0; u < R2; u++) base[(size_t)(j + R1 * u) * Kh + l] = a[u];
    }
}

// ------------------------------------------ z transform + influence -------
// A workgroup takes NP = 2^lnp consecutive (y, kx) positions of the flat
// half-plane index j = y (K/2+1) + kx (so every z plane is read in runs of
// NP) for one right-hand side. Stage 1 goes from global memory to LDS; the
// second stage, the influence multiply and the first stage of the inverse
// transform (its radices in the opposite order) work on the same registers
// and write back in place; the inverse's last stage goes from LDS to global
// memory. Where the registers of all components' butterflies would exceed
// the budget (NC R2 complex values), the middle part is three steps through
// LDS, spread over the components (K = 256 FP64 poly: 2.05 ms for 18 meshes
// against 2.86 with one thread taking all components in turn). The line lies
// below 192 registers of values, where kernels run one or two waves per SIMD. us
// in registers / three steps: unequal radii, FP64 with R2 = 8, 20 columns, K =
// 64: 123 / 95, 72: 164 / 136, 80: 354 / 186, 96: 844 / 368, 128: 940 / 868; FP32
// with R2 = 16, 8 columns, K = 256: 3286 / 2877, 288: 3549 / 2625; equal radii,
// FP64 with R2 = 16, 8 columns, K = 256: 2275 / 2230, 288: 2290 / 2222, 320: 2971 /
// 2965.
// 256 threads where the middle is in registers: K = 128 FP32, 100 columns
// 1.15 ms against 1.56 with 384 (two workgroups fit then, and more waves
// wait at each barrier). Chunks in XCD order: 1.15 against 1.18 ms, FP64 2.20
// against 2.45.
template <typename T, int R2, int NC>
struct ZShape {
    static constexpr bool in_regs = NC * R2 * 2 * (int)sizeof(T) / 4 < 192;
    static constexpr int NT = in_regs ? 256 : 512;
};

template <typename T, int R1, int R2, int NC>
__global__ void __launch_bounds__((ZShape<T, R2, NC>::NT))
fft2_z_influence_kernel(cplx<T>* __restrict__ spec, const double* __restrict__ tw_g,
                        const double* __restrict__ fac_g, int lnp, double box, double xi) {
    typedef Fft2<R1, R2> F;
    constexpr int K = F::K, Kh = F::Kh, nj = K * Kh;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    const int NP = 1 << lnp;
    cplx<T>* tw = reinterpret_cast<cplx<T>*>(smem_raw);
    cplx<T>* buf = tw + F::TWN;
    T* s_fac = reinterpret_cast<T*>(buf + (size_t)NC * NP * F::PSA);
    const int nch = (nj + NP - 1) >> lnp;
    // neighbouring chunks share cache lines where the runs are shorter than
    // one or the planes not whole lines: keep them on one XCD
    const unsigned lid = xcd_logical_id(blockIdx.x, gridDim.x);
    const int j0 = (int)(lid % nch) << lnp;
    const size_t mesh_sz = (size_t)nj * K;
    cplx<T>* base = spec + (size_t)(lid / nch) * NC * mesh_sz + j0;
    const int nv = min(NP, nj - j0);
    // lanes past the half plane's end repeat its last position
    auto load1 = [&](int it, cplx<T>* a) __attribute__((always_inline)) {
        const int l = min(it & (NP - 1), nv - 1), q = it >> lnp;
        const int c = q / R2, j = q % R2;
        const cplx<T>* s = base + (size_t)c * mesh_sz + (size_t)j * nj + l;
#pragma unroll
        for (int u = 0; u < R1; u++) a[u] = s[(size_t)(R2 * u) * nj];
    };
    const int nit = NC * NP * R2;
    {
        Twiddles<T, R1, R2, 2> t;
        t.fetch(tw_g);
        double f[2];
#pragma unroll
        for (int c = 0; c < 2; c++)
            f[c] = fac_g[min((int)(threadIdx.x + c * blockDim.x), K - 1)];
        cplx<T> a[R1];
        int it = threadIdx.x;
        if (it < nit) load1(it, a);
        t.store(tw, tw_g);
#pragma unroll
        for (int c = 0; c < 2; c++) {
            const int i = threadIdx.x + c * blockDim.x;
            if (i < K) s_fac[i] = (T)f[c];
        }
        for (int i = threadIdx.x + 2 * blockDim.x; i < K; i += blockDim.x) s_fac[i] = (T)fac_g[i];
        __syncthreads();
        while (it < nit) {
            const int l = it & (NP - 1), q = it >> lnp;
            const int c = q / R2, j = q % R2;
            small_dft<T, R1, -1>(a);
#pragma unroll
            for (int u = 1; u < R1; u++) a[u] = cmul(a[u], tw[j * F::RA + u]);
            cplx<T>* o = buf + (c * NP + l) * F::PSA + j * F::RA;
#pragma unroll
            for (int u = 0; u < R1; u++) o[u] = a[u];
            it += blockDim.x;
            if (it < nit) load1(it, a);
        }
    }
    __syncthreads();
    const Influence<T> inf(box, xi);
    const int cs = NP * F::PSA;    // component stride in LDS
    if constexpr (ZShape<T, R2, NC>::in_regs) {
        for (int it = threadIdx.x; it < NP * R1; it += blockDim.x) {
            const int l = it & (NP - 1), j = it >> lnp;
            if (l >= nv) continue;
            const int y = (j0 + l) / Kh, kxi = (j0 + l) % Kh;
            const int my = y <= K / 2 ? y : y - K;
            const T fxy = s_fac[kxi] * s_fac[y];
            cplx<T>* o = buf + l * F::PSA + j;
            cplx<T> a[NC][R2];
#pragma unroll
            for (int c = 0; c < NC; c++) {
#pragma unroll
                for (int u = 0; u < R2; u++) a[c][u] = o[c * cs + u * F::RA];
                small_dft<T, R2, -1>(a[c]);
            }
#pragma unroll
            for (int u = 0; u < R2; u++) {
                const int z = j + R1 * u;
                cplx<T> g[NC];
#pragma unroll
                for (int c = 0; c < NC; c++) g[c] = a[c][u];
                inf.template apply<NC>(kxi, my, z <= K / 2 ? z : z - K, fxy * s_fac[z], g);
#pragma unroll
                for (int c = 0; c < NC; c++) a[c][u] = g[c];
            }
#pragma unroll
            for (int c = 0; c < NC; c++) {
                small_dft<T, R2, +1>(a[c]);
                o[c * cs] = a[c][0];
#pragma unroll
                for (int u = 1; u < R2; u++)
                    o[c * cs + u * F::RA] = cmulc(a[c][u], tw[u * F::RA + j]);
            }
        }
    } else {
        for (int it = threadIdx.x; it < NC * NP * R1; it += blockDim.x) {
            const int l = it & (NP - 1), q = it >> lnp;
            if (l >= nv) continue;
            cplx<T>* o = buf + ((q / R1) * NP + l) * F::PSA + q % R1;
            cplx<T> a[R2];
#pragma unroll
            for (int u = 0; u < R2; u++) a[u] = o[u * F::RA];
            small_dft<T, R2, -1>(a);
#pragma unroll
            for (int u = 0; u < R2; u++) o[u * F::RA] = a[u];
        }
        __syncthreads();
        for (int it = threadIdx.x; it < NP * K; it += blockDim.x) {
            const int l = it & (NP - 1), z = it >> lnp;
            if (l >= nv) continue;
            const int y = (j0 + l) / Kh, kxi = (j0 + l) % Kh;
            cplx<T>* o = buf + l * F::PSA + F::posa(z);
            cplx<T> g[NC];
#pragma unroll
            for (int c = 0; c < NC; c++) g[c] = o[c * cs];
            inf.template apply<NC>(kxi, y <= K / 2 ? y : y - K, z <= K / 2 ? z : z - K,
                                   s_fac[kxi] * s_fac[y] * s_fac[z], g);
#pragma unroll
            for (int c = 0; c < NC; c++) o[c * cs] = g[c];
        }
        __syncthreads();
        for (int it = threadIdx.x; it < NC * NP * R1; it += blockDim.x) {
            const int l = it & (NP - 1), q = it >> lnp;
            if (l >= nv) continue;
            const int j = q % R1;
            cplx<T>* o = buf + ((q / R1) * NP + l) * F::PSA + j;
            cplx<T> a[R2];
#pragma unroll
            for (int u = 0; u < R2; u++) a[u] = o[u * F::RA];
            small_dft<T, R2, +1>(a);
            o[0] = a[0];
#pragma unroll
            for (int u = 1; u < R2; u++) o[u * F::RA] = cmulc(a[u], tw[u * F::RA + j]);
        }
    }
    __syncthreads();
    for (int it = threadIdx.x; it < NC * NP * R2; it += blockDim.x) {
        const int l = it & (NP - 1), q = it >> lnp;
        const int c = q / R2, j = q % R2;
        if (l >= nv) continue;
        const cplx<T>* o = buf + (c * NP + l) * F::PSA + j * F::RA;
        cplx<T> a[R1];
#pragma unroll
        for (int u = 0; u < R1; u++) a[u] = o[u];
        small_dft<T, R1, +1>(a);
        cplx<T>* s = base + (size_t)c * mesh_sz + (size_t)j * nj + l;
#pragma unroll
        for (int u = 0; u < R1; u++) s[(size_t)(R2 * u) * nj] = a[u];
    }
}

// ------------------------------------------------------------ dispatch -----
// Mesh sides with a two-stage kernel: K, R1 >= R2 with K = R1 R2 (every even
// 2^a 3^b 5^c from 16 to 324 except 250 = 2 5^3)
#define SDT_FFT2_SIDES(X)                                                                     \
    X(16, 4, 4) X(18, 6, 3) X(20, 5, 4) X(24, 6, 4) X(30, 6, 5) X(32, 8, 4) X(36, 6, 6)       \
    X(40, 8, 5) X(48, 8, 6) X(50, 10, 5) X(54, 9, 6) X(60, 10, 6) X(64, 8, 8) X(72, 9, 8)     \
    X(80, 10, 8) X(90, 10, 9) X(96, 12, 8) X(100, 10, 10) X(108, 12, 9) X(120, 12, 10)        \
    X(128, 16, 8) X(144, 16, 9) X(150, 15, 10) X(160, 16, 10) X(162, 18, 9) X(180, 18, 10)    \
    X(192, 16, 12) X(200, 20, 10) X(216, 18, 12) X(240, 16, 15) X(256, 16, 16)                \
    X(270, 18, 15) X(288, 18, 16) X(300, 20, 15) X(320, 20, 16) X(324, 18, 18)

// one workgroup's LDS on gfx950
constexpr size_t kMaxLds = 160 * 1024;

template <typename T>
bool Fft2Launch<T>::has(int K) {
    switch (K) {
#define X(KK, A, B) case KK:
        SDT_FFT2_SIDES(X)
#undef X
        return true;
    }
    return false;
}

template <typename T>
bool Fft2Launch<T>::plane_fits(int K) {
    switch (K) {
#define X(KK, A, B) case KK: return PlaneShape<T, A, B>::lds_fwd <= kMaxLds;
        SDT_FFT2_SIDES(X)
#undef X
    }
    return false;
}

template <typename T, int R1, int R2>
static void launch_plane(bool fwd, int nmesh, T* real, cplx<T>* spec, const double* tw,
                         hipStream_t s) {
    typedef PlaneShape<T, R1, R2> S;
    if constexpr (S::lds_fwd <= kMaxLds) {
        const dim3 grid((unsigned)(nmesh * R1 * R2));
        if (fwd) {
            allow_lds((const void*)fft2_plane_fwd_kernel<T, R1, R2>, S::lds_fwd);
            hipLaunchKernelGGL((fft2_plane_fwd_kernel<T, R1, R2>), grid, dim3(S::NT), S::lds_fwd, s,
                               real, spec, tw);
        } else {
            allow_lds((const void*)fft2_plane_inv_kernel<T, R1, R2>, S::lds_inv);
            hipLaunchKernelGGL((fft2_plane_inv_kernel<T, R1, R2>), grid, dim3(S::NT), S::lds_inv, s,
                               spec, real, tw);
        }
    }
}

template <typename T>
void Fft2Launch<T>::plane(int K, bool fwd, int nmesh, T* real, cplx<T>* spec, const double* tw,
                          hipStream_t s) {
    switch (K) {
#define X(KK, A, B) case KK: launch_plane<T, A, B>(fwd, nmesh, real, spec, tw, s); break;
        SDT_FFT2_SIDES(X)
#undef X
    }
    SDT_HIP_CHECK(hipGetLastError());
}

// the separate passes serve the sides from 128 up (below, a plane always fits)
template <typename T>
bool Fft2Launch<T>::has_xy(int K) { return K >= 128 && has(K); }

template <typename T, int R1, int R2>
static void launch_xy(bool fwd, int nmesh, T* real, cplx<T>* spec, const double* tw,
                      hipStream_t s) {
    typedef Fft2<R1, R2> F;
    if constexpr (F::K >= 128) {
        // pencils per workgroup: 16 (FP32) or 8 (FP64), runs of 128 bytes in
        // the y pass, 40 KB or less
        constexpr int lnp = sizeof(T) == 4 ? 4 : 3, NP = 1 << lnp;
        const size_t lds_a = (size_t)(F::TWN + NP * F::PSA) * sizeof(cplx<T>);
        const size_t lds_b = (size_t)(F::TWN + NP * F::PSB) * sizeof(cplx<T>);
        const long long npair = (long long)nmesh * F::K * F::H;
        const dim3 gx((unsigned)((npair + NP - 1) / NP));
        const dim3 gy((unsigned)((F::Kh + NP - 1) / NP * (long long)nmesh * F::K));
        if (fwd) {
            allow_lds((const void*)fft2_x_r2c_kernel<T, R1, R2>, lds_b);
            hipLaunchKernelGGL((fft2_x_r2c_kernel<T, R1, R2>), gx, dim3(kXYThreads), lds_b, s, npair,
                               real, spec, tw, NP);
            allow_lds((const void*)fft2_y_kernel<T, R1, R2, -1>, lds_a);
            hipLaunchKernelGGL((fft2_y_kernel<T, R1, R2, -1>), gy, dim3(kXYThreads), lds_a, s, spec,
                               tw, lnp);
        } else {
            allow_lds((const void*)fft2_y_kernel<T, R1, R2, +1>, lds_a);
            hipLaunchKernelGGL((fft2_y_kernel<T, R1, R2, +1>), gy, dim3(kXYThreads), lds_a, s, spec,
                               tw, lnp);
            allow_lds((const void*)fft2_x_c2r_kernel<T, R1, R2>, lds_a);
            hipLaunchKernelGGL((fft2_x_c2r_kernel<T, R1, R2>), gx, dim3(kXYThreads), lds_a, s, npair,
                               spec, real, tw, NP);
        }
    }
}

template <typename T>
void Fft2Launch<T>::xy(int K, bool fwd, int nmesh, T* real, cplx<T>* spec, const double* tw,
                       hipStream_t s) {
    switch (K) {
#define X(KK, A, B) case KK: launch_xy<T, A, B>(fwd, nmesh, real, spec, tw, s); break;
        SDT_FFT2_SIDES(X)
#undef X
    }
    SDT_HIP_CHECK(hipGetLastError());
}

template <typename T, int R1, int R2, int NC>
static void launch_z(int b, cplx<T>* spec, const double* tw, const double* fac, int ntmax,
                     int lnpmax, double box, double xi, hipStream_t s) {
    typedef Fft2<R1, R2> F;
    constexpr int nj = F::K * F::Kh;
    auto lds_of = [&](int l) {
        return ((size_t)F::TWN + ((size_t)NC << l) * F::PSA) * sizeof(cplx<T>) +
               F::K * sizeof(T);
    };
    int lnp = lnpmax;
    // at least two workgroups per CU by LDS, and a grid of four per CU
    while (lnp > 2 && (lds_of(lnp) > kMaxLds / 2 ||
                       (size_t)b * ((nj + (1 << lnp) - 1) >> lnp) < 1024))
        lnp--;
    while (lnp > 0 && lds_of(lnp) > kMaxLds) lnp--;
    const int items = (NC << lnp) * R2;
    const int nt = std::min({ntmax, ZShape<T, R2, NC>::NT, (items + 63) / 64 * 64});
    const size_t lds = lds_of(lnp);
    const dim3 grid((unsigned)(((nj + (1 << lnp) - 1) >> lnp) * (size_t)b));
    allow_lds((const void*)fft2_z_influence_kernel<T, R1, R2, NC>, lds);
    hipLaunchKernelGGL((fft2_z_influence_kernel<T, R1, R2, NC>), grid, dim3(nt), lds, s, spec, tw,
                       fac, lnp, box, xi);
}

template <typename T>
void Fft2Launch<T>::z(int K, int NC, int b, cplx<T>* spec, const double* tw, const double* fac,
                      int ntmax, int lnpmax, double box, double xi, hipStream_t s) {
    switch (K) {
#define X(KK, A, B)                                                                           \
    case KK:                                                                                  \
        if (NC == 3) launch_z<T, A, B, 3>(b, spec, tw, fac, ntmax, lnpmax, box, xi, s);       \
        else launch_z<T, A, B, 6>(b, spec, tw, fac, ntmax, lnpmax, box, xi, s);               \
        break;
        SDT_FFT2_SIDES(X)
#undef X
    }
    SDT_HIP_CHECK(hipGetLastError());
}

}  // namespace sdt
