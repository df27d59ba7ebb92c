// SPME reciprocal-space kernels for gfx950 (FP32 and FP64 instantiations).
//
// Reference algorithm: src/mob/spme.cc (UpdateSpmeEngine_ :366-509, Spread
// :313-363, ApplyInfluence :201-310, Interpolate :163-198, ComputeSpline
// :71-160, ComputeSpmeRecip_ :714-839). The GPU form keeps 3 p weights per
// particle or its fractional offsets instead of the N x p^3 P/ind tables,
// fuses all b right-hand sides into each launch, spreads by mesh blocks that
// sum their own points on the matrix cores (plain stores, no global atomics,
// no zero-fill pass), and fuses the influence multiply between the forward
// and inverse z-transforms.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <map>
#include <mutex>
#include <type_traits>
#include "fft_lds.hpp"
#include "spme_fft.hpp"
#include "real_gpu.hpp"
#include "spme_gpu.hpp"

namespace sdt {

// ----------------------------------------------------------- B-splines -----
// w[x] = M_P(x + 1 - frac), x = 0..P-1, by raising the order of
// a[k] = M_n(u + k), u = 1 - frac, from n = 1 to P (Cox-de Boor). Same values
// as BSpline(P, floor(c) - c + x) in src/mob/spme.cc:38-68,469-473.
template <typename T, int P>
__device__ __forceinline__ void bspline_weights(T frac, T* w) {
    const T u = T(1) - frac;
    w[0] = T(1);
#pragma unroll
    for (int k = 1; k < P; k++) w[k] = T(0);
#pragma unroll
    for (int n = 2; n <= P; n++) {
        const T inv = T(1) / T(n - 1);
#pragma unroll
        for (int k = n - 1; k >= 1; k--)
            w[k] = ((u + T(k)) * w[k] + (T(n) - u - T(k)) * w[k - 1]) * inv;
        w[0] = u * w[0] * inv;
    }
}

// the weights from the FP64 fractional offset, evaluated in FP64 and rounded
// to the arithmetic type once (FP32 weights carry no error from the offset)
template <typename T, int P>
__device__ __forceinline__ void bspline_weights_r(double frac, T* w) {
    double wd[P];
    bspline_weights<double, P>(frac, wd);
#pragma unroll
    for (int k = 0; k < P; k++) w[k] = (T)wd[k];
}

// ------------------------------------------------------------ prepare ------
// Wrap into [0, L) (pair-list convention, src/pairlist/pair_base.cc:94-99),
// scaled coordinate c = x / L * K, base index as src/mob/spme.cc:419-443.
template <typename T, int P>
__global__ void spme_prepare_kernel(int npos, const double* __restrict__ pos, double box, int K,
                                    int ts, int ntile, double* __restrict__ frac_u,
                                    int* __restrict__ base_u, int* __restrict__ key) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= npos) return;
    int t[3];
#pragma unroll
    for (int d = 0; d < 3; d++) {
        double x = fmod(pos[3 * i + d], box);
        x = (x >= 0.0 ? x : box + x);
        double c = x / box * K;
        double g = floor(c);
        int b0 = (P % 2 == 0) ? (int)(g - P / 2 + 1) : (int)(g - (P - 1) / 2);
        int b = ((b0 % K) + K) % K;
        frac_u[3 * i + d] = c - g;
        base_u[3 * i + d] = b;
        int tt = b / ts;
        t[d] = tt < ntile ? tt : ntile - 1;
    }
    key[i] = (t[2] * ntile + t[1]) * ntile + t[0];
}

// One particle's stencil record, made once per update and read by every
// spread and by the interpolation from blocks of tiles: the base index (3 ints
// in one 16-byte slot), then
// the 1D weights 0 0 0 wx[P] 0 0 0 wy[P] 0 0 0 wz[P] 0 0 0, padded to 16
// bytes. The zeros are the weights of the points up to 3 outside a stencil, so
// that 4 points of a mesh block read theirs without a range test. (The strip
// interpolation makes its weights from the offsets again: a record's bytes per
// group of 4 columns cost that kernel more, 3.56 against 3.19 ms for 100 FP64
// columns at K = 128.)
template <typename T, int P>
struct Sten {
    static constexpr int V = 16 / (int)sizeof(T);    // values per 16 bytes
    static constexpr int RUN = P + 3;                // from one run to the next
    static constexpr int OW = V + 3;                 // wx[0]
    static constexpr int N = (V + 3 * RUN + 3 + V - 1) / V * V;
};

template <typename T, int P>
__global__ void spme_gather_kernel(int npos, const int* __restrict__ perm,
                                   const double* __restrict__ frac_u, const int* __restrict__ base_u,
                                   const double* __restrict__ rdi, T* __restrict__ sten,
                                   double* __restrict__ frac, int* __restrict__ base,
                                   double* __restrict__ a2,
                                   unsigned long long* __restrict__ nids) {
    typedef Sten<T, P> St;
    const int is = blockIdx.x * blockDim.x + threadIdx.x;
    if (is == 0) *nids = 0;   // for spread_list_kernel, next on the stream
    if (is >= npos) return;
    const int i = perm[is];
    T* rec = sten + (size_t)is * St::N;
    int* rb = reinterpret_cast<int*>(rec);
#pragma unroll
    for (int d = 0; d < 3; d++) {
        const int b = base_u[3 * i + d];
        base[3 * is + d] = b;
        rb[d] = b;
        const double fr = frac_u[3 * i + d];
        frac[3 * is + d] = fr;
        T w[P];
        bspline_weights_r<T, P>(fr, w);
#pragma unroll
        for (int k = 0; k < P; k++) rec[St::OW + d * St::RUN + k] = w[k];
#pragma unroll
        for (int k = 1; k <= 3; k++) rec[St::OW + d * St::RUN - k] = T(0);
    }
#pragma unroll
    for (int k = St::V + 3 * St::RUN; k < St::N; k++) rec[k] = T(0);
    if (a2) a2[is] = rdi[i] * rdi[i];
}

// ------------------------------------------------------------- spread ------
__device__ __forceinline__ int wrapk(int d, int K) {
    d += (d < 0) ? K : 0;
    return d - ((d >= K) ? K : 0);
}

// Point-owner form: a workgroup of 8 waves owns a 32 x 4 x 4 block of mesh
// points (wave w: x in [4w, 4w+4); the last block of a dimension is partial, K
// is even: 2 points of 4). The block's candidates (particles whose stencil
// reaches it, spread_list_kernel) are staged in LDS in list order, stencil
// record and forces; every wave lists the candidates that reach its 4 x 4 x 4
// sub-block and adds w = wx[x - bx] wy[y - by] wz[z - bz] (0 outside the
// stencil) times their forces. Deterministic, no atomics.
constexpr int kPtThreads = 512;

// The candidates of every 32 x 4 x 4 mesh block, listed once per update: one
// wave per block goes through the particles of the tiles its window touches
// (the tiles of a row along x are one range of the sorted order, two where
// they wrap) and keeps those whose stencil reaches the block, in that order.
// blk[block] is its segment of ids; the offsets come from an atomic counter, so
// segments lie in any order, but each one's content is fixed. They have 64
// bits: a stencil reaches up to 18 blocks.
// Finding the candidates inside every spread took a third of its 89 us for one
// column at K = 128, N = 100 000 (62 us from the lists).
constexpr int kListWaves = 16;
constexpr int kListRanges = 64;   // ranges of one block (host-checked)
constexpr int kListMasks = 32;    // candidate groups whose test is kept for the second pass

template <int P>
__global__ void __launch_bounds__(64 * kListWaves)
spread_list_kernel(int K, int ts, int ntile, int nsx, int nblocks,
                   const int* __restrict__ tile_start, const int* __restrict__ base,
                   unsigned long long* __restrict__ nids, SpreadSeg* __restrict__ blk,
                   int* __restrict__ ids) {
    __shared__ int s_off_[kListWaves][kListRanges], s_beg_[kListWaves][kListRanges];
    __shared__ unsigned long long s_mask_[kListWaves][kListMasks];
    __shared__ int s_tot[kListWaves];
    __shared__ long long s_base;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    // waves past the last block repeat it and keep nothing
    const bool real = blockIdx.x * kListWaves + wave < nblocks;
    const int bl = min((int)(blockIdx.x * kListWaves + wave), nblocks - 1);
    int* s_off = s_off_[wave];
    int* s_beg = s_beg_[wave];
    unsigned long long* s_mask = s_mask_[wave];
    const int K4 = (K + 3) >> 2;
    const int yz = bl / nsx;
    const int org[3] = {(bl % nsx) * 32, (yz % K4) * 4, (yz / K4) * 4};
    const int ext[3] = {min(32, K - org[0]), min(4, K - org[1]), min(4, K - org[2])};
    // base tiles of the window [org - (P - 1), org + ext) in each dimension
    int first[3], cnt[3];
#pragma unroll
    for (int d = 0; d < 3; d++) {
        const int lo = org[d] - (P - 1), len = ext[d] + P - 1;
        if (len >= K) { first[d] = 0; cnt[d] = ntile; continue; }
        const int a = (lo >= 0) ? lo / ts : -((-lo + ts - 1) / ts);
        const int e = lo + len - 1;              // >= 0
        cnt[d] = min(e / ts - a + 1, ntile);
        first[d] = ((a % ntile) + ntile) % ntile;
    }
    const int nr = 2 * cnt[1] * cnt[2];
    int pb = 0, n = 0;
    if (lane < nr) {
        const int row = lane >> 1;
        const int ty = (first[1] + row % cnt[1]) % ntile, tz = (first[2] + row / cnt[1]) % ntile;
        const int n1 = min(cnt[0], ntile - first[0]);    // tiles before the wrap
        const int t0 = (tz * ntile + ty) * ntile + ((lane & 1) ? 0 : first[0]);
        const int nt = (lane & 1) ? cnt[0] - n1 : n1;
        pb = tile_start[t0];
        n = tile_start[t0 + nt] - pb;
    }
    int inc = n;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int t = __shfl_up(inc, o);
        if (lane >= o) inc += t;
    }
    s_off[lane] = inc - n;
    s_beg[lane] = pb;
    const int ncand = __shfl(inc, 63);
    // the LDS tables are this wave's own (its accesses complete in order)
    __builtin_amdgcn_wave_barrier();
    // particle of candidate ci: the last range whose offset is <= ci
    auto particle = [&](int ci) __attribute__((always_inline)) {
        int k = 0, hi = nr - 1;
        while (k < hi) {
            const int mid = (k + hi + 1) >> 1;
            if (s_off[mid] <= ci) k = mid;
            else hi = mid - 1;
        }
        return s_beg[k] + (ci - s_off[k]);
    };
    auto reaches = [&](const int* b3) __attribute__((always_inline)) {
        bool take = true;
#pragma unroll
        for (int d = 0; d < 3; d++) {
            const int r = wrapk(b3[d] - org[d], K);
            take = take && (r < ext[d] || K - r < P);
        }
        return take;
    };
    // U groups of 64 at a time, their loads in flight together
    constexpr int U = 4;
    int total = 0;
    for (int c0 = 0, g = 0; c0 < ncand; c0 += 64 * U, g += U) {
        int b3[U][3];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int is = particle(min(c0 + 64 * u + lane, ncand - 1));
#pragma unroll
            for (int d = 0; d < 3; d++) b3[u][d] = base[3 * is + d];
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            const unsigned long long m = __ballot(c0 + 64 * u + lane < ncand && reaches(b3[u]));
            if (lane == 0 && g + u < kListMasks) s_mask[g + u] = m;
            total += __popcll(m);
        }
    }
    // one atomic a workgroup: same-address atomics of every wave took 35 us
    if (!real) total = 0;
    if (lane == 0) s_tot[wave] = total;
    __syncthreads();
    if (threadIdx.x == 0) {
        int sum = 0;
        for (int w = 0; w < kListWaves; w++) {
            const int t = s_tot[w];
            s_tot[w] = sum;
            sum += t;
        }
        s_base = sum > 0 ? (long long)atomicAdd(nids, (unsigned long long)sum) : 0;
    }
    __syncthreads();
    if (!real) return;
    long long off = s_base + s_tot[wave];
    if (lane == 0) blk[bl] = SpreadSeg{off, total};
    for (int c0 = 0, g = 0; c0 < ncand; c0 += 64, g++) {
        const int ci = c0 + lane;
        const int is = particle(min(ci, ncand - 1));
        const unsigned long long m =
            g < kListMasks ? s_mask[g] : __ballot(ci < ncand && reaches(base + 3 * is));
        if ((m >> lane) & 1) ids[off + __popcll(m & ((1ull << lane) - 1ull))] = is;
        off += __popcll(m);
    }
}


// The sums run on the matrix cores (v_mfma_*_16x16x4): a wave's sub-block is
// the product W F of its 64 points x listed candidates weight matrix and the
// candidates' forces, 4 candidates at a time; m-tile m = the 16 points of z
// plane m (row i = 4 y + x), NT n-tiles of 16 force values. Each lane forms
// its A entry (point l % 16, candidate l / 16) from the staged 1D weights, so
// no lane is spent on points outside a stencil. The matrix cores add the 4
// products of a step in candidate order with one rounding each, so the sums
// are those of the vector form below to the bit.
//
// BLK (wide launches): the forces come from a column-blocked copy
// Xb[cb][j][c][r] of the packed input (NQ / 3 columns per block, arithmetic
// type T; with unequal radii the columns are f and a^2 f of every right-hand
// side in turn), so a candidate's NQ values are one contiguous run; value q
// belongs to component q / (NQ / 3) of column q % (NQ / 3). FP32: 48 values, 3
// n-tiles. FP64: 24 values, 2 n-tiles (8 slots of the second idle). A
// workgroup takes ncbw column blocks of its mesh block in turn. When all its
// candidates fit the stage they are staged and listed once; each further
// column block then only loads the candidates' forces before its sums and
// stores.
// Otherwise (at most 16 meshes): the forces of mesh q = NC r + c are read from
// the packed input, NQ = 4 or 16 slots, one n-tile.
//
// The meshes leave through LDS tiles after the stage (16 force values x 4 rows
// x 32 points of one z plane at a time; 4 values x 4 planes for NQ = 4; rows
// padded so that the waves' pieces land in distinct banks): every store
// instruction then writes whole rows of the block. Stores of 16-byte pieces
// per lane reached HBM 1.4 times. FP32 uses two tiles in turn, one barrier a
// round; FP64 one, to fit two workgroups per CU.
//
// Measured (with the candidates found and their weights made in every launch
// and the vector ALUs for narrow and FP64 launches -> now): one FP32 column,
// K = 128, N = 100 000: 96 -> 62 us (30 M wave instructions bounded it); 16
// columns 210 -> 180 us, 100 columns 1.06 -> 1.01 ms (the meshes alone take
// 0.5 ms to write); 8 columns, K = 216, N = 200 000: 620 -> 440 us; FP64, 100
// columns, K = 128: 3.2 -> 2.7 ms, 16 columns, K = 90: 144 -> 114 us.
constexpr int kTileRow = 132;    // values per force value and plane in a tile

template <typename T, int NQ>
struct SpreadTile {
    static constexpr int cols = NQ < 16 ? NQ : 16;      // force values of a round
    static constexpr int planes = NQ == 4 ? 4 : 1;      // z planes of a round
    static constexpr int bufs = sizeof(T) == 4 && planes == 1 ? 2 : 1;
    static constexpr size_t bytes = (size_t)bufs * planes * cols * kTileRow * sizeof(T);
};

// values per staged candidate: record, forces, and a pad that makes it an odd
// number of 16-byte slots (lanes reading consecutive candidates' bases then
// spread over the banks)
template <typename T>
__host__ __device__ constexpr int spread_slot(int sten_n, int nq) {
    constexpr int V = 16 / (int)sizeof(T);
    return ((sten_n + nq) / V | 1) * V;
}
// and its LDS bytes, with the eight waves' lists and the particle id
template <typename T>
static size_t spread_slot_bytes(int sten_n, int nq) {
    return (size_t)spread_slot<T>(sten_n, nq) * sizeof(T) + 8 * sizeof(unsigned) + sizeof(int);
}

typedef float f4v __attribute__((ext_vector_type(4)));
typedef double d4v __attribute__((ext_vector_type(4)));
__device__ __forceinline__ f4v mfma16(float a, float b, f4v c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ d4v mfma16(double a, double b, d4v c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// stages candidates list_g[0 .. n) of a block: their records with the base
// relative to the block origin (in (-P, K - P]), with NV > 0 followed by 16 NV
// bytes of blocked forces each; 16 bytes per load, the loads of a thread in
// flight together
template <typename T, int P, int NV>
__device__ __forceinline__ void spread_stage(int n, const int* __restrict__ list_g,
                                             const T* __restrict__ sten,
                                             const T* __restrict__ frc, const int* org, int K,
                                             int rec_n, T* stage, int* s_pid) {
    typedef Sten<T, P> St;
    typedef T VT __attribute__((ext_vector_type(16 / sizeof(T))));
    typedef int I4 __attribute__((ext_vector_type(4)));
    constexpr int HV = St::N / St::V, SV = HV + NV, U = NV > 0 ? 4 : 2;
    const VT* rec_g = reinterpret_cast<const VT*>(sten);
    const VT* frc_g = reinterpret_cast<const VT*>(frc);
    for (int e0 = threadIdx.x; e0 < n * SV; e0 += kPtThreads * U) {
        VT v[U];
        int pid[U];
#pragma unroll
        for (int u = 0; u < U; u++) pid[u] = list_g[min(e0 + u * kPtThreads, n * SV - 1) / SV];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int e = min(e0 + u * kPtThreads, n * SV - 1), q = e - (e / SV) * SV;
            v[u] = NV == 0 || q < HV ? rec_g[(size_t)pid[u] * HV + q]
                                     : frc_g[(size_t)pid[u] * NV + (q - HV)];
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int e = e0 + u * kPtThreads;
            if (e >= n * SV) continue;
            const int sl = e / SV, q = e - sl * SV;
            if (q == 0) {
                s_pid[sl] = pid[u];
                I4 b3 = *reinterpret_cast<I4*>(&v[u]);
#pragma unroll
                for (int d = 0; d < 3; d++) {
                    const int r = wrapk(b3[d] - org[d], K);
                    b3[d] = r > K - P ? r - K : r;
                }
                v[u] = *reinterpret_cast<VT*>(&b3);
            }
            *reinterpret_cast<VT*>(stage + (size_t)sl * rec_n + q * St::V) = v[u];
        }
    }
}

// the blocked forces of the staged candidates for another column block
template <typename T, int NQ>
__device__ __forceinline__ void spread_restage(int n, const int* s_pid, const T* __restrict__ frc,
                                               int rec_n, T* out) {
    typedef T VT __attribute__((ext_vector_type(16 / sizeof(T))));
    constexpr int V = 16 / (int)sizeof(T), NV = NQ / V, U = 4;
    const VT* src = reinterpret_cast<const VT*>(frc);
    for (int e0 = threadIdx.x; e0 < n * NV; e0 += kPtThreads * U) {
        VT v[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int e = min(e0 + u * kPtThreads, n * NV - 1);
            v[u] = src[(size_t)s_pid[e / NV] * NV + e % NV];
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int e = e0 + u * kPtThreads;
            if (e < n * NV)
                *reinterpret_cast<VT*>(out + (size_t)(e / NV) * rec_n + e % NV * V) = v[u];
        }
    }
}

// forces of the staged candidates from the packed input: slot q holds mesh
// q0 + q, mesh NC r + c the component c % 3 of right-hand side r, times a^2
// for c >= 3; zero beyond the last mesh. A thread serves one slot.
template <typename T, int NQ>
__device__ __forceinline__ void spread_stage_packed(int n, const int* s_pid,
                                                    const double* __restrict__ X,
                                                    const double* __restrict__ a2, int b, int NC,
                                                    int q0, int rec_n, T* frc) {
    static_assert(kPtThreads % NQ == 0, "one slot per thread");
    constexpr int U = 2, S = kPtThreads / NQ;
    const int q = threadIdx.x % NQ, r = (q0 + q) / NC, c = (q0 + q) - r * NC;
    const bool on = r < b, scaled = c >= 3;
    const double* x = X + (size_t)(c % 3) * b + r;
    for (int i0 = threadIdx.x / NQ; i0 < n; i0 += U * S) {
        double v[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            v[u] = 0.0;
            if (on && i0 + u * S < n) {
                const int p = s_pid[i0 + u * S];
                v[u] = x[(size_t)(3 * p) * b];
                if (scaled) v[u] *= a2[p];
            }
        }
#pragma unroll
        for (int u = 0; u < U; u++)
            if (i0 + u * S < n) frc[(size_t)(i0 + u * S) * rec_n + q] = (T)v[u];
    }
}

// lists the staged candidates (n of them) whose stencil reaches this wave's
// 4 x 4 x 4 sub-block; returns their number. An entry holds the record's value
// index (16 bits: the stage has fewer than 2^16 values) and the base relative
// to the sub-block, in (-P, 4) (K >= 16 > P + 3: one offset only), so that the
// sums need no second look at the record's base. The list is written and read
// by this wave only (LDS accesses of a wave complete in order).
template <typename T, int P>
__device__ __forceinline__ int spread_hits(int n, const T* stage, int rec_n, int K, int wave,
                                           int lane, unsigned* list) {
    int cnt = 0;
    for (int c0 = 0; c0 < n; c0 += 64) {
        const int c = c0 + lane;
        bool hit = c < n;
        unsigned entry = (unsigned)(c * rec_n);
        if (hit) {
            const int* rl = reinterpret_cast<const int*>(stage + c * rec_n);
#pragma unroll
            for (int d = 0; d < 3; d++) {
                int r = wrapk(rl[d] - (d == 0 ? 4 * wave : 0), K);
                r = r > K - P ? r - K : r;
                hit = hit && r < 4;
                entry |= (unsigned)(r + 8) << (16 + 4 * d);
            }
        }
        const unsigned long long m = __ballot(hit);
        if (hit) list[cnt + __popcll(m & ((1ull << lane) - 1ull))] = entry;
        cnt += __popcll(m);
    }
    __builtin_amdgcn_wave_barrier();
    return cnt;
}

// value index of a listed candidate's weight for coordinate x of the sub-block
// along dimension d (0 <= x < 4; a zero outside the stencil)
template <typename T, int P>
__device__ __forceinline__ int sten_at(int x, unsigned entry, int d) {
    typedef Sten<T, P> St;
    return (int)(entry & 0xffffu) + (St::OW + d * St::RUN + 8 + x) -
           (int)((entry >> (16 + 4 * d)) & 15u);
}

template <typename T, int P, int NQ, bool BLK>
__global__ void __launch_bounds__(kPtThreads) __attribute__((amdgpu_waves_per_eu(BLK ? 4 : (sizeof(T) == 4 ? 6 : 5))))
spread_mx_kernel(int K, int nsx, const SpreadSeg* __restrict__ blk, const int* __restrict__ ids,
                 const T* __restrict__ sten, const double* __restrict__ a2,
                 const double* __restrict__ X, const T* __restrict__ Xb, int npos, int b,
                 int ncbw, int NC, int cap, T* __restrict__ mesh) {
    typedef Sten<T, P> St;
    typedef SpreadTile<T, NQ> Tile;
    typedef T V4 __attribute__((ext_vector_type(4)));
    // four or two points of a mesh row: rows start on two values where K % 4 != 0
    typedef T V4m __attribute__((ext_vector_type(4), aligned(2 * sizeof(T))));
    typedef T V2m __attribute__((ext_vector_type(2), aligned(2 * sizeof(T))));
    constexpr int OF = St::N, REC = spread_slot<T>(OF, NQ), NT = (NQ + 15) / 16;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    T* stage = reinterpret_cast<T*>(smem_raw);
    int* s_pid = reinterpret_cast<int*>(stage + (size_t)cap * REC);            // [cap]
    unsigned* s_list = reinterpret_cast<unsigned*>(s_pid + cap);               // [8][cap]
    T* s_tile = reinterpret_cast<T*>(
        smem_raw + (((size_t)cap * (REC * sizeof(T) + 36) + 15) & ~(size_t)15));
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const unsigned lid = xcd_logical_id(blockIdx.x + blockIdx.y * gridDim.x, gridDim.x * gridDim.y);
    const int bxl = (int)(lid % gridDim.x), byl = (int)(lid / gridDim.x);
    const SpreadSeg seg = blk[bxl];
    const int ncand = seg.n;
    const int* __restrict__ list_g = ids + seg.off;
    const int K4 = (K + 3) >> 2;
    const int yz = bxl / nsx;
    const int org[3] = {(bxl % nsx) * 32, (yz % K4) * 4, (yz / K4) * 4};
    const int x0 = org[0], y0 = org[1], z0 = org[2];
    const int xlen = min(32, K - x0), ylen = min(4, K - y0), zlen = min(4, K - z0);
    const bool wave_on = 4 * wave < xlen;
    const size_t K3 = (size_t)K * K * K;
    V4 acc[4][NT];
    auto clear = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int m = 0; m < 4; m++)
#pragma unroll
            for (int t = 0; t < NT; t++) acc[m][t] = V4(T(0));
    };
    clear();
    // adds the first n staged candidates, listed anew or as they were
    int cnt = 0;
    auto accumulate = [&](int n, bool relist) __attribute__((always_inline)) {
        if (!wave_on) return;
        unsigned* list = s_list + wave * cap;
        if (relist) cnt = spread_hits<T, P>(n, stage, REC, K, wave, lane, list);
        if (cnt == 0) return;
        // A entry of lane l: point (x, y) = (l % 4, (l / 4) % 4) of the
        // sub-block, candidate l / 16 of the step (weight 0 past the list's
        // end); B entry: force value 16 t + l % 16 of the same candidate.
        const int kq = lane >> 4, jj = lane & 15, ax = lane & 3, ay = (lane >> 2) & 3;
        unsigned next = list[min(kq, cnt - 1)];
        for (int k0 = 0; k0 < cnt; k0 += 4) {
            const unsigned entry = next;
            next = list[min(k0 + 4 + kq, cnt - 1)];
            T wxy = stage[sten_at<T, P>(ax, entry, 0)] * stage[sten_at<T, P>(ay, entry, 1)];
            wxy = k0 + kq < cnt ? wxy : T(0);
            const T* wz = stage + sten_at<T, P>(0, entry, 2);
            const T* f = stage + (entry & 0xffffu) + OF + jj;
            T bf[NT];
#pragma unroll
            for (int t = 0; t < NT; t++)
                bf[t] = (NQ % 16 == 0 || 16 * t + jj < NQ) ? f[16 * t] : T(0);
#pragma unroll
            for (int m = 0; m < 4; m++) {
                const T a = wxy * wz[m];
#pragma unroll
                for (int t = 0; t < NT; t++) acc[m][t] = mfma16(a, bf[t], acc[m][t]);
            }
        }
    };
    constexpr int RBB = BLK ? NQ / 3 : 1;   // columns per block
    int cb = BLK ? byl * ncbw : 0;
    const int ncb = BLK ? min(cb + ncbw, (b + RBB - 1) / RBB) : 1;
    bool staged_all = false;   // the stage holds every candidate
    for (;;) {
        const T* frc = BLK ? Xb + (size_t)cb * npos * NQ : nullptr;
        constexpr int NV = BLK ? NQ / St::V : 0;
        for (int c0 = 0;; c0 += cap) {
            const int n = min(cap, ncand - c0);
            if (BLK && staged_all)
                spread_restage<T, NQ>(n, s_pid, frc, REC, stage + OF);
            else
                spread_stage<T, P, NV>(n, list_g + c0, sten, frc, org, K, REC, stage, s_pid);
            __syncthreads();
            if constexpr (!BLK) {
                spread_stage_packed<T, NQ>(n, s_pid, X, a2, b, NC, 0, REC, stage + OF);
                __syncthreads();
            }
            accumulate(n, !staged_all);
            if (c0 + cap >= ncand) break;
            __syncthreads();   // a full stage is summed and emptied
        }
        staged_all = ncand <= cap;
        // stores. FP32: result register v of lane l holds row 4 (l / 16) + v,
        // x = v and y = l / 16; FP64: row l / 16 + 4 v, x = l / 16 and y = v;
        // force value 16 t + l % 16 of z plane m
        const int jj = lane & 15, hi = lane >> 4;
        const int e = threadIdx.x;
        const int sx = (e & 7) * 4, sr = (e >> 3) & 3;
        const int sj = (e >> 5) % Tile::cols, sm = (e >> 5) / Tile::cols;
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int m0 = 0; m0 < 4; m0 += Tile::planes) {
                T* tb = s_tile + (Tile::bufs == 2 ? ((t * 4 + m0) & 1) : 0) *
                                     (Tile::planes * Tile::cols * kTileRow);
                if (wave_on && jj < Tile::cols) {
#pragma unroll
                    for (int m = m0; m < m0 + Tile::planes; m++) {
                        T* to = tb + ((m - m0) * Tile::cols + jj) * kTileRow + 4 * wave;
                        if constexpr (sizeof(T) == 4) {
                            *reinterpret_cast<V4*>(to + hi * 32) = acc[m][t];
                        } else {
#pragma unroll
                            for (int v = 0; v < 4; v++) to[v * 32 + hi] = acc[m][t][v];
                        }
                    }
                }
                __syncthreads();
                const int q = 16 * t + sj, m = m0 + sm;
                int mi;
                bool on;
                if constexpr (BLK) {
                    const int r = cb * RBB + q % RBB;
                    on = q < NQ && r < b;
                    mi = r * 3 + q / RBB;
                } else {
                    on = q < b * NC;
                    mi = q;
                }
                if (on && sm < Tile::planes && sx < xlen && sr < ylen && m < zlen) {
                    const V4 v = *reinterpret_cast<const V4*>(
                        tb + (sm * Tile::cols + sj) * kTileRow + sr * 32 + sx);
                    T* dst = mesh + (size_t)mi * K3 + ((size_t)(z0 + m) * K + (y0 + sr)) * K + x0 + sx;
                    if (sx + 4 <= xlen) *reinterpret_cast<V4m*>(dst) = v;
                    else *reinterpret_cast<V2m*>(dst) = V2m{v.x, v.y};
                }
                if (Tile::bufs == 1) __syncthreads();
            }
        if (++cb >= ncb) return;
        clear();
        // two tiles: a thread may be a round ahead, in the sums' LDS even more;
        // every wave is done with this column block's forces
        __syncthreads();
    }
}

// The same sums on the vector ALUs, kept as the comparison form: lane = point
// (x = l % 4, y = (l / 4) % 4, z = l / 16 of the wave's sub-block), kVecQ
// meshes in registers, one candidate at a time, forces from the packed input.
constexpr int kVecQ = 16;

template <typename T, int P>
__global__ void __launch_bounds__(kPtThreads)
spread_vec_kernel(int K, int nsx, const SpreadSeg* __restrict__ blk, const int* __restrict__ ids,
                  const T* __restrict__ sten, const double* __restrict__ a2,
                  const double* __restrict__ X, int b, int NC, int cap, T* __restrict__ mesh) {
    typedef Sten<T, P> St;
    constexpr int OF = St::N, REC = spread_slot<T>(OF, kVecQ);
    extern __shared__ __align__(16) unsigned char smem_raw[];
    T* stage = reinterpret_cast<T*>(smem_raw);
    int* s_pid = reinterpret_cast<int*>(stage + (size_t)cap * REC);
    unsigned* s_list = reinterpret_cast<unsigned*>(s_pid + cap);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int bxl = blockIdx.x, q0 = blockIdx.y * kVecQ;
    const SpreadSeg seg = blk[bxl];
    const int K4 = (K + 3) >> 2;
    const int yz = bxl / nsx;
    const int org[3] = {(bxl % nsx) * 32, (yz % K4) * 4, (yz / K4) * 4};
    const int lx = 4 * wave + (lane & 3), ly = (lane >> 2) & 3, lz = lane >> 4;
    T acc[kVecQ];
#pragma unroll
    for (int q = 0; q < kVecQ; q++) acc[q] = T(0);
    for (int c0 = 0; c0 < seg.n; c0 += cap) {
        const int n = min(cap, seg.n - c0);
        spread_stage<T, P, 0>(n, ids + seg.off + c0, sten, nullptr, org, K, REC, stage, s_pid);
        __syncthreads();
        spread_stage_packed<T, kVecQ>(n, s_pid, X, a2, b, NC, q0, REC, stage + OF);
        __syncthreads();
        // a wave past the mesh's end lists nothing: on sides below 28 its bases
        // would leave an entry's range
        unsigned* list = s_list + wave * cap;
        const int cnt = org[0] + 4 * wave < K ? spread_hits<T, P>(n, stage, REC, K, wave, lane, list)
                                              : 0;
        for (int k = 0; k < cnt; k++) {
            const unsigned entry = list[k];
            const T* rec = stage + (entry & 0xffffu);
            const T w = stage[sten_at<T, P>(lane & 3, entry, 0)] *
                        stage[sten_at<T, P>(ly, entry, 1)] * stage[sten_at<T, P>(lz, entry, 2)];
#pragma unroll
            for (int q = 0; q < kVecQ; q++) acc[q] = fma(w, rec[OF + q], acc[q]);
        }
        __syncthreads();
    }
    const int px = org[0] + lx, py = org[1] + ly, pz = org[2] + lz;
    if (lx >= 32 || px >= K || py >= K || pz >= K) return;
    const size_t K3 = (size_t)K * K * K, pt = ((size_t)pz * K + py) * K + px;
#pragma unroll
    for (int q = 0; q < kVecQ; q++)
        if (q0 + q < b * NC) mesh[(q0 + q) * K3 + pt] = acc[q];
}

// ------------------------------------------------------ x transforms -------
// Real rows (2 per complex FFT: z = a + i b). Each workgroup takes NR rows.
// LDS: K twiddles, then two buffers of NR / 2 pencils of stride PS.
template <typename T>
__device__ __forceinline__ void load_twiddles(cplx<T>* tw, const double* __restrict__ tw_g, int K) {
    for (int i = threadIdx.x; i < K; i += blockDim.x)
        tw[i] = cplx<T>{(T)tw_g[2 * i], (T)tw_g[2 * i + 1]};
}

template <typename T>
__global__ void __launch_bounds__(256)
fft_x_r2c_kernel(FFTArgs fa, long long nrows, const T* __restrict__ real,
                 cplx<T>* __restrict__ spec, const double* __restrict__ tw_g, int NR) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    const int K = fa.K, Kh = K / 2 + 1, PS = pencil_stride(K);
    const int npen = NR / 2;
    cplx<T>* tw = reinterpret_cast<cplx<T>*>(smem_raw);
    cplx<T>* bufa = tw + K;
    cplx<T>* bufb = bufa + npen * PS;
    load_twiddles(tw, tw_g, K);
    const long long row0 = (long long)blockIdx.x * NR;
    // the loads of a thread (XB rows pairs at a time) are in flight together
    constexpr int XB = 8;
    for (int i0 = threadIdx.x; i0 < npen * K; i0 += XB * blockDim.x) {
        T va[XB], vb[XB];
#pragma unroll
        for (int u = 0; u < XB; u++) {
            const int i = i0 + u * (int)blockDim.x;
            const int pen = (int)fdiv(i, fa.K_m), x = i - pen * K;
            const long long ra = row0 + 2 * pen;
            va[u] = vb[u] = T(0);
            if (i < npen * K && ra < nrows) {
                va[u] = real[ra * K + x];
                vb[u] = real[(ra + 1) * K + x];
            }
        }
#pragma unroll
        for (int u = 0; u < XB; u++) {
            const int i = i0 + u * (int)blockDim.x;
            const int pen = (int)fdiv(i, fa.K_m), x = i - pen * K;
            if (i < npen * K) bufa[pen * PS + lpad(x)] = cplx<T>{va[u], vb[u]};
        }
    }
    __syncthreads();
    const cplx<T>* res = fft_pencils<T, -1>(bufa, bufb, npen, PS, fa, tw);
    for (int i = threadIdx.x; i < npen * Kh; i += blockDim.x) {
        const int pen = (int)fdiv(i, fa.Kh_m), k = i - pen * Kh;
        const long long ra = row0 + 2 * pen;
        if (ra >= nrows) continue;
        const cplx<T> zk = res[pen * PS + lpad(k)];
        const cplx<T> zm = res[pen * PS + lpad(k == 0 ? 0 : K - k)];
        const T h = T(0.5);
        spec[ra * Kh + k] = cplx<T>{h * (zk.x + zm.x), h * (zk.y - zm.y)};
        spec[(ra + 1) * Kh + k] = cplx<T>{h * (zk.y + zm.y), h * (zm.x - zk.x)};
    }
}

template <typename T>
__global__ void __launch_bounds__(256)
fft_x_c2r_kernel(FFTArgs fa, long long nrows, const cplx<T>* __restrict__ spec,
                 T* __restrict__ real, const double* __restrict__ tw_g, int NR) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    const int K = fa.K, Kh = K / 2 + 1, PS = pencil_stride(K);
    const int npen = NR / 2;
    cplx<T>* tw = reinterpret_cast<cplx<T>*>(smem_raw);
    cplx<T>* bufa = tw + K;
    cplx<T>* bufb = bufa + npen * PS;
    load_twiddles(tw, tw_g, K);
    const long long row0 = (long long)blockIdx.x * NR;
    // the loads of a thread (XB at a time) are in flight together
    constexpr int XB = 8;
    for (int i0 = threadIdx.x; i0 < npen * K; i0 += XB * blockDim.x) {
        cplx<T> A[XB], B[XB];
#pragma unroll
        for (int u = 0; u < XB; u++) {
            const int i = i0 + u * (int)blockDim.x;
            const int pen = (int)fdiv(i, fa.K_m), k = i - pen * K;
            const long long ra = row0 + 2 * pen;
            A[u] = B[u] = cplx<T>{T(0), T(0)};
            if (i < npen * K && ra < nrows) {
                const int kk = (k <= K / 2) ? k : K - k;
                A[u] = spec[ra * Kh + kk];
                B[u] = spec[(ra + 1) * Kh + kk];
            }
        }
#pragma unroll
        for (int u = 0; u < XB; u++) {
            const int i = i0 + u * (int)blockDim.x;
            const int pen = (int)fdiv(i, fa.K_m), k = i - pen * K;
            const long long ra = row0 + 2 * pen;
            cplx<T> z{T(0), T(0)};
            if (i < npen * K && ra < nrows) {
                const int kk = (k <= K / 2) ? k : K - k;
                cplx<T> a = A[u], bb = B[u];
                if (kk == 0 || 2 * kk == K) { a.y = T(0); bb.y = T(0); }
                if (k <= K / 2) z = cplx<T>{a.x - bb.y, a.y + bb.x};
                else z = cplx<T>{a.x + bb.y, bb.x - a.y};
            }
            if (i < npen * K) bufa[pen * PS + lpad(k)] = z;
        }
    }
    __syncthreads();
    const cplx<T>* res = fft_pencils<T, +1>(bufa, bufb, npen, PS, fa, tw);
    for (int i = threadIdx.x; i < npen * K; i += blockDim.x) {
        const int pen = (int)fdiv(i, fa.K_m), x = i - pen * K;
        const long long ra = row0 + 2 * pen;
        if (ra >= nrows) continue;
        const cplx<T> v = res[pen * PS + lpad(x)];
        real[ra * K + x] = v.x;
        real[(ra + 1) * K + x] = v.y;
    }
}

// ------------------------------------------------------- y transform -------
// In place along y (element stride Kh) for NP = 2^lnp consecutive kx of one
// (mesh, z) plane.
template <typename T, int SIGN>
__global__ void __launch_bounds__(256)
fft_y_kernel(FFTArgs fa, cplx<T>* __restrict__ spec, const double* __restrict__ tw_g, int lnp) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    const int K = fa.K, Kh = K / 2 + 1, PS = pencil_stride(K);
    const int NP = 1 << lnp;
    cplx<T>* tw = reinterpret_cast<cplx<T>*>(smem_raw);
    cplx<T>* bufa = tw + K;
    cplx<T>* bufb = bufa + NP * PS;
    load_twiddles(tw, tw_g, K);
    const int nkb = (Kh + NP - 1) >> lnp;
    const int kx0 = (int)(blockIdx.x % nkb) * NP;
    const long long plane = blockIdx.x / nkb;    // mesh * K + z
    cplx<T>* base = spec + plane * K * Kh;
    // the loads of a thread (YB at a time) are in flight together
    constexpr int YB = 8;
    for (int i0 = threadIdx.x; i0 < NP * K; i0 += YB * blockDim.x) {
        cplx<T> v[YB];
#pragma unroll
        for (int u = 0; u < YB; u++) {
            const int i = i0 + u * (int)blockDim.x;
            const int y = i >> lnp, j = i & (NP - 1);
            const int kx = kx0 + j;
            v[u] = (i < NP * K && kx < Kh) ? base[(size_t)y * Kh + kx] : cplx<T>{T(0), T(0)};
        }
#pragma unroll
        for (int u = 0; u < YB; u++) {
            const int i = i0 + u * (int)blockDim.x;
            const int y = i >> lnp, j = i & (NP - 1);
            if (i < NP * K) bufa[j * PS + lpad(y)] = v[u];
        }
    }
    __syncthreads();
    const cplx<T>* res = fft_pencils<T, SIGN>(bufa, bufb, NP, PS, fa, tw);
    for (int i = threadIdx.x; i < NP * K; i += blockDim.x) {
        const int y = i >> lnp, j = i & (NP - 1);
        const int kx = kx0 + j;
        if (kx < Kh) base[(size_t)y * Kh + kx] = res[j * PS + lpad(y)];
    }
}

// ------------------------------------------ z transform + influence -------
// The mesh sides without a two-stage kernel (250 and those above 324): the
// same work as fft_kernels.hpp's fft2_z_influence_kernel with the general
// radix chain, in place in LDS.
constexpr int kZMaxI2 = 8;
constexpr int kZThreads = 512;

template <typename T, int NC>
__global__ void __launch_bounds__(kZThreads)
fft_z_influence_kernel(FFTArgs fa, cplx<T>* __restrict__ spec, const double* __restrict__ tw_g,
                       const double* __restrict__ fac_g, int lnp, double box, double xi) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    const int K = fa.K, Kh = K / 2 + 1, PS = pencil_stride(K);
    const int NP = 1 << lnp;
    const int nj = K * Kh;
    cplx<T>* tw = reinterpret_cast<cplx<T>*>(smem_raw);
    cplx<T>* buf = tw + K;
    load_twiddles(tw, tw_g, K);
    // influence factors in arithmetic T, after the spectrum buffer
    T* s_fac = reinterpret_cast<T*>(buf + (size_t)NC * NP * PS);
    for (int i = threadIdx.x; i < K; i += blockDim.x) s_fac[i] = (T)fac_g[i];
    const int nch = (nj + NP - 1) >> lnp;
    const int j0 = (int)(blockIdx.x % nch) * NP;
    const int rhs = (int)(blockIdx.x / nch);
    const size_t mesh_sz = (size_t)nj * K;
    cplx<T>* base = spec + (size_t)rhs * NC * mesh_sz + j0;
    const int nvalid = min(NP, nj - j0);
    // the loads of a thread (ZB at a time) are in flight together
    constexpr int ZB = 8;
    for (int i0 = threadIdx.x; i0 < NC * NP * K; i0 += ZB * kZThreads) {
        cplx<T> v[ZB];
#pragma unroll
        for (int u = 0; u < ZB; u++) {
            const int i = i0 + u * kZThreads;
            const int jl = i & (NP - 1);
            const int cz = i >> lnp;
            const int c = (int)fdiv(cz, fa.K_m), z = cz - c * K;
            v[u] = (i < NC * NP * K && jl < nvalid) ? base[c * mesh_sz + (size_t)z * nj + jl]
                                                    : cplx<T>{T(0), T(0)};
        }
#pragma unroll
        for (int u = 0; u < ZB; u++) {
            const int i = i0 + u * kZThreads;
            const int jl = i & (NP - 1);
            const int cz = i >> lnp;
            const int c = (int)fdiv(cz, fa.K_m), z = cz - c * K;
            if (i < NC * NP * K) buf[(c * NP + jl) * PS + lpad(z)] = v[u];
        }
    }
    __syncthreads();
    fft_pencils_inplace<T, -1, kZMaxI2>(buf, NC * NP, PS, fa, tw);
    const Influence<T> inf(box, xi);
    const int cs = NP * PS;    // component stride in LDS
    for (int i = threadIdx.x; i < NP * K; i += blockDim.x) {
        const int jl = (int)fdiv(i, fa.K_m), z = i - jl * K;
        if (jl >= nvalid) continue;
        const int j = j0 + jl;
        const int y = (int)fdiv(j, fa.Kh_m), kxi = j - y * Kh;
        cplx<T>* o = buf + jl * PS + lpad(z);
        cplx<T> g[NC];
#pragma unroll
        for (int c = 0; c < NC; c++) g[c] = o[c * cs];
        inf.template apply<NC>(kxi, y <= K / 2 ? y : y - K, z <= K / 2 ? z : z - K,
                               s_fac[kxi] * s_fac[y] * s_fac[z], g);
#pragma unroll
        for (int c = 0; c < NC; c++) o[c * cs] = g[c];
    }
    __syncthreads();
    fft_pencils_inplace<T, +1, kZMaxI2>(buf, NC * NP, PS, fa, tw);
    for (int i = threadIdx.x; i < NC * NP * K; i += blockDim.x) {
        const int jl = i & (NP - 1);
        const int cz = i >> lnp;
        const int c = (int)fdiv(cz, fa.K_m), z = cz - c * K;
        if (jl < nvalid) base[c * mesh_sz + (size_t)z * nj + jl] = buf[(c * NP + jl) * PS + lpad(z)];
    }
}

// ------------------------------------------------------------- interp ------
// A workgroup takes the particles whose base points lie in a strip of sxt
// tiles along x (ts x ts x ts each) for RB right-hand sides, i.e. the
// consecutive meshes r0 NC .. (r0 + rb) NC - 1. The meshes go through LDS MV
// at a time (one MV-vector per mesh point): each pass
// stages the region their stencils cover, (sxt ts + P - 1) x (ts + P - 1) x
// (ts + P - 1) points, while the next pass's region is loaded into
// registers. Items (particle, z line) sum their P x P stencil slice of all MV
// meshes with vector LDS reads, and each particle adds its P slices in fixed
// order (src/mob/spme.h:219-265 without the stored P/ind tables).
// Y = beta Y + alpha (sum_U + a^2 sum_W).
// A point's place within one mesh, in 32 bits: bytes where a mesh is no longer
// than 2^32 of them (FP32 up to K = 1024: one scaled add less per load), else
// elements (K^3 <= 2^30), widened before they are scaled (an FP64 mesh passes
// 2^32 bytes from K = 813).
constexpr int kMaxSide = 1024;
template <typename T>
struct MeshPoint {
    static constexpr bool bytes = (size_t)kMaxSide * kMaxSide * kMaxSide * sizeof(T) <= 1ull << 32;
    static_assert((size_t)kMaxSide * kMaxSide * kMaxSide <= 1ull << 32, "32-bit element index");
    static __device__ __forceinline__ unsigned at(int x, int y, int z, int K) {
        return (unsigned)((z * K + y) * K + x) * (bytes ? (unsigned)sizeof(T) : 1u);
    }
    static __device__ __forceinline__ T load(const T* mesh, unsigned at) {
        if constexpr (bytes)
            return *reinterpret_cast<const T*>(reinterpret_cast<const unsigned char*>(mesh) + at);
        else
            return mesh[at];
    }
};

template <typename T, int MV>
struct InterpVec {
    typedef T type __attribute__((ext_vector_type(MV)));
};

template <typename T, int P, int RREG, int MV>
__global__ void __launch_bounds__(256)
interp_tile_kernel(int K, int ts, int ntile, int nsx, int sxt, int ch,
                   const int* __restrict__ tile_start, const double* __restrict__ frac,
                   const int* __restrict__ base, const double* __restrict__ a2,
                   const T* __restrict__ mesh, int b, int RB, int NC, double alpha, double beta,
                   double* __restrict__ Y) {
    typedef typename InterpVec<T, MV>::type VT;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    const unsigned lid = xcd_logical_id(blockIdx.x + blockIdx.y * gridDim.x, gridDim.x * gridDim.y);
    const int bxl = (int)(lid % gridDim.x), byl = (int)(lid / gridDim.x);
    const int sxi = bxl % nsx;
    const int tyz = bxl / nsx;
    const int ty = tyz % ntile, tz = tyz / ntile;
    const int r0 = byl * RB;
    const int rb = min(RB, b - r0);
    const int nmesh = rb * NC;
    const int stx = sxi * sxt;
    const int nxt = min(sxt, ntile - stx);
    const int sx0 = stx * ts, sy0 = ty * ts, sz0 = tz * ts;
    const int RX = nxt * ts + P - 1, RY = ts + P - 1, RZ = ts + P - 1;
    const int nreg = RX * RY * RZ;
    // LDS: region VT[RZ][RY][RX] | partial sums VT[ch][P] | weights T[ch][3][P] |
    //      bases int[ch][3] | results double[ch][RB][3]
    VT* region = reinterpret_cast<VT*>(smem_raw);
    VT* s_part = region + (size_t)(sxt * ts + P - 1) * RY * RZ;
    T* s_w = reinterpret_cast<T*>(s_part + (size_t)ch * P);
    int* s_b = reinterpret_cast<int*>(s_w + ch * 3 * P);
    double* s_res = reinterpret_cast<double*>(
        (reinterpret_cast<uintptr_t>(s_b + ch * 3) + 7) & ~(uintptr_t)7);
    const size_t K3 = (size_t)K * K * K;
    // this thread's region points within one mesh (the same for every mesh,
    // added to its wave-uniform base): point u is region index
    // threadIdx.x + 256 u
    unsigned pt[RREG];
    {
        const unsigned rx_m = 0xffffffffu / (unsigned)RX + 1u;
        const unsigned ry_m = 0xffffffffu / (unsigned)RY + 1u;
#pragma unroll
        for (int u = 0; u < RREG; u++) {
            const int i = min((int)threadIdx.x + 256 * u, nreg - 1);
            const int row = (int)fdiv(i, rx_m), lx = i - row * RX;
            const int lz = (int)fdiv(row, ry_m), ly = row - lz * RY;
            pt[u] = MeshPoint<T>::at(wrapk(sx0 + lx, K), wrapk(sy0 + ly, K), wrapk(sz0 + lz, K), K);
        }
    }
    const T* mbase = mesh + (size_t)r0 * NC * K3;
    VT v[RREG];
    auto prefetch = [&](int pi) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < MV; j++) {
            const int q = pi * MV + j;
            const T* m = mbase + (size_t)min(q, nmesh - 1) * K3;
            const bool on = q < nmesh;
#pragma unroll
            for (int u = 0; u < RREG; u++) {
                const T x = MeshPoint<T>::load(m, pt[u]);
                v[u][j] = on ? x : T(0);
            }
        }
    };
    // own particles: base tiles stx .. stx+nxt-1 of row (ty, tz) are contiguous
    const int t_first = (tz * ntile + ty) * ntile + stx;
    const int pb = tile_start[t_first], pe = tile_start[t_first + nxt];
    const int npass = (nmesh + MV - 1) / MV;
    for (int c0 = pb; c0 < pe; c0 += ch) {
        const int cnt = min(ch, pe - c0);
        prefetch(0);
        for (int t = threadIdx.x; t < cnt; t += blockDim.x) {
            const int is = c0 + t;
            T w[P];
#pragma unroll
            for (int d = 0; d < 3; d++) {
                bspline_weights_r<T, P>(frac[3 * is + d], w);
#pragma unroll
                for (int k = 0; k < P; k++) s_w[(t * 3 + d) * P + k] = w[k];
            }
            // stencil origin relative to the region
            s_b[t * 3 + 0] = wrapk(base[3 * is + 0] - sx0, K);
            s_b[t * 3 + 1] = wrapk(base[3 * is + 1] - sy0, K);
            s_b[t * 3 + 2] = wrapk(base[3 * is + 2] - sz0, K);
            for (int q = 0; q < rb * 3; q++) s_res[t * RB * 3 + q] = 0.0;
        }
        for (int pi = 0; pi < npass; pi++) {
            __syncthreads();          // the previous pass no longer reads the region
#pragma unroll
            for (int u = 0; u < RREG; u++) {
                const int i = (int)threadIdx.x + 256 * u;
                if (i < nreg) region[i] = v[u];
            }
            __syncthreads();
            if (pi + 1 < npass) prefetch(pi + 1);
            for (int item = threadIdx.x; item < cnt * P; item += blockDim.x) {
                const int t = item / P, iz = item - t * P;
                const T* wx = s_w + (t * 3 + 0) * P;
                const T* wy = s_w + (t * 3 + 1) * P;
                const VT* rp = region + ((size_t)(s_b[t * 3 + 2] + iz) * RY + s_b[t * 3 + 1]) * RX +
                               s_b[t * 3 + 0];
                VT acc = VT(0);
                if constexpr (MV == 1) {
                    // rows in pairs: their reads are issued ahead of the sums
#pragma unroll 2
                    for (int iy = 0; iy < P; iy++) {
                        VT row = VT(0);
#pragma unroll
                        for (int ix = 0; ix < P; ix++) row += wx[ix] * rp[iy * RX + ix];
                        acc += wy[iy] * row;
                    }
                } else {
                    // one stencil row at a time keeps the live vector reads to P
#pragma unroll 1
                    for (int iy = 0; iy < P; iy++) {
                        VT row = VT(0);
#pragma unroll
                        for (int ix = 0; ix < P; ix++) row += wx[ix] * rp[iy * RX + ix];
                        acc += wy[iy] * row;
                    }
                }
                s_part[t * P + iz] = acc * s_w[(t * 3 + 2) * P + iz];
            }
            __syncthreads();
            for (int t = threadIdx.x; t < cnt; t += blockDim.x) {
                VT sum = VT(0);
#pragma unroll
                for (int iz = 0; iz < P; iz++) sum += s_part[t * P + iz];
#pragma unroll
                for (int j = 0; j < MV; j++) {
                    const int q = pi * MV + j;
                    if (q < nmesh) {
                        const int r = q / NC, c = q - r * NC;
                        double vv = (double)sum[j];
                        if (c >= 3) vv *= a2[c0 + t];
                        s_res[t * RB * 3 + r * 3 + (c % 3)] += vv;
                    }
                }
            }
        }
        __syncthreads();
        for (int i = threadIdx.x; i < cnt * rb * 3; i += blockDim.x) {
            const int t = i / (rb * 3), rc = i - t * rb * 3;
            const int r = rc / 3, c = rc - r * 3;
            double* y = &Y[(size_t)(3 * (c0 + t) + c) * b + r0 + r];
            *y = (beta == 0.0 ? 0.0 : beta * *y) + alpha * s_res[t * RB * 3 + r * 3 + c];
        }
        __syncthreads();
    }
}

// The same interpolation from blocks of tiles. A workgroup of 512 threads
// takes the particles whose base points lie in an st.x x st.y x st.z block of
// tiles (16 x 16 x 16 points where they are dense), for RB right-hand sides. A
// mesh's region is then (16 + P - 1)^3 points, 2.3 reads per mesh point (P =
// 6) where the strips above read each 3.1 times. An item (particle, z line)
// stays with its thread for all meshes, its x weights and stencil origin in
// registers, y and z weights in LDS; the particle sums of
// a pass run beside the next region's stores, two barriers a pass. Two
// workgroups per CU leave 128 registers: with all weights in registers 1.95
// instead of 1.78 ms, and as it is the FP32 kernels of 16 and 19 region points
// a thread still spill 12 to 116 bytes a lane (P = 6: 24 and 96; order 4 with
// 16 points none, FP64 none).
// Bound by the regions' loads, LDS reads with random bank conflicts and the
// barriers between them. HBM traffic of 100 FP32 columns, K = 128: 6.4 GB, of
// which 5.5 GB fetched (the meshes 2.2 times, strips 2.0) and 0.6 GB spilled
// values. Interpolation of 100 FP32 columns, strips -> blocks:
// K = 128, N = 100 000: 1.95 -> 1.78 ms, K = 108, N = 50 000: 1.39 -> 1.06; 32
// columns, K = 100, N = 50 000: 446 -> 302 us; 16 FP64 columns, K = 90,
// N = 20 011: 302 -> 188 us.
constexpr int kIbThreads = 512, kIbItems = 3;

template <typename T, int P, int RREG, bool POLY>
__global__ void __launch_bounds__(kIbThreads) __attribute__((amdgpu_waves_per_eu(sizeof(T) == 4 ? 4 : 2)))
interp_block_kernel(int K, int ts, int ntile, int3 nb, int3 st, const int* __restrict__ tile_start,
                    const T* __restrict__ sten, const double* __restrict__ a2,
                    const T* __restrict__ mesh, int b, int RB, double alpha, double beta,
                    double* __restrict__ Y) {
    typedef Sten<T, P> St;
    typedef typename std::conditional<POLY, double, T>::type RT;
    constexpr int NC = POLY ? 6 : 3, CH = kIbThreads * kIbItems / P;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    __shared__ int s_beg[16], s_off[17];
    const unsigned lid = xcd_logical_id(blockIdx.x + blockIdx.y * gridDim.x, gridDim.x * gridDim.y);
    const int bxl = (int)(lid % gridDim.x), byl = (int)(lid / gridDim.x);
    const int tx = bxl % nb.x * st.x, ty = bxl / nb.x % nb.y * st.y, tz = bxl / (nb.x * nb.y) * st.z;
    const int ntx = min(st.x, ntile - tx), nty = min(st.y, ntile - ty), ntz = min(st.z, ntile - tz);
    const int r0 = byl * RB, rb = min(RB, b - r0), nmesh = rb * NC;
    const int sx0 = tx * ts, sy0 = ty * ts, sz0 = tz * ts;
    const int RX = ntx * ts + P - 1, RY = nty * ts + P - 1, RZ = ntz * ts + P - 1;
    const int nreg = RX * RY * RZ;
    // LDS: region T[nreg] | partial sums T[2][CH][P] | results RT[CH][RB][3] | ids
    const int nreg_max = (st.x * ts + P - 1) * (st.y * ts + P - 1) * (st.z * ts + P - 1);
    T* region = reinterpret_cast<T*>(smem_raw);
    T* s_part = region + ((nreg_max + 3) & ~3);
    constexpr int WS = 2 * P + 1;   // wy, wz of a particle
    T* s_w = s_part + 2 * CH * P;
    RT* s_res = reinterpret_cast<RT*>(s_w + ((CH * WS + 3) & ~3));
    int* s_id = reinterpret_cast<int*>(s_res + CH * RB * 3);
    // the particles: one range of the sorted order per tile row
    if (threadIdx.x < 64) {
        const int nrow = nty * ntz, r = threadIdx.x;
        int pb = 0, n = 0;
        if (r < nrow) {
            const int t = ((tz + r / nty) * ntile + ty + r % nty) * ntile + tx;
            pb = tile_start[t];
            n = tile_start[t + ntx] - pb;
        }
        int inc = n;
#pragma unroll
        for (int o = 1; o < 16; o <<= 1) {
            const int v = __shfl_up(inc, o);
            if (r >= o) inc += v;
        }
        if (r < 16) {
            s_beg[r] = pb;
            s_off[r] = inc - n;
            if (r == 15) s_off[16] = inc;
        }
    }
    const size_t K3 = (size_t)K * K * K;
    unsigned pt[RREG];
    {
        const unsigned rx_m = 0xffffffffu / (unsigned)RX + 1u;
        const unsigned ry_m = 0xffffffffu / (unsigned)RY + 1u;
#pragma unroll
        for (int u = 0; u < RREG; u++) {
            const int i = min((int)threadIdx.x + kIbThreads * u, nreg - 1);
            const int row = (int)fdiv(i, rx_m), lx = i - row * RX;
            const int lz = (int)fdiv(row, ry_m), ly = row - lz * RY;
            pt[u] = MeshPoint<T>::at(wrapk(sx0 + lx, K), wrapk(sy0 + ly, K), wrapk(sz0 + lz, K), K);
        }
    }
    const T* mbase = mesh + (size_t)r0 * NC * K3;
    T v[RREG];
    auto prefetch = [&](int q) __attribute__((always_inline)) {
        const T* m = mbase + (size_t)q * K3;
#pragma unroll
        for (int u = 0; u < RREG; u++) v[u] = MeshPoint<T>::load(m, pt[u]);
    };
    __syncthreads();
    const int np = s_off[16];
    for (int c0 = 0; c0 < np; c0 += CH) {
        const int cnt = min(CH, np - c0);
        // the items' weights and stencil origins
        T wx[kIbItems][P];
        int at[kIbItems];
#pragma unroll
        for (int u = 0; u < kIbItems; u++) {
            const int it = threadIdx.x + u * kIbThreads, t = it / P, iz = it - t * P;
            at[u] = -1;
            if (t < cnt) {
                int k = 0;
                while (s_off[k + 1] <= c0 + t) k++;
                const int is = s_beg[k] + c0 + t - s_off[k];
                if (iz == 0) s_id[t] = is;
                const T* rec = sten + (size_t)is * St::N;
                const int* b3 = reinterpret_cast<const int*>(rec);
#pragma unroll
                for (int i = 0; i < P; i++) wx[u][i] = rec[St::OW + i];
                s_w[t * WS + iz] = rec[St::OW + St::RUN + iz];
                s_w[t * WS + P + iz] = rec[St::OW + 2 * St::RUN + iz];
                at[u] = ((wrapk(b3[2] - sz0, K) + iz) * RY + wrapk(b3[1] - sy0, K)) * RX +
                        wrapk(b3[0] - sx0, K);
            }
        }
        prefetch(0);
        // one more round than meshes: round pi stores region pi and adds up
        // the particle sums of mesh pi - 1
        for (int pi = 0; pi <= nmesh; pi++) {
            if (pi < nmesh) {
#pragma unroll
                for (int u = 0; u < RREG; u++) {
                    const int i = (int)threadIdx.x + kIbThreads * u;
                    if (i < nreg) region[i] = v[u];
                }
            }
            if (pi > 0) {
                const T* sp = s_part + ((pi - 1) & 1) * CH * P;
                const int q = pi - 1, r = q / NC, c = q - r * NC;
                for (int t = threadIdx.x; t < cnt; t += kIbThreads) {
                    T sum = T(0);
#pragma unroll
                    for (int iz = 0; iz < P; iz++) sum += sp[t * P + iz];
                    RT* o = s_res + (t * RB + r) * 3 + c % 3;
                    if (c < 3) *o = (RT)sum;
                    else *o += (RT)sum * (RT)a2[s_id[t]];
                }
            }
            __syncthreads();
            if (pi == nmesh) break;
            if (pi + 1 < nmesh) prefetch(pi + 1);
            T* sp = s_part + (pi & 1) * CH * P;
#pragma unroll
            for (int u = 0; u < kIbItems; u++) {
                if (at[u] < 0) continue;
                const int it = threadIdx.x + u * kIbThreads, t = it / P;
                const T* rp = region + at[u];
                const T* w = s_w + t * WS;
                T acc = T(0);
#pragma unroll 2
                for (int iy = 0; iy < P; iy++) {
                    T row = T(0);
#pragma unroll
                    for (int ix = 0; ix < P; ix++) row += wx[u][ix] * rp[iy * RX + ix];
                    acc += w[iy] * row;
                }
                sp[it] = acc * w[P + it - t * P];
            }
            __syncthreads();
        }
        for (int i = threadIdx.x; i < cnt * rb * 3; i += kIbThreads) {
            const int t = i / (rb * 3), cr = i - t * rb * 3;
            const int c = cr / rb, r = cr - c * rb;
            double* y = &Y[(size_t)(3 * s_id[t] + c) * b + r0 + r];
            *y = (beta == 0.0 ? 0.0 : beta * *y) + alpha * (double)s_res[(t * RB + r) * 3 + c];
        }
        __syncthreads();
    }
}

// ------------------------------------------------------------ host side ----
void bspline_moduli(int K, int P, std::vector<double>& out) {
    // |b(m)|^2 = 1 / |sum_{i<P-1} M_P(i+1) e^{2 pi i m i / K}|^2
    // (src/mob/spme.cc:80-128; Essmann et al. 1995)
    std::vector<double> sv(P - 1);
    for (int i = 0; i < P - 1; i++) {
        // M_P(i+1) by Cox-de Boor on integer knots
        std::vector<double> a(P + 1, 0.0);
        a[0] = 1.0;  // M_1(u + k) with u = 0 -> use u = 1 piece boundary
        double u = 1.0;
        for (int n = 2; n <= P; n++) {
            for (int k = n - 1; k >= 1; k--)
                a[k] = ((u + k) * a[k] + (n - u - k) * a[k - 1]) / (n - 1);
            a[0] = u * a[0] / (n - 1);
        }
        sv[i] = a[i];   // M_P(1 + i)
    }
    std::vector<double> den2(K);
    for (int m = 0; m < K; m++) {
        int mm = (m <= K / 2) ? m : m - K;
        double re = 0.0, im = 0.0;
        for (int i = 0; i < P - 1; i++) {
            double ph = 2.0 * M_PI * mm * i / K;
            re += sv[i] * cos(ph);
            im += sv[i] * sin(ph);
        }
        den2[m] = re * re + im * im;
    }
    // odd P: the sum vanishes at the Nyquist index (M_P is symmetric), and
    // rounding leaves |den|^2 ~ 1e-33; take the mean of the neighbours there
    // instead (Essmann et al. 1995). Even P is unaffected (|den|^2 > 1e-3).
    for (int m = 0; m < K; m++)
        if (den2[m] < 1e-7) den2[m] = 0.5 * (den2[(m + K - 1) % K] + den2[(m + 1) % K]);
    out.resize(K);
    for (int m = 0; m < K; m++) out[m] = 1.0 / den2[m];
}

bool make_fft_plan(int K, FFTPlan* plan, int order) {
    plan->K = K;
    plan->nst = 0;
    int m = K;
    auto take = [&](int r) {
        while (m % r == 0 && plan->nst < 16) { plan->radix[plan->nst++] = r; m /= r; }
    };
    if (order == 2) { take(3); take(5); }
    if (order != 1) take(8);
    take(4);
    take(2);
    take(3);
    take(5);
    return m == 1;
}

template <typename T>
void SpmeGpu<T>::set_tuning(const SpmeTuning& t, int width) {
    FFTPlan p;
    SDT_REQUIRE(t.fft_order >= 0 && t.fft_order <= 2 && make_fft_plan(K, &p, t.fft_order),
                SDT_EINVAL, "tuning: invalid FFT stage order");
    SDT_REQUIRE(t.spread_stage_kb == 0 || (t.spread_stage_kb >= 16 && t.spread_stage_kb <= 64),
                SDT_EINVAL, "tuning: spread stage must be 16 .. 64 KB");
    SDT_REQUIRE(t.interp_sxt == 0 || t.interp_sxt == 1 || t.interp_sxt == 2 || t.interp_sxt == 4,
                SDT_EINVAL, "tuning: interp strip width must be 1, 2 or 4 tiles");
    SDT_REQUIRE(t.interp_ch == 0 || (t.interp_ch >= 32 && t.interp_ch <= 128), SDT_EINVAL,
                "tuning: interp chunk must be 32 .. 128");
    SDT_REQUIRE(width == 0 || width == 1, SDT_EINVAL, "tuning: width class must be 0 or 1");
    plans[width] = p;
    tune[width] = t;
}

static FFTArgs fft_args(const FFTPlan& p) {
    FFTArgs a;
    memset(&a, 0, sizeof(a));
    a.K = p.K;
    a.nst = p.nst;
    a.K_m = fft_magic(p.K);
    a.Kh_m = fft_magic(p.K / 2 + 1);
    int len = p.K;
    for (int i = 0; i < p.nst; i++) {
        const int r = p.radix[i];
        a.radix[i] = r;
        a.per[i] = p.K / r;
        a.per_m[i] = fft_magic(a.per[i]);
        a.str[i] = p.K / len;
        a.str_m[i] = fft_magic(a.str[i]);
        len /= r;
    }
    return a;
}

// entries of the spread's candidate lists: the most blocks that one stencil can
// reach, over its base points and per dimension (blocks of 32 or 4 points, the
// last one partial), for every particle
static long long spread_list_cap(int npos, int K, int porder) {
    auto reach = [&](int len) {
        int most = 0;
        for (int b0 = 0; b0 < K; b0++) {
            std::vector<int> got;
            for (int q = 0; q < porder; q++) {
                const int bl = ((b0 + q) % K) / len;
                if (std::find(got.begin(), got.end(), bl) == got.end()) got.push_back(bl);
            }
            most = std::max(most, (int)got.size());
        }
        return (long long)most;
    };
    return reach(32) * reach(4) * reach(4) * npos;
}

// Sten<T, P>::N
template <typename T>
static int sten_values(int porder) {
    const int sv = 16 / (int)sizeof(T);
    return (sv + 3 * (porder + 3) + 3 + sv - 1) / sv * sv;
}

template <typename T>
double SpmeGpu<T>::system_bytes(int npos, int K, int porder) {
    // record, two offsets, two bases and a^2 of a particle; its list entries;
    // block segments; starts and sort counters of tiles of 4^3 points or more
    return npos * ((double)sten_values<T>(porder) * sizeof(T) + 2 * 24 + 2 * 12 + 8) +
           4.0 * spread_list_cap(npos, K, porder) +
           (double)K * K * K * (sizeof(SpreadSeg) / 512.0 + 12.0 / 64.0);
}

template <typename T>
void SpmeGpu<T>::create(int npos_, double box_, double xi_, int K_, int porder_, bool poly_) {
    npos = npos_; box = box_; xi = xi_; K = K_; porder = porder_; poly = poly_;
    // narrower than the reference (porder > 1 with 4 porder <= dim,
    // src/mob/mob_spme.cc:79-90): the kernels are instantiated for these
    SDT_REQUIRE(porder >= 4 && porder <= 8, SDT_EINVAL,
                "porder must be in [4, 8] on the GPU path (the reference accepts any porder > 1 "
                "with 4 porder <= dim)");
    SDT_REQUIRE(K % 2 == 0, SDT_EINVAL,
                "mesh dimension must be even on the GPU path (the reference's odd-dim wavenumber "
                "map is incomplete)");
    SDT_REQUIRE(make_fft_plan(K, &plan), SDT_EINVAL,
                "mesh dimension must factor into 2, 3 and 5 on the GPU path");
    SDT_REQUIRE(K <= kMaxSide, SDT_EINVAL, "mesh dimension must be <= 1024");
    plans[0] = plans[1] = plan;
    tune[0] = tune[1] = SpmeTuning();
    // tile side: a divisor of K in [P-1, 8], preferring 8 (one wave owns
    // ts x ts mesh rows)
    ts = 0;
    const int pref[] = {8, 6, 7, 5, 4};
    for (int c : pref)
        if (c >= porder - 1 && K % c == 0 && K / c >= 3) { ts = c; break; }
    SDT_REQUIRE(ts > 0, SDT_EINVAL, "no spread tile size divides the mesh dimension");
    ntile = K / ts;
    // tile rows of a 32 x 4 x 4 spread block's window, two ranges each
    const int trow = std::min(ntile, (porder + 3 + ts - 1) / ts + 1);
    SDT_REQUIRE(2 * trow * trow <= kListRanges, SDT_EINVAL,
                "spread: too many contributor tiles for this order and mesh");
    const size_t nblocks = (size_t)ceil_div(K, 32) * ceil_div(K, 4) * ceil_div(K, 4);
    d_nids.reserve(1);
    d_ids.reserve((size_t)spread_list_cap(npos, K, porder));
    d_blk.reserve(nblocks);
    std::vector<double> tw(2 * K);
    for (int j = 0; j < K; j++) {
        tw[2 * j] = cos(-2.0 * M_PI * j / K);
        tw[2 * j + 1] = sin(-2.0 * M_PI * j / K);
    }
    d_tw.reserve(2 * K);
    SDT_HIP_CHECK(sync_memcpy(d_tw.get(), tw.data(), sizeof(double) * 2 * K, hipMemcpyHostToDevice));
    std::vector<double> bs;
    bspline_moduli(K, porder, bs);
    // the influence factors |b(m)|^2 e^{-k_m^2 / 4 xi^2}, one per mesh index
    for (int m = 0; m < K; m++) {
        const double k = 2.0 * M_PI / box * (m <= K / 2 ? m : m - K);
        bs[m] *= exp(-k * k / (4.0 * xi * xi));
    }
    d_fac.reserve(K);
    SDT_HIP_CHECK(sync_memcpy(d_fac.get(), bs.data(), sizeof(double) * K, hipMemcpyHostToDevice));
    sten_n = sten_values<T>(porder);
    d_sten.reserve((size_t)sten_n * npos);
    d_frac.reserve(3 * (size_t)npos);
    d_base.reserve(3 * (size_t)npos);
    d_frac_u.reserve(3 * (size_t)npos);
    d_base_u.reserve(3 * (size_t)npos);
    d_a2.reserve(npos);
    d_tile_start.reserve((size_t)ntile * ntile * ntile + 1);
}

template <typename T>
void SpmeGpu<T>::reserve_rhs(int b) {
    if (b <= bcap) return;
    const size_t K3 = (size_t)K * K * K;
    const size_t Ksp = (size_t)K * K * (K / 2 + 1);
    d_real.reserve((size_t)nmesh(b) * K3);
    d_spec.reserve((size_t)nmesh(b) * Ksp);
    bcap = b;
}

template <typename T>
void SpmeGpu<T>::prepare(const double* d_pos, int* d_key, hipStream_t s) {
    const unsigned g = ceil_div(npos, 256);
#define SDT_PREP(PP)                                                                 \
    case PP:                                                                         \
        hipLaunchKernelGGL((spme_prepare_kernel<T, PP>), dim3(g), dim3(256), 0, s, npos, \
                           d_pos, box, K, ts, ntile, d_frac_u.get(), d_base_u.get(), d_key); \
        break;
    switch (porder) { SDT_PREP(4) SDT_PREP(5) SDT_PREP(6) SDT_PREP(7) SDT_PREP(8) }
#undef SDT_PREP
    SDT_HIP_CHECK(hipGetLastError());
}

template <typename T>
void SpmeGpu<T>::gather_sorted(const int* d_perm, const double* d_pos, const double* d_rdi,
                               hipStream_t s) {
    (void)d_pos;
    const int nsx = (K + 31) / 32;
    const int nblocks = nsx * (int)ceil_div(K, 4) * (int)ceil_div(K, 4);
#define SDT_GATHER(PP)                                                                        \
    case PP:                                                                                  \
        hipLaunchKernelGGL((spme_gather_kernel<T, PP>), dim3(ceil_div(npos, 256)), dim3(256), 0, s, \
                           npos, d_perm, d_frac_u.get(), d_base_u.get(), d_rdi, d_sten.get(), \
                           d_frac.get(), d_base.get(), poly ? d_a2.get() : (double*)nullptr, d_nids.get()); \
        hipLaunchKernelGGL((spread_list_kernel<PP>), dim3(ceil_div(nblocks, kListWaves)),     \
                           dim3(64 * kListWaves), 0, s, K, ts, ntile, nsx, nblocks,           \
                           d_tile_start.get(), d_base.get(), d_nids.get(), d_blk.get(),          \
                           d_ids.get());                                                      \
        break;
    switch (porder) { SDT_GATHER(4) SDT_GATHER(5) SDT_GATHER(6) SDT_GATHER(7) SDT_GATHER(8) }
#undef SDT_GATHER
    SDT_HIP_CHECK(hipGetLastError());
}

// force values per workgroup of the spread: 4 or 16 when few meshes are
// needed, else a column block of 16 (FP32) or 8 (FP64) columns
template <typename T>
static int spread_values(int b, int NC) {
    if (b * NC <= 4) return 4;
    return (b * NC <= 16) ? 16 : (sizeof(T) == 4 ? 48 : 24);
}

template <typename T>
int SpmeGpu<T>::blocked_cols(int b) const {
    if (poly) return 0;
    const int NQ = spread_values<T>(b, 3);
    return NQ <= 16 ? 0 : NQ / 3;
}

// Xs[cb][j][c][r], RC columns per block and zero beyond the last: the spread's
// own copy of the packed input where it cannot share the real space's. H = 1:
// column v is right-hand side v; H = 2 (unequal radii): column 2 r + h is
// right-hand side r, times a^2 for h = 1, so that mesh 3 v + c is mesh
// 6 r + 3 h + c.
template <typename T, int RC, int H>
__global__ void spread_copy_kernel(int npos, int b, int nblk, const double* __restrict__ x,
                                   const double* __restrict__ a2, T* __restrict__ y) {
    const long long n = (long long)nblk * npos * 3 * RC;
    const long long stride = (long long)gridDim.x * blockDim.x;
    for (long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += stride) {
        const int r = (int)(e % RC);
        const long long q = e / RC;            // (cb npos + j) 3 + c
        const long long row = q % (3LL * npos);
        const int v = (int)(q / (3LL * npos)) * RC + r;
        const int col = v / H;
        double f = 0.0;
        if (col < b) {
            f = x[row * b + col];
            if (H == 2 && (v & 1)) f *= a2[row / 3];
        }
        y[e] = (T)f;
    }
}

template <typename T>
void SpmeGpu<T>::spread(int b, const double* X, hipStream_t s, const T* xb) {
    SDT_REQUIRE(b <= bcap, SDT_ECAP, "spread: rhs count exceeds mesh capacity");
    SDT_REQUIRE(xb == nullptr || blocked_cols(b) > 0, SDT_EINVAL,
                "spread: no blocked input for this configuration");
    const SpmeTuning& tn = tune[width_class(b)];
    constexpr int NQL = sizeof(T) == 4 ? 48 : 24;
    const int NC = poly ? 6 : 3;
    const int NQ = spread_values<T>(b, NC);
    const int fr = spread_form & 3;
    const int nsx = (K + 31) / 32;
    const unsigned nblocks = nsx * ceil_div(K, 4) * ceil_div(K, 4);
    if (fr == 1 || fr == 2) {
        // the vector-ALU comparison form
        const size_t slot = spread_slot_bytes<T>(sten_n, kVecQ);
        const int cap = (int)(48 * 1024 / slot);
        const dim3 grid(nblocks, ceil_div(b * NC, kVecQ));
#define SDT_VEC(PP)                                                                            \
    case PP:                                                                                   \
        hipLaunchKernelGGL((spread_vec_kernel<T, PP>), grid, dim3(kPtThreads), cap * slot, s, \
                           K, nsx, d_blk.get(), d_ids.get(), d_sten.get(), d_a2.get(), X, b,  \
                           NC, cap, d_real.get());                                            \
        break;
        switch (porder) { SDT_VEC(4) SDT_VEC(5) SDT_VEC(6) SDT_VEC(7) SDT_VEC(8) }
#undef SDT_VEC
        SDT_HIP_CHECK(hipGetLastError());
        return;
    }
    // Wide launches read a blocked copy, their own where the real space's is
    // not there
    const bool wide = NQ == NQL;
    const int cols = wide && poly ? 2 * b : b;
    constexpr int RC = NQL / 3;
    if (wide && xb == nullptr) {
        const int nblk = ceil_div(cols, RC);
        const long long n = (long long)nblk * npos * 3 * RC;
        d_xs.reserve((size_t)n);
        const dim3 g((unsigned)std::min<long long>(ceil_div((size_t)n, 256), 8192));
        if (poly)
            hipLaunchKernelGGL((spread_copy_kernel<T, RC, 2>), g, dim3(256), 0, s, npos, b, nblk, X,
                               d_a2.get(), d_xs.get());
        else
            hipLaunchKernelGGL((spread_copy_kernel<T, RC, 1>), g, dim3(256), 0, s, npos, b, nblk, X,
                               (const double*)nullptr, d_xs.get());
        SDT_HIP_CHECK(hipGetLastError());
        xb = d_xs.get();
    }
    // stage: two workgroups per CU beside the output tiles for wide launches,
    // four (FP32, NQ = 4), three or (FP64 with 16 values) two for narrow ones
    const size_t slot = spread_slot_bytes<T>(sten_n, NQ);
    const size_t tile = NQ == 4 ? SpreadTile<T, 4>::bytes : SpreadTile<T, 16>::bytes;
    const int stage_kb = tn.spread_stage_kb > 0 ? tn.spread_stage_kb
                                                : (wide ? 62
                                                        : (sizeof(T) == 4 ? (NQ == 4 ? 31 : 35)
                                                                          : (NQ == 4 ? 35 : 62)));
    const int cap = (int)(stage_kb * 1024 / slot);
    const size_t lds = ((cap * slot + 15) & ~(size_t)15) + tile;
    // column blocks a workgroup takes in turn: all of them where the mesh
    // blocks alone fill the chip twice over (two workgroups per CU), fewer on
    // small meshes; one in form 3
    const int ncb = wide ? ceil_div(cols, RC) : 1;
    int ncbw = 1;
    if (fr == 0 || (spread_form & 8))
        ncbw = ceil_div(ncb, std::min<unsigned>(ncb, ceil_div(1024, nblocks)));
    const dim3 grid(nblocks, ceil_div(ncb, ncbw));
#define SDT_SPREAD_Q(PP, QQ, BB)                                                               \
    do {                                                                                      \
        allow_lds((const void*)spread_mx_kernel<T, PP, QQ, BB>, lds);                         \
        hipLaunchKernelGGL((spread_mx_kernel<T, PP, QQ, BB>), grid, dim3(kPtThreads), lds, s, \
                           K, nsx, d_blk.get(), d_ids.get(), d_sten.get(), d_a2.get(), X, xb, \
                           npos, cols, ncbw, NC, cap, d_real.get());                          \
    } while (0)
#define SDT_SPREAD_P(PP)                                                                       \
    case PP:                                                                                   \
        if (wide) SDT_SPREAD_Q(PP, NQL, true);                                                 \
        else if (NQ == 4) SDT_SPREAD_Q(PP, 4, false);                                          \
        else SDT_SPREAD_Q(PP, 16, false);                                                      \
        break;
    switch (porder) { SDT_SPREAD_P(4) SDT_SPREAD_P(5) SDT_SPREAD_P(6) SDT_SPREAD_P(7) SDT_SPREAD_P(8) }
#undef SDT_SPREAD_P
#undef SDT_SPREAD_Q
    SDT_HIP_CHECK(hipGetLastError());
}

template <typename T>
static int pick_lnp(int K, int ncomp_pen, size_t budget) {
    // log2 of the pencils per workgroup so that 2 padded buffers + twiddles
    // fit the budget
    int lnp = 4;
    while (lnp > 0 &&
           (2 * (size_t)ncomp_pen * ((size_t)1 << lnp) * pencil_stride(K) + K) * sizeof(cplx<T>) >
               budget)
        lnp--;
    return lnp;
}

template <typename T>
static size_t fft_lds_bytes(int K, int npen) {
    return (K + 2 * (size_t)npen * pencil_stride(K)) * sizeof(cplx<T>);
}

// largest dynamic LDS allocation of one workgroup on the current device
static size_t max_lds_bytes() {
    static size_t v = 0;
    if (!v) {
        int dev = 0, x = 0;
        SDT_HIP_CHECK(hipGetDevice(&dev));
        SDT_HIP_CHECK(hipDeviceGetAttribute(&x, hipDeviceAttributeMaxSharedMemoryPerBlock, dev));
        v = (size_t)x;
    }
    return v;
}

void allow_lds(const void* fn, size_t bytes) {
    if (bytes <= 64 * 1024) return;
    static std::mutex mu;
    static std::map<const void*, size_t> raised;
    std::lock_guard<std::mutex> lk(mu);
    size_t& have = raised[fn];
    if (have >= bytes) return;
    SDT_HIP_CHECK(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes));
    have = bytes;
}

template <typename T>
void SpmeGpu<T>::fft_forward(int b, hipStream_t s) {
    typedef Fft2Launch<T> F2;
    if (fft_form != 1 && F2::plane_fits(K)) {
        F2::plane(K, true, nmesh(b), d_real.get(), d_spec.get(), d_tw.get(), s);
        return;
    }
    if (F2::has_xy(K)) {
        F2::xy(K, true, nmesh(b), d_real.get(), d_spec.get(), d_tw.get(), s);
        return;
    }
    const FFTArgs fa = fft_args(plans[width_class(b)]);
    const int Kh = K / 2 + 1;
    const long long nrows = (long long)nmesh(b) * K * K;
    const int NR = 2 << pick_lnp<T>(K, 1, 48 * 1024);
    hipLaunchKernelGGL((fft_x_r2c_kernel<T>), dim3(ceil_div(nrows, NR)), dim3(256),
                       fft_lds_bytes<T>(K, NR / 2), s, fa, nrows, d_real.get(), d_spec.get(),
                       d_tw.get(), NR);
    SDT_HIP_CHECK(hipGetLastError());
    const int lnp = pick_lnp<T>(K, 1, 48 * 1024);
    hipLaunchKernelGGL((fft_y_kernel<T, -1>), dim3(ceil_div(Kh, 1 << lnp) * nmesh(b) * K),
                       dim3(256), fft_lds_bytes<T>(K, 1 << lnp), s, fa, d_spec.get(), d_tw.get(),
                       lnp);
    SDT_HIP_CHECK(hipGetLastError());
}

template <typename T>
void SpmeGpu<T>::influence(int b, hipStream_t s) {
    const int NC = poly ? 6 : 3;
    // at most this many threads and 2^lnp pencils per component in a
    // workgroup; z_form > 0 picks smaller ones
    static const int forms[][2] = {{512, 4}, {256, 4}, {128, 4}, {256, 3}, {128, 3}, {256, 2}};
    SDT_REQUIRE(z_form >= 0 && z_form <= 5, SDT_EINVAL, "z transform: form must be in [0, 5]");
    const int zf = z_form;
    if (Fft2Launch<T>::has(K)) {
        Fft2Launch<T>::z(K, NC, b, d_spec.get(), d_tw.get(), d_fac.get(), forms[zf][0],
                         forms[zf][1], box, xi, s);
        return;
    }
    const FFTArgs fa = fft_args(plans[width_class(b)]);
    const int Kh = K / 2 + 1;
    const int nj = K * Kh;
    int lnp = forms[zf][1];
    const size_t budget = std::min<size_t>(max_lds_bytes(), 112 * 1024);
    auto lds_of = [&](int l) {
        return (K + (size_t)NC * ((size_t)1 << l) * pencil_stride(K)) * sizeof(cplx<T>) +
               (size_t)K * sizeof(T);
    };
    while (lnp > 0 && (lds_of(lnp) > budget || NC * (K << lnp) > 2 * kZMaxI2 * kZThreads)) lnp--;
    SDT_REQUIRE(lds_of(lnp) <= max_lds_bytes() && NC * K <= 2 * kZMaxI2 * kZThreads, SDT_EINVAL,
                "z transform: mesh dimension too large");
    const size_t lds = lds_of(lnp);
    const unsigned nch = ceil_div(nj, (size_t)1 << lnp);
    const dim3 grid(nch * (unsigned)b);
    if (poly) {
        allow_lds((const void*)fft_z_influence_kernel<T, 6>, lds);
        hipLaunchKernelGGL((fft_z_influence_kernel<T, 6>), grid, dim3(kZThreads), lds, s, fa,
                           d_spec.get(), d_tw.get(), d_fac.get(), lnp, box, xi);
    } else {
        allow_lds((const void*)fft_z_influence_kernel<T, 3>, lds);
        hipLaunchKernelGGL((fft_z_influence_kernel<T, 3>), grid, dim3(kZThreads), lds, s, fa,
                           d_spec.get(), d_tw.get(), d_fac.get(), lnp, box, xi);
    }
    SDT_HIP_CHECK(hipGetLastError());
}

template <typename T>
void SpmeGpu<T>::fft_backward(int b, hipStream_t s) {
    typedef Fft2Launch<T> F2;
    if (fft_form != 1 && F2::plane_fits(K)) {
        F2::plane(K, false, nmesh(b), d_real.get(), d_spec.get(), d_tw.get(), s);
        return;
    }
    if (F2::has_xy(K)) {
        F2::xy(K, false, nmesh(b), d_real.get(), d_spec.get(), d_tw.get(), s);
        return;
    }
    const FFTArgs fa = fft_args(plans[width_class(b)]);
    const int Kh = K / 2 + 1;
    const long long nrows = (long long)nmesh(b) * K * K;
    const int lnp = pick_lnp<T>(K, 1, 48 * 1024);
    hipLaunchKernelGGL((fft_y_kernel<T, +1>), dim3(ceil_div(Kh, 1 << lnp) * nmesh(b) * K),
                       dim3(256), fft_lds_bytes<T>(K, 1 << lnp), s, fa, d_spec.get(), d_tw.get(),
                       lnp);
    SDT_HIP_CHECK(hipGetLastError());
    const int NR = 2 << pick_lnp<T>(K, 1, 48 * 1024);
    hipLaunchKernelGGL((fft_x_c2r_kernel<T>), dim3(ceil_div(nrows, NR)), dim3(256),
                       fft_lds_bytes<T>(K, NR / 2), s, fa, nrows, d_spec.get(), d_real.get(),
                       d_tw.get(), NR);
    SDT_HIP_CHECK(hipGetLastError());
}

template <typename T>
InterpPlan SpmeGpu<T>::interp_plan(int b) const {
    const int RB = 4;
    const int R = porder - 1;
    InterpPlan pl;
    int* sd = pl.sd;
    // Cubes of tiles, unless the tuning or a form asks for strips. Sides by
    // tile side and order: the larger the block the fewer its halo reads, up to
    // 19 region points in a thread's prefetch registers and to the particles of
    // a chunk. The lines, us of the stage (p = 6; more in
    // profiles/launch_rules.txt):
    // - flat (3, 2, 1) blocks of 8-point tiles in FP32 below 2.2 particles per
    //   4^3 points, whose passes are shorter: K = 128, 8 columns, flat / cube at
    //   1.6: 138 / 141, 2.4: 152 / 152, 3: 168 / 163. (On K = 216 flat stays
    //   ahead up to 4: 2.4: 632 / 724, 5: 1125 / 1091.)
    // - strips on large sparse meshes of 8-point tiles, whose passes are all
    //   staging (three workgroups per CU against two): below 48 particles a
    //   block on a grid above 2048. K = 192, 16 FP32 columns, strips / blocks at
    //   24 particles a block: 674 / 704, 48: 722 / 732, 75: 813 / 773. (Not so
    //   in FP64, K = 192, 8 columns, 16: 665 / 591, nor on K = 216, 36: 1058 /
    //   1005, which the line sends to strips too.)
    const SpmeTuning& tn = tune[width_class(b)];
    const double dens = (double)npos / ((double)K * K * K);
    if (ts == 6) { sd[0] = 3; }
    else if (ts == 5) { sd[0] = 4; sd[1] = 3; }
    else if (ts == 4) { sd[0] = 4; sd[1] = 4; sd[2] = 3; }
    else if (porder >= 7) { sd[2] = 1; }
    else if (sizeof(T) == 4 && dens * 64 < 2.2) { sd[0] = ntile >= 6 ? 3 : 2; sd[2] = 1; }
    for (int d = 0; d < 3; d++) sd[d] = std::min(sd[d], ntile);
    auto blocks = [&]() {
        size_t n = 1;
        for (int d = 0; d < 3; d++) n *= ceil_div(ntile, sd[d]);
        return n;
    };
    auto particles = [&]() { return dens * sd[0] * sd[1] * sd[2] * ts * ts * ts; };
    pl.strips = interp_form > 0 || tn.interp_sxt > 0 || tn.interp_ch > 0 ||
                (ts == 8 && particles() < 48 && blocks() * ceil_div(b, RB) > 2048);
    if (pl.strips) return pl;
    const int CH = kIbThreads * kIbItems / porder;
    auto reg_of = [&]() {
        return (size_t)(sd[0] * ts + R) * (sd[1] * ts + R) * (sd[2] * ts + R);
    };
    auto lds_b = [&](int rb) {
        return ((reg_of() + 3) / 4 * 4 + 2 * (size_t)CH * porder +
                (CH * (2 * porder + 1) + 3) / 4 * 4) * sizeof(T) +
               (size_t)CH * rb * 3 * (poly ? 8 : sizeof(T)) + CH * sizeof(int);
    };
    // smaller blocks where the particles exceed a chunk: K = 64, 8 FP32
    // columns, cubes of 0.85 chunks 39 us; of 1.0 chunks 51, blocks of half 36.
    // And on small meshes, where the grid would leave CUs idle: at least 512
    // workgroups. K = 64, 8 FP32 columns, at least 128: 39, 256: 38, 512: 32,
    // 1024: 38 us; K = 48, 20: 40, 31, 31, 39. FP64 (one or two workgroups per
    // CU) and single columns do better with fewer, one full round of the CUs:
    // K = 64, 4 FP64: 41, 21, 27, 31; K = 96, 1 FP32: 21, 21, 24, 27.
    for (int d = 2; sd[0] > 1 || sd[1] > 1 || sd[2] > 1; d = (d + 2) % 3) {
        if (reg_of() <= 19u * kIbThreads && lds_b(1) <= 150 * 1024 &&
            particles() <= 0.9 * CH && blocks() * b >= 512)
            break;
        if (sd[d] > 1) sd[d]--;
    }
    pl.rb = std::min(b, porder >= 7 && !poly ? 2 * RB : RB);
    while (pl.rb > 1 && (lds_b(pl.rb) > (sizeof(T) == 4 ? 80 : 155) * 1024 ||
                         blocks() * ceil_div(b, pl.rb) < 512))
        pl.rb--;
    pl.lds = lds_b(pl.rb);
    pl.rreg = (int)ceil_div(reg_of(), kIbThreads);
    return pl;
}

template <typename T>
void SpmeGpu<T>::interp(int b, double alpha, double beta, double* Y, hipStream_t s) {
    const int NC = poly ? 6 : 3;
    // alpha * K^3 / L^3 with the unnormalised inverse transform: alpha / L^3
    const double a_eff = alpha / (box * box * box);
    const int RB = 4;
    const int R = porder - 1;
    const SpmeTuning& tn = tune[width_class(b)];
    const InterpPlan pl = interp_plan(b);
    if (!pl.strips) {
        const int* sd = pl.sd;
        const int rbk = pl.rb, rreg = pl.rreg;
        const size_t lds = pl.lds;
        SDT_REQUIRE(rreg <= 19 && lds <= max_lds_bytes(), SDT_EINVAL, "interp: region too large");
        const int3 nb = make_int3(ceil_div(ntile, sd[0]), ceil_div(ntile, sd[1]), ceil_div(ntile, sd[2]));
        const dim3 grid(nb.x * nb.y * nb.z, ceil_div(b, rbk));
#define SDT_IB_R(PP, RR, PO)                                                                  \
    do {                                                                                      \
        allow_lds((const void*)interp_block_kernel<T, PP, RR, PO>, lds);                      \
        hipLaunchKernelGGL((interp_block_kernel<T, PP, RR, PO>), grid, dim3(kIbThreads), lds, s, K, \
                           ts, ntile, nb, make_int3(sd[0], sd[1], sd[2]), d_tile_start.get(), \
                           d_sten.get(), d_a2.get(), d_real.get(), b, rbk, a_eff, beta, Y);   \
    } while (0)
#define SDT_IB(PP)                                                                            \
    case PP:                                                                                  \
        if (rreg <= 8) { if (poly) SDT_IB_R(PP, 8, true); else SDT_IB_R(PP, 8, false); }      \
        else if (rreg <= 16) { if (poly) SDT_IB_R(PP, 16, true); else SDT_IB_R(PP, 16, false); } \
        else { if (poly) SDT_IB_R(PP, 19, true); else SDT_IB_R(PP, 19, false); }              \
        break;
        switch (porder) { SDT_IB(4) SDT_IB(5) SDT_IB(6) SDT_IB(7) SDT_IB(8) }
#undef SDT_IB
#undef SDT_IB_R
        SDT_HIP_CHECK(hipGetLastError());
        return;
    }
    // strip width (tiles along x) and particle chunk (measured at K = 128,
    // p = 6): FP32 4-tile strips, FP64 2-tile strips
    // interp_form > 0 overrides the meshes per pass (FP32 1, 2 or 4; FP64 1
    // or 2); one is fastest at K = 128, p = 6 in both precisions (the kernel
    // is bound by LDS reads, which wider vectors do not reduce)
    const int MV = interp_form > 0 ? interp_form : 1;
    SDT_REQUIRE(MV == 1 || MV == 2 || (MV == 4 && sizeof(T) == 4), SDT_EINVAL,
                "interp: meshes per pass must be 1, 2 or (FP32) 4");
    const int rlim = MV == 4 ? 16 : 26;
    int sxt = sizeof(T) == 8 ? 2 : 4, ch = sizeof(T) == 8 ? 64 : 128;
    if (tn.interp_sxt > 0) sxt = tn.interp_sxt;
    if (tn.interp_ch > 0) ch = tn.interp_ch;
    auto lds_of = [&](int sx, int c) {
        const size_t nreg = (size_t)(sx * ts + R) * (ts + R) * (ts + R);
        return nreg * MV * sizeof(T) + (size_t)c * porder * MV * sizeof(T) +
               (size_t)c * 3 * porder * sizeof(T) + (size_t)c * 3 * sizeof(int) + 8 +
               (size_t)c * RB * 3 * sizeof(double);
    };
    // narrower strips for wide stencils: the region must fit the prefetch
    // registers (26 points per thread)
    auto rreg_of = [&](int sx) {
        return (int)ceil_div((size_t)(sx * ts + R) * (ts + R) * (ts + R), 256);
    };
    while (rreg_of(sxt) > rlim && sxt > 1) sxt /= 2;
    while (lds_of(sxt, ch) > 80 * 1024 && (sxt > 1 || ch > 32)) {
        if (sxt > 1) sxt /= 2;
        else ch /= 2;
    }
    const size_t lds = lds_of(sxt, ch);
    SDT_REQUIRE(lds <= 80 * 1024, SDT_EINVAL, "interp: LDS region too large");
    const int nsx = (ntile + sxt - 1) / sxt;
    // region points per thread (registers of the prefetch)
    const int rreg = rreg_of(sxt);
    SDT_REQUIRE(rreg <= rlim, SDT_EINVAL, "interp: region too large for the prefetch registers");
    dim3 grid(nsx * ntile * ntile, ceil_div(b, RB));
#define SDT_INTERP_R(PP, RR)                                                                  \
    if (MV == 1) SDT_INTERP_M(PP, RR, 1);                                                     \
    else if (MV == 2) SDT_INTERP_M(PP, RR, 2);                                                \
    else if constexpr (sizeof(T) == 4) SDT_INTERP_M(PP, 16, 4);
#define SDT_INTERP_M(PP, RR, MM)                                                              \
    do {                                                                                      \
    allow_lds((const void*)interp_tile_kernel<T, PP, RR, MM>, lds);                            \
    hipLaunchKernelGGL((interp_tile_kernel<T, PP, RR, MM>), grid, dim3(256), lds, s, K, ts, ntile, \
                       nsx, sxt, ch, d_tile_start.get(), d_frac.get(), d_base.get(),              \
                       poly ? d_a2.get() : (double*)nullptr, d_real.get(), b, RB, NC, a_eff, beta, \
                       Y);                                                                \
    } while (0)
#define SDT_INTERP(PP)                                                                        \
    case PP:                                                                                  \
        if (rreg <= 16) { SDT_INTERP_R(PP, 16); }                                             \
        else { SDT_INTERP_R(PP, 26); }                                                        \
        break;
    switch (porder) { SDT_INTERP(4) SDT_INTERP(5) SDT_INTERP(6) SDT_INTERP(7) SDT_INTERP(8) }
#undef SDT_INTERP_R
#undef SDT_INTERP_M
#undef SDT_INTERP
    SDT_HIP_CHECK(hipGetLastError());
}

template <typename T>
void SpmeGpu<T>::apply(int b, double alpha, const double* X, double beta, double* Y,
                       hipStream_t s, T* xb, bool fill_xb) {
    reserve_rhs(b);
    {
        StageScope sc(timer, 0, s, b);
        if (fill_xb) real_block_copy<T>(npos, b, X, xb, s);
        spread(b, X, s, xb);
    }
    { StageScope sc(timer, 1, s, b); fft_forward(b, s); }
    { StageScope sc(timer, 2, s, b); influence(b, s); }
    { StageScope sc(timer, 3, s, b); fft_backward(b, s); }
    { StageScope sc(timer, 4, s, b); interp(b, alpha, beta, Y, s); }
}

template struct SpmeGpu<float>;
template struct SpmeGpu<double>;

}  // namespace sdt
