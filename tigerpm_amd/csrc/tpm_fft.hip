// tpm_fft.hip -- 3-D real FFTs of cubic meshes whose size is a power of two
// (16 .. 1024) or has a prime factor that rocFFT has no kernel for, LDS-tiled, in the layouts of fft3d_execute / fft3d_inv_execute
// (fft.cpp:51-84): R2C unnormalised, C2R unnormalised (the PM folds 1/M^3
// into its Green's function, fft.cpp:468, 512).
//
//   real  r[ix][iy][iz]           M^3 floats, iz fastest
//   spec  S[kx][ky][kz]           M * M * H complex, H = M/2 + 1, kz fastest
//   work  A[ix][kz][iy]           M * H * M complex, iy fastest
//   work  B[kz][ky][ix]           H * M * M complex, ix fastest
//
// Forward:  r --Z--> A --Y--> B --X--> S       (A in the output buffer)
// Inverse:  S --X'-> B --Y'-> A --Z'-> r       (A in the input buffer)
//
// Every pass reads and writes each element once: a workgroup loads T whole
// rows of its input (each row contiguous in memory), transforms them in LDS
// and writes T-element runs of its output, so the transposes that put the
// next pass's rows in contiguous memory are part of the pass.  Z and Z' make
// a real row of M points from a complex transform of M/2 points
// (z_n = x_2n + i x_2n+1) with the usual split of even and odd parts.
//
// The 1-D transforms are Stockham autosort FFTs (radix 8, 4 and 2 stages;
// each stage reads its butterflies' inputs from LDS, twiddles, applies the
// radix-R DFT and writes the outputs at their autosorted places), the
// twiddles read from a table e^{-2 pi i q / M} built in FP64.  The LDS tile
// holds T transforms with element (t, idx) at idx*T + (t ^ (idx % T)): rows
// of T consecutive t are whole bank rows, and the xor spreads a single
// transform's consecutive elements over the banks when rows are loaded.
#include <algorithm>
#include <cmath>
#include <vector>

#include "tpm_internal.hpp"

namespace {

constexpr int FFT_THREADS = 256;

constexpr int ilog2c(int v) { return v <= 1 ? 0 : 1 + ilog2c(v >> 1); }

__device__ __forceinline__ float2 cadd(float2 a, float2 b) { return make_float2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ float2 csub(float2 a, float2 b) { return make_float2(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ float2 cmul(float2 a, float2 b) {
    return make_float2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
__device__ __forceinline__ float2 conjc(float2 a) { return make_float2(a.x, -a.y); }
// a * (DIR i)
template <int DIR>
__device__ __forceinline__ float2 mul_i(float2 a) {
    return DIR < 0 ? make_float2(a.y, -a.x) : make_float2(-a.y, a.x);
}

// In-place DFTs of radix 2, 4, 8 with kernel e^{DIR 2 pi i r k / R},
// natural order in and out.
template <int R, int DIR>
struct Dft;

template <int DIR>
struct Dft<2, DIR> {
    static __device__ __forceinline__ void run(float2* v) {
        const float2 a = v[0];
        v[0] = cadd(a, v[1]);
        v[1] = csub(a, v[1]);
    }
};

template <int DIR>
__device__ __forceinline__ void dft4(float2& a0, float2& a1, float2& a2, float2& a3) {
    const float2 t0 = cadd(a0, a2), t1 = csub(a0, a2), t2 = cadd(a1, a3), t3 = mul_i<DIR>(csub(a1, a3));
    a0 = cadd(t0, t2);
    a1 = cadd(t1, t3);
    a2 = csub(t0, t2);
    a3 = csub(t1, t3);
}

template <int DIR>
struct Dft<4, DIR> {
    static __device__ __forceinline__ void run(float2* v) { dft4<DIR>(v[0], v[1], v[2], v[3]); }
};

template <int DIR>
struct Dft<8, DIR> {
    static __device__ __forceinline__ void run(float2* v) {
        // even and odd halves by radix 4, then y_k = E_k + w^k O_k and
        // y_k+4 = E_k - w^k O_k with w = e^{DIR 2 pi i / 8}
        float2 e0 = v[0], e1 = v[2], e2 = v[4], e3 = v[6];
        float2 o0 = v[1], o1 = v[3], o2 = v[5], o3 = v[7];
        dft4<DIR>(e0, e1, e2, e3);
        dft4<DIR>(o0, o1, o2, o3);
        const float h = 0.70710678118654752f;
        const float d = (float)DIR;
        o1 = make_float2(h * (o1.x - d * o1.y), h * (o1.y + d * o1.x));    // (1 + DIR i) / sqrt 2
        o2 = mul_i<DIR>(o2);                                                // DIR i
        o3 = make_float2(h * (-o3.x - d * o3.y), h * (-o3.y + d * o3.x));  // (-1 + DIR i) / sqrt 2
        v[0] = cadd(e0, o0);
        v[4] = csub(e0, o0);
        v[1] = cadd(e1, o1);
        v[5] = csub(e1, o1);
        v[2] = cadd(e2, o2);
        v[6] = csub(e2, o2);
        v[3] = cadd(e3, o3);
        v[7] = csub(e3, o3);
    }
};

template <int T>
__device__ __forceinline__ int lds_at(int t, int idx) {
    return idx * T + (t ^ (idx & (T - 1)));
}

// f(e) for e = threadIdx.x + 256 u < COUNT, fully unrolled, so that a
// phase's global loads are all in flight before the first wait.
template <int COUNT, class F>
__device__ __forceinline__ void for_each_elem(F f) {
    constexpr int NU = (COUNT + FFT_THREADS - 1) / FFT_THREADS;
#pragma unroll
    for (int u = 0; u < NU; u++) {
        const int e = (int)threadIdx.x + FFT_THREADS * u;
        if (COUNT % FFT_THREADS == 0 || e < COUNT) f(e);
    }
}

// Loads for e < COUNT into registers, then stores: every load of the phase
// is issued before any result is used.
template <int COUNT, class L, class S>
__device__ __forceinline__ void move_elems(L load, S store) {
    constexpr int NU = (COUNT + FFT_THREADS - 1) / FFT_THREADS;
    float2 v[NU];
#pragma unroll
    for (int u = 0; u < NU; u++) {
        const int e = (int)threadIdx.x + FFT_THREADS * u;
        if (COUNT % FFT_THREADS == 0 || e < COUNT) v[u] = load(e);
    }
#pragma unroll
    for (int u = 0; u < NU; u++) {
        const int e = (int)threadIdx.x + FFT_THREADS * u;
        if (COUNT % FFT_THREADS == 0 || e < COUNT) store(e, v[u]);
    }
}

// One Stockham stage of radix R over T transforms of length L whose first
// Ns-point sub-transforms are done: butterfly j (k = j mod Ns) takes
// x[j + r L/R] times e^{DIR 2 pi i r k / (Ns R)} and writes the R-point DFT
// to y[(j - k) R + k + r Ns].  Twiddles come from tf[q] = e^{-2 pi i q / M},
// M = L * SCALE.
template <int L, int T, int R, int Ns, int DIR, int SCALE>
__device__ __forceinline__ void fft_stage(float2* s, const float2* __restrict__ tf) {
    constexpr int NB = T * L / R;
    constexpr int NV = (NB + FFT_THREADS - 1) / FFT_THREADS;
    const int tid = (int)threadIdx.x;
    float2 v[NV][R];
#pragma unroll
    for (int u = 0; u < NV; u++) {
        const int b = tid + FFT_THREADS * u;
        if (NB % FFT_THREADS == 0 || b < NB) {
            const int t = b % T, j = b / T;
            const int k = j & (Ns - 1);
#pragma unroll
            for (int r = 0; r < R; r++) v[u][r] = s[lds_at<T>(t, j + r * (L / R))];
            if (Ns > 1) {
#pragma unroll
                for (int r = 1; r < R; r++) {
                    const float2 w = tf[r * k * (L / (Ns * R)) * SCALE];
                    v[u][r] = cmul(v[u][r], DIR < 0 ? w : conjc(w));
                }
            }
            Dft<R, DIR>::run(v[u]);
        }
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < NV; u++) {
        const int b = tid + FFT_THREADS * u;
        if (NB % FFT_THREADS == 0 || b < NB) {
            const int t = b % T, j = b / T;
            const int k = j & (Ns - 1);
            const int i0 = (j - k) * R + k;
#pragma unroll
            for (int r = 0; r < R; r++) s[lds_at<T>(t, i0 + r * Ns)] = v[u][r];
        }
    }
    __syncthreads();
}

// All stages: radix 8 while at least 8 points remain, except that 16 points
// go as 4 x 4 and 4 points as one radix-4 stage, 2 as radix 2.
template <int L, int T, int DIR, int SCALE, int Ns = 1>
__device__ __forceinline__ void fft_rows(float2* s, const float2* __restrict__ tf) {
    if constexpr (Ns < L) {
        constexpr int rem = ilog2c(L / Ns);
        constexpr int R = rem == 1 ? 2 : (rem == 2 || rem == 4) ? 4 : 8;
        fft_stage<L, T, R, Ns, DIR, SCALE>(s, tf);
        fft_rows<L, T, DIR, SCALE, Ns * R>(s, tf);
    }
}

// Z: real rows r[ix][iy0 + t][*] -> A[ix][kz][iy0 + t].  Grid M * (M / T).
// With Q32 the rows are the integer density grid (unit masses times 2^32,
// 16-byte aligned), converted as float(double(q) 2^-32) on the way in.
template <int M, int T, bool Q32>
__global__ __launch_bounds__(FFT_THREADS) void fft_z_r2c_kernel(const void* __restrict__ in, float2* __restrict__ A,
                                                               const float2* __restrict__ tf) {
    constexpr int N = M / 2, H = N + 1;
    __shared__ float2 s[T * N];
    const int iy0 = (int)(blockIdx.x % (M / T)) * T;
    const int64_t ix = blockIdx.x / (M / T);
    const int64_t row0 = (ix * M + iy0) * M;
    const float* src = static_cast<const float*>(in) + row0;
    const ulonglong2* qsrc = reinterpret_cast<const ulonglong2*>(static_cast<const unsigned long long*>(in) + row0);
    const bool aligned = (reinterpret_cast<uintptr_t>(src) & 7) == 0;
    move_elems<T * N>(
        [&](int e) {
            if (Q32) {
                const ulonglong2 q = qsrc[e];
                return make_float2((float)((double)q.x * 0x1p-32), (float)((double)q.y * 0x1p-32));
            }
            if (aligned) return reinterpret_cast<const float2*>(src)[e];
            return make_float2(src[2 * e], src[2 * e + 1]);
        },
        [&](int e, float2 v) { s[lds_at<T>(e / N, e % N)] = v; });
    __syncthreads();
    fft_rows<N, T, -1, 2>(s, tf);
    // X_k = (Z_k + conj Z_N-k) / 2 - i W^k (Z_k - conj Z_N-k) / 2, W = e^{-2 pi i / M}
    float2* dst = A + ix * H * M + iy0;
    for_each_elem<T * H>([&](int e) {
        const int k = e / T, t = e % T;
        const float2 a = s[lds_at<T>(t, k & (N - 1))];
        const float2 b = conjc(s[lds_at<T>(t, (N - k) & (N - 1))]);
        const float2 ev = make_float2(0.5f * (a.x + b.x), 0.5f * (a.y + b.y));
        const float2 od = mul_i<-1>(make_float2(0.5f * (a.x - b.x), 0.5f * (a.y - b.y)));
        dst[(int64_t)k * M + t] = cadd(ev, cmul(tf[k & (M - 1)], od));
    });
}

// Z': A[ix][kz][iy0 + t] -> real rows r[ix][iy0 + t][*].  Grid M * (M / T).
template <int M, int T>
__global__ __launch_bounds__(FFT_THREADS) void fft_z_c2r_kernel(const float2* __restrict__ A, float* __restrict__ out,
                                                               const float2* __restrict__ tf) {
    constexpr int N = M / 2, H = N + 1;
    constexpr int NV = (T * N + FFT_THREADS - 1) / FFT_THREADS;
    __shared__ float2 s[T * H];
    const int tid = (int)threadIdx.x;
    const int iy0 = (int)(blockIdx.x % (M / T)) * T;
    const int64_t ix = blockIdx.x / (M / T);
    const float2* src = A + ix * H * M + iy0;
    move_elems<T * H>([&](int e) { return src[(int64_t)(e / T) * M + e % T]; },
                      [&](int e, float2 v) { s[lds_at<T>(e % T, e / T)] = v; });
    __syncthreads();
    // Z'_k = (X_k + conj X_N-k) + i (X_k - conj X_N-k) conj(W^k), k < N;
    // the inverse N-point transform of Z' is x_2n + i x_2n+1 times M
    float2 z[NV];
#pragma unroll
    for (int u = 0; u < NV; u++) {
        const int e = tid + FFT_THREADS * u;
        if ((T * N) % FFT_THREADS == 0 || e < T * N) {
            const int k = e / T, t = e % T;
            const float2 a = s[lds_at<T>(t, k)];
            const float2 b = conjc(s[lds_at<T>(t, N - k)]);
            z[u] = cadd(cadd(a, b), mul_i<1>(cmul(csub(a, b), conjc(tf[k]))));
        }
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < NV; u++) {
        const int e = tid + FFT_THREADS * u;
        if ((T * N) % FFT_THREADS == 0 || e < T * N) s[lds_at<T>(e % T, e / T)] = z[u];
    }
    __syncthreads();
    fft_rows<N, T, 1, 2>(s, tf);
    float* dst = out + (ix * M + iy0) * M;
    const bool aligned = (reinterpret_cast<uintptr_t>(dst) & 7) == 0;
    for_each_elem<T * N>([&](int e) {
        const float2 v = s[lds_at<T>(e / N, e % N)];
        if (aligned) {
            reinterpret_cast<float2*>(dst)[e] = v;
        } else {
            dst[2 * e] = v.x;
            dst[2 * e + 1] = v.y;
        }
    });
}

// Y (FWD): A[ix0 + t][kz][*] -> B[kz][ky][ix0 + t];  Y' (!FWD): the reverse.
// Grid H * (M / T).
template <int M, int T, bool FWD>
__global__ __launch_bounds__(FFT_THREADS) void fft_y_kernel(const float2* __restrict__ in, float2* __restrict__ out,
                                                           const float2* __restrict__ tf) {
    constexpr int H = M / 2 + 1;
    __shared__ float2 s[T * M];
    const int ix0 = (int)(blockIdx.x % (M / T)) * T;
    const int64_t kz = blockIdx.x / (M / T);
    if (FWD)
        move_elems<T * M>([&](int e) { return in[((int64_t)(ix0 + e / M) * H + kz) * M + e % M]; },
                          [&](int e, float2 v) { s[lds_at<T>(e / M, e % M)] = v; });
    else
        move_elems<T * M>([&](int e) { return in[(kz * M + e / T) * M + ix0 + e % T]; },
                          [&](int e, float2 v) { s[lds_at<T>(e % T, e / T)] = v; });
    __syncthreads();
    fft_rows<M, T, FWD ? -1 : 1, 1>(s, tf);
    if (FWD)
        for_each_elem<T * M>([&](int e) { out[(kz * M + e / T) * M + ix0 + e % T] = s[lds_at<T>(e % T, e / T)]; });
    else
        for_each_elem<T * M>(
            [&](int e) { out[((int64_t)(ix0 + e / M) * H + kz) * M + e % M] = s[lds_at<T>(e / M, e % M)]; });
}

// X (FWD): B[kz0 + t][ky][*] -> S[kx][ky][kz0 + t];  X' (!FWD): the reverse.
// Grid M * ceil(H / T); rows past kz = M/2 are zeros and not stored.  With
// a Green's table g (FWD only, layout of S) each stored mode is g times the
// transform, as a separate multiply pass would make it.
template <int M, int T, bool FWD>
__global__ __launch_bounds__(FFT_THREADS) void fft_x_kernel(const float2* __restrict__ in, float2* __restrict__ out,
                                                           const float2* __restrict__ tf,
                                                           const float* __restrict__ g = nullptr) {
    constexpr int H = M / 2 + 1;
    constexpr int NKT = (H + T - 1) / T;
    __shared__ float2 s[T * M];
    const int kz0 = (int)(blockIdx.x % NKT) * T;
    const int64_t ky = blockIdx.x / NKT;
    const int tn = min(T, H - kz0);
    const float2 zero = make_float2(0.f, 0.f);
    // the Green's factors of this thread's stored modes, loaded before any
    // store (a load issued after stores waits for them too)
    constexpr int NU = T * M / FFT_THREADS;
    static_assert(T * M % FFT_THREADS == 0, "whole tiles per thread");
    float gv[FWD ? NU : 1];
    if (FWD && g) {
#pragma unroll
        for (int u = 0; u < NU; u++) {
            const int e = (int)threadIdx.x + FFT_THREADS * u;
            gv[u] = e % T < tn ? g[((int64_t)(e / T) * M + ky) * H + kz0 + e % T] : 0.f;
        }
    }
    if (FWD)
        move_elems<T * M>(
            [&](int e) { return e / M < tn ? in[((int64_t)(kz0 + e / M) * M + ky) * M + e % M] : zero; },
            [&](int e, float2 v) { s[lds_at<T>(e / M, e % M)] = v; });
    else
        move_elems<T * M>(
            [&](int e) { return e % T < tn ? in[((int64_t)(e / T) * M + ky) * H + kz0 + e % T] : zero; },
            [&](int e, float2 v) { s[lds_at<T>(e % T, e / T)] = v; });
    __syncthreads();
    fft_rows<M, T, FWD ? -1 : 1, 1>(s, tf);
    if (FWD) {
#pragma unroll
        for (int u = 0; u < NU; u++) {
            const int e = (int)threadIdx.x + FFT_THREADS * u;
            if (e % T < tn) {
                float2 v = s[lds_at<T>(e % T, e / T)];
                if (g) {
                    v.x *= gv[u];
                    v.y *= gv[u];
                }
                out[((int64_t)(e / T) * M + ky) * H + kz0 + e % T] = v;
            }
        }
    }
    else
        for_each_elem<T * M>([&](int e) {
            if (e / M < tn) out[((int64_t)(kz0 + e / M) * M + ky) * M + e % M] = s[lds_at<T>(e / M, e % M)];
        });
}

// X, Green's multiply and X' in one pass, in place on B (the PM's Poisson
// solve): the rows B[kz0 + t][ky][*] go forward along x, each mode (kx, ky,
// kz0 + t) is multiplied by its Green's factor, and the rows go back.  The
// same float operations as X, a Green's pass and X', without storing S.
// gt is the table regrouped by green_tiles_kernel: workgroup w reads the
// T * M factors gt[w * T * M ...] in one contiguous run.
// Grid M * ceil(H / T).
template <int M, int T>
__global__ __launch_bounds__(FFT_THREADS) void fft_xgx_kernel(float2* __restrict__ b, const float2* __restrict__ tf,
                                                             const float* __restrict__ gt) {
    constexpr int H = M / 2 + 1;
    constexpr int NKT = (H + T - 1) / T;
    constexpr int NU = T * M / FFT_THREADS;
    static_assert(T * M % FFT_THREADS == 0, "whole tiles per thread");
    __shared__ float2 s[T * M];
    const int kz0 = (int)(blockIdx.x % NKT) * T;
    const int64_t ky = blockIdx.x / NKT;
    const int tn = min(T, H - kz0);
    float gv[NU];
#pragma unroll
    for (int u = 0; u < NU; u++) gv[u] = gt[(int64_t)blockIdx.x * (T * M) + threadIdx.x + FFT_THREADS * u];
    move_elems<T * M>(
        [&](int e) {
            return e / M < tn ? b[((int64_t)(kz0 + e / M) * M + ky) * M + e % M] : make_float2(0.f, 0.f);
        },
        [&](int e, float2 v) { s[lds_at<T>(e / M, e % M)] = v; });
    __syncthreads();
    fft_rows<M, T, -1, 1>(s, tf);
#pragma unroll
    for (int u = 0; u < NU; u++) {
        const int e = (int)threadIdx.x + FFT_THREADS * u;
        float2& v = s[lds_at<T>(e % T, e / T)];
        v.x *= gv[u];
        v.y *= gv[u];
    }
    __syncthreads();
    fft_rows<M, T, 1, 1>(s, tf);
    for_each_elem<T * M>([&](int e) {
        if (e / M < tn) b[((int64_t)(kz0 + e / M) * M + ky) * M + e % M] = s[lds_at<T>(e / M, e % M)];
    });
}

#ifndef TPM_FFT_TILE
#define TPM_FFT_TILE 16
#endif
template <int M>
constexpr int tile_of() {
    return M * TPM_FFT_TILE <= 8192 ? TPM_FFT_TILE : 8192 / M;  // T * M complex <= 64 KiB of LDS
}

// Rows per workgroup of the fused x pass.  Its loads and stores are whole
// rows of B whatever T is, so T only sets the LDS per workgroup: with 4 rows
// (16 KiB at M = 512) eight workgroups share a CU, against two at 16 rows
// (64 KiB), and the pass takes 0.29 instead of 0.69 ms at M = 512 (8 rows:
// 0.30 ms).
#ifndef TPM_FFT_XGX_TILE
#define TPM_FFT_XGX_TILE 4
#endif
template <int M>
constexpr int xgx_tile_of() {
    constexpr int t = M * TPM_FFT_XGX_TILE <= 8192 ? TPM_FFT_XGX_TILE : 8192 / M;
    return t * M < FFT_THREADS ? FFT_THREADS / M : t;
}

// The Green's table (layout of S: [kx][ky][kz], kz < H) regrouped for
// fft_xgx_kernel: the factors of its workgroup w = ky * NKT + kz tile, in the
// order e = kx * T + t its threads use, zeros past kz = M/2.  The values are
// copied, not recomputed.
template <int M>
__global__ void green_tiles_kernel(const float* __restrict__ g, float* __restrict__ gt) {
    constexpr int T = xgx_tile_of<M>(), H = M / 2 + 1, NKT = (H + T - 1) / T;
    const int64_t total = (int64_t)M * NKT * T * M;
    for (int64_t l = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; l < total; l += (int64_t)gridDim.x * blockDim.x) {
        const int e = (int)(l % (T * M));
        const int64_t w = l / (T * M);
        const int kz = (int)(w % NKT) * T + e % T;
        const int64_t ky = w / NKT;
        gt[l] = kz < H ? g[((int64_t)(e / T) * M + ky) * H + kz] : 0.f;
    }
}

template <int M>
int64_t green_tiles(hipStream_t st, const float* g, float* gt) {
    constexpr int T = xgx_tile_of<M>(), H = M / 2 + 1;
    const int64_t n = (int64_t)M * ((H + T - 1) / T) * T * M;
    if (gt) green_tiles_kernel<M><<<(unsigned)std::min<int64_t>((n + 255) / 256, 65536), 256, 0, st>>>(g, gt);
    return n;
}

template <int M>
void launch_r2c(hipStream_t st, const void* in, bool q32, float2* out, float2* work, const float2* tf,
                const float* green) {
    constexpr int T = tile_of<M>(), H = M / 2 + 1;
    if (q32)
        fft_z_r2c_kernel<M, T, true><<<M * (M / T), FFT_THREADS, 0, st>>>(in, out, tf);
    else
        fft_z_r2c_kernel<M, T, false><<<M * (M / T), FFT_THREADS, 0, st>>>(in, out, tf);
    fft_y_kernel<M, T, true><<<H * (M / T), FFT_THREADS, 0, st>>>(out, work, tf);
    fft_x_kernel<M, T, true><<<M * ((H + T - 1) / T), FFT_THREADS, 0, st>>>(work, out, tf, green);
}

template <int M>
void launch_c2r(hipStream_t st, float2* in, float* out, float2* work, const float2* tf) {
    constexpr int T = tile_of<M>(), H = M / 2 + 1;
    fft_x_kernel<M, T, false><<<M * ((H + T - 1) / T), FFT_THREADS, 0, st>>>(in, work, tf);
    fft_y_kernel<M, T, false><<<H * (M / T), FFT_THREADS, 0, st>>>(work, in, tf);
    fft_z_c2r_kernel<M, T><<<M * (M / T), FFT_THREADS, 0, st>>>(in, out, tf);
}

// The PM's Poisson solve: Q32 density -> phi through spec (A layout) and
// work (B layout), both M * M * (M/2 + 1) complex.
template <int M>
void launch_pm(hipStream_t st, const unsigned long long* q, float* phi, float2* spec, float2* work,
               const float2* tf, const float* green) {
    constexpr int T = tile_of<M>(), H = M / 2 + 1;
    fft_z_r2c_kernel<M, T, true><<<M * (M / T), FFT_THREADS, 0, st>>>(q, spec, tf);
    fft_y_kernel<M, T, true><<<H * (M / T), FFT_THREADS, 0, st>>>(spec, work, tf);
    constexpr int TX = xgx_tile_of<M>();
    fft_xgx_kernel<M, TX><<<M * ((H + TX - 1) / TX), FFT_THREADS, 0, st>>>(work, tf, green);
    fft_y_kernel<M, T, false><<<H * (M / T), FFT_THREADS, 0, st>>>(work, spec, tf);
    fft_z_c2r_kernel<M, T><<<M * (M / T), FFT_THREADS, 0, st>>>(spec, phi, tf);
}


// ---- Sizes with a larger prime factor (runtime M) ---------------------------
// The same passes and layouts for M = product of the plan's radices.  Z and
// Z' take two real rows as one complex row of M points, which needs no even
// M.  A stage reads one LDS buffer and writes the other; radices up to 8 go
// through registers, a larger prime p pairs its inputs r and p - r in place
// (sum and difference) and makes outputs m and p - m together from
// p / 2 terms each, so that a row costs p fused multiply-adds per point and
// component.  Bound by LDS reads: a thread makes NM outputs and their
// mirrors from each pair that it reads (Poisson solve of a 97^3 mesh: 1 output
// 171 us, 2 155, 4 143; with eight rows per workgroup instead of sixteen, whose
// smaller LDS lets more of them share a CU, 2 outputs 124, 4 139).  The
// terms are summed in blocks of SUM_BLK: a density's mean makes the partial
// sums of one long chain grow to p / 2 terms before they cancel, and its rounding
// is the PM force's error (97^3, rms of the force: one chain 8.5e-6, blocks of 8
// 4.2e-6, rocFFT 5.6e-6; no change in time, nor blocks of 4 or 6 in either).
constexpr int NM = 2;
constexpr int SUM_BLK = 8;
struct GenPlan {
    int M;
    int nstage;
    int radix[10];
};

__device__ __forceinline__ constexpr float odd_cos(int P, int q) {
    // cos(2 pi q / P), q <= P / 2
    constexpr float c3[2] = {1.f, -0.5f}, c5[3] = {1.f, 0.30901699437494742f, -0.80901699437494742f},
                    c7[4] = {1.f, 0.62348980185873353f, -0.22252093395631440f, -0.90096886790241913f};
    return P == 3 ? c3[q] : P == 5 ? c5[q] : c7[q];
}
__device__ __forceinline__ constexpr float odd_sin(int P, int q) {
    constexpr float s3[2] = {0.f, 0.86602540378443865f}, s5[3] = {0.f, 0.95105651629515357f, 0.58778525229247313f},
                    s7[4] = {0.f, 0.78183148246802981f, 0.97492791218182361f, 0.43388373911755812f};
    return P == 3 ? s3[q] : P == 5 ? s5[q] : s7[q];
}

// DFT of odd length P in registers.
template <int P, int DIR>
__device__ __forceinline__ void dft_odd(float2* v) {
    constexpr int Q = (P - 1) / 2;
    float2 a[Q], b[Q];
#pragma unroll
    for (int r = 0; r < Q; r++) {
        a[r] = cadd(v[r + 1], v[P - 1 - r]);
        b[r] = csub(v[r + 1], v[P - 1 - r]);
    }
    const float2 x0 = v[0];
#pragma unroll
    for (int r = 0; r < Q; r++) v[0] = cadd(v[0], a[r]);
#pragma unroll
    for (int m = 1; m <= Q; m++) {
        float2 c = x0, d = make_float2(0.f, 0.f);
#pragma unroll
        for (int r = 1; r <= Q; r++) {
            const int q = (r * m) % P;
            const float co = odd_cos(P, q > Q ? P - q : q);
            const float si = q > Q ? -odd_sin(P, P - q) : odd_sin(P, q);
            c.x = fmaf(a[r - 1].x, co, c.x);
            c.y = fmaf(a[r - 1].y, co, c.y);
            d.x = fmaf(b[r - 1].x, si, d.x);
            d.y = fmaf(b[r - 1].y, si, d.y);
        }
        d = mul_i<DIR>(d);
        v[m] = cadd(c, d);
        v[P - m] = csub(c, d);
    }
}

template <int R, int DIR>
__device__ __forceinline__ void dft_any(float2* v) {
    if constexpr (R == 2 || R == 4 || R == 8)
        Dft<R, DIR>::run(v);
    else
        dft_odd<R, DIR>(v);
}

// e / d for e d < 2^32, by the multiplier ceil(2^32 / d); d = 1 has none.
struct FastDiv {
    unsigned d, mul;
    __device__ explicit FastDiv(unsigned d_) : d(d_), mul(0xffffffffu / d_ + 1u) {}
    __device__ unsigned div(unsigned e) const { return d == 1 ? e : __umulhi(e, mul); }
};

template <int T, int R, int DIR>
__device__ __forceinline__ void gen_stage(const float2* __restrict__ x, float2* __restrict__ y,
                                          const float2* __restrict__ tw, int M, int Ns) {
    const int mr = M / R, ws = mr / Ns;
    const FastDiv ns((unsigned)Ns);
    for (int b = (int)threadIdx.x; b < T * mr; b += FFT_THREADS) {
        const int t = b % T, j = b / T;
        const int k = j - (int)ns.div((unsigned)j) * Ns;
        float2 v[R];
#pragma unroll
        for (int r = 0; r < R; r++) v[r] = x[lds_at<T>(t, j + r * mr)];
        if (Ns > 1) {
#pragma unroll
            for (int r = 1; r < R; r++) {
                const float2 w = tw[r * k * ws];
                v[r] = cmul(v[r], DIR < 0 ? w : conjc(w));
            }
        }
        dft_any<R, DIR>(v);
        const int i0 = (j - k) * R + k;
#pragma unroll
        for (int r = 0; r < R; r++) y[lds_at<T>(t, i0 + r * Ns)] = v[r];
    }
}

// A prime p > 7; x is overwritten.  A thread makes NM outputs m and their
// mirrors p - m from each pair of inputs that it reads.
template <int T, int DIR>
__device__ __forceinline__ void gen_stage_prime(float2* __restrict__ x, float2* __restrict__ y,
                                                const float2* __restrict__ tw, int M, int Ns, int p) {
    const int mr = M / p, ws = mr / Ns, Q = (p - 1) / 2;
    const FastDiv ns((unsigned)Ns), dm((unsigned)mr);
    for (int b = (int)threadIdx.x; b < T * mr * Q; b += FFT_THREADS) {
        const int t = b % T, c = b / T;
        const int r0 = (int)dm.div((unsigned)c), j = c - r0 * mr, r = r0 + 1;
        const int i1 = lds_at<T>(t, j + r * mr), i2 = lds_at<T>(t, j + (p - r) * mr);
        float2 u = x[i1], v = x[i2];
        if (Ns > 1) {
            const int k = j - (int)ns.div((unsigned)j) * Ns;
            const float2 w1 = tw[r * k * ws], w2 = tw[(p - r) * k * ws];
            u = cmul(u, DIR < 0 ? w1 : conjc(w1));
            v = cmul(v, DIR < 0 ? w2 : conjc(w2));
        }
        x[i1] = cadd(u, v);
        x[i2] = csub(u, v);
    }
    __syncthreads();
    const int mg = (Q + NM) / NM;  // groups of the Q + 1 outputs m <= Q
    for (int b = (int)threadIdx.x; b < T * mr * mg; b += FFT_THREADS) {
        const int t = b % T, e = b / T;
        const int g = (int)dm.div((unsigned)e), j = e - g * mr;
        const int k = j - (int)ns.div((unsigned)j) * Ns;
        const float2 x0 = x[lds_at<T>(t, j)];
        float2 c[NM], d[NM];
        int m[NM], q[NM], i1 = j, i2 = j + M;
#pragma unroll
        for (int u = 0; u < NM; u++) {
            c[u] = x0;
            d[u] = make_float2(0.f, 0.f);
            m[u] = min(g * NM + u, Q);  // past the last: it again
            q[u] = 0;
        }
        for (int r0 = 1; r0 <= Q; r0 += SUM_BLK) {
            float2 cb[NM], db[NM];
#pragma unroll
            for (int u = 0; u < NM; u++) cb[u] = db[u] = make_float2(0.f, 0.f);
            const int r1 = min(r0 + SUM_BLK, Q + 1);
#pragma unroll 2
            for (int r = r0; r < r1; r++) {
                i1 += mr;
                i2 -= mr;
                const float2 xa = x[lds_at<T>(t, i1)], xb = x[lds_at<T>(t, i2)];
#pragma unroll
                for (int u = 0; u < NM; u++) {
                    q[u] += m[u];
                    q[u] -= q[u] >= p ? p : 0;
                    const float2 w = tw[q[u] * mr];
                    cb[u].x = fmaf(xa.x, w.x, cb[u].x);
                    cb[u].y = fmaf(xa.y, w.x, cb[u].y);
                    db[u].x = fmaf(xb.x, -w.y, db[u].x);
                    db[u].y = fmaf(xb.y, -w.y, db[u].y);
                }
            }
#pragma unroll
            for (int u = 0; u < NM; u++) {
                c[u] = cadd(c[u], cb[u]);
                d[u] = cadd(d[u], db[u]);
            }
        }
        const int i0 = (j - k) * p + k;
#pragma unroll
        for (int u = 0; u < NM; u++) {
            const float2 di = mul_i<DIR>(d[u]);
            y[lds_at<T>(t, i0 + m[u] * Ns)] = cadd(c[u], di);
            if (m[u] > 0) y[lds_at<T>(t, i0 + (p - m[u]) * Ns)] = csub(c[u], di);
        }
    }
}

// The T rows of length M in s (s2: a second buffer); returns the buffer that
// holds the result.  Begins and ends with a barrier.
template <int T, int DIR>
__device__ __forceinline__ float2* gen_rows(float2* s, float2* s2, const float2* tw, const GenPlan& P) {
    int Ns = 1;
    __syncthreads();
    for (int i = 0; i < P.nstage; i++) {
        const int R = P.radix[i];
        switch (R) {
            case 2: gen_stage<T, 2, DIR>(s, s2, tw, P.M, Ns); break;
            case 3: gen_stage<T, 3, DIR>(s, s2, tw, P.M, Ns); break;
            case 4: gen_stage<T, 4, DIR>(s, s2, tw, P.M, Ns); break;
            case 5: gen_stage<T, 5, DIR>(s, s2, tw, P.M, Ns); break;
            case 7: gen_stage<T, 7, DIR>(s, s2, tw, P.M, Ns); break;
            case 8: gen_stage<T, 8, DIR>(s, s2, tw, P.M, Ns); break;
            default: gen_stage_prime<T, DIR>(s, s2, tw, P.M, Ns, R); break;
        }
        Ns *= R;
        float2* const t = s;
        s = s2;
        s2 = t;
        __syncthreads();
    }
    return s;
}

__device__ __forceinline__ void gen_twiddles(float2* tw, const float2* __restrict__ tf, int M) {
    for (int q = (int)threadIdx.x; q < M; q += FFT_THREADS) tw[q] = tf[q];
}

extern __shared__ __align__(16) float2 gen_lds[];

// Z: real rows r[ix][iy0 + 0 .. 2T)[*], a pair per complex row.  Grid
// M * ceil(M / 2T).
template <int T>
__global__ __launch_bounds__(FFT_THREADS) void gen_z_r2c_kernel(const float* __restrict__ in, float2* __restrict__ A,
                                                               const float2* __restrict__ tf, GenPlan P) {
    const int M = P.M, H = M / 2 + 1, nt = (M + 2 * T - 1) / (2 * T);
    float2 *s = gen_lds, *s2 = s + T * M, *tw = s2 + T * M;
    const int64_t ix = blockIdx.x / nt;
    const int iy0 = (int)(blockIdx.x % nt) * 2 * T, tn = min(2 * T, M - iy0);
    const float* src = in + (ix * M + iy0) * M;
    const FastDiv dm((unsigned)M);
    gen_twiddles(tw, tf, M);
#pragma unroll 4
    for (int e = (int)threadIdx.x; e < 2 * T * M; e += FFT_THREADS) {
        const int row = (int)dm.div((unsigned)e), i = e - row * M;
        const float v = row < tn ? src[e] : 0.f;
        reinterpret_cast<float*>(&s[lds_at<T>(row >> 1, i)])[row & 1] = v;
    }
    const float2* z = gen_rows<T, -1>(s, s2, tw, P);
    float2* dst = A + ix * H * M + iy0;
    for (int e = (int)threadIdx.x; e < 2 * T * H; e += FFT_THREADS) {
        const int k = e / (2 * T), tt = e % (2 * T);
        if (tt >= tn) continue;
        const float2 a = z[lds_at<T>(tt >> 1, k)], b = conjc(z[lds_at<T>(tt >> 1, k ? M - k : 0)]);
        // first row (a + b) / 2, second (a - b) / 2i
        const float2 d = tt & 1 ? mul_i<-1>(csub(a, b)) : cadd(a, b);
        dst[(int64_t)k * M + tt] = make_float2(0.5f * d.x, 0.5f * d.y);
    }
}

// Z': the reverse.  The imaginary parts of modes 0 and M / 2, which a real
// row does not have, are left out.
template <int T>
__global__ __launch_bounds__(FFT_THREADS) void gen_z_c2r_kernel(const float2* __restrict__ A, float* __restrict__ out,
                                                               const float2* __restrict__ tf, GenPlan P) {
    const int M = P.M, H = M / 2 + 1, nt = (M + 2 * T - 1) / (2 * T);
    float2 *s = gen_lds, *s2 = s + T * M, *tw = s2 + T * M;
    const int64_t ix = blockIdx.x / nt;
    const int iy0 = (int)(blockIdx.x % nt) * 2 * T, tn = min(2 * T, M - iy0);
    const float2* src = A + ix * H * M + iy0;
    gen_twiddles(tw, tf, M);
#pragma unroll 4
    for (int e = (int)threadIdx.x; e < T * H; e += FFT_THREADS) {
        const int k = e / T, t = e % T;
        const float2 zero = make_float2(0.f, 0.f);
        float2 a = 2 * t < tn ? src[(int64_t)k * M + 2 * t] : zero;
        float2 b = 2 * t + 1 < tn ? src[(int64_t)k * M + 2 * t + 1] : zero;
        const int mk = k ? M - k : 0;
        if (mk == k) a.y = b.y = 0.f;
        s[lds_at<T>(t, k)] = make_float2(a.x - b.y, a.y + b.x);
        if (mk != k) s[lds_at<T>(t, mk)] = make_float2(a.x + b.y, b.x - a.y);
    }
    const float2* z = gen_rows<T, 1>(s, s2, tw, P);
    float* dst = out + (ix * M + iy0) * M;
    const FastDiv dm((unsigned)M);
    for (int e = (int)threadIdx.x; e < tn * M; e += FFT_THREADS) {
        const int row = (int)dm.div((unsigned)e), i = e - row * M;
        dst[e] = reinterpret_cast<const float*>(&z[lds_at<T>(row >> 1, i)])[row & 1];
    }
}

// Y (FWD): A[ix0 + t][kz][*] -> B[kz][ky][ix0 + t];  Y' (!FWD): the reverse.
// Grid H * ceil(M / T).
template <int T, bool FWD>
__global__ __launch_bounds__(FFT_THREADS) void gen_y_kernel(const float2* __restrict__ in, float2* __restrict__ out,
                                                           const float2* __restrict__ tf, GenPlan P) {
    const int M = P.M, H = M / 2 + 1, nt = (M + T - 1) / T;
    float2 *s = gen_lds, *s2 = s + T * M, *tw = s2 + T * M;
    const int64_t kz = blockIdx.x / nt;
    const int ix0 = (int)(blockIdx.x % nt) * T, tn = min(T, M - ix0);
    const FastDiv dm((unsigned)M);
    const float2 zero = make_float2(0.f, 0.f);
    gen_twiddles(tw, tf, M);
#pragma unroll 4
    for (int e = (int)threadIdx.x; e < T * M; e += FFT_THREADS) {
        if (FWD) {
            const int t = (int)dm.div((unsigned)e), i = e - t * M;
            s[lds_at<T>(t, i)] = t < tn ? in[((int64_t)(ix0 + t) * H + kz) * M + i] : zero;
        } else {
            const int i = e / T, t = e % T;
            s[lds_at<T>(t, i)] = t < tn ? in[(kz * M + i) * M + ix0 + t] : zero;
        }
    }
    const float2* z = gen_rows<T, FWD ? -1 : 1>(s, s2, tw, P);
    for (int e = (int)threadIdx.x; e < T * M; e += FFT_THREADS) {
        if (FWD) {
            const int i = e / T, t = e % T;
            if (t < tn) out[(kz * M + i) * M + ix0 + t] = z[lds_at<T>(t, i)];
        } else {
            const int t = (int)dm.div((unsigned)e), i = e - t * M;
            if (t < tn) out[((int64_t)(ix0 + t) * H + kz) * M + i] = z[lds_at<T>(t, i)];
        }
    }
}

// X (FWD): B[kz0 + t][ky][*] -> S[kx][ky][kz0 + t];  X' (!FWD): the reverse.
// Grid M * ceil(H / T).
template <int T, bool FWD>
__global__ __launch_bounds__(FFT_THREADS) void gen_x_kernel(const float2* __restrict__ in, float2* __restrict__ out,
                                                           const float2* __restrict__ tf, GenPlan P) {
    const int M = P.M, H = M / 2 + 1, nt = (H + T - 1) / T;
    float2 *s = gen_lds, *s2 = s + T * M, *tw = s2 + T * M;
    const int64_t ky = blockIdx.x / nt;
    const int kz0 = (int)(blockIdx.x % nt) * T, tn = min(T, H - kz0);
    const FastDiv dm((unsigned)M);
    const float2 zero = make_float2(0.f, 0.f);
    gen_twiddles(tw, tf, M);
#pragma unroll 4
    for (int e = (int)threadIdx.x; e < T * M; e += FFT_THREADS) {
        if (FWD) {
            const int t = (int)dm.div((unsigned)e), i = e - t * M;
            s[lds_at<T>(t, i)] = t < tn ? in[((int64_t)(kz0 + t) * M + ky) * M + i] : zero;
        } else {
            const int i = e / T, t = e % T;
            s[lds_at<T>(t, i)] = t < tn ? in[((int64_t)i * M + ky) * H + kz0 + t] : zero;
        }
    }
    const float2* z = gen_rows<T, FWD ? -1 : 1>(s, s2, tw, P);
    for (int e = (int)threadIdx.x; e < T * M; e += FFT_THREADS) {
        if (FWD) {
            const int i = e / T, t = e % T;
            if (t < tn) out[((int64_t)i * M + ky) * H + kz0 + t] = z[lds_at<T>(t, i)];
        } else {
            const int t = (int)dm.div((unsigned)e), i = e - t * M;
            if (t < tn) out[((int64_t)(kz0 + t) * M + ky) * M + i] = z[lds_at<T>(t, i)];
        }
    }
}

// Radices of M: primes above 7 first (no twiddles there), then 7 .. 3, 8, 4
// and 2.  Returns the largest radix.
int gen_plan(int M, GenPlan* P) {
    P->M = M;
    P->nstage = 0;
    int rest = M, big = 1;
    for (int p = 11; p <= rest; p += 2)
        while (rest % p == 0) {
            P->radix[P->nstage++] = p;
            rest /= p;
            big = std::max(big, p);
        }
    for (int R : {7, 5, 3, 8, 4, 2})
        while (rest % R == 0) {
            P->radix[P->nstage++] = R;
            rest /= R;
            big = std::max(big, R);
        }
    return big;
}

template <int T>
void gen_r2c(hipStream_t st, const GenPlan& P, const float* in, float2* out, float2* work, const float2* tf) {
    const int M = P.M, H = M / 2 + 1;
    const size_t lds = sizeof(float2) * (size_t)(2 * T + 1) * M;
    gen_z_r2c_kernel<T><<<M * ((M + 2 * T - 1) / (2 * T)), FFT_THREADS, lds, st>>>(in, out, tf, P);
    gen_y_kernel<T, true><<<H * ((M + T - 1) / T), FFT_THREADS, lds, st>>>(out, work, tf, P);
    gen_x_kernel<T, true><<<M * ((H + T - 1) / T), FFT_THREADS, lds, st>>>(work, out, tf, P);
}

template <int T>
void gen_c2r(hipStream_t st, const GenPlan& P, float2* in, float* out, float2* work, const float2* tf) {
    const int M = P.M, H = M / 2 + 1;
    const size_t lds = sizeof(float2) * (size_t)(2 * T + 1) * M;
    gen_x_kernel<T, false><<<M * ((H + T - 1) / T), FFT_THREADS, lds, st>>>(in, work, tf, P);
    gen_y_kernel<T, false><<<H * ((M + T - 1) / T), FFT_THREADS, lds, st>>>(work, in, tf, P);
    gen_z_c2r_kernel<T><<<M * ((M + 2 * T - 1) / (2 * T)), FFT_THREADS, lds, st>>>(in, out, tf, P);
}

#define GEN_T 8      // complex rows per workgroup
#define GEN_MAX 384  // two buffers of them and the twiddles: 51 KiB of LDS

}  // namespace

bool tpm_lds_fft_pow2(int M) { return M >= 16 && M <= 1024 && (M & (M - 1)) == 0; }

// rocFFT has kernels for the radices up to 17; a larger prime factor it
// transforms as a convolution of twice the length or more (chirps, two
// transforms, transposes: 30 to 60 launches for a solve).  Poisson solve, general kernels
// against rocFFT, in us: 38^3 50 / 102, 61^3 66 / 139, 93^3 86 / 212,
// 101^3 126 / 226, 155^3 189 / 501, 217^3 343 / 973, 244^3 591 / 719, 279^3
// 751 / 2968, 332^3 1871 / 2171, 380^3 2078 / 3085.  The rounding error is
// below the convolution's: the PM force's over 14 sizes from 38 to 155, uniform
// and Zel'dovich boxes, is 3.1e-6 / 4.6e-6 (rms), 0.66 of it in the mean.
// The lines: for p > 101 even sizes lose (202 = 2 101 is a draw, 226 = 2 113 648 / 614);
// above 384 large p lose (404 = 4 101: 5129 / 3710); without a factor
// above 17 rocFFT is faster (100^3: 110 / 66).
bool tpm_lds_fft_size(int M) {
    if (tpm_lds_fft_pow2(M)) return true;
    GenPlan P;
    const int p = M >= 16 && M <= GEN_MAX ? gen_plan(M, &P) : 0;
    return p >= 19 && p <= 101;
}

tpm_status tpm_lds_fft_twiddles(std::string& err, int M, float2** tf) {
    std::vector<float2> h(M);
    for (int q = 0; q < M; q++) {
        const double a = -2.0 * M_PI * (double)q / (double)M;
        h[q] = make_float2((float)std::cos(a), (float)std::sin(a));
    }
    TPM_HIPE(err, hipMalloc(tf, sizeof(float2) * M));
    TPM_HIPE(err, hipMemcpy(*tf, h.data(), sizeof(float2) * M, hipMemcpyHostToDevice));
    return TPM_OK;
}

tpm_status tpm_lds_fft_r2c(std::string& err, hipStream_t st, int M, const void* in, bool q32, float2* out,
                           float2* work, const float2* tf, const float* green) {
    switch (M) {
        case 16: launch_r2c<16>(st, in, q32, out, work, tf, green); break;
        case 32: launch_r2c<32>(st, in, q32, out, work, tf, green); break;
        case 64: launch_r2c<64>(st, in, q32, out, work, tf, green); break;
        case 128: launch_r2c<128>(st, in, q32, out, work, tf, green); break;
        case 256: launch_r2c<256>(st, in, q32, out, work, tf, green); break;
        case 512: launch_r2c<512>(st, in, q32, out, work, tf, green); break;
        case 1024: launch_r2c<1024>(st, in, q32, out, work, tf, green); break;
        default: {
            if (!tpm_lds_fft_size(M) || q32 || green) {
                err = "LDS FFT: unsupported size " + std::to_string(M);
                return TPM_ERR_FFT;
            }
            GenPlan P;
            gen_plan(M, &P);
            gen_r2c<GEN_T>(st, P, static_cast<const float*>(in), out, work, tf);
        }
    }
    TPM_HIPE(err, hipGetLastError());
    return TPM_OK;
}

tpm_status tpm_lds_fft_c2r(std::string& err, hipStream_t st, int M, float2* in, float* out, float2* work,
                           const float2* tf) {
    switch (M) {
        case 16: launch_c2r<16>(st, in, out, work, tf); break;
        case 32: launch_c2r<32>(st, in, out, work, tf); break;
        case 64: launch_c2r<64>(st, in, out, work, tf); break;
        case 128: launch_c2r<128>(st, in, out, work, tf); break;
        case 256: launch_c2r<256>(st, in, out, work, tf); break;
        case 512: launch_c2r<512>(st, in, out, work, tf); break;
        case 1024: launch_c2r<1024>(st, in, out, work, tf); break;
        default: {
            if (!tpm_lds_fft_size(M)) {
                err = "LDS FFT: unsupported size " + std::to_string(M);
                return TPM_ERR_FFT;
            }
            GenPlan P;
            gen_plan(M, &P);
            gen_c2r<GEN_T>(st, P, in, out, work, tf);
        }
    }
    TPM_HIPE(err, hipGetLastError());
    return TPM_OK;
}

tpm_status tpm_lds_green_tiles(std::string& err, hipStream_t st, int M, const float* green, float* gt,
                               int64_t* count) {
    int64_t n = 0;
    switch (M) {
        case 16: n = green_tiles<16>(st, green, gt); break;
        case 32: n = green_tiles<32>(st, green, gt); break;
        case 64: n = green_tiles<64>(st, green, gt); break;
        case 128: n = green_tiles<128>(st, green, gt); break;
        case 256: n = green_tiles<256>(st, green, gt); break;
        case 512: n = green_tiles<512>(st, green, gt); break;
        case 1024: n = green_tiles<1024>(st, green, gt); break;
        default: err = "LDS FFT: unsupported size " + std::to_string(M); return TPM_ERR_FFT;
    }
    if (count) *count = n;
    TPM_HIPE(err, hipGetLastError());
    return TPM_OK;
}

tpm_status tpm_lds_pm_solve(std::string& err, hipStream_t st, int M, const unsigned long long* q, float* phi,
                            float2* spec, float2* work, const float2* tf, const float* green) {
    switch (M) {
        case 16: launch_pm<16>(st, q, phi, spec, work, tf, green); break;
        case 32: launch_pm<32>(st, q, phi, spec, work, tf, green); break;
        case 64: launch_pm<64>(st, q, phi, spec, work, tf, green); break;
        case 128: launch_pm<128>(st, q, phi, spec, work, tf, green); break;
        case 256: launch_pm<256>(st, q, phi, spec, work, tf, green); break;
        case 512: launch_pm<512>(st, q, phi, spec, work, tf, green); break;
        case 1024: launch_pm<1024>(st, q, phi, spec, work, tf, green); break;
        default: err = "LDS FFT: unsupported size " + std::to_string(M); return TPM_ERR_FFT;
    }
    TPM_HIPE(err, hipGetLastError());
    return TPM_OK;
}
