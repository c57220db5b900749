// fft.hpp -- PADD2 + the forward 2D R2C FFT of the padded images
// (fmrs.f / fftw3.f: FFTW's forward sign), for N = 2^a 3^b 5^c 7^d, in two
// passes that skip the padding: three quarters of each padded image are zeros.
//
//   pad_mean_kernel (block per image): the ASTA mean (asta.f, FP64) of the
//                   pixels outside the inscribed circle;
//   row_fft_kernel  (block per image x group of rows): the NX nonzero rows of
//                   the padded image, two real rows per complex FFT of length
//                   N, unpacked to their N/2 + 1 outputs, written to rows
//                   IP .. IP + NX - 1 of the spectrum; the real values of
//                   columns 0 and N/2 are the two parts of column 0's;
//   col_fft_kernel  (block per image x slab of columns): each column's length-N
//                   transform from those NX rows (the others are zero),
//                   written to all N rows, and the image's largest |Re|, |Im|.
//                   Column 0's transform is that of columns 0 and N/2.
//
// The spectrum layout is the R2C layout of a row-major N x N transform: N
// rows of N/2 + 1 complex values, X[j][k] = sum_y sum_x P[y][x] e^{-2 pi i
// (x k + y j) / N}.  The transforms run in LDS as Stockham passes of radix 8,
// 4, 2, 3, 5 and 7, twiddles from an FP64-computed table of e^{-2 pi i m / N}
// copied into LDS.  Global loads are issued in groups of FFT_BATCH before
// their values are used, so that many are in flight per thread.
//
// Bound by memory: NX rows are read, NX rows of N/2 values written and read
// back, and N rows of N/2 + 1 written.  Columns pass, 20,000 images of 128^2 /
// 24,000 of 256^2: 2.48 / 15.2 ms with radix-4 passes over neighbouring
// butterflies of one sequence, slabs of one image on all XCDs and a block for
// column N/2; 2.23 / 11.2 ms with radix 8, butterflies of neighbouring
// sequences, an image's slabs on one XCD and columns 0 and N/2 in one
// transform (3.4 TB/s); rows pass 1.21 / 5.43 -> 1.02 / 5.00 ms.  Sizes that are
// no power of two went through hipFFT on whole padded images: pad, transforms
// and maxima of 4,000 BF16 images of 192^2 5.9 ms; means, rows and columns
// 2.1 ms here.
#pragma once
#include "common.hpp"

namespace spbp {

constexpr int FFT_ELEMS = 4096;             // complex values a columns-pass block transforms at a time
constexpr int FFT_LDS = FFT_ELEMS + 96;     // columns are N + 1 apart; min(N / 2, FFT_ELEMS / N) < 46 of them
constexpr int FFT_BATCH = 8;                // global loads in flight per thread
// The rows pass transforms fewer values per block, so that more blocks share
// a CU and their loads overlap: measured per 20,000 images of 128^2 (8,000 of
// 256^2), rows pass 1.78 ms (2.70) with 2048 values per block against 2.42
// (3.30) with 4096.
constexpr int FFT_ROW_ELEMS = 2048;
constexpr int FFT_ROW_LDS = FFT_ROW_ELEMS + 256;   // rows are N + 1 apart; FFT_ROW_ELEMS / N <= 204 of them (N >= 10)
// Threads of a columns-pass block: 512 (eight waves over the same LDS slab)
// hide its loads better than 256 (2.38 -> 2.31 ms per 20,000 images of 128^2,
// 5.43 -> 5.14 ms per 8,000 of 256^2).
constexpr int FFT_COL_NT = 512;

constexpr int FFT_PASSES = 12;
// Radices and, per pass, the product of the radices before it; reciprocals
// for n / d: __umulhi(n, 2^32 / d + 1), exact while n d < 2^32.
struct FftPlan {
    int N, np;
    int R[FFT_PASSES], Ns[FFT_PASSES];
    unsigned mNs[FFT_PASSES];   // by Ns
    unsigned mH, mL, mQ;        // by N / 2 + 1, N / 2 and N / 8 (0 for N < 16)
};
__host__ __device__ inline unsigned recip(int d) { return d > 1 ? 0xFFFFFFFFu / (unsigned)d + 1 : 0; }
__device__ __forceinline__ int div_by(int n, unsigned m) { return (int)__umulhi((unsigned)n, m); }   // d >= 2

// The plan of N, or np = 0 when N is no product of 2, 3, 5 and 7 (or too large for a block).
inline FftPlan fft_plan(int N) {
    FftPlan p{};
    if (N < 8 || N > FFT_ROW_ELEMS || N % 2) return p;
    p.N = N;
    p.mH = recip(N / 2 + 1);
    p.mL = recip(N / 2);
    p.mQ = N >= 16 ? recip(N / 8) : 0;
    int n = N, np = 0, Ns = 1;
    while (n > 1) {
        const int r = n % 7 == 0 ? 7 : n % 5 == 0 ? 5 : n % 3 == 0 ? 3 : n % 8 == 0 && n != 16 ? 8 : n % 4 == 0 ? 4 : n % 2 == 0 ? 2 : 0;
        if (!r) return p;   // another prime factor
        p.R[np] = r;
        p.Ns[np] = Ns;
        p.mNs[np] = recip(Ns);
        Ns *= r;
        n /= r;
        ++np;
    }
    p.np = np;
    return p;
}

// Dynamic LDS of the transform kernels: the data, then the N twiddles.
inline size_t fft_lds_bytes(int N, int lds) { return (size_t)(lds + N) * sizeof(float2); }
__device__ inline void load_twiddles(float2* stw, const float2* __restrict__ tw, int N) {
    for (int i = threadIdx.x; i < N; i += blockDim.x) stw[i] = tw[i];
}

// Blocks go round the eight XCDs in turn; work item xcd_order(b, n) gives each
// XCD a contiguous range of the n items, so neighbouring slabs, whose rows
// share cache lines at their unaligned ends, meet in one L2.
__device__ __forceinline__ unsigned xcd_order(unsigned b, unsigned n) {
    const unsigned q = n >> 3, r = n & 7, x = b & 7;
    return x * q + min(x, r) + (b >> 3);
}

__device__ inline float2 c_mul(float2 a, float2 b) {
    return make_float2(__fmaf_rn(a.x, b.x, -__fmul_rn(a.y, b.y)), __fmaf_rn(a.x, b.y, __fmul_rn(a.y, b.x)));
}
__device__ inline float2 c_add(float2 a, float2 b) { return make_float2(__fadd_rn(a.x, b.x), __fadd_rn(a.y, b.y)); }
__device__ inline float2 c_sub(float2 a, float2 b) { return make_float2(__fsub_rn(a.x, b.x), __fsub_rn(a.y, b.y)); }

__device__ __forceinline__ void dft4(float2& x0, float2& x1, float2& x2, float2& x3) {
    const float2 a0 = c_add(x0, x2), a1 = c_sub(x0, x2), a2 = c_add(x1, x3), d = c_sub(x1, x3);
    const float2 a3 = make_float2(d.y, -d.x);   // (x1 - x3) (-i)
    x0 = c_add(a0, a2);
    x1 = c_add(a1, a3);
    x2 = c_sub(a0, a2);
    x3 = c_sub(a1, a3);
}

// Forward DFT of R values in place: 8 as 2 x 4, odd radices from the sums and
// differences of the pairs (j, R - j).
template <int R>
__device__ __forceinline__ void dft(float2 (&x)[R]) {
    if constexpr (R == 2) {
        const float2 a = x[0], b = x[1];
        x[0] = c_add(a, b);
        x[1] = c_sub(a, b);
    } else if constexpr (R == 4) {
        dft4(x[0], x[1], x[2], x[3]);
    } else if constexpr (R == 8) {
        constexpr float h = 0.70710678118654752f;
        dft4(x[0], x[2], x[4], x[6]);
        dft4(x[1], x[3], x[5], x[7]);
        const float2 o0 = x[1], o1 = make_float2(h * __fadd_rn(x[3].x, x[3].y), h * __fsub_rn(x[3].y, x[3].x));   // e^{-i pi/4}
        const float2 o2 = make_float2(x[5].y, -x[5].x);
        const float2 o3 = make_float2(h * __fsub_rn(x[7].y, x[7].x), -h * __fadd_rn(x[7].x, x[7].y));
        const float2 e0 = x[0], e1 = x[2], e2 = x[4], e3 = x[6];
        x[0] = c_add(e0, o0);
        x[4] = c_sub(e0, o0);
        x[1] = c_add(e1, o1);
        x[5] = c_sub(e1, o1);
        x[2] = c_add(e2, o2);
        x[6] = c_sub(e2, o2);
        x[3] = c_add(e3, o3);
        x[7] = c_sub(e3, o3);
    } else {
        // cos and sin of 2 pi m / R
        constexpr float C3[3] = {1.0f, -0.5f, -0.5f}, S3[3] = {0.0f, 0.86602540378443865f, -0.86602540378443865f};
        constexpr float C5[5] = {1.0f, 0.30901699437494742f, -0.80901699437494742f, -0.80901699437494742f, 0.30901699437494742f};
        constexpr float S5[5] = {0.0f, 0.95105651629515357f, 0.58778525229247313f, -0.58778525229247313f, -0.95105651629515357f};
        constexpr float C7[7] = {1.0f, 0.62348980185873353f, -0.22252093395631440f, -0.90096886790241913f, -0.90096886790241913f,
                                 -0.22252093395631440f, 0.62348980185873353f};
        constexpr float S7[7] = {0.0f, 0.78183148246802981f, 0.97492791218182361f, 0.43388373911755812f, -0.43388373911755812f,
                                 -0.97492791218182361f, -0.78183148246802981f};
        constexpr int P = (R - 1) / 2;
        float2 s[P], d[P];
#pragma unroll
        for (int j = 0; j < P; ++j) {
            s[j] = c_add(x[j + 1], x[R - 1 - j]);
            d[j] = c_sub(x[j + 1], x[R - 1 - j]);
        }
        const float2 x0 = x[0];
#pragma unroll
        for (int j = 0; j < P; ++j) x[0] = c_add(x[0], s[j]);
#pragma unroll
        for (int k = 1; k <= P; ++k) {
            float2 a = x0, b = make_float2(0.f, 0.f);
#pragma unroll
            for (int j = 0; j < P; ++j) {
                const int m = ((j + 1) * k) % R;
                const float c = R == 3 ? C3[m % 3] : R == 5 ? C5[m % 5] : C7[m % 7], sn = R == 3 ? S3[m % 3] : R == 5 ? S5[m % 5] : S7[m % 7];
                a.x = __fmaf_rn(s[j].x, c, a.x);
                a.y = __fmaf_rn(s[j].y, c, a.y);
                b.x = __fmaf_rn(d[j].x, sn, b.x);
                b.y = __fmaf_rn(d[j].y, sn, b.y);
            }
            x[k] = make_float2(a.x + b.y, a.y - b.x);       // a - i b
            x[R - k] = make_float2(a.x - b.y, a.y + b.x);   // a + i b
        }
    }
}

// One Stockham pass.  Consecutive threads take the same butterfly of
// consecutive sequences, S (odd) values apart: LDS accesses that hardly
// conflict at any stride Ns, and one twiddle for all of them.
template <int R, int E, int NT>
__device__ __forceinline__ void fft_pass(float2* buf, int M, unsigned mM, int N, int S, int Ns, unsigned mNs,
                                         const float2* __restrict__ tw) {
    constexpr int U = (E / R + NT - 1) / NT;
    const int q = (int)((unsigned)N / R), nb = M * q;
    const int step = Ns > 1 ? div_by(q, mNs) : q;
    float2 x[U][R];
    int dst[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int t = threadIdx.x + u * NT;
        dst[u] = -1;
        if (t < nb) {
            const int j = mM ? div_by(t, mM) : t, m = t - j * M;
            const int k = Ns > 1 ? j - div_by(j, mNs) * Ns : 0;
            const float2* s = buf + m * S + j;
#pragma unroll
            for (int r = 0; r < R; ++r) x[u][r] = s[r * q];
            if (Ns > 1) {
                const int ks = k * step;
#pragma unroll
                for (int r = 1; r < R; ++r) x[u][r] = c_mul(x[u][r], tw[ks * r]);
            }
            dft<R>(x[u]);
            dst[u] = m * S + (j - k) * R + k;
        }
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < U; ++u)
        if (dst[u] >= 0) {
#pragma unroll
            for (int r = 0; r < R; ++r) buf[dst[u] + r * Ns] = x[u][r];
        }
    __syncthreads();
}

// Forward DFTs of M sequences of length p.N in LDS (sequence m at buf + m S),
// in place, by a block of NT threads: every pass reads all its inputs into
// registers, synchronises, then writes.  M N <= E.  Ends synchronised.  P2: N
// is a power of two (without the odd radices a kernel takes 64 VGPRs or fewer
// instead of 77, and four blocks of the columns pass share a CU, not three).
template <int E, int NT, bool P2>
__device__ __forceinline__ void lds_fft(float2* buf, int M, const FftPlan& p, int S, const float2* __restrict__ tw) {
    const unsigned mM = recip(M);
    for (int i = 0; i < p.np; ++i) {
        const int Ns = p.Ns[i];
        const unsigned mNs = p.mNs[i];
        switch (p.R[i]) {
            case 8: fft_pass<8, E, NT>(buf, M, mM, p.N, S, Ns, mNs, tw); break;
            case 4: fft_pass<4, E, NT>(buf, M, mM, p.N, S, Ns, mNs, tw); break;
            case 2: fft_pass<2, E, NT>(buf, M, mM, p.N, S, Ns, mNs, tw); break;
            default:
                if constexpr (!P2) {
                    if (p.R[i] == 3) fft_pass<3, E, NT>(buf, M, mM, p.N, S, Ns, mNs, tw);
                    else if (p.R[i] == 5) fft_pass<5, E, NT>(buf, M, mM, p.N, S, Ns, mNs, tw);
                    else fft_pass<7, E, NT>(buf, M, mM, p.N, S, Ns, mNs, tw);
                }
        }
    }
}

// PADD2's mean: FP64 mean of the pixels outside the inscribed circle
// (asta.f, bp3f.f:1316); block per image.  Also zeroes the image's vmax.
// Each thread reads 16 bytes at a time (4 fp32 or 8 BF16 pixels), FFT_BATCH /
// 2 such loads in flight; an image that does not start 16-byte aligned, or
// whose pixel count is not a multiple of the vector (NX < 4), takes the
// scalar loop.  mL: reciprocal of NX.
template <typename T>
__global__ __launch_bounds__(TPB) void pad_mean_kernel(const T* __restrict__ imgs, int nx, unsigned mL,
                                                       double* __restrict__ mean, float* __restrict__ vmax) {
    constexpr int VW = 16 / sizeof(T);   // pixels per 16-byte load
    const int b = blockIdx.x;
    const T* img = imgs + (size_t)b * nx * nx;
    const int c = nx / 2, n = nx * nx;
    const float r2 = (float)c * (float)c;
    double s = 0.0;
    unsigned cnt = 0;
    auto add = [&](int idx, float v) {
        const int j = div_by(idx, mL), i = idx - j * nx;
        const float tj = (float)(j - c), ti = (float)(i - c);
        if (tj * tj + ti * ti > r2) { s += (double)v; ++cnt; }
    };
    if (n % VW == 0 && ((uintptr_t)img & 15) == 0) {
        constexpr int MB = FFT_BATCH / 2;
        const int nv = n / VW;
        const uint4* img4 = reinterpret_cast<const uint4*>(img);
        for (int i0 = threadIdx.x; i0 < nv; i0 += MB * TPB) {
            uint4 q[MB];
#pragma unroll
            for (int u = 0; u < MB; ++u) {
                const int k = i0 + u * TPB;
                q[u] = k < nv ? img4[k] : make_uint4(0u, 0u, 0u, 0u);
            }
#pragma unroll
            for (int u = 0; u < MB; ++u) {
                const int k = i0 + u * TPB;
                if (k >= nv) continue;
                const unsigned w[4] = {q[u].x, q[u].y, q[u].z, q[u].w};
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    if constexpr (sizeof(T) == 4) {
                        add(k * VW + e, __uint_as_float(w[e]));
                    } else {   // two BF16 pixels per word, the lower address in the low half
                        add(k * VW + 2 * e, __uint_as_float(w[e] << 16));
                        add(k * VW + 2 * e + 1, __uint_as_float(w[e] & 0xFFFF0000u));
                    }
                }
            }
        }
    } else {
        for (int idx = threadIdx.x; idx < n; idx += TPB) add(idx, load_img(img, idx));
    }
    block_sum2(s, cnt);
    if (threadIdx.x == 0) { mean[b] = s / (double)cnt; vmax[b] = 0.0f; }
}

// Four consecutive pixels (an aligned 16- or 8-byte load) as fp32.
__device__ inline float4 load_img4(const float* p) { return *reinterpret_cast<const float4*>(p); }
__device__ inline float4 load_img4(const uint16_t* p) {
    const uint2 w = *reinterpret_cast<const uint2*>(p);   // pixel 0 in the low half of w.x
    return make_float4(__uint_as_float(w.x << 16), __uint_as_float(w.x & 0xFFFF0000u), __uint_as_float(w.y << 16),
                       __uint_as_float(w.y & 0xFFFF0000u));
}

// Rows pass.  Block per (image, group of FFT_ROW_ELEMS / N row pairs); the
// spectrum's rows IP .. IP + NX - 1 receive the row transforms of the padded
// image (PADD2: image minus the FP64 mean, bp3f.f:1316-1345), columns 0 ..
// N/2 - 1, with column N/2's (real) value as the imaginary part of column 0's.
template <typename T, bool P2>
__global__ __launch_bounds__(TPB) void row_fft_kernel(const T* __restrict__ imgs, int nx, FftPlan p, int groups,
                                                      const float2* __restrict__ tw, const double* __restrict__ mean,
                                                      float2* __restrict__ spec) {
    extern __shared__ float2 lds[];
    float2* buf = lds;
    float2* stw = lds + FFT_ROW_LDS;
    const int N = p.N, H = nx + 1, S = N + 1, ip = (N - nx) / 2 + (nx % 2);
    load_twiddles(stw, tw, N);
    const unsigned b = blockIdx.x / (unsigned)groups;
    const T* img = imgs + (size_t)b * nx * nx;
    const double qs = mean[b];
    const int pairs = (nx + 1) / 2, M = min(FFT_ROW_ELEMS / N, pairs);
    const int p0 = (int)(blockIdx.x - b * (unsigned)groups) * M, mc = min(M, pairs - p0);
    for (int i = threadIdx.x; i < mc * nx; i += TPB) {   // the padding: N - NX = NX columns of each sequence
        const int m = div_by(i, p.mL), n = i - m * nx;
        buf[m * S + (n < ip ? n : n + nx)] = make_float2(0.f, 0.f);
    }
    if ((nx & 3) == 0 && p.mQ && ((uintptr_t)img & (4 * sizeof(T) - 1)) == 0) {
        // four pixels of each of the pair's rows per load
        const int nq = nx >> 2, totq = mc * nq;
        constexpr int BQ = FFT_BATCH / 2;
        for (int q0 = threadIdx.x; q0 < totq; q0 += BQ * TPB) {
            float4 a[BQ], c[BQ];
            int at[BQ];
#pragma unroll
            for (int u = 0; u < BQ; ++u) {
                const int q = q0 + u * TPB;
                const int m = div_by(q, p.mQ), xq = q - m * nq;
                const int r = 2 * (p0 + m);
                at[u] = m * S + ip + 4 * xq;
                if (q < totq) {
                    a[u] = load_img4(img + r * nx + 4 * xq);
                    c[u] = load_img4(img + (r + 1) * nx + 4 * xq);
                }
            }
#pragma unroll
            for (int u = 0; u < BQ; ++u) {
                if (q0 + u * TPB >= totq) continue;
                float2* o = buf + at[u];
                o[0] = make_float2((float)((double)a[u].x - qs), (float)((double)c[u].x - qs));
                o[1] = make_float2((float)((double)a[u].y - qs), (float)((double)c[u].y - qs));
                o[2] = make_float2((float)((double)a[u].z - qs), (float)((double)c[u].z - qs));
                o[3] = make_float2((float)((double)a[u].w - qs), (float)((double)c[u].w - qs));
            }
        }
    } else {
        const int total = mc * nx;
        for (int i0 = threadIdx.x; i0 < total; i0 += FFT_BATCH * TPB) {
            float2 v[FFT_BATCH];
            int at[FFT_BATCH];
#pragma unroll
            for (int u = 0; u < FFT_BATCH; ++u) {
                const int idx = i0 + u * TPB;
                const int m = div_by(idx, p.mL), x = idx - m * nx, r = 2 * (p0 + m);
                at[u] = m * S + ip + x;
                v[u] = make_float2(0.f, 0.f);
                if (idx < total) {
                    v[u].x = (float)((double)load_img(img, (size_t)r * nx + x) - qs);
                    if (r + 1 < nx) v[u].y = (float)((double)load_img(img, (size_t)(r + 1) * nx + x) - qs);   // odd NX: the last row alone
                }
            }
#pragma unroll
            for (int u = 0; u < FFT_BATCH; ++u)
                if (i0 + u * TPB < total) buf[at[u]] = v[u];
        }
    }
    __syncthreads();
    lds_fft<FFT_ROW_ELEMS, TPB, P2>(buf, mc, p, S, stw);
    // Z = FFT(x_r + i x_{r+1}): X_r[k] = (Z[k] + conj Z[N-k]) / 2,
    // X_{r+1}[k] = -i (Z[k] - conj Z[N-k]) / 2
    float2* out = spec + (size_t)b * N * H + (size_t)(ip + 2 * p0) * H;
    for (int idx = threadIdx.x; idx < mc * nx; idx += TPB) {
        const int m = div_by(idx, p.mL), k = idx - m * nx;
        const float2 z = buf[m * S + k], w = buf[m * S + N - (k ? k : nx)];   // k = 0: w = Z[N/2]
        float2 u, v;
        if (k) {
            u = make_float2(0.5f * __fadd_rn(z.x, w.x), 0.5f * __fsub_rn(z.y, w.y));
            v = make_float2(0.5f * __fadd_rn(z.y, w.y), 0.5f * __fsub_rn(w.x, z.x));
        } else {
            u = make_float2(z.x, w.x);
            v = make_float2(z.y, w.y);
        }
        out[2 * m * H + k] = u;
        if (2 * (p0 + m) + 1 < nx) out[(2 * m + 1) * H + k] = v;
    }
}

// Columns pass.  Block per (image, slab of cw <= FFT_ELEMS / N of the columns 0
// .. N/2 - 1; the last slab may be narrower): the columns' transforms over all
// N rows, from rows IP .. IP + NX - 1; the image's largest |Re|, |Im| into vmax
// (zeroed by the caller).  A thread keeps its column: rows n0, n0 + dn, ...
//
// ADJ: the raw values the insertion takes in the projector's adjoint applied to
// real images (the transpose of images = crop(irfft2(BI completed by Hermitian
// symmetry in column 0))) instead: R(I, jp) cx(I) / N^2 with cx = 2 for 0 < I <
// NX and 1 at I = 0 and NX (the columns irfft2 counts twice), and in column 0
// the transpose of the completion, R(0, jp) + conj(R(0, N - jp)) = 2 R(0, jp) for
// 0 < jp < NX and 0 for jp > NX.  Two passes over the spectra did this before,
// scaling and maxima: 0.85 ms per 4,096 images of 128^2, nothing measurable here.
template <bool P2, bool ADJ>
__global__ __launch_bounds__(FFT_COL_NT) void col_fft_kernel(int nx, FftPlan p, int slabs, int width,
                                                             const float2* __restrict__ tw, float2* __restrict__ spec,
                                                             float* __restrict__ vmax) {
    extern __shared__ float2 lds[];
    float2* buf = lds;
    float2* stw = lds + FFT_LDS;
    __shared__ float wmax[FFT_COL_NT / 64];
    const int N = p.N, H = nx + 1, S = N + 1, ip = (N - nx) / 2 + (nx % 2);
    load_twiddles(stw, tw, N);
    const unsigned w = xcd_order(blockIdx.x, gridDim.x), b = w / (unsigned)slabs;
    const int c0 = (int)(w - b * (unsigned)slabs) * width, cw = min(width, nx - c0);
    float2* sp = spec + (size_t)b * N * H + c0;
    const int lc = cw > 1 ? 32 - __clz(cw - 1) : 0, cp = 1 << lc;
    const int m = threadIdx.x & (cp - 1), n0 = threadIdx.x >> lc, dn = FFT_COL_NT >> lc;
    if (m < cw) {
        for (int nb = n0; nb < nx; nb += FFT_BATCH * dn) {   // only rows IP .. IP + NX - 1 are nonzero
            float2 v[FFT_BATCH];
#pragma unroll
            for (int u = 0; u < FFT_BATCH; ++u) v[u] = sp[(ip + min(nb + u * dn, nx - 1)) * H + m];
#pragma unroll
            for (int u = 0; u < FFT_BATCH; ++u)
                if (nb + u * dn < nx) buf[m * S + ip + nb + u * dn] = v[u];
        }
        for (int n = n0; n < N - nx; n += dn) buf[m * S + (n < ip ? n : n + nx)] = make_float2(0.f, 0.f);
    }
    __syncthreads();
    lds_fft<FFT_ELEMS, FFT_COL_NT, P2>(buf, cw, p, S, stw);
    float mx = 0.0f;
    const float inv = 1.0f / (float)((double)N * (double)N);
    if (m < cw)
        for (int n = n0; n < N; n += dn) {
            float2 v = buf[m * S + n];
            if (c0 + m == 0) {   // F of columns 0 + i N/2: (F[n] + conj F[N-n]) / 2 and -i (F[n] - conj F[N-n]) / 2
                const float2 c = buf[n ? N - n : 0];
                float2 h = make_float2(0.5f * __fadd_rn(v.y, c.y), 0.5f * __fsub_rn(c.x, v.x));
                v = make_float2(0.5f * __fadd_rn(v.x, c.x), 0.5f * __fsub_rn(v.y, c.y));
                if constexpr (ADJ) {
                    h = make_float2(h.x * inv, h.y * inv);
                    if (n > nx) v = make_float2(0.f, 0.f);
                }
                mx = fmaxf(mx, fmaxf(fabsf(h.x), fabsf(h.y)));
                sp[n * H + nx] = h;
            }
            if constexpr (ADJ) {
                const float sc = c0 + m == 0 && (n == 0 || n == nx) ? inv : 2.0f * inv;
                v = make_float2(v.x * sc, v.y * sc);
            }
            sp[n * H + m] = v;
            mx = fmaxf(mx, fmaxf(fabsf(v.x), fabsf(v.y)));
        }
    for (int off = 32; off > 0; off >>= 1) mx = fmaxf(mx, __shfl_down(mx, off, 64));
    if ((threadIdx.x & 63) == 0) wmax[threadIdx.x >> 6] = mx;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int k = 1; k < FFT_COL_NT / 64; ++k) mx = fmaxf(mx, wmax[k]);
        atomicMax((unsigned*)&vmax[b], __float_as_uint(mx));   // non-negative floats order as their bits
    }
}

}  // namespace spbp
