// fft_any.hpp -- the passes of fft.hpp for padded sizes N = 2^a 3^b 5^c 7^d that
// are no power of two: Stockham passes of radix 4, 2, 3, 5 and 7 in LDS, the
// index arithmetic by multiplication with host-computed reciprocals.
//
// Bound by memory: the NX rows are read, NX rows of N/2 + 1 values written and
// read back, and N rows written.  hipFFT transforms the whole padded images,
// three quarters of them zeros, in up to four passes with transposes.  4,000
// BF16 images of 192^2: pad 0.89, transforms 4.6 and maxima 0.45 ms by hipFFT;
// means, rows 0.72 and columns 1.62 ms here.
#pragma once
#include "fft.hpp"

namespace spbp {

constexpr int ANY_PASSES = 12;
// Radices and, per pass, the product of the radices before it; reciprocals
// for n / d with n, d < 2^16: __umulhi(n, 2^32 / d + 1).
struct FftPlan {
    int N, np;
    int R[ANY_PASSES], Ns[ANY_PASSES];
    unsigned mq[ANY_PASSES], mNs[ANY_PASSES];   // by N / R and by Ns
    unsigned mN, mH, mL;                        // by N, by N / 2 + 1 and by N / 2
};
inline unsigned recip(int d) { return (unsigned)((1ull << 32) / (unsigned)d + 1); }   // d >= 2

// The plan of N, or np = 0 when N is no product of 2, 3, 5 and 7 (or too large for a block).
inline FftPlan fft_plan(int N) {
    FftPlan p{};
    if (N < 8 || N > FFT_ROW_ELEMS) return p;
    p.N = N;
    p.mN = recip(N);
    p.mH = recip(N / 2 + 1);
    p.mL = recip(N / 2);
    int n = N, np = 0, Ns = 1;
    const int rad[5] = {7, 5, 3, 4, 2};
    for (int r : rad)
        while (n % r == 0) {
            p.R[np] = r;
            p.Ns[np] = Ns;
            p.mq[np] = recip(N / r);
            p.mNs[np] = Ns > 1 ? recip(Ns) : 0;
            Ns *= r;
            n /= r;
            ++np;
        }
    if (n == 1) p.np = np;
    return p;
}

__device__ __forceinline__ int div_by(int n, unsigned m) { return (int)__umulhi((unsigned)n, m); }

// Forward DFT of R values in place: radix 2 and 4 as in lds_fft, odd radices
// from the sums and differences of the pairs (j, R - j).
template <int R>
__device__ __forceinline__ void dft(float2 (&x)[R]) {
    if constexpr (R == 2) {
        const float2 a = x[0], b = x[1];
        x[0] = c_add(a, b);
        x[1] = c_sub(a, b);
    } else if constexpr (R == 4) {
        const float2 a0 = c_add(x[0], x[2]), a1 = c_sub(x[0], x[2]), a2 = c_add(x[1], x[3]), d = c_sub(x[1], x[3]);
        const float2 a3 = make_float2(d.y, -d.x);
        x[0] = c_add(a0, a2);
        x[1] = c_add(a1, a3);
        x[2] = c_sub(a0, a2);
        x[3] = c_sub(a1, a3);
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

template <int R, int E, int NT>
__device__ __forceinline__ void any_pass(float2* buf, int M, int N, int S, int Ns, unsigned mq, unsigned mNs,
                                         const float2* __restrict__ tw) {
    constexpr int U = (E / R + NT - 1) / NT;
    const int q = N / R, nb = M * q, step = q / Ns;
    float2 x[U][R];
    int dst[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int t = threadIdx.x + u * NT;
        dst[u] = -1;
        if (t < nb) {
            const int m = div_by(t, mq), j = t - m * q;
            const int k = Ns > 1 ? j - div_by(j, mNs) * Ns : 0;
            const float2* s = buf + m * S;
#pragma unroll
            for (int r = 0; r < R; ++r) x[u][r] = r == 0 ? s[j] : c_mul(s[j + r * q], tw[k * step * r]);
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
// in place, by NT threads; M N <= E.  Ends synchronised.
template <int E, int NT>
__device__ __forceinline__ void any_fft(float2* buf, int M, const FftPlan& p, int S, const float2* __restrict__ tw) {
    for (int i = 0; i < p.np; ++i) {
        const int Ns = p.Ns[i];
        const unsigned mq = p.mq[i], mNs = p.mNs[i];
        switch (p.R[i]) {
            case 2: any_pass<2, E, NT>(buf, M, p.N, S, Ns, mq, mNs, tw); break;
            case 3: any_pass<3, E, NT>(buf, M, p.N, S, Ns, mq, mNs, tw); break;
            case 4: any_pass<4, E, NT>(buf, M, p.N, S, Ns, mq, mNs, tw); break;
            case 5: any_pass<5, E, NT>(buf, M, p.N, S, Ns, mq, mNs, tw); break;
            default: any_pass<7, E, NT>(buf, M, p.N, S, Ns, mq, mNs, tw); break;
        }
    }
}

// PADD2's mean for any NX (pad_mean_kernel): a wave per row.
template <typename T>
__global__ __launch_bounds__(TPB) void pad_mean_any_kernel(const T* __restrict__ imgs, int nx, double* __restrict__ mean,
                                                           float* __restrict__ vmax) {
    const int b = blockIdx.x, c = nx / 2;
    const T* img = imgs + (size_t)b * nx * nx;
    const float r2 = (float)c * (float)c;
    double s = 0.0;
    unsigned cnt = 0;
    for (int j = threadIdx.x >> 6; j < nx; j += TPB / 64) {
        const float tj = (float)(j - c);
        for (int i = threadIdx.x & 63; i < nx; i += 64) {
            const float ti = (float)(i - c);
            if (tj * tj + ti * ti > r2) { s += (double)load_img(img, (size_t)j * nx + i); ++cnt; }
        }
    }
    block_sum2(s, cnt);
    if (threadIdx.x == 0) { mean[b] = s / (double)cnt; vmax[b] = 0.0f; }
}

// Rows pass (row_fft_kernel): block per (image, group of FFT_ROW_ELEMS / N row pairs).
template <typename T>
__global__ __launch_bounds__(TPB) void row_any_kernel(const T* __restrict__ imgs, int nx, FftPlan p, const float2* __restrict__ tw,
                                                      const double* __restrict__ mean, float2* __restrict__ spec) {
    extern __shared__ float2 lds[];
    float2* buf = lds;
    float2* stw = lds + FFT_ROW_ELEMS + 64;
    const int N = p.N, H = nx + 1, ip = (N - nx) / 2 + (nx % 2);
    load_twiddles(stw, tw, N);
    const int b = blockIdx.y;
    const T* img = imgs + (size_t)b * nx * nx;
    const double qs = mean[b];
    const int pairs = (nx + 1) / 2, M = min(FFT_ROW_ELEMS / N, pairs);
    const int p0 = blockIdx.x * M, mc = min(M, pairs - p0);
    const int total = mc * N;
    for (int i0 = threadIdx.x; i0 < total; i0 += FFT_BATCH * TPB) {
        float2 v[FFT_BATCH];
#pragma unroll
        for (int u = 0; u < FFT_BATCH; ++u) {
            const int idx = i0 + u * TPB;
            const int m = div_by(idx, p.mN), x = idx - m * N - ip;
            const int r = 2 * (p0 + m);
            v[u] = make_float2(0.f, 0.f);
            if (idx < total && (unsigned)x < (unsigned)nx) {
                v[u].x = (float)((double)load_img(img, (size_t)r * nx + x) - qs);
                if (r + 1 < nx) v[u].y = (float)((double)load_img(img, (size_t)(r + 1) * nx + x) - qs);   // odd NX: the last row alone
            }
        }
#pragma unroll
        for (int u = 0; u < FFT_BATCH; ++u)
            if (i0 + u * TPB < total) buf[i0 + u * TPB] = v[u];
    }
    __syncthreads();
    any_fft<FFT_ROW_ELEMS, TPB>(buf, mc, p, N, stw);
    float2* out = spec + (size_t)b * N * H;
    for (int idx = threadIdx.x; idx < mc * H; idx += TPB) {
        const int m = div_by(idx, p.mH), k = idx - m * H;
        const float2 z = buf[m * N + k], w = buf[m * N + (k ? N - k : 0)];
        const int r = 2 * (p0 + m);
        out[(size_t)(ip + r) * H + k] = make_float2(0.5f * __fadd_rn(z.x, w.x), 0.5f * __fsub_rn(z.y, w.y));
        if (r + 1 < nx) out[(size_t)(ip + r + 1) * H + k] = make_float2(0.5f * __fadd_rn(z.y, w.y), 0.5f * __fsub_rn(w.x, z.x));
    }
}

// Columns pass (col_fft_kernel): block per (image, slab of FFT_ELEMS / N columns).
__global__ __launch_bounds__(FFT_COL_NT) void col_any_kernel(int nx, FftPlan p, const float2* __restrict__ tw,
                                                             float2* __restrict__ spec, float* __restrict__ vmax) {
    extern __shared__ float2 lds[];
    float2* buf = lds;
    float2* stw = lds + FFT_LDS;
    __shared__ float wmax[FFT_COL_NT / 64];
    const int N = p.N, H = nx + 1, ip = (N - nx) / 2 + (nx % 2);
    load_twiddles(stw, tw, N);
    const int b = blockIdx.y;
    // the columns split evenly over the image's blocks
    const int c0 = (int)((long long)H * blockIdx.x / gridDim.x), cw = (int)((long long)H * (blockIdx.x + 1) / gridDim.x) - c0;
    const int S = N + 1;   // odd column stride: a row of the slab spreads over the banks
    float2* sp = spec + (size_t)b * N * H + c0;
    int lc = 0;
    while ((1 << lc) < cw) ++lc;
    const int cp = 1 << lc;
    const int total = cp * nx;   // only rows IP .. IP + NX - 1 are nonzero
    for (int i0 = threadIdx.x; i0 < total; i0 += FFT_BATCH * FFT_COL_NT) {
        float2 v[FFT_BATCH];
#pragma unroll
        for (int u = 0; u < FFT_BATCH; ++u) {
            const int idx = i0 + u * FFT_COL_NT;
            const int n = idx >> lc, m = idx & (cp - 1);
            v[u] = (idx < total && m < cw) ? sp[(size_t)(ip + n) * H + m] : make_float2(0.f, 0.f);
        }
#pragma unroll
        for (int u = 0; u < FFT_BATCH; ++u) {
            const int idx = i0 + u * FFT_COL_NT;
            const int n = idx >> lc, m = idx & (cp - 1);
            if (idx < total && m < cw) buf[m * S + ip + n] = v[u];
        }
    }
    for (int idx = threadIdx.x; idx < cp * (N - nx); idx += FFT_COL_NT) {   // the zero rows
        const int n = idx >> lc, m = idx & (cp - 1);
        if (m < cw) buf[m * S + (n < ip ? n : n + nx)] = make_float2(0.f, 0.f);
    }
    __syncthreads();
    any_fft<FFT_ELEMS, FFT_COL_NT>(buf, cw, p, S, stw);
    float mx = 0.0f;
    for (int idx = threadIdx.x; idx < cp * N; idx += FFT_COL_NT) {
        const int n = idx >> lc, m = idx & (cp - 1);
        if (m >= cw) continue;
        const float2 v = buf[m * S + n];
        sp[(size_t)n * H + m] = v;
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
