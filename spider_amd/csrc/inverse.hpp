// inverse.hpp -- NRMW2, the inverse transform and WINDKB2A of a volume in three
// passes over the half grid, for N = 2^a 3^b 5^c 7^d:
//
//   inv_y_kernel  (block per (plane k, slab of columns kx)): normalised values of
//                 the accumulators, transformed along y; the NX rows the window
//                 keeps are written;
//   inv_z_kernel  (block per (row, slab)): along z; the NX planes it keeps;
//   inv_x_kernel  (block per group of row pairs): two rows' half spectra make one
//                 complex transform of length N, whose real and imaginary parts
//                 are the rows; cropped, scaled, divided by the window, with the
//                 outer shell's sum.
//
// Bound by memory: 12 bytes per half-grid voxel and half are read, then (1/2 +
// 1/2 + 1/4 + 1/4) of 8 bytes pass through the intermediates.  Normalising
// into a full half grid, hipFFT's 3D transform with its transposes and a window
// pass over N^3 reals moved over three times as much, and a context's plan cost
// ~5 ms to make and ~5 ms to destroy.  Three volumes of two halves, before and
// after: 256^3 into 128^3 0.93 -> 0.25 ms; a context of 64^3 from 300
// projections, made, used and destroyed: 10.7 -> 1.8 ms.
//
// y before z: the accumulators' rows of a plane are N / 2 + 1 values apart, those
// of a column of planes ~N^2 / 2, each in a page of its own (z first: 1.20 ms
// for the first pass at 384^3, y first: 1.09).  4,096 values per block of 512
// threads leave three blocks on a CU (0.89 ms; 8,192 values 1.06, 256 threads
// 1.05); then the Friedel mates are loaded with the column kx = 0's lanes only
// (0.68 ms).
//
// The volume is the forward transform of the Hermitian normalised grid: SPIDER
// conjugates first and transforms backward (fmrs_3.f), which gives the
// conjugate of the same, real, sum.  Of the kx = 0 and kx = N/2 planes a C2R
// transform uses the Hermitian parts only; their transform along y and z is the
// real part of the planes' own, which is what the x pass reads.
#pragma once
#include "finalize.hpp"

namespace spbp {

struct Slab {
    int row, c0, cw, lc;   // lc: log2 of the power of two >= cw
};
__device__ __forceinline__ Slab slab_of(unsigned w, int slabs, int H) {
    Slab s;
    s.row = (int)(w / (unsigned)slabs);
    const int k = (int)w - s.row * slabs;
    s.c0 = (int)((long long)H * k / slabs);
    s.cw = (int)((long long)H * (k + 1) / slabs) - s.c0;
    s.lc = s.cw > 1 ? 32 - __clz(s.cw - 1) : 0;
    return s;
}

// Element (n, m) of a slab: row n, column m; a thread keeps its column, and its
// rows are n0, n0 + dn, ...  Columns m >= cw idle (they load a column that exists).

template <bool P2>
__global__ __launch_bounds__(INV_NT) void inv_y_kernel(const FinalJob* __restrict__ jobs, int nj) {
    __shared__ float2 buf[INV_LDS];
    extern __shared__ float2 stw[];
    const FinalJob& f = jobs[job_of_block<0>(jobs, nj, blockIdx.x)];
    const FftPlan& p = f.fft;
    const int nx = f.nx, N = f.N, H = nx + 1, S = N + 1, ip = (N - nx) / 2 + (nx % 2);
    const Slab s = slab_of(xcd_order(blockIdx.x - f.hb0, (unsigned)(N * f.slabs)), f.slabs, H);
    const int k = s.row, cp = 1 << s.lc;
    for (int i = threadIdx.x; i < N; i += INV_NT) stw[i] = f.tw[i];
    const int m = threadIdx.x & (cp - 1), n0 = threadIdx.x >> s.lc, dn = INV_NT >> s.lc, i = s.c0 + m;
    const size_t plane = (size_t)k * N * H, mirror = (size_t)(k ? N - k : 0) * N * H;
    const bool comp = f.a.Wc[0] != nullptr, masked = f.a.mask != nullptr;
    const int halves = f.a.n, mshift = f.a.mshift;
    const Global<const unsigned char> mask = as_global(f.a.mask) + plane;
    constexpr int U = 4;
    for (int nb = n0; nb < N; nb += U * dn) {
        float2 x[U];
        float w[U];
        double wd[U];
        int md[U];
        unsigned o[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            o[u] = (unsigned)(min(nb + u * dn, N - 1) * H + min(i, nx));
            x[u] = make_float2(0.f, 0.f);
            w[u] = 0.f;
            wd[u] = 0.0;
            md[u] = 0;
        }
        if (masked)
#pragma unroll
            for (int u = 0; u < U; ++u) md[u] = mask[o[u]];
        for (int h = 0; h < halves; ++h) {
            const Global<const float2> X = as_global(f.a.X[h]) + plane;
            const Global<const float> W = as_global(f.a.W[h]) + plane, C = as_global(f.a.Wc[h]) + plane;
            float2 xh[U];
            float wh[U], ch[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                xh[u] = load2(X + o[u]);
                wh[u] = W[o[u]];
                ch[u] = 0.f;
            }
            if (comp)
#pragma unroll
                for (int u = 0; u < U; ++u) ch[u] = C[o[u]];
            double dh[U];
#pragma unroll
            for (int u = 0; u < U; ++u) dh[u] = (double)wh[u] + (double)ch[u];
            if (i == 0) {   // SYMPLANE0: the voxel's Friedel mate, as in load_sym
                const Global<const float2> Xm = as_global(f.a.X[h]) + mirror;
                const Global<const float> Wm = as_global(f.a.W[h]) + mirror, Cm = as_global(f.a.Wc[h]) + mirror;
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const int j = min(nb + u * dn, N - 1);
                    if (!sym_pair(j, k, nx)) continue;
                    const unsigned om = (unsigned)((j ? N - j : 0) * H);
                    const float2 xm = load2(Xm + om);
                    const float wm = Wm[om];
                    xh[u].x = xh[u].x + xm.x;
                    xh[u].y = xh[u].y + (-xm.y);
                    wh[u] = wh[u] + wm;
                    dh[u] += comp ? (double)wm + (double)Cm[om] : (double)wm;
                }
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                x[u].x = x[u].x + xh[u].x;
                x[u].y = x[u].y + xh[u].y;
                w[u] = w[u] + wh[u];
                wd[u] += dh[u];
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int j = nb + u * dn;
            if (j < N && m < s.cw) buf[m * S + j] = norm_div(comp, x[u], w[u], wd[u], (md[u] >> mshift) & 3, (i + j + k) & 1);
        }
    }
    __syncthreads();
    lds_fft<INV_ELEMS, INV_NT, P2>(buf, s.cw, p, S, stw);
    const Global<float2> out = as_global(f.work) + (size_t)k * nx * H;
    if (m < s.cw)
        for (int y = n0; y < nx; y += dn) store2(out + (unsigned)(y * H + i), buf[m * S + ip + y]);
}

template <bool P2>
__global__ __launch_bounds__(INV_NT) void inv_z_kernel(const FinalJob* __restrict__ jobs, int nj) {
    __shared__ float2 buf[INV_LDS];
    extern __shared__ float2 stw[];
    const FinalJob& f = jobs[job_of_block<1>(jobs, nj, blockIdx.x)];
    const FftPlan& p = f.fft;
    const int nx = f.nx, N = f.N, H = nx + 1, S = N + 1, ip = (N - nx) / 2 + (nx % 2);
    const Slab s = slab_of(xcd_order(blockIdx.x - f.zb0, (unsigned)(nx * f.slabs)), f.slabs, H);
    const int cp = 1 << s.lc;
    for (int i = threadIdx.x; i < N; i += INV_NT) stw[i] = f.tw[i];
    const int m = threadIdx.x & (cp - 1), n0 = threadIdx.x >> s.lc, dn = INV_NT >> s.lc;
    const size_t pitch = (size_t)nx * H;   // a plane of the intermediate
    const Global<const float2> in = as_global((const float2*)f.work) + (size_t)s.row * H + s.c0 + min(m, s.cw - 1);
    constexpr int U = 8;
    for (int nb = n0; nb < N; nb += U * dn) {
        float2 v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) v[u] = load2(in + (size_t)min(nb + u * dn, N - 1) * pitch);
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (nb + u * dn < N && m < s.cw) buf[m * S + nb + u * dn] = v[u];
    }
    __syncthreads();
    lds_fft<INV_ELEMS, INV_NT, P2>(buf, s.cw, p, S, stw);
    const Global<float2> out = as_global(f.work) + (size_t)nx * N * H + (size_t)s.row * H + s.c0 + m;
    if (m < s.cw)
        for (int z = n0; z < nx; z += dn) store2(out + (size_t)z * pitch, buf[m * S + ip + z]);
}

template <bool P2>
__global__ __launch_bounds__(TPB) void inv_x_kernel(const FinalJob* __restrict__ jobs, int nj) {
    __shared__ float2 buf[FFT_ROW_LDS];
    extern __shared__ float2 stw[];
    const FinalJob& f = jobs[job_of_block<2>(jobs, nj, blockIdx.x)];
    const FftPlan& p = f.fft;
    const int nx = f.nx, N = f.N, H = nx + 1, S = N + 1, ip = (N - nx) / 2 + (nx % 2);
    const unsigned lb = blockIdx.x - f.xb0;
    for (int i = threadIdx.x; i < N; i += TPB) stw[i] = f.tw[i];
    const int rows = nx * nx, M = f.pairs, r0 = 2 * M * (int)lb, mc = min(M, (rows - r0 + 1) / 2);
    const Global<const float2> in = as_global((const float2*)f.work) + (size_t)nx * N * H + (size_t)r0 * H;
    constexpr int U = 4;
    for (int i0 = threadIdx.x; i0 < mc * H; i0 += U * TPB) {
        float2 a[U], b[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int idx = min(i0 + u * TPB, mc * H - 1), m = div_by(idx, p.mH), i = idx - m * H;
            const int ra = 2 * m, rb = min(ra + 1, rows - 1 - r0);   // the last row of an odd number pairs with itself
            a[u] = load2(in + (size_t)ra * H + i);
            b[u] = load2(in + (size_t)rb * H + i);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int idx = i0 + u * TPB;
            if (idx >= mc * H) continue;
            const int m = div_by(idx, p.mH), i = idx - m * H;
            if (i == 0 || i == nx) {
                buf[m * S + i] = make_float2(a[u].x, b[u].x);
            } else {
                buf[m * S + i] = make_float2(a[u].x - b[u].y, a[u].y + b[u].x);
                buf[m * S + N - i] = make_float2(a[u].x + b[u].y, b[u].x - a[u].y);
            }
        }
    }
    __syncthreads();
    lds_fft<FFT_ROW_ELEMS, TPB, P2>(buf, mc, p, S, stw);
    double sum = 0.0;
    unsigned cnt = 0;
    const int cc = nx / 2, nr = min(2 * mc, rows - r0);
    const Global<const float> wkb = as_global(f.wkb);
    const Global<float> out = as_global(f.out) + (size_t)r0 * nx;
    for (int idx = threadIdx.x; idx < nr * nx; idx += TPB) {
        const int q = div_by(idx, p.mL), x = idx - q * nx, r = r0 + q, z = r / nx, y = r - z * nx;
        const float2 t = buf[(q >> 1) * S + ip + x];
        float v = (q & 1 ? t.y : t.x) * f.pix;   // FMRS_3 scale
        const int lr = (x - cc) * (x - cc) + (y - cc) * (y - cc) + (z - cc) * (z - cc);
        if (lr <= cc * cc) {
            v = __fdiv_rn(v, wkb[lr]);
            if (lr >= (cc - 1) * (cc - 1)) { sum += v; ++cnt; }
        } else {
            v = 0.0f;
        }
        out[idx] = v;
    }
    block_sum2(sum, cnt);
    if (threadIdx.x == 0) { f.psum[lb] = sum; f.pcnt[lb] = cnt; }
}

}  // namespace spbp
