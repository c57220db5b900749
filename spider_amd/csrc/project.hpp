// project.hpp -- central-slice KB gather: the exact adjoint of the ONELINE
// scatter (oneline.f:38-158), and the BI -> raw spectrum conversion that lets
// BI-layout spectra go through the insertion kernels.
#pragma once
#include "common.hpp"
#include "fft.hpp"

namespace spbp {

// four floats at an 8-byte aligned address (global loads need only dword
// alignment on gfx950)
typedef float float4a8 __attribute__((ext_vector_type(4), aligned(8)));

// For lattice sample (I, J) of projection p, ONELINE adds w * v to X at each
// direct tap t (t_x >= 0) and w * conj(v) at -t for each reflected tap
// (t_x < 0), where v is BI(I, J), conjugated when the sample is Friedel-
// flipped (x < 0).  Viewing complex numbers as pairs of reals, the transpose
// of that map is
//     out(I, J) = c( sum_direct w X[t] + conj(sum_reflected w X[-t]) ),
// c = conj when flipped, identity otherwise; samples ONELINE skips give 0.
// The taps, the table lookups and the fp32 weights w are computed exactly as
// the insertion kernels compute them, and the sum is accumulated in FP64.
// One thread per output entry; out is nproj x N x H in the BI layout (row
// jp = J mod N, I fastest).  A workgroup covers a GT x GT tile of (I, jp), so
// its samples form a patch of the section and share most of their taps in
// the caches; blockIdx.x = tile (I tiles fastest), blockIdx.y = projection.
constexpr int GT = 16;
// P: sample-position precision, float (the reference's geometry) or double
// (contexts with FP64 geometry), as in the insertion kernels it transposes.
template <typename P>
__global__ __launch_bounds__(GT * GT) void gather_kernel(const float2* __restrict__ X, const Geom* __restrict__ geom,
                                                         int nx, int N, const float* __restrict__ tab, float fltb_f,
                                                         float2* __restrict__ out) {
    const int H = nx + 1;
    const int p = blockIdx.y;
    const int ti = (H + GT - 1) / GT;
    const int tj = blockIdx.x / ti;
    const int I = (blockIdx.x - tj * ti) * GT + (threadIdx.x & (GT - 1));
    const int jp = tj * GT + threadIdx.x / GT;
    if (I >= H || jp >= N) return;
    const int J = jp <= nx ? jp : jp - N;
    float2* o = out + ((size_t)p * N + jp) * H + I;
    if (!(I * I + J * J < (N * N) / 4) || (I == 0 && J < 0)) { *o = make_float2(0.f, 0.f); return; }
    const Geom g = geom[p];
    const P fltb = fltb_of<P>(fltb_f);
    P x, y, z;
    sample_pos(g, I, J, x, y, z);
    const bool flip = x < (P)0;
    if (flip) { x = -x; y = -y; z = -z; }
    const int ix = nearest_voxel(x, N), iy = nearest_voxel(y, N), iz = nearest_voxel(z, N);
    if (!in_bounds(ix, iy, iz, nx)) { *o = make_float2(0.f, 0.f); return; }
    const size_t plane = (size_t)N * H;
    if (ix >= LN2) {
        // no reflected taps (every tap has p_x >= ix - 2 >= 0); the nonzero
        // taps of each axis are a run of at most 4 (the table vanishes beyond
        // 1.8 voxels): from i - 2 when its weight is nonzero, else from i - 1.
        // Same nonzero terms in the same order as the general loop below.
        float tx[4], ty[4], tz[4];
        const float wx0 = kb_weight(tab, dsub(x, ix - 2), fltb);
        const float wy0 = kb_weight(tab, dsub(y, iy - 2), fltb);
        const float wz0 = kb_weight(tab, dsub(z, iz - 2), fltb);
        const int sx = wx0 != 0.0f ? ix - 2 : ix - 1;
        const int sy = wy0 != 0.0f ? iy - 2 : iy - 1;
        const int sz = wz0 != 0.0f ? iz - 2 : iz - 1;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            tx[t] = (t == 0 && sx == ix - 2) ? wx0 : kb_weight(tab, dsub(x, sx + t), fltb);
            ty[t] = (t == 0 && sy == iy - 2) ? wy0 : kb_weight(tab, dsub(y, sy + t), fltb);
            tz[t] = (t == 0 && sz == iz - 2) ? wz0 : kb_weight(tab, dsub(z, sz + t), fltb);
        }
        // each tap row is read whole (columns sx .. sx + 3 <= ix + 2 <= nx - 1,
        // inside the row) as two 16-byte loads; zero-weight taps add exact
        // zeros, so the sums equal those over the nonzero taps alone
        double dre = 0.0, dim = 0.0;
#pragma unroll
        for (int lz = 0; lz < 4; ++lz) {
            const int izp = sz + lz;
            const float2* Xz = X + (size_t)(izp >= 0 ? izp : N + izp) * plane;
#pragma unroll
            for (int ly = 0; ly < 4; ++ly) {
                const float tyz = __fmul_rn(ty[ly], tz[lz]);
                const int iyp = sy + ly;
                const float2* Xy = Xz + (size_t)(iyp >= 0 ? iyp : N + iyp) * H + sx;
                const float4a8 a = *(const float4a8*)Xy, b = *(const float4a8*)(Xy + 2);
                const float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
                for (int lx = 0; lx < 4; ++lx) {
                    const double w = (double)__fmul_rn(tx[lx], tyz);
                    dre += w * (double)v[2 * lx];
                    dim += w * (double)v[2 * lx + 1];
                }
            }
        }
        // the general form adds the (empty) reflected sums: + 0 and - 0
        const double re = dre + 0.0, im = dim - 0.0;
        *o = make_float2((float)re, (float)(flip ? -im : im));
        return;
    }
    float tx[5], ty[5], tz[5];
#pragma unroll
    for (int l = 0; l < 5; ++l) {
        tx[l] = kb_weight(tab, dsub(x, ix + l - LN2), fltb);
        ty[l] = kb_weight(tab, dsub(y, iy + l - LN2), fltb);
        tz[l] = kb_weight(tab, dsub(z, iz + l - LN2), fltb);
    }
    double dre = 0.0, dim = 0.0, mre = 0.0, mim = 0.0;
    for (int lz = 0; lz < 5; ++lz) {
        if (tz[lz] == 0.0f) continue;
        const int izp = iz + lz - LN2;
        const size_t za = (size_t)(izp >= 0 ? izp : N + izp) * plane;
        const size_t zt = (size_t)(izp <= 0 ? -izp : N - izp) * plane;   // wrap(-izp)
        for (int ly = 0; ly < 5; ++ly) {
            const float tyz = __fmul_rn(ty[ly], tz[lz]);
            if (tyz == 0.0f) continue;
            const int iyp = iy + ly - LN2;
            const size_t ya = (size_t)(iyp >= 0 ? iyp : N + iyp) * H;
            const size_t yt = (size_t)(iyp <= 0 ? -iyp : N - iyp) * H;
#pragma unroll
            for (int lx = 0; lx < 5; ++lx) {
                const float wg = __fmul_rn(tx[lx], tyz);
                if (wg == 0.0f) continue;
                const int px = ix + lx - LN2;
                const double w = (double)wg;
                if (px >= 0) {
                    const float2 v = X[za + ya + px];
                    dre += w * (double)v.x;
                    dim += w * (double)v.y;
                } else {
                    const float2 v = X[zt + yt + (size_t)(-px)];
                    mre += w * (double)v.x;
                    mim += w * (double)v.y;
                }
            }
        }
    }
    const double re = dre + mre, im = dim - mim;
    *o = make_float2((float)re, (float)(flip ? -im : im));
}

// ------------------------------------------------------------------ image synthesis
// images = crop(irfft2(C)), C(I, jp) = conj(BI(I, jp) (-1)^(I + jp)) with column 0
// completed by Hermitian symmetry, as the forward transform of conj(C), which
// has the same real sum: synth_col_kernel transforms slabs of columns and keeps
// the NX rows of the crop (in place: rows 0 .. NX - 1), synth_row_kernel makes
// one complex transform of two rows' half spectra and writes their crop.  Of
// columns 0 and N/2 the row transform uses the real parts.
//
// Bound by memory: N rows read, NX written and read, NX rows of pixels written.
// hipFFT transformed and stored all N rows, after a pass that completed the
// spectra and before one that cropped: 4,096 images of 128^2 1.92 ms, here 0.56.
template <bool P2>
__global__ __launch_bounds__(FFT_COL_NT) void synth_col_kernel(int nx, FftPlan p, int slabs, int width,
                                                               const float2* __restrict__ tw, float2* __restrict__ spec) {
    extern __shared__ float2 lds[];
    float2* buf = lds;
    float2* stw = lds + FFT_LDS;
    const int N = p.N, H = nx + 1, S = N + 1, ip = (N - nx) / 2 + (nx % 2);
    load_twiddles(stw, tw, N);
    const unsigned w = xcd_order(blockIdx.x, gridDim.x), b = w / (unsigned)slabs;
    const int c0 = (int)(w - b * (unsigned)slabs) * width, cw = min(width, H - c0);
    float2* sp = spec + (size_t)b * N * H + c0;
    const int lc = cw > 1 ? 32 - __clz(cw - 1) : 0, cp = 1 << lc;
    const int m = threadIdx.x & (cp - 1), n0 = threadIdx.x >> lc, dn = FFT_COL_NT >> lc;
    if (m < cw) {
        for (int nb = n0; nb < N; nb += FFT_BATCH * dn) {
            float2 v[FFT_BATCH];
#pragma unroll
            for (int u = 0; u < FFT_BATCH; ++u) {
                const int n = min(nb + u * dn, N - 1);
                v[u] = sp[(c0 + m == 0 && n > nx ? N - n : n) * H + m];
            }
#pragma unroll
            for (int u = 0; u < FFT_BATCH; ++u) {
                const int n = nb + u * dn;
                const float sg = ((c0 + m + n) & 1) ? -1.0f : 1.0f;   // N is even: the mirror row has the same sign
                if (n < N) buf[m * S + n] = make_float2(v[u].x * sg, c0 + m == 0 && n > nx ? -(v[u].y * sg) : v[u].y * sg);
            }
        }
    }
    __syncthreads();
    lds_fft<FFT_ELEMS, FFT_COL_NT, P2>(buf, cw, p, S, stw);
    if (m < cw)
        for (int n = n0; n < nx; n += dn) sp[n * H + m] = buf[m * S + ip + n];
}

// Block per (image, group of FFT_ROW_ELEMS / N row pairs).
template <bool P2>
__global__ __launch_bounds__(TPB) void synth_row_kernel(int nx, FftPlan p, int groups, const float2* __restrict__ tw,
                                                        const float2* __restrict__ spec, float* __restrict__ imgs) {
    extern __shared__ float2 lds[];
    float2* buf = lds;
    float2* stw = lds + FFT_ROW_LDS;
    const int N = p.N, H = nx + 1, S = N + 1, ip = (N - nx) / 2 + (nx % 2);
    load_twiddles(stw, tw, N);
    const int pairs = (nx + 1) / 2, M = min(FFT_ROW_ELEMS / N, pairs);
    const unsigned img = blockIdx.x / (unsigned)groups;
    const int p0 = (int)(blockIdx.x - img * (unsigned)groups) * M, mc = min(M, pairs - p0), nr = min(2 * mc, nx - 2 * p0);
    const float2* in = spec + (size_t)img * N * H + (size_t)2 * p0 * H;
    constexpr int U = FFT_BATCH / 2;
    for (int i0 = threadIdx.x; i0 < mc * H; i0 += U * TPB) {
        float2 a[U], b[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int idx = min(i0 + u * TPB, mc * H - 1), m = div_by(idx, p.mH), i = idx - m * H;
            a[u] = in[2 * m * H + i];
            b[u] = in[min(2 * m + 1, nr - 1) * H + i];   // odd NX: the last row pairs with itself
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
    const float inv = 1.0f / (float)((double)N * (double)N);   // the inverse transform's normalisation
    float* out = imgs + (size_t)img * nx * nx + (size_t)2 * p0 * nx;
    for (int idx = threadIdx.x; idx < nr * nx; idx += TPB) {
        const int q = div_by(idx, p.mL), x = idx - q * nx;
        const float2 t = buf[(q >> 1) * S + ip + x];
        out[idx] = (q & 1 ? t.y : t.x) * inv;
    }
}

// The same through hipFFT, for other N: before the C2R transform, in place, C(I, jp) = conj(BI(I, jp) (-1)^(I + jp)), and column 0
// completed by Hermitian symmetry, C(0, N - jp) = conj(C(0, jp)) for
// 0 < jp < NX (the rows J < 0 of column 0 are not gathered).  One thread per
// entry; column 0's pairs by the thread of jp.
__global__ __launch_bounds__(TPB) void bi_complete_kernel(float2* __restrict__ spec, int N, int H, int nx, size_t n) {
    const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= n) return;
    const size_t per = (size_t)N * H;
    const size_t r = idx % per;
    const int jp = (int)(r / H), I = (int)(r - (size_t)jp * H);
    if (I == 0 && jp > nx) return;   // written by the thread of N - jp
    const float sg = ((I + jp) & 1) ? -1.0f : 1.0f;
    const float2 v = spec[idx];
    const float2 c = make_float2(v.x * sg, -(v.y * sg));
    spec[idx] = c;
    if (I == 0 && jp > 0 && jp < nx) spec[(idx - r) + (size_t)(N - jp) * H] = make_float2(c.x, -c.y);
}

// Crop of the C2R outputs (N x N each, unnormalised) to the NX x NX images at
// offset IP, scaled by 1 / N^2 (the inverse transform's normalisation).
__global__ __launch_bounds__(TPB) void crop_images_kernel(const float* __restrict__ full, int N, int nx, int ip,
                                                          size_t n, float* __restrict__ out) {
    const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= n) return;
    const size_t npix = (size_t)nx * nx;
    const size_t img = idx / npix, q = idx - img * npix;
    const int y = (int)(q / nx), x = (int)(q - (size_t)y * nx);
    const float inv = 1.0f / (float)((double)N * (double)N);
    out[idx] = full[(img * N + (size_t)(ip + y)) * N + (size_t)(ip + x)] * inv;
}

// BI(I, J) -> the raw R2C value s that spectrum_value() maps to it:
// BI = c conj(s), c = (-1)^(I + jp), so s = c conj(BI); and the spectrum's
// largest |Re|, |Im| into vmax (zero on entry).  Block per (image, BI_BLOCK
// values).  A pass of its own for the maxima, a block per image, took 65 us
// for 256 spectra of 128^2.
constexpr int BI_BLOCK = 8 * TPB;
__global__ __launch_bounds__(TPB) void bi_to_raw_kernel(const float2* __restrict__ bi, int N, int H, unsigned blocks,
                                                        float2* __restrict__ raw, float* __restrict__ vmax) {
    const int per = N * H, r0 = (int)(blockIdx.x % blocks) * BI_BLOCK + threadIdx.x;
    const unsigned b = blockIdx.x / blocks;
    const size_t img = (size_t)b * per;
    float2 v[BI_BLOCK / TPB];
#pragma unroll
    for (int u = 0; u < BI_BLOCK / TPB; ++u) v[u] = bi[img + min(r0 + u * TPB, per - 1)];
    float m = 0.0f;
#pragma unroll
    for (int u = 0; u < BI_BLOCK / TPB; ++u) {
        const int r = r0 + u * TPB;
        if (r >= per) continue;
        const int jp = r / H, I = r - jp * H;
        const float sg = ((I + jp) & 1) ? -1.0f : 1.0f;
        raw[img + r] = make_float2(v[u].x * sg, -v[u].y * sg);
        m = fmaxf(m, fmaxf(fabsf(v[u].x), fabsf(v[u].y)));
    }
    for (int off = 32; off > 0; off >>= 1) m = fmaxf(m, __shfl_down(m, off, 64));
    __shared__ float sm[TPB / 64];
    if ((threadIdx.x & 63) == 0) sm[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int k = 1; k < TPB / 64; ++k) m = fmaxf(m, sm[k]);
        atomicMax((unsigned*)&vmax[b], __float_as_uint(m));   // non-negative floats order as their bits
    }
}

}  // namespace spbp
