// project_cells.hpp -- the central-slice KB gather by bricks of unit cells: the
// transpose of insert_cells_kernel.
//
// gather_kernel reads each sample's 64 taps from the half grid in memory; its
// loads wait on the caches (84% L2 hits, VALU 0.31 per CU-cycle).  Here a
// workgroup loads a brick's region of the grid into LDS once, walks the
// samples of up to `C` sections whose planes cross the brick (the insertion's
// lists and lattice walk), and every sample, one per lane, takes its taps
// from LDS.  The region's layer kx = -1 holds conj X(1, -ky, -kz), so a
// reflected tap is read like a direct one.  Taps, table lookups and the fp32
// weights are the insertion's, as in gather_kernel; the products are summed
// in FP64.  (A row of four x taps summed first and weighted by an unrounded
// FP64 product took 3% less time, but transposed other weights than the
// scatter's.)
//
// Measured, 2,048 sections of 128^2 (with lists and zero fill): 4.46 -> 1.42 ms;
// 512 of 256^2 4.87 -> 1.63 ms.  It is bound by VALU issue (920 per 64
// gathered samples) with the LDS reads (one conflict-free 8-byte read per
// tap) at about half of that.
#pragma once
#include "common.hpp"
#include "insert_cells.hpp"

namespace spbp {

constexpr int GATHER_NT = 256;      // against four groups of 256, 512 threads in two took 6% more per 2,048 of 128^2, 25% per 512 of 256^2
constexpr int GATHER_GROUPS = 4;    // workgroups per CU
constexpr int GATHER_SECS = 128;    // sections of a work item at most

template <typename P>
struct GatherLds {
    static constexpr int B = CELL_EDGE + 3, NS = B * B * B, T = B / 4;
    // the region in 4 x 4 tiles of (x, y), as CellLds
    __device__ static int xpart(int x) { return ((x >> 2) << 4) | (x & 3); }
    __device__ static int ypart(int y) { return (((y >> 2) * T) << 4) | ((y & 3) << 2); }
    __device__ static int zpart(int z) { return (z * T * T) << 4; }
    f2v v[NS];
    float tab[CELL_TAB];
    P g[GATHER_SECS][6];
    f2v* out[GATHER_SECS];              // the sections' spectra
    unsigned mark[GATHER_NT / 64][64];
    int item, pnext;
};

// The gathered value of the sample at (x, y, z) in cell (xl, yl, zl) of the region.
template <typename P>
__device__ __forceinline__ f2v gather_taps(const GatherLds<P>& L, P x, P y, P z, int xl, int yl, int zl, int x0, int y0, int z0,
                                           P fltb) {
    using Lds = GatherLds<P>;
    // this lane's x and y taps in the cyclic order that gives the 16 lanes of a group distinct banks (own_taps)
    const int lane = threadIdx.x & 63;
    const int rx = (lane - xl) & 3, ry = ((lane >> 2) - yl) & 3;
    float tx[4], ty[4], tz[4];
    int xo[4], yo[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        const int dx = (t + rx) & 3, dy = (t + ry) & 3;
        xo[t] = Lds::xpart(xl + dx);
        yo[t] = Lds::ypart(yl + dy) + Lds::zpart(zl);
        tx[t] = cell_weight(L.tab, x - (P)(x0 - 1 + xl + dx), fltb);
        ty[t] = cell_weight(L.tab, y - (P)(y0 - 1 + yl + dy), fltb);
        tz[t] = cell_weight(L.tab, z - (P)(z0 - 1 + zl + t), fltb);
    }
    double re = 0.0, im = 0.0;
#pragma unroll
    for (int ly = 0; ly < 4; ++ly) {
#pragma unroll
        for (int lz = 0; lz < 4; ++lz) {
            const float tyz = __fmul_rn(ty[ly], tz[lz]);               // TY = TABI(Y) * TZ
#pragma unroll
            for (int lx = 0; lx < 4; ++lx) {
                const f2v v = L.v[xo[lx] + yo[ly] + Lds::zpart(lz)];
                const double w = (double)__fmul_rn(tx[lx], tyz);       // WG = TABI(X) * TY
                re = __fma_rn(w, (double)v.x, re);
                im = __fma_rn(w, (double)v.y, im);
            }
        }
    }
    f2v o;
    o.x = (float)re;
    o.y = (float)im;
    return o;
}

// A wave's share of an item's samples: gathered and stored in the BI layout (conjugated for a flipped sample).
template <bool EDGE, typename P>
__device__ __forceinline__ void gather_walk(GatherLds<P>& L, int ns, int nx, int N, int x0, int y0, int z0, P fltb) {
    constexpr int E = CELL_EDGE;
    const int H = nx + 1;
    unsigned* mark = L.mark[threadIdx.x >> 6];
    const P(*g)[6] = L.g;
    CellWalk wk;
    wk.s0 = wk.q0 = wk.total = wk.start = wk.cnt = 0;
    wk.lrec = wk.open = 0u;
    while (cell_sections<E, E, E, P>(wk, &L.pnext, g, ns, nx, x0, y0, z0)) {
        for (; wk.q0 < wk.total; wk.q0 += 64) {
            CellPoint<P> p;
            wk.open = cell_points<E, E, E, EDGE, P>(p, wk, mark, g, ns, nx, N, x0, y0, z0);
            if (!p.ok) continue;
            f2v v = gather_taps<P>(L, p.x, p.y, p.z, p.xc, p.yc, p.zc, x0, y0, z0, fltb);
            const int I = p.canon ? p.a : -p.a, J = p.canon ? p.b : -p.b;
            if (!p.canon) v.y = -v.y;
            *(as_global(L.out[p.s]) + ((J >= 0 ? J : J + N) * H + I)) = v;
        }
    }
}

// Persistent workgroups pull (brick, slice of its sections) items from a
// queue whose head must be zero at launch.  out holds the spectra of images
// img0 .. and must be zero: only samples are written.  The lists are those of
// the unit-cell bricks, GATHER_SECS sections per item at most.
template <typename P>
__global__ __launch_bounds__(GATHER_NT) __attribute__((amdgpu_waves_per_eu(GATHER_GROUPS * GATHER_NT / 256)))
void gather_cells_kernel(const float2* __restrict__ X, const Geom* __restrict__ geom, int img0, BrickGrid bg, int nx, int N,
                         const float* __restrict__ tab, float fltb_f, const int* __restrict__ cnt,
                         const int* __restrict__ off, const int* __restrict__ item_off, const int* __restrict__ item_key,
                         const int* __restrict__ list, float2* __restrict__ out, int* __restrict__ next_item) {
    using Lds = GatherLds<P>;
    __shared__ Lds L;
    const int H = nx + 1;
    for (int i = threadIdx.x; i < CELL_TAB; i += GATHER_NT) L.tab[i] = tab[i];
    const int total = item_off[2 * bg.nb];
    const P fltb = fltb_of<P>(fltb_f);
    for (;;) {
        __syncthreads();   // the item before is done with the region
        if (threadIdx.x == 0) {
            L.item = atomicAdd(next_item, 1);
            L.pnext = 0;
        }
        __syncthreads();
        const int item = __builtin_amdgcn_readfirstlane(L.item);
        if (item >= total) break;
        const int key = item_key[item], b = key % bg.nb;
        // the key's sections split evenly over its items
        const int i0 = item_off[key], ni = item_off[key + 1] - i0, kc = cnt[key];
        const int s_lo = (int)((long long)kc * (item - i0) / ni), ns = (int)((long long)kc * (item - i0 + 1) / ni) - s_lo;
        const int* lst = list + off[key] + s_lo;
        int x0, y0, z0;
        brick_origin(bg, b, nx, x0, y0, z0);
        for (int s = threadIdx.x; s < ns; s += GATHER_NT) {
            const Geom& g = geom[lst[s]];
#pragma unroll
            for (int k = 0; k < 6; ++k) L.g[s][k] = sizeof(P) == 8 ? (P)g.d[k] : (P)g.r[k];
            L.out[s] = (f2v*)(out + (size_t)(g.img - img0) * N * H);
        }
        for (int v = threadIdx.x; v < Lds::NS; v += GATHER_NT) {
            const int lx = v % Lds::B, r = v / Lds::B, ly = r % Lds::B, lz = r / Lds::B;
            int kx = x0 - 1 + lx, ky = y0 - 1 + ly, kz = z0 - 1 + lz;
            const bool refl = kx < 0;
            if (refl) { kx = -kx; ky = -ky; kz = -kz; }
            f2v q = {0.f, 0.f};
            if (kx <= nx && ky >= -nx + 1 && ky <= nx && kz >= -nx + 1 && kz <= nx) {   // beyond: zero-weight taps only
                const float2 t = X[((size_t)(kz >= 0 ? kz : N + kz) * N + (ky >= 0 ? ky : N + ky)) * H + kx];
                q.x = t.x;
                q.y = refl ? -t.y : t.y;
            }
            L.v[Lds::xpart(lx) + Lds::ypart(ly) + Lds::zpart(lz)] = q;
        }
        __syncthreads();
        if (cell_edge<CELL_EDGE, CELL_EDGE, CELL_EDGE>(nx, x0, y0, z0)) gather_walk<true, P>(L, ns, nx, N, x0, y0, z0, fltb);
        else gather_walk<false, P>(L, ns, nx, N, x0, y0, z0, fltb);
    }
}

}  // namespace spbp
