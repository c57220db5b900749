// insert_cells.hpp -- the ONELINE scatter with samples binned by unit cell.
//
// A brick owns the samples whose effective position E (after the Friedel
// flip) lies in its box of CX x CY x CZ unit cells [x, x + 1).  The KB table
// vanishes beyond 1.8 voxels, so a sample's nonzero taps lie, per axis, in
// floor(E) - 1 .. floor(E) + 2: every sample of a cell writes the same 4x4x4
// window of the brick's LDS region (the cells plus 1 voxel before and 2
// after).  These are always among the reference's taps (the nearest voxel
// and two to each side, oneline.f:77-152), whose others carry zero weight.
//
// With one LDS add per tap and component the scatter is bound by LDS atomic
// issue (a ds_add_u64 wave instruction costs ~6.35 CU-cycles) with the VALU
// close behind.  So a work item first bins its samples: a pass over its
// sections stores every sample (lattice point, section, spectrum value: 12
// bytes) in a pool in LDS and links it to its cell.  Then each lane takes up
// to four samples of one cell and adds their terms for a tap in registers
// before one LDS add.  The terms, their fixed-point encoding and so the sums
// are insert_brick_kernel's (each term rounded once, the weights to units of
// 2^-WBITS, see CELL_WOFF; the sums exact).  The table is in LDS too: as
// global loads its lookups, 64 scattered addresses each, took the cache's tag
// rate (20.4 -> 18.8 ms, below).
//
// Measured against the nearest-voxel bricks, insertion per 20,000 images of
// 128^2 (8 of 9 samples grouped by four, ~118 sections and ~5,900 samples per
// item): 22.8 -> 14.8 ms; 24,000 of 256^2: 111 -> 74 ms; 6,000 of 128^2 with
// FP64 geometry 10.9 -> 5.1 ms.  What bounds it now is VALU issue: of ~38 us per
// item 12 bin (~210 VALU per 64 lattice points), 18 add groups (~1,930 VALU
// per 64 groups of four), 2 flush, 6 wait at the barriers between.  Choices,
// insertion per 20,000 images of 128^2: cells of fixed slots with the
// overflow added singly 16.0 ms; rank by compare-and-swap against a chain
// walked per cell 14.6 / 14.3; 9x9x5 cells in two groups per CU 19.8 (their
// bricks hold too few samples per section); products of unrounded FP64
// weights, fewer instructions but more registers, 17.2 against 16.0.
//
// Reflected taps (p_x < 0, written conjugated at -p) are exactly the region's
// layer kx = -1 of the bricks at kx = 0: the flush sends that layer to
// (1, -ky, -kz), conjugated, so no second pass over the samples is needed.
#pragma once
#include "common.hpp"
#include "insert.hpp"

namespace spbp {

constexpr int CELL_POOL = 6336;   // samples an item groups at a time (12 bytes and a link each)
constexpr unsigned CELL_THREE = 0x8000u;   // list entry of a group of three
constexpr int CELL_TAB = 3336;    // table entries a window's taps reach (distances up to 2 voxels)
constexpr int CELL_SECS = 120;    // sections of a work item at most
constexpr int CELL_SECS64 = 96;   // with FP64 geometry
constexpr int CELL_NT = 768;      // threads per workgroup, one workgroup per CU
constexpr int CELL_EDGE = 9;      // cells per brick edge
// Weights are positive, so a tap's sum over four samples is formed from 2^52
// up, not from the middle of [2^52, 2^53) as signed terms are (fixed_term): at
// four weights of exactly 1, the most it can be, it ends at 2^53, whose bit
// pattern still is that of 2^52 plus the sum.
constexpr double CELL_WOFF = 4503599627370496.0;                       // 2^52
constexpr unsigned long long CELL_WOFF_BITS = 0x4330000000000000ull;   // its bits
static_assert(4.0 * WSCALE <= 4503599627370496.0, "four weights of at most 1 stay within 2^52 units");

__device__ __forceinline__ void add_global(Global<float> p, float v) {
    (void)__hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// A work item: the sections of one brick and half, CELL_SECS at most.
struct CellItem {
    int item, job, x0, y0, z0, half, ns, edge, e;   // item < 0: none; e: its largest |Re|, |Im| is below 2^e
};

// Region layout: 4 x 4 tiles of (x, y) as in TileLds, each lane's taps in the
// order that gives the 16 lanes of a group 16 distinct bank pairs.
template <int CX, int CY, int CZ, int NT, bool WGT, typename P>
struct CellLds {
    static constexpr int BX = CX + 3, BY = CY + 3, BZ = CZ + 3, NS = BX * BY * BZ, NC = CX * CY * CZ;
    static_assert(BX % 4 == 0 && BY % 4 == 0, "the tile layout needs x and y edges divisible by 4");
    static constexpr int POOL = sizeof(P) == 8 ? CELL_POOL - 256 : CELL_POOL;
    static_assert(POOL < (int)CELL_THREE && NC <= NT, "16-bit links and entries; one thread per cell");
    static constexpr int TX = BX / 4, TY = BY / 4;
    __device__ static int xpart(int x) { return ((x >> 2) << 4) | (x & 3); }
    __device__ static int ypart(int y) { return (((y >> 2) * TX) << 4) | ((y & 3) << 2); }
    __device__ static int zpart(int z) { return (z * TY * TX) << 4; }
    __device__ static void coords(int v, int& x, int& y, int& z) {
        const int t = v >> 4;
        x = ((t % TX) << 2) | (v & 3);
        y = (((t / TX) % TY) << 2) | ((v >> 2) & 3);
        z = t / (TX * TY);
    }
    static constexpr int SECS = sizeof(P) == 8 ? CELL_SECS64 : CELL_SECS;
    unsigned long long re[NS], im[NS], w[WGT ? NS : 1];
    float2 val[POOL];                     // the item's samples: value,
    unsigned rec[POOL];                   // cell_rec,
    unsigned short next[POOL];            // and the sample before it in the same cell
    unsigned head[NC];                    // per cell: samples so far << 16 | the last one
    // the item's groups, each by its last sample: of four, or three (CELL_THREE), from 0; of two from POOL / 3 up;
    // of one from the end down (a cell has one group of less than three at most)
    unsigned short list[POOL / 3 + NC];
    float tab[CELL_TAB];
    P g[2][SECS][6];                      // the sections of this item and the next: DM(1..6)
    const float2* spec[2][SECS];          // their spectra
    unsigned mark[NT / 64][64];
    CellItem info[2];
    int pnext, tnext, npool, blocked, nl[3];
};

// A binned sample: lattice point (a, b) with E = a DM(1:3) + b DM(4:6), and
// the section's place in the round.
__device__ __forceinline__ unsigned cell_rec(int a, int b, int s) {
    return (unsigned)(a + 1024) | ((unsigned)(b + 1024) << 12) | ((unsigned)s << 24);
}

// E of lattice point (a, b), with sample_pos's operations (the negated sample
// of a Friedel flip has exactly the negated position).
__device__ __forceinline__ void cell_pos(const float* g, int a, int b, float& x, float& y, float& z) {
    const float fa = (float)a, fb = (float)b;
    x = __fadd_rn(__fmul_rn(fa, g[0]), __fmul_rn(fb, g[3]));
    y = __fadd_rn(__fmul_rn(fa, g[1]), __fmul_rn(fb, g[4]));
    z = __fadd_rn(__fmul_rn(fa, g[2]), __fmul_rn(fb, g[5]));
}
__device__ __forceinline__ void cell_pos(const double* g, int a, int b, double& x, double& y, double& z) {
    const double fa = (double)a, fb = (double)b;
    x = __dadd_rn(__dmul_rn(fa, g[0]), __dmul_rn(fb, g[3]));
    y = __dadd_rn(__dmul_rn(fa, g[1]), __dmul_rn(fb, g[4]));
    z = __dadd_rn(__dmul_rn(fa, g[2]), __dmul_rn(fb, g[5]));
}

// kb_weight's table index without roundf's sequence: for 0 <= x < 2^22,
// adding the largest value below one half and truncating rounds half away
// from zero, as roundf does (checked for every float in [0, 5000) on the CPU).
__host__ __device__ __forceinline__ int half_away(float x) { return (int)(x + 0.49999997f); }
__host__ __device__ __forceinline__ int half_away(double x) { return (int)(x + 0.49999999999999994); }
__device__ __forceinline__ float cell_weight(const float* tab, float d, float fltb) {
    const unsigned o = (unsigned)half_away(__fmul_rn(fabsf(d), fltb)) << 2;   // unsigned: a 32-bit offset from a scalar base
    return *(const float*)((const char*)tab + o);
}
__device__ __forceinline__ float cell_weight(const float* tab, double d, double fltb) {
    const unsigned o = (unsigned)half_away(__dmul_rn(fabs(d), fltb)) << 2;
    return *(const float*)((const char*)tab + o);
}

// The terms of K samples of one cell, summed per tap and added to the region.
// rec[0] is a sample; rec[k], k >= n, are not (their weights are zeroed).
template <int K, typename Lds, typename P, bool WGT>
__device__ __forceinline__ void cell_taps(Lds& L, const P (*g)[6], const unsigned (&rec)[K], const float2 (&v)[K], int n, int xl, int yl,
                                          int zl, int x0, int y0, int z0, const float* tab, P fltb,
                                          double vscale, double wscale) {
    const int lane = threadIdx.x & 63;
    const int rx = (lane - xl) & 3, ry = ((lane >> 2) - yl) & 3;
    int x8[4], y8[4];
    P px[4], py[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        const int dx = (t + rx) & 3, dy = (t + ry) & 3;
        x8[t] = Lds::xpart(xl + dx) * 8;
        y8[t] = Lds::ypart(yl + dy) * 8;
        px[t] = (P)(x0 - 1 + xl + dx);
        py[t] = (P)(y0 - 1 + yl + dy);
    }
    float tx[K][4], ty[K][4];
    P zk[K];
    double vx[K], vy[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const unsigned r = k < n ? rec[k] : rec[0];
        P x, y, z;
        cell_pos(g[r >> 24], (int)(r & 0xFFFu) - 1024, (int)((r >> 12) & 0xFFFu) - 1024, x, y, z);
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            tx[k][t] = cell_weight(L.tab, x - px[t], fltb);
            ty[k][t] = cell_weight(L.tab, y - py[t], fltb);
        }
        zk[k] = z;
        vx[k] = (double)v[k].x * vscale;
        vy[k] = (double)v[k].y * vscale;
    }
    // one z layer at a time (rolled: its weights are looked up here; unrolled, the registers would not fit 768 threads)
    int z8 = Lds::zpart(zl) * 8;
    P pz = (P)(z0 - 1 + zl);
#pragma unroll 1
    for (int lz = 0; lz < 4; ++lz, z8 += Lds::zpart(1) * 8, pz += (P)1) {
        float tz[K];
#pragma unroll
        for (int k = 0; k < K; ++k) {
            tz[k] = cell_weight(L.tab, zk[k] - pz, fltb);
            if (K > 1) tz[k] = k < n ? tz[k] : 0.0f;
        }
#pragma unroll
        for (int ly = 0; ly < 4; ++ly) {
            constexpr double OFF = 6755399441055744.0;   // 1.5 * 2^52 (fixed_term)
            const int row = y8[ly] + z8;
            float tyz[K];
#pragma unroll
            for (int k = 0; k < K; ++k) tyz[k] = __fmul_rn(ty[k][ly], tz[k]);     // TY = TABI(Y) * TZ
#pragma unroll
            for (int lx = 0; lx < 4; ++lx) {
                double re = OFF, im = OFF, w = CELL_WOFF;
#pragma unroll
                for (int k = 0; k < K; ++k) {
                    const double wd = (double)__fmul_rn(tx[k][lx], tyz[k]);       // WG = TABI(X) * TY
                    re = __fma_rn(vx[k], wd, re);
                    im = __fma_rn(vy[k], wd, im);
                    if constexpr (WGT) w = __fma_rn(wd, wscale, w);
                }
                const int ob = row + x8[lx];
                lds_add(L.re, ob, (unsigned long long)__double_as_longlong(re));
                lds_add(L.im, ob, (unsigned long long)__double_as_longlong(im));
                if constexpr (WGT) lds_add(L.w, ob, (unsigned long long)__double_as_longlong(w));
            }
        }
    }
}

// Inclusive sum over the wave by DPP row shifts and row broadcasts.
__device__ __forceinline__ int wave_scan(int v) {
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);   // row_shr:1
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);   // row_shr:2
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);   // row_shr:4
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);   // row_shr:8
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);   // row_bcast:15
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);   // row_bcast:31
    return v;
}

// A wave's place in an item's sections.
struct CellWalk {
    int s0, q0, total;         // first of the current sections, next point of their sequence, its length
    int start, cnt;            // this lane's line: first point in the sequence, points
    unsigned lrec, open;       // its record; the line open at q0
};
// A lattice point of the walk: E = a DM(1:3) + b DM(4:6) of section s, its cell in the brick; `canon`: (a, b) is the
// sample (I, J) itself, else its Friedel twin (-I, -J).
template <typename P>
struct CellPoint {
    int a, b, s, xc, yc, zc;
    P x, y, z;
    bool ok, canon;
};
// Lattice lines of a section across the cells' box (at most the diagonal + 2), sections a wave takes at a time.
template <int CX, int CY, int CZ>
struct CellLines {
    static constexpr double D2 = (CX + 0.04) * (CX + 0.04) + (CY + 0.04) * (CY + 0.04) + (CZ + 0.04) * (CZ + 0.04);
    static constexpr int LINES = 21;
    static constexpr int WSEC = 64 / LINES;
    static_assert(D2 <= (LINES - 2) * (LINES - 2), "a section crosses at most the box diagonal + 2 lines");
};

// The next sections of the walk (WSEC from *pnext), LINES lanes each: a lane
// computes the interval of one lattice line in the cells' box, and a scan lays
// the intervals end to end.  False past the last section (no points then).
template <int CX, int CY, int CZ, typename P>
__device__ __forceinline__ bool cell_sections(CellWalk& wk, int* pnext, const P (*g)[6], int ns, int nx, int x0, int y0,
                                              int z0) {
    using Ln = CellLines<CX, CY, CZ>;
    const int lane = threadIdx.x & 63;
    const int sec = lane / Ln::LINES, line = lane - sec * Ln::LINES;
    int s0 = 0;
    if (lane == 0) s0 = atomicAdd(pnext, Ln::WSEC);
    wk.s0 = __builtin_amdgcn_readfirstlane(s0);
    wk.q0 = 0;
    // this lane's line b of section s: lattice points a0 .. a0 + cnt - 1
    const float lo[3] = {x0 - 0.02f, y0 - 0.02f, z0 - 0.02f};
    const float hi[3] = {x0 + CX + 0.02f, y0 + CY + 0.02f, z0 + CZ + 0.02f};
    const int s = min(wk.s0 + sec, ns - 1);
    float r2[3];
    float bmn = 0.f, bmx = 0.f;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        r2[k] = (float)g[s][3 + k];
        const float u = r2[k] * lo[k], w = r2[k] * hi[k];
        bmn += fminf(u, w);
        bmx += fmaxf(u, w);
    }
    const int b = (int)ceilf(bmn - 0.01f) + line;
    const float bb = (float)b;
    float amin = -(float)nx, amax = (float)nx;   // |a|, |b| <= nx <= 1024: the records' fields
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        // 1 / DM, |DM| below 10^-6 taken as 10^-6: the line's points then lie inside the box's slab or
        // outside it for every |a| <= 1024, as they do for the true value
        const float d = (float)g[s][k], r1 = __builtin_amdgcn_rcpf(fabsf(d) > 1e-6f ? d : 1e-6f);
        const float off = bb * r2[k];
        const float u = (lo[k] - off) * r1, w = (hi[k] - off) * r1;
        amin = fmaxf(amin, fminf(u, w));
        amax = fminf(amax, fmaxf(u, w));
    }
    const int a0 = (int)ceilf(amin - 0.001f);
    wk.cnt = max(0, (int)floorf(amax + 0.001f) - a0 + 1);
    if (!(sec < Ln::WSEC && wk.s0 + sec < ns && bb <= bmx + 0.01f && abs(b) <= nx)) wk.cnt = 0;
    const int pref = wave_scan(wk.cnt);
    wk.total = __builtin_amdgcn_readlane(pref, 63);
    wk.start = pref - wk.cnt;
    // line record: a - q for its points (q: position in the sequence), b, section
    wk.lrec = (unsigned)(a0 - wk.start + 2048) | ((unsigned)(b + 1024) << 13) | ((unsigned)sec << 25) | 0x80000000u;
    return wk.s0 < ns;
}

// The next 64 points of the walk, one per lane (wk.q0 stays).  A line's first
// point among the 64 marks its lane with the line; every lane takes the last
// mark at or before it, or the line that was open before.  Returns the
// record of the line open after the 64.  EDGE: the brick may hold lattice
// points that are no samples (outside the disk, outside ONELINE's bounds, or
// the flipped twin at kx = 0).
template <int CX, int CY, int CZ, bool EDGE, typename P>
__device__ __forceinline__ unsigned cell_points(CellPoint<P>& t, const CellWalk& wk, unsigned* mark, const P (*g)[6], int ns,
                                                int nx, int N, int x0, int y0, int z0) {
    const int lane = threadIdx.x & 63;
    mark[lane] = 0u;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    if (wk.cnt > 0 && (unsigned)(wk.start - wk.q0) < 64u) mark[wk.start - wk.q0] = wk.lrec;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    const unsigned m = mark[lane];
    const unsigned long long M = __ballot(m != 0u) & ((2ull << lane) - 1ull);
    unsigned ln = (unsigned)__shfl((int)m, M ? 63 - __clzll((long long)M) : 0, 64);
    if (!M) ln = wk.open;
    const int q = wk.q0 + lane;
    t.a = (int)(ln & 0x1FFFu) - 2048 + q;
    t.b = (int)((ln >> 13) & 0xFFFu) - 1024;
    t.s = min(wk.s0 + (int)((ln >> 25) & 3u), ns - 1);
    cell_pos(g[t.s], t.a, t.b, t.x, t.y, t.z);
    t.xc = (int)floor(t.x) - x0;
    t.yc = (int)floor(t.y) - y0;
    t.zc = (int)floor(t.z) - z0;
    t.ok = q < wk.total && (unsigned)t.xc < (unsigned)CX && (unsigned)t.yc < (unsigned)CY && (unsigned)t.zc < (unsigned)CZ;
    t.canon = t.a > 0 || (t.a == 0 && t.b >= 0);
    if constexpr (EDGE) {
        t.ok = t.ok && t.a * t.a + t.b * t.b < nx * nx;                   // oneline.f:53-55
        t.ok = t.ok && (t.canon || t.x > (P)0);                           // oneline.f:60-67 (E_x >= 0 holds)
        t.ok = t.ok && in_bounds(nearest_voxel(t.x, N), nearest_voxel(t.y, N), nearest_voxel(t.z, N), nx);
    }
    return (unsigned)__builtin_amdgcn_readlane((int)ln, 63);
}
// May the brick at (x0, y0, z0) hold a lattice point that is no sample?
template <int CX, int CY, int CZ>
__device__ __forceinline__ bool cell_edge(int nx, int x0, int y0, int z0) {
    const int fx = x0 + CX, fy = max(-y0, y0 + CY), fz = max(-z0, z0 + CZ);
    return x0 == 0 || fx > nx - 3 || y0 < -nx + 4 || y0 + CY > nx - 3 || z0 < -nx + 4 || z0 + CZ > nx - 3 ||
           fx * fx + fy * fy + fz * fz >= (nx - 1) * (nx - 1);
}

// Bin the item's sections (geometry buffer `buf`) until they or the pool end;
// true: the pool ended, call again when it is empty.  Two sets of 64 points
// are in flight: a set's spectrum values are stored while the next set's are
// on their way.
template <int CX, int CY, int CZ, int NT, bool EDGE, bool WGT, typename P>
__device__ __forceinline__ bool cell_bin(CellLds<CX, CY, CZ, NT, WGT, P>& L, CellWalk& wk, int buf, int ns, int nx, int N,
                                         int x0, int y0, int z0) {
    using Lds = CellLds<CX, CY, CZ, NT, WGT, P>;
    const int H = nx + 1;
    const int lane = threadIdx.x & 63;
    unsigned* mark = L.mark[threadIdx.x >> 6];
    const P(*g)[6] = L.g[buf];
    const unsigned long long below = (1ull << lane) - 1ull;
    // 64 points on their way: record, signs, value, cell, place in the pool (< 0: no sample)
    struct Set {
        unsigned rec, sg;
        f2v val;
        int cell, slot;
    };
    bool blocked = false, ended = false;
    // The next 64 points.  No early way out: every set loads, so that the wait for a set's values is for them alone;
    // past the last section or a full pool a set holds no samples.
    auto take = [&](Set& t) {
        if (wk.q0 >= wk.total) ended = !cell_sections<CX, CY, CZ, P>(wk, &L.pnext, g, ns, nx, x0, y0, z0);
        CellPoint<P> p;
        const unsigned open = cell_points<CX, CY, CZ, EDGE, P>(p, wk, mark, g, ns, nx, N, x0, y0, z0);
        const unsigned long long mk = __ballot(p.ok);
        const int n = (int)__popcll(mk);
        int base = 0;
        if (lane == 0) base = atomicAdd(&L.npool, n);
        {
            // spectrum_value: sign (-1)^(I + J), conjugated, and conjugated back for a flipped sample.  Every lane
            // loads, the section's first value where no sample is
            const int I = p.canon ? p.a : -p.a, J = p.canon ? p.b : -p.b;
            t.val = *(Global<const f2v>)(as_global(L.spec[buf][p.s]) + (p.ok ? (J >= 0 ? J : J + N) * H + I : 0));
        }
        t.sg = ((unsigned)((p.a + p.b) & 1) << 31) | (p.canon ? 1u : 0u);
        t.rec = cell_rec(p.a, p.b, p.s);
        t.cell = (p.zc * CY + p.yc) * CX + p.xc;
        base = __builtin_amdgcn_readfirstlane(base);
        // no room: these points again when the pool is empty (npool stays past its end until then)
        const bool room = base + n <= Lds::POOL;
        t.slot = p.ok && room ? base + (int)__popcll(mk & below) : -1;
        blocked = !room;
        if (room) {
            wk.open = open;
            wk.q0 += 64;
        }
    };
    // store a set
    auto put = [&](const Set& t) {
        unsigned prev = 0;
        float2 v = make_float2(__uint_as_float(__float_as_uint(t.val.x) ^ (t.sg & 0x80000000u)),
                               __uint_as_float(__float_as_uint(t.val.y) ^ (t.sg & 0x80000000u) ^ (t.sg << 31)));
        asm volatile("" : "+v"(v.x), "+v"(v.y));   // formed here, outside the branch: see take's load
        if (t.slot >= 0) {
            // the cell's count and last sample change together
            unsigned old = __hip_atomic_load(&L.head[t.cell], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            do {
                prev = old;
                old = atomicCAS(&L.head[t.cell], prev, ((prev & 0xFFFF0000u) + 0x10000u) | (unsigned)t.slot);
            } while (old != prev);
            L.rec[t.slot] = t.rec;
            L.next[t.slot] = (unsigned short)prev;
            L.val[t.slot] = v;
        }
        // every fourth sample of a cell completes a group
        const bool four = t.slot >= 0 && (prev >> 16 & 3u) == 3u;
        const unsigned long long m4 = __ballot(four);
        if (m4 != 0ull) {
            int base = 0;
            if (lane == 0) base = atomicAdd(&L.nl[0], (int)__popcll(m4));
            base = __builtin_amdgcn_readfirstlane(base);
            if (four) L.list[base + (int)__popcll(m4 & below)] = (unsigned short)t.slot;
        }
    };
    Set t0, t1;
    take(t0);
    while (!blocked && !ended) {
        take(t1);
        put(t0);
        take(t0);
        put(t1);
    }
    put(t0);
    return blocked;
}

// The group of list entry p: K samples of a cell (of four, the last may be missing).
template <int K, typename Lds, typename P, bool WGT>
__device__ __forceinline__ void cell_group(Lds& L, const P (*g)[6], unsigned p, int x0, int y0, int z0, const float* tab,
                                           P fltb, double vscale, double wscale) {
    unsigned r[K];
    float2 v[K];
    const int n = K == 4 && (p & CELL_THREE) ? 3 : K;
    p &= CELL_THREE - 1u;
#pragma unroll
    for (int k = 0; k < K; ++k) {
        r[k] = L.rec[p];
        v[k] = L.val[p];
        if (k + 1 < K) p = k + 1 < n ? L.next[p] : p;
    }
    if (n < K) v[K - 1] = make_float2(0.f, 0.f);
    P x, y, z;
    cell_pos(g[r[0] >> 24], (int)(r[0] & 0xFFFu) - 1024, (int)((r[0] >> 12) & 0xFFFu) - 1024, x, y, z);
    cell_taps<K, Lds, P, WGT>(L, g, r, v, n, (int)floor(x) - x0, (int)floor(y) - y0, (int)floor(z) - z0, x0, y0, z0, tab,
                                   fltb, vscale, wscale);
}

// One wave takes the next work item from the queue and puts its description
// and its sections' geometry into buffer `buf`.
template <int CX, int CY, int CZ, int NT, bool WGT, typename P>
__device__ __forceinline__ void cell_load(CellLds<CX, CY, CZ, NT, WGT, P>& L, int buf, const BrickJob* __restrict__ jobs,
                                          const int* jbase, int total, int* __restrict__ next_item) {
    const int lane = threadIdx.x & 63;
    int gitem = 0;
    if (lane == 0) gitem = atomicAdd(next_item, 1);
    gitem = __builtin_amdgcn_readfirstlane(gitem);
    if (gitem >= total) {
        if (lane == 0) L.info[buf].item = -1;
        return;
    }
    int j = 0;
    while (gitem >= jbase[j + 1]) ++j;
    const BrickJob& J = jobs[j];
    const int nx = J.nx, item = gitem - jbase[j];
    const int key = as_global(J.item_key)[item];
    const int b = key % J.bg.nb, half = key / J.bg.nb;
    // the key's sections split evenly over its items
    const int i0 = as_global(J.item_off)[key], ni = as_global(J.item_off)[key + 1] - i0, kc = as_global(J.cnt)[key];
    const int s_lo = (int)((long long)kc * (item - i0) / ni), ns = (int)((long long)kc * (item - i0 + 1) / ni) - s_lo;
    const Global<const int> lst = as_global(J.list) + as_global(J.off)[key] + s_lo;
    const size_t nspec = (size_t)J.N * (nx + 1);
    float m = 0.0f;
    for (int s = lane; s < ns; s += 64) {
        const Global<const Geom> g = as_global(J.geom) + lst[s];
        const int img = g->img - J.img0;
        m = fmaxf(m, as_global(J.vmax)[img]);
#pragma unroll
        for (int k = 0; k < 6; ++k) L.g[buf][s][k] = sizeof(P) == 8 ? (P)g->d[k] : (P)g->r[k];
        L.spec[buf][s] = J.spec + (size_t)img * nspec;
    }
    for (int off = 32; off > 0; off >>= 1) m = fmaxf(m, __shfl_down(m, off, 64));
    if (lane == 0) {
        CellItem c;
        c.item = gitem;
        c.job = j;
        brick_origin(J.bg, b, nx, c.x0, c.y0, c.z0);
        c.half = half;
        c.ns = ns;
        c.edge = cell_edge<CX, CY, CZ>(nx, c.x0, c.y0, c.z0);
        // fixed-point unit (as insert_brick_kernel's): terms below 2^VBITS units
        c.e = 0;
        if (m > 0.0f && isfinite(m)) (void)frexpf(m, &c.e);
        L.info[buf] = c;
    }
}

// Persistent workgroups, one per CU (the region and the cells' slots fill its
// LDS), pull (job, brick and half, slice of its sections) items from one
// queue as insert_brick_kernel's do.  Per item: bin, list the groups left in
// the cells, add the groups (again while the pool fills before the sections
// end), flush.  While the groups are added one wave loads the next item's
// sections; a wave that has flushed its part of the region goes on to bin the
// next item.  The queue head must be zero at launch.
template <int CX, int CY, int CZ, typename P, int NT, bool WGT>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(NT / 256))) void insert_cells_kernel(
    const BrickJob* __restrict__ jobs, int njobs, int* __restrict__ next_item) {
    using Lds = CellLds<CX, CY, CZ, NT, WGT, P>;
    __shared__ Lds L;
    __shared__ int jbase[MAX_JOBS + 1];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (threadIdx.x == 0) {
        int acc = 0;
        for (int j = 0; j < njobs; ++j) {
            jbase[j] = acc;
            acc += jobs[j].item_off[2 * jobs[j].bg.nb];
        }
        jbase[njobs] = acc;
        L.pnext = 0;
        L.tnext = 0;
        L.npool = 0;
        L.blocked = 0;
        L.nl[0] = L.nl[1] = L.nl[2] = 0;
    }
    for (int i = threadIdx.x; i < Lds::NC; i += NT) L.head[i] = 0u;
    for (int i = threadIdx.x; i < Lds::NS; i += NT) {
        L.re[i] = 0ull;
        L.im[i] = 0ull;
        if constexpr (WGT) L.w[i] = 0ull;
    }
    __syncthreads();
    const int total = jbase[njobs];
    if (wave == 0) cell_load<CX, CY, CZ, NT, WGT, P>(L, 0, jobs, jbase, total, next_item);
    __syncthreads();
    int job = -1;   // whose table is in LDS
    for (int buf = 0;; buf ^= 1) {
        if (__builtin_amdgcn_readfirstlane(L.info[buf].item) < 0) break;
        const int j = __builtin_amdgcn_readfirstlane(L.info[buf].job), ns = __builtin_amdgcn_readfirstlane(L.info[buf].ns);
        const int x0 = __builtin_amdgcn_readfirstlane(L.info[buf].x0), y0 = __builtin_amdgcn_readfirstlane(L.info[buf].y0),
                  z0 = __builtin_amdgcn_readfirstlane(L.info[buf].z0);
        const int e = __builtin_amdgcn_readfirstlane(L.info[buf].e);
        const bool half = __builtin_amdgcn_readfirstlane(L.info[buf].half) != 0,
                   edge = __builtin_amdgcn_readfirstlane(L.info[buf].edge) != 0;
        const BrickJob& J = jobs[j];
        const int nx = J.nx, N = J.N, H = nx + 1;
        if (j != job) {   // another context's table
            for (int i = threadIdx.x; i < CELL_TAB; i += NT) L.tab[i] = as_global(J.tab)[i];
            job = j;
            __syncthreads();
        }
        const float* tab = L.tab;
        const P fltb = fltb_of<P>(J.fltb);
        const double vscale = ldexp(1.0, VBITS - e), vinv = ldexp(1.0, e - VBITS);
        const double wscale = J.wscale;   // a run-time value: kept in registers
        CellWalk wk;
        wk.s0 = wk.q0 = wk.total = wk.start = wk.cnt = 0;
        wk.lrec = wk.open = 0u;
        for (bool again = true, first = true; again; first = false) {
            const bool bl = edge ? cell_bin<CX, CY, CZ, NT, true, WGT, P>(L, wk, buf, ns, nx, N, x0, y0, z0)
                                 : cell_bin<CX, CY, CZ, NT, false, WGT, P>(L, wk, buf, ns, nx, N, x0, y0, z0);
            if (bl && lane == 0) L.blocked = 1;
            __syncthreads();
            again = __builtin_amdgcn_readfirstlane(L.blocked) != 0;   // part of the sections is left for another round
            // the samples past each cell's last whole group of four, a lane per cell
            if (wave * 64 < Lds::NC) {
                const int c = threadIdx.x;
                const unsigned long long below = (1ull << lane) - 1ull;
                unsigned h = 0;
                if (c < Lds::NC) {
                    h = L.head[c];
                    L.head[c] = 0u;
                }
                const int rest = (int)(h >> 16 & 3u);
                const unsigned long long m3 = __ballot(rest == 3), m2 = __ballot(rest == 2), m1 = __ballot(rest == 1);
                int base = 0;
                if (lane < 3) base = atomicAdd(&L.nl[lane], (int)(lane == 0 ? __popcll(m3) : lane == 1 ? __popcll(m2) : __popcll(m1)));
                const int b3 = __builtin_amdgcn_readlane(base, 0), b2 = Lds::POOL / 3 + __builtin_amdgcn_readlane(base, 1),
                          b1 = Lds::POOL / 3 + Lds::NC - 1 - __builtin_amdgcn_readlane(base, 2);
                if (rest == 3) L.list[b3 + (int)__popcll(m3 & below)] = (unsigned short)(h | CELL_THREE);
                if (rest == 2) L.list[b2 + (int)__popcll(m2 & below)] = (unsigned short)h;
                if (rest == 1) L.list[b1 - (int)__popcll(m1 & below)] = (unsigned short)h;
            }
            __syncthreads();
            if (threadIdx.x == 0) {
                L.npool = 0;
                L.blocked = 0;
                if (!again) L.pnext = 0;
            }
            if (first && wave == NT / 64 - 1) cell_load<CX, CY, CZ, NT, WGT, P>(L, buf ^ 1, jobs, jbase, total, next_item);
            const int n4 = L.nl[0], n2 = L.nl[1], n1 = L.nl[2];
            const int t4 = (n4 + 63) / 64, t2 = t4 + (n2 + 63) / 64, t1 = t2 + (n1 + 63) / 64;   // 64 groups to a task
            const P(*g)[6] = L.g[buf];
            for (;;) {
                int t = 0;
                if (lane == 0) t = atomicAdd(&L.tnext, 1);
                t = __builtin_amdgcn_readfirstlane(t);
                if (t >= t1) break;
                if (t < t4) {
                    const int i = t * 64 + lane;
                    if (i < n4) cell_group<4, Lds, P, WGT>(L, g, L.list[i], x0, y0, z0, tab, fltb, vscale, wscale);
                } else if (t < t2) {
                    const int i = (t - t4) * 64 + lane;
                    if (i < n2)
                        cell_group<2, Lds, P, WGT>(L, g, L.list[Lds::POOL / 3 + i], x0, y0, z0, tab, fltb, vscale, wscale);
                } else {
                    const int i = (t - t2) * 64 + lane;
                    if (i < n1)
                        cell_group<1, Lds, P, WGT>(L, g, L.list[Lds::POOL / 3 + Lds::NC - 1 - i], x0, y0, z0, tab, fltb, vscale,
                                                        wscale);
                }
            }
            __syncthreads();
            if (threadIdx.x == 0) {
                L.tnext = 0;
                L.nl[0] = L.nl[1] = L.nl[2] = 0;
            }
            __syncthreads();
        }
        // add the region to the half grid and zero it; its layer kx = -1 holds the reflected taps
        const Global<float> X = as_global((float*)(half ? J.X1 : J.X0));
        [[maybe_unused]] const Global<float> W = as_global(half ? J.W1 : J.W0);
        [[maybe_unused]] float* __restrict__ Wc = half ? J.Wc1 : J.Wc0;   // null unless compensated weights
        for (int v = threadIdx.x; v < Lds::NS; v += NT) {
            const unsigned long long sre = L.re[v];
            if (sre == 0ull) continue;   // no tap reached the voxel (n = 0)
            const unsigned long long sim = L.im[v];
            [[maybe_unused]] const unsigned long long sw = WGT ? L.w[v] : 0ull;
            L.re[v] = 0ull;
            L.im[v] = 0ull;
            if constexpr (WGT) L.w[v] = 0ull;
            int lx, ly, lz;
            Lds::coords(v, lx, ly, lz);
            int kx = x0 - 1 + lx, ky = y0 - 1 + ly, kz = z0 - 1 + lz;
            const bool refl = kx < 0;
            if (refl) { kx = -kx; ky = -ky; kz = -kz; }
            if (kx > nx || ky < -nx + 1 || ky > nx || kz < -nx + 1 || kz > nx) continue;
            const size_t o = ((size_t)(kz >= 0 ? kz : N + kz) * N + (ky >= 0 ? ky : N + ky)) * H + kx;
            const long long tre = fixed_sum48(sre), tim = fixed_sum48(sim);
            if constexpr (WGT) {
                const long long tw = (long long)(sw - (unsigned long long)fixed_count(sre, tre) * CELL_WOFF_BITS);
                if (tw == 0 && tre == 0 && tim == 0) continue;   // zero-weight taps only
                const double wd = __dmul_rn((double)tw, WINV);
                const float wi = (float)wd;
                if (Wc) twosum_atomic_add((float*)W, Wc, o, wi, (float)(wd - (double)wi));
                else if (W) add_global(W + o, wi);
            }
            const double di = __dmul_rn((double)tim, vinv);
            add_global(X + 2 * o, (float)__dmul_rn((double)tre, vinv));
            add_global(X + 2 * o + 1, (float)(refl ? -di : di));
        }
    }
}

}  // namespace spbp
