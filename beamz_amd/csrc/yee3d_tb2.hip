// Two-step temporally blocked 3D Yee kernel for gfx950: steps n -> n+2 of
// FDTD._update_3d_fields (beamz/simulation/fdtd.py:200-310) with the soft
// sources of helper.py:62-118 after each E update, in one pass over HBM.
//
// Every cell update is the arithmetic of the one-step fused kernel
// (yee3d_fused.hip) applied twice, so two launches of that kernel and one
// launch of this one give identical bits. The intermediate state (step n+1)
// never goes to HBM; monitor samples of it are written to a staging box.
//
// Decomposition:
//   * a workgroup of W waves owns a tile of 60 x-columns, T = W*R y-rows and a
//     z-segment [k0, k1); lane l of a wave covers column i0-2+l (lanes 0, 1,
//     62, 63 are halo lanes), wave w covers rows J0 + w*R .. J0 + w*R + R - 1,
//     with J0 = tile_y*(T-4) - 2, so the first two and last two rows of the
//     workgroup are halo rows and T-4 rows are stored;
//   * the workgroup marches z with a two-level pipeline: at iteration k it
//     computes H and E of step n+1 on plane k, H of step n+2 on plane k-1 and
//     E of step n+2 on plane k-2 (which it stores with H of step n+2 on that
//     plane). x neighbours move between lanes by wave shuffles; y neighbours
//     move between register rows and, at wave edges, through LDS (two
//     workgroup barriers per plane); z neighbours are carried in registers.
//   * a segment starting at k0 > 0 begins two planes early (recomputed halo).
// Validity: every value outside the cells the reference updates keeps its
// old value, exactly as in the one-step kernel; halo lanes, rows and planes
// (clamped in-grid reads) only feed values that are not stored.
// HBM traffic per two cell-updates: 8 reads + 6 writes of FP32 (56 B) plus
// the halo columns, rows and planes.
// What bounds it: on a large grid HBM (480x240x160: 1.228 GB a pair, 1.19 times one pass, at 4.35 TB/s, 0.89 of a large
// copy; vector ALUs 40% busy, waves waiting 64% of their time), at two workgroups of 512 per CU (97 VGPRs); on a small
// one the serial march of a segment of kseg + 3 planes. Sources and staging box sit in LDS, with the planes on which a
// wave can meet them worked out once: as kernel arguments tested on every plane they cost 130 spilled scalar registers
// and 120 VGPRs.
// us per pair before / after: 480x240x160 295 / 286, 300x200x100 112 / 97, 200x120x64 46 / 37, 120x72x40 24 / 20.
// Tried and slower: 80 VGPRs for three workgroups per CU (20 spills: 609 at 480x240x160, 31 at 120x72x40), loads one
// plane ahead (378 at 480x240x160), three rows per wave (322), 16 waves (22 at 120x72x40).
#include "common.h"

#include <algorithm>
#include <mutex>
#include <string>

// No multiply-add contraction in this file or in yee3d_fused.hip: both kernels then evaluate every
// update with the same rounded operations, which is what makes them bit-identical.
#pragma clang fp contract(off)

namespace {

constexpr int LANES = 64;
constexpr int OXT = LANES - 4;   // stored columns per wave
constexpr int NXCD = 8;
constexpr int MANY_BOXES = 3;
#define BZ_GLOBAL __attribute__((address_space(1)))

struct Fields6 {
    float* p[6];
};

struct Boxes2 {
    int n;
    int x0, y0, z0, x1, y1, z1;    // the cells the boxes cover lie in [x0, x1) x [y0, y1) x [z0, z1)
    bz_box_source b[BZ_MAX_BOX];   // b[q].amp: amplitude of step n
    float amp1[BZ_MAX_BOX];        // amplitude of step n + 1
};

struct Stage {
    float* p;   // [6][sz][sy][sx] (Ex, Ey, Ez, Hx, Hy, Hz of step n+1), or NULL
    int x0, y0, z0, sx, sy, sz;
};

// Monitor samples of the previous pair, taken by extra workgroups of a launch (n 0: none): 4 us a pair as a launch
// of its own at 120x72x40, hidden beside the tiles here.
struct Gather3D {
    const float* base0[6];       // the staging slot that holds its first step
    const int* comp;
    const int64_t* off0;
    const int64_t* off1;         // offsets into the field buffer this launch only reads (its second step)
    int n, act0, act1, nfreq;
    float* series0;
    float* series1;
    const double* phasor0;
    const double* phasor1;
    double* dft;
};

__device__ __forceinline__ float fast_rcp(float x) { return __builtin_amdgcn_rcpf(x); }

__device__ __forceinline__ float at(const float* __restrict__ base, uint32_t byte_off) {
    return *reinterpret_cast<const float*>(reinterpret_cast<const char*>(base) + byte_off);
}
__device__ __forceinline__ void put(float* __restrict__ base, uint32_t byte_off, float v) {
    *reinterpret_cast<float*>(reinterpret_cast<char*>(base) + byte_off) = v;
}

__device__ __forceinline__ void hcoef(float sig, const Coef& c, float& fa, float& fb) {
    const float s = sig * c.kh;
    const float r = fast_rcp(1.0f + s);
    fa = (1.0f - s) * r;
    fb = c.kbh * r;
}

__device__ __forceinline__ void ecoef(float sig, float eps, const Coef& c, float& ca, float& cb) {
    const float ie = fast_rcp(eps);
    const float s = sig * c.ke * ie;
    const float r = fast_rcp(1.0f + s);
    ca = (1.0f - s) * r;
    cb = c.kbe * ie * r;
}

__device__ __forceinline__ void add_box(float& ex, float& ey, float& ez, int i, int j, int k, const bz_box_source& b,
                                        float amp) {
    const int a = i - b.x0, bb = j - b.y0, cc = k - b.z0;
    if (a >= 0 && a < b.sx && bb >= 0 && bb < b.sy && cc >= 0 && cc < b.sz) {
        const long rr = ((long)cc * b.sy + bb) * b.sx + a;
        // (global, not flat, accesses, also where the pointers come from LDS)
        const float m = b.mul ? ((const BZ_GLOBAL float*)b.mul)[rr] : 1.0f;
        const float v = ((const BZ_GLOBAL float*)b.add)[rr] * amp;
        // selects, not a component-indexed write (which would place ex, ey, ez in scratch memory)
        ex = b.comp == 0 ? m * ex + v : ex;
        ey = b.comp == 1 ? m * ey + v : ey;
        ez = b.comp == 2 ? m * ez + v : ez;
    }
}

// MANY: the boxes as kernel arguments, unrolled; else from LDS, one after the other.
template <bool MANY>
__device__ __forceinline__ void add_sources(float& ex, float& ey, float& ez, int i, int j, int k, const Boxes2& src,
                                            bool second) {
    if (MANY) {
#pragma unroll
        for (int q = 0; q < BZ_MAX_BOX; ++q) {
            if (q >= src.n) break;
            add_box(ex, ey, ez, i, j, k, src.b[q], second ? src.amp1[q] : src.b[q].amp);
        }
    } else {
#pragma unroll 1
        for (int q = 0; q < src.n; ++q) add_box(ex, ey, ez, i, j, k, src.b[q], second ? src.amp1[q] : src.b[q].amp);
    }
}

// Register state of one wave's R rows carried from plane to plane.
template <int R>
struct Carry2 {
    float ex0[R], ey0[R];              // E(step n) x, y at plane k
    float h1x[R], h1y[R], h1z[R];      // H(step n+1) at plane k-1
    float fa1[R], fb1[R], ca1[R], cb1[R];   // update coefficients at plane k-1
    float e1x[R], e1y[R], e1z[R];      // E(step n+1) at plane k-1
    float f1x[R], f1y[R], f1z[R];      // E(step n+1) at plane k-2
    float h2x[R], h2y[R], h2z[R];      // H(step n+2) at plane k-2
    float g2x[R], g2y[R];              // H(step n+2) x, y at plane k-3
    float ca2[R], cb2[R];              // E coefficients at plane k-2
};

// Terms of the previous pair's two steps for (point, frequency) g, in step order: k_gather2's operations (there
// the compiler contracts each multiply and add; this file switches contraction off).
__device__ __forceinline__ void gather_prev(const Gather3D& G, const Fields6& S, long g) {
    const int p = (int)(g % G.n), k = (int)(g / G.n);
    if (k >= max(G.nfreq, 1)) return;
    const int c = G.comp[p];
    float v0 = 0.0f, v1 = 0.0f;
#pragma unroll
    for (int q = 0; q < 6; ++q)
        if (q == c) {
            if (G.act0) v0 = G.base0[q][G.off0[p]];
            if (G.act1) v1 = S.p[q][G.off1[p]];
        }
    if (k == 0) {
        if (G.act0 && G.series0) G.series0[p] = v0;
        if (G.act1 && G.series1) G.series1[p] = v1;
    }
    if (k >= G.nfreq) return;
    double* a = G.dft + 2 * ((long)k * G.n + p);
    double re = a[0], im = a[1];
    if (G.act0) {
        const double dv = (double)v0;
        re = fma(dv, G.phasor0[2 * k], re);
        im = fma(dv, G.phasor0[2 * k + 1], im);
    }
    if (G.act1) {
        const double dv = (double)v1;
        re = fma(dv, G.phasor1[2 * k], re);
        im = fma(dv, G.phasor1[2 * k + 1], im);
    }
    a[0] = re;
    a[1] = im;
}

template <int R, int W, bool MANY>
__global__ __launch_bounds__(LANES* W) void k_yee3d_tb2(Fields6 S, Fields6 D, const float* __restrict__ eps,
                                                       const float* __restrict__ sig, int nx, int ny, int nz, int ld,
                                                       int kseg, int gx, int gy, int gz, int per_xcd, Coef c,
                                                       float rdx, float rdy, float rdz, Boxes2 src_arg,
                                                       Stage stg_arg, Gather3D G) {
    constexpr int T = W * R;
    if ((int)blockIdx.x >= per_xcd * NXCD) {
        gather_prev(G, S, (long)((int)blockIdx.x - per_xcd * NXCD) * (LANES * W) + threadIdx.y * LANES + threadIdx.x);
        return;
    }
    __shared__ float xa[W][4][LANES];   // first row of each wave: Ez(n), Ex(n) at k; Ez(n+1), Ex(n+1) at k-1
    __shared__ float xh[W][2][LANES];   // last row: Hz(n+2), Hx(n+2) at k-2
    __shared__ float xb[W][2][LANES];   // last row: Hz(n+1), Hx(n+1) at k

    // the source boxes and the staging box, written before the first barrier and read after it by the few waves
    // and planes that meet them: as kernel arguments their 80 values sat in spilled scalar registers in every wave
    // (MANY, three and more boxes: as arguments all the same, since one after the other from LDS each costs a chain of
    // its own: us per pair with 4 boxes on one line, 39 from LDS and 35 as arguments at 120x72x40, 149 and 140 at
    // 240x160x100 with wide boxes; with 3 boxes of a few cells 34 and 32, 84 and 92)
    __shared__ Boxes2 src_lds;
    __shared__ Stage stg;
    if (threadIdx.x == 0 && threadIdx.y == 0) {
        if (!MANY) src_lds = src_arg;
        stg = stg_arg;
    }
    const Boxes2& src = MANY ? src_arg : src_lds;

    const int h = blockIdx.x;
    const int tile = (h % NXCD) * per_xcd + h / NXCD;
    if (tile >= gx * gy * gz) return;     // uniform over the workgroup
    const int tx = tile % gx;
    const int ty = (tile / gx) % gy;
    const int tz = tile / (gx * gy);
    const int l = threadIdx.x;
    const int w = threadIdx.y;
    const int i = tx * OXT - 2 + l;
    const int J0 = ty * (T - 4) - 2;
    const int jb = J0 + w * R;            // first row of this wave
    const int k0 = tz * kseg;
    const int k1 = min(nz, k0 + kseg);
    const uint32_t ps = (uint32_t)ny * (uint32_t)ld * 4u;
    const int ic = min(max(i, 0), nx - 1);
    uint32_t ro[R];
#pragma unroll
    for (int r = 0; r < R; ++r)
        ro[r] = ((uint32_t)min(max(jb + r, 0), ny - 1) * (uint32_t)ld + (uint32_t)ic) * 4u;
    const bool hyok = i < nx - 1;
    const bool xin = i >= 1 && i <= nx - 2;
    const bool xe = i <= nx - 2;
    const bool lane_out = l >= 2 && l <= LANES - 3 && i >= 0 && i < nx;
    const int wd = min(w + 1, W - 1), wu = max(w - 1, 0);   // neighbour waves (edge waves read their own slot)

    // planes on which this wave's rows and columns can meet a source, or the staging box (empty: never)
    const int wr = __builtin_amdgcn_readfirstlane(jb), wx = tx * OXT - 2;
    const bool src_xy = src_arg.n > 0 && wr < src_arg.y1 && wr + R > src_arg.y0 && wx < src_arg.x1 &&
                        wx + LANES > src_arg.x0;
    const int sz0 = src_xy ? src_arg.z0 : 0, sz1 = src_xy ? src_arg.z1 : 0;
    const bool stg_xy = stg_arg.p && wr < stg_arg.y0 + stg_arg.sy && wr + R > stg_arg.y0 &&
                        wx < stg_arg.x0 + stg_arg.sx && wx + LANES > stg_arg.x0;
    const int gz0 = stg_xy ? max(k0, stg_arg.z0) : 0, gz1 = stg_xy ? min(k1, stg_arg.z0 + stg_arg.sz) : 0;

    Carry2<R> C;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        C.h1x[r] = C.h1y[r] = C.h1z[r] = 0.0f;
        C.e1x[r] = C.e1y[r] = C.e1z[r] = 0.0f;
        C.f1x[r] = C.f1y[r] = C.f1z[r] = 0.0f;
        C.h2x[r] = C.h2y[r] = C.h2z[r] = 0.0f;
        C.g2x[r] = C.g2y[r] = 0.0f;
        // the coefficients of sigma 0, eps 1 (planes before the march has loaded any)
        hcoef(0.0f, c, C.fa1[r], C.fb1[r]);
        ecoef(0.0f, 1.0f, c, C.ca1[r], C.cb1[r]);
        C.ca2[r] = C.ca1[r];
        C.cb2[r] = C.cb1[r];
    }
    const int kstart = k0 > 0 ? k0 - 2 : 0;
    {
        const uint32_t kp = (uint32_t)min(max(kstart, 0), nz - 1) * ps;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            C.ex0[r] = at(S.p[0], kp + ro[r]);
            C.ey0[r] = at(S.p[1], kp + ro[r]);
        }
    }

    for (int k = kstart; k <= k1 + 1; ++k) {
        // ---- loads of plane k (E x, y of plane k+1) ----
        const uint32_t kp = (uint32_t)min(max(k, 0), nz - 1) * ps;
        const uint32_t kq = (uint32_t)min(max(k + 1, 0), nz - 1) * ps;
        float ex1[R], ey1[R], ez[R], hx[R], hy[R], hz[R], sg[R], ee[R];
#pragma unroll
        for (int r = 0; r < R; ++r) {
            ex1[r] = at(S.p[0], kq + ro[r]);
            ey1[r] = at(S.p[1], kq + ro[r]);
            ez[r] = at(S.p[2], kp + ro[r]);
            hx[r] = at(S.p[3], kp + ro[r]);
            hy[r] = at(S.p[4], kp + ro[r]);
            hz[r] = at(S.p[5], kp + ro[r]);
            sg[r] = at(sig, kp + ro[r]);
            ee[r] = at(eps, kp + ro[r]);
        }
        // the update coefficients of plane k, once: step n+1 uses them here, step n+2 one and two planes later
        float fa0[R], fb0[R], ca0[R], cb0[R];
#pragma unroll
        for (int r = 0; r < R; ++r) {
            hcoef(sg[r], c, fa0[r], fb0[r]);
            ecoef(sg[r], ee[r], c, ca0[r], cb0[r]);
        }
        // ---- exchange A: first rows go up a wave, last rows go down ----
        xa[w][0][l] = ez[0];
        xa[w][1][l] = C.ex0[0];
        xa[w][2][l] = C.e1z[0];
        xa[w][3][l] = C.e1x[0];
        xh[w][0][l] = C.h2z[R - 1];
        xh[w][1][l] = C.h2x[R - 1];
        __syncthreads();
        const float dEz0 = xa[wd][0][l], dEx0 = xa[wd][1][l], dE1z = xa[wd][2][l], dE1x = xa[wd][3][l];
        const float uH2z = xh[wu][0][l], uH2x = xh[wu][1][l];

        // ---- H of step n+1 at plane k ----
        float h1x[R], h1y[R], h1z[R];
        {
            const bool kh = k < nz - 1;
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const int j = jb + r;
                const float ezN = r + 1 < R ? ez[r + 1] : dEz0;
                const float exN = r + 1 < R ? C.ex0[r + 1] : dEx0;
                const float ezR = __shfl_down(ez[r], 1, LANES);
                const float eyR = __shfl_down(C.ey0[r], 1, LANES);
                const float fa = fa0[r], fb = fb0[r];
                const bool jh = j < ny - 1;
                h1x[r] = (kh && jh) ? fa * hx[r] - fb * ((ezN - ez[r]) * rdy - (ey1[r] - C.ey0[r]) * rdz) : hx[r];
                h1y[r] = (kh && hyok) ? fa * hy[r] - fb * ((ex1[r] - C.ex0[r]) * rdz - (ezR - ez[r]) * rdx) : hy[r];
                h1z[r] = (jh && hyok) ? fa * hz[r] - fb * ((eyR - C.ey0[r]) * rdx - (exN - C.ex0[r]) * rdy) : hz[r];
            }
        }
        // ---- exchange B: last row of H(n+1) goes down a wave ----
        xb[w][0][l] = h1z[R - 1];
        xb[w][1][l] = h1x[R - 1];
        __syncthreads();
        const float uH1z = xb[wu][0][l], uH1x = xb[wu][1][l];

        // ---- E of step n+1 at plane k ----
        float e1x[R], e1y[R], e1z[R];
        {
            const bool kin = k >= 1 && k <= nz - 2;
            const bool kz = k <= nz - 2;
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const int j = jb + r;
                const float hzU = r > 0 ? h1z[r - 1] : uH1z;
                const float hxU = r > 0 ? h1x[r - 1] : uH1x;
                const float hzL = __shfl_up(h1z[r], 1, LANES);
                const float hyL = __shfl_up(h1y[r], 1, LANES);
                const bool yin = j >= 1 && j <= ny - 2;
                const float ca = ca0[r], cb = cb0[r];
                float ex = (kin && yin && xe) ? ca * C.ex0[r] + cb * ((h1z[r] - hzU) * rdy - (h1y[r] - C.h1y[r]) * rdz)
                                              : C.ex0[r];
                float ey = (kin && j <= ny - 2 && xin)
                               ? ca * C.ey0[r] + cb * ((h1x[r] - C.h1x[r]) * rdz - (h1z[r] - hzL) * rdx)
                               : C.ey0[r];
                float ezz = (kz && yin && xin) ? ca * ez[r] + cb * ((h1y[r] - hyL) * rdx - (h1x[r] - hxU) * rdy) : ez[r];
                if (k >= sz0 && k < sz1) add_sources<MANY>(ex, ey, ezz, i, j, k, src, false);
                e1x[r] = ex;
                e1y[r] = ey;
                e1z[r] = ezz;
            }
        }
        // ---- monitor samples of step n+1 (owned cells inside the staging box) ----
        if (k >= gz0 && k < gz1 && lane_out) {
            const long plane = (long)stg.sz * stg.sy * stg.sx;
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const int j = jb + r;
                const int a = i - stg.x0, b = j - stg.y0, cc = k - stg.z0;
                if (j >= J0 + 2 && j < J0 + T - 2 && j < ny && a >= 0 && a < stg.sx && b >= 0 && b < stg.sy &&
                    cc >= 0 && cc < stg.sz) {
                    BZ_GLOBAL float* q = (BZ_GLOBAL float*)stg.p + ((long)cc * stg.sy + b) * stg.sx + a;
                    q[0] = e1x[r];
                    q[plane] = e1y[r];
                    q[2 * plane] = e1z[r];
                    q[3 * plane] = h1x[r];
                    q[4 * plane] = h1y[r];
                    q[5 * plane] = h1z[r];
                }
            }
        }

        // ---- H of step n+2 at plane m = k-1 ----
        float h2x[R], h2y[R], h2z[R];
        {
            const int m = k - 1;
            const bool kh = m < nz - 1;
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const int j = jb + r;
                const float ezN = r + 1 < R ? C.e1z[r + 1] : dE1z;
                const float exN = r + 1 < R ? C.e1x[r + 1] : dE1x;
                const float ezR = __shfl_down(C.e1z[r], 1, LANES);
                const float eyR = __shfl_down(C.e1y[r], 1, LANES);
                const float fa = C.fa1[r], fb = C.fb1[r];
                const bool jh = j < ny - 1;
                h2x[r] = (kh && jh) ? fa * C.h1x[r] - fb * ((ezN - C.e1z[r]) * rdy - (e1y[r] - C.e1y[r]) * rdz)
                                    : C.h1x[r];
                h2y[r] = (kh && hyok) ? fa * C.h1y[r] - fb * ((e1x[r] - C.e1x[r]) * rdz - (ezR - C.e1z[r]) * rdx)
                                      : C.h1y[r];
                h2z[r] = (jh && hyok) ? fa * C.h1z[r] - fb * ((eyR - C.e1y[r]) * rdx - (exN - C.e1x[r]) * rdy)
                                      : C.h1z[r];
            }
        }
        // ---- E of step n+2 at plane m2 = k-2, stores of plane m2 ----
        {
            const int m2 = k - 2;
            const bool kin = m2 >= 1 && m2 <= nz - 2;
            const bool kz = m2 <= nz - 2;
            const bool kst = m2 >= k0 && m2 < k1;
            const uint32_t mp = (uint32_t)max(m2, 0) * ps;
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const int j = jb + r;
                const float hzU = r > 0 ? C.h2z[r - 1] : uH2z;
                const float hxU = r > 0 ? C.h2x[r - 1] : uH2x;
                const float hzL = __shfl_up(C.h2z[r], 1, LANES);
                const float hyL = __shfl_up(C.h2y[r], 1, LANES);
                const bool yin = j >= 1 && j <= ny - 2;
                const float ca = C.ca2[r], cb = C.cb2[r];
                float ex = (kin && yin && xe)
                               ? ca * C.f1x[r] + cb * ((C.h2z[r] - hzU) * rdy - (C.h2y[r] - C.g2y[r]) * rdz)
                               : C.f1x[r];
                float ey = (kin && j <= ny - 2 && xin)
                               ? ca * C.f1y[r] + cb * ((C.h2x[r] - C.g2x[r]) * rdz - (C.h2z[r] - hzL) * rdx)
                               : C.f1y[r];
                float ezz = (kz && yin && xin) ? ca * C.f1z[r] + cb * ((C.h2y[r] - hyL) * rdx - (C.h2x[r] - hxU) * rdy)
                                               : C.f1z[r];
                if (kst && lane_out && j >= J0 + 2 && j < J0 + T - 2 && j < ny) {
                    if (m2 >= sz0 && m2 < sz1) add_sources<MANY>(ex, ey, ezz, i, j, m2, src, true);
                    const uint32_t o = mp + ro[r];
                    put(D.p[0], o, ex);
                    put(D.p[1], o, ey);
                    put(D.p[2], o, ezz);
                    put(D.p[3], o, C.h2x[r]);
                    put(D.p[4], o, C.h2y[r]);
                    put(D.p[5], o, C.h2z[r]);
                }
            }
        }
        // ---- rotate the carried planes ----
#pragma unroll
        for (int r = 0; r < R; ++r) {
            C.g2x[r] = C.h2x[r];
            C.g2y[r] = C.h2y[r];
            C.h2x[r] = h2x[r];
            C.h2y[r] = h2y[r];
            C.h2z[r] = h2z[r];
            C.f1x[r] = C.e1x[r];
            C.f1y[r] = C.e1y[r];
            C.f1z[r] = C.e1z[r];
            C.e1x[r] = e1x[r];
            C.e1y[r] = e1y[r];
            C.e1z[r] = e1z[r];
            C.h1x[r] = h1x[r];
            C.h1y[r] = h1y[r];
            C.h1z[r] = h1z[r];
            C.ca2[r] = C.ca1[r];
            C.cb2[r] = C.cb1[r];
            C.fa1[r] = fa0[r];
            C.fb1[r] = fb0[r];
            C.ca1[r] = ca0[r];
            C.cb1[r] = cb0[r];
            C.ex0[r] = ex1[r];
            C.ey0[r] = ey1[r];
        }
        // No barrier here: every wave read the exchange-A slots before barrier B and the exchange-B slots
        // before it can reach the next barrier A, so the next iteration's writes cannot race those reads.
    }
}

template <int R, int W>
int launch(const Fields6& S, const Fields6& D, const float* eps, const float* sig, int nx, int ny, int nz, int ld,
           int kseg, const Coef& c, float rdx, float rdy, float rdz, const Boxes2& bs, const Stage& stg,
           const Gather3D& G, hipStream_t st) {
    constexpr int T = W * R;
    const int gx = (nx + OXT - 1) / OXT;
    const int gy = (ny + (T - 4) - 1) / (T - 4);
    const int gz = (nz + kseg - 1) / kseg;
    const int n = gx * gy * gz;
    const int per_xcd = (n + NXCD - 1) / NXCD;
    const long gt = (long)G.n * (G.nfreq > 0 ? G.nfreq : 1);
    const dim3 grid(per_xcd * NXCD + (unsigned)((gt + LANES * W - 1) / (LANES * W)));
    const auto kern = bs.n >= MANY_BOXES ? k_yee3d_tb2<R, W, true> : k_yee3d_tb2<R, W, false>;
    hipLaunchKernelGGL(kern, grid, dim3(LANES, W), 0, st, S, D, eps, sig, nx, ny, nz, ld, kseg, gx, gy,
                       gz, per_xcd, c, rdx, rdy, rdz, bs, stg, G);
    BZ_CHECK_LAUNCH("bz_yee3d_step2");
    return BZ_OK;
}

// One pair of checked arguments.
int launch_pair(const Fields6& S, const Fields6& D, const float* eps, const float* sig, int nx, int ny, int nz, int ld,
                int kseg, int rows, int waves, const Coef& c, float rx, float ry, float rz, const Boxes2& bs,
                const Stage& stg, const Gather3D& G, hipStream_t st) {
    if (waves == 16) return launch<2, 16>(S, D, eps, sig, nx, ny, nz, ld, kseg, c, rx, ry, rz, bs, stg, G, st);
    switch (rows) {
        case 2: return launch<2, 8>(S, D, eps, sig, nx, ny, nz, ld, kseg, c, rx, ry, rz, bs, stg, G, st);
        case 3: return launch<3, 8>(S, D, eps, sig, nx, ny, nz, ld, kseg, c, rx, ry, rz, bs, stg, G, st);
        default: return launch<4, 8>(S, D, eps, sig, nx, ny, nz, ld, kseg, c, rx, ry, rz, bs, stg, G, st);
    }
}

// The checks and the launch structs that bz_yee3d_step2 and bz_yee3d_run2 share.
int check_pair(const std::string& name, float* const src[6], float* const dst[6], const float* eps_r,
               const float* sigma, int nx, int ny, int nz, int ld, const bz_box_source* boxes, const float* amps,
               int nbox, const float* stage, const int* stage_box, int& kseg, int rows, int waves, Boxes2& bs,
               Stage& stg, Fields6& S, Fields6& D) {
    BZ_REQUIRE(src && dst && eps_r && sigma, name + ": null pointer");
    for (int q = 0; q < 6; ++q)
        BZ_REQUIRE(src[q] && dst[q] && src[q] != dst[q], name + ": bad field buffers");
    BZ_REQUIRE(nx >= 2 && ny >= 2 && nz >= 2 && ld >= nx, name + ": bad shape");
    BZ_REQUIRE(4.0 * nz * ny * ld < 4294967295.0, name + ": a field array exceeds 4 GiB (32-bit offsets)");
    BZ_REQUIRE(nbox >= 0 && nbox <= BZ_MAX_BOX && (nbox == 0 || (boxes && amps)), name + ": bad source list");
    bs = Boxes2{};
    bs.n = nbox;
    for (int q = 0; q < nbox; ++q) {
        const bz_box_source& b = boxes[q];
        BZ_REQUIRE(b.comp >= 0 && b.comp <= 2 && b.add && b.sx > 0 && b.sy > 0 && b.sz > 0 && b.x0 >= 0 &&
                       b.y0 >= 0 && b.z0 >= 0 && b.x0 + b.sx <= nx && b.y0 + b.sy <= ny && b.z0 + b.sz <= nz,
                   name + ": source box outside the grid");
        bs.b[q] = b;
        bs.x0 = q ? std::min(bs.x0, b.x0) : b.x0;
        bs.y0 = q ? std::min(bs.y0, b.y0) : b.y0;
        bs.z0 = q ? std::min(bs.z0, b.z0) : b.z0;
        bs.x1 = q ? std::max(bs.x1, b.x0 + b.sx) : b.x0 + b.sx;
        bs.y1 = q ? std::max(bs.y1, b.y0 + b.sy) : b.y0 + b.sy;
        bs.z1 = q ? std::max(bs.z1, b.z0 + b.sz) : b.z0 + b.sz;
    }
    stg.p = const_cast<float*>(stage);
    stg.x0 = stg.y0 = stg.z0 = stg.sx = stg.sy = stg.sz = 0;
    if (stage) {
        BZ_REQUIRE(stage_box, name + ": staging buffer without its box");
        stg.x0 = stage_box[0];
        stg.y0 = stage_box[1];
        stg.z0 = stage_box[2];
        stg.sx = stage_box[3];
        stg.sy = stage_box[4];
        stg.sz = stage_box[5];
        BZ_REQUIRE(stg.sx > 0 && stg.sy > 0 && stg.sz > 0 && stg.x0 >= 0 && stg.y0 >= 0 && stg.z0 >= 0 &&
                       stg.x0 + stg.sx <= nx && stg.y0 + stg.sy <= ny && stg.z0 + stg.sz <= nz,
                   name + ": staging box outside the grid");
    }
    if (kseg <= 0) kseg = 32;
    BZ_REQUIRE(kseg >= 2, name + ": kseg must be at least 2");
    BZ_REQUIRE(waves == 8 || (waves == 16 && rows == 2), name + ": waves must be 8 (rows 2, 3, 4) or 16 (rows 2)");
    if (rows < 2 || rows > 4) {
        bz::set_error(name + ": rows must be 2, 3 or 4");
        return BZ_EINVAL;
    }
    for (int q = 0; q < 6; ++q) {
        S.p[q] = src[q];
        D.p[q] = dst[q];
    }
    return BZ_OK;
}

}  // namespace

extern "C" int bz_yee3d_step2(float* const src[6], float* const dst[6], const float* eps_r, const float* sigma,
                              int nx, int ny, int nz, int ld, double dx, double dy, double dz, double dt, double mu0,
                              double eps0, const bz_box_source* boxes, const float* amp1, int nbox, float* stage,
                              const int* stage_box, int kseg, int rows, int waves, void* stream) {
    Boxes2 bs;
    Stage stg;
    Fields6 S, D;
    const int rc = check_pair("bz_yee3d_step2", src, dst, eps_r, sigma, nx, ny, nz, ld, boxes, amp1, nbox, stage,
                              stage_box, kseg, rows, waves, bs, stg, S, D);
    if (rc != BZ_OK) return rc;
    for (int q = 0; q < nbox; ++q) bs.amp1[q] = amp1[q];
    return launch_pair(S, D, eps_r, sigma, nx, ny, nz, ld, kseg, rows, waves, make_coef(dt, mu0, eps0),
                       (float)(1.0 / dx), (float)(1.0 / dy), (float)(1.0 / dz), bs, stg, Gather3D{},
                       (hipStream_t)stream);
}

extern "C" int bz_yee3d_run2(float* const src[6], float* const dst[6], const float* eps_r, const float* sigma, int nx,
                             int ny, int nz, int ld, double dx, double dy, double dz, double dt, double mu0,
                             double eps0, const bz_box_source* boxes, const float* amps, int nbox, int npairs,
                             float* stage, const int* stage_box, const bz_gather_table* tables, int ntables, int kseg,
                             int rows, int waves, void* stream) {
    BZ_REQUIRE(npairs >= 0 && ntables >= 0 && (ntables == 0 || (tables && stage && stage_box)),
               "bz_yee3d_run2: bad arguments");
    for (int t = 0; t < ntables; ++t) {
        const bz_gather_table& g = tables[t];
        BZ_REQUIRE(g.n > 0 && g.comp && g.stage_off && g.off && g.row && g.nfreq >= 0 &&
                       (g.nfreq == 0 || (g.phasor && g.dft)),
                   "bz_yee3d_run2: incomplete monitor table");
        BZ_REQUIRE((long)g.n * (g.nfreq > 0 ? g.nfreq : 1) / 256 < (1L << 31) - 1,
                   "bz_yee3d_run2: too many points x frequencies");
    }
    Boxes2 bs;
    Stage stg;
    Fields6 F[2];
    const int rc = check_pair("bz_yee3d_run2", src, dst, eps_r, sigma, nx, ny, nz, ld, boxes, amps, nbox, stage,
                              stage_box, kseg, rows, waves, bs, stg, F[0], F[1]);
    if (rc != BZ_OK || npairs == 0) return rc;
    const Coef c = make_coef(dt, mu0, eps0);
    const float rx = (float)(1.0 / dx), ry = (float)(1.0 / dy), rz = (float)(1.0 / dz);
    const hipStream_t st = (hipStream_t)stream;
    const long cells = (long)stg.sx * stg.sy * stg.sz;
    const bool fused = ntables == 1;
    auto slot = [&](int q) { return fused ? q & 1 : 0; };
    // table t's arguments for pair q: its first step's samples in staging slot `slot(q)`
    auto of_pair = [&](int t, int q) {
        const bz_gather_table& g = tables[t];
        Gather3D G{};
        const int r0 = g.row[2 * q], r1 = g.row[2 * q + 1];
        if (r0 < 0 && r1 < 0) return G;
        for (int k = 0; k < 6; ++k) G.base0[k] = stage + (6 * slot(q) + k) * cells;
        G.comp = g.comp;
        G.off0 = g.stage_off;
        G.off1 = g.off;
        G.n = g.n;
        G.act0 = r0 >= 0;
        G.act1 = r1 >= 0;
        G.nfreq = g.nfreq;
        if (r0 >= 0 && g.series) G.series0 = g.series + (long)r0 * g.n;
        if (r1 >= 0 && g.series) G.series1 = g.series + (long)r1 * g.n;
        if (r0 >= 0 && g.nfreq) G.phasor0 = g.phasor + 2L * r0 * g.nfreq;
        if (r1 >= 0 && g.nfreq) G.phasor1 = g.phasor + 2L * r1 * g.nfreq;
        G.dft = g.dft;
        return G;
    };
    auto gather = [&](const Gather3D& G, const Fields6& after) {
        if (G.n == 0) return (int)BZ_OK;
        const float* base1[6];
        for (int k = 0; k < 6; ++k) base1[k] = after.p[k];
        return bz_gather2(G.base0, G.off0, base1, G.comp, G.off1, G.n, G.act0, G.act1, G.series0, G.series1, G.nfreq,
                          G.phasor0, G.phasor1, G.dft, stream);
    };
    // One call, since a pair on a small grid is shorter than its two Python calls were (33 us at 120x72x40; now 20 per
    // pair with the samples). With one table, pair q - 1's samples are taken by extra workgroups of pair q's launch:
    // its first step sits in the staging slot that launch does not write, its second step in the buffer that launch
    // only reads
    for (int q = 0; q < npairs; ++q) {
        for (int k = 0; k < nbox; ++k) {
            bs.b[k].amp = amps[(long)2 * q * nbox + k];
            bs.amp1[k] = amps[(long)(2 * q + 1) * nbox + k];
        }
        bool need = false;
        for (int t = 0; t < ntables; ++t) need = need || tables[t].row[2 * q] >= 0;
        Stage sq = stg;
        sq.p = need ? stage + 6 * slot(q) * cells : nullptr;
        const Fields6 &S = F[q & 1], &D = F[(q & 1) ^ 1];
        const int e = launch_pair(S, D, eps_r, sigma, nx, ny, nz, ld, kseg, rows, waves, c, rx, ry, rz, bs, sq,
                                  fused && q > 0 ? of_pair(0, q - 1) : Gather3D{}, st);
        if (e != BZ_OK) return e;
        for (int t = 0; t < ntables && (!fused || q == npairs - 1); ++t) {
            const int g = gather(of_pair(t, q), D);
            if (g != BZ_OK) return g;
        }
    }
    return BZ_OK;
}

// ---------------- allocation-free variant: staging box in a library-owned device array ----------------
// bz_yee3d_step2 with a staging box, then bz_gather2 of both steps' samples, where the box lives in
// `scratch`, a file-scope device array (one copy per GPU, held until the process ends). Its address on a
// device is looked up once, with that device current, and kept per device: the array's name is a host-side
// stand-in that no kernel may be given.
namespace {
static __device__ __align__(256) float scratch[BZ_NOALLOC_STAGE_FLOATS];

constexpr int MAX_DEVICES = 64;
float* g_scratch[MAX_DEVICES] = {};
std::mutex g_scratch_mu;

int scratch_ptr(float** out) {
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return bz::hip_fail("bz_yee3d_step2_noalloc: hipGetDevice", e);
    BZ_REQUIRE(dev >= 0 && dev < MAX_DEVICES, "bz_yee3d_step2_noalloc: device index beyond 64");
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch[dev]) {
        void* p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return bz::hip_fail("bz_yee3d_step2_noalloc: hipGetSymbolAddress", e);
        BZ_REQUIRE(p, "bz_yee3d_step2_noalloc: no device address for the staging array");
        g_scratch[dev] = static_cast<float*>(p);
    }
    *out = g_scratch[dev];
    return BZ_OK;
}
}  // namespace

extern "C" int bz_yee3d_step2_noalloc(float* const src[6], float* const dst[6], const float* eps_r,
                                      const float* sigma, int nx, int ny, int nz, int ld, double dx, double dy,
                                      double dz, double dt, double mu0, double eps0, const bz_box_source* boxes,
                                      const float* amp1, int nbox, const int* stage_box, const int* comp,
                                      const int64_t* stage_off, const int64_t* field_off, int npts, int act0,
                                      int act1, float* series0, float* series1, int nfreq, const double* phasor0,
                                      const double* phasor1, double* dft, int kseg, int rows, int waves,
                                      void* stream) {
    BZ_REQUIRE(npts >= 0, "bz_yee3d_step2_noalloc: negative point count");
    const bool sample = npts > 0 && (act0 || act1);
    float* stage = nullptr;
    if (sample) {
        BZ_REQUIRE(stage_box && comp && stage_off && field_off, "bz_yee3d_step2_noalloc: monitor table incomplete");
        BZ_REQUIRE(stage_box[3] > 0 && stage_box[4] > 0 && stage_box[5] > 0,
                   "bz_yee3d_step2_noalloc: empty staging box");
        const double need = 6.0 * stage_box[3] * stage_box[4] * stage_box[5];
        if (need > (double)BZ_NOALLOC_STAGE_FLOATS) {
            bz::set_error("bz_yee3d_step2_noalloc: staging box of " + std::to_string((long long)need) +
                          " floats exceeds the library's " + std::to_string(BZ_NOALLOC_STAGE_FLOATS) +
                          "-float array");
            return BZ_EINVAL;
        }
        const int rc = scratch_ptr(&stage);
        if (rc != BZ_OK) return rc;
    }
    int rc = bz_yee3d_step2(src, dst, eps_r, sigma, nx, ny, nz, ld, dx, dy, dz, dt, mu0, eps0, boxes, amp1, nbox,
                            stage, sample ? stage_box : nullptr, kseg, rows, waves, stream);
    if (rc != BZ_OK || !sample) return rc;
    // the staged step n+1 is every cell of the box, written by the launch above before this gather reads it
    // (same stream), so the array needs no clearing
    const long plane = (long)stage_box[3] * stage_box[4] * stage_box[5];
    const float* base0[6];
    const float* base1[6];
    for (int c = 0; c < 6; ++c) {
        base0[c] = stage + c * plane;
        base1[c] = dst[c];
    }
    return bz_gather2(base0, stage_off, base1, comp, field_off, npts, act0, act1, series0, series1, nfreq, phasor0,
                      phasor1, dft, stream);
}
