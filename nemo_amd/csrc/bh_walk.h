// Device code shared by the group walks (bh_walk.hip, bh_team.hip): wave
// reductions, the interaction tiles, the local expansions and the walks'
// arguments.  The tiles' arithmetic is written once, so that every walk gives
// a tile the same sums.
#pragma once

#include "bh_ctx.h"

namespace bh {
namespace {

__device__ __forceinline__ int lane_id() { return threadIdx.x & 63; }

__device__ __forceinline__ void wave_lds_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ float wave_min(float v)
{
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) v = fminf(v, __shfl_xor(v, d, 64));
    return v;
}
__device__ __forceinline__ float wave_max(float v)
{
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) v = fmaxf(v, __shfl_xor(v, d, 64));
    return v;
}
__device__ __forceinline__ int wave_min_i(int v)
{
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) v = min(v, __shfl_xor(v, d, 64));
    return v;
}
__device__ __forceinline__ int wave_max_i(int v)
{
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) v = max(v, __shfl_xor(v, d, 64));
    return v;
}
__device__ __forceinline__ int wave_excl_scan(int v, int *total)
{
    const int lane = lane_id();
    int x = v;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        int t = __shfl_up(x, d, 64);
        if (lane >= d) x += t;
    }
    *total = __shfl(x, 63, 64);
    return x - v;
}
__device__ __forceinline__ int mbcnt(unsigned long long m)
{
    return __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0));
}

// TwoSum fold of a tile sum into a compensated accumulator.
__device__ __forceinline__ void fold(float &hi, float &lo, float v)
{
    float s = hi + v;
    float bb = s - hi;
    float err = (hi - (s - bb)) + (v - bb);
    hi = s;
    lo += err;
}

__device__ __forceinline__ float rsq(float x) { return __builtin_amdgcn_rsqf(x); }

template <int NPL>
struct Lane {
    float px[NPL], py[NPL], pz[NPL];
    float axh[NPL], axl[NPL], ayh[NPL], ayl[NPL], azh[NPL], azl[NPL], ph[NPL], pl[NPL];
};

// Sums of one tile: cnt sources on the particles (px, py, pz)[q], q < NQ.
template <int NQ, bool SOFT0>
__device__ __forceinline__ void tile_p2p(const float *px, const float *py, const float *pz, const float4 *src, int cnt,
                                         float eps2, float *sx, float *sy, float *sz, float *sp)
{
#pragma unroll
    for (int q = 0; q < NQ; q++) sx[q] = sy[q] = sz[q] = sp[q] = 0.f;
#pragma unroll 4
    for (int j = 0; j < cnt; j++) {
        const float4 s = src[j];
#pragma unroll
        for (int q = 0; q < NQ; q++) {
            float dx = s.x - px[q], dy = s.y - py[q], dz = s.z - pz[q];
            float r2 = fmaf(dx, dx, fmaf(dy, dy, fmaf(dz, dz, eps2)));
            float ri = rsq(r2);
            if (SOFT0) ri = r2 > 0.f ? ri : 0.f;
            float mr = s.w * ri;
            sp[q] += mr;
            float mr3 = mr * ri * ri;
            sx[q] = fmaf(dx, mr3, sx[q]);
            sy[q] = fmaf(dy, mr3, sy[q]);
            sz[q] = fmaf(dz, mr3, sz[q]);
        }
    }
}

// NQ <= NPL: the particle slots in use (a group of at most 64 points uses
// one slot per lane).
template <int NPL, int NQ, bool SOFT0>
__device__ __forceinline__ void eval_p2p(Lane<NPL> &L, const float4 *src, int cnt, float eps2)
{
    float sx[NQ], sy[NQ], sz[NQ], sp[NQ];
    tile_p2p<NQ, SOFT0>(L.px, L.py, L.pz, src, cnt, eps2, sx, sy, sz, sp);
#pragma unroll
    for (int q = 0; q < NQ; q++) {
        fold(L.axh[q], L.axl[q], sx[q]);
        fold(L.ayh[q], L.ayl[q], sy[q]);
        fold(L.azh[q], L.azl[q], sz[q]);
        fold(L.ph[q], L.pl[q], sp[q]);
    }
}

// P2C entry: e[0] = (dx0, dy0, dz0, m) relative to the group centre,
// e[1] = (qxx, qxy, qxz, qyy), e[2] = (qyz, qzz, -, -).
template <int NQ, bool QUAD, bool SOFT0>
__device__ __forceinline__ void tile_p2c(const float *px, const float *py, const float *pz, const float4 *src, int cnt,
                                         float eps2, float *sx, float *sy, float *sz, float *sp)
{
    constexpr int S = QUAD ? 3 : 1;
#pragma unroll
    for (int q = 0; q < NQ; q++) sx[q] = sy[q] = sz[q] = sp[q] = 0.f;
#pragma unroll 2
    for (int j = 0; j < cnt; j++) {
        const float4 s = src[S * j];
        float4 q0, q1;
        if (QUAD) {
            q0 = src[S * j + 1];
            q1 = src[S * j + 2];
        }
#pragma unroll
        for (int q = 0; q < NQ; q++) {
            float dx = s.x - px[q], dy = s.y - py[q], dz = s.z - pz[q];
            float r2 = fmaf(dx, dx, fmaf(dy, dy, fmaf(dz, dz, eps2)));
            float ri = rsq(r2);
            if (SOFT0) ri = r2 > 0.f ? ri : 0.f;
            float ri2 = ri * ri;
            float mr = s.w * ri;
            if (QUAD) {
                float qx = fmaf(q0.x, dx, fmaf(q0.y, dy, q0.z * dz));
                float qy = fmaf(q0.y, dx, fmaf(q0.w, dy, q1.x * dz));
                float qz = fmaf(q0.z, dx, fmaf(q1.x, dy, q1.y * dz));
                float dqd = fmaf(dx, qx, fmaf(dy, qy, dz * qz));
                float r5 = ri2 * ri2 * ri;
                float phq = -0.5f * r5 * dqd;          // quadrupole potential term
                float coef = (mr - 5.f * phq) * ri2;   // radial factor of a
                sp[q] += mr - phq;
                sx[q] = fmaf(dx, coef, fmaf(-qx, r5, sx[q]));
                sy[q] = fmaf(dy, coef, fmaf(-qy, r5, sy[q]));
                sz[q] = fmaf(dz, coef, fmaf(-qz, r5, sz[q]));
            } else {
                float mr3 = mr * ri2;
                sp[q] += mr;
                sx[q] = fmaf(dx, mr3, sx[q]);
                sy[q] = fmaf(dy, mr3, sy[q]);
                sz[q] = fmaf(dz, mr3, sz[q]);
            }
        }
    }
}

template <int NPL, int NQ, bool QUAD, bool SOFT0>
__device__ __forceinline__ void eval_p2c(Lane<NPL> &L, const float4 *src, int cnt, float eps2)
{
    float sx[NQ], sy[NQ], sz[NQ], sp[NQ];
    tile_p2c<NQ, QUAD, SOFT0>(L.px, L.py, L.pz, src, cnt, eps2, sx, sy, sz, sp);
#pragma unroll
    for (int q = 0; q < NQ; q++) {
        fold(L.axh[q], L.axl[q], sx[q]);
        fold(L.ayh[q], L.ayl[q], sy[q]);
        fold(L.azh[q], L.azl[q], sz[q]);
        fold(L.ph[q], L.pl[q], sp[q]);
    }
}

// Tiles for the first nq particle slots of each lane (groups of at most
// 64 nq points leave the other slots idle).
template <int NPL, bool SOFT0>
__device__ __forceinline__ void p2p_slots(int nq, Lane<NPL> &L, const float4 *src, int cnt, float eps2)
{
    if (nq <= 1) eval_p2p<NPL, 1, SOFT0>(L, src, cnt, eps2);
    else if (NPL > 2 && nq == 2) eval_p2p<NPL, (NPL > 2 ? 2 : NPL), SOFT0>(L, src, cnt, eps2);
    else if (NPL > 3 && nq == 3) eval_p2p<NPL, (NPL > 3 ? 3 : NPL), SOFT0>(L, src, cnt, eps2);
    else eval_p2p<NPL, NPL, SOFT0>(L, src, cnt, eps2);
}

template <int NPL, bool QUAD, bool SOFT0>
__device__ __forceinline__ void p2c_slots(int nq, Lane<NPL> &L, const float4 *src, int cnt, float eps2)
{
    if (nq <= 1) eval_p2c<NPL, 1, QUAD, SOFT0>(L, src, cnt, eps2);
    else if (NPL > 2 && nq == 2) eval_p2c<NPL, (NPL > 2 ? 2 : NPL), QUAD, SOFT0>(L, src, cnt, eps2);
    else if (NPL > 3 && nq == 3) eval_p2c<NPL, (NPL > 3 ? 3 : NPL), QUAD, SOFT0>(L, src, cnt, eps2);
    else eval_p2c<NPL, NPL, QUAD, SOFT0>(L, src, cnt, eps2);
}

// Local expansion coefficients, in the order G0, G1 (x y z), G2 (xx xy xz yy
// yz zz), G3 (xxx xxy xxz xyy xyz xzz yyy yyz yzz zzz).
constexpr int kLoc = 20;

// v + (v of another lane chosen by the DPP control CTRL); rows outside RM add 0.
template <int CTRL, int RM = 0xF>
__device__ __forceinline__ float dpp_add(float v)
{
    return v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, RM, 0xF, true));
}

// Sum over the wave, valid in lane 63: quad swaps (xor 1, xor 2), half-row
// and row mirrors (sums of 8 and 16 lanes), then row 15 -> next row and
// lane 31 -> rows 2-3 broadcasts.  All VALU, no LDS round trips.
__device__ __forceinline__ float wave_sum63(float v)
{
    v = dpp_add<0xB1>(v);          // quad_perm [1,0,3,2]
    v = dpp_add<0x4E>(v);          // quad_perm [2,3,0,1]
    v = dpp_add<0x141>(v);         // row_half_mirror
    v = dpp_add<0x140>(v);         // row_mirror
    v = dpp_add<0x142, 0xA>(v);    // row_bcast:15 into rows 1 and 3
    v = dpp_add<0x143, 0xC>(v);    // row_bcast:31 into rows 2 and 3
    return v;
}

// Adds the first cnt far cells of F (c.o.m. relative to the centre, mass) to
// the group's coefficients row[kLoc]: lane k takes cell k, then the wave sums.
__device__ __forceinline__ void local_flush(const float4 *F, int cnt, float *row, float eps2, float ell)
{
    const int lane = lane_id();
    const float4 e = lane < cnt ? F[lane] : make_float4(1.f, 0.f, 0.f, 0.f);   // massless: no terms
    const float rho2 = fmaf(e.x, e.x, fmaf(e.y, e.y, fmaf(e.z, e.z, eps2)));
    const float ri = rsq(rho2);
    const float nx = e.x * ri, ny = e.y * ri, nz = e.z * ri;
    const float F0 = e.w * ri * ri;
    const float sc = ell * ri;
    const float Fs = F0 * sc, Fs2 = Fs * sc;
    const float e3 = 3.f * Fs, t15 = 15.f * Fs2, f3 = 3.f * Fs2;
    // one coefficient at a time: its wave sum, added by lane 63
    auto put = [&](int k, float v) {
        v = wave_sum63(v);
        if (lane == 63) row[k] += v;
    };
    put(0, e.w * ri);
    put(1, F0 * nx);
    put(2, F0 * ny);
    put(3, F0 * nz);
    put(4, fmaf(e3 * nx, nx, -Fs));
    put(5, e3 * nx * ny);
    put(6, e3 * nx * nz);
    put(7, fmaf(e3 * ny, ny, -Fs));
    put(8, e3 * ny * nz);
    put(9, fmaf(e3 * nz, nz, -Fs));
    put(10, fmaf(t15 * nx, nx * nx, -3.f * f3 * nx));
    put(11, fmaf(t15 * nx, nx * ny, -f3 * ny));
    put(12, fmaf(t15 * nx, nx * nz, -f3 * nz));
    put(13, fmaf(t15 * nx, ny * ny, -f3 * nx));
    put(14, t15 * nx * (ny * nz));
    put(15, fmaf(t15 * nx, nz * nz, -f3 * nx));
    put(16, fmaf(t15 * ny, ny * ny, -3.f * f3 * ny));
    put(17, fmaf(t15 * ny, ny * nz, -f3 * nz));
    put(18, fmaf(t15 * ny, nz * nz, -f3 * ny));
    put(19, fmaf(t15 * nz, nz * nz, -3.f * f3 * nz));
}

// Field and potential sum (+m/r convention of the tiles) of the summed
// coefficients G at the member u = (x - centre)/l.
__device__ __forceinline__ void local_eval(const float *G, float ux, float uy, float uz, float ell, float &ax,
                                           float &ay, float &az, float &ph)
{
    const float gx = fmaf(G[4], ux, fmaf(G[5], uy, G[6] * uz));
    const float gy = fmaf(G[5], ux, fmaf(G[7], uy, G[8] * uz));
    const float gz = fmaf(G[6], ux, fmaf(G[8], uy, G[9] * uz));
    const float xx = ux * ux, yy = uy * uy, zz = uz * uz;
    const float xy2 = 2.f * ux * uy, xz2 = 2.f * ux * uz, yz2 = 2.f * uy * uz;
    const float hx = fmaf(G[10], xx, fmaf(G[11], xy2, fmaf(G[12], xz2, fmaf(G[13], yy, fmaf(G[14], yz2, G[15] * zz)))));
    const float hy = fmaf(G[11], xx, fmaf(G[13], xy2, fmaf(G[14], xz2, fmaf(G[16], yy, fmaf(G[17], yz2, G[18] * zz)))));
    const float hz = fmaf(G[12], xx, fmaf(G[14], xy2, fmaf(G[15], xz2, fmaf(G[17], yy, fmaf(G[18], yz2, G[19] * zz)))));
    ax = fmaf(0.5f, hx, G[1] + gx);
    ay = fmaf(0.5f, hy, G[2] + gy);
    az = fmaf(0.5f, hz, G[3] + gz);
    const float px = fmaf(1.f / 6.f, hx, fmaf(0.5f, gx, G[1]));
    const float py = fmaf(1.f / 6.f, hy, fmaf(0.5f, gy, G[2]));
    const float pz = fmaf(1.f / 6.f, hz, fmaf(0.5f, gz, G[3]));
    ph = fmaf(ell, fmaf(ux, px, fmaf(uy, py, uz * pz)), G[0]);
}

}  // namespace

struct WalkArgs {
    const float4 *thi, *tlo;
    const int *tself, *tinv;
    int selfmode;
    const uint32_t *tperm;
    int64_t ntest;
    const unsigned long long *stat;
    const int *gfirst, *gcount;
    const float4 *bhi, *blo;
    const float4 *cA, *cB, *cQ0, *cQ1;
    const int *sub, *nkids;
    const int2 *fnb;
    int nleaf;
    const uint8_t *level;
    int nb;
    const unsigned long long *ncellp;
    float tolsq, eps2;
    int *frontier;
    int fcap;
    int *gctr;
    unsigned long long *counters;
    double *phi, *acc;
    double4 *sacc;        // lmode 1: (a, phi) per test point in sorted order (the correction pass writes phi, acc)
    // learned correction: record, per group, the accepted cells whose
    // size/distance lies in [lr_lo, lr_hi] (squared bounds) into a per-wave
    // region: [used][g, n, cx, cy, cz, cell ids ...] ...
    int lmode;            // 0 off, 1 every group, 2 every lstride-th group
    int lstride;
    float lr_lo2, lr_hi2;
    int *lrec;
    int lcap;
    // batches: system offsets, per-system (tol^2, eps^2) and walk roots
    int nsys;
    const int64_t *boff;
    const float2 *sysp;
    const int *sysroot;
    // treecode1 criteria: root box; cB.w holds each cell's Rcrit2
    const double4 *box;
    // super-groups: K consecutive groups share one traversal; per-wave
    // scratch for the shared lists (shcap entries each)
    int K;
    float lalpha2;        // local expansions: local_alpha^2 (0 = off)
    float4 *shlist;       // [wave][shcap P entries][shcap * S C entries]
    int *shid;            // [wave][shcap body ids of the P entries][shcap deferred nodes]
    int shcap;
    // teams: rows of 64 points a team holds, and rows of the largest group
    // (group_size / 64); one row per team of a group when rows < grows
    int rows, grows;
};

// bh_team.hip: the walk with a team of W waves (4 or 8) per group, grid blocks.
void walk_team(bh_ctx *ctx, const WalkArgs &a, int W, int grid, bool quad, bool soft0, bool crit);
// Dynamic LDS of a block of that walk (bytes).
size_t walk_team_lds(int W, bool quad, bool local, int rows);

}  // namespace bh
