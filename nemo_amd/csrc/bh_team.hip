// The group walk by a team of waves: one block walks one group.
//
// k_walk (bh_walk.hip) gives a group to one wave.  That fills the device when
// there are several groups for each of its ~4096 resident waves; below that
// the walk's time is one wave's serial walk of its group (N = 10^4, quadrupole
// cells: 120 groups, 0.45 ms; here 0.077 ms).  Here the W waves of a block
// share the group's work:
//   traversal  each step tests 64 W frontier nodes, 64 per wave, and appends
//              bodies, accepted cells and children at offsets from a scan of
//              the waves' counts, so the lists hold what k_walk's lists hold,
//              in the same order;
//   tiles      the full 64-entry tiles of the lists are the same tiles; each
//              is evaluated by one wave for all rows of the group, and the
//              tile sums meet in LDS, where each (row, component) is folded in
//              the order in which k_walk completes the tiles (per 64 nodes:
//              first its body tile, then its cell tile).
// Every sum is therefore k_walk's bit for bit, whatever W is.  With few groups
// (WalkArgs::rows < grows) a team takes one row of a group: the traversal is
// repeated per row, the tiles, which are most of the work, are not.
//
// What bounds it: up to N ~ 2 10^4 the traversal's chain of levels (about 15,
// each an LDS read, one round of cell loads and two barriers, ~3 us), then the
// vector ALU with half the waves' life in barrier waits, which is why k_walk
// keeps the large runs (walkers() in bh_walk.hip has both sides measured).
#include "bh_walk.h"

#include <algorithm>
#include <type_traits>

namespace bh {
namespace {

// Lists of a team of W waves: rings of whole tiles.  A step needs room for 64 W
// entries of each; tiles are evaluated W at a time, so a ring also holds what
// waits for the W-th tile (for cells, whose entries are the larger, not
// always: then fewer than W tiles are evaluated).
template <int W>
struct TeamCap {
    static constexpr int kP = (W == 4 ? 96 : 128) * W;     // bodies
    static constexpr int kC = 96 * W;                      // cells
    static constexpr int kF = 64 * W + 64;                 // far cells (local expansions)
    static constexpr int kFr = (W == 4 ? 96 : 128) * W;    // frontier entries kept in LDS, per level parity
    static constexpr int kEv = 4 * W;                      // tiles waiting, in order (power of two)
    static_assert(kP / 64 + kC / 64 + 2 <= kEv && (kEv & (kEv - 1)) == 0, "pending tiles");
};

// Dynamic LDS of a team (bytes) for groups of `rows` rows of 64 points.
template <int W, bool QUAD, bool LOCAL>
constexpr size_t team_lds(int rows)
{
    using T = TeamCap<W>;
    return sizeof(float4) * (T::kP + T::kC * (QUAD ? 3 : 1) + (LOCAL ? T::kF : 0))   // lists
           + sizeof(float) * 256 * (size_t)(W * rows)                                // tile sums
           + sizeof(float) * 192 * (size_t)rows                                      // positions
           + sizeof(int) * (2 * T::kFr + T::kEv + 8 * W + 4)                         // frontier, tiles, counts
           + sizeof(float) * (LOCAL ? (W + 1) * kLoc : 0)                            // expansion terms
           + 64 * (size_t)rows;                                                      // self flags
}

// min / max over the wave in every lane (order does not matter to either).
template <int CTRL, int RM = 0xF>
__device__ __forceinline__ float dpp_of(float v)
{
    const int i = __float_as_int(v);
    return __int_as_float(__builtin_amdgcn_update_dpp(i, i, CTRL, RM, 0xF, false));
}
__device__ __forceinline__ float lane63(float v) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63)); }
__device__ __forceinline__ float dpp_min(float v)
{
    v = fminf(v, dpp_of<0xB1>(v));
    v = fminf(v, dpp_of<0x4E>(v));
    v = fminf(v, dpp_of<0x141>(v));
    v = fminf(v, dpp_of<0x140>(v));
    v = fminf(v, dpp_of<0x142, 0xA>(v));
    v = fminf(v, dpp_of<0x143, 0xC>(v));
    return lane63(v);
}
__device__ __forceinline__ float dpp_max(float v) { return -dpp_min(-v); }

// Inclusive scan over the wave.
template <int CTRL, int RM = 0xF>
__device__ __forceinline__ int dpp_addi(int v) { return v + __builtin_amdgcn_update_dpp(0, v, CTRL, RM, 0xF, true); }
__device__ __forceinline__ int dpp_incl_scan(int v)
{
    v = dpp_addi<0x111>(v);        // row_shr:1
    v = dpp_addi<0x112>(v);        // row_shr:2
    v = dpp_addi<0x114>(v);        // row_shr:4
    v = dpp_addi<0x118>(v);        // row_shr:8
    v = dpp_addi<0x142, 0xA>(v);   // row_bcast:15 into rows 1 and 3
    v = dpp_addi<0x143, 0xC>(v);   // row_bcast:31 into rows 2 and 3
    return v;
}

// Sums of one pending tile for the nq rows of the group into the slot
// (slot[(4 row + component) * 64 + lane]; components ax ay az phi).
template <int NQ, bool CELLS, bool QUAD, bool SOFT0>
__device__ __forceinline__ void team_tile(const float *pos, const float4 *src, int cnt, float eps2, float *slot)
{
    const int lane = lane_id();
    float px[NQ], py[NQ], pz[NQ], sx[NQ], sy[NQ], sz[NQ], sp[NQ];
#pragma unroll
    for (int q = 0; q < NQ; q++) {
        px[q] = pos[192 * q + lane];
        py[q] = pos[192 * q + 64 + lane];
        pz[q] = pos[192 * q + 128 + lane];
    }
    if (CELLS) tile_p2c<NQ, QUAD, SOFT0>(px, py, pz, src, cnt, eps2, sx, sy, sz, sp);
    else tile_p2p<NQ, SOFT0>(px, py, pz, src, cnt, eps2, sx, sy, sz, sp);
#pragma unroll
    for (int q = 0; q < NQ; q++) {
        slot[256 * q + lane] = sx[q];
        slot[256 * q + 64 + lane] = sy[q];
        slot[256 * q + 128 + lane] = sz[q];
        slot[256 * q + 192 + lane] = sp[q];
    }
}

template <bool CELLS, bool QUAD, bool SOFT0>
__device__ __forceinline__ void team_tile_rows(int nq, const float *pos, const float4 *src, int cnt, float eps2,
                                               float *slot)
{
    if (nq <= 1) team_tile<1, CELLS, QUAD, SOFT0>(pos, src, cnt, eps2, slot);
    else if (nq == 2) team_tile<2, CELLS, QUAD, SOFT0>(pos, src, cnt, eps2, slot);
    else if (nq == 3) team_tile<3, CELLS, QUAD, SOFT0>(pos, src, cnt, eps2, slot);
    else team_tile<4, CELLS, QUAD, SOFT0>(pos, src, cnt, eps2, slot);
}

// Inclusive scan over the first W lanes (4 or 8: within a DPP row).
template <int W>
__device__ __forceinline__ int scan_w(int v)
{
    v = dpp_addi<0x111>(v);
    v = dpp_addi<0x112>(v);
    if (W > 4) v = dpp_addi<0x114>(v);
    return v;
}

extern __shared__ __attribute__((aligned(16))) unsigned char team_mem[];

template <int W, bool QUAD, bool SOFT0, bool LREC, bool CRIT, bool LOCAL>
__global__ __launch_bounds__(64 * W) void k_walk_team(WalkArgs a)
{
    static_assert(!(LOCAL && QUAD), "local expansions take monopole cells");
    static_assert(W == 4 || W == 8, "scan_w and the list sizes");
    using T = TeamCap<W>;
    constexpr int S = QUAD ? 3 : 1;
    constexpr int kTasks = 16 / W;    // (row, component) sums per wave, at most 4 rows
    const int rows = a.rows;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = lane_id();
    float4 *P = reinterpret_cast<float4 *>(team_mem);
    float4 *Cl = P + T::kP;
    float4 *Fl = Cl + S * T::kC;
    float *slots = reinterpret_cast<float *>(Fl + (LOCAL ? T::kF : 0));
    float *pos = slots + 256 * W * rows;
    float *lrow = pos + 192 * rows;                     // LOCAL: the group's coefficients, then W rows of terms
    int *fr = reinterpret_cast<int *>(lrow + (LOCAL ? (W + 1) * kLoc : 0));
    int *ev = fr + 2 * T::kFr;
    int4 *cnt = reinterpret_cast<int4 *>(ev + T::kEv);
    int *next = reinterpret_cast<int *>(cnt + 2 * W);
    unsigned char *self = reinterpret_cast<unsigned char *>(next + 1);
    int *fr0 = a.frontier + (int64_t)blockIdx.x * 2 * a.fcap, *fr1 = fr0 + a.fcap;   // entries past kFr
    int *lf0 = fr, *lf1 = fr + T::kFr;
    int *lreg = a.lrec + (int64_t)blockIdx.x * a.lcap;
    int lused = 1, par = 0;
    const unsigned long long lt = lane ? ~0ULL >> (64 - lane) : 0ULL;
    const int split = rows < a.grows ? a.grows : 1;     // teams per group
    const int nitem = (int)a.stat[S_NGROUPS] * split;

    // The first item by the block's number, the others by tickets, drawn as late
    // in a group as the round trip can still be hidden (a team that holds its
    // next ticket through a long walk leaves work waiting: 2 10^5 bodies 390 us,
    // now 343); the range of the next group is loaded before it is begun.
    int item = blockIdx.x;
    const bool nocell = *a.ncellp == 0, once = nitem <= (int)gridDim.x;
    int gfirst = a.gfirst[item / split], gsize = a.gcount[item / split];
    auto enter = [&](int to) {
        item = to;
        gfirst = a.gfirst[min(to, nitem - 1) / split];
        gsize = a.gcount[min(to, nitem - 1) / split];
    };
    auto advance = [&]() {
        if (threadIdx.x == 0) *next = once ? nitem : (int)gridDim.x + atomicAdd(a.gctr, 1);
        __syncthreads();
        enter(*next);
        __syncthreads();
    };
    while (item < nitem) {
        const int g = item / split, r0 = item % split;  // group, and this team's first row
        const int64_t gbase = gfirst;
        const int gcount = gsize;
        const int nq = (gcount + 63) >> 6;
        const int nr = split > 1 ? 1 : nq;              // this team's rows and points
        const int mine0 = 64 * r0, mcount = min(gcount - mine0, 64 * nr);
        if (mcount <= 0) {
            advance();
            continue;
        }
        float tolsq = a.tolsq, eps2 = a.eps2;
        int sys = -1;
        if (a.nsys) {
            int lo = 0, hi = a.nsys;
            while (hi - lo > 1) {
                const int mid = (lo + hi) >> 1;
                if (a.boff[mid] <= gbase) lo = mid;
                else hi = mid;
            }
            sys = lo;
            const float2 pp = a.sysp[sys];
            tolsq = pp.x;
            eps2 = pp.y;
        }

        // the group's frame (every wave computes it; k_walk's expressions)
        float4 h[4], l[4];
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int k = q * 64 + lane;
            const int64_t i = gbase + (q < nq && k < gcount ? k : 0);
            if (q == 0 || q < nq) {
                h[q] = a.thi[i];
                l[q] = a.tlo[i];
            } else {
                h[q] = h[0];
                l[q] = l[0];
            }
        }
        float mnx = h[0].x, mny = h[0].y, mnz = h[0].z, mxx = mnx, mxy = mny, mxz = mnz;
#pragma unroll
        for (int q = 1; q < 4; q++) {
            mnx = fminf(mnx, h[q].x); mny = fminf(mny, h[q].y); mnz = fminf(mnz, h[q].z);
            mxx = fmaxf(mxx, h[q].x); mxy = fmaxf(mxy, h[q].y); mxz = fmaxf(mxz, h[q].z);
        }
        const float cx = 0.5f * (dpp_min(mnx) + dpp_max(mxx));
        const float cy = 0.5f * (dpp_min(mny) + dpp_max(mxy));
        const float cz = 0.5f * (dpp_min(mnz) + dpp_max(mxz));
        float bminx = 3.0e38f, bminy = 3.0e38f, bminz = 3.0e38f, bmaxx = -3.0e38f, bmaxy = -3.0e38f, bmaxz = -3.0e38f;
        float lrg2 = 0.f, lell = 0.f;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            if (q >= nq) break;
            const float px = (h[q].x - cx) + l[q].x, py = (h[q].y - cy) + l[q].y, pz = (h[q].z - cz) + l[q].z;
            if (q >= r0 && q < r0 + nr && w == (q - r0) % W) {
                float *to = pos + 192 * (q - r0) + lane;
                to[0] = px;
                to[64] = py;
                to[128] = pz;
                self[(q - r0) * 64 + lane] = 0;
            }
            bminx = fminf(bminx, px); bminy = fminf(bminy, py); bminz = fminf(bminz, pz);
            bmaxx = fmaxf(bmaxx, px); bmaxy = fmaxf(bmaxy, py); bmaxz = fmaxf(bmaxz, pz);
            if (LOCAL) lrg2 = fmaxf(lrg2, fmaf(px, px, fmaf(py, py, pz * pz)));
        }
        bminx = dpp_min(bminx); bminy = dpp_min(bminy); bminz = dpp_min(bminz);
        bmaxx = dpp_max(bmaxx); bmaxy = dpp_max(bmaxy); bmaxz = dpp_max(bmaxz);
        if (LOCAL) {
            lrg2 = dpp_max(lrg2);
            lell = sqrtf(lrg2);
            if (threadIdx.x < kLoc) lrow[threadIdx.x] = 0.f;
        }
        int ulo[3] = {0, 0, 0}, uhi[3] = {0, 0, 0};
        float uoff[3] = {0.f, 0.f, 0.f}, uunit = 0.f, urs = 0.f;
        if (CRIT) {
            const double4 bb = *a.box;
            const double org[3] = {bb.x, bb.y, bb.z}, cen[3] = {cx, cy, cz};
            const double sc = 2097152.0 / bb.w;
#pragma unroll
            for (int k = 0; k < 3; k++) {
                int lo = INT32_MAX, hi = INT32_MIN;
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const float hk = k == 0 ? h[q].x : (k == 1 ? h[q].y : h[q].z);
                    const float lk = k == 0 ? l[q].x : (k == 1 ? l[q].y : l[q].z);
                    double f = floor((((double)hk + (double)lk) - org[k]) * sc);
                    f = fmin(fmax(f, -536870912.0), 536870912.0);
                    lo = min(lo, (int)f);
                    hi = max(hi, (int)f);
                }
                ulo[k] = wave_min_i(lo);
                uhi[k] = wave_max_i(hi);
                uoff[k] = (float)((org[k] + (double)ulo[k] * (bb.w / 2097152.0)) - cen[k]);
            }
            uunit = (float)(bb.w / 2097152.0);
            urs = (float)bb.w;
        }

        int np = 0, nc = 0, nfl = 0, nf = 0;            // entries listed so far, frontier
        int wp = 0, wc = 0, wf = 0;                     // the rings' write positions
        int dp = 0, dc = 0, df = 0;                     // tiles evaluated
        int ne = 0, eh = 0;                             // tiles waiting, the first one's place in ev
        const bool lrecord = LREC && r0 == 0 && (a.lmode == 1 || (a.lmode == 2 && g % a.lstride == 0));
        int lhead = 0, lcnt = 0;
        if (lrecord) {
            lhead = lused;
            if (lhead + 5 + 64 > a.lcap) {
                if (threadIdx.x == 0) atomicOr(&a.counters[S_FLAGS], (unsigned long long)F_LREC_OVF);
            } else if (threadIdx.x == 0) {
                lreg[lhead] = g;
                lreg[lhead + 2] = __float_as_int(cx);
                lreg[lhead + 3] = __float_as_int(cy);
                lreg[lhead + 4] = __float_as_int(cz);
            }
        }
        int root = ~0;
        nf = 1;
        if (sys >= 0) {
            root = a.sysroot[sys];
        } else if (nocell) {
            root = 0;
            nf = a.nb == 1 ? 1 : 0;
        }
        if (threadIdx.x == 0) lf0[0] = root;
        float ahi[kTasks], alo[kTasks];                 // this wave's (row, component) sums
#pragma unroll
        for (int t = 0; t < kTasks; t++) ahi[t] = alo[t] = 0.f;
        __syncthreads();

        // Evaluates the first min(W, ne) waiting tiles, one per wave, and folds
        // their sums in order.  Ends with a barrier.
        auto eval_tiles = [&]() {
            const int m = min(W, ne);
            if (w < m) {
                const int e = ev[(eh + w) & (T::kEv - 1)], n = (e >> 1) & 127, at = 64 * (e >> 8);
                float *slot = slots + 256 * rows * w;
                if (e & 1) team_tile_rows<true, QUAD, SOFT0>(nr, pos, Cl + S * at, n, eps2, slot);
                else team_tile_rows<false, QUAD, SOFT0>(nr, pos, P + at, n, eps2, slot);
            }
            const int cells = __popcll(__ballot(lane < m && (ev[(eh + lane) & (T::kEv - 1)] & 1)));
            __syncthreads();
#pragma unroll
            for (int t = 0; t < kTasks; t++) {
                const int k = w + W * t;
                if (k < 4 * nr)
                    for (int e = 0; e < m; e++) fold(ahi[t], alo[t], slots[256 * rows * e + 64 * k + lane]);
            }
            dp += m - cells;
            dc += cells;
            ne -= m;
            eh += m;
            __syncthreads();
        };
        // the expansion terms of the next n far cells (at most 64 W; fewer
        // than 64 only in the last)
        auto eval_far = [&](int n) {
            if constexpr (LOCAL) {
                float *mine = lrow + kLoc * (1 + w);
                const int at = 64 * w;
                if (at < n) {
                    if (lane < kLoc) mine[lane] = 0.f;
                    wave_lds_sync();
                    local_flush(Fl + 64 * ((df + w) % (T::kF / 64)), min(64, n - at), mine, eps2, lell);
                }
                __syncthreads();
                if (threadIdx.x < kLoc)
                    for (int k = 0; k < W && 64 * k < n; k++) lrow[threadIdx.x] += lrow[kLoc * (1 + k) + threadIdx.x];
                df += n >> 6;
                __syncthreads();
            }
        };

        bool overflow = false;
        while (nf > 0 && !overflow) {
            int nn = 0;
            for (int base = 0; base < nf; base += 64 * W) {
                // room for this step's entries?
                const bool full = np - 64 * dp > T::kP - 64 * W || nc - 64 * dc > T::kC - 64 * W;
                if (full || ne >= 2 * W || (LOCAL && nfl - 64 * df > T::kF - 64 * W)) {
                    __syncthreads();
                    while (ne >= W) eval_tiles();
                    if (ne && (np - 64 * dp > T::kP - 64 * W || nc - 64 * dc > T::kC - 64 * W)) eval_tiles();
                    if (LOCAL && nfl - 64 * df >= 64) eval_far(min(64 * W, (nfl - 64 * df) & ~63));
                }
                // (a wave whose 64 nodes lie past the level's end only keeps step)
                const bool busy = base + 64 * w < nf;
                int node = 0, c = 0, nk = 0, off = 0, wk = 0, bfirst = -1;
                bool isBody = false, open = false, accept = false, take = false, far = false;
                float4 A = make_float4(0.f, 0.f, 0.f, 0.f), bl = A, q0 = A, q1 = A;
                float rx = 0.f, ry = 0.f, rz = 0.f, size2 = 0.f;
                int4 s0 = make_int4(kNoChild, kNoChild, kNoChild, kNoChild), s1 = s0;
                unsigned long long mP = 0, mC = 0, mF = 0, mR = 0;
                if (busy) {
                    const int k = base + 64 * w + lane;
                    const bool v = k < nf;
                    node = v ? (k < T::kFr ? lf0[k] : fr0[k - T::kFr]) : 0;
                    isBody = v && node >= 0;
                    const bool isCell = v && node < 0;
                    if (isBody) {
                        A = a.bhi[node];
                        bl = a.blo[node];
                    }
                    if (isCell) {
                        c = ~node;
                        s0 = reinterpret_cast<const int4 *>(a.sub)[2 * (int64_t)c];
                        s1 = reinterpret_cast<const int4 *>(a.sub)[2 * (int64_t)c + 1];
                        A = a.cA[c];
                        const float4 B = a.cB[c];
                        if (QUAD) {      // (with the record: after the decision they are a round trip more per step)
                            q0 = a.cQ0[c];
                            q1 = a.cQ1[c];
                        }
                        const int2 fn = a.fnb[c];
                        const int lv = a.level[c];
                        size2 = B.w;
                        rx = (A.x - cx) + B.x;
                        ry = (A.y - cy) + B.y;
                        rz = (A.z - cz) + B.z;
                        const float dx = fmaxf(fmaxf(bminx - rx, rx - bmaxx), 0.f);
                        const float dy = fmaxf(fmaxf(bminy - ry, ry - bmaxy), 0.f);
                        const float dz = fmaxf(fmaxf(bminz - rz, rz - bmaxz), 0.f);
                        const float d2 = fmaf(dx, dx, fmaf(dy, dy, dz * dz));
                        const bool small = fn.y <= a.nleaf || lv == kMaxLevel;
                        if (CRIT) {
                            const int sh = kMaxLevel - lv, step = 1 << sh;
                            const float side = ldexpf(urs, -lv), rr[3] = {rx, ry, rz};
                            float dd[3];
#pragma unroll
                            for (int k3 = 0; k3 < 3; k3++) {
                                const float flo = (float)((ulo[k3] >> sh) * step - ulo[k3]) * uunit + uoff[k3];
                                const float fhi = (float)(((uhi[k3] >> sh) + 1) * step - ulo[k3]) * uunit + uoff[k3];
                                dd[k3] = fmaxf(fmaxf(flo - rr[k3], rr[k3] - fhi), 0.f);
                            }
                            const float usq = fmaf(dd[0], dd[0], fmaf(dd[1], dd[1], dd[2] * dd[2]));
                            const bool adj_ok = fmaxf(dd[0], fmaxf(dd[1], dd[2])) > side;
                            open = !(usq > B.w && adj_ok) || fn.y <= a.nleaf;
                        } else {
                            open = tolsq * d2 < B.w || fn.y <= a.nleaf;
                        }
                        accept = !open;
                        if (open) {
                            int cc = 0;
                            const int so[8] = {s0.x, s0.y, s0.z, s0.w, s1.x, s1.y, s1.z, s1.w};
#pragma unroll
                            for (int o = 0; o < 8; o++) cc += so[o] != kNoChild;
                            nk = small ? fn.y : cc;
                        }
                        bfirst = small ? fn.x : -1;
                    }
                    if (LREC && lrecord) {
                        const float r2 = fmaf(rx, rx, fmaf(ry, ry, rz * rz));
                        take = accept && size2 >= a.lr_lo2 * r2 && size2 <= a.lr_hi2 * r2;
                    }
                    if (LOCAL) {
                        far = accept && lrg2 < a.lalpha2 * fmaf(rx, rx, fmaf(ry, ry, rz * rz));
                        accept = accept && !far;
                    }
                    mP = __ballot(isBody);
                    mC = __ballot(accept);
                    mF = LOCAL ? __ballot(far) : 0ULL;
                    mR = LREC ? __ballot(take) : 0ULL;
                    const int ki = dpp_incl_scan(nk);
                    off = ki - nk;
                    wk = __builtin_amdgcn_readlane(ki, 63);
                }
                par ^= 1;
                if (lane == 0)
                    cnt[par * W + w] = make_int4(__popcll(mP) | (__popcll(mC) << 16), __popcll(mF) | (__popcll(mR) << 16), wk, 0);
                __syncthreads();
                // every wave scans the W waves' counts (lane i: wave i's)
                const int4 mine = lane < W ? cnt[par * W + lane] : make_int4(0, 0, 0, 0);
                const int pc = scan_w<W>(mine.x), fq = scan_w<W>(mine.y), kk = scan_w<W>(mine.z);
                const int pcx = __builtin_amdgcn_readlane(pc - mine.x, w), kx = __builtin_amdgcn_readlane(kk - mine.z, w);
                const int pct = __builtin_amdgcn_readlane(pc, W - 1), tot = __builtin_amdgcn_readlane(kk, W - 1);
                const int fqx = LOCAL || LREC ? __builtin_amdgcn_readlane(fq - mine.y, w) : 0;
                const int fqt = LOCAL || LREC ? __builtin_amdgcn_readlane(fq, W - 1) : 0;
                if (nn + tot > T::kFr + a.fcap) {
                    overflow = true;
                    break;
                }
                if (w == 0) {
                    // tiles that the chunk of wave i (lane i) completes
                    const int pi = np + (pc & 0xffff), ci = nc + (pc >> 16);
                    const int pb = pi - (mine.x & 0xffff), cb = ci - (mine.x >> 16);
                    const int pt = (pb >> 6) % (T::kP / 64), ct = (cb >> 6) % (T::kC / 64);
                    const bool tp = lane < W && (pi >> 6) > (pb >> 6), tc = lane < W && (ci >> 6) > (cb >> 6);
                    const unsigned long long bp = __ballot(tp), bc = __ballot(tc);
                    const int at = eh + ne + __popcll(bp & lt) + __popcll(bc & lt);
                    if (tp) ev[at & (T::kEv - 1)] = (64 << 1) | (pt << 8);
                    if (tc) ev[(at + (tp ? 1 : 0)) & (T::kEv - 1)] = 1 | (64 << 1) | (ct << 8);
                }
                ne += ((np + (pct & 0xffff)) >> 6) - (np >> 6) + ((nc + (pct >> 16)) >> 6) - (nc >> 6);
                if (isBody) {
                    int at = wp + (pcx & 0xffff) + mbcnt(mP);
                    at -= at >= T::kP ? T::kP : 0;
                    P[at] =
                        make_float4((A.x - cx) + bl.x, (A.y - cy) + bl.y, (A.z - cz) + bl.z, A.w);
                    const int64_t rel = a.selfmode == 1   ? (int64_t)node - gbase - mine0
                                        : a.selfmode == 2 ? (int64_t)a.tinv[node] - gbase - mine0
                                                          : -1;
                    if (rel >= 0 && rel < mcount) self[rel] = 1;
                }
                np += pct & 0xffff;
                wp += pct & 0xffff;
                wp -= wp >= T::kP ? T::kP : 0;
                if (accept) {
                    int slot = wc + (pcx >> 16) + mbcnt(mC);
                    slot -= slot >= T::kC ? T::kC : 0;
                    Cl[S * slot] = make_float4(rx, ry, rz, A.w);
                    if (QUAD) {
                        Cl[S * slot + 1] = q0;
                        Cl[S * slot + 2] = q1;
                    }
                }
                nc += pct >> 16;
                wc += pct >> 16;
                wc -= wc >= T::kC ? T::kC : 0;
                if (LOCAL) {
                    int at = wf + (fqx & 0xffff) + mbcnt(mF);
                    at -= at >= T::kF ? T::kF : 0;
                    if (far) Fl[at] = make_float4(rx, ry, rz, A.w);
                    nfl += fqt & 0xffff;
                    wf += fqt & 0xffff;
                    wf -= wf >= T::kF ? T::kF : 0;
                }
                if (LREC && lrecord) {
                    const int at = lhead + 5 + lcnt;
                    if (at + 64 * W <= a.lcap) {
                        if (take) lreg[at + (fqx >> 16) + mbcnt(mR)] = c;
                        lcnt += fqt >> 16;
                    } else if (fqt >> 16 && threadIdx.x == 0) {
                        atomicOr(&a.counters[S_FLAGS], (unsigned long long)F_LREC_OVF);
                    }
                }
                if (open) {
                    const int at = nn + kx + off;
                    auto put = [&](int j, int r) {
                        if (at + j < T::kFr) lf1[at + j] = r;
                        else fr1[at + j - T::kFr] = r;
                    };
                    if (bfirst >= 0) {
                        for (int j = 0; j < nk; j++) put(j, bfirst + j);
                    } else {
                        const int so[8] = {s0.x, s0.y, s0.z, s0.w, s1.x, s1.y, s1.z, s1.w};
                        int j = 0;
#pragma unroll
                        for (int o = 0; o < 8; o++)
                            if (so[o] != kNoChild) put(j++, so[o]);
                    }
                }
                nn += tot;
            }
            int *tmp = fr0;
            fr0 = fr1;
            fr1 = tmp;
            tmp = lf0;
            lf0 = lf1;
            lf1 = tmp;
            nf = nn;
            __syncthreads();
        }
        if (overflow) {
            if (threadIdx.x == 0) atomicOr(&a.counters[S_FLAGS], (unsigned long long)F_FRONTIER);
            __syncthreads();
            advance();
            continue;
        }
        // the last full tiles, then the two partial ones (bodies first)
        // and the next ticket
        int ticket = 0;
        if (threadIdx.x == 0) {
            if (!once) ticket = (int)gridDim.x + atomicAdd(a.gctr, 1);
            int at = eh + ne;
            if (np & 63) ev[at++ & (T::kEv - 1)] = ((np & 63) << 1) | (((np >> 6) % (T::kP / 64)) << 8);
            if (nc & 63) ev[at & (T::kEv - 1)] = 1 | ((nc & 63) << 1) | (((nc >> 6) % (T::kC / 64)) << 8);
        }
        ne += ((np & 63) != 0) + ((nc & 63) != 0);
        __syncthreads();
        if (!once) {
            if (ne > 0) eval_tiles();
            if (threadIdx.x == 0) *next = ticket;
            __syncthreads();
            enter(*next);
        }
        while (ne > 0) eval_tiles();
        if (LOCAL && nfl > 0) {
            for (int rest = nfl - 64 * df; rest > 0; rest -= 64 * W) eval_far(min(64 * W, rest));
            float Gs[kLoc];
#pragma unroll
            for (int k = 0; k < kLoc; k++) Gs[k] = lrow[k];
            const float linv = lell > 0.f ? 1.f / lell : 0.f;
#pragma unroll
            for (int t = 0; t < kTasks; t++) {
                const int k = w + W * t, q = k >> 2;
                if (k < 4 * nr) {
                    float e[4];
                    local_eval(Gs, pos[192 * q + lane] * linv, pos[192 * q + 64 + lane] * linv,
                               pos[192 * q + 128 + lane] * linv, lell, e[0], e[1], e[2], e[3]);
                    fold(ahi[t], alo[t], (k & 3) == 0 ? e[0] : (k & 3) == 1 ? e[1] : (k & 3) == 2 ? e[2] : e[3]);
                }
            }
        }
        if (lrecord && lhead + 5 + 64 <= a.lcap) {
            lused = lhead + 5 + lcnt;
            if (threadIdx.x == 0) {
                lreg[lhead + 1] = lcnt;
                lreg[0] = lused;
            }
        }
        int nself = 0;
#pragma unroll
        for (int t = 0; t < kTasks; t++) {
            const int k = w + W * t, q = k >> 2, comp = k & 3, i = q * 64 + lane;
            if (k >= 4 * nr || i >= mcount) continue;
            const int64_t tp = gbase + mine0 + i;       // the point, in sorted order
            double r = (double)ahi[t] + (double)alo[t];
            if (comp == 3) {
                if (self[i]) {
                    nself++;
                    if (eps2 > 0.f) {
                        const int64_t tb = a.selfmode == 1 ? tp : a.tself[tp];
                        r -= (double)(a.bhi[tb].w * rsq(eps2));
                    }
                }
                r = -r;
            }
            if (LREC && a.lmode == 1) {
                reinterpret_cast<double *>(a.sacc + tp)[comp] = r;
            } else {
                const int64_t o = a.tperm[tp];
                if (comp == 3) a.phi[o] = r;
                else a.acc[3 * o + comp] = r;
            }
        }
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) nself += __shfl_xor(nself, d, 64);
        if (lane == 0) {
            const long long pp = w == 0 ? (long long)np * mcount - nself : -(long long)nself;
            if (pp) atomicAdd(&a.counters[0], (unsigned long long)pp);
            if (w == 0) {
                atomicAdd(&a.counters[1], (unsigned long long)((long long)(nc + nfl) * mcount));
                if (LOCAL) atomicAdd(&a.counters[S_NLOC], (unsigned long long)((long long)nfl * mcount));
            }
        }
        if (once) break;
        __syncthreads();   // the lists, positions and self flags are reused
    }
}

template <int W, bool QUAD, bool SOFT0, bool LREC, bool CRIT, bool LOCAL>
void launch_team(bh_ctx *ctx, const WalkArgs &a, int grid)
{
    k_walk_team<W, QUAD, SOFT0, LREC, CRIT, LOCAL>
        <<<grid, 64 * W, team_lds<W, QUAD, LOCAL>(a.rows), ctx->stream>>>(a);
}

template <int W, bool QUAD, bool SOFT0>
void launch_team_for(bh_ctx *ctx, const WalkArgs &a, int grid, bool crit)
{
    if (!QUAD && a.lalpha2 > 0.f) {
        if (a.lmode) launch_team<W, false, SOFT0, true, false, true>(ctx, a, grid);
        else if (crit) launch_team<W, false, SOFT0, false, true, true>(ctx, a, grid);
        else launch_team<W, false, SOFT0, false, false, true>(ctx, a, grid);
    } else if (crit) launch_team<W, QUAD, SOFT0, false, true, false>(ctx, a, grid);
    else if (a.lmode) launch_team<W, QUAD, SOFT0, true, false, false>(ctx, a, grid);
    else launch_team<W, QUAD, SOFT0, false, false, false>(ctx, a, grid);
}

template <int W>
void launch_team_w(bh_ctx *ctx, const WalkArgs &a, int grid, bool quad, bool soft0, bool crit)
{
    if (quad) soft0 ? launch_team_for<W, true, true>(ctx, a, grid, crit) : launch_team_for<W, true, false>(ctx, a, grid, crit);
    else soft0 ? launch_team_for<W, false, true>(ctx, a, grid, crit) : launch_team_for<W, false, false>(ctx, a, grid, crit);
}

}  // namespace

size_t walk_team_lds(int W, bool quad, bool local, int rows)
{
    auto of = [&](auto w) -> size_t {
        constexpr int V = decltype(w)::value;
        return quad ? team_lds<V, true, false>(rows) : local ? team_lds<V, false, true>(rows) : team_lds<V, false, false>(rows);
    };
    if (W == 8) return of(std::integral_constant<int, 8>());
    return of(std::integral_constant<int, 4>());
}

void walk_team(bh_ctx *ctx, const WalkArgs &a, int W, int grid, bool quad, bool soft0, bool crit)
{
    if (W == 8) launch_team_w<8>(ctx, a, grid, quad, soft0, crit);
    else launch_team_w<4>(ctx, a, grid, quad, soft0, crit);
    BH_HIP(hipGetLastError());
}

}  // namespace bh
