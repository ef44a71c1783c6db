// vx3mi_tile.h -- the tiled persistent timestep for batches of small robots.
//
// Robots are bin-packed (longest processing time first, by link count) into
// tiles of at most LMAX links and VMAX voxels; one workgroup of NT threads owns
// a tile for a whole launch of many steps.  Each thread owns up to KL links and
// KV voxels and keeps their state in registers across steps; the only data
// exchanged between threads are the voxel poses (position field, quaternion,
// temperature) and the link-end forces, both in LDS as structure of arrays.
// Global memory is read at the start of a launch and written at its end.
// The per-link and per-voxel arithmetic is the same as k_links / k_voxels
// (link_forces / voxel_step, link ends summed in direction order), so every
// launch mode produces the same bits.
#pragma once

#include <hip/hip_runtime.h>

namespace vx3mi {

// Tile configurations: NT threads, up to KL links and KV voxels per thread,
// MINW the minimum waves per SIMD the register budget must allow (the second
// __launch_bounds__ argument).  The large tile
// uses ~158 KB of LDS (one workgroup per compute unit); the FP32 one runs 768
// threads, 12 waves, so each SIMD holds three waves of at most 168 VGPRs (the
// kernel is VALU-issue bound, and a third wave hides the LDS and barrier
// waits: +33 % over 512 threads holding four links each at two waves).  The
// small tile stays within 78 KB of LDS, so two workgroups fit a compute unit's
// 160 KB (one computes while the other waits at a barrier), 384 threads each,
// again three waves per SIMD.  The batch's autotuner picks one.
template <typename T, int SMALL> struct TileCfg;
template <> struct TileCfg<float, 0> {
    static constexpr int NT = 768, KL = 3, KV = 2, LMAX = 2048, VMAX = 1536, RMAX = 128, MINW = 1;
};
template <> struct TileCfg<float, 1> {
    static constexpr int NT = 384, KL = 3, KV = 2, LMAX = 960, VMAX = 768, RMAX = 64, MINW = 3;
};
template <> struct TileCfg<double, 0> {
    static constexpr int NT = 512, KL = 2, KV = 2, LMAX = 1024, VMAX = 768, RMAX = 64, MINW = 2;
};
template <> struct TileCfg<double, 1> {
    static constexpr int NT = 256, KL = 2, KV = 2, LMAX = 512, VMAX = 384, RMAX = 32, MINW = 2;
};

// Collision tiles (large configuration): the partner momenta of the contact
// phase sit in LDS beside the poses, so the capacities are smaller (every
// robot of the batched workload still fits: at most 1,861 links, 1,077 voxels).
// The FP32 tile holds fewer robots (64) to keep 1,984 links and 1,280 voxels:
// the batched workload then packs into 256 tiles, one per compute unit, where
// 1,920 links made 259 and three compute units ran a second tile after the
// first (the launch took twice as long).
template <typename T> struct TileColCfg;
template <> struct TileColCfg<float> {
    static constexpr int NT = 768, KL = 3, KV = 2, LMAX = 1984, VMAX = 1280, RMAX = 64, MINW = 1;
};
template <> struct TileColCfg<double> {
    static constexpr int NT = 512, KL = 2, KV = 2, LMAX = 896, VMAX = 640, RMAX = 64, MINW = 2;
};
// the thinner list skin goes to the robots the FP32 collision tile can hold
static_assert(kSmallRobotVoxels == TileColCfg<float>::VMAX, "small-robot skin threshold");
template <typename T, int SMALL, int COL> struct TileSel { using C = TileCfg<T, SMALL>; };
template <typename T, int SMALL> struct TileSel<T, SMALL, 1> { using C = TileColCfg<T>; };

// LDS robot table of a tile
template <int RMAX, int COL> struct TileRobots {
    int rid[RMAX];
    int voffG[RMAX], loffG[RMAX];
    int vpre[RMAX + 1], lpre[RMAX + 1];
    double time[2][RMAX];
    float prevDt[2][RMAX];
    float dt[RMAX];
    int diverged[RMAX];
    int steps[RMAX];
    double tempAmp[RMAX], tempPeriod[RMAX];  // actuation of each robot (FP32: 1 / period)
    int tempFlags[RMAX];                     // varyTemp | enableExpansion << 1
    int col[RMAX];                           // the robot has collisions (surface voxels in the lists)
    // collision tiles: the robot lists its candidates at the start of the next
    // step (set by the tracking of the voxel phase), its stale distance, a link
    // of this step passed the divergence strain (merged into diverged once the
    // contact and link phases that read diverged are done), and per step parity
    // whether some robot of the tile is stale
    int stale[COL ? RMAX : 1];
    float staleD2[COL ? RMAX : 1];
    int divNow[RMAX];
    int anyStale[2];
};

// material tables of at most this many entries (large / small tile) are
// copied into LDS at launch; the small tile keeps within half the LDS
template <int SMALL> struct TileMatCache { static constexpr int N = SMALL ? 12 : 24; };

// largest j with pre[j] <= x (pre ascending, pre[0] = 0, pre[n] = total)
__device__ __forceinline__ int tile_slot(const int *pre, int n, int x) {
    int lo = 0, hi = n - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (pre[mid] <= x) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

// LDSMAT: the batch has at most kTileMatCache voxel and link materials, which
// are read from LDS in the step loop instead of global memory
// COL: collision tiles.  Each step, robots whose candidate lists are stale list
// them first: sixteen lanes to a voxel test its robot's pairs outright, from the
// poses in LDS, and write its list and the packed words the tile reads.  After the
// links the lanes of a wave test their voxels' candidates, and what may be in
// contact is dealt out over the wave for the exact test and the force, from the
// poses and momenta entering the step (LDS), summed in list order as in
// k_col_contact.  The stale flags stay in LDS during a launch.
template <typename T, int SMALL, int LDSMAT, int COL>
__global__ __launch_bounds__((TileSel<T, SMALL, COL>::C::NT), (TileSel<T, SMALL, COL>::C::MINW)) void k_tile(
    Dev<T> a, const int4 *tiles, const int *tileRobots, int nsteps, int parity0, int nLinkMats, int nVoxMats) {
    using C = typename TileSel<T, SMALL, COL>::C;
    constexpr int NT = C::NT, KL = C::KL, KV = C::KV;
    constexpr int LMAX = C::LMAX, VMAX = C::VMAX, RMAX = C::RMAX;
    static_assert(KL * NT >= LMAX && KV * NT >= VMAX && RMAX <= NT && NT <= 3 * LMAX,
                  "a tile's threads must cover its capacity");
    static_assert(RMAX <= 128 && VMAX <= 2048, "robot slots take 7 bits, packed candidates 11");
    __shared__ T sPose[8][VMAX];    // position field xyz, qw, qx, qy, qz, temperature
    __shared__ T sForce[12][LMAX];  // forceNeg, momentNeg, forcePos, momentPos (in the link frame)
    __shared__ T sMom[COL ? 3 : 1][COL ? VMAX : 1];  // linear momentum entering the step (contacts)
    __shared__ TileRobots<RMAX, COL> tr;
    __shared__ LinkMat sLM[LDSMAT ? TileMatCache<SMALL>::N : 1];
    __shared__ VoxelMat sVM[LDSMAT ? TileMatCache<SMALL>::N : 1];
    __shared__ unsigned char sOwner[COL && LDSMAT ? NT : 1];  // contact_wave: the lane whose candidate a lane takes
    __shared__ float2 sEnv[COL && LDSMAT ? TileMatCache<SMALL>::N : 1];  // a material's size at temperature 0, and per degree

    int tid = threadIdx.x;
    // threads take links from the front and voxels from the back: the waves left
    // without a link in the last round are those with a voxel more, and in a tile
    // of few links the contact sums run in other waves than the links (they need
    // no barrier between them).  An FP64 tile without collisions has neither, and
    // steps 2 % faster with both from the front.
    int vt = COL || sizeof(T) == 4 ? NT - 1 - tid : tid;
    const int4 info = tiles[blockIdx.x];  // robot begin, robot count, voxels, links
    const int nr = info.y, nv = info.z, nl = info.w;

    if (tid < nr) {
        const int r = tileRobots[info.x + tid];
        const RobotParams &p = a.rp[r];
        const RobotTime &t = a.rt[r];
        tr.rid[tid] = r;
        tr.voffG[tid] = p.voff;
        tr.loffG[tid] = p.loff;
        tr.vpre[tid + 1] = p.vcount;
        tr.lpre[tid + 1] = p.lcount;
        tr.time[0][tid] = t.time[0];
        tr.time[1][tid] = t.time[1];
        tr.prevDt[0][tid] = t.prevDt[0];
        tr.prevDt[1][tid] = t.prevDt[1];
        tr.dt[tid] = t.dt;
        tr.diverged[tid] = (t.diverged | t.divergedNow) ? 2 : 0;  // (1: in this launch)
        tr.steps[tid] = t.steps;
        tr.tempAmp[tid] = p.tempAmp;
        tr.tempPeriod[tid] = std::is_same<T, float>::value ? p.tempInvPeriod : p.tempPeriod;
        tr.tempFlags[tid] = (p.varyTemp ? 1 : 0) | (p.enableExpansion ? 2 : 0);
        tr.col[tid] = COL && p.collisions && p.scount > 0;
        if constexpr (COL) {
            tr.stale[tid] = tr.col[tid] && t.stale[parity0 & 1];
            tr.staleD2[tid] = p.staleD2;
        }
        tr.divNow[tid] = 0;
    }
    if (LDSMAT) {
        for (int i = tid; i < nLinkMats; i += NT) sLM[i] = a.lmats[i];
        for (int i = tid; i < nVoxMats; i += NT) {
            sVM[i] = a.vmats[i];
            if (COL) sEnv[i] = float2{(float)a.vmats[i].nomSize, (float)a.vmats[i].nomSize * a.vmats[i].alphaCTE};
        }
    }
    __syncthreads();
    if (tid == 0) {
        tr.vpre[0] = 0;
        tr.lpre[0] = 0;
        int any = 0;
#pragma unroll 1  // (code every launch has to fetch: unrolled, 2 us of a call of ten steps)
        for (int j = 0; j < nr; j++) {
            tr.vpre[j + 1] += tr.vpre[j];
            tr.lpre[j + 1] += tr.lpre[j];
            if constexpr (COL) any |= tr.stale[j] && !tr.diverged[j];
        }
        tr.anyStale[parity0 & 1] = any;
        tr.anyStale[(parity0 & 1) ^ 1] = 0;
    }
    __syncthreads();

    // ---- owned links: static description and state in registers
    int lEnds[KL], lInfo[KL];  // neg | pos << 16 (tile indices); axis | robot slot << 2 | material << 9
    LinkState<T> ls[KL];
    // the strain is an output only: collision tiles, short of registers, store it
    // in a launch's last step
    float lStrain[COL ? 1 : KL];
#pragma unroll
    for (int k = 0; k < KL; k++) {
        const int ll = tid + k * NT;
        if (ll < nl) {
            const int j = tile_slot(tr.lpre, nr, ll);
            const int gl = tr.loffG[j] + (ll - tr.lpre[j]);
            const int2 e = a.lends[gl];
            const int base = tr.vpre[j] - tr.voffG[j];
            lEnds[k] = (e.x + base) | ((e.y + base) << 16);
            lInfo[k] = (a.lmeta[gl].x & 3) | (j << 2) | ((a.lmeta[gl].x >> 2) << 9);
            const T4<T> s0 = a.ls0[gl], s1 = a.ls1[gl], s2 = a.ls2[gl];
            ls[k].pos2 = {s0.x, s0.y, s0.z};
            ls[k].a1v = {s0.w, s1.x, s1.y};
            ls[k].a2v = {s1.z, s1.w, s2.x};
            ls[k].maxStrain = (float)s2.y;
            ls[k].flags = (int)s2.z;
            if constexpr (!COL) lStrain[k] = (float)s2.w;
        }
    }
    // ---- owned voxels
    int vInfo[KV], vLat[KV];  // robot slot | material << 7; lattice position
    int vLinks[KV][3];  // local link ids, two 16-bit fields each (0xffff = none)
    // the rest of a voxel's state in registers.  Collision tiles keep only its
    // angular momentum and flags there: pose and momentum are in LDS anyway, phase
    // and position at the last listing are read from memory each step, ahead of
    // their use -- the contact phase needs the registers (with all of it held, 69
    // were spilled, and the scratch of an XCD's 32 workgroups outgrew its L2)
    constexpr bool KEEP = !COL;
    VoxelState<T> vs[KEEP ? KV : 1];
    T vPhase[KEEP ? KV : 1];
    V3<T> vH[KEEP ? 1 : KV];
    int vFlags[KEEP ? 1 : KV];
    // collision tiles: the voxel's candidates (kNoCand: none, not a surface voxel
    // of a robot with collisions; kWideCand: read the candidate list itself; else
    // the number of packed entries)
    constexpr int kNoCand = -2, kWideCand = -1;
    int vCand[KV];
#pragma unroll
    for (int k = 0; k < KV; k++) {
        const int lv = vt + k * NT;
        vCand[k] = kNoCand;
        if (lv < nv) {
            const int j = tile_slot(tr.vpre, nr, lv);
            const int gv = tr.voffG[j] + (lv - tr.vpre[j]);
            vInfo[k] = j | (a.vmat[gv] << 7);
            vLat[k] = a.lat[gv];
            const int lbase = tr.lpre[j] - tr.loffG[j];
#pragma unroll
            for (int d = 0; d < 3; d++) {
                const int l0 = a.vlinks[6 * gv + 2 * d], l1 = a.vlinks[6 * gv + 2 * d + 1];
                vLinks[k][d] = (l0 < 0 ? 0xffff : l0 + lbase) | ((l1 < 0 ? 0xffff : l1 + lbase) << 16);
            }
            const T4<T> q0 = a.pq0[gv], q1 = a.pq1[gv], m0 = a.mo0[gv], m1 = a.mo1[gv];
            if constexpr (KEEP) {
                vPhase[k] = a.phase[gv];
                vs[k].u = {q0.x, q0.y, q0.z};
                vs[k].q = {q0.w, q1.x, q1.y, q1.z};
                vs[k].p = {m0.x, m0.y, m0.z};
                vs[k].h = {m0.w, m1.x, m1.y};
                vs[k].flags = (int)m1.z;
            } else {
                vH[k] = {m0.w, m1.x, m1.y};
                vFlags[k] = (int)m1.z;
            }
            sPose[0][lv] = q0.x; sPose[1][lv] = q0.y; sPose[2][lv] = q0.z; sPose[3][lv] = q0.w;
            sPose[4][lv] = q1.x; sPose[5][lv] = q1.y; sPose[6][lv] = q1.z; sPose[7][lv] = q1.w;
            if constexpr (COL) { sMom[0][lv] = m0.x; sMom[1][lv] = m0.y; sMom[2][lv] = m0.z; }
        }
    }
    __syncthreads();

    // owned voxel k: its robot's slot, its material, its global id
    auto vSlot = [&](int k) { return vInfo[k] & 127; };
    auto vMat = [&](int k) { return vInfo[k] >> 7; };
    auto vGlob = [&](int k) {
        const int j = vInfo[k] & 127;
        return tr.voffG[j] + (vt + k * NT - tr.vpre[j]);
    };
    // packed candidates of the tile's voxels: one word per candidate holding the
    // partner's tile index (11 bits), its material (5 bits; the materials are in
    // LDS) and its lattice offset from the voxel (5 signed bits per axis); four
    // candidates of a voxel per int4, laid out by (rank / 4, owned voxel slot k,
    // thread), so the threads of a wave read consecutive int4s, and a tile's
    // entries stay in its XCD's L2
    int4 *const tc4 = reinterpret_cast<int4 *>(a.tcand);
    const size_t cbase = COL ? (size_t)blockIdx.x * (kMaxCand / 4) * KV * NT : 0;
    auto cand4_at = [&](int c4, int k) -> size_t { return cbase + ((size_t)c4 * KV + k) * NT + tid; };
    // owned voxel k's packed entries from its candidate list (at the start of a
    // launch and after each listing)
    auto pack = [&](int k) {
        vCand[k] = kNoCand;
        if (vt + k * NT >= nv || !tr.col[vSlot(k)]) return;
        const int gv = vGlob(k);
        const int s = a.vsurf[gv];
        if (s < 0) return;
        vCand[k] = kWideCand;
        const int n = a.ccount[s];
        if (!LDSMAT || n > kMaxCand) return;
        const int *list = a.clist + (long)s * kMaxCand;
        const int lbase = tr.vpre[vSlot(k)] - tr.voffG[vSlot(k)];
        int4 q = {0, 0, 0, 0};
        for (int c = 0; c < n; c++) {
            const int w = list[c];
            const int3 o = lat_offset(vLat[k], a.lat[w]);
            if (o.x < -16 || o.x > 15 || o.y < -16 || o.y > 15 || o.z < -16 || o.z > 15) return;
            const int e = (w + lbase) | (a.vmat[w] << 11) | ((o.x & 31) << 16) | ((o.y & 31) << 21) | ((o.z & 31) << 26);
            if ((c & 3) == 0) q.x = e;
            else if ((c & 3) == 1) q.y = e;
            else if ((c & 3) == 2) q.z = e;
            else q.w = e;
            if ((c & 3) == 3 || c == n - 1) {
                tc4[cand4_at(c >> 2, k)] = q;
                q = int4{0, 0, 0, 0};
            }
        }
        vCand[k] = n;
    };
    // the force on voxel li (tile index, material mi) of the robot in slot j from
    // its candidate lw at lattice offset o (material mj) when the two are in
    // contact now: col_contact's partner test and force with the poses and momenta
    // of the tile (the robots of a tile lose neither links nor voxels, and have no
    // signals)
    auto partner = [&](int j, int li, const VoxelMat &mi, int lw, int3 o, const VoxelMat &mj, V3<T> &fw) -> bool {
        // everything it takes from LDS is read at once (a read behind each test
        // that returns early would wait by itself)
        T4<T> qi0 = {sPose[0][li], sPose[1][li], sPose[2][li], sPose[7][li]};
        T4<T> qj0 = {sPose[0][lw], sPose[1][lw], sPose[2][lw], sPose[7][lw]};
        V3<T> pi = {sMom[0][li], sMom[1][li], sMom[2][li]}, pj = {sMom[0][lw], sMom[1][lw], sMom[2][lw]};
        const float mInvI = mi.massInv, pkI = mi.penKinv, cdI = mi.cDampT;
        float mInvJ = mj.massInv, pkJ = mj.penKinv, cdJ = mj.cDampT, alphaJ = mj.alphaCTE;
        double sizeJ = mj.nomSize;
        pin(qi0);
        pin(qj0);
        pin(pi.x);
        pin(pi.y);
        pin(pi.z);
        pin(pj.x);
        pin(pj.y);
        pin(pj.z);
        pin(mInvJ);
        pin(pkJ);
        pin(cdJ);
        pin(alphaJ);
        pin(sizeJ);
        if (mi.fixed && mj.fixed) return false;
        T bsaI = base_size_average<T>(mi.nomSize, (float)qi0.w, mi.alphaCTE);
        pin(bsaI);  // rounded by itself, as where one size serves a voxel's whole list
        const V3<T> diff = col_diff<T>(qi0, qj0, o, (T)mi.nomSize);
        const T bsaJ = base_size_average<T>(sizeJ, (float)qj0.w, alphaJ);
        if (!in_contact_envelope(diff, bsaI, bsaJ)) return false;
        if (a.vtarget || a.pairRec) {
            const int lbase = tr.vpre[j] - tr.voffG[j], v = li - lbase, w = lw - lbase;
            if (a.vtarget && a.vtarget[w] != a.vtarget[v] && v < w) atomicAdd(&a.rt[tr.rid[j]].collisionCount, 1);
            if (a.pairRec && v < w) {
                const int q = atomicAdd(a.pairN, 1);
                if (q < a.pairCap) a.pairRec[q] = int2{v, w};
            }
        }
        const V3<T> velI = pi * (T)mInvI, velJ = pj * (T)mInvJ;
        fw = contact_force(diff, bsaI, bsaJ, velI, velJ, pkI, pkJ, cdI, cdJ);
        return true;
    };
    // the contact force on owned voxel k when its candidates are not packed: the
    // list in memory, or the grid
    auto contact_wide = [&](int k, int lv, int parity) -> V3<T> {
        V3<T> f = {0, 0, 0};
        const int j = vSlot(k), gv = vGlob(k);
        const int lbase = tr.vpre[j] - tr.voffG[j];  // tile index of a voxel of the robot = global id + lbase
        const VoxelMat &mi = LDSMAT ? sVM[vMat(k)] : a.vmats[vMat(k)];
        // a partner by voxel id; links: test the current links first
        auto partner_id = [&](int w, bool links) {
            const int3 o = lat_offset(vLat[k], a.lat[w]);
            if (links && col_linked(a, gv, o.x, o.y, o.z)) return;
            V3<T> fw;
            if (partner(j, lv, mi, w + lbase, o, LDSMAT ? sVM[a.vmat[w]] : a.vmats[a.vmat[w]], fw)) f = f + fw;
        };
        const int s = a.vsurf[gv];
        const int nc = a.ccount[s];
        const bool wide = nc > kMaxCand;  // the grid of this step, ascending
        const int *list = a.clist + (long)s * kMaxCand;
        if (wide) {
            tr.stale[j] = 1;  // rebuilt every step while this lasts
            tr.anyStale[parity ^ 1] = 1;
        }
        const RobotParams &rp = a.rp[tr.rid[j]];
        int prev = -1;
        for (int c = 0; wide || c < nc; c++) {
            int next = INT_MAX;
            if (wide) {
                col_grid_each<false>(a, rp, s, -1, [&](int w, const T4<T> &) {
                    if (w > prev && w < next && w != gv) next = w;
                });
                if (next == INT_MAX) break;
            } else {
                next = list[c];
            }
            partner_id(next, wide);
            prev = next;
        }
        return f;
    };
    // the contact forces on the voxels k of a wave's threads, n packed candidates
    // each (0: none; every lane of the wave calls it).  Twelve candidates at a
    // time in three registers of four.  A first pass over them keeps those that
    // may be in contact (no square root and no branch, so the LDS reads of
    // all of them are in flight together).  What is kept, about one for every
    // second voxel, goes through the exact test and the force: the wave's kept
    // candidates are dealt out over its lanes, so that this long part runs once for
    // up to 64 of them instead of once for each candidate of the busiest voxel,
    // and the forces are taken back and added in candidate order.  1024 robots of
    // 4..12 voxels per axis (311,088 voxels), a step with the listing: 44 us with a
    // loop over the kept candidates in each lane, 32 like this, 20 with the
    // registers above no longer spilled (56 before any of it, one round of tiles).
    auto contact_wave = [&](int k, int n) -> V3<T> {
        V3<T> f = {0, 0, 0};
        const int lv = n > 0 ? vt + k * NT : 0, info = n > 0 ? vInfo[k] : 0;
        const VoxelMat &mi = sVM[n > 0 ? vMat(k) : 0];
        const T qx = sPose[0][lv], qy = sPose[1][lv], qz = sPose[2][lv];
        const float Lf = (float)mi.nomSize;
        const float bi = Lf + (float)sPose[7][lv] * (Lf * mi.alphaCTE);
        auto near = [&](int e) -> unsigned {
            const unsigned u = (unsigned)e;
            const int lw = e & 2047, m = (e >> 11) & 31;
            const float2 env = sEnv[m];
            const float w = 0.6250125f * (bi + env.x + (float)sPose[7][lw] * env.y);  // the envelope radius, rounded up by 2e-5
            float dx = (float)(qx - sPose[0][lw]), dy = (float)(qy - sPose[1][lw]), dz = (float)(qz - sPose[2][lw]);
            if constexpr (!kAbsolutePositions<T>) {
                dx -= (float)((int)(u << 11) >> 27) * Lf;
                dy -= (float)((int)(u << 6) >> 27) * Lf;
                dz -= (float)((int)(u << 1) >> 27) * Lf;
            }
            return dx * dx + dy * dy + dz * dz < w * w;
        };
        const int me = tid & 63;
        for (int c0 = 0; __any(c0 < n); c0 += 12) {
            int4 A = {0, 0, 0, 0}, B = A, D = A;
            if (c0 < n) A = tc4[cand4_at(c0 >> 2, k)];
            if (c0 + 4 < n) B = tc4[cand4_at((c0 >> 2) + 1, k)];
            if (c0 + 8 < n) D = tc4[cand4_at((c0 >> 2) + 2, k)];
            unsigned hits = near(A.x) | near(A.y) << 1 | near(A.z) << 2 | near(A.w) << 3;
            if (__any(c0 + 4 < n)) hits |= near(B.x) << 4 | near(B.y) << 5 | near(B.z) << 6 | near(B.w) << 7;
            if (__any(c0 + 8 < n)) hits |= near(D.x) << 8 | near(D.y) << 9 | near(D.z) << 10 | near(D.w) << 11;
            hits &= (1u << max(0, min(n - c0, 12))) - 1u;  // (the words after the last candidate are zero)
            // places of the lanes' candidates: prefix sums of the counts, bit by bit
            const int h = __popc(hits);
            int first = 0, total = 0;
#pragma unroll
            for (int b = 0; b < 4; b++) {
                const unsigned long long m = __ballot((h >> b) & 1);
                first += __popcll(m & ((1ull << me) - 1)) << b;
                total += __popcll(m) << b;
            }
            for (int base = 0; base < total; base += 64) {
                int at = first - base;
                for (unsigned left = hits; left; left &= left - 1, at++)
                    if (at >= 0 && at < 64) sOwner[(tid & ~63) + at] = (unsigned char)me;
                __builtin_amdgcn_wave_barrier();  // (a wave's LDS accesses are carried out in order)
                asm volatile("" ::: "memory");
                const bool mine = base + me < total;
                const int owner = mine ? sOwner[tid] : me;
                unsigned oh = __shfl(hits, owner);
                const int oinfo = __shfl(info, owner);
                V3<T> fw = {0, 0, 0};
                int in = 0;
                for (int rank = base + me - __shfl(first, owner); mine && rank > 0; rank--) oh &= oh - 1;
                if (mine) {
                    const int q = __ffs(oh) - 1, own = (tid & ~63) + owner;
                    const int e = a.tcand[4 * (cbase + ((size_t)((c0 + q) >> 2) * KV + k) * NT + own) + (q & 3)];
                    const unsigned u = (unsigned)e;
                    const int3 o = {(int)(u << 11) >> 27, (int)(u << 6) >> 27, (int)(u << 1) >> 27};
                    in = partner(oinfo & 127, NT - 1 - own + k * NT, sVM[oinfo >> 7], e & 2047, o, sVM[(e >> 11) & 31], fw);
                }
                at = first - base;
                for (int r = 0; __any(r < h); r++, at++) {
                    const int src = min(max(at, 0), 63);
                    const V3<T> g = {__shfl(fw.x, src), __shfl(fw.y, src), __shfl(fw.z, src)};
                    const int on = __shfl(in, src);
                    if (r < h && at >= 0 && at < 64 && on) f = f + g;
                }
            }
        }
        return f;
    };
    if constexpr (COL) {
#pragma unroll
        for (int k = 0; k < KV; k++) pack(k);
    }

    for (int s = 0; s < nsteps; s++) {
        const int parity = (parity0 + s) & 1;
        // the packed words are taken apart in each step anew: what is derived from
        // them (the LDS addresses of a voxel's six links alone are two dozen
        // registers) is otherwise kept over the steps and pushes state into scratch.
        // Without collisions there is room for the rest, and taking it apart again
        // costs 1.5 % of the step.
        if constexpr (COL || sizeof(T) == 4) {
#pragma unroll
            for (int k = 0; k < KV; k++)
#pragma unroll
                for (int d = 0; d < 3; d++) pin(vLinks[k][d]);
        }
        if constexpr (COL) {
            pin(tid);
            pin(vt);
#pragma unroll
            for (int k = 0; k < KL; k++) { pin(lEnds[k]); pin(lInfo[k]); }
#pragma unroll
            for (int k = 0; k < KV; k++) { pin(vInfo[k]); pin(vLat[k]); pin(vCand[k]); }
        }
        if constexpr (COL) {
            // ---- candidate lists of the robots whose lists are stale (rare)
            if (tr.anyStale[parity]) {
                auto listing = [&](int j) { return tr.col[j] && !tr.diverged[j] && tr.stale[j]; };
                // Each robot's pairs are tested outright, from LDS: 16 lanes a
                // voxel, each a run of the robot's surface voxels, so that what
                // the lanes find, one after the other, is in ascending order.  A
                // robot of a tile has at most VMAX voxels, and its n^2 tests take
                // less time than the chain of grid lookups in memory that the
                // large robots' listing is (about 300 us of the workgroup, 6.6 us
                // of each step of the 1024-robot batch, against about 1).  The
                // forces' LDS is free until the link phase.
                constexpr int G = 16, RUN = (VMAX + G - 1) / G, WORDS = (RUN + 31) / 32;
                int *const work = reinterpret_cast<int *>(&sForce[0][0]);
                int *const sIdx = work, *const sLat = work + VMAX, *const sMt = work + 2 * VMAX, *const sCnt = work + 3 * VMAX;
                int *const sOver = work + 4 * VMAX, *const wsum = sOver + 1;
                for (int j = 0; j < nr; j++) {
                    if (!listing(j)) continue;  // (the same for every thread)
                    const int r = tr.rid[j];
                    const RobotParams &rp = a.rp[r];
                    const int soff = rp.soff, ns = rp.scount, lbase = tr.vpre[j] - tr.voffG[j];
                    if (tid == 0) *sOver = 0;
                    for (int i = tid; i < ns; i += NT) {
                        const int w = a.surf[soff + i], lw = w + lbase;
                        sIdx[i] = lw;
                        sLat[i] = a.lat[w];
                        sMt[i] = a.vmat[w];
                        a.bpos[w] = T4<T>{sPose[0][lw], sPose[1][lw], sPose[2][lw], sPose[3][lw]};
                    }
                    __syncthreads();
                    const int lane = tid % G, run = (ns + G - 1) / G, b0 = min(ns, lane * run), b1 = min(ns, b0 + run);
                    const T R2 = (T)rp.listR * (T)rp.listR;
                    for (int i = tid / G; i < ns; i += NT / G) {
                        const int lv = sIdx[i], pk = sLat[i], gv = lv - lbase;
                        const VoxelMat &mi = LDSMAT ? sVM[sMt[i]] : a.vmats[sMt[i]];
                        const T L = (T)mi.nomSize;
                        const T4<T> pv = {sPose[0][lv], sPose[1][lv], sPose[2][lv], (T)0};
                        const unsigned linked = (unsigned)(__ballot(lane < 6 && a.vlinks[6 * gv + min(lane, 5)] >= 0) >> (tid & 48)) & 63u;
                        unsigned found[WORDS];
                        int own = 0;
#pragma unroll
                        for (int m = 0; m < WORDS; m++) {
                            unsigned bits = 0;
                            for (int q = 0; q < 32 && b0 + 32 * m + q < b1; q++) {
                                const int c = b0 + 32 * m + q, lw = sIdx[c];
                                const int3 o = lat_offset(pk, sLat[c]);
                                const V3<T> df = col_diff<T>(pv, T4<T>{sPose[0][lw], sPose[1][lw], sPose[2][lw], (T)0}, o, L);
                                if (df.x * df.x + df.y * df.y + df.z * df.z > R2 || lw == lv) continue;
                                if (abs(o.x) + abs(o.y) + abs(o.z) == 1) {  // a lattice neighbour: left out when linked
                                    const int d = o.x ? (o.x > 0 ? 0 : 1) : (o.y ? (o.y > 0 ? 2 : 3) : (o.z > 0 ? 4 : 5));
                                    if ((linked >> d) & 1) continue;
                                }
                                if (mi.fixed && (LDSMAT ? sVM[sMt[c]] : a.vmats[sMt[c]]).fixed) continue;
                                bits |= 1u << q;
                            }
                            found[m] = bits;
                            own += __popc(bits);
                        }
                        int at = own;  // inclusive, then exclusive prefix over the voxel's lanes
                        for (int q = 1; q < G; q <<= 1) {
                            const int y = __shfl_up(at, q, G);
                            if (lane >= q) at += y;
                        }
                        const int n = __shfl(at, G - 1, G);
                        at -= own;
                        int *const list = a.clist + (long)(soff + i) * kMaxCand;
                        const int k = lv / NT, ownerTid = NT - 1 - lv % NT;
                        auto word = [&](int rank) -> int & {
                            return a.tcand[4 * (cbase + ((size_t)(rank >> 2) * KV + k) * NT + ownerTid) + (rank & 3)];
                        };
                        bool wide = !LDSMAT || n > kMaxCand;
#pragma unroll
                        for (int m = 0; m < WORDS; m++)
                            for (unsigned bits = found[m]; bits; bits &= bits - 1, at++) {
                                const int c = b0 + 32 * m + __ffs(bits) - 1, lw = sIdx[c];
                                const int3 o = lat_offset(pk, sLat[c]);
                                wide |= o.x < -16 || o.x > 15 || o.y < -16 || o.y > 15 || o.z < -16 || o.z > 15;
                                if (at >= kMaxCand) continue;
                                list[at] = lw - lbase;
                                word(at) = lw | (sMt[c] << 11) | ((o.x & 31) << 16) | ((o.y & 31) << 21) | ((o.z & 31) << 26);
                            }
                        if (lane < 3 && n + lane < ((n + 3) & ~3) && n + lane < kMaxCand) word(n + lane) = 0;
                        const bool anyWide = ((__ballot(wide) >> (tid & 48)) & 0xffff) != 0;
                        if (lane == 0) {
                            a.ccount[soff + i] = n;
                            sCnt[lv] = anyWide ? kWideCand : n;
                            if (n > kMaxCand) *sOver = 1;
                        }
                    }
                    __syncthreads();
#pragma unroll
                    for (int k = 0; k < KV; k++)
                        if (vt + k * NT < nv && vSlot(k) == j && vCand[k] != kNoCand) vCand[k] = sCnt[vt + k * NT];
                    // a voxel with more candidates than a list holds searches the
                    // grid of the listing: count, prefix sum, scatter
                    if (*sOver) {
                        for (int i = tid; i < ns; i += NT) {
                            const int lw = sIdx[i];
                            col_cell(a, rp, soff + i, lw - lbase, T4<T>{sPose[0][lw], sPose[1][lw], sPose[2][lw], sPose[3][lw]});
                        }
                        __syncthreads();
                        col_scan<false>(a, r, wsum);  // at most VMAX surface voxels: a few buckets per thread
                        __syncthreads();
                        for (int i = soff + tid; i < soff + ns; i += NT) col_record(a, rp, i, a.surf[i]);
                    }
                    __syncthreads();
                }
                if (tid < nr && listing(tid)) {
                    RobotTime &t = a.rt[tr.rid[tid]];
                    t.stale[parity] = 0;
                    t.listings += 1;
                    tr.stale[tid] = 0;
                }
                __syncthreads();  // before the contact phase may set them again
            }
        }
        // ---- links; a link past the divergence strain stops its robot before
        // the voxel phase (diverged itself changes only after the barrier, so
        // every link and contact of the step sees the same flag)
#pragma unroll
        for (int k = 0; k < KL; k++) {
            const int ll = tid + k * NT;
            if (ll >= nl) continue;
            const int j = (lInfo[k] >> 2) & 127;
            if (tr.diverged[j]) continue;
            const LinkMat &lm = LDSMAT ? sLM[lInfo[k] >> 9] : a.lmats[lInfo[k] >> 9];
            if (lm.fixedBoth) continue;
            const int n = lEnds[k] & 0xffff, p = lEnds[k] >> 16;
            const V3<T> du = {sPose[0][p] - sPose[0][n], sPose[1][p] - sPose[1][n], sPose[2][p] - sPose[2][n]};
            const Q4<T> qn = {sPose[3][n], sPose[4][n], sPose[5][n], sPose[6][n]};
            const Q4<T> qp = {sPose[3][p], sPose[4][p], sPose[5][p], sPose[6][p]};
            LinkOut<T> o;
            link_forces<T, true>(lm, a.curves, lInfo[k] & 3, du, qn, qp, (float)sPose[7][n], (float)sPose[7][p], tr.prevDt[parity][j],
                           ls[k], o);
            sForce[0][ll] = o.fN.x; sForce[1][ll] = o.fN.y; sForce[2][ll] = o.fN.z;
            sForce[3][ll] = o.mN.x; sForce[4][ll] = o.mN.y; sForce[5][ll] = o.mN.z;
            sForce[6][ll] = o.fP.x; sForce[7][ll] = o.fP.y; sForce[8][ll] = o.fP.z;
            sForce[9][ll] = o.mP.x; sForce[10][ll] = o.mP.y; sForce[11][ll] = o.mP.z;
            if constexpr (!COL) lStrain[k] = o.strain;
            else if (s == nsteps - 1) a.ls2[tr.loffG[j] + (ll - tr.lpre[j])].w = (T)o.strain;
            if (o.strain > 100.0f) tr.divNow[j] = 1;
        }
        // ---- contact forces, from the poses and momenta entering the step
        V3<T> cf[KV];
#pragma unroll
        for (int k = 0; k < KV; k++) {
            cf[k] = V3<T>{0, 0, 0};
            if constexpr (COL) {
                const int n = vCand[k] == kNoCand || tr.diverged[vSlot(k)] ? 0 : vCand[k];
                if constexpr (LDSMAT) {
                    if (__any(n > 0)) cf[k] = contact_wave(k, max(n, 0));
                }
                if (n == kWideCand) cf[k] = contact_wide(k, vt + k * NT, parity);
            }
        }
        __syncthreads();
        if (tid < nr && tr.divNow[tid]) tr.diverged[tid] = 1;  // (the voxel phase reads both)
        if (COL && tid == 0) tr.anyStale[parity] = 0;            // every thread has read it
        // ---- voxels
#pragma unroll
        for (int k = 0; k < KV; k++) {
            const int lv = vt + k * NT;
            if (lv >= nv) continue;
            const int j = vSlot(k);
            if (tr.diverged[j] || tr.divNow[j]) continue;
            const float dt = tr.dt[j];
            const double tnext = tr.time[parity][j] + (double)dt;
            if (lv == tr.vpre[j]) {
                tr.time[parity ^ 1][j] = tnext;
                tr.prevDt[parity ^ 1][j] = dt;
                tr.steps[j] += 1;
            }
            const VoxelMat &vm = LDSMAT ? sVM[vMat(k)] : a.vmats[vMat(k)];
            if (vm.fixed) continue;
            T phase;
            T4<T> bp{};
            if constexpr (KEEP) {
                phase = vPhase[k];
            } else {
                const int gv = vGlob(k);
                phase = a.phase[gv];
                bp = a.bpos[gv];
            }
            V3<T> fs = {0, 0, 0}, ms = {0, 0, 0};
#pragma unroll
            for (int d = 0; d < 6; d++) {
                const int l = (vLinks[k][d >> 1] >> (16 * (d & 1))) & 0xffff;
                if (l == 0xffff) continue;
                const int o = (d & 1) ? 6 : 0;  // NEG direction: this voxel is the pVPos end
                // link-frame end vectors back to the lattice frame (axis d / 2, known here)
                fs = fs + to_axis_original(V3<T>{sForce[o + 0][l], sForce[o + 1][l], sForce[o + 2][l]}, d >> 1);
                ms = ms + to_axis_original(V3<T>{sForce[o + 3][l], sForce[o + 4][l], sForce[o + 5][l]}, d >> 1);
            }
            float temp = (float)sPose[7][lv];
            const int tf = tr.tempFlags[j];
            VoxelState<T> now;
            VoxelState<T> &v = KEEP ? vs[k] : now;
            if constexpr (!KEEP) {
                v.u = {sPose[0][lv], sPose[1][lv], sPose[2][lv]};
                v.q = {sPose[3][lv], sPose[4][lv], sPose[5][lv], sPose[6][lv]};
                v.p = {sMom[0][lv], sMom[1][lv], sMom[2][lv]};
                v.h = vH[k];
                v.flags = vFlags[k];
            }
            voxel_step<T>(vm, a.exts, dt, vLat[k], temp, fs, ms, cf[k], V3<T>{0, 0, 0}, v);
            if ((tf & 1) && !(vm.thermalOnAfter > tnext)) {
                if constexpr (std::is_same<T, float>::value)
                    temp = actuation_temperature_f32(tr.tempAmp[j], tr.tempPeriod[j], tnext, (double)phase, tf >> 1);
                else
                    temp = actuation_temperature<T>(tr.tempAmp[j], tr.tempPeriod[j], tnext, (double)phase, tf >> 1);
            }
            if constexpr (!KEEP) {
                vH[k] = v.h;
                vFlags[k] = v.flags;
            }
            sPose[0][lv] = v.u.x; sPose[1][lv] = v.u.y; sPose[2][lv] = v.u.z; sPose[3][lv] = v.q.w;
            sPose[4][lv] = v.q.x; sPose[5][lv] = v.q.y; sPose[6][lv] = v.q.z; sPose[7][lv] = (T)temp;
            if constexpr (COL) {
                sMom[0][lv] = v.p.x; sMom[1][lv] = v.p.y; sMom[2][lv] = v.p.z;
                if (vCand[k] != kNoCand) {  // a moved surface voxel: its robot lists again next step
                    const T dx = v.u.x - bp.x, dy = v.u.y - bp.y, dz = v.u.z - bp.z;
                    if (dx * dx + dy * dy + dz * dz > (T)tr.staleD2[j]) {
                        tr.stale[j] = 1;
                        tr.anyStale[parity ^ 1] = 1;
                    }
                }
            }
        }
        __syncthreads();
    }

    // ---- write back
#pragma unroll
    for (int k = 0; k < KL; k++) {
        const int ll = tid + k * NT;
        if (ll >= nl) continue;
        const int j = (lInfo[k] >> 2) & 127;
        const int gl = tr.loffG[j] + (ll - tr.lpre[j]);
        a.ls0[gl] = T4<T>{ls[k].pos2.x, ls[k].pos2.y, ls[k].pos2.z, ls[k].a1v.x};
        a.ls1[gl] = T4<T>{ls[k].a1v.y, ls[k].a1v.z, ls[k].a2v.x, ls[k].a2v.y};
        if constexpr (!COL) {
            a.ls2[gl] = T4<T>{ls[k].a2v.z, (T)ls[k].maxStrain, (T)ls[k].flags, (T)lStrain[k]};
        } else {
            T *const l2 = &a.ls2[gl].x;
            l2[0] = ls[k].a2v.z;
            l2[1] = (T)ls[k].maxStrain;
            l2[2] = (T)ls[k].flags;
            if (tr.diverged[j] == 1 || (tr.diverged[j] == 0 && tr.divNow[j])) {
                // a robot that stopped in this launch: its last update was not the
                // launch's last step, the voxels are still where that update saw them
                const LinkMat &lm = LDSMAT ? sLM[lInfo[k] >> 9] : a.lmats[lInfo[k] >> 9];
                if (!lm.fixedBoth)
                    l2[3] = (T)(float)qdiv(ls[k].pos2.x, rest_length<T>(lm, (float)sPose[7][lEnds[k] & 0xffff], (float)sPose[7][lEnds[k] >> 16]));
            }
        }
    }
#pragma unroll
    for (int k = 0; k < KV; k++) {
        const int lv = vt + k * NT;
        if (lv >= nv) continue;
        const int gv = vGlob(k);
        a.pq0[gv] = T4<T>{sPose[0][lv], sPose[1][lv], sPose[2][lv], sPose[3][lv]};
        a.pq1[gv] = T4<T>{sPose[4][lv], sPose[5][lv], sPose[6][lv], sPose[7][lv]};
        V3<T> p, h;
        int flags;
        if constexpr (KEEP) {
            p = vs[k].p;
            h = vs[k].h;
            flags = vs[k].flags;
        } else {
            p = {sMom[0][lv], sMom[1][lv], sMom[2][lv]};
            h = vH[k];
            flags = vFlags[k];
        }
        a.mo0[gv] = T4<T>{p.x, p.y, p.z, h.x};
        a.mo1[gv] = T4<T>{h.y, h.z, (T)flags, (T)0};
    }
    if (tid < nr) {
        RobotTime &t = a.rt[tr.rid[tid]];
        t.time[0] = tr.time[0][tid];
        t.time[1] = tr.time[1][tid];
        t.prevDt[0] = tr.prevDt[0][tid];
        t.prevDt[1] = tr.prevDt[1][tid];
        t.diverged = (tr.diverged[tid] | tr.divNow[tid]) != 0;
        t.steps = tr.steps[tid];
        if constexpr (COL) {
            if (tr.col[tid]) {  // lists to build at the next step, as the flat path's tracking leaves them
                const int pe = (parity0 + nsteps) & 1;
                t.stale[pe] = tr.stale[tid];
                t.stale[pe ^ 1] = 0;
            }
        }
    }
    // the flat path's hint that some robot may be stale (per-robot flags decide)
    if (COL && blockIdx.x == 0 && tid == 0) a.anyStale[0] = a.anyStale[1] = 1;
}

}  // namespace vx3mi
