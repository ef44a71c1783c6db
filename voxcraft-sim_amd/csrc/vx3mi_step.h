// vx3mi_step.h -- the flat timestep with collisions for batches whose links stay
// as they are (no removal, detach or attach): the grid of a listing of contact
// candidates is filled by the voxel updates, the lists are made in the contact
// launch that needs them, and the contact phase takes each voxel's candidates at
// once.  Two launches a step, none of them for listing.
//
// The lists are those of the other paths, made in the same steps: a robot lists in
// the step after one that leaves a surface voxel beyond the limit of its skin
// (hardStep).  The grid that takes is a hashed table of chains.  The voxel updates
// of a step put their surface voxels at the heads of the chains (gridStep: the step
// whose updates do), so it is whole when the contact launch comes, whatever the
// robot's size.  Whether the updates of a step are to do that is known a step
// before: a voxel that may pass the limit by then, at twice the speed it has, asks
// for it.  A robot that passes the limit with no such warning (a blow: within one
// step from 0.9 of the limit less twice its speed) tests every pair of its surface
// voxels in one step, and from then on until its state is replaced (jumped) its
// updates fill the grid in every step.  So a step costs at the most a listing,
// however fast the voxels are.
//
// us per call with a launch for the listings before every step, and like this: one
// body of 45,700 voxels in FP32, 500 steps, 11,430 and 10,350; one of 17,200 in FP64,
// 150 steps, 3,815 and 3,195; 200 robots, 62,800 voxels, in FP64, 200 steps, 10,280 and
// 7,630; 48 robots with signals, cilia and force fields in FP32, 300 steps, 9,700 and
// 8,050.  The same body of 45,700 voxels from a new state, thrown at 150 m/s (it lists
// in every fourth step), 100 steps: 76 and 28 us a step.
//
// What bounds the step: two launches, each a chain of loads at one or two waves a
// SIMD (the body in FP32: 12.5 us of contacts and links, 7.4 us of voxels), and with
// many robots the lists some of them make in nearly every step (200 robots: 34 us of
// contacts and links, 15 without a list).
#pragma once

#include <hip/hip_runtime.h>

namespace vx3mi {

// a robot is warned of a listing from this part of its limit on
constexpr float kListWarn = 0.9f;

struct ListArgs {
    ulonglong2 *head;  // per bucket the heads of its two chains: serial number of the filling (upper half), first voxel
    int4 *node;        // per voxel: its cell at the last filling, the voxel after it in the chain (-1: none)
    int nmats;         // voxel materials
    int step;          // number of the step within the run, from 0
    unsigned serial;   // of the grid that step 0 of the run takes; step k takes serial + k
};

template <typename T = void> __global__ __launch_bounds__(256) void k_clear_heads(ulonglong2 *head, long n) {
    for (long i = blockIdx.x * 256l + threadIdx.x; i < n; i += gridDim.x * 256l) head[i] = ulonglong2{0, 0};
}

// the bucket of a cell.  Four buckets to one of the counting sort's table: what a chain
// holds of other cells is walked for nothing (200 robots in FP64, 200 steps, 7.95 ms
// with one, 7.73 with four).
constexpr int kGridSpread = 4;
__device__ __forceinline__ long grid_bucket(const RobotParams &rp, int cx, int cy, int cz) {
    return kGridSpread * (long)rp.toff + (cell_hash(cx, cy, cz) & (unsigned)(kGridSpread * (rp.mask + 1) - 1));
}

// surface voxel v at position field q put into the grid
template <typename T>
__device__ __forceinline__ void grid_put(const Dev<T> &a, const ListArgs &f, const RobotParams &rp, int v, const T4<T> &q, unsigned serial) {
    const V3<double> p = position_d<T>(a.lat[v], a.vmats[a.vmat[v]].nomSize, V3<T>{q.x, q.y, q.z});
    const double h = rp.listR;
    const int cx = (int)floor(p.x / h), cy = (int)floor(p.y / h), cz = (int)floor(p.z / h);
    unsigned long long *const head = &f.head[grid_bucket(rp, cx, cy, cz)].x + (v & 1);
    const unsigned long long was = atomicExch(head, (unsigned long long)serial << 32 | (unsigned)v);
    f.node[v] = int4{cx, cy, cz, (unsigned)(was >> 32) == serial ? (int)(unsigned)was : -1};
}
// the first voxels of a cell's chains, -1 for none
__device__ __forceinline__ int2 grid_heads(const ListArgs &f, const RobotParams &rp, int cx, int cy, int cz) {
    const ulonglong2 w = f.head[grid_bucket(rp, cx, cy, cz)];
    const unsigned serial = f.serial + (unsigned)f.step;
    return int2{(unsigned)(w.x >> 32) == serial ? (int)(unsigned)w.x : -1, (unsigned)(w.y >> 32) == serial ? (int)(unsigned)w.y : -1};
}

// LDS of a wave that makes lists: its 16 voxels, their candidates, the chains to walk
template <typename T> struct alignas(16) ListRoom {
    static constexpr int N = 64 / kContactLanes;
    static constexpr int CHAINS = N * 27 * 2;
    int row[N][kMaxCand + 4];  // (rows of 52 words: 16 rows' 16-byte words fall on different banks)
    union {
        int chain[CHAINS + 1];      // first voxel of a chain (the last place: of none)
        int list[N][kMaxCand + 4];  // the row in ascending order, when the chains are done
    };
    unsigned short place[CHAINS + 1];  // of the voxel a chain is for, and the cell of the 27 around it
    T x[N], y[N], z[N], L[N], R2[N];
    int cx[N], cy[N], cz[N], lat[N], info[N], count[N];  // info: links by direction, bit 6: fixed
};

// The lists and counts of the wave's voxels, kContactLanes lanes each (every lane
// calls; want: the voxel has one to make), as col_list_group makes them, from the grid
// of this step, whose positions are the state entering it.  Returns the count to the
// voxel's lanes, nc to those with nothing to make.  The heads of all the wave's
// chains are requested at once; the chains with a voxel are walked by whichever lane
// is free, two to a lane, a node's cell and position in one load level: some ten
// dependent loads for the wave, where sixteen lanes to a voxel walked each voxel's
// chains on their own, four voxels after four (some thirty; the 200 robots in FP64
// 10.0 ms, 7.6 like this).  What is left is issue: three or four chains to a lane are
// no faster than two.
template <typename T>
__device__ __forceinline__ int step_list_wave(const Dev<T> &a, const ListArgs &f, int s, int v, bool want, int nc, const T4<T> &q0,
                                              const int4 &cs, int pk, int mat, const RobotParams &rp,
                                              ListRoom<T> &room) {
    constexpr int CELLS = (27 + kContactLanes - 1) / kContactLanes, NB = 2;
    const int me = threadIdx.x & 63, slot = me / kContactLanes, lane = me % kContactLanes;
    const unsigned long long below = (1ull << me) - 1;
    const int la = a.vlinks[6 * v + lane], lb = lane < 2 ? a.vlinks[6 * v + kContactLanes + lane] : -1;
    const int linked = (int)(__ballot(la >= 0) >> (slot * kContactLanes) & 15) | (int)(__ballot(lb >= 0) >> (slot * kContactLanes) & 3) << 4;
    if (lane == 0) {
        const VoxelMat &mi = a.vmats[mat];
        room.x[slot] = q0.x;
        room.y[slot] = q0.y;
        room.z[slot] = q0.z;
        room.L[slot] = (T)mi.nomSize;
        room.R2[slot] = (T)rp.listR * (T)rp.listR;
        room.cx[slot] = cs.x;
        room.cy[slot] = cs.y;
        room.cz[slot] = cs.z;
        room.lat[slot] = pk;
        room.info[slot] = linked | (mi.fixed ? 64 : 0);
        room.count[slot] = 0;
    }
    int2 head[CELLS];
    int total = 0, next = 0;
#pragma unroll
    for (int t = 0; t < CELLS; t++) {
        const int c = lane + t * kContactLanes;
        const int2 h = grid_heads(f, rp, cs.x + c % 3 - 1, cs.y + (c / 3) % 3 - 1, cs.z + c / 9 - 1);
        head[t] = want && c < 27 ? h : int2{-1, -1};
    }
#pragma unroll
    for (int t = 0; t < 2 * CELLS; t++) {
        const int h = t & 1 ? head[t / 2].y : head[t / 2].x;
        const unsigned long long m = __ballot(h >= 0);
        const int at = h >= 0 ? total + __popcll(m & below) : ListRoom<T>::CHAINS;
        room.chain[at] = h;
        room.place[at] = (unsigned short)(slot | (lane + t / 2 * kContactLanes) << 4);
        total += __popcll(m);
    }
    __builtin_amdgcn_wave_barrier();  // (a wave's LDS accesses are carried out in order)
    asm volatile("" ::: "memory");
    int w[NB], tag[NB];
#pragma unroll
    for (int j = 0; j < NB; j++) {
        w[j] = -1;
        tag[j] = 0;
    }
    for (;;) {
#pragma unroll
        for (int j = 0; j < NB; j++) {  // the free lanes take the next chains
            const unsigned long long m = __ballot(w[j] < 0);
            const int at = next + __popcll(m & below);
            if (w[j] < 0 && at < total) {
                w[j] = room.chain[at];
                tag[j] = room.place[at];
            }
            next = min(total, next + __popcll(m));
        }
        if (!__any(w[0] >= 0 || w[1] >= 0)) break;
        int4 g[NB];
        T4<T> pw[NB];
        int lw[NB];
#pragma unroll
        for (int j = 0; j < NB; j++) {
            const int at = w[j] >= 0 ? w[j] : v;
            g[j] = f.node[at];
            pw[j] = a.pq0[at];
            lw[j] = a.lat[at];
        }
#pragma unroll
        for (int j = 0; j < NB; j++) {  // (tests joined without branches: a branch costs more than the test)
            const int i = tag[j] & 15, c = tag[j] >> 4;
            const int dx = g[j].x - room.cx[i] + 1, dy = g[j].y - room.cy[i] + 1, dz = g[j].z - room.cz[i] + 1;
            const int3 o = lat_offset(room.lat[i], lw[j]);
            const T4<T> pv = {room.x[i], room.y[i], room.z[i], (T)0};
            const V3<T> d = col_diff<T>(pv, pw[j], o, room.L[i]);
            const int far = abs(o.x) + abs(o.y) + abs(o.z);
            // direction of a lattice neighbour, as of its link
            const int k = (o.y != 0 ? 2 : 0) + (o.z != 0 ? 4 : 0) + (o.x + o.y + o.z < 0 ? 1 : 0);
            // another cell of the bucket, beyond the radius, itself, linked
            const int in = (w[j] >= 0) & ((unsigned)dx < 3) & ((unsigned)dy < 3) & ((unsigned)dz < 3) & (dx + 3 * dy + 9 * dz == c) &
                           !(d.x * d.x + d.y * d.y + d.z * d.z > room.R2[i]) & (far != 0) & !((far == 1) & (room.info[i] >> (k & 7)));
            bool keep = in != 0;
            if (keep && (room.info[i] & 64)) keep = !a.vmats[a.vmat[w[j]]].fixed;
            if (keep) {
                const int at = atomicAdd(&room.count[i], 1);
                if (at < kMaxCand) room.row[i][at] = w[j];
            }
            w[j] = w[j] >= 0 ? g[j].w : -1;
        }
    }
    __builtin_amdgcn_wave_barrier();
    asm volatile("" ::: "memory");
    const int n = room.count[slot];
    int *const list = a.clist + (long)s * kMaxCand;
    if (want) {
        for (int k = lane; k < (n <= kMaxCand ? n : 0); k += kContactLanes) {  // each to the place its rank among all gives it
            const int e = room.row[slot][k];
            int rank = 0;
            for (int m = 0; m < n; m += 4) {
                const int4 o = *reinterpret_cast<const int4 *>(&room.row[slot][m]);
                rank += (o.x < e) + (m + 1 < n && o.y < e) + (m + 2 < n && o.z < e) + (m + 3 < n && o.w < e);
            }
            list[rank] = room.list[slot][rank] = e;
        }
        if (lane == 0) a.ccount[s] = n;
    }
    __threadfence_block();  // the list, for the other lanes
    __builtin_amdgcn_wave_barrier();
    asm volatile("" ::: "memory");
    return want ? n : nc;
}

// the force on surface voxel v from candidate w when the two are in contact now
// (bit 0 of the result), from the state a holds; bit 1: a target touches a
// non-target.  col_contact_sum's partner for robots whose links stay.
template <typename T> __device__ __forceinline__ int step_pair(const Dev<T> &a, int v, int w, V3<T> &fw) {
    const int pkv = a.lat[v], pkw = a.lat[w], matV = a.vmat[v], matW = a.vmat[w];
    T4<T> qi0 = a.pq0[v], qj0 = a.pq0[w], mi0 = a.mo0[v], mj0 = a.mo0[w];
    T ti = a.pq1[v].w, tj = a.pq1[w].w;
    const VoxelMat &mi = a.vmats[matV], &mj = a.vmats[matW];
    pin(qi0);
    pin(qj0);
    pin(mi0);
    pin(mj0);
    pin(ti);
    pin(tj);
    if (mi.fixed && mj.fixed) return 0;
    T bsaI = base_size_average<T>(mi.nomSize, (float)ti, mi.alphaCTE);
    pin(bsaI);  // rounded by itself, as where one size serves a voxel's whole list
    const V3<T> diff = col_diff<T>(qi0, qj0, lat_offset(pkv, pkw), (T)mi.nomSize);
    const T bsaJ = base_size_average<T>(mj.nomSize, (float)tj, mj.alphaCTE);
    if (!in_contact_envelope(diff, bsaI, bsaJ)) return 0;
    int got = 1;
    if (a.vtarget && a.vtarget[w] != a.vtarget[v]) {  // a target touching a non-target (:711-726)
        if (v < w) atomicAdd(&a.rt[a.vrob[v]].collisionCount, 1);
        got = 3;
    }
    if (a.pairRec && v < w) {
        const int k = atomicAdd(a.pairN, 1);
        if (k < a.pairCap) a.pairRec[k] = int2{v, w};
    }
    const V3<T> velI = V3<T>{mi0.x, mi0.y, mi0.z} * (T)mi.massInv, velJ = V3<T>{mj0.x, mj0.y, mj0.z} * (T)mj.massInv;
    fw = contact_force(diff, bsaI, bsaJ, velI, velJ, mi.penKinv, mj.penKinv, mi.cDampT, mj.cDampT);
    return got;
}

// materials whose size a wave keeps in LDS for the first test of its candidates
constexpr int kStepMats = 64;

// The contact force on surface voxel s (every lane of a wave calls it, s >= S for
// none; kContactLanes lanes a voxel), and the list of its voxel where its robot lists
// in this step.  Each lane takes three of a dozen candidates, whose words are
// requested as soon as the list's are there, and keeps those that may be in contact;
// what the wave keeps, about one for every second voxel, is dealt out over its lanes
// for the exact test and the force, which are added in candidate order (as in the
// collision tiles' contact phase).
// room, owner, env: LDS of the wave.
template <typename T>
__device__ __forceinline__ void step_contact(const Dev<T> &a, const ListArgs &f, int S, int s, int lane, int parity, ListRoom<T> &room,
                                             unsigned char *owner, float2 *env) {
    constexpr int NB = 3, STEP = NB * kContactLanes;
    const int me = threadIdx.x & 63;
    const bool there = s < S;
    const int sv = there ? s : S - 1;
    int *const list = a.clist + (long)sv * kMaxCand;
    int nc = there ? a.ccount[sv] : 0;
    int id[NB];
#pragma unroll
    for (int b = 0; b < NB; b++) id[b] = list[b * kContactLanes + lane];
    const int v = a.surf[sv];
    const int r = a.vrob[v], pk = a.lat[v], mat = a.vmat[v];
    const T4<T> q0 = a.pq0[v];
    int4 cell = {0, 0, 0, 0};  // of the grid, in a step that lists
    const float temp = (float)a.pq1[v].w;
    RobotTime *rt = a.rt + r;
    const RobotParams &rp = a.rp[r];
    if (me < f.nmats) env[me] = float2{(float)a.vmats[me].nomSize, (float)a.vmats[me].nomSize * a.vmats[me].alphaCTE};
    const bool all = f.nmats > kStepMats;  // (then every candidate goes to the exact test)
    const bool live = there && rp.collisions && !rt->diverged;
    const bool hard = live && rt->hardStep[parity] == f.step;
    const bool lists = hard && rt->gridStep[parity ^ 1] == f.step - 1;
    if (__any(lists)) {
        cell = f.node[v];
        nc = step_list_wave(a, f, sv, v, lists, nc, q0, cell, pk, mat, rp, room);
        if (lists)
#pragma unroll
            for (int b = 0; b < NB; b++) id[b] = room.list[me / kContactLanes][b * kContactLanes + lane];
        if (lists && lane == 0) {
            a.bpos[v] = q0;
            if (sv == rp.soff) rt->listings += 1;
            if (nc > kMaxCand) {  // searches the grid, in every step while this lasts
                rt->hardStep[parity ^ 1] = f.step + 1;
                rt->gridStep[parity] = f.step;
            }
        }
    }
    // lists that may miss a pair, with no grid to list from; a voxel with more candidates than a list holds
    const bool odd = (hard && !lists) || (live && nc > kMaxCand);
    const int n = live && !odd ? nc : 0;
    V3<T> c = {0, 0, 0};
    int hit = 0;
    const unsigned long long below = (1ull << me) - 1;
    for (int c0 = 0; __any(c0 < n); c0 += STEP) {
        unsigned long long near[NB];
        int total = 0, first[NB];
        T4<T> qw[NB];
        float tw[NB];
        int pw[NB], mw[NB];
#pragma unroll
        for (int b = 0; b < NB; b++) {
            if (c0 > 0) id[b] = c0 + b * kContactLanes + lane < n ? list[c0 + b * kContactLanes + lane] : v;
            const int w = c0 + b * kContactLanes + lane < n ? id[b] : v;
            qw[b] = a.pq0[w];
            tw[b] = (float)a.pq1[w].w;
            pw[b] = a.lat[w];
            mw[b] = a.vmat[w];
        }
        __builtin_amdgcn_wave_barrier();  // (a wave's LDS accesses are carried out in order)
        asm volatile("" ::: "memory");
        const float Lf = all ? 0.0f : env[mat].x, bi = all ? 0.0f : Lf + temp * env[mat].y;
#pragma unroll
        for (int b = 0; b < NB; b++) {
            // the exact test's own difference: over hundreds of lattice lengths its FP32
            // rounding passes the margin below
            const V3<T> df = col_diff<T>(q0, qw[b], lat_offset(pk, pw[b]), (T)Lf);
            const float dx = (float)df.x, dy = (float)df.y, dz = (float)df.z;
            bool keep = true;
            if (!all) {
                const float2 ew = env[mw[b]];
                const float w = 0.6250125f * (bi + ew.x + tw[b] * ew.y);  // the envelope radius, rounded up by 2e-5
                keep = dx * dx + dy * dy + dz * dz < w * w;
            }
            near[b] = __ballot(keep && c0 + b * kContactLanes + lane < n);
            first[b] = total;
            total += __popcll(near[b]);
        }
        for (int base = 0; base < total; base += 64) {
#pragma unroll
            for (int b = 0; b < NB; b++) {
                const int at = first[b] + __popcll(near[b] & below) - base;
                if (((near[b] >> me) & 1) && at >= 0 && at < 64) owner[at] = (unsigned char)(me | b << 6);
            }
            __builtin_amdgcn_wave_barrier();
            asm volatile("" ::: "memory");
            const bool mine = base + me < total;
            const int o = mine ? owner[me] : me, ol = o & 63, ob = o >> 6;
            const int ov = __shfl(v, ol), w0 = __shfl(id[0], ol), w1 = __shfl(id[1], ol), w2 = __shfl(id[2], ol);
            V3<T> fw = {0, 0, 0};
            int got = 0;
            if (mine) got = step_pair(a, ov, ob == 0 ? w0 : ob == 1 ? w1 : w2, fw);
#pragma unroll
            for (int b = 0; b < NB; b++) {
                unsigned mask = (unsigned)(near[b] >> (me & ~(kContactLanes - 1))) & ((1u << kContactLanes) - 1);
                while (__any(mask != 0)) {
                    const int src = (me & ~(kContactLanes - 1)) + (mask ? __ffs(mask) - 1 : 0);
                    const int at = first[b] + __popcll(near[b] & ((1ull << src) - 1)) - base, from = min(max(at, 0), 63);
                    const V3<T> g = {__shfl(fw.x, from), __shfl(fw.y, from), __shfl(fw.z, from)};
                    const int on = __shfl(got, from);
                    if (mask && at >= 0 && at < 64 && on) {
                        c = c + g;
                        hit |= on >> 1;
                    }
                    mask &= mask - 1;
                }
            }
        }
    }
    if (odd)
        c = col_contact_sum(
            a, rp, rt, sv, v, lane, lists ? COL_GRID : COL_ALL, nc, 0, mat, pk, q0, a.pq1[v], a.mo0[v], hit, [&](auto &&use) {
                for (int k = 0; k < 27; k++) {
                    const int cx = cell.x + k % 3 - 1, cy = cell.y + (k / 3) % 3 - 1, cz = cell.z + k / 9 - 1;
                    const int2 h = grid_heads(f, rp, cx, cy, cz);
                    for (int w0 = h.x, w1 = h.y; w0 >= 0 || w1 >= 0;) {
                        const int4 g0 = f.node[max(w0, 0)], g1 = f.node[max(w1, 0)];
                        if (w0 >= 0 && w0 != v && g0.x == cx && g0.y == cy && g0.z == cz) use(w0);
                        if (w1 >= 0 && w1 != v && g1.x == cx && g1.y == cy && g1.z == cz) use(w1);
                        w0 = w0 >= 0 ? g0.w : -1;
                        w1 = w1 >= 0 ? g1.w : -1;
                    }
                }
            });
    if (!live || lane != 0) return;
    // with signals a non-target voxel touching a target receives a forced 100
    if (hit && !(a.vtarget && a.vtarget[v]) && a.sig && rp.signals) {
        VoxelSignal sg = a.sig[v];
        signal_receive(sg, a.sigMat[v], 100, rt->time[parity], true);
        a.sig[v] = sg;
    }
    a.contactW[v] = T4<T>{c.x, c.y, c.z, 0};
}

// the contact phase and the link updates of a step side by side in one launch (as
// k_contact_links), and with FIELD the force fields (7 us as a launch of their own,
// formula by formula in each voxel)
template <typename T, int FIELD>
__global__ __launch_bounds__(256) void k_list_contact_links(Dev<T> a, ListArgs f, int nv, int nbf, int nl, int nbl, int ns, int parity) {
    __shared__ ListRoom<T> sRoom[4];
    __shared__ unsigned char sOwner[256];
    __shared__ float2 sEnv[4][kStepMats];
    int blk = blockIdx.x;
    if (FIELD && blk < nbf) {
        const int v = blk * blockDim.x + threadIdx.x;
        if (v < nv) field_update(a, v, parity);
    } else if ((blk -= FIELD ? nbf : 0) < nbl) {
        const int l = blk * blockDim.x + threadIdx.x;
        if (l < nl) link_update(a, l, parity);
    } else {
        const int i = (blk - nbl) * blockDim.x + threadIdx.x;
        step_contact(a, f, ns, i / kContactLanes, i % kContactLanes, parity, sRoom[threadIdx.x >> 6],
                     sOwner + (threadIdx.x & ~63), sEnv[threadIdx.x >> 6]);
    }
}

// the voxel update, which fills the grid and tells whose lists the next step cannot use
template <typename T> __global__ __launch_bounds__(256) void k_list_voxels(Dev<T> a, ListArgs f, int V, int parity) {
    const int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= V) return;
    const int sv = a.vsurf[v], r = a.vrob[v];
    const T4<T> b = a.bpos[v];
    const T4<T> was = a.pq0[v];
    voxel_update<true>(a, v, parity);
    RobotTime *rt = a.rt + r;
    if (sv < 0 || rt->diverged) return;
    const bool put = rt->gridStep[parity] == f.step, jumped = rt->jumped != 0;  // (set by earlier launches)
    const RobotParams &rp = a.rp[r];
    const T4<T> now = a.pq0[v];
    const T d2 = col_moved2(now, b);
    if (d2 > (T)rp.staleD2) {
        rt->hardStep[parity ^ 1] = f.step + 1;
        if (!put) rt->jumped = 1;
    }
    const float ahead = fsqrt((float)d2) + 2.0f * fsqrt((float)col_moved2(now, was));
    if (jumped || ahead > kListWarn * fsqrt(rp.staleD2)) rt->gridStep[parity ^ 1] = f.step + 1;
    if (put) grid_put(a, f, rp, v, now, f.serial + f.step + 1);
}

// before a run of such steps: robots whose lists are stale list in its first step.
// What that step moves is not known: its voxel updates fill the grid.
template <typename T> __global__ __launch_bounds__(256) void k_list_begin(Dev<T> a, ListArgs f, int R, int S, int parity) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    for (int r = i; r < R; r += gridDim.x * blockDim.x) {
        RobotTime &rt = a.rt[r];
        const bool any = a.rp[r].scount > 0;
        rt.hardStep[parity] = any && rt.stale[parity] ? 0 : -2;
        rt.hardStep[parity ^ 1] = any && rt.stale[parity ^ 1] ? 1 : -2;  // (a new state: both)
        rt.gridStep[parity] = 0;
        rt.gridStep[parity ^ 1] = -1;
    }
    if (i >= S) return;
    const int v = a.surf[i], r = a.vrob[v];
    if (a.rt[r].stale[parity]) grid_put(a, f, a.rp[r], v, a.pq0[v], f.serial);
}

// and after it: the listing flags of the other modes.  n: steps of the run, parity:
// of the step to come
template <typename T> __global__ __launch_bounds__(256) void k_list_end(Dev<T> a, int R, int n, int parity) {
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r == 0) a.anyStale[0] = a.anyStale[1] = 1;
    if (r >= R) return;
    a.rt[r].stale[parity] = a.rt[r].hardStep[parity] == n;
    a.rt[r].stale[parity ^ 1] = 0;
}

}  // namespace vx3mi
