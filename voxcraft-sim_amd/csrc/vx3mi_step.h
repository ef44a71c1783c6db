// vx3mi_step.h -- the flat timestep with collisions for batches whose links stay
// as they are (no removal, detach or attach): the listing of contact candidates
// runs beside the steps, and the contact phase takes each voxel's candidates at
// once.
//
// A listing is a launch of its own before every step, which waits for it: 3 us with
// nothing to list, 7 with, and the lists in the contact launch on top.  A batch of
// many robots lists some robot in almost every step (200 robots in FP64: 61 us a
// step, 26 without collisions, before lists were made by lane groups and beside the
// steps; 40 now).  Here the step that sees a voxel near the limit of its robot's
// skin starts a listing (RobotTime::listStep = the next step): workgroups of that
// step's contact launch build the robot's grid, and each of the four contact
// launches after it makes the lists of a quarter of each wave's voxels (all four
// quarters at once: 47 us a step there, half and half 43, a quarter 40).  Until then
// the old lists serve: "near the limit" looks kListLead steps ahead at the speed of
// the step, and should a voxel pass the limit with old lists in use all the same, the
// next step tests every pair of its robot (hardStep).  The partners are the all-pairs
// loop's in every step, so nothing else depends on when the lists were built.
//
// What bounds the step: two launches, each a chain of loads at one or two waves a
// SIMD; one body of 45,700 voxels in FP32 runs 12.5 us of contacts and links and
// 7.4 us of voxels (23.2 -> 20.6 us a step).
#pragma once

#include <hip/hip_runtime.h>

namespace vx3mi {

template <typename T> struct ListArgs {
    T4<T> *bold;           // per voxel: position field at the listing before the one under way
    int nmats;             // voxel materials
    int step;              // number of the step within the run, from 0
    int *hard, *hardHost;  // surface voxels of a robot that tested every pair, summed over the steps of the run,
                           // and the last such step; of the last run, for the host
};

constexpr int kListPerStep = 1;                           // rounds of a wave's lists a step
constexpr int kListSteps = kListRounds / kListPerStep;    // the step whose contact phase makes the last lists
constexpr float kListLead = 1.5f * (kListSteps + 1);
// robots of more surface voxels than this (all pairs: a millisecond and more of the
// device) take their first kListYoung steps from a new state with a listing before
// each step that needs one: bodies whose actuation starts at once move through the
// skin in a step or two (first call of 500 steps of a body of 45,700 voxels: 8 such
// steps 35 ms, 24 14.0, 64 13.1, 128 13.0)
constexpr int kListYoungVoxels = 4096, kListYoung = 64;

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
// none; kContactLanes lanes a voxel), and the passes of a listing under way that
// belong to the contact phase.  Each lane takes three of a dozen candidates, whose
// words are requested as soon as the list's are there, and keeps those that may be
// in contact; what the wave keeps, about one for every second voxel, is dealt out
// over its lanes for the exact test and the force, which are added in candidate
// order (as in the collision tiles' contact phase).
// q: LDS for listing, of the lane's kListLanes; owner, env: the wave's.
template <typename T>
__device__ __forceinline__ void step_contact(const Dev<T> &a, const ListArgs<T> &f, int S, int s, int lane, int parity, int *q,
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
    const float temp = (float)a.pq1[v].w;
    RobotTime *rt = a.rt + r;
    const RobotParams &rp = a.rp[r];
    if (me < f.nmats) env[me] = float2{(float)a.vmats[me].nomSize, (float)a.vmats[me].nomSize * a.vmats[me].alphaCTE};
    const bool all = f.nmats > kStepMats;  // (then every candidate goes to the exact test)
    const bool live = there && !rt->diverged;
    const int phase = f.step - rt->listStep;  // of the listing under way
    const bool lists = live && phase >= 1 && phase <= kListSteps;
    if (__any(lists)) {
        nc = col_list_wave(a, sv, v, lists, nc, max(phase - 1, 0) * kListPerStep, kListPerStep, q);
#pragma unroll
        for (int b = 0; b < NB; b++) id[b] = list[b * kContactLanes + lane];
    }
    // the step whose lists may miss a pair; a voxel with more candidates than a list holds
    const bool odd = live && rp.collisions && (rt->hardStep[parity] == f.step || nc > kMaxCand);
    const int n = live && rp.collisions && !odd ? nc : 0;
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
            float dx = (float)(q0.x - qw[b].x), dy = (float)(q0.y - qw[b].y), dz = (float)(q0.z - qw[b].z);
            if constexpr (!kAbsolutePositions<T>) {
                const int3 o = lat_offset(pk, pw[b]);
                dx -= (float)o.x * Lf;
                dy -= (float)o.y * Lf;
                dz -= (float)o.z * Lf;
            }
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
    if (odd) {
        // the grid and the cells go together outside a listing only
        const bool grid = rt->hardStep[parity] != f.step && phase != 0;
        c = col_contact_sum(a, rp, rt, sv, v, lane, grid ? COL_GRID : COL_ALL, nc, 0, mat, pk, q0, a.pq1[v], a.mo0[v], hit);
    }
    if (!live || !rp.collisions || lane != 0) return;
    // with signals a non-target voxel touching a target receives a forced 100
    if (hit && !(a.vtarget && a.vtarget[v]) && a.sig && rp.signals) {
        VoxelSignal sg = a.sig[v];
        signal_receive(sg, a.sigMat[v], 100, rt->time[parity], true);
        a.sig[v] = sg;
    }
    a.contactW[v] = T4<T>{c.x, c.y, c.z, 0};
}

// the contact phase and the link updates of a step side by side in one launch (as
// k_contact_links), the grids of robots that begin a listing, and with FIELD the
// force fields (7 us as a launch of their own, formula by formula in each voxel)
template <typename T, int FIELD>
__global__ __launch_bounds__(256) void k_list_contact_links(Dev<T> a, ListArgs<T> f, int nbg, int parts, int nv, int nbf, int nl,
                                                            int nbl, int ns, int parity) {
    __shared__ int sQueue[256 / kListLanes * kListQueue];
    __shared__ unsigned char sOwner[256];
    __shared__ float2 sEnv[4][kStepMats];
    __shared__ int wsum[16], lastPart;
    int blk = blockIdx.x;
    if (blk < nbg) {
        const int r = blk / parts;
        // (not the robot's diverged: a link of this launch may set it)
        if (a.rt[r].listStep == f.step) col_grid_part(a, a.rp[r], r, blk % parts, wsum, lastPart, f.bold);
    } else if (FIELD && (blk -= nbg) < nbf) {
        const int v = blk * blockDim.x + threadIdx.x;
        if (v < nv) field_update(a, v, parity);
    } else if ((blk -= FIELD ? nbf : nbg) < nbl) {
        const int l = blk * blockDim.x + threadIdx.x;
        if (l < nl) link_update(a, l, parity);
    } else {
        const int i = (blk - nbl) * blockDim.x + threadIdx.x;
        step_contact(a, f, ns, i / kContactLanes, i % kContactLanes, parity, sQueue + threadIdx.x / kListLanes * kListQueue,
                     sOwner + (threadIdx.x & ~63), sEnv[threadIdx.x >> 6]);
    }
}

// the voxel update with the passes of a listing under way that belong to it
template <typename T> __global__ __launch_bounds__(256) void k_list_voxels(Dev<T> a, ListArgs<T> f, int V, int parity) {
    const int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= V) return;
    const int sv = a.vsurf[v], r = a.vrob[v];
    const T4<T> b = a.bpos[v];
    const T4<T> was = a.pq0[v];
    float before;
    {
        const T dx = was.x - b.x, dy = was.y - b.y, dz = was.z - b.z;
        before = fsqrt((float)(dx * dx + dy * dy + dz * dz));
    }
    voxel_update<true>(a, v, parity);
    RobotTime *rt = a.rt + r;
    const RobotParams &rp = a.rp[r];
    if (rp.scount == 0 || rt->diverged) return;
    const int phase = f.step - rt->listStep;
    if (v == rp.voff) {
        if (phase == kListSteps || (f.step == 0 && rt->stale[parity])) rt->listings += 1;
        if (f.step == 0) rt->stale[0] = rt->stale[1] = 0;
        // (the robots of a step do it side by side)
        if (rt->hardStep[parity] == f.step && atomicExch(&f.hard[1], f.step) != f.step) atomicAdd(f.hard, rp.scount);
    }
    if (sv < 0) return;
    const T4<T> now = a.pq0[v];
    const T dx = now.x - b.x, dy = now.y - b.y, dz = now.z - b.z;
    float moved = fsqrt((float)(dx * dx + dy * dy + dz * dz));
    const float ahead = kListLead * (moved - before), limit = fsqrt(rp.staleD2);
    if (phase >= kListSteps && moved + ahead > limit) rt->listStep = f.step + 1;
    if (phase >= 0 && phase < kListSteps - 1) {  // some lists of the next step are the old ones
        const T4<T> o = f.bold[v];
        const T ox = now.x - o.x, oy = now.y - o.y, oz = now.z - o.z;
        moved = fmaxf(moved, fsqrt((float)(ox * ox + oy * oy + oz * oz)));
    }
    if (moved > limit) rt->hardStep[parity ^ 1] = f.step + 1;
}

// before a run of such steps: the lists of the robots whose lists are stale (their
// grid is built by the listing launch before)
template <typename T> __global__ __launch_bounds__(256) void k_list_begin(Dev<T> a, ListArgs<T> f, int R, int S, int parity) {
    __shared__ int sQueue[256 / kListLanes * kListQueue];
    const int i = blockIdx.x * blockDim.x + threadIdx.x, s = min(i / kListLanes, S - 1);
    if (i < 2) f.hard[i] = -i;
    for (int r = i; r < R; r += gridDim.x * blockDim.x) {  // no listing under way, no step of all pairs
        a.rt[r].listStep = -2 * kListSteps;
        a.rt[r].hardStep[0] = a.rt[r].hardStep[1] = -1;
    }
    if (!a.anyStale[parity]) return;
    const int v = a.surf[s], r = a.vrob[v];
    const bool live = i / kListLanes < S && a.rt[r].stale[parity] && !a.rt[r].diverged;
    if (__any(live)) col_list_group(a, s, v, live, sQueue + threadIdx.x / kListLanes * kListQueue);
}

// and after it: the listing flags of the other modes.  n: steps of the run, parity:
// of the step to come
template <typename T> __global__ __launch_bounds__(256) void k_list_end(Dev<T> a, ListArgs<T> f, int n, int parity) {
    const int r = blockIdx.x;
    RobotTime &rt = a.rt[r];
    const RobotParams &rp = a.rp[r];
    const int phase = n - 1 - rt.listStep;
    // a listing half way, lists that are out of date: listed again first
    if (threadIdx.x == 0 && rp.scount > 0 && (rt.hardStep[parity] == n || phase < kListSteps)) rt.stale[parity] = 1;
    if (r == 0 && threadIdx.x == 0) {
        a.anyStale[0] = a.anyStale[1] = 1;
        *f.hardHost = *f.hard;
    }
}

}  // namespace vx3mi
