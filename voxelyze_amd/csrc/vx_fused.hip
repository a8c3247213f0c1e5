/*
 * vx_fused.hip -- the FP64 step as one kernel per step, bit for bit the split step.
 *
 * CVoxelyze::doTimeStep (src/Voxelyze.cpp:251-284) updates every link, then every voxel.
 * The split step (vx_kernels.hip) does that with two kernels and hands each link's four
 * end vectors to its voxels through HBM (96 B per link written, then read).  Here one lane
 * per voxel evaluates the <= 6 links it touches with the split step's own link function
 * (every link is evaluated by both of its voxels, on identical inputs, so both get the
 * split step's bits), sums its end vectors in direction order 0..5 and integrates with the
 * split step's voxel function.  Nothing is handed over through HBM.
 *
 * Voxel state, voxel flags, link state and robot clocks are double-buffered: a step reads
 * "in" and writes "out", so no lane sees a neighbour's new state.  The link's negative
 * voxel owns it and writes its new state.  previousDt (VX_Voxel.cpp:163), read only by
 * links with a valid local velocity, is the robot's dt of the previous step.
 *
 * Divergence (a strain > 100, Voxelyze.cpp:265-269): every link of that step is updated
 * but the voxels and the clock must not move.  The lanes record the step in the robot's
 * rdiv entry and still write their (discarded) voxel output; from the next step on the
 * robot's lanes copy whichever ping-pong buffer is stale, so the robot ends the launch with
 * its voxels as before the diverging step and its links as after it.  The first of those
 * copies also saves the link state from before the diverging step, from which the host
 * recomputes that step's end forces after the launch (k_step_fp64<true, ...>).
 *
 * End forces (what CVX_Link::force() returns) are written to the split step's force slots
 * on the launch's last step only.
 *
 * Actuation: temperatures are double-buffered like the state.  A launch starts with k_fused_temps
 * (as k_actuate_fp64 sets them), and every step but the last writes its voxels' temperatures at the
 * robot's time after it, which the next step's rest lengths and contacts read: one correctly
 * rounded sine per voxel and step instead of one for each link end as well (a population of 48
 * robots, 74,400 voxels: 21.5 -> 18.1 ms for 200 steps).
 */
#include "vx_contact_force.h"
#include "vx_device.h"
#include "vx_math.h"
#include "vx_step_fp64.h"

#pragma clang fp contract(off)

namespace vx {

/* a robot that diverged at step d (or, d = -1, does not step in this launch) */
__device__ void frozen_fp64(const FusedPtrs& s, int i, int rob, int d) {
    const int nv = s.nv, nl = s.nl;
    const bool idle = d < 0;
    if (s.vpsOut) /* as the temperatures */
        for (int c = 0; c < 3; c++) {
            if (idle) s.vpsOut[c * nv + i] = s.vps[c * nv + i];
            else if (s.k == d + 1) s.vps[c * nv + i] = s.vpsOut[c * nv + i];
        }
    if (s.vphase) { /* both halves keep the temperatures of the last step that counted */
        if (idle) s.vtempOut[i] = s.vtempIn[i];
        else if (s.k == d + 1) s.vtempIn[i] = s.vtempOut[i];
    }
    if (idle || ((s.k - d) & 1) == 0) {
        for (int c = 0; c < VD_COUNT; c++) s.vdOut[c * nv + i] = s.vdIn[c * nv + i];
        s.vflOut[i] = s.vflIn[i];
        if (i == 0 || s.vrobot[i - 1] != rob) s.rtimeOut[rob] = s.rtimeIn[rob];
    }
    if (idle || ((s.k - d) & 1) == 1) {
        const bool save = !idle && s.k == d + 1; /* "out" still holds the links before step d */
        for (int axis = 0; axis < 3; axis++) {
            const int slot = axis * nv + i;
            for (int c = 0; c < LDEV_COUNT; c++) {
                if (save) s.ldSide[c * nl + slot] = s.ldOut[c * nl + slot];
                s.ldOut[c * nl + slot] = s.ldIn[c * nl + slot];
            }
            for (int c = 0; c < LF_COUNT; c++) {
                if (save) s.lfSide[c * nl + slot] = s.lfOut[c * nl + slot];
                s.lfOut[c * nl + slot] = s.lfIn[c * nl + slot];
            }
            if (save) s.lflSide[slot] = s.lflOut[slot];
            s.lflOut[slot] = s.lflIn[slot];
        }
    }
}

__device__ __forceinline__ double axis_size(const VoxMat& m, int axis) {
    return axis == 0 ? m.sizeX : axis == 1 ? m.sizeY : m.sizeZ;
}

/* what one end of a link reads: the neighbour's pose and material, the link's material and state */
struct LinkIn {
    int meta, mo;
    float to; /* the neighbour's temperature (read under actuation) */
    dvec po;
    dquat qo;
    double rest;
    LinkPrev old;
};
/* the loads of one link of voxel i (direction dir, neighbour o), those that wait for nothing but
   the slot first */
template <bool Neg, bool Poisson>
__device__ __forceinline__ void link_load(const FusedPtrs& s, int i, int o, int dir, LinkIn& in) {
    const int nv = s.nv, nl = s.nl;
    const double* __restrict__ vd = s.vdIn;
    const int slot = (dir >> 1) * nv + (Neg ? i : o);
    in.meta = s.lmeta[slot];
    in.old.flags = s.lflIn[slot];
    in.old.pos2 = dv(s.ldIn[LP2X * nl + slot], s.ldIn[LP2Y * nl + slot], s.ldIn[LP2Z * nl + slot]);
    in.old.a1 = dv(s.ldIn[LA1X * nl + slot], s.ldIn[LA1Y * nl + slot], s.ldIn[LA1Z * nl + slot]);
    in.old.a2 = dv(s.ldIn[LA2X * nl + slot], s.ldIn[LA2Y * nl + slot], s.ldIn[LA2Z * nl + slot]);
    in.old.maxStrain = s.lfIn[LMAXSTRAIN * nl + slot];
    in.old.strainOffset = s.lfIn[LOFFSET * nl + slot];
    if (Poisson) {
        in.old.tArea = s.lfIn[LTAREA * nl + slot];
        in.old.tss = s.lfIn[LTSS * nl + slot];
    }
    in.rest = s.ldIn[LREST * nl + slot];
    in.mo = s.vmat[o];
    if (s.vphase) in.to = s.vtempIn[o];
    in.po = dv(vd[VPX * nv + o], vd[VPY * nv + o], vd[VPZ * nv + o]);
    in.qo = dq(vd[VQW * nv + o], vd[VQX * nv + o], vd[VQY * nv + o], vd[VQZ * nv + o]);
}

/* one link of voxel i (direction dir, neighbour o, material mi) as CVX_Link::updateForces
   (VX_Link.cpp:149-217): its end vectors on voxel i (force f, moment mm), written to the force
   slot on the last step; the negative end (Neg) owns the link state.
   Poisson: some material has Poisson's ratio != 0 (the transverse info is read and kept) */
template <bool ForcesOnly, bool Neg, bool Poisson, bool Cached>
__device__ __forceinline__ void link_end(const FusedPtrs& s, LinkIn& in, int i, int o, int mi, int dir, int rob,
                                         float prevDt, float tempI, const dvec& pos0, const dquat& q0,
                                         dvec& f, dvec& mm, float& strain) {
    const int nv = s.nv, nl = s.nl;
    const int axis = dir >> 1;
    const int n = Neg ? i : o, p = Neg ? o : i;
    const int slot = axis * nv + n;
    const LinkMat m = s.lmats[in.meta];
    const VoxMat& mn = s.vmats[Neg ? mi : in.mo];
    const VoxMat& mp = s.vmats[Neg ? in.mo : mi];
    const dvec po = in.po;
    const dquat qo = in.qo;
    double rest = in.rest;
    if (s.vphase) { /* updateRestLength (VX_Link.cpp:137-140) at this step's temperatures */
        const float tempO = in.to;
        rest = 0.5 * (base_size(axis_size(mn, axis), Neg ? tempI : tempO, mn.alphaCTE) +
                      base_size(axis_size(mp, axis), Neg ? tempO : tempI, mp.alphaCTE));
    }
    LinkPrev old = in.old;
    if (Poisson) { /* volume effects (VX_Link.cpp:160) */
        link_transverse(m, mn, mp, s.vps, nv, n, p, axis, &old.tArea, &old.tss);
    } else {
        old.tArea = m.transverseArea;
        old.tss = 0.0f;
    }
    float dmN = 0.0f, dmP = 0.0f;
    if (old.flags & LF_LVV) { /* dampingMultiplier (VX_Voxel.h:130) of both voxels */
        dmN = mn.dampNum / prevDt;
        dmP = mp.dampNum / prevDt;
    }
    LinkEval e;
    link_eval_fp64<Poisson>(m, s.curveStrain + m.curveOff, s.curveStress + m.curveOff, axis, Neg ? pos0 : po,
                   Neg ? q0 : qo, Neg ? po : pos0, Neg ? qo : q0, rest, old, dmN, dmP, &e);
    strain = e.strain;
    f = Neg ? e.fN : e.fP;
    mm = Neg ? e.mN : e.mP;
    if (s.storeForces) {
        double* slotF = s.vf + vf_index(dir, 0, nv, i);
        slotF[0] = f.x; slotF[1] = f.y; slotF[2] = f.z;
        slotF[3] = mm.x; slotF[4] = mm.y; slotF[5] = mm.z;
    }
    if (!ForcesOnly && Neg) {
        double* ld = s.ldOut;
        put<Cached>(&ld[LP2X * nl + slot], e.pos2.x); put<Cached>(&ld[LP2Y * nl + slot], e.pos2.y);
        put<Cached>(&ld[LP2Z * nl + slot], e.pos2.z);
        put<Cached>(&ld[LA1X * nl + slot], e.a1v.x); put<Cached>(&ld[LA1Y * nl + slot], e.a1v.y);
        put<Cached>(&ld[LA1Z * nl + slot], e.a1v.z);
        put<Cached>(&ld[LA2X * nl + slot], e.a2v.x); put<Cached>(&ld[LA2Y * nl + slot], e.a2v.y);
        put<Cached>(&ld[LA2Z * nl + slot], e.a2v.z);
        if (!s.restConst) put<Cached>(&ld[LREST * nl + slot], rest);
        float* lf = s.lfOut;
        put<Cached>(&lf[LSTRAIN * nl + slot], e.strain);
        put<Cached>(&lf[LMAXSTRAIN * nl + slot], e.maxStrain);
        if (!s.offsetConst) put<Cached>(&lf[LOFFSET * nl + slot], e.strainOffset);
        put<Cached>(&lf[LSTRESS * nl + slot], e.stress);
        if (Poisson) {
            lf[LTAREA * nl + slot] = old.tArea;
            lf[LTSS * nl + slot] = old.tss;
        }
        put<Cached>(&s.lflOut[slot], e.flags);
        if (e.strain > 100) {
            atomicMin(&s.rdiv[rob], s.k);
            atomicOr(&s.ctl[0], 1);
        }
    }
}

#ifndef VX_FUSED64_WAVES
#define VX_FUSED64_WAVES 3
#endif
/* ForcesOnly: after a launch, the end forces of the step in which a robot diverged, for the
   robots that diverged before the launch's last step (k is that step); "in" is the voxel
   state (as before the diverging step) and the saved link state.  Poisson: s.poisson, as a
   compile-time switch */
/* The voxel and link material tables staged in LDS by every workgroup (when they fit these
   sizes): each lane reads its materials' constants (about 20 words per link end) from LDS
   instead of gathering them through the vector caches. On the drop lattice 255 -> 248 us per
   step, on the porous block 67 -> 66 us, the same bits. */
#ifndef VX_MATS_LDS
#define VX_MATS_LDS 1
#endif
constexpr int kLdsVoxMats = 32, kLdsLinkMats = 64;
__device__ __forceinline__ void stage_materials(const FusedPtrs& s, VoxMat* svm, LinkMat* slm) {
    const int nv32 = s.nvmats * (int)(sizeof(VoxMat) / 4), nl32 = s.nlmats * (int)(sizeof(LinkMat) / 4);
    for (int t = threadIdx.x; t < nv32; t += blockDim.x) ((uint32_t*)svm)[t] = ((const uint32_t*)s.vmats)[t];
    for (int t = threadIdx.x; t < nl32; t += blockDim.x) ((uint32_t*)slm)[t] = ((const uint32_t*)s.lmats)[t];
    __syncthreads();
}

/* voxel i's temperature for the next step, at its robot's time after this one */
__device__ __forceinline__ void next_temperature(const FusedPtrs& s, int i, int rob, float dt) {
    if (s.vphase && s.tempNext)
        s.vtempOut[i] = actuation_temperature(s.actBase, s.actAmp, s.actFreq, s.rtimeIn[rob] + dt, s.vphase[i]);
}

/* contacts in partner order (VX_Voxel.cpp:250-253), each pair's force from voxel i's side as the
   split step's contact kernel forms it */
__device__ __forceinline__ void subtract_contacts(const FusedPtrs& s, const VoxMat& m, int i, float tempI, dvec& t) {
    if (!s.colCnt) return;
    const int nv = s.nv;
    const int cnt = s.colCnt[i], off = s.colOff[i];
    if (cnt == 0) return;
    const ContactSelf me = contact_self(m, s.vdIn, nv, i, tempI);
    for (int c = 0; c < cnt; c++) {
        const int j = s.partners[off + c];
        const fvec f = contact_pair_force(me, s.vmats[s.vmat[j]], s.vdIn, nv, j, s.vtempIn[j]);
        t.x -= f.x; t.y -= f.y; t.z -= f.z;
    }
}

/* Driven: instances for contact-batch steps (the watch-list test on the positions written),
   prescribed-displacement ramps and actuation; the others carry none of them, nor their registers. */
template <bool ForcesOnly, bool Poisson, bool MatsLds, bool Driven>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(VX_FUSED64_WAVES, 8))) k_step_fp64(FusedPtrs s0) {
    FusedPtrs s = s0;
    if (!Driven && !ForcesOnly) s.vphase = nullptr;
    if (MatsLds) {
        __shared__ VoxMat svm[kLdsVoxMats];
        __shared__ LinkMat slm[kLdsLinkMats];
        stage_materials(s0, svm, slm);
        s.vmats = svm;
        s.lmats = slm;
    }
    const int i = lane_index(s.xcd);
    const int nv = s.nv, nl = s.nl;
    if (i >= nv) return;
    if (!ForcesOnly && s.halt && s.halt[0] <= s.k) return; /* a contact batch halted before this step */
    const int rob = s.vrobot[i];
    const int d = s.rdiv[rob];
    const float dt = s.rdt[rob];
    float prevDt;
    if (ForcesOnly) {
        if (d < 0 || d >= s.k) return;
        prevDt = d == 0 ? s.rprev[rob] : dt;
    } else {
        if (d < s.k) {
            frozen_fp64(s, i, rob, d);
            if (Driven && s.haltTest)
                halt_if_stale(s.halt, s.k + 1, s.colLast, s.recalcSq, s.vflIn, nv, i, s.vdOut[VPX * nv + i],
                              s.vdOut[VPY * nv + i], s.vdOut[VPZ * nv + i]);
            return;
        }
        prevDt = s.k == 0 ? s.rprev[rob] : dt;
        next_temperature(s, i, rob, dt);
        if (i == 0 || s.vrobot[i - 1] != rob) s.rtimeOut[rob] = s.rtimeIn[rob] + dt; /* currentTime += dt */
        /* here, before the link loop, where few registers are live; read back further down */
        if (Driven) apply_ramp(s.exts, s.ramps, s.vext[i], s.rtimeIn[rob]);
    }
    const double* __restrict__ vd = s.vdIn;
    const dvec pos0 = dv(vd[VPX * nv + i], vd[VPY * nv + i], vd[VPZ * nv + i]);
    const dquat q0 = dq(vd[VQW * nv + i], vd[VQX * nv + i], vd[VQY * nv + i], vd[VQZ * nv + i]);
    const int mi = s.vmat[i];
    const float tempI = s.vtempIn[i];

    /* force() and moment() (VX_Voxel.cpp:234-271): the end vectors of the links in direction
       order 0..5, each link evaluated as CVX_Link::updateForces (VX_Link.cpp:149-217) */
    dvec sf = dv(0.0, 0.0, 0.0), sm = dv(0.0, 0.0, 0.0);
#pragma unroll 1
    for (int dir = 0; dir < 6; dir++) {
        const int o = s.vnbr[dir * nv + i];
        if (o < 0) {
            if (s.storeForces)
                for (int c = 0; c < 6; c++) s.vf[vf_index(dir, c, nv, i)] = 0.0;
            continue;
        }
        /* the two ends as separate instances, each computing only its own end vectors */
        dvec f, mm;
        float strain;
        LinkIn in;
        if ((dir & 1) == 0) {
            link_load<true, Poisson>(s, i, o, dir, in);
            link_end<ForcesOnly, true, Poisson, false>(s, in, i, o, mi, dir, rob, prevDt, tempI, pos0, q0, f, mm, strain);
        } else {
            link_load<false, Poisson>(s, i, o, dir, in);
            link_end<ForcesOnly, false, Poisson, false>(s, in, i, o, mi, dir, rob, prevDt, tempI, pos0, q0, f, mm, strain);
        }
        sf.x += f.x; sf.y += f.y; sf.z += f.z;
        sm.x += mm.x; sm.y += mm.y; sm.z += mm.z;
    }
    if (ForcesOnly) return;
    /* the voxel's index through an opaque copy: its addresses are formed here, after the link
       loop, instead of being kept live (and spilled) across it */
    int iv = i;
    __asm__ volatile("" : "+v"(iv));

    /* CVX_Voxel::timeStep (VX_Voxel.cpp:162-232) */
    const VoxMat m = s.vmats[mi];
    const int e = s.vext[iv];
    const ExtRec* ex = e >= 0 ? &s.exts[e] : nullptr;
    uint32_t flags = s.vflIn[iv];
    if (ex && (ex->dof & 0x3F) == 0x3F) {
        voxel_pinned(m, ex, s.vijk, nv, iv, s.vdOut);
        s.vflOut[iv] = flags;
        if (Driven && s.haltTest)
            halt_if_stale(s.halt, s.k + 1, s.colLast, s.recalcSq, s.vflIn, nv, iv, s.vdOut[VPX * nv + iv],
                          s.vdOut[VPY * nv + iv], s.vdOut[VPZ * nv + iv]);
        return;
    }
    /* the momenta only this lane reads: loaded past the caches */
    dvec pos = pos0, lin = dv(ld_nt(&vd[VLX * nv + iv]), ld_nt(&vd[VLY * nv + iv]), ld_nt(&vd[VLZ * nv + iv]));
    dvec ang = dv(ld_nt(&vd[VAX * nv + iv]), ld_nt(&vd[VAY * nv + iv]), ld_nt(&vd[VAZ * nv + iv]));
    dquat q = q0;
    voxel_step_fp64(m, ex, s.vijk, nv, iv, dt, tempI, sf, sm, pos, lin, ang, q, flags,
                    [&](dvec& t) { subtract_contacts(s, m, iv, tempI, t); });
    store_voxel(s.vdOut, nv, iv, pos, lin, ang, q);
    st_nt(&s.vflOut[iv], flags & ~(uint32_t)VF_PS_VALID); /* poissonsStrainInvalid = true (VX_Voxel.cpp:231) */
    if (Driven && s.haltTest) halt_if_stale(s.halt, s.k + 1, s.colLast, s.recalcSq, s.vflIn, nv, iv, pos.x, pos.y, pos.z);
}

/* The same step for models that do not fill the chip: a workgroup takes 64 voxels and splits
   their link directions over its waves, PerWave directions to a wave, so a voxel's <= 6 links run
   side by side instead of one after the other; the end vectors meet in LDS (18 KB), where wave 0
   sums the forces in direction order and integrates the translations while wave 1 does the same
   with the moments and rotations.  Each link end is evaluated by link_end on the same inputs and
   the sums keep their order (an absent link adds +0.0), so the bits are k_step_fp64's.
   With a Poisson's ratio, wave 2 forms the voxel's Poisson strain for the next step from the
   strains its links just took, which k_poisson_fp64 otherwise does in a launch before every step
   (8,385 voxels: 15.2 us a step with that launch, 9.3 without).

   What bounds it: the chain of dependent loads and FP64 operations of one link (2.7 us of the 5 us
   a workgroup lives; 2.5 us more pass between two launches), which k_step_fp64 walks through six
   times over.  us per step of a two-material lattice, k_step_fp64 at its best launch shape -> here:
   290 voxels 14.7 -> 6.6; 7,169 15.5 -> 6.7; 15,784 15.9 -> 7.3 (PerWave 1: six waves with 185
   VGPRs, two a SIMD, everything a lane reads asked for up front);
   17,676 16.9 -> 10.1; 45,352 19.4 -> 13.8; 112,451 29.9 -> 26.8; 235,932 59.9 -> 48.8 (PerWave 2:
   three waves at three a SIMD; PerWave 1 takes 12.2 at 24,286 voxels where PerWave 2 takes 10.4,
   since a second workgroup of six waves no longer finds room beside the first).
   The blocks map to the XCDs in contiguous ranges and the stores go through the caches, so that
   the next step finds a tile's state, and most of its neighbours', in the same L2 (45,352 voxels:
   15.9 linear and non-temporal, 15.0 contiguous, 13.8 contiguous and cached). */
template <int PerWave, bool Poisson, bool MatsLds, bool Driven>
__global__ void __launch_bounds__(6 / PerWave * kEndsTile) __attribute__((amdgpu_waves_per_eu(PerWave == 1 ? 2 : 3, 8))) k_step_fp64_ends(FusedPtrs s0) {
    FusedPtrs s = s0;
    if (!Driven) s.vphase = nullptr;
    const int nv = s.nv;
    if (s.halt && s.halt[0] <= s.k) return; /* the whole grid: a halt recorded by this step is k + 1 */
    const int lane = threadIdx.x & (kEndsTile - 1);
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x / kEndsTile);
    const int at = xcd_block() * kEndsTile + lane;
    const double* __restrict__ vd = s.vdIn;
    __shared__ double ends[6][6][kEndsTile];
    __shared__ float strains[6][Poisson ? kEndsTile : 1]; /* at the voxel's ends */
    __shared__ VoxMat svm[MatsLds ? kLdsVoxMats : 1];
    __shared__ LinkMat slm[MatsLds ? kLdsLinkMats : 1];
    const int c0 = 3 * wave; /* wave 0 integrates the translations, wave 1 the rotations */
    int i = at, rob = 0, mi = 0, o = -1, ei = -1, d = 0;
    float dt = 0.0f, tnow = 0.0f, tempI = 0.0f;
    uint32_t flags = 0;
    dvec pos0, mom = dv(0.0, 0.0, 0.0);
    dquat q0;
    bool live;
    if (PerWave == 1) {
        /* what a lane reads is asked for at once, before the material tables' barrier and the
           test of its robot (a lane past the end reads the last voxel's) */
        i = at < nv ? at : nv - 1;
        o = s.vnbr[wave * nv + i];
        rob = s.vrobot[i];
        mi = s.vmat[i];
        pos0 = dv(vd[VPX * nv + i], vd[VPY * nv + i], vd[VPZ * nv + i]);
        q0 = dq(vd[VQW * nv + i], vd[VQX * nv + i], vd[VQY * nv + i], vd[VQZ * nv + i]);
        tempI = s.vtempIn[i];
        if (wave < 2) {
            mom = dv(vd[(VLX + c0) * nv + i], vd[(VLY + c0) * nv + i], vd[(VLZ + c0) * nv + i]);
            ei = s.vext[i];
            flags = s.vflIn[i];
        }
    }
    if (MatsLds) {
        stage_materials(s0, svm, slm);
        s.vmats = svm;
        s.lmats = slm;
    }
    if (PerWave == 1) {
        d = s.rdiv[rob];
        dt = s.rdt[rob];
        tnow = s.rtimeIn[rob];
        live = at < nv && d >= s.k;
    } else {
        live = at < nv;
        if (live) {
            rob = s.vrobot[i];
            d = s.rdiv[rob];
            live = d >= s.k;
        }
    }
    if (at < nv && !live && wave == 0) {
        frozen_fp64(s, i, rob, d);
        if (Driven && s.haltTest)
            halt_if_stale(s.halt, s.k + 1, s.colLast, s.recalcSq, s.vflIn, nv, i, s.vdOut[VPX * nv + i],
                          s.vdOut[VPY * nv + i], s.vdOut[VPZ * nv + i]);
    }
    if (live) {
        if (PerWave > 1) {
            mi = s.vmat[i];
            pos0 = dv(vd[VPX * nv + i], vd[VPY * nv + i], vd[VPZ * nv + i]);
            q0 = dq(vd[VQW * nv + i], vd[VQX * nv + i], vd[VQY * nv + i], vd[VQZ * nv + i]);
            tempI = s.vtempIn[i];
            dt = s.rdt[rob];
            tnow = s.rtimeIn[rob];
        }
        const float prevDt = s.k == 0 ? s.rprev[rob] : dt;
#pragma unroll 1
        for (int dir = PerWave * wave; dir < PerWave * (wave + 1); dir++) {
            if (PerWave > 1) o = s.vnbr[dir * nv + i];
            dvec f = dv(0.0, 0.0, 0.0), mm = dv(0.0, 0.0, 0.0);
            float strain = 0.0f;
            if (o >= 0) {
                LinkIn in;
                if ((dir & 1) == 0) {
                    link_load<true, Poisson>(s, i, o, dir, in);
                    link_end<false, true, Poisson, true>(s, in, i, o, mi, dir, rob, prevDt, tempI, pos0, q0, f, mm, strain);
                } else {
                    link_load<false, Poisson>(s, i, o, dir, in);
                    link_end<false, false, Poisson, true>(s, in, i, o, mi, dir, rob, prevDt, tempI, pos0, q0, f, mm, strain);
                }
            } else if (s.storeForces) {
                for (int c = 0; c < 6; c++) s.vf[vf_index(dir, c, nv, i)] = 0.0;
            }
            ends[dir][0][lane] = f.x; ends[dir][1][lane] = f.y; ends[dir][2][lane] = f.z;
            ends[dir][3][lane] = mm.x; ends[dir][4][lane] = mm.y; ends[dir][5][lane] = mm.z;
            if (Poisson && o >= 0 && s.psNext)
                strains[dir][lane] = axial_strain_end(strain, s.lratio[(dir >> 1) * nv + ((dir & 1) ? o : i)], (dir & 1) != 0);
        }
    }
    __syncthreads();
    if (!live) return;
    if (wave == 2) next_temperature(s, i, rob, dt);
    if (Poisson && wave == 2 && s.psNext) {
        /* the next step's Poisson strain (a voxel that k_poisson_fp64 would leave keeps its own) */
        const VoxMat& m = s.vmats[mi];
        const uint32_t fl = s.vflIn[i];
        const int e = s.vext[i];
        const ExtRec* ex = e >= 0 ? &s.exts[e] : nullptr;
        float ps[3];
        if (m.nu != 0.0f && (fl & (0x3Fu * VF_LINK0)) && !(ex && (ex->dof & 0x3F) == 0x3F))
            poisson_strain(m, ex, fl, [&](int dir) { return strains[dir][lane]; }, ps);
        else
            for (int c = 0; c < 3; c++) ps[c] = s.vps[c * nv + i];
        for (int c = 0; c < 3; c++) s.vpsOut[c * nv + i] = ps[c];
    }
    if (wave > 1) return;
    if (PerWave > 1) {
        mom = dv(vd[(VLX + c0) * nv + i], vd[(VLY + c0) * nv + i], vd[(VLZ + c0) * nv + i]);
        ei = s.vext[i];
        flags = s.vflIn[i];
    }

    /* CVX_Voxel::timeStep (VX_Voxel.cpp:162-232): translation in wave 0, rotation in wave 1 */
    const VoxMat m = s.vmats[mi];
    const ExtRec* ex = ei >= 0 ? &s.exts[ei] : nullptr;
    const bool pinned = ex && (ex->dof & 0x3F) == 0x3F;
    dvec sum = dv(0.0, 0.0, 0.0);
    for (int e = 0; e < 6; e++) {
        sum.x += ends[e][c0][lane]; sum.y += ends[e][c0 + 1][lane]; sum.z += ends[e][c0 + 2][lane];
    }
    double* __restrict__ out = s.vdOut;
    if (wave == 1) {
        if (pinned) return;
        dvec ang = mom;
        dquat q = q0;
        voxel_rotate_fp64(m, ex, dt, sum, ang, q);
        if (ex) voxel_fix_rotation(ex, ang, q);
        out[VAX * nv + i] = ang.x; out[VAY * nv + i] = ang.y; out[VAZ * nv + i] = ang.z;
        out[VQW * nv + i] = q.w; out[VQX * nv + i] = q.x; out[VQY * nv + i] = q.y; out[VQZ * nv + i] = q.z;
        return;
    }
    if (i == 0 || s.vrobot[i - 1] != rob) s.rtimeOut[rob] = tnow + dt; /* currentTime += dt */
    if (Driven) apply_ramp(s.exts, s.ramps, ei, tnow);
    if (pinned) {
        voxel_pinned(m, ex, s.vijk, nv, i, out);
        s.vflOut[i] = flags;
        if (Driven && s.haltTest)
            halt_if_stale(s.halt, s.k + 1, s.colLast, s.recalcSq, s.vflIn, nv, i, out[VPX * nv + i], out[VPY * nv + i],
                          out[VPZ * nv + i]);
        return;
    }
    dvec pos = pos0, lin = mom;
    voxel_translate_fp64(m, ex, dt, tempI, sum, q0, pos, lin, flags,
                         [&](dvec& t) { subtract_contacts(s, m, i, tempI, t); });
    if (ex) voxel_fix_translation(m, ex, s.vijk, nv, i, pos, lin);
    out[VPX * nv + i] = pos.x; out[VPY * nv + i] = pos.y; out[VPZ * nv + i] = pos.z;
    out[VLX * nv + i] = lin.x; out[VLY * nv + i] = lin.y; out[VLZ * nv + i] = lin.z;
    /* poissonsStrainInvalid = true (VX_Voxel.cpp:231); the next step's strain is valid again */
    const bool psValid = Poisson && s.psNext && m.nu != 0.0f && (flags & (0x3Fu * VF_LINK0));
    s.vflOut[i] = psValid ? flags | VF_PS_VALID : flags & ~(uint32_t)VF_PS_VALID;
    if (Driven && s.haltTest) halt_if_stale(s.halt, s.k + 1, s.colLast, s.recalcSq, s.vflIn, nv, i, pos.x, pos.y, pos.z);
}

/* temperatures at each robot's current time, before the first step of an actuated launch (robots
   that do not step keep theirs, which the other half holds if `moved`) */
__global__ void __launch_bounds__(256) k_fused_temps(FusedPtrs s, int moved) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= s.nv) return;
    const int rob = s.vrobot[i];
    if (s.rdiv[rob] < 0) {
        if (moved) s.vtempIn[i] = s.vtempOut[i];
        return;
    }
    s.vtempIn[i] = actuation_temperature(s.actBase, s.actAmp, s.actFreq, s.rtimeIn[rob], s.vphase[i]);
}

/* a robot that diverged in the launch's last step takes back its voxels (and clock, and for
   the mixed step its temperatures) from before that step, which the other ping-pong buffer
   holds */
__global__ void __launch_bounds__(256) k_fused_restore(double* vd, const double* vdPrev, uint32_t* vfl,
                                                      const uint32_t* vflPrev, float* vtemp, const float* vtempPrev,
                                                      float* rtime, const float* rtimePrev, int nv, int first,
                                                      int count, int rob) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= count) return;
    const int i = first + t;
    for (int c = 0; c < VD_COUNT; c++) vd[c * nv + i] = vdPrev[c * nv + i];
    vfl[i] = vflPrev[i];
    if (vtemp) vtemp[i] = vtempPrev[i];
    if (t == 0) rtime[rob] = rtimePrev[rob];
}

void launch_step_fp64(const FusedPtrs& s, int block, bool forcesOnly, hipStream_t st) {
    if (s.nv <= 0) return;
    const dim3 grid((unsigned)((s.nv + block - 1) / block));
    const bool lds = VX_MATS_LDS && !forcesOnly && s.nvmats <= kLdsVoxMats && s.nlmats <= kLdsLinkMats;
    const bool driven = s.haltTest || s.ramps || s.vphase;
    if (forcesOnly) {
        if (s.poisson) hipLaunchKernelGGL((k_step_fp64<true, true, false, false>), grid, dim3(block), 0, st, s);
        else hipLaunchKernelGGL((k_step_fp64<true, false, false, false>), grid, dim3(block), 0, st, s);
        return;
    }
#define VX_STEP64(P, L)                                                                                  \
    if (driven) hipLaunchKernelGGL((k_step_fp64<false, P, L, true>), grid, dim3(block), 0, st, s);      \
    else hipLaunchKernelGGL((k_step_fp64<false, P, L, false>), grid, dim3(block), 0, st, s)
    if (s.poisson) {
        if (lds) { VX_STEP64(true, true); }
        else { VX_STEP64(true, false); }
    } else {
        if (lds) { VX_STEP64(false, true); }
        else { VX_STEP64(false, false); }
    }
#undef VX_STEP64
}
void launch_step_fp64_ends(const FusedPtrs& s, hipStream_t st) {
    if (s.nv <= 0) return;
    const int perWave = s.nv <= kEndsWideMax ? 1 : 2;
    const dim3 grid((unsigned)((s.nv + kEndsTile - 1) / kEndsTile)), block(6 / perWave * kEndsTile);
    const bool lds = VX_MATS_LDS && s.nvmats <= kLdsVoxMats && s.nlmats <= kLdsLinkMats;
    const bool driven = s.haltTest || s.ramps || s.vphase;
#define VX_ENDS64(W, P, L)                                                                                \
    if (driven) hipLaunchKernelGGL((k_step_fp64_ends<W, P, L, true>), grid, block, 0, st, s);            \
    else hipLaunchKernelGGL((k_step_fp64_ends<W, P, L, false>), grid, block, 0, st, s)
#define VX_ENDS64_W(W)                                                                                    \
    if (s.poisson) {                                                                                      \
        if (lds) { VX_ENDS64(W, true, true); }                                                            \
        else { VX_ENDS64(W, true, false); }                                                               \
    } else {                                                                                              \
        if (lds) { VX_ENDS64(W, false, true); }                                                           \
        else { VX_ENDS64(W, false, false); }                                                              \
    }
    if (perWave == 1) { VX_ENDS64_W(1) }
    else { VX_ENDS64_W(2) }
#undef VX_ENDS64_W
#undef VX_ENDS64
}
void launch_fused_temps(const FusedPtrs& s, bool moved, hipStream_t st) {
    if (s.nv > 0)
        hipLaunchKernelGGL(k_fused_temps, dim3((unsigned)((s.nv + 255) / 256)), dim3(256), 0, st, s, moved ? 1 : 0);
}
void launch_fused_restore(double* vd, const double* vdPrev, uint32_t* vfl, const uint32_t* vflPrev, float* vtemp,
                          const float* vtempPrev, float* rtime, const float* rtimePrev, int nv, int first, int count,
                          int rob, hipStream_t st) {
    if (count > 0)
        hipLaunchKernelGGL(k_fused_restore, dim3((unsigned)((count + 255) / 256)), dim3(256), 0, st, vd, vdPrev, vfl,
                           vflPrev, vtemp, vtempPrev, rtime, rtimePrev, nv, first, count, rob);
}

}  // namespace vx
