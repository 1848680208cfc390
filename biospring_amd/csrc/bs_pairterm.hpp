// bs_pairterm.hpp -- one non-bonded pair as the pair kernels and the step
// kernel evaluate it.
#pragma once

#include "bs_device.hpp"

namespace bs
{

namespace
{

constexpr int WAVES = BLOCK / 64;

__device__ inline int32_t lanes_below(uint64_t b)
{
    return (int32_t)__builtin_amdgcn_mbcnt_hi((uint32_t)(b >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)b, 0u));
}

// ---------------------------------------------------------------------------
// One pair from i's side.  Energies are weighted 1/2 for a dynamic partner
// and 1 for a static one (Particle.cpp:231-249).  Formulas: energy/steric.hpp,
// electrostatic.hpp, hydrophobic.hpp; per-bead sqrt(r), sqrt(eps) for the
// Lorentz-Berthelot / Good-Hope modes (CombinationRules.hpp:18-31).  The
// force is accumulated in FP64 (same rate as FP32 on CDNA4), which keeps
// small net forces accurate when many pair terms cancel.
//
// Branch-free: every lane evaluates the terms with a safe distance and the
// results are selected by the pair's predicates.  Across a wave the pairs are
// half inside the cutoff at best, so branching would not skip work; it only
// costs exec-mask bookkeeping and keeps loads from being issued early.  The
// exact two-stage test runs for pairs in the guard band around rc^2 only.
//
// The kernel is bound by VALU issue, so the per-pair instruction count is
// what is minimised: the force prefactors carry C_spring, the term scales
// and i's own factor (PairI, formed once per lane); the pair predicates gate
// FP32 values (one select each) instead of FP64 results; a charge that is
// zero, or a pair gated off, zeroes the Coulomb term through q_j.
// ---------------------------------------------------------------------------
struct PairI
{
    float ks;  // steric force: C_spring x scale x {12 eps_i', 24 eps_i', eps_i} (Amber, Lewitt, Zacharias), C_spring x scale (linear)
    float kh;  // hydrophobic force: scale x C_spring x h_i
    double qe; // Coulomb energy: q_i ke
    double qf; // Coulomb force: q_i kf, doubled for eps(r) = eps r
};

// An FP32 value kept as computed: a select of it stays one FP32 select
// instead of being sunk past a later FP64 conversion (two selects).
__device__ inline float keep(float x)
{
    asm("" : "+v"(x));
    return x;
}

template <int SMODE, int EMODE>
__device__ inline PairI pair_i(float4 pi, float4 ri, const PairArgs &a)
{
    PairI c;
    const float cs = (float)a.k.c_spring;
    const float m = SMODE == 1 ? 12.0f : SMODE == 2 ? 24.0f : 1.0f;
    c.ks = SMODE == 0 ? cs * a.steric_scale : m * cs * a.steric_scale * ri.y;
    c.kh = a.hydro_scale * cs * ri.z;
    c.qe = (double)pi.w * a.ke;
    c.qf = (double)pi.w * a.kf * (EMODE == 2 ? 2.0 : 1.0);
    return c;
}

template <int SMODE, int EMODE, int HYDRO, bool ENERGY>
__device__ inline void interact(bool masked, float4 pi, float4 ri, float4 pj, float4 rj, const PairArgs &a,
                                const PairI &c, double &fx, double &fy, double &fz, double &es, double &ee,
                                double &eh)
{
    const float dx = pj.x - pi.x, dy = pj.y - pi.y, dz = pj.z - pi.z;
    const double xd = dx, yd = dy, zd = dz;
    // r^2 in FP64 where the Coulomb term needs it; the FP32 value is its
    // rounding there
    double r2d = 0.0;
    float r2;
    if (EMODE > 0)
    {
        r2d = fma(xd, xd, fma(yd, yd, zd * zd));
        r2 = (float)r2d;
    }
    else
        r2 = dx * dx + dy * dy + dz * dz;
    constexpr bool POWER = SMODE > 0; // power-law sterics: none below 0.1 A (steric.hpp:62)
    const bool inside = r2 < a.rc2lo;
    bool on = masked && inside, fon = on, qon = on; // pair inside the cutoff; its power-law and Coulomb terms
    // rare: within the guard band of the cutoff (decide exactly), or closer
    // than the terms' floors
    if (masked && (r2 < 0.01f || (!inside && r2 < a.rc2hi)))
    {
        if (!inside)
            on = exact_two_stage(pi, pj, a.rc);
        fon = on && r2 >= 0.01f;
        qon = on && r2 >= 1.0e-6f;
    }
    const bool pos2 = r2 > 0.0f;
    const float r2s = pos2 ? r2 : 1.0f;
    // the distance itself is needed by the vacuum Coulomb term, the linear
    // steric wall and the hydrophobic term; the others need 1/r^2 only
    constexpr bool NEED_D = EMODE == 1 || SMODE == 0 || HYDRO != 0;
    float inv = 0.0f, inv2;
    double invd = 0.0, i2d = 0.0;
    if (EMODE > 0)
    {
        // 1/d or 1/r^2 to ~1e-13: the FP32 seed (its input kept at or above
        // the smallest normal float, so it is finite) and one FP64 Newton
        // step on the exact r^2 of the float components.  The FP32 values of
        // the other terms are its rounding.
        const float seed = fmaxf(r2, 1.1754944e-38f);
        if (NEED_D)
        {
            const double y = (double)__builtin_amdgcn_rsqf(seed);
            invd = y * fma(-0.5 * r2d, y * y, 1.5);
            i2d = invd * invd;
            inv = (float)invd;
            inv2 = inv * inv;
        }
        else
        {
            const double y = (double)__builtin_amdgcn_rcpf(seed);
            i2d = y * fma(-r2d, y, 2.0);
            inv2 = (float)i2d;
        }
    }
    else
    {
        inv = __builtin_amdgcn_rsqf(r2s);
        inv = inv * (1.5f - 0.5f * r2s * inv * inv);
        inv2 = inv * inv;
    }
    const uint32_t flj = fbits(rj.w);
    const float wgt = (flj & PF_STATIC) ? 1.0f : 0.5f;
    float fs = 0.0f; // FP32 terms of the force scalar: force on i = (dx, dy, dz) * (fs + fsd)
    if (SMODE == 0)
    { // linear: ri + rj from raw radii; a coincident pair has energy, no force
        const float sr = ri.x + rj.x;
        const float d = r2s * inv;
        const float dv = pos2 ? d - sr : -sr;
        const bool ov = !(dv > 0.0f);
        if (ENERGY)
            es += on ? (double)(wgt * a.steric_scale * (ov ? 0.5f * dv * dv : 0.0f)) : 0.0;
        fs = (on && ov && pos2) ? dv * c.ks * inv : 0.0f; // -|dv| * C / d
    }
    else if (POWER)
    {
        // the factors' product is R^2 (jprm_of)
        const float s2 = ri.x * (rj.x * inv2), s6 = s2 * s2 * s2;
        float g, e0 = 0.0f;
        if (SMODE == 1)
        { // Amber 12-6: F = 12 eps (s6 - s12) / r^2, E = eps (s12 - 2 s6)
            g = fmaf(-s6, s6, s6);
            if (ENERGY)
                e0 = ri.y * rj.y * (s6 * s6 - 2.0f * s6);
        }
        else if (SMODE == 2)
        { // Lewitt 8-6: F = 24 eps (s6 - s8) / r^2, E = eps (3 s8 - 4 s6)
            const float s8 = s6 * s2;
            g = s6 - s8;
            if (ENERGY)
                e0 = ri.y * rj.y * (3.0f * s8 - 4.0f * s6);
        }
        else
        { // Zacharias 8-6: raw r, eps, product rules
            const float s8 = s6 * s2;
            g = 6.0f * s6 - 8.0f * s8;
            if (ENERGY)
                e0 = ri.y * rj.y * (s8 - s6);
        }
        if (ENERGY)
            es += fon ? (double)(wgt * a.steric_scale * e0) : 0.0;
        fs = fon ? c.ks * rj.y * g * inv2 : 0.0f;
    }
    double fsd = 0.0;
    if (EMODE > 0)
    {
        // Coulomb dominates the non-bonded force: its scalar is formed in FP64
        const double qj = (double)keep(qon ? pj.w : 0.0f);
        if (EMODE == 1)
        {
            if (ENERGY)
                ee += (double)wgt * c.qe * qj * invd;
            fsd = -(c.qf * qj) * (i2d * invd);
        }
        else
        { // eps(r) = eps * r
            if (ENERGY)
                ee += (double)wgt * c.qe * qj * i2d;
            fsd = -(c.qf * qj) * (i2d * i2d);
        }
    }
    if (HYDRO)
    {
        // h_i h_j vanishes unless both are hydrophobic
        const float e = __expf(-(r2s * inv));
        if (ENERGY)
        {
            const float hh = pos2 ? ri.z * rj.z * e : 0.0f;
            eh += on ? (double)(wgt * a.hydro_scale) * (-(double)hh * 6.02214169E23 * 1.0E-3) : 0.0;
        }
        fs += (on && pos2) ? c.kh * rj.z * e * inv : 0.0f;
    }
    const double s = EMODE > 0 ? fsd + (double)keep(fs) : (double)fs;
    fx = fma(xd, s, fx);
    fy = fma(yd, s, fy);
    fz = fma(zd, s, fz);
}

// ---------------------------------------------------------------------------
// Queue layout (BS_PAIR_QUEUES).  A wave takes its cluster's list 64 words at
// a time.  Each word's j data is loaded once (one lane per word) into an LDS
// ring of the last QSTRETCH stretches, and each of the 8 cluster particles
// has an LDS queue of the ring's words it sees (one ballot per particle and
// stretch).  The 8 lanes of a particle drain its queue, 8 entries per round,
// so the lanes evaluate listed pairs instead of idling on entries their
// particle does not see (an entry is seen by about half of a cluster's
// particles when springs empty the inner shell).
//
// A stretch takes as many rounds as keep every lane busy, and at least those
// that drain the oldest stretch in the ring, whose place the next one takes;
// what the longer queues hold beyond that waits for the next stretch.  The
// imbalance of a single stretch (a slab of the cluster's surroundings, which
// the particles see unevenly) mostly cancels over three: 84 % useful lanes in
// an emulation of dense networks, against 69 % when every 128 words are
// drained to the end.  Which particles see which words, and so the rounds of
// each stretch, follow from the list alone: the list build plans them
// (QPlan, queue_plan) and the walk reads the plan through the scalar cache.
//
// Each lane sums a fixed subset of its particle's entries in a fixed order
// and the 8 partial sums are combined at the end: deterministic.  The next
// stretch's words and j data are loaded while the current one is evaluated.
//
// W waves share a cluster: wave w takes stretches w, w + W, ... (pair_waves).
//
// Bound by VALU issue (FP64 and conversions take 4 cycles a wave, as FP32).
// Measured at 250,000 dense beads (51.7 M pairs, a list every 10 steps): 1.26e8
// VALU instructions and 0.272 ms a launch; draining 128 words at a time, with
// the ballots and counts taken in the walk and four clusters to a block, took
// 1.70e8 and 0.307 ms.  Sharing the launch with the springs as well: k_step.
// ---------------------------------------------------------------------------
constexpr int32_t QSTRETCH = 3;           // stretches of 64 words in the ring
constexpr int32_t QRING = 64 * QSTRETCH;
constexpr int32_t QLEN = 256;             // queue entries (a power of two >= QRING)

// One wave's queues in LDS.  Their stride keeps the 8 particles' entries in
// different banks.
struct QueueIdx
{
    uint8_t at[CLUSTER][QLEN + 16];
};

// One wave's ring of a pair walk.  j's parameters: all of jprm where the
// hydrophobicity or the flags are read (WIDE: hydrophobic term, energies),
// else the two steric factors.
template <bool WIDE> struct QueueLds
{
    float4 pos[QRING];
    float4 prm[QRING];
    QueueIdx idx;
    __device__ void put(int s, float4 r) { prm[s] = r; }
    __device__ float4 get(int s) const { return prm[s]; }
};
template <> struct QueueLds<false>
{
    float4 pos[QRING];
    float2 prm[QRING];
    QueueIdx idx;
    __device__ void put(int s, float4 r) { prm[s] = make_float2(r.x, r.y); }
    __device__ float4 get(int s) const
    {
        const float2 r = prm[s];
        return make_float4(r.x, r.y, 0.0f, 0.0f);
    }
};

// A stretch as planned: the words each particle sees, how many those are (a
// byte per particle), and the rounds the stretch takes.
struct QPlan
{
    uint64_t sees[CLUSTER];
    uint64_t counts;
    uint64_t rounds;
};
static_assert(sizeof(QPlan) == QPLAN_BYTES, "plan records");

// Over the 8 lanes of an aligned group (every lane gets the result).
__device__ inline int32_t max8(int32_t v)
{
    v = max(v, __builtin_amdgcn_update_dpp(v, v, 0xB1, 0xF, 0xF, false)); // quad_perm 1 0 3 2
    v = max(v, __builtin_amdgcn_update_dpp(v, v, 0x4E, 0xF, 0xF, false)); // quad_perm 2 3 0 1
    return max(v, __builtin_amdgcn_update_dpp(v, v, 0x141, 0xF, 0xF, false)); // row_half_mirror
}

// The plan of a cluster's list: cnt words at L, for W waves.  One wave; the
// words were written before by the same wave.
__device__ inline void queue_plan(const uint32_t *L, int32_t cnt, int32_t W, QPlan *plan)
{
    const int lane = threadIdx.x & 63, il = lane & 7;
    for (int32_t w = 0; w < W; ++w)
    {
        // of the lane's particle: entries waiting, and those of the last stretch
        int32_t wait = 0, last = 0;
        int32_t t = 64 * w;
        uint32_t next = t + lane < cnt ? L[t + lane] : 0u;
        for (; t < cnt; t += 64 * W)
        {
            const uint32_t wd = next;
            const int32_t tn = t + 64 * W + lane;
            next = tn < cnt ? L[tn] : 0u;
            uint64_t mine = 0, counts = 0;
            int32_t c = 0;
#pragma unroll
            for (int k = 0; k < CLUSTER; ++k)
            {
                const uint64_t b = __ballot((wd >> (24 + k)) & 1u);
                const int32_t n = __popcll(b);
                counts |= (uint64_t)n << (8 * k);
                mine = il == k ? b : mine;
                c = il == k ? n : c;
            }
            const bool more = t + 64 * W < cnt;
            // waiting from before the last stretch: the next one takes their places
            const int32_t old = wait - last;
            wait += c;
            const int32_t must = more ? max(old, 0) : wait;
            const int32_t least = max8((must + 7) >> 3), full = -max8(-(wait >> 3));
            const int32_t rounds = max(least, full);
            wait = max(wait - 8 * rounds, 0);
            last = c;
            QPlan *p = plan + t / 64;
            if (lane < CLUSTER)
                p->sees[lane] = mine;
            if (lane == 0)
            {
                p->counts = counts;
                p->rounds = (uint64_t)rounds;
            }
        }
    }
}

// One lane's share of its particle's pair force and energies.
struct PairSums
{
    double fx = 0.0, fy = 0.0, fz = 0.0, es = 0.0, ee = 0.0, eh = 0.0;

    // over the 8 lanes of each particle (lanes il, il + 8, ..., il + 56)
    template <bool ENERGY> __device__ void reduce()
    {
        for (int off = 8; off < 64; off <<= 1)
        {
            fx += __shfl_xor(fx, off, 64);
            fy += __shfl_xor(fy, off, 64);
            fz += __shfl_xor(fz, off, 64);
            if (ENERGY)
            {
                es += __shfl_xor(es, off, 64);
                ee += __shfl_xor(ee, off, 64);
                eh += __shfl_xor(eh, off, 64);
            }
        }
    }
    template <bool ENERGY> __device__ void store(double *o) const
    {
        o[0] = fx;
        o[1] = fy;
        o[2] = fz;
        if (ENERGY)
        {
            o[3] = es;
            o[4] = ee;
            o[5] = eh;
        }
    }
    template <bool ENERGY> __device__ void add(const double *o)
    {
        fx += o[0];
        fy += o[1];
        fz += o[2];
        if (ENERGY)
        {
            es += o[3];
            ee += o[4];
            eh += o[5];
        }
    }
};

// The walk of wave w of W over cluster ci's list.  ev.fetch(j) loads a word's
// data (one j per lane), ev.put(slot) stores it in the ring, ev.pair(valid,
// slot) evaluates one pair of the lane's particle.
template <class Args, class Eval>
__device__ inline void queue_walk(const Args &a, int32_t ci, int32_t w, int32_t W, QueueIdx &idx, Eval &ev)
{
    const int lane = threadIdx.x & 63;
    const int32_t il = lane & 7, sl = lane >> 3;
    const int32_t cnt = __builtin_amdgcn_readfirstlane(a.cln[ci]);
    const uint32_t *L = a.cl + (size_t)ci * a.cap;
    // constant during the kernel: read with scalar loads
    typedef const __attribute__((address_space(4))) QPlan *PlanPtr;
    PlanPtr plan = (PlanPtr)(a.plan + ((size_t)ci * a.nst + w) * QPLAN_BYTES);
    // the first stretch in flight
    int32_t t = 64 * w;
    ev.fetch(t + lane < cnt ? L[t + lane] & CL_JMASK : 0u);
    // the stretch's plan (scalar registers), and entries queued per particle
    uint64_t sees[CLUSTER], counts = 0;
    int32_t rounds = 0;
    uint32_t tail[CLUSTER];
    auto read_plan = [&]() {
#pragma unroll
        for (int k = 0; k < CLUSTER; ++k)
            sees[k] = plan->sees[k];
    };
#pragma unroll
    for (int k = 0; k < CLUSTER; ++k)
        tail[k] = 0;
    if (t < cnt)
        read_plan();
    // of the lane's particle: entries drained and queued
    int32_t head = 0, mine = 0;
    int32_t slot = 0;
    while (t < cnt)
    {
        ev.put(slot + lane);
#pragma unroll
        for (int k = 0; k < CLUSTER; ++k)
        {
            const uint64_t b = sees[k];
            if (__builtin_amdgcn_inverse_ballot_w64(b))
                idx.at[k][__builtin_amdgcn_mbcnt_hi((uint32_t)(b >> 32),
                                                    __builtin_amdgcn_mbcnt_lo((uint32_t)b, tail[k])) &
                          (QLEN - 1)] = (uint8_t)(slot + lane);
            tail[k] += (uint32_t)__popcll(b);
        }
        counts = plan->counts;
        rounds = (int32_t)plan->rounds;
        mine += (int32_t)(((il < 4 ? (uint32_t)counts : (uint32_t)(counts >> 32)) >> (8 * (il & 3))) & 255u);
        // the next stretch in flight while this one is evaluated
        t += 64 * W;
        plan += W;
        if (t < cnt)
        {
            read_plan();
            ev.fetch(t + lane < cnt ? L[t + lane] & CL_JMASK : 0u);
        }
        wave_lds_sync();
        int32_t e = head + sl;
        for (int32_t r = 0; r < rounds; ++r, e += 8)
        {
            const bool valid = e < mine;
            ev.pair(valid, valid ? (int32_t)idx.at[il][e & (QLEN - 1)] : 0);
        }
        head = min(head + 8 * rounds, mine);
        wave_lds_sync();
        slot = slot == QRING - 64 ? 0 : slot + 64;
    }
}

// The pair terms as the walk evaluates them.
template <int SMODE, int EMODE, int HYDRO, bool ENERGY> struct PairEval
{
    const PairArgs &a;
    QueueLds<ENERGY || HYDRO> &q;
    float4 pi = make_float4(0.f, 0.f, 0.f, 0.f), ri = make_float4(0.f, 0.f, 0.f, 0.f);
    PairI c;
    float4 pj, rj;
    PairSums s;

    __device__ PairEval(const PairArgs &args, int32_t ci, QueueLds<ENERGY || HYDRO> &lds) : a(args), q(lds)
    {
        const int32_t i = ci * CLUSTER + (int32_t)(threadIdx.x & 7u);
        if (i < a.n)
        {
            pi = a.pos[i];
            ri = a.jprm[i];
        }
        c = pair_i<SMODE, EMODE>(pi, ri, a);
    }
    __device__ void fetch(uint32_t j)
    {
        pj = partner(a.pos, j);
        rj = partner(a.jprm, j);
    }
    __device__ void put(int32_t slot)
    {
        q.pos[slot] = pj;
        q.put(slot, rj);
    }
    __device__ void pair(bool valid, int32_t src)
    {
        interact<SMODE, EMODE, HYDRO, ENERGY>(valid, pi, ri, q.pos[src], q.get(src), a, c, s.fx, s.fy, s.fz, s.es,
                                              s.ee, s.eh);
    }
};

} // namespace

} // namespace bs
