// bs_step.hip -- the step kernel: the last neighbour list's pair forces, the
// springs and the integrator of a cluster's 8 particles in one launch.
//
// Each wave takes its springs first, then its share of the pairs.  The spring
// gather waits on memory (its edge words are read once a step, from HBM) and
// the pair walk keeps the VALU busy, so waves in one phase run beside waves
// in the other, and the pair forces never leave the chip.  At 250,000 dense
// beads a step takes 0.46 ms, 0.40 of it here.  When the kernels were joined a
// step took 0.50 ms, against 0.56 ms with the two as kernels of their own before
// the pair walk was planned and 0.53 ms after (list builds have become shorter
// since).  Measured then and left out: one spring edge per lane between the stretches of the pair walk (its
// partner in flight meanwhile: 0.53 ms; 8-lane rows read a line in two halves,
// a stretch apart); half the blocks taking their pairs first (0.51 ms; the
// second copy's registers cost a wave per SIMD); six or eight spring edges in
// flight (0.51, 0.55 ms, also for the registers).
#include "bs_pairterm.hpp"
#include "bs_spring.hpp"

namespace bs
{

namespace
{

// The springs of one wave: of `rows` rows from `first` on, G = 64 / rows lanes
// each (one pass: rows of 50 to 200 springs fill 8 lanes).  out: each row's
// force and, with ENERGY, energy.
template <bool COMP, bool ENERGY>
__device__ inline void spring_walk(const SpringArgs &a, int32_t first, int32_t rows, double (*out)[ENERGY ? 4 : 3])
{
    const int lane = threadIdx.x & 63;
    const int32_t G = 64 / rows, sub = lane / G;
    const bool live = first + sub < a.n && a.spring_enable;
    const int32_t row = min(first + sub, a.n - 1);
    const float4 pi = a.pos[row];
    float4 li = make_float4(0.f, 0.f, 0.f, 0.f);
    if (COMP)
        li = a.plo[row];
    RowSum<COMP> sum(pi, li);
    if (a.spring_enable)
    {
        EdgeRow er(a, min(first, a.n - 1), row, lane & (G - 1), G, live && !(fbits(a.jprm[row].w) & PF_STATIC));
        row_springs<4, true, COMP>(a, er, sum, ENERGY, er.steps<CLUSTER>());
    }
    for (int off = G / 2; off > 0; off >>= 1)
    {
        sum.fx += __shfl_xor(sum.fx, off, 64);
        sum.fy += __shfl_xor(sum.fy, off, 64);
        sum.fz += __shfl_xor(sum.fz, off, 64);
        if (ENERGY)
            sum.e += __shfl_xor(sum.e, off, 64);
    }
    if ((lane & (G - 1)) == 0)
    {
        const double cs = a.k.c_spring * (double)a.spring_scale;
        double *o = out[sub];
        o[0] = sum.fx * cs;
        o[1] = sum.fy * cs;
        o[2] = sum.fz * cs;
        if (ENERGY)
            o[3] = sum.e;
    }
}

template <bool WIDE, bool ENERGY> struct StepLds
{
    QueueLds<WIDE> q;
    double pair[CLUSTER][ENERGY ? 6 : 3];   // the wave's pair sums
    double spring[CLUSTER][ENERGY ? 4 : 3]; // spring sums of the wave's 8 / W rows
};

// A block of W waves per cluster: its springs and pairs (queue_walk), then its
// 8 rows end on the first lanes.  Small blocks: a slot is free as soon as
// its cluster is done.
template <int SMODE, int EMODE, int HYDRO, bool ENERGY, bool COMP>
__global__ void __launch_bounds__(BLOCK) k_step(PairArgs p, SpringArgs a)
{
    extern __shared__ __align__(16) char lds[];
    auto *part = reinterpret_cast<StepLds<ENERGY || HYDRO, ENERGY> *>(lds); // one per wave
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int W = blockDim.x >> 6;
    const int32_t ci = blockIdx.x;
    if (halted(a.status))
    { // a stopped call: the state is carried over to the other position buffer
        const int32_t row = ci * CLUSTER + threadIdx.x;
        if (threadIdx.x < CLUSTER && row < a.n)
        {
            a.pos_out[row] = a.pos[row];
            if (COMP)
                a.plo_out[row] = a.plo[row];
        }
        return;
    }
    if (blockIdx.x == 0 && threadIdx.x == 0 && a.steps_done)
        atomicAdd(a.steps_done, 1);
    const int rows = CLUSTER / W;
    spring_walk<COMP, ENERGY>(a, ci * CLUSTER + w * rows, rows, part[w].spring);
    {
        PairEval<SMODE, EMODE, HYDRO, ENERGY> ev(p, ci, part[w].q);
        queue_walk(p, ci, w, W, part[w].q.idx, ev);
        ev.s.template reduce<ENERGY>();
        if (lane < CLUSTER)
            ev.s.template store<ENERGY>(part[w].pair[lane]);
    }
    __syncthreads();
    const int t = threadIdx.x;
    const int32_t row = ci * CLUSTER + t;
    if (t >= CLUSTER || row >= a.n)
        return;
    const double *spring = part[t / rows].spring[t % rows];
    PairSums s;
    for (int v = 0; v < W; ++v)
        s.add<ENERGY>(part[v].pair[t]);
    RowOut o;
    const float4 pi = a.pos[row];
    const uint32_t fli = fbits(a.jprm[row].w);
    const bool lost = lost_row(a, row, pi, fli);
    if (!(fli & PF_STATIC))
    {
        float4 li = make_float4(0.f, 0.f, 0.f, 0.f);
        if (COMP)
            li = a.plo[row];
        double fx = s.fx, fy = s.fy, fz = s.fz;
        if (p.accumulate)
        {
            const double4 f = p.fnb[row];
            fx += f.x;
            fy += f.y;
            fz += f.z;
        }
        if (!lost)
        {
            fx += spring[0];
            fy += spring[1];
            fz += spring[2];
        }
        finish_row<true, COMP>(a, row, pi, li, fli, fx, fy, fz, o);
    }
    if (ENERGY)
    {
        double4 en = make_double4(s.es, s.ee, s.eh, 0.0);
        if (p.accumulate)
        {
            const double4 v = p.epp[row];
            en.x += v.x;
            en.y += v.y;
            en.z += v.z;
        }
        p.epp[row] = en;
        a.eps[row] = make_double4(lost ? 0.0 : spring[3], o.eke, o.eimp, o.efld);
    }
}

template <int S, int E, int H, bool EN, bool C> static void step4(const PairArgs &p, const SpringArgs &a, hipStream_t s)
{
    const int32_t W = pair_waves(p.ncl);
    k_step<S, E, H, EN, C><<<p.ncl, 64 * W, W * sizeof(StepLds<EN || H, EN>), s>>>(p, a);
}

template <int S, int E, int H> static void step3(const PairArgs &p, const SpringArgs &a, hipStream_t s)
{
    if (a.plo)
        p.energy ? step4<S, E, H, true, true>(p, a, s) : step4<S, E, H, false, true>(p, a, s);
    else
        p.energy ? step4<S, E, H, true, false>(p, a, s) : step4<S, E, H, false, false>(p, a, s);
}

template <int S> static void step2(const PairArgs &p, const SpringArgs &a, int32_t em, int32_t h, hipStream_t s)
{
    if (em == 0)
        h ? step3<S, 0, 1>(p, a, s) : step3<S, 0, 0>(p, a, s);
    else if (em == 1)
        h ? step3<S, 1, 1>(p, a, s) : step3<S, 1, 0>(p, a, s);
    else
        h ? step3<S, 2, 1>(p, a, s) : step3<S, 2, 0>(p, a, s);
}

} // namespace

void launch_step_kernel(const PairArgs &p, const SpringArgs &a, int32_t elec_mode, int32_t hydro, hipStream_t s)
{
    if (p.ncl <= 0)
        return;
    switch (p.steric_mode)
    {
    case -1: step2<-1>(p, a, elec_mode, hydro, s); break;
    case 0: step2<0>(p, a, elec_mode, hydro, s); break;
    case 1: step2<1>(p, a, elec_mode, hydro, s); break;
    case 2: step2<2>(p, a, elec_mode, hydro, s); break;
    default: step2<3>(p, a, elec_mode, hydro, s); break;
    }
}

} // namespace bs
