// bs_spring.hpp -- the spring edge and what ends a particle's force: external,
// probe, field and membrane forces, viscosity and the Euler step.  Shared by
// the spring kernel and the step kernel.
#pragma once

#include "bs_device.hpp"

namespace bs
{

namespace
{

// ---------------------------------------------------------------------------
// IMPALA (imp.hpp:29-159, ForceField.cpp:62-86) in FP64: returns the energy
// and adds the force (the negated gradient vector times the scale) to f.
// The curved geometry z' = sqrt(x^2 + (z - c)^2) - R cancels two numbers of
// the size of the tube radius, so it is formed in double.
// ---------------------------------------------------------------------------
__device__ inline double imp_eval(float xf, float zf, float sasa, float tr, float uo, float lo, float uc, float lc,
                                  float scale, double c_spring, double f[3])
{
    const double alpha = (double)1.99f, z0 = 15.75, alip = (double)-0.018f;
    const bool flat = uo == 0.0f && lo == 0.0f && uc == 0.0f && lc == 0.0f;
    const double x = xf, z = zf;
    const double ru = uc == 0.0f ? 1000000.0 : fabs(1.0 / (double)uc);
    const double rl = lc == 0.0f ? 1000000.0 : fabs(1.0 / (double)lc);
    const int su = (uc > 0.0f) - (uc < 0.0f), sl = (lc > 0.0f) - (lc < 0.0f);
    const double cu = (double)uo - su * ru, cl = -(double)lo - sl * rl;
    const double vu0 = x, vu2 = z - cu, vl0 = x, vl2 = z - cl;
    const double nu = sqrt(vu0 * vu0 + vu2 * vu2);
    const double nl = sqrt(vl0 * vl0 + vl2 * vl2);
    const double zu = su == 0 ? z : (z > cu ? su * nu + uo - ru : -su * nu + uo - ru);
    const double zl = sl == 0 ? z : (z > cl ? sl * nl - lo - rl : -sl * nl - lo - rl);
    const double wu = zu - uo, wl = zl + lo;
    const double xu = exp(alpha * (fabs(wu) - z0)), xl = exp(alpha * (fabs(wl) - z0));
    const double pre = -(double)sasa * tr + alip * sasa;
    const double eu = pre * (0.5 - 1.0 / (1.0 + xu));
    const double el = pre * (0.5 - 1.0 / (1.0 + xl));
    double dcu = alpha * wu * xu / ((xu + 1.0) * (xu + 1.0) * fabs(wu));
    double dcl = alpha * wl * xl / ((xl + 1.0) * (xl + 1.0) * fabs(wl));
    if (!isfinite(dcu))
        dcu = 0.0;
    if (!isfinite(dcl))
        dcl = 0.0;
    double du[3] = {0.0, 0.0, 1.0}, dl[3] = {0.0, 0.0, 1.0};
    if (su != 0)
    {
        const double inv = nu > 1e-40 ? 1.0 / nu : 0.0;
        du[0] = vu0 * inv;
        du[2] = vu2 * inv;
    }
    if (sl != 0)
    {
        const double inv = nl > 1e-40 ? 1.0 / nl : 0.0;
        dl[0] = vl0 * inv;
        dl[2] = vl2 * inv;
    }
    const double mu = pre * dcu * c_spring, ml = pre * dcl * c_spring;
    for (int c = 0; c < 3; ++c)
        f[c] -= (double)scale * (flat ? du[c] * mu : du[c] * mu + dl[c] * ml);
    return (double)scale * (flat ? eu : eu + el);
}

// A row's springs as one of its lanes reads them: edge words {j | static bit
// 31, L0 bits} and stiffnesses of the lane's edges, one every `step` bytes,
// at 32-bit offsets from the wave's first row (the base stays in scalar
// registers).  Every row ends in at least one null edge (j = the row itself,
// L0 = 0: no extension, no force), so an offset past the row's end is moved
// to its last word and nothing else guards the edge.
struct EdgeRow
{
    const char *eb, *kb; // kb null: every spring has stiffness k_uni
    float k_uni;
    uint32_t off, last, step, self; // self: the row, partner of its null edges

    // G lanes per row, 64 / G rows from row0 on (wave-uniform) of the wave;
    // row0 < n.  Rows past n, static rows and disabled springs read the null
    // edge of their (of the last) row.
    template <class Args> __device__ EdgeRow(const Args &a, int32_t row0, int32_t row, int32_t lane, int32_t G, bool on)
    {
        const int32_t c0 = __builtin_amdgcn_readfirstlane(a.sp_ptr[row0]), r = min(row, a.n - 1);
        eb = reinterpret_cast<const char *>(a.sp_e + (size_t)c0 * EDGE_PAD);
        kb = a.sp_k ? reinterpret_cast<const char *>(a.sp_k + (size_t)c0 * EDGE_PAD) : nullptr;
        k_uni = a.k_uni;
        step = (uint32_t)G * sizeof(uint2);
        self = (uint32_t)r;
        const uint32_t unit = EDGE_PAD * sizeof(uint2);
        last = (uint32_t)(a.sp_ptr[r + 1] - c0) * unit - (uint32_t)sizeof(uint2);
        off = on ? (uint32_t)(a.sp_ptr[r] - c0) * unit + (uint32_t)lane * (uint32_t)sizeof(uint2) : last;
    }
    // the longest row of the wave in steps (wave-uniform): a row's first lane
    // takes the most, and rows start at lanes that STRIDE divides
    template <int STRIDE> __device__ int32_t steps() const
    {
        const int32_t s = ((int32_t)(last - off) + (int32_t)(sizeof(uint2) + step) - 1) >> (31 - __builtin_clz(step));
        int32_t m = 0;
#pragma unroll
        for (int o = 0; o < 64; o += STRIDE)
            m = max(m, __builtin_amdgcn_readlane(s, o));
        return m;
    }
    __device__ void word(int u, uint32_t &j, float &l0, float &k) const
    {
        const uint32_t o = min(off + (uint32_t)u * step, last);
        const uint2 w = *reinterpret_cast<const uint2 *>(eb + o);
        j = w.x;
        l0 = __uint_as_float(w.y);
        k = kb ? *reinterpret_cast<const float *>(kb + (o >> 1)) : k_uni;
    }
};

// The positions of a row's particle in FP64, and the sums over the lane's
// edges: force (without the factor C_spring x scale) and energy.
template <bool COMP> struct RowSum
{
    double px, py, pz, lx = 0.0, ly = 0.0, lz = 0.0;
    double fx = 0.0, fy = 0.0, fz = 0.0, e = 0.0;

    __device__ RowSum(float4 p, float4 l) : px(p.x), py(p.y), pz(p.z)
    {
        if (COMP)
        {
            lx = l.x;
            ly = l.y;
            lz = l.z;
        }
    }
    // One spring: force k ext d / len.  The FP64 length comes from the FP32
    // reciprocal square root and one Newton step (1e-14 relative), so that
    // the extension keeps its accuracy near rest; its seed's argument is kept
    // at or above the smallest normal float (a coincident pair: length 0,
    // finite factor, no force; closer than 1e-19 A: finite, inexact).
    __device__ void edge(float4 pj, const float4 *plo, uint32_t j, float k, float l0, bool energy, float scale)
    {
        double dx = (double)pj.x - px, dy = (double)pj.y - py, dz = (double)pj.z - pz;
        if (COMP)
        {
            const float4 lj = partner(plo, j);
            dx += (double)lj.x - lx;
            dy += (double)lj.y - ly;
            dz += (double)lj.z - lz;
        }
        const double r2 = fma(dx, dx, fma(dy, dy, dz * dz));
        const double y0 = (double)__builtin_amdgcn_rsqf(fmaxf((float)r2, 1.1754944e-38f));
        const double y = y0 * fma(-0.5 * y0, r2 * y0, 1.5);
        const double ext = fma(r2, y, -(double)l0);
        const double f = (double)k * ext * y;
        fx = fma(dx, f, fx);
        fy = fma(dy, f, fy);
        fz = fma(dz, f, fz);
        if (energy)
            e += ((int32_t)j < 0 ? 1.0 : 0.5) * 0.5 * (double)scale * (double)k * ext * ext;
    }
};

// Cell of a field grid holding a position, -1 off the grid
// (GridCoordinatesSystem.hpp:85-93,206-218: off when x < min or x > max - 1e-6).
__device__ inline int64_t grid_cell(const GridView &g, float x, float y, float z)
{
    const double p[3] = {x, y, z};
    int64_t q[3];
    for (int c = 0; c < 3; ++c)
    {
        if (!(p[c] >= g.origin[c]) || p[c] > g.bmax[c] - 1e-6)
            return -1;
        q[c] = (int64_t)(int32_t)((p[c] - g.origin[c]) / g.cell[c]);
        if (q[c] >= g.shape[c])
            return -1;
    }
    return (q[0] * g.shape[1] + q[1]) * g.shape[2] + q[2];
}

// One particle's interactions with the probe (Particle::addStericProbeForce /
// addElectrostaticProbeForce, Particle.cpp:434-465), in FP64: the force on
// the particle goes to f; the pair energies (in full) to es, ee.  The
// formulas are the pair kernel's (energy/steric.hpp, electrostatic.hpp) with
// the probe as the first particle; no cutoff and no spring exclusion.
__device__ inline void probe_pair(const ProbeArgs &p, const float4 q, float4 pi, float4 ri, double cs, double f[3],
                                  double &es, double &ee)
{
    const double dx = (double)q.x - (double)pi.x, dy = (double)q.y - (double)pi.y, dz = (double)q.z - (double)pi.z;
    const double r = sqrt(dx * dx + dy * dy + dz * dz);
    const double inv = r > 1e-40 ? 1.0 / r : 0.0; // a zero vector stays zero (Vector3f::normalize)
    double fm = 0.0;
    if (p.steric)
    {
        double e = 0.0, m = 0.0;
        if (p.steric_mode == 0)
        { // linear: overlap of the raw radii
            const double dv = r - ((double)p.radius + (double)ri.x);
            if (!(dv > 0.0))
            {
                e = 0.5 * dv * dv;
                m = -fabs(dv) * cs;
            }
        }
        else if (r >= 0.1)
        {
            const bool prod = p.steric_mode == 3; // Zacharias: raw products; else square-root factors
            const double eij = (double)p.eps * (double)ri.y;
            const double R2 = (double)p.radius * (double)ri.x; // the factors' product (jprm)
            const double s2 = R2 * inv * inv, s6 = s2 * s2 * s2;
            if (p.steric_mode == 1)
            { // Amber 12-6
                e = eij * s6 * s6 - 2.0 * eij * s6;
                m = (-12.0 * eij * s6 * s6 + 12.0 * eij * s6) * inv * cs;
            }
            else if (p.steric_mode == 2)
            { // Lewitt 8-6
                e = 3.0 * eij * s6 * s2 - 4.0 * eij * s6;
                m = (-24.0 * eij * s6 * s2 + 24.0 * eij * s6) * inv * cs;
            }
            else if (prod)
            { // Zacharias 8-6
                e = eij * s6 * s2 - eij * s6;
                m = (-8.0 * eij * s6 * s2 + 6.0 * eij * s6) * inv * cs;
            }
        }
        es += (double)p.steric_scale * e;
        fm += (double)p.steric_scale * m;
    }
    if (p.elec && r >= 0.001)
    {
        const double qq = (double)q.w * (double)pi.w;
        if (p.ddd)
        { // eps(r) = eps r
            ee += p.ke * qq * inv * inv;
            fm += -2.0 * p.kf * qq * inv * inv * inv;
        }
        else
        {
            ee += p.ke * qq * inv;
            fm += -p.kf * qq * inv * inv;
        }
    }
    f[0] += dx * inv * fm;
    f[1] += dy * inv * fm;
    f[2] += dz * inv * fm;
}

// The springs of the wave's rows (at most `steps` edges a lane), D edges in
// flight per lane: the edge words of the next D load while these gather and
// compute (two dependent loads per edge: the word, then x_j).  A lane with null
// edges alone adds nothing, also for a particle whose position is not finite
// (a null edge of a lane that has a real one cannot make that one's sum worse);
// with ALL the caller sees to that, a row at a time (lost_row).
//
// Every edge in flight costs a row its loads, needed or not: with ALL none is
// skipped, which suits D = 4 beside the pair walk (skipped there: 71 -> 69 us
// a step for chains of 250,000 beads, but 465 -> 467 for rows of 182); with D =
// 8 and the springs alone the branches pay at every length (100,000 rows of 5,
// 71 and 185 springs: 39.4, 43.5 and 59.8 us with all loads, 28.9, 37.2 and
// 55.6 without the idle ones).
template <int D, bool ALL, bool COMP>
__device__ inline void row_springs(const SpringArgs &a, EdgeRow &er, RowSum<COMP> &sum, bool energy, int32_t steps)
{
    uint32_t j[D], jn[D];
    float k[D], l[D], kn[D], ln[D];
#pragma unroll
    for (int u = 0; u < D; ++u)
        if (ALL || u < steps)
            er.word(u, j[u], l[u], k[u]);
    const bool real = j[0] != er.self;
    for (int32_t left = steps; left > 0; left -= D) // wave-uniform
    {
        float4 p[D];
#pragma unroll
        for (int u = 0; u < D; ++u)
            if (ALL || u < left)
                p[u] = partner(a.pos, j[u]);
        er.off += D * er.step;
#pragma unroll
        for (int u = 0; u < D; ++u)
            if (ALL || D + u < left)
                er.word(u, jn[u], ln[u], kn[u]);
#pragma unroll
        for (int u = 0; u < D; ++u)
            if (u < left)
                sum.edge(p[u], a.plo, j[u], k[u], l[u], energy, a.spring_scale);
#pragma unroll
        for (int u = 0; u < D; ++u)
        {
            j[u] = jn[u];
            k[u] = kn[u];
            l[u] = ln[u];
        }
    }
    if (!ALL && !real)
        sum.fx = sum.fy = sum.fz = sum.e = 0.0;
}

// Whether row's springs add nothing although its position, not being finite,
// made its null edges' sums NaN: a static row, or one without springs.
__device__ inline bool lost_row(const SpringArgs &a, int32_t row, float4 pi, uint32_t fli)
{
    return !(fabsf(pi.x) < INFINITY && fabsf(pi.y) < INFINITY && fabsf(pi.z) < INFINITY) &&
           ((fli & PF_STATIC) || a.sp_e[(size_t)a.sp_ptr[row] * EDGE_PAD].x == (uint32_t)row);
}

// What a particle's row adds to the sums beside its force: energies, and the
// opposite of the probe's force on it with the probe's pair energies.
struct RowOut
{
    double eke = 0.0, eimp = 0.0, efld = 0.0;
    double pf[3] = {0.0, 0.0, 0.0}, pes = 0.0, pee = 0.0;
};

// Ends row `row` (dynamic) from the sum (sx, sy, sz) of its spring and pair
// forces: the other forces, then (INTEGRATE) the viscous semi-implicit Euler
// step (SpringNetwork.cpp:202-241; Particle.cpp:80-128), else the force.
template <bool INTEGRATE, bool COMP>
__device__ inline void finish_row(const SpringArgs &a, int32_t row, float4 pi, float4 li, uint32_t fli, double sx,
                                  double sy, double sz, RowOut &o)
{
    float4 v = a.vel[row];
    if (a.fext)
    {
        const float4 fe = a.fext[row];
        sx += fe.x;
        sy += fe.y;
        sz += fe.z;
    }
    if (a.probe.state)
    { // the probe: the particle's share here, the opposite on the probe
        double f[3] = {0.0, 0.0, 0.0};
        probe_pair(a.probe, a.probe.state->x, pi, a.jprm[row], a.k.c_spring, f, o.pes, o.pee);
        sx += f[0];
        sy += f[1];
        sz += f[2];
        o.pf[0] = -f[0];
        o.pf[1] = -f[1];
        o.pf[2] = -f[2];
    }
    const float4 ip = a.iprm[row];
    // field forces: nearest-lower-cell lookup, no interpolation
    // (Particle.cpp:136-189); off-grid particles get nothing
    if (a.gpot.cells)
    {
        const int64_t c = grid_cell(a.gpot, pi.x, pi.y, pi.z);
        if (c >= 0)
        {
            const float4 g = a.gpot.cells[c];
            const double qs = (double)pi.w * (double)a.gpot.scale;
            sx += (double)g.x * qs;
            sy += (double)g.y * qs;
            sz += (double)g.z * qs;
            o.efld += (double)g.w * qs * a.e_field;
        }
    }
    if (a.gden.cells)
    {
        const int64_t c = grid_cell(a.gden, pi.x, pi.y, pi.z);
        if (c >= 0)
        {
            const float4 g = a.gden.cells[c];
            const double bs = (double)ip.w * (double)a.gden.scale;
            sx += (double)g.x * bs;
            sy += (double)g.y * bs;
            sz += (double)g.z * bs;
        }
    }
    if (a.imp_enable)
    {
        double f[3] = {sx, sy, sz};
        o.eimp += imp_eval(pi.x, pi.z, ip.y, ip.z, a.imp_uo, a.imp_lo, a.imp_uc, a.imp_lc, a.imp_scale,
                         a.k.c_spring, f);
        sx = f[0];
        sy = f[1];
        sz = f[2];
    }
    // the position-dependent sum is rounded once; the viscous term
    // -gamma v follows in FP32 (Particle.cpp:80-84)
    float fxf = (float)sx, fyf = (float)sy, fzf = (float)sz;
    if (a.visc_enable)
    {
        fxf -= v.x * a.visc;
        fyf -= v.y * a.visc;
        fzf -= v.z * a.visc;
    }
    const float fx = fxf, fy = fyf, fz = fzf;
    if (!INTEGRATE)
    {
        a.fout[row] = make_float4(fx, fy, fz, 0.0f);
    }
    else if (fli & PF_RIGID)
    {
        // placed by its body after the body solve (k_rigid_place); a rigid
        // particle's kinetic energy is reset before it is summed
        // (RigidBody.cpp:629, SpringNetwork.cpp:232)
        a.frig[row] = make_double4(fx, fy, fz, 0.0);
    }
    else
    {
        const float m = ip.x;
        const float dt = a.dt;
        if (m > 0.0f)
        {
            v.x = v.x + (fx / m) * dt;
            v.y = v.y + (fy / m) * dt;
            v.z = v.z + (fz / m) * dt;
        }
        o.eke += 0.5 * (double)m * ((double)v.x * v.x + (double)v.y * v.y + (double)v.z * v.z) * a.k.c_kinetic;
        float4 xn = pi;
        if (COMP)
        {
            // two-sum of hi + v*dt, carried into the low word
            float4 ln = li;
            const float u[3] = {v.x * dt, v.y * dt, v.z * dt};
            float *hp[3] = {&xn.x, &xn.y, &xn.z};
            float *lp[3] = {&ln.x, &ln.y, &ln.z};
#pragma unroll
            for (int c = 0; c < 3; ++c)
            {
                const float h = *hp[c];
                const float s = h + u[c];
                const float bb = s - h;
                const float err = (h - (s - bb)) + (u[c] - bb);
                const float lo = *lp[c] + err;
                const float h2 = s + lo;
                *lp[c] = lo - (h2 - s);
                *hp[c] = h2;
            }
            a.plo_out[row] = ln;
        }
        else
        {
            xn.x = pi.x + v.x * dt;
            xn.y = pi.y + v.y * dt;
            xn.z = pi.z + v.z * dt;
        }
        if (!isfinite(xn.x) || !isfinite(xn.y) || !isfinite(xn.z))
            atomicMin(&a.status[1], a.perm[row]);
        const float4 xr = a.xref[row];
        const float ex = xn.x - xr.x, ey = xn.y - xr.y, ez = xn.z - xr.z;
        if (!(ex * ex + ey * ey + ez * ez <= a.half_skin2))
            atomicOr(&a.status[7], 1);
        a.vel[row] = v;
        a.pos_out[row] = xn;
    }
}

} // namespace

} // namespace bs
