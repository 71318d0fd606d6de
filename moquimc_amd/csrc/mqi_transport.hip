// Transport kernels for gfx950: fippel stepping, ionization with straggling,
// multiple Coulomb scattering, p-p elastic, p-O elastic/inelastic, the
// dose / LETd / statistics / Dij scorers, and the two launch forms:
//
//   batched  one persistent launch over every (scenario, spot) history of a
//            plan; lanes pull histories from a device counter with one
//            atomic per wavefront refill (ballot + popcount), so a lane whose
//            track ends takes the next secondary or history on the next
//            iteration while its neighbours keep stepping.
//   plain    histories split statically over threads (the reference's
//            mc::transport_particles_patient launch, mqi_transport.hpp:
//            113-250, mqi_tps_env.hpp:1058-1129), consecutive spots sharing
//            a launch while a lane per history holds them.
//
// Compiled three times: MQI_EXACT=1 (namespace mqi_exact, -ffp-contract=off,
// portable math: bit-identical to the CPU restatement), MQI_EXACT=0
// (namespace mqi_fast, device math library, FMA contraction), and the latter
// again with MQI_DEFER=6 (namespace mqi_fast6) for launches of five or six
// scorers.  A fifth scorer added on every step cost 2.5 ms of the 11.9 of 3e5
// histories with dose and four LET scorers (9.4 with its sum in LDS too, 8.5
// with the register budget of 3 waves/SIMD); built into mqi_fast the two slots
// cost every launch registers (143 -> 153 VGPRs, Dij field 18.9 -> 20.1 ms).
#include "mqi_device.hpp"
#include "mqi_kernels.h"
#if MQI_EXACT
#define MQI_VOXEL_EXIT mqi_dev::intersect_in
#else
#include "mqi_prod.hpp"
#define MQI_VOXEL_EXIT mqi_dev::exit_distance
#endif

#define MQI_TABLE_QUALIFIER static __constant__
#include "mqi_tables.inc"

#if MQI_EXACT
#define MQI_NS mqi_exact
#elif MQI_DEFER > MQI_GROUP
#define MQI_NS mqi_fast6
#else
#define MQI_NS mqi_fast
#endif

using namespace mqi_dev;

namespace MQI_NS
{

// The launch's parameters as read where they are needed: loads through this
// reference are not moved out of the history loop.  Parameters of the rare
// paths (new histories, secondaries, beamline children) otherwise end up
// loaded before the loop, spilled from the scalar registers into VGPR lanes
// and read back by v_readlane wherever they are used.  With the scoring modes
// of a step in two words and its cell's edges read once: 33 spilled scalars
// for 171 and 138 VGPRs for 151; slab phantom 37.3 -> 33.5 ms, water spot 5.55
// -> 5.31 ms.
MQI_DI const transport_params& cold() {
    uint64_t a = (uint64_t) __builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(a));
    auto p = (const __attribute__((address_space(4))) transport_params*) a;
    return *(const transport_params*) p;
}

// ------------------------------------------------------------------ physics
// Per-lane context: LDS tables, grid view, RNG, the lane's secondary stack.
struct ctx {
    const float* T;   // LDS tables
    grid_view    g;
    rng_t        rng;
    int          sp;
    unsigned     drops;
    int          child;    // world child the track is in: 0 .. nbl - 1 beamline, nbl the patient
    int          nbl;      // beamline children
};

#if MQI_EXACT
// p_ionization_tabulated::cross_section (mqi_p_ionization.hpp:254-268): Ei=0.1, Ef=299.6, step 0.5
MQI_DI float cs_ion(const ctx& c, float Ek, float rho) {
    float cs = 0;
    if (Ek >= 0.1f && Ek <= 299.6f) {
        uint16_t idx0 = uint16_t((Ek - 0.1f) / 0.5f);
        uint16_t idx1 = idx0 + 1;
        float    x0   = 0.1f + idx0 * 0.5f;
        float    x1   = x0 + 0.5f;
        cs            = intpl(Ek, x0, x1, c.T[T_CS_ION + idx0], c.T[T_CS_ION + idx1]);
    }
    cs *= rho;
    return cs;
}
// pp / p-O tables: Ek_min 0.5, Ek_max 300, dEk 0.5 (mqi_pp_elastic.hpp:221-235 and twins)
MQI_DI float cs_tab(const ctx& c, int off, float Ek, float rho) {
    float cs = 0;
    if (Ek >= 0.5f && Ek <= 300.0f) {
        uint16_t idx0 = uint16_t((Ek - 0.5f) / 0.5f);
        uint16_t idx1 = idx0 + 1;
        float    x0   = 0.5f + idx0 * 0.5f;
        float    x1   = x0 + 0.5;
        cs            = intpl(Ek, x0, x1, c.T[off + idx0], c.T[off + idx1]);
    }
    cs *= rho;
    return cs;
}
// dEdx (mqi_p_ionization.hpp:271-286)
MQI_DI float dedx(const ctx& c, float Ek) {
    float pw = 0;
    if (Ek >= 0.1f && Ek <= 299.6f) {
        uint16_t idx0 = uint16_t((Ek - 0.1f) / 0.5f);
        uint16_t idx1 = idx0 + 1;
        float    x0   = 0.1f + idx0 * 0.5f;
        float    x1   = x0 + 0.5f;
        pw            = intpl(Ek, x0, x1, c.T[T_DEDX + idx0], c.T[T_DEDX + idx1]);
    } else if (Ek < 0.1f && Ek > 0) {
        pw = c.T[T_DEDX];
    }
    return -1.0 * pw;
}

// energy_loss + energy_straggling (mqi_p_ionization.hpp:297-345); the
// residual-range walk stops at index 0 where the reference's uint16_t
// counter would wrap past zero.
template<bool DBG>
MQI_DI float energy_loss(ctx& c, const rel_q& rel, float rho, float step_length, float sp) {
    const float* R   = c.T + T_RANGE;
    float        L_w = step_length * sp * rho / units::water_density;
    uint16_t     n   = uint16_t((rel.Ek - 0.1f) / 0.5f);
    float        x0  = 0.1f + n * 0.5f;
    float        x1  = x0 + 0.5f;
    if (x0 > rel.Ek) n -= 1;
    if (x1 < rel.Ek) n += 1;
    float r = intpl(rel.Ek, x0, x1, R[n], R[n + 1]);
    if (r < L_w) return rel.Ek;
    r -= L_w;
    for (;;) {
        if (r >= R[n]) break;
        if (n == 0) break;
        --n;
        if (n == 0) break;
    }
    x0            = 0.1f + n * 0.5f;
    x1            = x0 + 0.5f;
    float dE_mean = rel.Ek - intpl(r, R[n], R[n + 1], x0, x1);
    float Te      = (rel.Te_max >= 0.08511) ? 0.08511 : rel.Te_max;
    float O_sq    = units::two_pi_re2_mc2_h2o * rho / units::water_density * L_w;
    O_sq *= Te / rel.beta_sq * (1.0 - 0.5 * rel.beta_sq);
    float ret = c.rng.normal(dE_mean, MQ_SQRTF(O_sq));
    if (ret < 0) ret *= -1.0;
    return ret;
}

// along_step (mqi_p_ionization.hpp:348-420)
template<bool DBG>
MQI_DI void along_step(ctx& c, trk& t, float len, float rho, float sp) {
    rel_q rel = relq(t.ke0);
    float dE  = energy_loss<DBG>(c, rel, rho, len, sp);
    float r   = 1.0;
    if (dE >= t.ke0) {
        r         = t.ke0 / dE;
        t.stopped = true;
    }
    float P     = momentum(rel);
    float X0    = radiation_length<DBG>(rho);
    float th_sq = ((13.9f / P) * (13.9f / P) / rel.beta_sq) * len / X0;
    float th    = MQ_SQRTF(th_sq);
    th          = c.rng.normal(0, MQ_SQRTF(2.0f) * th);
    if (th < 0) th *= -1.0;
    float phi = 2.0 * 3.14159265358979323846 * c.rng.uniform();
    rotate_direction(t.d1, th, phi);
    t.dE += dE * r;
    update_pos(t, r * len);
    t.ke1 -= dE * r;
}

#else
// Cross sections per density of the four processes at Ek (cs_ion, cs_tab)
// and, with DEDX, dEdx: the two index grids of the tables (0.1 + 0.5 i and
// 0.5 + 0.5 i MeV) are evaluated once for the tables that share them.
struct q_cs {
    float ion, pp, poe, poi;
};
template<bool DEDX>
MQI_DI q_cs q_cross(const float* T, float Ek, float* pw) {
    MQI_NO_CONTRACT
    q_cs         c;
    const bool   in = Ek >= 0.1f && Ek <= 299.6f;
    const int    i  = in ? (int) ((Ek - 0.1f) * 2.0f) : 0;
    const float  x0 = __builtin_fmaf((float) i, 0.5f, 0.1f);
    const float  dx = Ek - x0;
    const float  rw = __builtin_amdgcn_rcpf((x0 + 0.5f) - x0);
    const float* t  = T + i;
    c.ion           = t[T_CS_ION] + dx * (t[T_CS_ION + 1] - t[T_CS_ION]) * rw;
    if (DEDX) {
        *pw = t[T_DEDX] + dx * (t[T_DEDX + 1] - t[T_DEDX]) * rw;
        if (!in) *pw = (Ek < 0.1f && Ek > 0) ? T[T_DEDX] : 0.0f;
    }
    const bool   jn = Ek >= 0.5f && Ek <= 300.0f;
    const int    j  = jn ? (int) ((Ek - 0.5f) * 2.0f) : 0;
    const float  dy = Ek - __builtin_fmaf((float) j, 0.5f, 0.5f);
    const float* u  = T + j;
    // the bins are 0.5 wide exactly: the quotient is a doubling
    c.pp  = __builtin_fmaf(dy * (u[T_CS_PP + 1] - u[T_CS_PP]), 2.0f, u[T_CS_PP]);
    c.poe = __builtin_fmaf(dy * (u[T_CS_POE + 1] - u[T_CS_POE]), 2.0f, u[T_CS_POE]);
    c.poi = __builtin_fmaf(dy * (u[T_CS_POI + 1] - u[T_CS_POI]), 2.0f, u[T_CS_POI]);
    if (!in) c.ion = 0.0f;
    if (!jn) c.pp = c.poe = c.poi = 0.0f;
    return c;
}
MQI_DI float q_sum(const q_cs& c, float rho) {
    MQI_NO_CONTRACT
    return __builtin_fmaf(rho, c.poi, __builtin_fmaf(rho, c.poe, __builtin_fmaf(rho, c.ion, rho * c.pp)));
}

// energy_loss + energy_straggling: the residual-range walk of the
// verification build ends at the largest n in [1, n0] with R[n] <= r (0 if
// none), R being non-decreasing.  Walking from the current bin takes one LDS
// round trip per 0.5 MeV lost, the longest lane setting the wave's count (8.3
// per step on the 2000-spot CT plan); here the walk starts at the bin the
// range slope of the current bin predicts, and goes down or up from there to
// the same n (1.7 round trips).
MQI_DI float q_energy_loss(ctx& c, const q_rel& rel, float Ek, float rho, float L_w) {
    MQI_NO_CONTRACT
    const float* R  = c.T + T_RANGE;
    int          n  = (int) ((Ek - 0.1f) * 2.0f);
    const float  x0 = __builtin_fmaf((float) n, 0.5f, 0.1f);
    const float  x1 = x0 + 0.5f;
    if (x0 > Ek) n -= 1;
    if (x1 < Ek) n += 1;
    const float slope = R[n + 1] - R[n];   // mm per 0.5 MeV
    float       r     = R[n] + q_div((Ek - x0) * slope, x1 - x0);
    if (r < L_w) return Ek;
    r -= L_w;
    int k = slope > 0.0f ? (int) q_div(L_w, slope) : 0;
    k     = k < 0 ? 0 : k;
    int   m = n - (k < n ? k : n);
    float a = R[m], b = R[m + 1];
    while (m >= 1 && a > r) {
        --m;
        b = a;
        a = R[m];
    }
    while (m < n && b <= r) {
        ++m;
        a = b;
        b = R[m + 1];
    }
    const float y0 = __builtin_fmaf((float) m, 0.5f, 0.1f);
    const float w  = b - a;
    const float E1 = w == 0.0f ? y0 : y0 + q_div((r - a) * ((y0 + 0.5f) - y0), w);
    const float te = q_te_max(rel);
    const float Te = te >= at_least(0.08511) ? 0.08511f : te;
    const float  O = q_div(units::two_pi_re2_mc2_h2o * rho, units::water_density) * L_w;
    const double g = __builtin_fma((double) rel.beta_sq, -0.5, 1.0) * (double) q_div(Te, rel.beta_sq);
    const float  O_sq = (float) (g * (double) O);
    return fabsf(__builtin_fmaf(c.rng.st_z0, q_sqrt(O_sq), Ek - E1));
}

// along_step (mqi_p_ionization.hpp:348-420) from the step's sp * len
template<bool DBG>
MQI_DI void q_along_step(ctx& c, trk& t, float len, float rho, float sp) {
    MQI_NO_CONTRACT
    const q_rel rel = q_relq(t.ke0);
    const float L_w = q_div(len * sp * rho, units::water_density);
    const float dE  = q_energy_loss(c, rel, t.ke0, rho, L_w);
    float       r   = 1.0f;
    if (dE >= t.ke0) {
        r         = r_div(t.ke0, dE);
        t.stopped = true;
    }
    const float q     = q_div(13.9f, q_sqrt(rel.pp));
    const float th_sq = q_div(q_div(q * q, rel.beta_sq) * len, q_radiation_length<DBG>(rho));
    const float th    = fabsf(c.rng.st_z1 * (0x1.6a09e6p+0f * q_sqrt(th_sq)));   // sqrt(2)
    const float phi   = (float) (2.0 * 3.14159265358979323846 * (double) c.rng.st_u1);
    t.d1 = q_turn(q_align<false, false>(t.d1), th, phi);
    t.dE = __builtin_fmaf(dE, r, t.dE);
    update_pos(t, r * len);
    t.ke1 = __builtin_fmaf(-dE, r, t.ke1);
}

#endif

// secondary placement: pos -> fwd (pos - T) + T, dir -> fwd dir (e.g.
// mqi_pp_elastic.hpp:190-196), with the transform of the child the track is
// in.  In the patient (P.fwd, P.trans) at the push; a secondary made in a
// beamline child is stored unplaced with the child's index and placed with
// that child's transform when it is popped (the same operations, so the same
// bits), which keeps the beamline transforms out of the physics.
MQI_DI v3 place(const transport_params& P, v3 p) {
    MQI_NO_CONTRACT
    v3 q = mk(p.x - P.trans[0], p.y - P.trans[1], p.z - P.trans[2]);
    q    = mv(P.fwd, q);
    return mk(q.x + P.trans[0], q.y + P.trans[1], q.z + P.trans[2]);
}
MQI_DI v3 turn(const transport_params& P, v3 d) { return mv(P.fwd, d); }
// the same with a child's transform (fwd[9], inv[9], translation[3]) in HBM
MQI_DI v3 place_xf(const float* f, v3 p) {
    MQI_NO_CONTRACT
    v3 q = mv(f, mk(p.x - f[18], p.y - f[19], p.z - f[20]));
    return mk(q.x + f[18], q.y + f[19], q.z + f[20]);
}

// track_stack_t::push_secondary: dropped when the stack is full (mqi_track_stack.hpp:36-41).
// A pushed track keeps vtx0, vtx1.ke and dE; vtx1 position/direction are
// overwritten when it is popped, local_dE is always zero, status is CREATED.
// The lane's stack (P.stack_cap entries in HBM) is addressed from the launch
// at the few pushes and pops, not from a pointer held through the loop.
MQI_DI float* stack_entry(const transport_params& P, int k) {
    const uint64_t tid = (uint64_t) blockIdx.x * blockDim.x + threadIdx.x;
    return P.stack + (tid * (uint32_t) P.stack_cap + (uint32_t) k) * MQI_STACK_FLOATS;
}
MQI_DI void push(const transport_params& P, ctx& c, float ke0, v3 p0, v3 d0, float ke1, float dE, float tag) {
    if (c.sp < P.stack_cap) {
        float* s = stack_entry(P, c.sp);
        s[0]     = ke0;
        s[1]     = p0.x;
        s[2]     = p0.y;
        s[3]     = p0.z;
        s[4]     = d0.x;
        s[5]     = d0.y;
        s[6]     = d0.z;
        s[7]     = ke1;
        s[8]     = dE;
        s[9]     = tag;
        ++c.sp;
    } else {
        ++c.drops;
    }
}

// push a daughter made at (p, d) in the current child
MQI_DI void push_placed(const transport_params& P, ctx& c, float ke0, v3 p, v3 d, float ke1, float dE) {
    if (c.child < c.nbl)
        push(P, c, ke0, p, d, ke1, dE, (float) c.child);
    else
        push(P, c, ke0, place(P, p), turn(P, d), ke1, dE, -1.0f);
}

#if MQI_EXACT
// p_ionization_tabulated::post_step: delta-ray (mqi_p_ionization.hpp:424-477)
template<bool DBG>
MQI_DI void post_ion(const transport_params& P, ctx& c, trk& t) {
    rel_q       rel   = relq(t.ke1);
    const float T_cut = DBG ? 0.08511 * 1.0 : 0.0815 * 1.0;
    float       Te, n;
    // acceptance probability is above 1/2 for any finite energy; the bound
    // only ends the loop for non-finite input (which the reference would spin on)
    for (int it = 0; it < 4096; ++it) {
        n  = c.rng.uniform();
        Te = T_cut * rel.Te_max;
        Te /= ((1.0 - n) * rel.Te_max + n * T_cut);
        const float acc = c.rng.uniform();
        if (acc < 1.0 - rel.beta_sq * Te / rel.Te_max + Te * Te / (2.0 * rel.Et_sq)) break;
    }
    if (DBG) {
        push_placed(P, c, 0.0f, t.p0, t.d0, 0.0f, Te);
    } else {
        t.dE += Te;
    }
    t.ke1 -= Te;
}
#else
// p_ionization_tabulated::post_step: delta-ray (mqi_p_ionization.hpp:424-477).
// The first trial's numbers come from the interaction's block; the later
// ones (acceptance is above 1/2) from the history's stream.
template<bool DBG>
MQI_DI void post_ion(const transport_params& P, ctx& c, trk& t) {
    MQI_NO_CONTRACT
    const q_rel  rel    = q_relq(t.ke1);
    const float  te_max = q_te_max(rel);
    const float  T_cut  = DBG ? 0.08511 * 1.0 : 0.0815 * 1.0;
    const double num    = (double) (T_cut * te_max);
    const double temd   = (double) te_max;
    const float  rte    = __builtin_amdgcn_rcpf(te_max);
    const double e2     = 2.0 * (double) rel.Et_sq;
    const double re2    = d_recip(e2);
    float        n = c.rng.it_u1, acc = c.rng.it_u2, Te;
    // the bound only ends the loop for non-finite input
    for (int it = 0;; ++it) {
        const double den = __builtin_fma(1.0 - (double) n, temd, (double) (n * T_cut));
        Te               = (float) d_quot(num, den, d_recip(den));
        const double a   = 1.0 - (double) (rel.beta_sq * Te * rte);
        if ((double) acc < a + d_quot((double) (Te * Te), e2, re2) || it == 4095) break;
        c.rng.pair(n, acc);
    }
    if (DBG) {
        push_placed(P, c, 0.0f, t.p0, t.d0, 0.0f, Te);
    } else {
        t.dE += Te;
    }
    t.ke1 -= Te;
}
#endif

#if MQI_EXACT
// pp_elastic_tabulated::post_step (mqi_pp_elastic.hpp:119-219)
template<bool DBG>
MQI_DI void post_pp(const transport_params& P, ctx& c, trk& t) {
    rel_q rel       = relq(t.ke1);
    float min_value = 0.5f / rel.Ek;
    float r0, r1;
    c.rng.pair(r0, r1);
    float u         = r0 * (1.0 - 2.0 * min_value) + min_value;
    float E1        = rel.Et;
    float dE        = rel.Ek * u;
    float E3        = (rel.Ek - dE) + units::Mp;
    float E4        = dE + units::Mp;
    float P1        = momentum(rel);
    float P3        = MQ_SQRTF(E3 * E3 - units::Mp_sq);
    float P4        = MQ_SQRTF(E4 * E4 - units::Mp_sq);
    float cos_th3   = E1 * E3 - units::Mp_sq - units::Mp * (E1 - E3);
    cos_th3 /= (P1 * P3);
    float cos_th34 = E3 * E4 - E1 * units::Mp;
    cos_th34 /= (P3 * P4);
    if (cos_th3 > 1.0)
        cos_th3 = 1.0;
    else if (cos_th3 < -1.0)
        cos_th3 = -1.0;
    if (cos_th34 > 1.0)
        cos_th34 = 1.0;
    else if (cos_th34 < -1.0)
        cos_th34 = -1.0;
    float th3 = MQ_ACOSF(cos_th3);
    float th4 = th3 - MQ_ACOSF(cos_th34);
    float phi = 2.0 * 3.14159265358979323846 * r1;
    t.ke1 -= dE;
    rotate_direction(t.d1, th3, phi);
    v3 dd = t.d1;
    rotate_direction(dd, th4, phi);
    push_placed(P, c, dE, t.p1, dd, dE, 0.0f);
}

// po_elastic::post_step (mqi_po_elastic.hpp:96-217); exponential not truncated (CPU semantics)
template<bool DBG>
MQI_DI void post_poe(const transport_params& P, ctx& c, trk& t) {
    rel_q rel = relq(t.ke1);
    if (rel.Ek <= 5.5f) {
        float dE = rel.Ek;
        if (DBG)
            push_placed(P, c, dE, t.p1, t.d1, 0.0f, dE);
        else
            t.ldE += dE;
        t.ke1 -= dE;
        t.stopped = true;
    } else {
        float Tp_avg = 0.65 * MQ_EXPD(-0.0013 * rel.Ek);
        Tp_avg -= 0.71 * MQ_EXPD(-0.0177 * rel.Ek);
        float Tp_max = (2.0 * units::Mo * rel.beta_sq * rel.gamma_sq);
        Tp_max /= (1.0 + 2.0 * rel.gamma * units::MoMp + units::MoMp_sq);
        (void) Tp_max;
        float avg     = (float) (1.0 / Tp_avg);
        float uu, u1;
        c.rng.pair(uu, u1);
        float dE      = -MQ_LOGF(uu) / avg;
        float E1      = rel.Ek * (rel.Ek + 2.0 * units::Mp);
        float E3      = (rel.Ek - dE) * (rel.Ek - dE + 2.0 * units::Mp);
        float cos_th3 = (E1 + E3 - dE * (dE + 2.0 * units::Mo)) / 2.0 / MQ_SQRTF(E1 * E3);
        if (cos_th3 > 1.0) cos_th3 = 1.0;
        if (cos_th3 < -1.0) cos_th3 = -1.0;
        float th3 = MQ_ACOSF(cos_th3);
        float phi = 2.0 * 3.14159265358979323846 * u1;
        if (DBG)
            push_placed(P, c, dE, t.p0, t.d0, 0.0f, dE);
        else
            t.ldE += dE;
        t.ke1 -= dE;
        rotate_direction(t.d1, th3, phi);
    }
}

// po_inelastic_tabulated::post_step (mqi_po_inelastic.hpp:158-288)
template<bool DBG>
MQI_DI void post_poi(const transport_params& P, ctx& c, trk& t) {
    const float Ek = t.ke1;
    float       Eb = 5.0f;
    float       Er = Ek;
    const float E_mini = 2.0f, E_ratio = 0.65f;
    float       Prob_2nd, Prob_long, power;
    if (Ek <= 215 && Ek > 200) {
        Prob_2nd  = 0.78f;
        Prob_long = Prob_2nd + (1 - Prob_2nd) * 0.9;
        power     = 0.4f;
    } else if (Ek > 215) {
        Prob_2nd  = 0.78f;
        Prob_long = Prob_2nd + (1 - Prob_2nd) * 1.0;
        power     = 0.4f;
    } else if (Ek <= 200 && Ek > 150) {
        Prob_2nd  = 0.72f;
        Prob_long = Prob_2nd + (1 - Prob_2nd) * 0.83;
        power     = 0.45f;
    } else {
        Prob_2nd  = 0.7f;
        Prob_long = Prob_2nd + (1 - Prob_2nd) * 0.83;
        power     = 0.52f;
    }
    while ((Er - Eb) > E_mini) {
        Er -= Eb;
        float u, zeta;
        c.rng.pair(u, zeta);
        float dE = MQ_POWF(u, power) * (Er - E_mini) + E_mini;
        if (dE >= Er) dE = Er;
        Er -= dE;
        t.ke1 -= dE + Eb;
        if (zeta < Prob_2nd) {
            float r0, r1;
            c.rng.pair(r0, r1);
            float cos_th = (2.0 * dE / Ek - 1.0) + 2.0 * (1 - dE / Ek) * r0;
            if (cos_th < -1) cos_th = -1;
            if (cos_th > 1) cos_th = 1;
            float th  = MQ_ACOSF(cos_th);
            float phi = 2.0 * 3.14159265358979323846 * r1;
            v3    dd  = t.d1;
            rotate_direction(dd, th, phi);
            push_placed(P, c, dE, t.p1, dd, dE, 0.0f);
        } else if (zeta < Prob_long) {
            // long-range energy leaves the track
        } else if (DBG) {
            push_placed(P, c, dE, t.p0, t.d0, 0.0f, dE);
        }
        Eb *= E_ratio;
    }
    t.dE += Er;
    t.ke1 -= Er;
    t.stopped = true;
}
#else
// pp_elastic_tabulated::post_step (mqi_pp_elastic.hpp:119-219)
template<bool DBG>
MQI_DI void post_pp(const transport_params& P, ctx& c, trk& t) {
    MQI_NO_CONTRACT
    const float Mp = units::Mp, Ek = t.ke1;
    const q_rel rel = q_relq(Ek);
    float       r0, r1;
    c.rng.pair(r0, r1);
    const double mv_ = (double) q_div(0.5f, Ek);
    const float  u   = (float) __builtin_fma(__builtin_fma(mv_, -2.0, 1.0), (double) r0, mv_);
    const float  E1 = rel.Et, dE = Ek * u, Ek1 = __builtin_fmaf(-Ek, u, Ek);
    const float  E3 = Ek1 + Mp, E4 = dE + Mp;
    const float  P1 = q_sqrt(rel.pp);
    const float  P3 = q_sqrt(__builtin_fmaf(E3, E3, -units::Mp_sq));
    const float  P4 = q_sqrt(__builtin_fmaf(E4, E4, -units::Mp_sq));
    float cos_th3  = q_div(__builtin_fmaf(-Mp, E1 - E3, __builtin_fmaf(E1, E3, -units::Mp_sq)), P1 * P3);
    float cos_th34 = q_div(__builtin_fmaf(E4, E3, -(Mp * E1)), P4 * P3);
    if (cos_th3 > 1.0f)
        cos_th3 = 1.0f;
    else if (cos_th3 < -1.0f)
        cos_th3 = -1.0f;
    if (cos_th34 > 1.0f)
        cos_th34 = 1.0f;
    else if (cos_th34 < -1.0f)
        cos_th34 = -1.0f;
    const float th3 = MQ_ACOSF(cos_th3);
    const float th4 = th3 - MQ_ACOSF(cos_th34);
    const float phi = (float) (2.0 * 3.14159265358979323846 * (double) r1);
    t.ke1           = Ek1;
    t.d1            = q_turn(q_align<false, true>(t.d1), th3, phi);
    const v3 dd     = q_turn(q_align<false, false>(t.d1), th4, phi);
    push_placed(P, c, dE, t.p1, dd, dE, 0.0f);
}

// po_elastic::post_step (mqi_po_elastic.hpp:96-217); exponential not truncated (CPU semantics)
template<bool DBG>
MQI_DI void post_poe(const transport_params& P, ctx& c, trk& t) {
    MQI_NO_CONTRACT
    const float Ek = t.ke1;
    if (Ek <= 5.5f) {
        if (DBG)
            push_placed(P, c, Ek, t.p1, t.d1, 0.0f, Ek);
        else
            t.ldE += Ek;
        t.ke1 -= Ek;
        t.stopped = true;
    } else {
        const double ek = (double) Ek;
        float        Tp_avg = (float) (0.65 * MQ_EXPD(-0.0013 * ek));
        Tp_avg              = (float) ((double) Tp_avg - 0.71 * MQ_EXPD(-0.0177 * ek));
        float uu, u1;
        c.rng.pair(uu, u1);
        const float  dE  = q_div(-q_log(uu), r_div(1.0f, Tp_avg));
        const float  Ek1 = Ek - dE;
        const double ek1 = (double) Ek1, de = (double) dE;
        const float  E1 = (float) ((ek + 2.0 * (double) units::Mp) * ek);
        const float  E3 = (float) ((ek1 + 2.0 * (double) units::Mp) * ek1);
        const double q  = (double) q_sqrt(E1 * E3);
        const double n  = __builtin_fma(-(de + 2.0 * (double) units::Mo), de, (double) (E1 + E3)) * 0.5;
        float        cos_th3 = (float) d_quot(n, q, d_recip(q));
        if (cos_th3 > 1.0f) cos_th3 = 1.0f;
        if (cos_th3 < -1.0f) cos_th3 = -1.0f;
        const float th3 = MQ_ACOSF(cos_th3);
        const float phi = (float) (2.0 * 3.14159265358979323846 * (double) u1);
        if (DBG)
            push_placed(P, c, dE, t.p0, t.d0, 0.0f, dE);
        else
            t.ldE += dE;
        t.ke1 = Ek1;
        t.d1  = q_turn(q_align<false, true>(t.d1), th3, phi);
    }
}

// po_inelastic_tabulated::post_step (mqi_po_inelastic.hpp:158-288)
template<bool DBG>
MQI_DI void post_poi(const transport_params& P, ctx& c, trk& t) {
    MQI_NO_CONTRACT
    const float Ek = t.ke1;
    float       Eb = 5.0f;
    float       Er = Ek;
    const float E_mini = 2.0f, E_ratio = 0.65f;
    float       Prob_2nd, Prob_long, power;
    if (Ek <= 215 && Ek > 200) {
        Prob_2nd  = 0.78f;
        Prob_long = Prob_2nd + (1 - Prob_2nd) * 0.9;
        power     = 0.4f;
    } else if (Ek > 215) {
        Prob_2nd  = 0.78f;
        Prob_long = Prob_2nd + (1 - Prob_2nd) * 1.0;
        power     = 0.4f;
    } else if (Ek <= 200 && Ek > 150) {
        Prob_2nd  = 0.72f;
        Prob_long = Prob_2nd + (1 - Prob_2nd) * 0.83;
        power     = 0.45f;
    } else {
        Prob_2nd  = 0.7f;
        Prob_long = Prob_2nd + (1 - Prob_2nd) * 0.83;
        power     = 0.52f;
    }
    float rest = Er - Eb;   // the energy left, less the next binding energy
    if (rest > E_mini) {
        // every daughter leaves from the same direction
        const q_mat  m  = q_align<true, true>(t.d1);
        const double ek = (double) Ek, rk = d_recip(ek);
        do {
            Er = rest;
            float u, zeta;
            c.rng.pair(u, zeta);
            float dE = __builtin_fmaf(Er - E_mini, MQ_POWF(u, power), E_mini);
            if (dE >= Er) dE = Er;
            Er -= dE;
            t.ke1 -= dE + Eb;
            if (zeta < Prob_2nd) {
                float r0, r1;
                c.rng.pair(r0, r1);
                const double a  = d_quot((double) dE + (double) dE, ek, rk) - 1.0;
                const double b  = (double) (1.0f - q_div(dE, Ek));
                float        cos_th = (float) __builtin_fma(b + b, (double) r0, a);
                if (cos_th < -1.0f) cos_th = -1.0f;
                if (cos_th > 1.0f) cos_th = 1.0f;
                const float th  = MQ_ACOSF(cos_th);
                const float phi = (float) (2.0 * 3.14159265358979323846 * (double) r1);
                push_placed(P, c, dE, t.p1, q_turn(m, th, phi), dE, 0.0f);
            } else if (zeta < Prob_long) {
                // long-range energy leaves the track
            } else if (DBG) {
                push_placed(P, c, dE, t.p0, t.d0, 0.0f, dE);
            }
            rest = __builtin_fmaf(-E_ratio, Eb, Er);
            Eb *= E_ratio;
        } while (rest > E_mini);
    }
    t.dE += Er;
    t.ke1 -= Er;
    t.stopped = true;
}
#endif

#if MQI_EXACT
// fippel_physics::stepping (mqi_fippel_physics.hpp:68-216).  The three
// branches' along_step calls are merged into one call with the branch's
// length; the random-number order is unchanged.  The stopping power ratio
// the reference evaluates at several points of a step (stepping,
// energy_loss, last_step, the dose hit) always has the arguments (rho,
// ke0 of the step): it is evaluated once and returned in sp for scoring.
template<bool DBG>
MQI_DI void stepping(ctx& c, trk& t, float rho, float d2b, float& sp) {
    sp = 0.0f;   // vacuum: the dose hit returns before reading it
    if (rho < 1.0e-7) {
        update_pos(t, d2b);
        return;
    } else if (rho > 99.9) {
        t.stopped = true;
        sp        = spr<DBG>(rho, t.ke0);
        return;
    }
    if (t.ke0 <= 0.5f) {
        if (t.ke0 < 0) t.ke0 = 0;
        sp = spr<DBG>(rho, t.ke0);
        t.dE += t.ke0;
        t.ke1 -= t.ke0;
        // last_step (mqi_p_ionization.hpp:481-490)
        rel_q rel = relq(t.ke0);
        float L_w = 0;
        if (t.dE > 0) L_w = -t.dE / dedx(c, rel.Ek);
        float step_length = L_w * units::water_density / (sp * rho);
        update_pos(t, step_length);
        t.stopped = true;
        return;
    }
    rel_q rel = relq(t.ke0);
    float cms = 1.0f;
    sp        = spr<DBG>(rho, rel.Ek);   // rel.Ek == t.ke0
    cms       = cms * sp * rho / units::water_density;
    float max_loss_energy = -1.0 * cms * dedx(c, rel.Ek);
    float cs1[4]  = { cs_ion(c, rel.Ek, rho), cs_tab(c, T_CS_PP, rel.Ek, rho), cs_tab(c, T_CS_POE, rel.Ek, rho),
                      cs_tab(c, T_CS_POI, rel.Ek, rho) };
    float cs1_sum = cs1[0] + cs1[1] + cs1[2] + cs1[3];
    rel_q rel_de  = relq(t.ke0 - max_loss_energy);
    float cs2[4]  = { cs_ion(c, rel_de.Ek, rho), cs_tab(c, T_CS_PP, rel_de.Ek, rho),
                      cs_tab(c, T_CS_POE, rel_de.Ek, rho), cs_tab(c, T_CS_POI, rel_de.Ek, rho) };
    float cs2_sum = cs2[0] + cs2[1] + cs2[2] + cs2[3];
    const bool first = cs1_sum >= cs2_sum;
    float cs_sum  = first ? cs1_sum : cs2_sum;
    float cs0 = first ? cs1[0] : cs2[0], csa = first ? cs1[1] : cs2[1], csb = first ? cs1[2] : cs2[2],
          csc = first ? cs1[3] : cs2[3];
    float prob       = c.rng.uniform();
    float mfp        = -1.0f * MQ_LOGF(prob) / cs_sum;
    float step_limit = cms * units::water_density / (sp * rho);
    int   br;
    float len;
    if (d2b < mfp && d2b < step_limit) {
        br  = 0;
        len = d2b;
    } else if ((mfp < d2b || fabsf(mfp - d2b) < 1e-3f) &&
               (mfp < step_limit || fabsf(mfp - step_limit) < 1e-3f)) {
        br  = 1;
        len = mfp;
    } else {
        br  = 2;
        len = step_limit;
    }
    along_step<DBG>(c, t, len, rho, sp);
    if (br != 1) return;
    if (t.ke1 <= 0.5f) return;
    float u = cs_sum * c.rng.uniform();
    t.d1    = t.d0;
    if (u < cs0) {
        post_ion<DBG>(cold(), c, t);
    } else if (u < (cs0 + csa)) {
        post_pp<DBG>(cold(), c, t);
    } else if (u < (cs0 + csa + csb)) {
        post_poe<DBG>(cold(), c, t);
    } else if (u < (cs0 + csa + csb + csc)) {
        post_poi<DBG>(cold(), c, t);
    }
}
#else
// The same with the step's common terms formed once (mqi_prod.hpp): one
// stopping power ratio for every kind of step, both energies' cross sections
// from shared table indices.
template<bool DBG>
MQI_DI void stepping(ctx& c, trk& t, float rho, float d2b, float& sp) {
    MQI_NO_CONTRACT
    if (rho < at_least(1.0e-7)) {
        sp = 0.0f;   // vacuum: the dose hit returns before reading it
        update_pos(t, d2b);
        return;
    }
    const bool block = rho > at_most(99.9);
    if (!block && t.ke0 < 0) t.ke0 = 0;
    sp = q_spr<DBG>(rho, t.ke0);
    if (block) {
        t.stopped = true;
        return;
    }
    if (t.ke0 <= 0.5f) {
        t.dE += t.ke0;
        t.ke1 -= t.ke0;
        // last_step (mqi_p_ionization.hpp:481-490)
        float L_w = 0;
        if (t.dE > 0) {
            float pw;
            q_cross<true>(c.T, t.ke0, &pw);
            L_w = geo_div(t.dE, pw);
        }
        update_pos(t, q_div(L_w * units::water_density, sp * rho));
        t.stopped = true;
        return;
    }
    const float sr  = sp * rho;
    const float cms = q_div(sr, units::water_density);
    float       pw;
    const q_cs  c1   = q_cross<true>(c.T, t.ke0, &pw);
    const q_cs  c2   = q_cross<false>(c.T, t.ke0 - cms * pw, nullptr);
    const float sum1 = q_sum(c1, rho), sum2 = q_sum(c2, rho);
    const bool  first  = sum1 >= sum2;
    const float cs_sum = first ? sum1 : sum2;
    const float ion = first ? c1.ion : c2.ion, pp = first ? c1.pp : c2.pp, poe = first ? c1.poe : c2.poe,
                poi = first ? c1.poi : c2.poi;
    c.rng.begin_step();
    const float mfp        = q_div(-q_log(c.rng.st_u0), cs_sum);
    const float step_limit = q_div(cms * units::water_density, sr);
    float       len        = step_limit;
    bool        interact   = false;
    if (d2b < mfp && d2b < step_limit) {
        len = d2b;
    } else if ((mfp < d2b || fabsf(mfp - d2b) < 1e-3f) &&
               (mfp < step_limit || fabsf(mfp - step_limit) < 1e-3f)) {
        len      = mfp;
        interact = true;
    }
    q_along_step<DBG>(c, t, len, rho, sp);
    if (!interact || t.ke1 <= 0.5f) return;
    c.rng.begin_interaction();
    const float u  = cs_sum * c.rng.it_u0;
    const float s0 = rho * ion, s1 = s0 + rho * pp, s2 = s1 + rho * poe, s3 = s2 + rho * poi;
    t.d1           = t.d0;
    if (u < s0) {
        post_ion<DBG>(cold(), c, t);
    } else if (u < s1) {
        post_pp<DBG>(cold(), c, t);
    } else if (u < s2) {
        post_poe<DBG>(cold(), c, t);
    } else if (u < s3) {
        post_poi<DBG>(cold(), c, t);
    }
}
#endif

// ------------------------------------------------------------------ scoring
// hit functions (mqi_scorer_energy_deposit.hpp:43-139)
template<bool DBG>
MQI_DI double dose_hit(const trk& t, float density, float volume, float sp) {
    if (density < 1.0e-7) return 0.0;
#if MQI_EXACT
    return (t.dE + t.ldE) * 1.60218e-10 / (volume * density * sp);
#else
    // production: the per-step value in float (it is accumulated in FP64)
    return (double) ((t.dE + t.ldE) * 1.60218e-10f / (volume * density * sp));
#endif
}
// energy_deposit (:14-20); dose_to_medium of primaries in J/kg (:80-92)
MQI_DI double edep_hit(const trk& t) { return t.dE + t.ldE; }
MQI_DI double dm_hit(const trk& t, float density, float volume) {
    return t.primary ? t.dE * 1.60218e-13 * 1000.0 / (volume * density) : 0.0;
}
// step length and dE / length / density of the LETd and LETt scorers
// (LETd_weight1/2 :93-139, LETt_weight1/2 :141-177); false for no length.
// One square root and two divisions in FP64: formed once per step, and only
// for plans that score a LET (evaluated per scorer they were hoisted out of
// the scorers' branches and ran for every plan, 90 FP64 instructions a step).
MQI_DI bool let_terms(const trk& t, float density, double& length, double& let) {
    density *= 1000.0;
    length = (t.p1.x - t.p0.x) * (t.p1.x - t.p0.x);
    length += (t.p1.y - t.p0.y) * (t.p1.y - t.p0.y);
    length += (t.p1.z - t.p0.z) * (t.p1.z - t.p0.z);
#if MQI_EXACT
    length = MQ_SQRTD(length);
    if (length <= 0) return false;
    let = t.dE / length / density;
#else
    if (length <= 0) return false;
    length          = d_sqrt(length);
    const double dn = (double) density;
    let             = d_quot(d_quot((double) t.dE, length, d_recip(length)), dn, d_recip(dn));
#endif
    return true;
}

// Dij: per-spot open-addressing table of (voxel, dose) in HBM.  Keys are
// claimed with one 32-bit CAS, values added with FP64 atomics.  Linear
// probing stops after MQI_DIJ_MAX_PROBE slots (a table that full is an
// overflow: the run reports it instead of crawling through a full table).
#define MQI_DIJ_MAX_PROBE 4096
// A table's slots in groups of 32 for the 4 x 4 x 2 voxels of a block, so the
// keys of a block share a 128-byte line and its values two: the lanes of a
// spot work in the same few blocks.  A voxel's home is its place in the group
// that its block's number hashes to; on a conflict it tries its place in the
// next groups, then the slots behind its home one by one (a table smaller
// than a group has no groups).
#define MQI_DIJ_GROUP_PROBES 16
MQI_DI uint32_t dij_home(const transport_params& P, int cx, int cy, int cz, uint32_t groups) {
    const uint32_t nbx = (uint32_t) (P.nx + 3) >> 2, nby = (uint32_t) (P.ny + 3) >> 2;
    const uint32_t id  = ((uint32_t) (cz >> 1) * nby + (uint32_t) (cy >> 2)) * nbx + (uint32_t) (cx >> 2);
    const uint32_t g   = __umulhi(id * 2654435761u, groups);
    return g << 5 | (uint32_t) (cx & 3) | (uint32_t) (cy & 3) << 2 | (uint32_t) (cz & 1) << 4;
}
// A key changes once, from empty to its voxel, so a plain load that shows a
// voxel is final: the slot is ours, or taken by another voxel.  Only a load
// that shows it empty (possibly a stale cached line) needs the
// compare-and-swap, which is performed beyond the caches.
MQI_DI bool dij_claim(uint32_t* key, uint32_t voxel) {
    uint32_t k = *key;
    if (k == 0xffffffffu) k = atomicCAS(key, 0xffffffffu, voxel);
    return k == 0xffffffffu || k == voxel;
}
MQI_DI void dij_insert(const transport_params& P, uint32_t item, uint32_t voxel, double value) {
    if (value <= 0) return;
    const uint64_t base   = P.dij_off[item];
    const uint64_t cap    = P.dij_off[item + 1] - base;
    uint32_t*      keys   = P.dij_keys + base;
    double*        vals   = P.dij_vals + base;
    const uint32_t groups = (uint32_t) (cap >> 5), tries = groups ? MQI_DIJ_GROUP_PROBES : 0;
    const uint32_t last   = tries + (uint32_t) (cap < MQI_DIJ_MAX_PROBE ? cap : MQI_DIJ_MAX_PROBE);
    uint32_t       home   = 0;
    if (groups) {
        const uint32_t yz = voxel / (uint32_t) P.nx, cz = yz / (uint32_t) P.ny;
        home = dij_home(P, (int) (voxel - yz * (uint32_t) P.nx), (int) (yz - cz * (uint32_t) P.ny), (int) cz, groups);
    }
    uint32_t slot = home;
    for (uint32_t probe = 1; probe <= last; ++probe) {
        if (dij_claim(keys + slot, voxel)) {
            atomicAdd(vals + slot, value);
            return;
        }
        if (probe < tries)
            slot = slot >> 5 < groups - 1 ? slot + 32 : slot & 31;
        else if (probe == tries)
            slot = home;
        else
            slot = (uint64_t) slot + 1 < cap ? slot + 1 : 0;
    }
    atomicOr(P.status, MQI_STATUS_DIJ_FULL);
    if (P.dij_dose) atomicAdd(P.dij_dose + P.out_scenario_stride * (item / (uint32_t) P.n_spots) + voxel, value);
}

#if !MQI_EXACT
// Deposits whose slot the key loaded with the voxel's density did not show
// wait in their wave's queue in LDS until half of it may be in use, and then
// go into the tables side by side: a first touch, a conflict or a probe by
// one lane costs the other 63 nothing.  The lanes of a wave share the queue
// without barriers (LDS accesses of one wave are performed in order).
MQI_DI void wave_fence() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}
MQI_DI uint32_t lane_rank(unsigned long long m) {   // lanes of m below this one
    return __builtin_amdgcn_mbcnt_hi((uint32_t) (m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t) m, 0u));
}
MQI_DI void dij_defer(mqi_dij_queue* q, const mqi_dij_entry& e) {
    const unsigned long long m    = __ballot(1);
    const uint32_t           rank = lane_rank(m), at = q->n;
    wave_fence();
    q->e[at + rank] = e;
    if (rank == 0) q->n = at + (uint32_t) __popcll(m);
    wave_fence();
}
// The queue if it holds more than `keep` entries, by the lanes that are here;
// without a queue each lane's own deposit (voxel 0xffffffff: none).
MQI_DI void dij_drain(const transport_params& P, mqi_dij_queue* q, const mqi_dij_entry& own, uint32_t keep) {
    uint32_t i = 0, n = own.voxel != 0xffffffffu ? 1 : 0, step = 1;
    if (q) {
        const unsigned long long m = __ballot(1);
        n    = q->n;
        i    = lane_rank(m);
        step = (uint32_t) __popcll(m);
        if (n <= keep) return;
        wave_fence();
    }
    const bool first = i == 0;
    for (; i < n; i += step) {
        const mqi_dij_entry x = q ? q->e[i] : own;
        dij_insert(P, x.item, x.voxel, x.value);
    }
    if (q) {
        wave_fence();
        if (first) q->n = 0;
        wave_fence();
    }
}
#endif

// The launch's scoring as the loop's code reads it: two words, taken apart
// where a field is used (a compiler that sees the fields' comparisons before
// the history loop keeps each one's lane mask in a pair of scalar registers).
struct scoring {
    uint32_t kinds, mode;
    MQI_DI int  n() const { return mode & 7; }
    MQI_DI int  kind(int s) const { return kinds >> 4 * s & 15; }
    MQI_DI bool let() const { return mode & 8; }
    MQI_DI int  loops() const { return mode >> 4 & 3; }
    MQI_DI int  pair() const { return mode >> 6 & 7; }
    MQI_DI int  grouped() const { return mode >> 9 & 7; }
    MQI_DI int  dij_slot() const { return (int) (mode >> 12 & 15) - 1; }
    MQI_DI bool dij_deferred() const { return loops() == MQI_LOOPS_ONCE && (uint32_t) dij_slot() < MQI_DEFER; }
};
MQI_DI scoring scoring_of(const transport_params& P) {
    scoring S;
    S.kinds = P.kind_word;
    S.mode  = P.mode_word;
    asm volatile("" : "+s"(S.kinds), "+s"(S.mode));
    return S;
}

// Deposits of consecutive steps into the same voxel (and scenario, and Dij
// table) are summed per lane and added to the scorer arrays, or inserted
// into the Dij table, once, when the lane moves on (each-scorer-once scoring
// only; the sums differ from per-step atomics only in FP64 summation order).
// Scorer slots beyond MQI_DEFER are scored per step.  The sums live in the lane's LDS slots (v[s * blockDim.x]), not
// in registers: held across the loop they pushed the kernel into scratch,
// and every scratch reload waits on the one counter the atomics in flight
// also hold.
struct pending {
    int32_t  cnb;    // voxel of the pending sums, -1: none
    uint32_t scen;   // their scenario
    uint32_t item;   // their Dij table (scenario, spot)
#if !MQI_EXACT
    uint32_t key;    // what the voxel's home slot in that table showed
#endif
};
MQI_DI uint64_t pend_element(const transport_params& P, const pending& A) {
    return P.out_scenario_stride * A.scen + (uint32_t) A.cnb;
}

// accumulated slots are positive, +inf or NaN (every value that is not <= 0
// is added, NaN included); untouched slots are 0
MQI_DI void flush(const transport_params& P, const scoring& S, pending& A, double* v, mqi_dij_entry& own,
                  mqi_dij_queue* q) {
    if (A.cnb >= 0) {
        const uint64_t k  = pend_element(P, A);
        double         dx = 0.0;   // the Dij slot's sum: inserted behind the loop, from one place
#pragma unroll
        for (int s = 0; s < MQI_DEFER; ++s) {
            if (s >= S.n()) break;
            const double x = v[s * blockDim.x];
            if (s == S.dij_slot()) {
                dx = x;
            } else if (x != 0.0) {
#if !MQI_EXACT
                if (s < S.grouped())
                    atomicAdd(P.pair_out + (uint64_t) S.pair() * k + s, x);
                else
#endif
                    atomicAdd(P.out[s] + k, x);
            }
        }
        if (dx != 0.0) {
#if MQI_EXACT
            dij_insert(P, A.item, (uint32_t) A.cnb, dx);
#else
            if (q && A.key == (uint32_t) A.cnb) {
                atomicAdd(P.dij_vals + q->slot[__lane_id()], dx);
            } else {
                const mqi_dij_entry e = { (uint32_t) A.cnb, A.item, dx };
                if (q)
                    dij_defer(q, e);
                else
                    own = e;
            }
#endif
        }
    }
    A.cnb = -1;
}

#if !MQI_EXACT
// a lane's value from another lane of its group of four (DPP quad_perm: one
// instruction, no LDS round trip as ds_bpermute has); lanes that are not
// active read as `old`
template<int CTRL>
MQI_DI int quad_get(int old, int x) {
    return __builtin_amdgcn_update_dpp(old, x, CTRL, 0xf, 0xf, false);
}
template<int CTRL>
MQI_DI uint64_t quad_get(uint64_t x) {
    const uint32_t lo = (uint32_t) quad_get<CTRL>(0, (int) (uint32_t) x);
    const uint32_t hi = (uint32_t) quad_get<CTRL>(0, (int) (uint32_t) (x >> 32));
    return (uint64_t) hi << 32 | lo;
}
template<int CTRL>
MQI_DI double quad_get(double x) {
    return __longlong_as_double((long long) quad_get<CTRL>((uint64_t) __double_as_longlong(x)));
}
#define QUAD_XOR1 0xB1          // quad_perm [1, 0, 3, 2]
#define QUAD_XOR2 0x4E          // quad_perm [2, 3, 0, 1]
#define QUAD_OF(j) ((j) * 0x55) // quad_perm [j, j, j, j]

// The flush of the step with paired scoring, run by every lane that steps
// (f: this lane leaves its voxel).  Lanes 2m and 2m+1 exchange their sums:
// the first atomic instruction adds both of lane 2m's sums (scorer 0 from
// lane 2m, scorer 1 from lane 2m+1), the second both of lane 2m+1's, so the
// two adds of a voxel land in one line of the interleaved array in one
// instruction.  A lane whose partner does not step adds both of its own.
MQI_DI void flush_pair(const transport_params& P, pending& A, double* v, bool f) {
    const bool     has  = f && A.cnb >= 0;
    const double   a    = has ? v[0] : 0.0;
    const double   b    = has ? v[blockDim.x] : 0.0;
    const uint64_t k    = 2 * (has ? pend_element(P, A) : 0);
    const bool     pact = quad_get<QUAD_XOR1>(0, 1) != 0;
    const uint64_t kp   = quad_get<QUAD_XOR1>(k);
    const double   ap   = quad_get<QUAD_XOR1>(a);
    const double   bp   = quad_get<QUAD_XOR1>(b);
    const bool     odd  = __lane_id() & 1;
    const bool     swA = pact && odd, swB = pact && !odd;
    const uint64_t eA = swA ? kp + 1 : k, eB = swB ? kp : k + 1;
    const double   xA = swA ? bp : a, xB = swB ? ap : b;
    if (xA != 0.0) atomicAdd(P.pair_out + eA, xA);
    if (xB != 0.0) atomicAdd(P.pair_out + eB, xB);
    if (has) A.cnb = -1;
}

// lanes q and q ^ D of each group exchange halves of (x, y): the even lane
// keeps its x and gets the other's x as y, the odd one the reverse
template<int CTRL>
MQI_DI void quad_swap(bool up, double& x, double& y) {
    const double t = quad_get<CTRL>(up ? x : y);
    if (up)
        x = t;
    else
        y = t;
}

// The same for three or four grouped scorers (interleaved four doubles per
// element): in a group of four stepping lanes, instruction j adds the sums of
// lane 4m+j's voxel, lane 4m+q adding that lane's sum of scorer q, so all of
// a voxel's sums go out as one line request (the sums are transposed within
// the group in two exchanges).  Lanes of a group with a lane that does not
// step add their own sums.
MQI_DI void flush_quad(const transport_params& P, const scoring& S, pending& A, double* v, bool f) {
    const bool     has = f && A.cnb >= 0;
    double         x0  = has ? v[0] : 0.0;
    double         x1  = has ? v[blockDim.x] : 0.0;
    double         x2  = has ? v[2 * blockDim.x] : 0.0;
    double         x3  = (has && S.grouped() > 3) ? v[3 * blockDim.x] : 0.0;
    const uint64_t k   = 4 * (has ? pend_element(P, A) : 0);
    const int      q   = __lane_id() & 3;
    const int      all = quad_get<QUAD_OF(0)>(0, 1) & quad_get<QUAD_OF(1)>(0, 1) & quad_get<QUAD_OF(2)>(0, 1) &
                    quad_get<QUAD_OF(3)>(0, 1);
    if (all) {
        const bool u1 = q & 1, u2 = q & 2;
        quad_swap<QUAD_XOR1>(u1, x0, x1);
        quad_swap<QUAD_XOR1>(u1, x2, x3);
        quad_swap<QUAD_XOR2>(u2, x0, x2);
        quad_swap<QUAD_XOR2>(u2, x1, x3);
        // x_j: scorer q of lane 4m+j
        const uint64_t k0 = quad_get<QUAD_OF(0)>(k), k1 = quad_get<QUAD_OF(1)>(k), k2 = quad_get<QUAD_OF(2)>(k),
                       k3 = quad_get<QUAD_OF(3)>(k);
        if (x0 != 0.0) atomicAdd(P.pair_out + k0 + q, x0);
        if (x1 != 0.0) atomicAdd(P.pair_out + k1 + q, x1);
        if (x2 != 0.0) atomicAdd(P.pair_out + k2 + q, x2);
        if (x3 != 0.0) atomicAdd(P.pair_out + k3 + q, x3);
    } else if (has) {
        if (x0 != 0.0) atomicAdd(P.pair_out + k, x0);
        if (x1 != 0.0) atomicAdd(P.pair_out + k + 1, x1);
        if (x2 != 0.0) atomicAdd(P.pair_out + k + 2, x2);
        if (x3 != 0.0) atomicAdd(P.pair_out + k + 3, x3);
    }
#if MQI_DEFER > MQI_GROUP
    // the scorers behind the group, each into its own array
    if (has) {
#pragma unroll
        for (int s = MQI_GROUP; s < MQI_DEFER; ++s) {
            if (s >= S.n()) break;
            const double x = v[s * blockDim.x];
            if (x != 0.0) atomicAdd(P.out[s] + (k >> 2), x);
        }
    }
#endif
    if (has) A.cnb = -1;
}
#endif

template<bool DBG>
MQI_DI void score(const transport_params& P, const scoring& S, const trk& t, uint32_t cnb, float density, float volume, float sp,
                  uint32_t dij_item, uint32_t scen, pending& A, double* pv) {
    const int n = S.n();
    // regular scorers score through roi_->idx(cnb) > 0, the statistics pair
    // through get_mask_idx(cnb) >= 0 (mqi_transport.hpp:342-364), under
    // roi_t DIRECT every voxel but 0 and every voxel; a CONTOUR ROI's answer
    // per voxel is in roi_flags
    const uint32_t fl      = P.roi_flags ? (uint32_t) P.roi_flags[cnb] : ((int32_t) cnb > 0 ? 3u : 2u);
    const bool     in_reg  = fl & 1u;
    const bool     in_stat = fl & 2u;
    const uint64_t k       = P.out_scenario_stride * scen + cnb;
    const double   d       = dose_hit<DBG>(t, density, volume, sp);
    // the deposits of a voxel the lane has just entered start from 0
    const bool fresh = (int32_t) cnb != A.cnb;
    double     length = 0.0, let = 0.0;
    bool       has_let = false;
    if (S.let()) has_let = let_terms(t, density, length, let);
    double dv = 0.0;   // the Dij scorer's value and repeats when it is not deferred
    int    dr = 0;
    // The loop runs over the fixed maximum with constant indices so that the
    // scorer table stays in kernel arguments / registers (a runtime index
    // into it would move the whole argument block to private memory).
#pragma unroll
    for (int s = 0; s < MQI_MAX_SCORERS; ++s) {
        if (s >= n) break;
        const int kind = S.kind(s);
        double    v    = d;
        if (kind == MQI_KIND_STAT_DOSE2) {
            v = d * d;
        } else if (S.let() && kind != MQI_KIND_DOSE) {
            if (kind == MQI_KIND_LETD_NUM)
                v = (!has_let || let >= 25.0) ? 0.0 : t.dE * let;
            else if (kind == MQI_KIND_LETD_DEN)
                v = (!has_let || let >= 25.0) ? 0.0 : (double) t.dE;
            else if (kind == MQI_KIND_LETT_NUM)
                v = has_let ? length * let : 0.0;
            else if (kind == MQI_KIND_LETT_DEN)
                v = has_let ? length : 0.0;
        }
        if (kind == MQI_KIND_EDEP)
            v = edep_hit(t);
        else if (kind == MQI_KIND_DM)
            v = dm_hit(t, density, volume);
        const bool stat = (kind == MQI_KIND_STAT_DOSE || kind == MQI_KIND_STAT_DOSE2);
        if (S.loops() == MQI_LOOPS_ONCE && s < MQI_DEFER) {
            double*      acc = pv + s * blockDim.x;
            const double o   = fresh ? 0.0 : *acc;
            *acc             = (!(stat ? in_stat : in_reg) || v <= 0) ? o : o + v;
            continue;
        }
        int reps = 0;
        if (S.loops() == MQI_LOOPS_ONCE) {
            reps = (stat ? in_stat : in_reg) ? 1 : 0;
        } else if (S.loops() == MQI_LOOPS_PLAIN) {
            // mqi_transport.hpp:204-225: scorers 0..n-3 in both loops
            reps = in_reg ? ((s < n - 2) ? 2 : 1) : 0;
        } else {
            // mqi_transport.hpp:343-364: last two through get_mask_idx >= 0
            if (s < n - 2)
                reps = in_reg ? 1 : 0;
            else if (n >= 2)
                reps = in_stat ? 1 : 0;
        }
        if (v <= 0) continue;
        if (kind == MQI_KIND_DIJ) {
            dv = v;
            dr = reps;
            continue;
        }
        for (int r = 0; r < reps; ++r) atomicAdd(P.out[s] + k, v);
    }
    // one insert site for every slot and loop
    for (int r = 0; r < dr; ++r) dij_insert(P, dij_item, cnb, dv);
    if (S.loops() == MQI_LOOPS_ONCE) {
        A.cnb  = (int32_t) cnb;
        A.scen = scen;
        A.item = dij_item;
    }
}

// ------------------------------------------------------------------ lane machine
struct lane {
    trk      t;
    bool     active;
    uint32_t item;       // work item (spot of a scenario) of the current history
    uint64_t hist;       // history index within the item
    uint64_t g;          // history index in the flattened list
    int      nsteps;     // trace mode: steps logged for this history
    float    scale;      // scenario density scale
    uint32_t scen;       // scenario
    uint32_t dij_item;   // Dij table of (scenario, spot): scenario * n_spots + spot
    int      tsteps;     // steps of the current track
    pending  acc;        // deferred deposits of the current voxel
    bool     newhist;    // the first step of a history: the pending deposits are another one's
    bool     reenter;    // left a beamline child: enter the next child
};

// pop + enter the child grid: transport loop head (mqi_transport.hpp:158-191)
MQI_DI bool enter(const transport_params& P, ctx& c, trk& t) {
    MQI_NO_CONTRACT
    v3 pp = mk(t.p0.x - P.trans[0], t.p0.y - P.trans[1], t.p0.z - P.trans[2]);
    t.p0  = mv(P.inv, pp);
    t.d0  = mv(P.inv, t.d0);
    normalize(t.d0);
    t.p1 = t.p0;
    t.d1 = t.d0;
    int cx, cy, cz;
    index3(c.g, t.p0, t.d0, cx, cy, cz);
    if (!is_valid(c.g, cx, cy, cz)) {
        int   ox, oy, oz;
        float dist = intersect_out(c.g, t.p0, t.d0, ox, oy, oz);
        t.its      = dist;
        if (dist < 0) return false;
        update_pos(t, dist);
        move(t);
        index3(c.g, t.p0, t.d0, t.cx, t.cy, t.cz);
    } else {
        t.its = 0.0f;
        t.cx  = cx;
        t.cy  = cy;
        t.cz  = cz;
    }
    return is_valid(c.g, t.cx, t.cy, t.cz) && !t.stopped;
}

// ------------------------------------------------------------------ beamline children
// The world's children are transported in order, the patient last
// (mqi_transport.hpp:158-240): the track goes into the child's frame, to its
// first voxel, steps until it leaves or stops, and back to the world frame
// (also when it misses the child) before the next child.  Beamline children
// have no scorers and no scenario shift or density scale; their edges sit in
// LDS after the patient's.
MQI_DI grid_view bl_view(const transport_params& P, const float* shb, int k) {
    const int* m = P.bl_meta + 8 * k;
    grid_view  g;
    g.nx = m[0];
    g.ny = m[1];
    g.nz = m[2];
    g.xe = shb + m[3];
    g.ye = g.xe + g.nx + 1;
    g.ze = g.ye + g.ny + 1;
    g.sx = g.sy = g.sz = 0.0f;
    return g;
}

// into child k's frame and to its first voxel (as enter() for the patient)
MQI_DI bool enter_bl(const transport_params& P, const grid_view& g, int k, trk& t) {
    MQI_NO_CONTRACT
    const float* f = P.bl_xf + 21 * k;
    v3           pp = mk(t.p0.x - f[18], t.p0.y - f[19], t.p0.z - f[20]);
    t.p0            = mv(f + 9, pp);
    t.d0            = mv(f + 9, t.d0);
    normalize(t.d0);
    t.p1 = t.p0;
    t.d1 = t.d0;
    int cx, cy, cz;
    index3(g, t.p0, t.d0, cx, cy, cz);
    if (!is_valid(g, cx, cy, cz)) {
        int   ox, oy, oz;
        float dist = intersect_out(g, t.p0, t.d0, ox, oy, oz);
        t.its      = dist;
        if (dist < 0) return false;
        update_pos(t, dist);
        move(t);
        index3(g, t.p0, t.d0, t.cx, t.cy, t.cz);
    } else {
        t.its = 0.0f;
        t.cx  = cx;
        t.cy  = cy;
        t.cz  = cz;
    }
    return is_valid(g, t.cx, t.cy, t.cz) && !t.stopped;
}

// back from child k's frame to the world: pos -> fwd pos + T, dir -> fwd dir
MQI_DI void leave_bl(const transport_params& P, int k, trk& t) {
    MQI_NO_CONTRACT
    const float* f = P.bl_xf + 21 * k;
    v3           q = mv(f, t.p0);
    t.p0           = mk(q.x + f[18], q.y + f[19], q.z + f[20]);
    t.d0           = mv(f, t.d0);
    t.p1 = t.p0;
    t.d1 = t.d0;
}

// the track (in the world frame) enters the first child it reaches from
// c.child on; false when it reaches none
MQI_DI bool enter_chain(const transport_params& P, ctx& c, trk& t, const float* shb) {
    while (c.child < c.nbl) {
        const grid_view g = bl_view(P, shb, c.child);
        if (enter_bl(P, g, c.child, t)) return true;
        leave_bl(P, c.child, t);
        ++c.child;
    }
    return enter(P, c, t);
}

MQI_DI void pop(const transport_params& P, ctx& c, trk& t) {
    --c.sp;
    const float* s = stack_entry(P, c.sp);
    t.ke0          = s[0];
    t.p0           = mk(s[1], s[2], s[3]);
    t.d0           = mk(s[4], s[5], s[6]);
    if (s[9] >= 0.0f) {   // made in beamline child s[9]: place it now
        const float* f = P.bl_xf + 21 * (int) s[9];
        t.p0           = place_xf(f, t.p0);
        t.d0           = mv(f, t.d0);
    }
    t.ke1          = s[7];
    t.dE           = s[8];
    t.ldE          = 0.0f;
    t.stopped      = false;
    t.primary      = false;
}

// Vertex of history h of item (scenario, spot): phsp_6d + norm_1d/const_1d
// beamlet, then rotation/translation (mqi_beamlet.hpp:81-90, mqi_phsp6d.hpp:62-79).
MQI_DI void sample_vertex(const transport_params& P, const mqi_spot& sp, uint32_t spot_id, uint32_t scenario,
                          uint64_t h, trk& t) {
    vertex_rng r;
    r.s.init(P.seed, (uint32_t) h, spot_id, scenario, mqi_rng::STREAM_VERTEX);
    float Ux, Vx, Uy, Vy, Uz;
    if (sp.phsp == MQI_PHSP_UNIFORM) {   // U(-1, 1) draws (phsp_6d_uniform)
        Ux = 2.0f * r.uniform() - 1.0f;
        Vx = 2.0f * r.uniform() - 1.0f;
        Uy = 2.0f * r.uniform() - 1.0f;
        Vy = 2.0f * r.uniform() - 1.0f;
        Uz = 2.0f * r.uniform() - 1.0f;
    } else {
        Ux = r.gauss();
        Vx = r.gauss();
        Uy = r.gauss();
        Vy = r.gauss();
        Uz = r.gauss();
    }
    float ke = sp.energy;
    if (!sp.energy_const) {
        float z = r.gauss();
        ke      = z * sp.sigma_energy + sp.energy;
    }
    float ph[6];
    for (int k = 0; k < 6; ++k) ph[k] = sp.mean[k];
    ph[0] += sp.sigma[0] * Ux;
    ph[1] += sp.sigma[1] * Uy;
    ph[2] += sp.sigma[2] * Uz;
    const float rho0 = sp.corr[0], rho1 = sp.corr[1];
    ph[3] += sp.sigma[3] * (rho0 * Ux + Vx * MQ_SQRTD(1.0 - rho0 * rho0));
    ph[4] += sp.sigma[4] * (rho1 * Uy + Vy * MQ_SQRTD(1.0 - rho1 * rho1));
    ph[5]  = -1.0 * MQ_SQRTD(1.0 - ph[3] * ph[3] - ph[4] * ph[4]);
    v3 pos = mv(sp.rotation, mk(ph[0], ph[1], ph[2]));
    t.p0   = mk(pos.x + sp.translation[0], pos.y + sp.translation[1], pos.z + sp.translation[2]);
    t.d0   = mv(sp.rotation, mk(ph[3], ph[4], ph[5]));
    t.ke0  = ke;
    t.ke1  = ke;
    t.p1   = t.p0;
    t.d1   = t.d0;
    t.dE   = 0;
    t.ldE  = 0;
    t.stopped = false;
    t.primary = true;
}

// history g of the flattened work list -> (item, history-in-item)
MQI_DI void locate(const transport_params& P, uint64_t g, uint32_t& item, uint64_t& h) {
    int lo = 0, hi = P.n_items - 1;   // first item with item_end > g
    while (lo < hi) {
        int mid = (lo + hi) >> 1;
        if (P.item_end[mid] > g)
            hi = mid;
        else
            lo = mid + 1;
    }
    item = (uint32_t) lo;
    h    = g - (lo ? P.item_end[lo - 1] : 0);
}

MQI_DI void trace_record(const transport_params& P, lane& L, uint64_t cnb) {
    // per-history slots: history index g of the flattened list
    const uint64_t g = L.g;
    if (L.nsteps < P.trace_cap) {
        const uint64_t k = g * P.trace_cap + L.nsteps;
        P.trace_cnb[k]   = (int64_t) cnb;
        float* r         = P.trace_rec + 12 * k;
        r[0]             = L.t.its;
        r[1]             = L.t.p0.x;
        r[2]             = L.t.p0.y;
        r[3]             = L.t.p0.z;
        r[4]             = L.t.d0.x;
        r[5]             = L.t.d0.y;
        r[6]             = L.t.d0.z;
        r[7]             = L.t.p1.x;
        r[8]             = L.t.p1.y;
        r[9]             = L.t.p1.z;
        r[10]            = L.t.ke0;
        r[11]            = L.t.dE;
    }
    L.nsteps++;
    P.trace_n[g] = L.nsteps;
}

// one voxel-loop iteration (mqi_transport.hpp:192-233), in the patient or
// in a beamline child (no scoring there; leaving it hands the track to the
// next child).  One stepping call site serves both.
template<bool DBG, bool TRACE>
MQI_DI void step(const transport_params& P, ctx& c, lane& L, const float* shb, double* pv, mqi_dij_queue* q) {
    trk&       t  = L.t;
    const bool bl = c.child < c.nbl;
    uint64_t   cnb;
    float      rho;
    // a track starts its step where it stands (said here so that the end point
    // is not kept beside the start from one step to the next)
    t.p1 = t.p0;
    t.d1 = t.d0;
    if (bl) {
        // the beamline child's grid view is rebuilt after stepping rather
        // than kept live across it (register pressure of the patient path)
        const transport_params& B  = cold();
        const grid_view         gb = bl_view(B, shb, c.child);
        const int*              m  = B.bl_meta + 8 * c.child;
        const uint64_t off = (uint64_t) (uint32_t) m[4] | ((uint64_t) (uint32_t) m[5] << 32);
        cnb                = (uint64_t) (int32_t) (t.cz * gb.nx * gb.ny + t.cy * gb.nx + t.cx);
        t.its              = MQI_VOXEL_EXIT(gb, t.p0, t.d0, t.cx, t.cy, t.cz);
        rho                = B.bl_density[off + cnb];
    } else {
        cnb              = (uint64_t) (int32_t) (t.cz * c.g.nx * c.g.ny + t.cy * c.g.nx + t.cx);
        const float dens = P.density[cnb];
        const scoring S  = scoring_of(P);
#if !MQI_EXACT
        // the voxel's home in the spot's Dij table: its key, read now, is
        // looked at when the lane leaves the voxel
        uint64_t home = 0;
        uint32_t key  = 0xffffffffu;
        if (q) {
            const uint32_t groups = q->groups[__lane_id()];
            if (groups) {
                home = q->base[__lane_id()] + dij_home(P, t.cx, t.cy, t.cz, groups);
                key  = P.dij_keys[home];
            }
        }
#endif
        t.its            = MQI_VOXEL_EXIT(c.g, t.p0, t.d0, t.cx, t.cy, t.cz);
        rho              = dens * L.scale;
        // The deposits gathered in the voxel the lane has left go out here,
        // after the wait for the density and ahead of the physics of the
        // step: one counter tracks loads, stores and atomics alike, so atomics
        // issued just before the next wait on a load would add their round
        // trip to every step.
        // (A history's deposits are its own scenario's and Dij table's.)
        const bool leave = S.loops() == MQI_LOOPS_ONCE && ((int32_t) cnb != L.acc.cnb || L.newhist);
        L.newhist        = false;
#if !MQI_EXACT
        if (S.pair() == 2)
            flush_pair(P, L.acc, pv, leave);
        else if (S.pair() == 4)
            flush_quad(P, S, L.acc, pv, leave);
        else
#endif
        {
            mqi_dij_entry own = { 0xffffffffu, 0, 0.0 };
            if (leave) flush(P, S, L.acc, pv, own, q);
#if !MQI_EXACT
            if (S.dij_deferred()) dij_drain(cold(), q, own, MQI_DIJ_QUEUE - 64);
#endif
        }
#if !MQI_EXACT
        if (q) {
            q->slot[__lane_id()] = home;
            L.acc.key            = key;
        }
#endif
    }
    float sp;   // stopping power ratio of the step
    stepping<DBG>(c, t, rho, t.its, sp);
    if (bl) {
        const transport_params& B     = cold();
        const grid_view         gb    = bl_view(B, shb, c.child);
        bool                    leave = t.its < 0;
        if (!leave && !t.stopped) {
            t.cx += step_cell(t.p1.x, t.d1.x, gb.X(t.cx), gb.X(t.cx + 1));
            t.cy += step_cell(t.p1.y, t.d1.y, gb.Y(t.cy), gb.Y(t.cy + 1));
            t.cz += step_cell(t.p1.z, t.d1.z, gb.Z(t.cz), gb.Z(t.cz + 1));
            move(t);
            leave = !is_valid(gb, t.cx, t.cy, t.cz);
        }
        if (t.stopped) {
            // a stopped track does nothing in the children after this one
            L.active = false;
        } else if (leave) {
            leave_bl(B, c.child, t);
            ++c.child;
            L.reenter = true;
        }
        if (++L.tsteps > MQI_MAX_TRACK_STEPS && L.active) {
            L.active = false;
            atomicOr(cold().status, MQI_STATUS_TRACK_CAP);
        }
        return;
    }
    if (t.its < 0) {
        L.active = false;
        return;
    }
    // the voxel's edges: its volume and the cell after the step.
    // get_volume(cnb) (mqi_grid3d.hpp:471-487) goes through cnb2ijk; the
    // lane's cell indices are that (i, j, k) already
    const float x0 = c.g.X(t.cx), x1 = c.g.X(t.cx + 1);
    const float y0 = c.g.Y(t.cy), y1 = c.g.Y(t.cy + 1);
    const float z0 = c.g.Z(t.cz), z1 = c.g.Z(t.cz + 1);
    if (TRACE) {
        trace_record(P, L, cnb);
    } else {
        float vol = x1 - x0;
        vol *= y1 - y0;
        vol *= z1 - z0;
        score<DBG>(P, scoring_of(P), t, (uint32_t) cnb, rho, vol, sp, L.dij_item, L.scen, L.acc, pv);
    }
    if (!t.stopped) {
        t.cx += step_cell(t.p1.x, t.d1.x, x0, x1);
        t.cy += step_cell(t.p1.y, t.d1.y, y0, y1);
        t.cz += step_cell(t.p1.z, t.d1.z, z0, z1);
        move(t);
    }
    L.active = is_valid(c.g, t.cx, t.cy, t.cz) && !t.stopped;
    // a finite track takes a few thousand steps at most; the cap only ends
    // tracks whose state went non-finite
    if (++L.tsteps > MQI_MAX_TRACK_STEPS && L.active) {
        L.active = false;
        atomicOr(cold().status, MQI_STATUS_TRACK_CAP);
    }
}

// LDS staging of the tables and edges
MQI_DI void stage(const transport_params& P, float* sh) {
    for (int i = threadIdx.x; i < 600; i += blockDim.x) {
        sh[T_CS_ION + i] = kCsPIon[i];
        sh[T_DEDX + i]   = kDedxRestricted[i];
        sh[T_RANGE + i]  = kRangeSteps[i];
        sh[T_CS_PP + i]  = kCsPPElastic[i];
        sh[T_CS_POE + i] = kCsPOElastic[i];
        sh[T_CS_POI + i] = kCsPOInelastic[i];
    }
    float* xe = sh + T_TABLES;
    float* ye = xe + P.nx + 1;
    float* ze = ye + P.ny + 1;
    for (int i = threadIdx.x; i <= P.nx; i += blockDim.x) xe[i] = P.xe[i];
    for (int i = threadIdx.x; i <= P.ny; i += blockDim.x) ye[i] = P.ye[i];
    for (int i = threadIdx.x; i <= P.nz; i += blockDim.x) ze[i] = P.ze[i];
    float* blx = ze + P.nz + 1;
    for (int i = threadIdx.x; i < P.bl_n_edges; i += blockDim.x) blx[i] = P.bl_edges[i];
    __syncthreads();
}

// The transport kernel.  DYNAMIC: histories from the device counter
// (batched persistent form); otherwise each thread takes a contiguous slice
// [start, start+len) of the work list (plain form; start_and_length,
// mqi_utils.hpp:138-147).
// W > 0 asks the register allocator for at least W resident waves per SIMD
// (more memory latency hidden, at the price of spills past the budget).
template<bool DBG, bool DYNAMIC, bool TRACE, int W>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(W > 0 ? W : 1)))
k_transport(transport_params P) {
    extern __shared__ float sh[];
    stage(P, sh);
    ctx c;
    c.T     = sh;
    c.g.nx  = P.nx;
    c.g.ny  = P.ny;
    c.g.nz  = P.nz;
    c.g.xe  = sh + T_TABLES;
    c.g.ye  = c.g.xe + P.nx + 1;
    c.g.ze  = c.g.ye + P.ny + 1;
    c.sp    = 0;
    c.drops = 0;
    c.child = 0;
    c.nbl   = P.n_bl;
#if !MQI_EXACT
    c.rng.set_seed(P.seed);
#endif
    const float* shb = c.g.ze + P.nz + 1;   // beamline edges in LDS
    // the lane's pending deposit sums (MQI_DEFER doubles, blockDim.x apart),
    // after the beamline edges at an 8-byte boundary
    double* pv = reinterpret_cast<double*>(sh + mqi_pend_offset(P.nx, P.ny, P.nz, P.bl_n_edges)) + threadIdx.x;
#pragma unroll
    for (int s = 0; s < MQI_DEFER; ++s) pv[s * blockDim.x] = 0.0;
    mqi_dij_queue* q = nullptr;   // the wave's, if the launch has room for them
#if !MQI_EXACT
    if (P.dij_queued) {
        q = reinterpret_cast<mqi_dij_queue*>(pv - threadIdx.x + MQI_DEFER * blockDim.x) + (threadIdx.x >> 6);
        q->n = 0;
    }
#endif
    const uint64_t tid      = (uint64_t) blockIdx.x * blockDim.x + threadIdx.x;
    const uint64_t nthreads = (uint64_t) gridDim.x * blockDim.x;

    // plain: the thread's start_and_length slice; dynamic: the lane's current
    // chunk of P.fetch_chunk consecutive histories from the device counter
    uint64_t s_next = 0, s_end = 0;
    if (!DYNAMIC) {   // start_and_length over the flattened list
        const uint64_t q = P.total / nthreads, r = P.total % nthreads;
        s_next           = q * tid + (tid < r ? tid : r);
        s_end            = s_next + q + (tid < r ? 1 : 0);
    }
    lane     L;
    L.active = false;
    L.item   = 0;
    L.hist   = 0;
    L.nsteps   = 0;
    L.scale    = 1.0f;
    L.scen     = 0;
    L.dij_item = 0;
    L.acc.cnb  = -1;
    L.acc.scen = 0;
    L.acc.item = 0;
#if !MQI_EXACT
    L.acc.key = 0xffffffffu;
#endif
    L.newhist  = false;
    L.reenter  = false;
    c.g.sx = c.g.sy = c.g.sz = 0.0f;
    uint32_t           done = 0, nstep = 0;
    uint32_t           scen = 0;
    const uint64_t     hoff = P.hist_offset ? *P.hist_offset : 0;
    int                qx   = 0;   // work range this wave fetches from (dynamic form)
    if (DYNAMIC) {
        unsigned xcc;
        asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID)" : "=s"(xcc));
        qx = (int) (xcc & (MQI_QUEUES - 1));
    }

    for (;;) {
        // A lane whose history and secondaries are done takes a new history.
        // With refill_lanes > 1 (dynamic form) it first waits until that
        // many lanes of its wave need one, so the wave runs the new-history
        // path (sampling, work-list search, grid entry) once for all of
        // them; with no lane left to step it refills at once.
        const bool need   = !L.active && c.sp == 0;
        bool       refill = need;
        if (DYNAMIC && P.refill_lanes > 1) {
            const unsigned long long nm   = __ballot(need);
            const unsigned long long busy = __ballot(!need);
            refill = need && (__popcll(nm) >= (unsigned) P.refill_lanes || busy == 0);
        }
        if (need && !refill) continue;
        if (refill) {
            const transport_params& C = cold();
            uint64_t                g;
            if (DYNAMIC) {
                if (s_next >= s_end) {
                    // Wave-aggregated fetch of fetch_chunk histories per dry
                    // lane from range qx (initially this XCD's own range; a
                    // range that runs dry sends the wave to the next one).
                    const uint64_t chunk = (uint64_t) C.fetch_chunk;
                    const int      me    = __lane_id();
                    bool           got   = false;
                    for (int r = 0; r < MQI_QUEUES; ++r) {
                        const unsigned long long m = __ballot(!got);
                        if (m == 0) break;
                        const int          lead = __builtin_ctzll(m);
                        const int          rank = __popcll(m & ((1ull << me) - 1ull));
                        // the leader's range for every lane (lanes that were
                        // busy during earlier fetches may hold a stale qx)
                        const int          q    = __shfl(qx, lead);
                        unsigned long long base = 0;
                        if (me == lead)
                            base = atomicAdd(C.queue + q * MQI_QUEUE_STRIDE, (unsigned long long) __popcll(m) * chunk);
                        base               = __shfl(base, lead);
                        const uint64_t end = mqi_range_begin(C.total, q + 1);
                        if (!got) {
                            const uint64_t s0 = base + rank * chunk;
                            if (s0 < end) {
                                s_next = s0;
                                s_end  = s0 + chunk < end ? s0 + chunk : end;
                                got    = true;
                            }
                        }
                        // a range that could not serve every lane is dry: move on
                        qx = (__ballot(!got) != 0) ? ((q + 1) & (MQI_QUEUES - 1)) : q;
                    }
                    if (!got) break;
                }
                g = s_next++;
            } else {
                if (s_next >= s_end) break;
                g = s_next++;
            }
            L.g = g;
            uint32_t spot_id;
            if (C.vertices) {
                // caller-made vertex (upload_vertices path); scenario 0
                spot_id  = C.vertex_spot ? C.vertex_spot[g] : 0;
                L.item   = spot_id;
                L.hist   = g;
                scen     = 0;
            } else {
                locate(C, g, L.item, L.hist);
                spot_id = C.item_spot[L.item];
                scen    = C.item_scenario[L.item];
            }
            c.g.sx                 = C.scen_shift ? C.scen_shift[3 * scen] : 0.0f;
            c.g.sy                 = C.scen_shift ? C.scen_shift[3 * scen + 1] : 0.0f;
            c.g.sz                 = C.scen_shift ? C.scen_shift[3 * scen + 2] : 0.0f;
            L.scale                = C.scen_scale ? C.scen_scale[scen] : 1.0f;
            L.scen                 = scen;
            L.dij_item             = scen * (uint32_t) C.n_spots + spot_id;
            L.newhist              = true;
#if !MQI_EXACT
            if (q) {
                const uint64_t b        = C.dij_off[L.dij_item];
                q->base[__lane_id()]    = b;
                q->groups[__lane_id()]  = (uint32_t) ((C.dij_off[L.dij_item + 1] - b) >> 5);
            }
#endif
            if (C.vertices) {
                const float* v = C.vertices + 7 * g;
                L.t.ke0        = v[0];
                L.t.p0         = mk(v[1], v[2], v[3]);
                L.t.d0         = mk(v[4], v[5], v[6]);
                L.t.ke1        = L.t.ke0;
                L.t.p1         = L.t.p0;
                L.t.d1         = L.t.d0;
                L.t.dE         = 0;
                L.t.ldE        = 0;
                L.t.stopped    = false;
                L.t.primary    = true;
            } else {
                sample_vertex(C, C.spots[spot_id], spot_id, scen, L.hist + hoff, L.t);
            }
#if MQI_EXACT
            c.rng.init(C.seed, (uint32_t) (L.hist + hoff), spot_id, scen);
#else
            c.rng.init((uint32_t) (L.hist + hoff), spot_id, scen);
#endif
            L.nsteps = 0;
            L.tsteps = 0;
            ++done;
            c.child   = 0;
            L.reenter = true;
        } else if (!L.active) {
            pop(cold(), c, L.t);
            L.tsteps  = 0;
            c.child   = 0;
            L.reenter = true;
        }
        // a new or popped track, or one that left a beamline child, enters
        // the next child it reaches (one call site for all three)
        if (L.reenter) {
            L.reenter = false;
            L.active  = enter_chain(cold(), c, L.t, shb);
            if (!L.active) continue;
        }
        step<DBG, TRACE>(P, c, L, shb, pv, q);
        ++nstep;
    }
    mqi_dij_entry own = { 0xffffffffu, 0, 0.0 };
    flush(P, scoring_of(P), L.acc, pv, own, q);
#if !MQI_EXACT
    if (scoring_of(P).dij_deferred()) dij_drain(cold(), q, own, 0);
#endif
    atomicAdd(cold().tracked, (unsigned long long) done);
    atomicAdd(cold().steps, (unsigned long long) nstep);
    if (c.drops) atomicAdd(cold().drops, (unsigned long long) c.drops);
}

namespace
{
using launch_fn = void (*)(const transport_params&, int, int, size_t, hipStream_t);

struct variant {
    launch_fn   launch;
    const void* fn;
};

template<bool D, bool Y, bool T, int W>
void launch_one(const transport_params& P, int blocks, int threads, size_t shmem, hipStream_t stream) {
    hipLaunchKernelGGL((k_transport<D, Y, T, W>), dim3(blocks), dim3(threads), shmem, stream, P);
}

template<bool D, bool Y, bool T, int W>
variant make() {
    return {&launch_one<D, Y, T, W>, reinterpret_cast<const void*>(&k_transport<D, Y, T, W>)};
}

template<bool D, bool Y, bool T>
variant pick_waves(int waves) {
#if MQI_EXACT
    (void) waves;   // the verification kernels are not tuned
    return make<D, Y, T, 0>();
#else
    if (T) return make<D, Y, T, 0>();
    // by default the callers choose between 3 and 4 (the budgets without spills
    // in the step, 3 where it sums six scorers; 5 spills and is slower
    // everywhere), a caller's config any of them; 2: the compiler's own budget
    switch (waves) {
    case 2: return make<D, Y, T, 0>();
    case 4: return make<D, Y, T, 4>();
    case 5: return make<D, Y, T, 5>();
    case 6: return make<D, Y, T, 6>();
    case 8: return make<D, Y, T, 8>();
    default: return make<D, Y, T, 3>();
    }
#endif
}

variant pick(int debug, int dynamic, int trace, int waves) {
    if (debug) {
        if (dynamic) return trace ? pick_waves<true, true, true>(waves) : pick_waves<true, true, false>(waves);
        return trace ? pick_waves<true, false, true>(waves) : pick_waves<true, false, false>(waves);
    }
    if (dynamic) return trace ? pick_waves<false, true, true>(waves) : pick_waves<false, true, false>(waves);
    return trace ? pick_waves<false, false, true>(waves) : pick_waves<false, false, false>(waves);
}
}   // namespace

int
launch_transport(const transport_params& P, int debug, int dynamic, int trace, int waves, int blocks, int threads,
                 size_t shmem, hipStream_t stream) {
    pick(debug, dynamic, trace, waves).launch(P, blocks, threads, shmem, stream);
    return (int) hipGetLastError();
}

#if MQI_DEFER == MQI_GROUP
// Verification probes of the material and physics functions as the
// transport kernels evaluate them: fn 0 spr (rho, ek), fn 1 radiation length
// (rho), fn 2 per (rho, ek) the four cross sections at rho, dEdx and the
// relativistic quantities beta^2, gamma, Et, Te_max, momentum (10 floats).
template<bool DBG>
__global__ void __launch_bounds__(256) k_physics_probe(int fn, const float* rho, const float* ek, int64_t n, float* out) {
    __shared__ float sh[T_TABLES];
    for (int i = threadIdx.x; i < 600; i += blockDim.x) {
        sh[T_CS_ION + i] = kCsPIon[i];
        sh[T_DEDX + i]   = kDedxRestricted[i];
        sh[T_RANGE + i]  = kRangeSteps[i];
        sh[T_CS_PP + i]  = kCsPPElastic[i];
        sh[T_CS_POE + i] = kCsPOElastic[i];
        sh[T_CS_POI + i] = kCsPOInelastic[i];
    }
    __syncthreads();
    const int64_t i = (int64_t) blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    if (fn == 0) {
#if MQI_EXACT
        out[i] = spr<DBG>(rho[i], ek[i]);
#else
        out[i] = q_spr<DBG>(rho[i], ek[i]);
#endif
    } else if (fn == 1) {
#if MQI_EXACT
        out[i] = radiation_length<DBG>(rho[i]);
#else
        out[i] = q_radiation_length<DBG>(rho[i]);
#endif
    } else {
        float* o = out + 10 * i;
#if MQI_EXACT
        ctx c;
        c.T           = sh;
        const rel_q r = relq(ek[i]);
        o[0]          = cs_ion(c, r.Ek, rho[i]);
        o[1]          = cs_tab(c, T_CS_PP, r.Ek, rho[i]);
        o[2]          = cs_tab(c, T_CS_POE, r.Ek, rho[i]);
        o[3]          = cs_tab(c, T_CS_POI, r.Ek, rho[i]);
        o[4]          = dedx(c, r.Ek);
        o[5]          = r.beta_sq;
        o[6]          = r.gamma;
        o[7]          = r.Et;
        o[8]          = r.Te_max;
        o[9]          = momentum(r);
#else
        float       pw;
        const q_cs  c = q_cross<true>(sh, ek[i], &pw);
        const q_rel r = q_relq(ek[i]);
        o[0]          = c.ion * rho[i];
        o[1]          = c.pp * rho[i];
        o[2]          = c.poe * rho[i];
        o[3]          = c.poi * rho[i];
        o[4]          = -pw;
        o[5]          = r.beta_sq;
        o[6]          = q_div(r.Et, units::Mp);
        o[7]          = r.Et;
        o[8]          = q_te_max(r);
        o[9]          = q_sqrt(r.pp);
#endif
    }
}

int
physics_probe(int debug, int fn, const float* rho, const float* ek, int64_t n, float* out, hipStream_t stream) {
    if (n <= 0) return 0;
    const dim3 grid((unsigned) ((n + 255) / 256));
    if (debug)
        hipLaunchKernelGGL(k_physics_probe<true>, grid, dim3(256), 0, stream, fn, rho, ek, n, out);
    else
        hipLaunchKernelGGL(k_physics_probe<false>, grid, dim3(256), 0, stream, fn, rho, ek, n, out);
    return (int) hipGetLastError();
}

#if !MQI_EXACT
// Verification probe of the step's arithmetic (mqi_prod.hpp) as this build
// compiles it: fn 10 q_div, 11 q_sqrt, 12 q_log, 13 r_div (floats), 14 d_quot
// by d_recip, 15 d_sqrt (doubles), and what the build's own float division
// (16), square root (17) and logarithm (18) give.
__global__ void __launch_bounds__(256)
k_arith_probe(int fn, const double* x, const double* y, double* out, int64_t n) {
    const int64_t i = (int64_t) blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float a = (float) x[i], b = (float) y[i];
    double      r = 0.0;
    switch (fn) {
    case 10: r = (double) q_div(a, b); break;
    case 11: r = (double) q_sqrt(a); break;
    case 12: r = (double) q_log(a); break;
    case 13: r = (double) r_div(a, b); break;
    case 14: r = d_quot(x[i], y[i], d_recip(y[i])); break;
    case 15: r = d_sqrt(x[i]); break;
    case 16: r = (double) (a / b); break;
    case 17: r = (double) sqrtf(a); break;
    default: r = (double) logf(a); break;
    }
    out[i] = r;
}

int
arith_probe(int fn, const double* x, const double* y, double* out, int64_t n, hipStream_t stream) {
    if (n <= 0) return 0;
    hipLaunchKernelGGL(k_arith_probe, dim3((unsigned) ((n + 255) / 256)), dim3(256), 0, stream, fn, x, y, out, n);
    return (int) hipGetLastError();
}
#endif

#endif

// resident workgroups per CU of one instantiation
int
occupancy(int debug, int dynamic, int trace, int waves, int threads, size_t shmem) {
    int n = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, pick(debug, dynamic, trace, waves).fn, threads, shmem) !=
        hipSuccess)
        return 1;
    return n < 1 ? 1 : n;
}

}   // namespace MQI_NS
