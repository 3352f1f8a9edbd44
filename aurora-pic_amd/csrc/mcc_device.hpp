// mcc_device.hpp - device side of the null-collision MCC (FP32), shared by
// the standalone collide (mcc.hip), the 1D collision step (mcc.hip,
// ensemble.hip) and the batched swarm kernel (swarm.hip).
//
// Restates NullCollisionModel::collide (Collision.cpp:907-993) with
// collision_energy (579-594: projectile or centre-of-mass frame),
// rates_for_speed (596-625), the thermal frequency bound (627-685),
// apply_channel (738-829: attachment, resonant charge exchange, isotropic,
// backward and Henyey-Greenstein scattering, finite-mass elastic
// kinematics) and the ionization secondary (966-977).  Uniforms come from
// Philox4x32-10 in a fixed draw order, the order of the oracle's
// or_mcc_collide_3v.
//
// Everything is templated on the channel count NCH so per-channel rates and
// counters live in registers (fully unrolled loops); launch sites dispatch
// on the model's channel count with with_nchan().
#pragma once

#include <algorithm>
#include <cmath>

#include "aurora_internal.hpp"
#include "push_device.hpp"

namespace aurora {

constexpr int kMccLdsWords = 4096;  // FP32 table words staged in LDS (16 KiB)

enum : int { SCATTER_ISOTROPIC = 0, SCATTER_BACKWARD = 1, SCATTER_HENYEY_GREENSTEIN = 2 };

struct MccParams {
    int nchan;
    int kind[kMaxChannels];
    int angular[kMaxChannels];
    float threshold[kMaxChannels];
    float half_emass[kMaxChannels];  // half the collision-energy mass (projectile or reduced)
    int rows[kMaxChannels];
    int offset[kMaxChannels];
    int mc_rows[kMaxChannels];       // Henyey-Greenstein mean-cosine rows (0: none)
    int mc_offset[kMaxChannels];
    int shared_grid;         // every channel uses channel 0's energy grid and energy frame
    int grid_shared;         // every channel's energies equal channel 0's (one copy suffices)
    int total_rows;
    const float* energy;     // concatenated tables (global)
    const float* sigma;
    const float* mc_energy;  // concatenated mean-cosine tables (global)
    const float* mc_value;
    float neutral_density;
    float max_frequency;
    float inv_max_frequency;
    int max_candidates;
    float mass;
    float half_mass;
    float neutral_mass;      // 0: infinitely heavy neutral
    float neutral_vstd;      // 0: cold neutral
    float safe_speed;        // below it the rate bound is provably under max_frequency
    float safe_speed2;       // just under its square: the check is looked at only above
    uint32_t no_candidate;   // a step's first draws below this (of 2^23) hold no candidate
    // The 1D step books the kinetic energy of each ionization's secondary
    // and ion into the ionization channel (Simulation.cpp:880-902); half
    // their masses, 0 for the bare collide (NullCollisionModel::collide).
    float half_sec_mass;
    float half_ion_mass;
};

template <int NCH>
struct MccTally {
    uint32_t candidates;
    uint32_t nulls;
    uint32_t chan[NCH];
    float energy_change[NCH];
    int nsec;                // ionization events this call
    float sec[2][3];         // first two secondary velocities
    float ion[2][3];         // matching ion velocities
    uint32_t err;
};

// the counters alone (fixed-population swarms keep no products or energy
// ledger; the draws are the same)
template <int NCH>
struct MccCounts {
    uint32_t candidates;
    uint32_t nulls;
    uint32_t chan[NCH];
    uint32_t err;
};

// Host-side dispatch on the channel count: f.template operator()<NCH>().
template <typename F>
void with_nchan(int nchan, F&& f) {
    switch (nchan) {
        case 1: f.template operator()<1>(); break;
        case 2: f.template operator()<2>(); break;
        case 3: f.template operator()<3>(); break;
        case 4: f.template operator()<4>(); break;
        case 5: f.template operator()<5>(); break;
        case 6: f.template operator()<6>(); break;
        case 7: f.template operator()<7>(); break;
        default: f.template operator()<8>(); break;
    }
}

// with_nchan plus where the tables live: f.template operator()<NCH, LDS>().
template <typename F>
void with_model(int nchan, bool lds, F&& f) {
    with_nchan(nchan, [&]<int NCH>() {
        if (lds) f.template operator()<NCH, true>();
        else f.template operator()<NCH, false>();
    });
}

// First of n increasing energies at E + eo (LDS or global) that is above x
// (n: none).  (Three probes a step instead of one, so that half the reads wait
// for each other: no faster in the collide, 5 % slower in the swarm.)
__device__ __forceinline__ int xs_upper(const float* E, int eo, int n, float x) {
    int lo = 0, hi = n;
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (x < E[eo + mid]) hi = mid; else lo = mid + 1;
    }
    return lo;
}

// Linear interpolation with constant extrapolation (Collision.cpp:221-237,
// MeanCosineTable::evaluate 296-313) of the table whose n energies start at
// E + eo and values at S + so; up = xs_upper of x.
__device__ __forceinline__ float xs_at(const float* E, const float* S, int eo, int so, int n,
                                       int up, float x) {
    const int i0 = up > 0 ? up - 1 : 0, i1 = up < n ? up : n - 1;
    const float first = E[eo], e0 = E[eo + i0], e1 = E[eo + i1];
    const float s0 = S[so + i0], s1 = S[so + i1];
    const float f = (x - e0) / (e1 - e0);
    if (x <= first) return S[so];       // (rows may round to one FP32 energy)
    return i0 < i1 && up > 0 ? s0 + f * (s1 - s0) : s0;
}

// Cross-section tables as the kernels read them: E holds one energy grid
// for all channels when eshared (LDS staging of a shared grid), else the
// concatenated per-channel grids.
struct XsView {
    const float* E;
    const float* S;
    int eshared;
};

// collision energy of channel c at relative speed g (Collision.cpp:579-594)
__device__ __forceinline__ float collision_energy(const MccParams& m, int c, float g) {
    return m.half_emass[c] * g * g;
}

// per-channel rates n sigma(E) g for relative speed g; returns the total
template <int NCH>
__device__ __forceinline__ float mcc_rates(const MccParams& m, const XsView& X, float g,
                                           float* rate) {
    float total = 0.f;
    int up0 = -1;
    if (m.shared_grid) up0 = xs_upper(X.E, 0, m.rows[0], collision_energy(m, 0, g));
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
        const float e = collision_energy(m, c, g);
        float r = 0.f;
        if (e >= m.threshold[c]) {
            const int eo = X.eshared ? 0 : m.offset[c];
            const int up = m.shared_grid ? up0 : xs_upper(X.E, eo, m.rows[c], e);
            r = m.neutral_density * xs_at(X.E, X.S, eo, m.offset[c], m.rows[c], up, e) * g;
        }
        rate[c] = r;
        total += r;
    }
    return total;
}

__device__ __forceinline__ bool above_bound(const MccParams& m, float total) {
    // tolerance of 64 units of roundoff (Collision.cpp:617-623), FP32
    const float mx = total > m.max_frequency ? total : m.max_frequency;
    return total > m.max_frequency + 64.0f * 1.1920929e-7f * mx;
}

// Collision.cpp:627-685 for thermal neutrals: bound over the speed window.
// The largest cross section of the window is that of its ends and of the
// table rows inside it, found by two binary searches (the energies increase)
// instead of a pass over the whole table.
template <int NCH>
__device__ bool thermal_bound_exceeded(const MccParams& m, const XsView& X, float speed) {
    const float lim = 8.0f * m.neutral_vstd;
    const float vmax = speed + lim;
    float bound = 0.f;
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
        const float emax = collision_energy(m, c, vmax);
        if (emax < m.threshold[c]) continue;
        const float vmin = speed - lim > 0.f ? speed - lim : 0.f;
        float emin = collision_energy(m, c, vmin);
        if (emin < m.threshold[c]) emin = m.threshold[c];
        const int so = m.offset[c], eo = X.eshared ? 0 : so, n = m.rows[c];
        const int up0 = xs_upper(X.E, eo, n, emin), up1 = xs_upper(X.E, eo, n, emax);
        float best = xs_at(X.E, X.S, eo, so, n, up0, emin);
        const float smax = xs_at(X.E, X.S, eo, so, n, up1, emax);
        if (smax > best) best = smax;
        // rows with emin <= E <= emax (rows that round to one FP32 energy
        // are all looked at)
        int i = up0;
        while (i > 0 && X.E[eo + i - 1] >= emin) --i;
        for (; i < up1; ++i)
            if (X.S[so + i] > best) best = X.S[so + i];
        bound += m.neutral_density * best * vmax;
    }
    return above_bound(m, bound);
}

__device__ __forceinline__ void isotropic(float speed, Philox& rng, float* out) {
    // Collision.cpp:53-64
    const float cosine = 2.0f * rng.u01() - 1.0f;
    const float s2 = 1.0f - cosine * cosine;
    const float sine = sqrtf(s2 > 0.f ? s2 : 0.f);
    const float az = 6.28318530717958647692f * rng.u01();
    float sa, ca;
    sincosf(az, &sa, &ca);
    out[0] = speed * sine * ca;
    out[1] = speed * sine * sa;
    out[2] = speed * cosine;
}

// Henyey-Greenstein deflection of the relative velocity g0 (Collision.cpp:
// 66-134): inverse-CDF cosine for mean cosine mc, uniform azimuth about g0.
__device__ __forceinline__ void henyey_greenstein(const float* g0, float speed, float mc, Philox& rng,
                                  float* out) {
    const float inc = sqrtf(g0[0] * g0[0] + g0[1] * g0[1] + g0[2] * g0[2]);
    if (!(inc > 0.f)) {
        isotropic(speed, rng, out);
        return;
    }
    const float sample = rng.u01();
    float cosine = 2.0f * sample - 1.0f;
    if (mc != 0.f) {
        const float num = 1.0f - mc * mc;
        const float den = 1.0f - mc + 2.0f * mc * sample;
        const float ratio = num / den;
        cosine = (1.0f + mc * mc - ratio * ratio) / (2.0f * mc);
        cosine = fminf(fmaxf(cosine, -1.0f), 1.0f);
    }
    const float s2 = 1.0f - cosine * cosine;
    const float sine = sqrtf(s2 > 0.f ? s2 : 0.f);
    const float az = 6.28318530717958647692f * rng.u01();
    const float d[3] = {g0[0] / inc, g0[1] / inc, g0[2] / inc};
    const bool zaxis = fabsf(d[2]) < 0.9f;
    const float h[3] = {0.f, zaxis ? 0.f : 1.f, zaxis ? 1.f : 0.f};
    float t[3] = {h[1] * d[2] - h[2] * d[1], h[2] * d[0] - h[0] * d[2],
                  h[0] * d[1] - h[1] * d[0]};
    const float tn = sqrtf(t[0] * t[0] + t[1] * t[1] + t[2] * t[2]);
    t[0] /= tn;
    t[1] /= tn;
    t[2] /= tn;
    const float b[3] = {d[1] * t[2] - d[2] * t[1], d[2] * t[0] - d[0] * t[2],
                        d[0] * t[1] - d[1] * t[0]};
    float sa, ca;
    sincosf(az, &sa, &ca);
    const float tf = sine * ca, bf = sine * sa;
#pragma unroll
    for (int a = 0; a < 3; ++a) out[a] = speed * (cosine * d[a] + tf * t[a] + bf * b[a]);
}

// bounded Maxwellian neutral velocity: Box-Muller, rejected above 8 sigma
__device__ __forceinline__ void neutral_velocity(const MccParams& m, Philox& rng, float* w) {
    w[0] = w[1] = w[2] = 0.f;
    if (m.neutral_vstd == 0.f) return;
    const float lim = 8.0f * m.neutral_vstd;
    for (int attempt = 0; attempt < 1024; ++attempt) {
        const float u1 = rng.u01(), u2 = rng.u01(), u3 = rng.u01(), u4 = rng.u01();
        const float r1 = sqrtf(-2.0f * logf(u1)), r2 = sqrtf(-2.0f * logf(u3));
        float s1, c1, s2, c2;
        sincosf(6.28318530717958647692f * u2, &s1, &c1);
        sincosf(6.28318530717958647692f * u4, &s2, &c2);
        w[0] = m.neutral_vstd * r1 * c1;
        w[1] = m.neutral_vstd * r1 * s1;
        w[2] = m.neutral_vstd * r2 * c2;
        if (sqrtf(w[0] * w[0] + w[1] * w[1] + w[2] * w[2]) <= lim) return;
    }
}

// Parameters of one channel; the per-channel table lives in LDS so the
// accepted channel is read with a dynamic index without touching scratch.
struct ChannelSel {
    int kind;
    int angular;
    float threshold;
    float half_emass;
    int mc_offset;
    int mc_rows;
};

// apply_channel (Collision.cpp:738-829) for the accepted channel ch:
// relative velocity g (speed gs) against neutral velocity w
__device__ __forceinline__ void apply_channel(const MccParams& m, const ChannelSel& ch, float* v, const float* w,
                              const float* g, float gs, Philox& rng) {
    const int kind = ch.kind;
    if (kind == AURORA_ATTACHMENT) {
        v[0] = v[1] = v[2] = 0.f;
        return;
    }
    if (kind == AURORA_CHARGE_EXCHANGE) {
        v[0] = w[0];
        v[1] = w[1];
        v[2] = w[2];
        return;
    }
    float energy = m.half_mass * gs * gs;
    if (kind == AURORA_EXCITATION || kind == AURORA_IONIZATION) {
        energy -= ch.threshold;
        if (energy < 0.f) energy = 0.f;
    }
    if (kind == AURORA_IONIZATION) energy *= 0.5f;
    const float sp = sqrtf(energy / m.half_mass);
    float sc[3];
    if (ch.angular == SCATTER_BACKWARD) {
        sc[0] = -g[0];
        sc[1] = -g[1];
        sc[2] = -g[2];
    } else if (ch.angular == SCATTER_HENYEY_GREENSTEIN) {
        const float ec = ch.half_emass * gs * gs;     // collision_energy
        const int o = ch.mc_offset, n = ch.mc_rows;
        const float mc =
            xs_at(m.mc_energy, m.mc_value, o, o, n, xs_upper(m.mc_energy, o, n, ec), ec);
        henyey_greenstein(g, sp, mc, rng, sc);
    } else {
        isotropic(sp, rng, sc);
    }
    if (kind == AURORA_ELASTIC && m.neutral_mass > 0.f) {
        const float mt = m.mass + m.neutral_mass;
        const float rf = m.neutral_mass / mt;
        v[0] = (m.mass * v[0] + m.neutral_mass * w[0]) / mt + rf * sc[0];
        v[1] = (m.mass * v[1] + m.neutral_mass * w[1]) / mt + rf * sc[1];
        v[2] = (m.mass * v[2] + m.neutral_mass * w[2]) / mt + rf * sc[2];
    } else {
        v[0] = w[0] + sc[0];
        v[1] = w[1] + sc[1];
        v[2] = w[2] + sc[2];
    }
}

// validate_frequency_bound before a waiting time (Collision.cpp:617-632):
// below safe_speed it cannot fail, so it is evaluated only above
template <int NCH>
__device__ __forceinline__ bool mcc_rate_fails(const MccParams& m, const XsView& X,
                                               const float* v) {
    const float speed = sqrtf(v[0] * v[0] + v[1] * v[1] + v[2] * v[2]);
    if (!(speed > m.safe_speed)) return false;
    if (m.neutral_vstd != 0.f) return thermal_bound_exceeded<NCH>(m, X, speed);
    float rate[NCH];
    return above_bound(m, mcc_rates<NCH>(m, X, speed, rate));
}

// The candidate loop of one particle-step, in two resumable pieces (the
// swarm kernel interleaves particles' candidates): mcc_next_candidate is the
// loop top -- the rate-bound checks at the current speed, then the next
// waiting time -- and returns true when another candidate falls inside the
// step; mcc_candidate handles that candidate and returns false when the
// particle stops colliding in this step (attachment, or an error in t.err).
template <int NCH, typename Tally>
__device__ __forceinline__ bool mcc_next_candidate(const MccParams& m, const XsView& X,
                                                   const float* v, float dt, Philox& rng,
                                                   float& elapsed, Tally& t) {
    if (mcc_rate_fails<NCH>(m, X, v)) {
        t.err = DEV_ERR_RATE;
        return false;
    }
    const float waiting = -logf(rng.u01()) * m.inv_max_frequency;
    if (!(waiting < dt - elapsed)) return false;
    elapsed += waiting;
    ++t.candidates;
    if (t.candidates > static_cast<uint32_t>(m.max_candidates)) {
        t.err = DEV_ERR_CANDIDATES;
        return false;
    }
    return true;
}

template <int NCH, typename Tally>
__device__ __forceinline__ bool mcc_candidate(const MccParams& m, const XsView& X,
                                              const ChannelSel* chan, float* v, Philox& rng,
                                              Tally& t) {
    constexpr bool kLedger = requires { t.energy_change[0]; };
    float rate[NCH];
    float w[3];
    neutral_velocity(m, rng, w);
    const float g[3] = {v[0] - w[0], v[1] - w[1], v[2] - w[2]};
    const float gs = sqrtf(g[0] * g[0] + g[1] * g[1] + g[2] * g[2]);
    // rates at the relative speed (Collision.cpp:943-944); with a cold
    // neutral gs equals the speed checked above
    const float total = mcc_rates<NCH>(m, X, gs, rate);
    if (m.neutral_vstd != 0.f && above_bound(m, total)) {
        t.err = DEV_ERR_RATE;
        return false;
    }
    const float selection = rng.u01() * m.max_frequency;
    float cumulative = 0.f;
    int accepted = -1;
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
        cumulative += rate[c];
        if (accepted < 0 && selection < cumulative) accepted = c;
    }
    if (accepted < 0) {
        ++t.nulls;
        return true;
    }
    const int c = accepted;
    const ChannelSel ch = chan[c];
    const float e_before = m.half_mass * (v[0] * v[0] + v[1] * v[1] + v[2] * v[2]);
    apply_channel(m, ch, v, w, g, gs, rng);
    const float de = m.half_mass * (v[0] * v[0] + v[1] * v[1] + v[2] * v[2]) - e_before;
#pragma unroll
    for (int k = 0; k < NCH; ++k)
        if (k == c) {
            if constexpr (kLedger) t.energy_change[k] += de;
            ++t.chan[k];
        }
    if (ch.kind == AURORA_IONIZATION) {
        const float r0 = v[0] - w[0], r1 = v[1] - w[1], r2 = v[2] - w[2];
        float sec[3];
        isotropic(sqrtf(r0 * r0 + r1 * r1 + r2 * r2), rng, sec);
        if constexpr (!kLedger) return ch.kind != AURORA_ATTACHMENT;   // draws consumed
        else {
        const float s0 = w[0] + sec[0], s1 = w[1] + sec[1], s2 = w[2] + sec[2];
        if constexpr (requires { t.prod; }) {
            if (t.prod && t.nsec < 2) {
                float* d = t.prod + 6 * t.nsec;
                d[0] = s0;
                d[1] = s1;
                d[2] = s2;
#pragma unroll
                for (int a = 0; a < 3; ++a) d[3 + a] = w[a];
            }
        } else {
        // selects, not a store through a computed index (which would put the
        // tally in scratch memory)
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const bool here = t.nsec == k;
            t.sec[k][0] = here ? s0 : t.sec[k][0];
            t.sec[k][1] = here ? s1 : t.sec[k][1];
            t.sec[k][2] = here ? s2 : t.sec[k][2];
#pragma unroll
            for (int a = 0; a < 3; ++a) t.ion[k][a] = here ? w[a] : t.ion[k][a];
        }
        }
        ++t.nsec;
        if (m.half_sec_mass != 0.f) {
            const float added = m.half_sec_mass * (s0 * s0 + s1 * s1 + s2 * s2) +
                                m.half_ion_mass * (w[0] * w[0] + w[1] * w[1] + w[2] * w[2]);
#pragma unroll
            for (int k = 0; k < NCH; ++k)
                if (k == c) t.energy_change[k] += added;
        }
        }
    }
    return ch.kind != AURORA_ATTACHMENT;
}

template <int NCH>
__device__ __forceinline__ void mcc_tally_reset(MccTally<NCH>& t) {
    t.candidates = 0;
    t.nulls = 0;
#pragma unroll
    for (int c = 0; c < NCH; ++c) { t.chan[c] = 0; t.energy_change[c] = 0.f; }
    t.nsec = 0;
    t.err = 0;
}

template <int NCH>
__device__ __forceinline__ void mcc_tally_reset(MccCounts<NCH>& t) {
    t.candidates = 0;
    t.nulls = 0;
#pragma unroll
    for (int c = 0; c < NCH; ++c) t.chan[c] = 0;
    t.err = 0;
}

// One particle-step of null-collision MCC on velocity v (in place).
template <int NCH>
__device__ void mcc_collide(const MccParams& m, const XsView& X, const ChannelSel* chan, float* v,
                            float dt, Philox& rng, MccTally<NCH>& t) {
    mcc_tally_reset(t);
    if (!isfinite(v[0]) || !isfinite(v[1]) || !isfinite(v[2])) {
        t.err = DEV_ERR_NONFINITE;
        return;
    }
    float elapsed = 0.f;
    while (mcc_next_candidate<NCH>(m, X, v, dt, rng, elapsed, t))
        if (!mcc_candidate<NCH>(m, X, chan, v, rng, t)) break;
}

// bounded Maxwellian neutral velocity of the 1V collide: one normal from
// Box-Muller (u1, u2), rejected beyond 8 sigma (Collision.cpp:686-699)
__device__ __forceinline__ float neutral_velocity_1v(const MccParams& m, Philox& rng) {
    if (m.neutral_vstd == 0.f) return 0.f;
    const float lim = 8.0f * m.neutral_vstd;
    float w = 0.f;
    for (int attempt = 0; attempt < 1024; ++attempt) {
        const float u1 = rng.u01(), u2 = rng.u01();
        w = m.neutral_vstd * sqrtf(-2.0f * logf(u1)) * cosf(6.28318530717958647692f * u2);
        if (fabsf(w) <= lim) return w;
    }
    return w;
}

// One particle-step of the 1V null-collision MCC (Collision.cpp:831-905) on
// the scalar velocity v: the candidate loop of the 3V form on |v - w|, and
// apply_channel's 1V branch (Collision.cpp:717-760): attachment stops the
// particle, charge exchange takes the neutral's velocity, otherwise the
// speed after the energy loss is scattered forward or backward with equal
// probability (in the centre-of-mass frame for elastic channels with a
// neutral mass).  Ionization and anisotropic channels are 3V only; the host
// rejects them.
template <int NCH>
__device__ void mcc_collide_1v(const MccParams& m, const XsView& X, const ChannelSel* chan,
                               float& v, float dt, Philox& rng, MccTally<NCH>& t) {
    t.candidates = 0;
    t.nulls = 0;
#pragma unroll
    for (int c = 0; c < NCH; ++c) { t.chan[c] = 0; t.energy_change[c] = 0.f; }
    t.nsec = 0;
    t.err = 0;
    if (!isfinite(v)) {
        t.err = DEV_ERR_NONFINITE;
        return;
    }
    float elapsed = 0.f;
    float rate[NCH];
    for (;;) {
        const float speed = fabsf(v);
        if (m.neutral_vstd == 0.f) {
            if (speed > m.safe_speed && above_bound(m, mcc_rates<NCH>(m, X, speed, rate))) {
                t.err = DEV_ERR_RATE;
                return;
            }
        } else if (speed > m.safe_speed && thermal_bound_exceeded<NCH>(m, X, speed)) {
            t.err = DEV_ERR_RATE;
            return;
        }
        const float waiting = -logf(rng.u01()) * m.inv_max_frequency;
        if (!(waiting < dt - elapsed)) break;
        elapsed += waiting;
        ++t.candidates;
        if (t.candidates > static_cast<uint32_t>(m.max_candidates)) {
            t.err = DEV_ERR_CANDIDATES;
            return;
        }
        const float w = neutral_velocity_1v(m, rng);
        const float g = v - w;
        mcc_rates<NCH>(m, X, fabsf(g), rate);
        const float selection = rng.u01() * m.max_frequency;
        float cumulative = 0.f;
        int accepted = -1;
#pragma unroll
        for (int c = 0; c < NCH; ++c) {
            cumulative += rate[c];
            if (accepted < 0 && selection < cumulative) accepted = c;
        }
        if (accepted < 0) { ++t.nulls; continue; }
        const int c = accepted;
        const ChannelSel ch = chan[c];
        const float e_before = m.half_mass * v * v;
        if (ch.kind == AURORA_ATTACHMENT) {
            v = 0.f;
        } else if (ch.kind == AURORA_CHARGE_EXCHANGE) {
            v = w;
        } else {
            float energy = m.half_mass * g * g;
            if (ch.kind == AURORA_EXCITATION) {
                energy -= ch.threshold;
                if (energy < 0.f) energy = 0.f;
            }
            const float sp = sqrtf(energy / m.half_mass);
            const float scattered = rng.u01() < 0.5f ? -sp : sp;
            if (ch.kind == AURORA_ELASTIC && m.neutral_mass > 0.f) {
                const float mt = m.mass + m.neutral_mass;
                v = (m.mass * v + m.neutral_mass * w) / mt + (m.neutral_mass / mt) * scattered;
            } else {
                v = w + scattered;
            }
        }
        const float de = m.half_mass * v * v - e_before;
#pragma unroll
        for (int k = 0; k < NCH; ++k)
            if (k == c) {
                t.energy_change[k] += de;
                ++t.chan[k];
            }
        if (ch.kind == AURORA_ATTACHMENT) break;
    }
}

// The tallies of a launch without atomics: each lane adds up its particles',
// at the end the block's lanes are summed in a fixed order and one row per
// workgroup is stored: NCH energy sums (J, unweighted) at [0, NCH), then
// candidates, nulls, per-channel collisions and secondaries as integers at
// [kMaxChannels, kMaxChannels + NCH + 3), and the error bits.  The rows are
// added in row order, so counts are exact and energies repeat to the bit;
// and many waves never contend for one counter.
constexpr int kTallyStride = 2 * kMaxChannels + 4;
constexpr int kTallyErr = 2 * kMaxChannels + 3;

// A lane's tally: the counters of mcc_candidate, of which candidates, nsec
// and err are the current particle's (begin, finish) and the others sums.
// Products go to memory when they are made (prod: 2 x (secondary, ion), or
// null).  32 bits hold a lane's sums: its particles (2^32 / (64 waves) at
// most) times their candidates of the launch, each a chain of some hundred
// cycles, stay below 2^32 in any launch that ends within hours.
template <int NCH>
struct LaneTally {
    uint32_t candidates, nsec, err;
    float* prod;
    uint32_t nulls, chan[NCH];
    double energy_change[NCH];
    uint32_t all_candidates, all_nsec, all_err;
    __device__ __forceinline__ void begin(float* products) {
        candidates = nsec = err = 0u;
        prod = products;
    }
    __device__ __forceinline__ void finish() {
        all_candidates += candidates;
        all_nsec += nsec;
        all_err |= err;
    }
    __device__ __forceinline__ void add(const MccTally<NCH>& t) {
        all_candidates += t.candidates;
        all_nsec += static_cast<uint32_t>(t.nsec);
        all_err |= t.err;
        nulls += t.nulls;
#pragma unroll
        for (int c = 0; c < NCH; ++c) {
            chan[c] += t.chan[c];
            energy_change[c] += static_cast<double>(t.energy_change[c]);
        }
    }
};

// One row per workgroup (BLOCK threads, every thread calls it): the lanes'
// tallies summed per wave, the waves' in wave order, stored at
// rows + row * kTallyStride.
template <int NCH, int BLOCK>
__device__ __forceinline__ void store_block_row(const LaneTally<NCH>& t, double* rows,
                                                int64_t row) {
    constexpr int W = BLOCK / 64;
    __shared__ double se[W][NCH];
    __shared__ unsigned long long sc[W][NCH + 3];
    __shared__ uint32_t sx[W];
    const int wid = static_cast<int>(threadIdx.x) >> 6;
    const bool lead = (threadIdx.x & 63) == 0;
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
        const double e = wave_sum(t.energy_change[c]);
        if (lead) se[wid][c] = e;
    }
#pragma unroll
    for (int k = 0; k < NCH + 3; ++k) {
        const unsigned long long n = wave_sum_u64(k == 0         ? t.all_candidates
                                                  : k == 1       ? t.nulls
                                                  : k == NCH + 2 ? t.all_nsec
                                                                 : t.chan[k - 2 < NCH ? k - 2 : 0]);
        if (lead) sc[wid][k] = n;
    }
    const uint32_t err = wave_or(t.all_err);
    if (lead) sx[wid] = err;
    __syncthreads();
    double* r = rows + row * kTallyStride;
    unsigned long long* n = reinterpret_cast<unsigned long long*>(r + kMaxChannels);
    const int i = static_cast<int>(threadIdx.x);
    if (i < NCH) {
        double e = se[0][i];
#pragma unroll
        for (int v = 1; v < W; ++v) e += se[v][i];
        r[i] = e;
    } else if (i >= 16 && i < 16 + NCH + 3) {
        unsigned long long k = 0;
#pragma unroll
        for (int v = 0; v < W; ++v) k += sc[v][i - 16];
        n[i - 16] = k;
    } else if (i == 32) {
        uint32_t e = 0u;
#pragma unroll
        for (int v = 0; v < W; ++v) e |= sx[v];
        reinterpret_cast<unsigned long long*>(r)[kTallyErr] = e;
    }
}

// Exclusive scan of one int per thread over a BLOCK-thread block: the
// wave's prefix by shuffles, the wave totals through LDS (wsum: BLOCK / 64
// ints); sets total.
template <int BLOCK>
__device__ __forceinline__ int block_scan_int(int x, int* wsum, int& total) {
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    int incl = x;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int y = __shfl_up(incl, d, 64);
        if (lane >= d) incl += y;
    }
    if (lane == 63) wsum[wid] = incl;
    __syncthreads();
    int before = 0;
    total = 0;
#pragma unroll
    for (int k = 0; k < BLOCK / 64; ++k) {
        const int sk = wsum[k];
        before += k < wid ? sk : 0;
        total += sk;
    }
    __syncthreads();
    return before + incl - x;
}

// off[c] = tot[0] + ... + tot[c - 1] for c < nchunks, by one BLOCK-thread
// block: each thread sums a consecutive run, its loads issued together; returns the sum of all totals.
template <int BLOCK>
__device__ int chunk_offsets(const int32_t* tot, int32_t* off, int64_t nchunks, int* wsum) {
    constexpr int kB = BLOCK >= 1024 ? 4 : 8;
    const int64_t per = (nchunks + BLOCK - 1) / BLOCK;
    const int64_t c0 = static_cast<int64_t>(threadIdx.x) * per;
    const int64_t c1 = c0 + per < nchunks ? c0 + per : nchunks;
    int mine = 0;
    for (int64_t c = c0; c < c1; c += kB) {
        int v[kB];
#pragma unroll
        for (int b = 0; b < kB; ++b) v[b] = c + b < c1 ? tot[c + b] : 0;
#pragma unroll
        for (int b = 0; b < kB; ++b) mine += v[b];
    }
    int total = 0;
    int run = block_scan_int<BLOCK>(mine, wsum, total);
    for (int64_t c = c0; c < c1; c += kB) {
        int v[kB];
#pragma unroll
        for (int b = 0; b < kB; ++b) v[b] = c + b < c1 ? tot[c + b] : 0;
#pragma unroll
        for (int b = 0; b < kB; ++b)
            if (c + b < c1) {
                off[c + b] = run;
                run += v[b];
            }
    }
    return total;
}

// Rows [0, nrows) added in row order and the sums added to (ADD) or stored at
// energy[NCH] and counts[NCH + 3]; returns the rows' error bits to every
// thread.  Block of BLOCK threads; every thread calls it.
// A thread's rows r, r + BLOCK, ... are loaded kFoldBatch at a time (the
// loads in flight together) and added in that same order.
template <int NCH, int BLOCK, bool ADD = true>
__device__ uint32_t fold_tally_rows(const double* rows, int64_t nrows, double* energy,
                                    unsigned long long* counts) {
    constexpr int kFoldBatch = BLOCK >= 1024 ? 2 : (NCH <= 4 ? 8 : 4);
    double v[NCH] = {};
    unsigned long long u[NCH + 3] = {};
    uint32_t err = 0u;
    for (int64_t r0 = threadIdx.x; r0 < nrows; r0 += kFoldBatch * BLOCK) {
        double e[kFoldBatch][NCH];
        unsigned long long n[kFoldBatch][NCH + 3], x[kFoldBatch];
#pragma unroll
        for (int b = 0; b < kFoldBatch; ++b) {
            const int64_t r = r0 + static_cast<int64_t>(b) * BLOCK;
            const double* row = rows + (r < nrows ? r : 0) * kTallyStride;
            const unsigned long long* cnt =
                reinterpret_cast<const unsigned long long*>(row + kMaxChannels);
#pragma unroll
            for (int c = 0; c < NCH; ++c) e[b][c] = row[c];
#pragma unroll
            for (int k = 0; k < NCH + 3; ++k) n[b][k] = cnt[k];
            x[b] = reinterpret_cast<const unsigned long long*>(row)[kTallyErr];
        }
#pragma unroll
        for (int b = 0; b < kFoldBatch; ++b) {
            if (r0 + static_cast<int64_t>(b) * BLOCK >= nrows) break;
#pragma unroll
            for (int c = 0; c < NCH; ++c) v[c] += e[b][c];
#pragma unroll
            for (int k = 0; k < NCH + 3; ++k) u[k] += n[b][k];
            err |= static_cast<uint32_t>(x[b]);
        }
    }
    const double s = block_sum<NCH, BLOCK>(v);
    if (threadIdx.x < NCH) energy[threadIdx.x] = ADD ? energy[threadIdx.x] + s : s;
    // counts: integer sums, any order gives the same value
    __shared__ unsigned long long cs[NCH + 3];
    __shared__ uint32_t sx;
    if (threadIdx.x < NCH + 3) cs[threadIdx.x] = 0;
    if (threadIdx.x == 0) sx = 0u;
    __syncthreads();
    if (err) atomicOr(&sx, err);
#pragma unroll
    for (int k = 0; k < NCH + 3; ++k) {
        const unsigned long long x = wave_sum_u64(u[k]);
        if ((threadIdx.x & 63) == 0 && x) atomicAdd(cs + k, x);
    }
    __syncthreads();
    if (threadIdx.x < NCH + 3)
        counts[threadIdx.x] = (ADD ? counts[threadIdx.x] : 0ull) + cs[threadIdx.x];
    const uint32_t all = sx;
    __syncthreads();
    return all;
}

struct AppendSide {
    int32_t* cell;
    float* off;
    float* v0;
    float* v1;
    float* v2;
    uint32_t* uid;
    int64_t base_slot;
    uint32_t base_uid;
    float half_qm_dt;
};

// Write the np product pairs of one parent (cell c, offset o) at product
// index j0.. of the secondary and ion species; their v_half comes from the
// current field (Simulation.cpp:989-994).
__device__ __forceinline__ void append_products_of(int c, float o, int np, int64_t j0,
                                                   const float* prod, const float* E32, int nx,
                                                   const AppendSide& sec, const AppendSide& ion) {
    const float ex = gather_1d_f32(E32, nx, c, o);
    for (int k = 0; k < np; ++k) {
        const int64_t j = j0 + k;
        const float* s = prod + 6 * k;
        const AppendSide* sides[2] = {&sec, &ion};
        for (int q = 0; q < 2; ++q) {
            const AppendSide& d = *sides[q];
            const int64_t slot = d.base_slot + j;
            d.cell[slot] = c;
            d.off[slot] = o;
            d.v0[slot] = s[3 * q] - d.half_qm_dt * ex;
            d.v1[slot] = s[3 * q + 1];
            d.v2[slot] = s[3 * q + 2];
            d.uid[slot] = d.base_uid + static_cast<uint32_t>(j);
        }
    }
}

// The tables go to LDS when they fit in kMccLdsWords (a shared energy grid
// is stored once), else the kernels read them from global memory (L2);
// the per-channel parameter table always goes to LDS.
struct MccLds {
    float words[kMccLdsWords];
    ChannelSel chan[kMaxChannels];
    MccParams params;        // collide_run's copy
};

// energy rows staged: one grid for all channels, or every channel's
__host__ __device__ __forceinline__ int mcc_energy_rows(const MccParams& m) {
    return m.grid_shared ? m.rows[0] : m.total_rows;
}
inline bool mcc_tables_fit(const MccParams& m) {
    return mcc_energy_rows(m) + m.total_rows <= kMccLdsWords;
}

__device__ __forceinline__ void stage_channels(const MccParams& m, MccLds& lds) {
    if (threadIdx.x == 0) {
#pragma unroll
        for (int k = 0; k < kMaxChannels; ++k)
            if (k < m.nchan)
                lds.chan[k] = ChannelSel{m.kind[k], m.angular[k], m.threshold[k], m.half_emass[k],
                                         m.mc_offset[k], m.mc_rows[k]};
    }
}

__device__ __forceinline__ XsView stage_tables(const MccParams& m, MccLds& lds) {
    stage_channels(m, lds);
    XsView X{m.energy, m.sigma, 0};
    const int ne = mcc_energy_rows(m);
    if (ne + m.total_rows <= kMccLdsWords) {
        for (int i = threadIdx.x; i < ne; i += blockDim.x) lds.words[i] = m.energy[i];
        for (int i = threadIdx.x; i < m.total_rows; i += blockDim.x)
            lds.words[ne + i] = m.sigma[i];
        X = XsView{lds.words, lds.words + ne, m.grid_shared};
    }
    __syncthreads();
    return X;
}

// The same with the choice made at compile time (LDS: mcc_tables_fit): the
// tables' address space is known, so their reads are LDS reads and not
// generic ones.
template <bool LDS>
__device__ __forceinline__ void stage_tables_as(const MccParams& m, MccLds& lds) {
    stage_channels(m, lds);
    if constexpr (LDS) {
        const int ne = mcc_energy_rows(m);
        for (int i = threadIdx.x; i < ne; i += blockDim.x) lds.words[i] = m.energy[i];
        for (int i = threadIdx.x; i < m.total_rows; i += blockDim.x)
            lds.words[ne + i] = m.sigma[i];
    }
    __syncthreads();
}
// and the parameters
template <bool LDS>
__device__ __forceinline__ void stage_model(MccLds& lds) {
    using Words = const __attribute__((address_space(4))) uint32_t*;
    const Words m = (Words)__builtin_amdgcn_kernarg_segment_ptr();
    for (unsigned i = threadIdx.x; i < sizeof(MccParams) / 4; i += blockDim.x)
        reinterpret_cast<uint32_t*>(&lds.params)[i] = m[i];
    stage_tables_as<LDS>(first_kernel_argument<MccParams>(), lds);
}
template <bool LDS>
__device__ __forceinline__ XsView table_view(const MccParams& m, const MccLds& lds) {
    if constexpr (LDS)
        return XsView{lds.words, lds.words + mcc_energy_rows(m), m.grid_shared};
    else
        return XsView{m.energy, m.sigma, 0};
}

// ------------------------------------------------ collisions of many particles
// One step's collisions of a run of slots, by one wave.  Nine particles in
// ten meet no candidate, so the wave goes over its slots twice:
//   sweep    every particle's first Philox block; a first draw that cannot
//            hold a candidate (no_candidate, proved on the host) ends its
//            step, the others' indices go to the wave's LDS queue
//   collide  each lane takes a queued particle and runs its candidate loop
//            one waiting time at a time; a lane that is done takes the next,
//            so the long code runs on full waves
// A particle's operations and draws are those of mcc_collide, and its result
// does not depend on its lane, so neither does anything written per particle.
// A run holds at most 64 kRunChunks slots.  Latency bounds a launch of up to a
// million particles (62 % of the wave cycles wait, mostly on LDS), VALU issue
// larger ones.  Measured, 1e6 bare collides 55.8 -> 21.6 us; the 1D step at
// 5e5 electrons 38.5 -> 25.1 us, 64 instances of 1e5 155 -> 60.7 us (one
// particle per lane before, every lane through the whole candidate code).
constexpr int kRunChunks = 16;
constexpr int kSweepUnroll = 4;     // chunks whose loads are in flight together
constexpr int kRefill = 32;         // lanes that are done before the wave takes new ones

struct WaveQueue {
    uint16_t index[64 * kRunChunks];
    uint8_t products[64 * kRunChunks];   // ionizations of each particle
};

// The runs of n slots over `waves` waves: `passes` runs each, of `chunks`
// 64-slot chunks (one pass of short runs until they are full).
struct RunPlan {
    uint32_t chunks, runs;
    __host__ __device__ __forceinline__ RunPlan(int64_t n, uint32_t waves) {
        const uint32_t all = static_cast<uint32_t>((n + 63) >> 6);
        chunks = (all + waves - 1) / waves;
        if (chunks > kRunChunks) {
            const uint32_t passes = (chunks + kRunChunks - 1) / kRunChunks;
            chunks = (chunks + passes - 1) / passes;
        }
        if (chunks < 1) chunks = 1;
        runs = (all + chunks - 1) / chunks;
    }
};
// at least the runs of any slot count up to n
inline int64_t max_runs(int64_t n, int64_t waves) {
    const int64_t full = 64 * kRunChunks * waves;
    return waves * std::max<int64_t>(1, (n + full - 1) / full);
}

// The waves that collide one population: kMccWaves per SIMD of the chip, in
// workgroups of kMccBlock; fewer when there are fewer chunks.  More
// waves hide more latency, fewer pack their lanes better: 2, 3 and 4 per SIMD
// take 26.8, 27.0 and 28.7 us at 5e5 electrons, 76.8, 63.4 and 59.7 us at 64
// instances (3.2e6), and the one-workgroup folds grow with them.
constexpr int kMccBlock = 256;
constexpr int kMccWaves = 3;
inline int mcc_groups(int cu_count, int64_t n) {
    const int64_t resident = static_cast<int64_t>(cu_count) * kMccWaves * 4 / (kMccBlock / 64);
    return static_cast<int>(std::clamp<int64_t>((n + kMccBlock - 1) / kMccBlock, 1, resident));
}

// orders a wave's LDS accesses before and after it (its lanes run together)
__device__ __forceinline__ void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Collides the run's `slots` slots; Io gives them:
//   fetch(i, state)     loads slot i; false: nothing alive there
//   velocity(state, u)  the velocity to collide
//   id(state, i)        the random stream
//   products(i)         where its products go, or null
//   pass(i, state, u)   a particle that meets no candidate
//   store(i, state, u)  one that went through the candidate loop
// and whether any particle of the run made products (their numbers in
// q.products) is returned.
template <int NCH, bool LDS, bool ONE_V, typename Io>
__device__ __forceinline__ bool collide_run(const MccLds& lds, WaveQueue& q, const Io& io,
                                            int slots, float dt, uint64_t seed, uint32_t stream,
                                            uint32_t step, LaneTally<NCH>& t) {
    const int lane = threadIdx.x & 63;
    const uint64_t below = (uint64_t{1} << lane) - 1;
    int queued = 0;
    {
        const MccParams& m = lds.params;
        const uint32_t no_candidate = m.no_candidate;
        const float safe_speed2 = m.safe_speed2;
        for (int base = 0; base < slots; base += 64 * kSweepUnroll) {
            typename Io::State st[kSweepUnroll];
            bool in[kSweepUnroll];
            float u[kSweepUnroll][3];
#pragma unroll
            for (int k = 0; k < kSweepUnroll; ++k) {
                const int i = base + 64 * k + lane;
                in[k] = io.fetch(i < slots ? i : 0, st[k]) && i < slots;
            }
#pragma unroll
            for (int k = 0; k < kSweepUnroll; ++k) io.velocity(st[k], u[k]);
#pragma unroll
            for (int k = 0; k < kSweepUnroll; ++k) {
                if (base + 64 * k >= slots) break;
                const int i = base + 64 * k + lane;
                Philox rng;
                rng.init(seed, stream, io.id(st[k], i), step);
                rng.refill();
                const float v2 = ONE_V ? u[k][0] * u[k][0]
                                       : u[k][0] * u[k][0] + u[k][1] * u[k][1] + u[k][2] * u[k][2];
                const bool collide =
                    in[k] && ((rng.b0 >> 9) >= no_candidate || !(v2 <= safe_speed2));
                if (in[k] && !collide) io.pass(i, st[k], u[k]);
                const uint64_t mask = __ballot(collide);
                if (collide) q.index[queued + __popcll(mask & below)] = static_cast<uint16_t>(i);
                queued += __popcll(mask);
                if (Io::kProducts) q.products[i] = 0;
            }
        }
    }
    wave_lds_fence();
    if constexpr (ONE_V) {
        for (int h = lane; h < queued; h += 64) {
            const MccParams& m = lds.params;
            const XsView X = table_view<LDS>(m, lds);
            const int i = q.index[h];
            typename Io::State st;
            float u[3];
            io.fetch(i, st);
            io.velocity(st, u);
            Philox rng;
            rng.init(seed, stream, io.id(st, i), step);
            MccTally<NCH> one{};
            mcc_collide_1v<NCH>(m, X, lds.chan, u[0], dt, rng, one);
            io.store(i, st, u);
            t.add(one);
        }
        wave_lds_fence();
        return false;
    } else {
        int head = 0, i = -1;
        bool made = false;
        typename Io::State st{};
        float u[3] = {0.f, 0.f, 0.f};
        float elapsed = 0.f;
        Philox rng;
        rng.init(seed, stream, 0u, step);
        while (head < queued || __ballot(i >= 0) != 0ull) {
            const uint64_t idle = __ballot(i < 0);
            if (head < queued && __popcll(idle) >= kRefill) {
                const int h = head + __popcll(idle & below);
                if (i < 0 && h < queued) {
                    i = q.index[h];
                    io.fetch(i, st);
                    io.velocity(st, u);
                    rng.c0 = 0u;
                    rng.c1 = io.id(st, i);
                    rng.used = 4;
                    t.begin(io.products(i));
                    elapsed = 0.f;
                }
                head += __popcll(idle);
            }
            if (i >= 0) {
                // mcc_collide from one waiting time to the next
                const MccParams& m = lds.params;
                const XsView X = table_view<LDS>(m, lds);
                bool again = false;
                if (!(u[0] * u[0] + u[1] * u[1] + u[2] * u[2] <= m.safe_speed2)) {
                    if (t.candidates == 0u &&
                        (!isfinite(u[0]) || !isfinite(u[1]) || !isfinite(u[2])))
                        t.err = DEV_ERR_NONFINITE;
                    else if (mcc_rate_fails<NCH>(m, X, u))
                        t.err = DEV_ERR_RATE;
                }
                if (t.err == 0u) {
                    const float waiting = -logf(rng.u01()) * m.inv_max_frequency;
                    if (waiting < dt - elapsed) {
                        elapsed += waiting;
                        ++t.candidates;
                        if (t.candidates > static_cast<uint32_t>(m.max_candidates))
                            t.err = DEV_ERR_CANDIDATES;
                        else
                            again = mcc_candidate<NCH>(m, X, lds.chan, u, rng, t);
                    }
                }
                if (!again) {
                    io.store(i, st, u);
                    if (Io::kProducts && t.nsec != 0u) {
                        q.products[i] = static_cast<uint8_t>(t.nsec < 2u ? t.nsec : 2u);
                        made = true;
                        if (t.nsec > 2u) t.err |= DEV_ERR_CAPACITY;
                    }
                    t.finish();
                    i = -1;
                }
            }
        }
        wave_lds_fence();
        return __ballot(made) != 0ull;
    }
}

// The parents of a run with products, in slot order, as words
// slot | products << 10 | products before it in the run << 12; written at
// list, their number to *parents and the products' to *total.
__device__ __forceinline__ void list_parents(const WaveQueue& q, int slots, bool made,
                                             int32_t* list, int32_t* parents, int32_t* total) {
    const int lane = threadIdx.x & 63;
    const uint64_t below = (uint64_t{1} << lane) - 1;
    int np = 0, nt = 0;
    if (made)
        for (int base = 0; base < slots; base += 64) {
            const int i = base + lane;
            const int c = i < slots ? q.products[i] : 0;
            const uint64_t m1 = __ballot(c > 0), m2 = __ballot(c > 1);
            if (c > 0)
                list[np + __popcll(m1 & below)] =
                    i | (c << 10) |
                    ((nt + __popcll(m1 & below) + __popcll(m2 & below)) << 12);
            np += __popcll(m1);
            nt += __popcll(m1) + __popcll(m2);
        }
    if (lane == 0) {
        *parents = np;
        *total = nt;
    }
}

// A 1D target species' run (Simulation.cpp:900-926): the velocity to collide
// is v synchronised from v_half with E(x) at t+dt (Pusher.cpp:74-76), the
// stored one v_half rebuilt (Pusher.cpp:66-68), also without a collision.
struct Run1d {
    const int32_t* cell;     // the run's first slot, as all below
    const float* off;
    float* v0;
    float* v1;
    float* v2;
    const uint32_t* uid;
    float* prod;             // per slot: 2 x (secondary v[3], ion v[3])
    const float* E32;
    int nx;
    float half_qm_dt;
    static constexpr bool kProducts = true;
    struct State {
        float kick;
        float v[3];
        uint32_t uid;
        int c;
        float o;
    };
    __device__ __forceinline__ bool fetch(int i, State& s) const {
        s.c = cell[i];
        s.o = off[i];
        s.v[0] = v0[i];
        s.v[1] = v1[i];
        s.v[2] = v2[i];
        s.uid = uid[i];
        return s.c >= 0;
    }
    __device__ __forceinline__ void velocity(State& s, float* u) const {
        s.kick = half_qm_dt * gather_1d_f32(E32, nx, s.c >= 0 ? s.c : 0, s.o);
        u[0] = s.v[0] + s.kick;
        u[1] = s.v[1];
        u[2] = s.v[2];
    }
    __device__ __forceinline__ uint32_t id(const State& s, int) const { return s.uid; }
    __device__ __forceinline__ float* products(int i) const {
        return prod ? prod + 12 * static_cast<int64_t>(i) : nullptr;
    }
    __device__ __forceinline__ void pass(int i, const State& s, const float* u) const {
        v0[i] = u[0] - s.kick;
    }
    __device__ __forceinline__ void store(int i, const State& s, const float* u) const {
        v0[i] = u[0] - s.kick;
        v1[i] = u[1];
        v2[i] = u[2];
    }
};

// Adds a run's products to the secondary and ion species: lane after lane
// takes a listed parent (see list_parents), whose products start at index
// first + (those before it in the run).
__device__ __forceinline__ void append_run(const int32_t* list, int parents, int64_t first,
                                           const int32_t* cell, const float* off,
                                           const float* prod, const float* E32, int nx,
                                           const AppendSide& sec, const AppendSide& ion) {
    for (int k = threadIdx.x & 63; k < parents; k += 64) {
        const int e = list[k];
        const int i = e & 1023;
        append_products_of(cell[i], off[i], (e >> 10) & 3, first + (e >> 12),
                           prod + 12 * static_cast<int64_t>(i), E32, nx, sec, ion);
    }
}

// ------------------------------------------------------------- host side
// Draws of a step's first uniform u = (2k + 1) 2^-24 that cannot hold a
// candidate: -log(u) / max_frequency >= dt for every k below this, with 1e-4
// of the exponent left for the FP32 logarithm, product and timestep (off by
// a few 1e-7 of it).
inline uint32_t no_candidate_draws(float dt, float inv_max_frequency) {
    const double x = static_cast<double>(dt) / static_cast<double>(inv_max_frequency);
    const double k = std::floor(std::exp(-x * (1.0 + 1.0e-4)) * 0x1p23) - 2.0;
    return k > 0.0 ? static_cast<uint32_t>(k) : 0u;
}

// Validated model tables (NullCollisionModel ctor, Collision.cpp:315-577)
// into h; particle_mass is the projectile mass.
void load_mcc_model(MccModelHost& h, int nchan, const int* kind, const double* threshold,
                    const int64_t* rows, const double* const* energy,
                    const double* const* sigma, double neutral_density, double max_frequency,
                    int64_t max_candidates, double particle_mass, double neutral_mass,
                    double neutral_temperature);
// Per-channel angular model and energy frame (CollisionChannelConfig).
void set_channel_options(MccModelHost& h, int channel, int angular, int frame, int64_t rows,
                         const double* energy, const double* mean_cosine);
MccParams mcc_params_of(const MccModelHost& h);
MccParams mcc_params(const Context& c);
// the parameters of the context's model `model` plus the product masses of
// the 1D step's energy tally
MccParams mcc_step_params(const Context& c, int model = 0);

}  // namespace aurora
