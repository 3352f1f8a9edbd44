// swarm.hip - batched homogeneous electron swarms (run_field,
// Swarm.cpp:940-1250, fixed population), many requests of uneven particle
// count per launch.
//
// Work is split into chunks of kChunk electrons of one request.  A
// persistent kernel's workgroups pull chunks from a queue; each chunk's
// velocities stay in registers for the launch's step range (half kick,
// energy guard, MCC, half kick, guard - Swarm.cpp:998-1060).  Sampling
// statistics go to per-(chunk, uncertainty block) integer fixed-point
// partials (power-of-two scales per request, sized from its energy ceiling
// and block length so a chunk's block sum cannot overflow) and integer
// counters;
// integer sums are associative, so a request's result does not depend on
// which other requests share its launches or on how its steps are split
// into launches.  Each electron's displacement since the end of burn-in is
// kept (x += v dt after the first half kick, Swarm.cpp:1026-1031); after
// the last step every chunk reduces its displacement moments in FP64 in a
// fixed order, for the diffusion coefficients (Swarm.cpp:1139-1176).
#include <algorithm>
#include <cmath>
#include <limits>
#include <map>
#include <cstring>
#include <memory>
#include <string>
#include <vector>

#include "mcc_device.hpp"

namespace aurora {

namespace {

constexpr int kChunk = 256;
constexpr double kElectronMass = 9.1093837139e-31;   // Swarm.cpp:23
constexpr double kElementaryCharge = 1.602176634e-19; // Swarm.cpp:24
constexpr double kTownsend = 1.0e-21;                 // Swarm.cpp:26

struct RequestDesc {
    float* vx;
    float* vy;
    float* vz;
    float* dx;                    // displacement since burn-in (3 x particles)
    double* moments;              // [chunk][5]: sums of dx, dy, dz, dx^2, dy^2 + dz^2
    long long* part;              // [chunk][block][2] fixed-point sums of v_x, energy
    unsigned long long* counts;   // [candidates, nulls, chan...]
    unsigned* max_energy_bits;
    uint32_t* status;
    int64_t particles;
    float half_kick;
    float dt;
    float v2_max;                 // largest squared speed whose energy is within the ceiling
    float ev_per_v2;              // 0.5 m / e
    float scale_v;                // fixed-point scales (powers of two)
    float scale_e;
    int step0;                    // first step of this launch
    int nsteps;                   // steps this launch
    int burn_in;
    int sampling;                 // steps - burn_in
    int blocks;
    uint32_t no_candidate;        // first draws below this (of 2^23) hold no candidate
    uint64_t seed;
};

struct WorkItem {
    int request;
    int chunk;
};

// lanes of a wave that wait with a collision candidate before the wave
// runs the candidate code for them together
constexpr int kCandidateBatch = 32;
constexpr int kLdsBlocks = 32;

// the largest FP32 squared speed x with fl(ev x) <= limit: the energy check
// e > limit on an electron is x > v2_ceiling
float v2_ceiling(float limit, float ev) {
    float x = limit / ev;
    while (x > 0.0f && ev * x > limit) x = std::nextafter(x, 0.0f);
    for (;;) {
        const float y = std::nextafter(x, std::numeric_limits<float>::infinity());
        if (!(y < std::numeric_limits<float>::infinity()) || ev * y > limit) return x;
        x = y;
    }
}

// (m_arg is the first argument: first_kernel_argument<MccParams>)
template <int NCH, bool LDS>
__global__ void __launch_bounds__(kChunk, 4) k_swarm(MccParams m_arg,
                                                     const RequestDesc* __restrict__ descs,
                                                     const WorkItem* __restrict__ items, int nitems,
                                                     int* head) {
    __shared__ MccLds lds;
    __shared__ int item_s;
    // half a chunk for the cross-wave steps of the FP64 moment tree
    __shared__ double red_m[5][kChunk / 2];
    stage_tables_as<LDS>(m_arg, lds);
    const float safe_speed2 = m_arg.safe_speed2;
    // sums of v_x and energy per uncertainty block of the launch (further
    // blocks of a launch go to global memory)
    __shared__ unsigned long long block_sum_s[2 * kLdsBlocks];
    for (int q = threadIdx.x; q < 2 * kLdsBlocks; q += kChunk) block_sum_s[q] = 0ull;
    for (;;) {
        if (threadIdx.x == 0) item_s = atomicAdd(head, 1);
        __syncthreads();
        // uniform across the workgroup: the work item and its request
        // descriptor go to scalar registers
        const int item = __builtin_amdgcn_readfirstlane(item_s);
        __syncthreads();
        if (item >= nitems) break;
        const WorkItem w = items[item];
        const RequestDesc d = descs[w.request];
        const int64_t p = static_cast<int64_t>(w.chunk) * kChunk + threadIdx.x;
        const bool active = p < d.particles;
        float v[3] = {0.f, 0.f, 0.f};
        float x[3] = {0.f, 0.f, 0.f};
        if (active) { v[0] = d.vx[p]; v[1] = d.vy[p]; v[2] = d.vz[p]; }
        if (active && d.step0 > d.burn_in) {
            x[0] = d.dx[p];
            x[1] = d.dx[d.particles + p];
            x[2] = d.dx[2 * d.particles + p];
        }
        uint32_t cand = 0, nulls = 0, chan[NCH] = {};
        uint32_t err = 0;
        // the largest squared speed, as bits (squares order like integers)
        uint32_t max_v2 = 0u;
        // a step needs a closer look where the squared speed exceeds this:
        // the energy ceiling, the rate bound, or not a number
        const float look_v2 = fminf(safe_speed2, d.v2_max);
        // The launch's steps in two segments, before and after the burn-in
        // end.  Inside a segment every lane steps on its own, and the common
        // step -- no collision candidate -- is all a lane runs by itself: two
        // half kicks with their energy checks, one Philox block and an
        // integer compare of its first draw (no_candidate_draws).  A lane
        // waits when its draw may hold a candidate, and when it reaches the
        // end of its uncertainty block; once kCandidateBatch lanes of the
        // wave wait (or no lane can step on) the wave takes the waiting time,
        // the candidate and the next draw for all of the former at once, and
        // the latter add their block sums in LDS.  Each lane's operations and
        // draws are those of the step-synchronous loop and the sums are of
        // integers, so results are unchanged.  VALU issue bounds the kernel:
        // 1.2e11 electron-steps/s in runs of 8,000 steps (6.8e10 with the logarithm,
        // square root and tallies in every step and blocks as segments).
        const int s_stop = d.step0 + d.nsteps;
        for (int s0 = d.step0; s0 < s_stop;) {
            const bool sampling = s0 >= d.burn_in;
            const int seg_end = sampling ? s_stop : min(s_stop, d.burn_in);
            // block sums of the lane: integers below 2^53 (the scales leave
            // a chunk's 256 lanes 2^61), so FP64 adds them exactly
            double acc_v = 0.0, acc_e = 0.0;
            MccCounts<NCH> t;
            mcc_tally_reset(t);
            int s = active ? s0 : seg_end;
            // uncertainty block b covers samples [floor(b S / B),
            // floor((b + 1) S / B)); blocks are at least one sample long
            int group = -1, first_group = 0, block_end = seg_end;
            auto end_of = [&](int g) {
                const int64_t e = (static_cast<int64_t>(g) + 1) * d.sampling / d.blocks;
                return static_cast<int>(min(static_cast<int64_t>(seg_end), d.burn_in + e));
            };
            if (sampling) {
                const int64_t k = s0 - d.burn_in;
                first_group = group = static_cast<int>(((k + 1) * d.blocks - 1) / d.sampling);
                block_end = end_of(group);
            }
            int run_to = block_end;    // a lane with a candidate: 0, it does not step
            float elapsed = 0.f;
            int step_candidates = 0;
            Philox rng;
            rng.init(d.seed, 0u, static_cast<uint32_t>(p), 0u);
            auto square = [&]() { return v[0] * v[0] + v[1] * v[1] + v[2] * v[2]; };
            // a failed particle keeps its velocity; the block sums still
            // take it at every step left (a product of exact integers)
            auto book_rest = [&]() {
                const double k = static_cast<double>(block_end - s);
                if (sampling && s < block_end) {
                    acc_v += k * static_cast<double>(rintf(v[0] * d.scale_v));
                    acc_e += k * static_cast<double>(rintf(d.ev_per_v2 * square() * d.scale_e));
                }
                s = block_end;
            };
            // the step's end: second half kick, energy check, block sums
            auto end_step = [&]<bool SAMPLING>() {
                v[0] += d.half_kick;
                const float v2 = square();
                max_v2 = max(max_v2, __float_as_uint(v2));
                if constexpr (SAMPLING) {
                    acc_v += static_cast<double>(rintf(v[0] * d.scale_v));
                    acc_e += static_cast<double>(rintf(d.ev_per_v2 * v2 * d.scale_e));
                }
                ++s;
                if (v2 > d.v2_max) err |= DEV_ERR_ENERGY;
                if (err) book_rest();
            };
            if (err && active) book_rest();
            // every lane steps until enough wait or none can step on
            auto step_lanes = [&]<bool SAMPLING>() {
                for (;;) {
                    if (s < run_to) {
                        v[0] += d.half_kick;
                        const float v2 = square();
                        max_v2 = max(max_v2, __float_as_uint(v2));
                        if constexpr (SAMPLING) {
                            x[0] += v[0] * d.dt;
                            x[1] += v[1] * d.dt;
                            x[2] += v[2] * d.dt;
                        }
                        rng.c0 = 0u;
                        rng.c2 = static_cast<uint32_t>(s);
                        rng.refill();
                        bool may_collide = (rng.b0 >> 9) >= d.no_candidate;
                        if (!(v2 <= look_v2)) {
                            if (v2 > d.v2_max) err |= DEV_ERR_ENERGY;
                            if (!(v2 <= safe_speed2)) {
                                const MccParams& m = first_kernel_argument<MccParams>();
                                const XsView X = table_view<LDS>(m, lds);
                                uint32_t failed = 0u;
                                if (!isfinite(v[0]) || !isfinite(v[1]) || !isfinite(v[2]))
                                    failed = DEV_ERR_NONFINITE;
                                else if (mcc_rate_fails<NCH>(m, X, v))
                                    failed = DEV_ERR_RATE;
                                err |= failed;
                                may_collide = may_collide && failed == 0u;
                            }
                        }
                        if (may_collide) {
                            run_to = 0;
                            elapsed = 0.f;
                            step_candidates = 0;
                        } else {
                            end_step.template operator()<SAMPLING>();
                        }
                    }
                    const uint64_t stepping = __ballot(s < run_to);
                    const uint64_t waiting = __ballot(s < seg_end) & ~stepping;
                    if (stepping == 0ull || __popcll(waiting) >= kCandidateBatch) break;
                }
            };
            for (;;) {
                if (sampling) step_lanes.template operator()<true>();
                else step_lanes.template operator()<false>();
                if (s < seg_end && run_to == 0) {
                    // mcc_collide's loop from one waiting time to the next
                    const MccParams& m = first_kernel_argument<MccParams>();
                    const XsView X = table_view<LDS>(m, lds);
                    bool again = false;
                    const float waiting = -logf(rng.u01()) * m.inv_max_frequency;
                    if (waiting < d.dt - elapsed) {
                        elapsed += waiting;
                        ++t.candidates;
                        if (++step_candidates > m.max_candidates)
                            err |= DEV_ERR_CANDIDATES;
                        else if (mcc_candidate<NCH>(m, X, lds.chan, v, rng, t)) {
                            if (!(square() <= safe_speed2) && mcc_rate_fails<NCH>(m, X, v))
                                err |= DEV_ERR_RATE;
                            else
                                again = true;
                        }
                        err |= t.err;
                        t.err = 0u;
                    }
                    if (!again) {
                        run_to = block_end;
                        if (sampling) end_step.template operator()<true>();
                        else end_step.template operator()<false>();
                    }
                }
                // lanes at the end of their block add its sums
                if (sampling && active && s == block_end && group >= 0) {
                    const int slot = 2 * (group - first_group);
                    if (slot < 2 * kLdsBlocks) {
                        atomicAdd(&block_sum_s[slot],
                                  static_cast<unsigned long long>(__double2ll_rn(acc_v)));
                        atomicAdd(&block_sum_s[slot + 1],
                                  static_cast<unsigned long long>(__double2ll_rn(acc_e)));
                    } else {
                        unsigned long long* q = reinterpret_cast<unsigned long long*>(
                            d.part + (static_cast<int64_t>(w.chunk) * d.blocks + group) * 2);
                        atomicAdd(q, static_cast<unsigned long long>(__double2ll_rn(acc_v)));
                        atomicAdd(q + 1, static_cast<unsigned long long>(__double2ll_rn(acc_e)));
                    }
                    acc_v = 0.0;
                    acc_e = 0.0;
                    ++group;
                    if (s < seg_end) {
                        block_end = end_of(group);
                        run_to = block_end;
                        if (err) book_rest();
                    } else {
                        group = -1;
                    }
                }
                if (__ballot(s < seg_end || (sampling && active && group >= 0)) == 0ull) break;
            }
            if (sampling) {
                cand += t.candidates;
                nulls += t.nulls;
#pragma unroll
                for (int c = 0; c < NCH; ++c) chan[c] += t.chan[c];
                // the chunk's block sums of this launch (every lane has added
                // its own) to the request's partials
                const int64_t k1 = s_stop - d.burn_in;
                const int last_group = static_cast<int>((k1 * d.blocks - 1) / d.sampling);
                const int nsum = 2 * min(last_group - first_group + 1, kLdsBlocks);
                __syncthreads();
                for (int q = threadIdx.x; q < nsum; q += kChunk) {
                    d.part[(static_cast<int64_t>(w.chunk) * d.blocks + first_group) * 2 + q] +=
                        static_cast<long long>(block_sum_s[q]);
                    block_sum_s[q] = 0ull;
                }
                __syncthreads();
            }
            s0 = seg_end;
        }
        const float emax = d.ev_per_v2 * __uint_as_float(max_v2);
        const bool last = d.step0 + d.nsteps == d.burn_in + d.sampling;
        if (last) {
            // displacement moments of the chunk, reduced in a fixed order
            const double m0 = active ? static_cast<double>(x[0]) : 0.0;
            const double m1 = active ? static_cast<double>(x[1]) : 0.0;
            const double m2 = active ? static_cast<double>(x[2]) : 0.0;
            double mv[5] = {m0, m1, m2, m0 * m0, m1 * m1 + m2 * m2};
            // the pairwise tree: at stride st, element i < st adds element
            // i + st; strides of a wave or more through LDS, the rest by
            // shuffles within the first wave (the same pairs and sums)
            for (int st = kChunk / 2; st >= 64; st >>= 1) {
                if (threadIdx.x >= st && threadIdx.x < 2 * st)
#pragma unroll
                    for (int k = 0; k < 5; ++k) red_m[k][threadIdx.x - st] = mv[k];
                __syncthreads();
                if (threadIdx.x < st)
#pragma unroll
                    for (int k = 0; k < 5; ++k) mv[k] += red_m[k][threadIdx.x];
                __syncthreads();
            }
            for (int st = 32; st > 0; st >>= 1)
#pragma unroll
                for (int k = 0; k < 5; ++k) mv[k] += __shfl_down(mv[k], st, 64);
            if (threadIdx.x == 0)
#pragma unroll
                for (int k = 0; k < 5; ++k) d.moments[static_cast<int64_t>(w.chunk) * 5 + k] = mv[k];
            __syncthreads();
        } else if (active && d.step0 + d.nsteps > d.burn_in) {
            d.dx[p] = x[0];
            d.dx[d.particles + p] = x[1];
            d.dx[2 * d.particles + p] = x[2];
        }
        if (active) {
            d.vx[p] = v[0];
            d.vy[p] = v[1];
            d.vz[p] = v[2];
        }
        // one atomic per wave and counter (per lane they queue up on the
        // request's few addresses: 20 ms of a 66 ms launch of 1,000 steps)
        uint64_t sums[2 + NCH];
        sums[0] = cand;
        sums[1] = nulls;
#pragma unroll
        for (int c = 0; c < NCH; ++c) sums[2 + c] = chan[c];
        float top = active ? emax : 0.f;
        for (int o = 32; o > 0; o >>= 1) {
            top = fmaxf(top, __shfl_xor(top, o, 64));
            err |= __shfl_xor(err, o, 64);
        }
#pragma unroll
        for (int k = 0; k < 2 + NCH; ++k) {
            const unsigned long long n = wave_sum_u64(sums[k]);
            if ((threadIdx.x & 63) == 0 && n) atomicAdd(d.counts + k, n);
        }
        if ((threadIdx.x & 63) == 0) {
            atomicMax(d.max_energy_bits, __float_as_uint(top));
            if (err) atomicOr(d.status, err);
        }
    }
}

// initial Maxwellian velocities with mean energy E0 (Swarm.cpp:951-957),
// Box-Muller from the request's Philox stream (step slot 0xFFFFFFFF)
__global__ void k_swarm_init(float* vx, float* vy, float* vz, int64_t n, float sigma,
                             uint64_t seed) {
    for (int64_t p = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; p < n;
         p += static_cast<int64_t>(gridDim.x) * blockDim.x) {
        Philox rng;
        rng.init(seed, 0u, static_cast<uint32_t>(p), 0xFFFFFFFFu);
        const float u1 = rng.u01(), u2 = rng.u01(), u3 = rng.u01(), u4 = rng.u01();
        const float r1 = sqrtf(-2.0f * logf(u1)), r2 = sqrtf(-2.0f * logf(u3));
        float s1, c1, s2, c2;
        sincosf(6.28318530717958647692f * u2, &s1, &c1);
        sincosf(6.28318530717958647692f * u4, &s2, &c2);
        vx[p] = sigma * r1 * c1;
        vy[p] = sigma * r1 * s1;
        vz[p] = sigma * r2 * c2;
    }
}

struct RequestState {
    aurora_hip_swarm_request req{};
    int64_t chunks = 0;
    int64_t steps_done = 0;
    uint64_t footprint = 0;
    // One allocation, laid out by RequestLayout: the sums that start at zero,
    // then the moments (together the request's result, read back in one copy),
    // then the electrons.
    DevBuf<uint8_t> slab;
    long long* part = nullptr;             // chunks x blocks x 2
    unsigned long long* counts = nullptr;  // kMaxChannels + 3
    unsigned* maxe = nullptr;
    uint32_t* status = nullptr;
    double* moments = nullptr;             // chunks x 5
    float* v = nullptr;                    // 3 x particles (SoA)
    float* dx = nullptr;                   // 3 x particles displacement (SoA)
};

// byte offsets of a request's arrays in its slab; zeroed: the bytes that start
// at zero, result: those read back at its end
struct RequestLayout {
    size_t counts, maxe, status, zeroed, moments, result, v, dx, bytes;
    RequestLayout(const aurora_hip_swarm_request& q, int64_t chunks) {
        const size_t lanes = static_cast<size_t>(3 * q.particles) * sizeof(float);
        counts = static_cast<size_t>(chunks * q.blocks * 2) * sizeof(long long);   // part at 0
        maxe = counts + (kMaxChannels + 3) * sizeof(unsigned long long);
        status = maxe + sizeof(unsigned);
        zeroed = status + sizeof(uint32_t);
        moments = (zeroed + 7) / 8 * 8;
        result = moments + static_cast<size_t>(chunks * 5) * sizeof(double);
        v = (result + 63) / 64 * 64;
        dx = v + lanes;
        bytes = dx + lanes;   // at most footprint_of(q), which leaves 64 bytes for the alignment
    }
};

// Descriptor and work-item arrays of one launch: pinned host staging and
// device copies, reused once the event recorded after the launch completes.
struct LaunchBuffers {
    RequestDesc* h_descs = nullptr;
    WorkItem* h_items = nullptr;
    size_t cap_descs = 0, cap_items = 0;
    DevBuf<RequestDesc> descs;
    DevBuf<WorkItem> items;
    DevBuf<int> head;
    hipEvent_t done = nullptr;
    ~LaunchBuffers() {
        if (h_descs) (void)hipHostFree(h_descs);
        if (h_items) (void)hipHostFree(h_items);
        if (done) (void)hipEventDestroy(done);
    }
};

struct SwarmState {
    MccModelHost gas;
    bool gas_loaded = false;
    std::map<int64_t, std::unique_ptr<RequestState>> active;
    std::map<int64_t, aurora_hip_swarm_result> finished;
    int64_t next_handle = 1;
    uint64_t bytes_in_use = 0;
    double table_max_ev = 0.0;
    LaunchBuffers buf[2];           // alternate between launches
    int cur = 0;
    bool in_flight = false;         // a launch has been queued and not collected
    std::vector<int64_t> finishing; // requests whose last steps the launch in flight runs
    int blocks_per_cu = 0;          // resident k_swarm workgroups per CU (occupancy)
    // Slabs of requests that are done, for the next ones: 64 served requests
    // spent 5 of 40 ms in allocating and freeing them (and 5 to 10 more while
    // each request had seven allocations).  Used on the context's stream alone,
    // after it has drained past the request; at most kSpareBytes, which a
    // request's budget covers with the slabs in use (fit_budget), freed with
    // the context or when an allocation of the context needs the memory.
    std::vector<DevBuf<uint8_t>> spare;
    size_t spare_bytes = 0;
    bool budgeted = false;          // a request came with an HBM budget
};
constexpr size_t kSpareBytes = size_t{256} << 20;

// the smallest spare slab of bytes to most, or none
DevBuf<uint8_t> take_spare(SwarmState& s, size_t bytes, size_t most) {
    size_t best = s.spare.size();
    for (size_t k = 0; k < s.spare.size(); ++k)
        if (s.spare[k].count >= bytes && s.spare[k].count <= most &&
            (best == s.spare.size() || s.spare[k].count < s.spare[best].count))
            best = k;
    DevBuf<uint8_t> slab;
    if (best < s.spare.size()) {
        slab = std::move(s.spare[best]);
        s.spare.erase(s.spare.begin() + static_cast<std::ptrdiff_t>(best));
        s.spare_bytes -= slab.count;
    }
    return slab;
}

// Spare slabs freed, the last kept first, until the budget holds them, the
// slabs in use and the bytes of one more.
void fit_budget(SwarmState& s, uint64_t bytes, uint64_t budget) {
    while (!s.spare.empty() && s.bytes_in_use + bytes + s.spare_bytes > budget) {
        s.spare_bytes -= s.spare.back().count;
        s.spare.pop_back();
    }
}

void keep_slab(SwarmState& s, DevBuf<uint8_t>&& slab) {
    if (slab.count > kSpareBytes - s.spare_bytes) return;   // freed by its owner
    s.spare_bytes += slab.count;
    s.spare.push_back(std::move(slab));
}

SwarmState& state(Context& c) {
    if (!c.swarm) c.swarm = new SwarmState();
    return *static_cast<SwarmState*>(c.swarm);
}

uint64_t footprint_of(const aurora_hip_swarm_request& r) {
    const uint64_t chunks = (static_cast<uint64_t>(r.particles) + kChunk - 1) / kChunk;
    return static_cast<uint64_t>(r.particles) * 24u + chunks * static_cast<uint64_t>(r.blocks) * 16u +
           chunks * 40u + (kMaxChannels + 3) * 8u + 64u;
}

MccParams swarm_params(const SwarmState& s) { return mcc_params_of(s.gas); }

// power-of-two fixed-point scales for the v_x and energy sums of one
// (chunk, uncertainty block): kChunk x (block length) values each bounded by
// the request's energy ceiling (with 2x headroom) stay below 2^61
std::pair<double, double> scales(const aurora_hip_swarm_request& q) {
    const double S = static_cast<double>(q.steps - q.burn_in);
    const double per_block = std::ceil(S / static_cast<double>(q.blocks));
    const double emax = 2.0 * q.max_energy_ev;
    const double vmax = std::sqrt(2.0 * emax * kElementaryCharge / kElectronMass);
    const double room = std::ldexp(1.0, 61) / (kChunk * per_block);
    auto pow2_floor = [](double x) {
        int e = static_cast<int>(std::floor(std::log2(x)));
        e = std::max(-120, std::min(120, e));
        return std::ldexp(1.0, e);
    };
    return {pow2_floor(room / vmax), pow2_floor(room / emax)};
}

void block_mean_error(const std::vector<double>& means, double& mean, double& se) {
    // Swarm.cpp:103-134 on block means
    const size_t b = means.size();
    double m = 0.0;
    for (double v : means) m += v;
    m /= static_cast<double>(b);
    double sq = 0.0;
    for (double v : means) sq += (v - m) * (v - m);
    mean = m;
    se = b == 1 ? 0.0 : std::sqrt(sq / (static_cast<double>(b) * static_cast<double>(b - 1)));
}

void finalize(Context& c, SwarmState& s, int64_t handle, RequestState& r) {
    aurora_hip_swarm_result out{};
    const auto& q = r.req;
    const int64_t B = q.blocks, S = q.steps - q.burn_in, N = q.particles;
    const RequestLayout lay(q, r.chunks);
    std::vector<long long> part(lay.result / sizeof(long long));   // the whole result, part first
    AUR_HIP(hipMemcpyAsync(part.data(), r.slab.ptr, lay.result, hipMemcpyDeviceToHost,
                           c.stream));
    AUR_HIP(hipStreamSynchronize(c.stream));
    const uint8_t* bytes = reinterpret_cast<const uint8_t*>(part.data());
    unsigned long long counts[kMaxChannels + 3];
    unsigned maxe = 0;
    uint32_t status = 0;
    std::memcpy(counts, bytes + lay.counts, sizeof counts);
    std::memcpy(&maxe, bytes + lay.maxe, sizeof maxe);
    std::memcpy(&status, bytes + lay.status, sizeof status);
    std::vector<double> mom(static_cast<size_t>(r.chunks * 5));
    std::memcpy(mom.data(), bytes + lay.moments, mom.size() * sizeof(double));
    {
        // Swarm.cpp:1139-1176: variance of the displacement over the
        // sampling window; D_L = var_x / 2T, D_T = var_yz / 4T
        double sx = 0, sy = 0, sz = 0, sxx = 0, syz = 0;
        for (int64_t ch = 0; ch < r.chunks; ++ch) {   // fixed chunk order
            sx += mom[ch * 5];
            sy += mom[ch * 5 + 1];
            sz += mom[ch * 5 + 2];
            sxx += mom[ch * 5 + 3];
            syz += mom[ch * 5 + 4];
        }
        const double n = static_cast<double>(N);
        const double mx = sx / n, my = sy / n, mz = sz / n;
        const double var_x = sxx / n - mx * mx;
        const double var_yz = syz / n - my * my - mz * mz;
        const double T = static_cast<double>(S) * q.timestep;
        out.longitudinal_diffusion = var_x / (2.0 * T);
        out.transverse_diffusion = var_yz / (4.0 * T);
    }
    std::vector<double> vm(static_cast<size_t>(B)), em(static_cast<size_t>(B));
    for (int64_t b = 0; b < B; ++b) {
        double sv = 0.0, se = 0.0;
        for (int64_t ch = 0; ch < r.chunks; ++ch) {   // fixed chunk order
            sv += static_cast<double>(part[(ch * B + b) * 2]) / scales(q).first;
            se += static_cast<double>(part[(ch * B + b) * 2 + 1]) / scales(q).second;
        }
        const int64_t len = (b + 1) * S / B - b * S / B;
        vm[b] = sv / (static_cast<double>(N) * static_cast<double>(len));
        em[b] = se / (static_cast<double>(N) * static_cast<double>(len));
    }
    double mv, sev, me, see;
    block_mean_error(vm, mv, sev);
    block_mean_error(em, me, see);
    out.drift = -mv;
    out.drift_se = sev;
    out.mean_energy_ev = me;
    out.mean_energy_se = see;
    const double exposure = static_cast<double>(N) * q.timestep * static_cast<double>(S);
    out.candidates = counts[0];
    out.nulls = counts[1];
    for (int k = 0; k < s.gas.nchan; ++k) {
        out.collisions[k] = counts[2 + k];
        out.rate[k] = static_cast<double>(counts[2 + k]) / exposure;
        out.rate_se[k] = std::sqrt(static_cast<double>(counts[2 + k])) / exposure;
        if (s.gas.kind[k] == AURORA_IONIZATION) {
            out.ionization_rate += out.rate[k];
            out.ionization_rate_se = std::hypot(out.ionization_rate_se, out.rate_se[k]);
        }
    }
    float mx;
    std::memcpy(&mx, &maxe, sizeof mx);
    out.max_energy_ev = mx;
    out.status = AURORA_OK;
    if (status & DEV_ERR_ENERGY) out.status = AURORA_ERR_ENERGY_ABOVE_MAX;
    else if (status & DEV_ERR_RATE) out.status = AURORA_ERR_RATE_ABOVE_BOUND;
    else if (status & DEV_ERR_CANDIDATES) out.status = AURORA_ERR_CANDIDATE_LIMIT;
    else if (status) out.status = AURORA_ERR_INVALID_ARGUMENT;
    s.finished[handle] = out;
    s.bytes_in_use -= r.footprint;
}

// validate_config (Swarm.cpp:277-559), the checks common to both
// population models
void validate_request(const SwarmState& s, const aurora_hip_swarm_request* r) {
    AUR_REQUIRE(std::isfinite(r->timestep) && r->timestep > 0.0, AURORA_ERR_INVALID_ARGUMENT,
                "swarm timestep must be positive and finite");
    AUR_REQUIRE(s.gas.max_frequency * r->timestep <= 0.1, AURORA_ERR_INVALID_ARGUMENT,
                "swarm max_frequency * timestep must not exceed 0.1");
    AUR_REQUIRE(r->steps > 0 && r->burn_in < r->steps, AURORA_ERR_INVALID_ARGUMENT,
                "swarm steps must exceed burn_in_steps");
    AUR_REQUIRE(r->steps < 2147483647, AURORA_ERR_INVALID_ARGUMENT, "swarm steps too large");
    AUR_REQUIRE(r->particles > 0, AURORA_ERR_INVALID_ARGUMENT,
                "swarm particles must be positive");
    AUR_REQUIRE(r->blocks > 0 && r->blocks <= r->steps - r->burn_in,
                AURORA_ERR_INVALID_ARGUMENT,
                "swarm block statistics require at least one sample per block");
    AUR_REQUIRE(std::isfinite(r->reduced_field_td) && r->reduced_field_td >= 0.0,
                AURORA_ERR_INVALID_ARGUMENT,
                "swarm reduced fields must be finite and non-negative");
    AUR_REQUIRE(std::isfinite(r->initial_mean_energy_ev) && r->initial_mean_energy_ev >= 0.0,
                AURORA_ERR_INVALID_ARGUMENT,
                "swarm initial_mean_energy_ev must be finite and non-negative");
    AUR_REQUIRE(std::isfinite(r->max_energy_ev) && r->max_energy_ev > 0.0,
                AURORA_ERR_INVALID_ARGUMENT, "swarm max_energy_ev must be positive and finite");
    AUR_REQUIRE(r->max_energy_ev <= s.table_max_ev, AURORA_ERR_INVALID_ARGUMENT,
                "swarm max_energy_ev exceeds channel table coverage");
}

// ------------------------------------------- branching / resampled population
// Swarm.cpp:1063-1104 and systematic_resample (616-643).  Every electron of
// a step carries the same weight w: secondaries inherit their parent's and
// resampling gives all outputs W / N.  So the population is N velocities
// plus one weight, and the systematic resample of the M survivors and
// secondaries (equal weights) takes for output j the source
// ceil((u + j) M / N) - 1, where the cumulative weight first reaches the
// threshold (u + j) W / N.  Survivors come first, in order, then the
// secondaries in parent order.  Two forms of the same step:
//   k_br_small    up to kBrSmall electrons: one workgroup keeps the
//                 population in LDS and runs up to 512 steps in one launch.
//                 A step is bound by its chain of dependent phases, so
//                 launches are what it must not have: 512 electrons 25.0 ->
//                 10.4 us a step (six launches before).  512 threads up to
//                 512 electrons, else 1024 (1,024 electrons 13.8 us against
//                 17.7; the register cap of 1024 threads costs 4 % at 512);
//                 at 2,048 electrons (24.7 us) the launches take over (24.1)
//   three launches per step otherwise: collide (each 256-electron chunk
//                 compacts its survivors and secondaries in place), a
//                 one-workgroup scan of the chunk totals that also books the
//                 step, and the resample, which finds a source's chunk by
//                 bisecting the scanned totals (33,000 electrons 29 us a step)
constexpr int kBr = 256;
constexpr int kBrSmall = 2048;
constexpr int kBrSmallSteps = 512;

struct BranchArgs {
    float* v;                    // the population, 3 x N (SoA)
    float* pre;                  // survivors, compacted per chunk, 3 x N (SoA)
    float* sec;                  // secondaries, per chunk 2 kBr x 3 (per slot 2 x 3 in k_br_small)
    int32_t* tot;                // [chunks] survivors, then [chunks] secondaries
    int32_t* off;                // their exclusive sums
    long long* pop;              // survivors and secondaries of the step
    unsigned long long* step_counts;  // [candidates, nulls, chan...] of the step
    unsigned long long* totals;       // the same, summed over sampled steps
    unsigned* max_energy_bits;
    uint32_t* status;
    double* part;                // per resample block: sum v_x, sum energy (eV)
    double* state;               // [w, exposure, weighted[8], squared[8]]
    double* samples;             // [3][sampling]: mean v_x, mean energy, log W
    int64_t N, limit;
    int chunks;
    float half_kick, dt, max_energy_ev, ev_per_v2;
    uint64_t seed;
    int step, burn_in, sampling;
    uint32_t attach_mask;        // channels whose collision removes the electron
};

// One electron's step: kick, energy check, collisions, kick, check.  Returns
// whether it survives; v, t and err hold the outcome.
template <int NCH>
__device__ __forceinline__ bool br_electron(const BranchArgs& a, const MccParams& m,
                                            const XsView& X, const ChannelSel* chan, int64_t p,
                                            int step, float* v, MccTally<NCH>& t, float& emax,
                                            uint32_t& err) {
    v[0] += a.half_kick;
    const float e_pre = a.ev_per_v2 * (v[0] * v[0] + v[1] * v[1] + v[2] * v[2]);
    emax = fmaxf(emax, e_pre);
    if (e_pre > a.max_energy_ev) err |= DEV_ERR_ENERGY;
    Philox rng;
    rng.init(a.seed, 0u, static_cast<uint32_t>(p), static_cast<uint32_t>(step));
    mcc_collide<NCH>(m, X, chan, v, a.dt, rng, t);
    err |= t.err;
    v[0] += a.half_kick;
    const float e = a.ev_per_v2 * (v[0] * v[0] + v[1] * v[1] + v[2] * v[2]);
    emax = fmaxf(emax, e);
    if (e > a.max_energy_ev) err |= DEV_ERR_ENERGY;
    bool alive = true;
#pragma unroll
    for (int c = 0; c < NCH; ++c)
        if (((a.attach_mask >> c) & 1u) && t.chan[c]) alive = false;
    if (t.nsec > 2) err |= DEV_ERR_PRODUCTS;
    return alive;
}

// the step's resample offset u
__device__ __forceinline__ double br_offset(const BranchArgs& a, int step) {
    Philox rng;
    rng.init(a.seed, 1u, 0xFFFFFFFFu, static_cast<uint32_t>(step));
    return static_cast<double>(rng.u01());
}

__device__ __forceinline__ int64_t br_source(double u, int64_t j, int64_t M, int64_t N) {
    if (M == N) return j;
    const int64_t s = static_cast<int64_t>(ceil((u + static_cast<double>(j)) *
                                                static_cast<double>(M) / static_cast<double>(N))) - 1;
    return s < 0 ? 0 : (s > M - 1 ? M - 1 : s);
}

__device__ __forceinline__ double br_energy(const BranchArgs& a, float vx, float vy, float vz) {
    return static_cast<double>(a.ev_per_v2) *
           (static_cast<double>(vx) * vx + static_cast<double>(vy) * vy +
            static_cast<double>(vz) * vz);
}

// the checks of a step with A survivors and S secondaries (Swarm.cpp:1069-1100)
__device__ __forceinline__ uint32_t br_checks(const BranchArgs& a, int64_t A, int64_t S) {
    return (a.N + S > a.limit ? DEV_ERR_POPULATION : 0u) | (A + S == 0 ? DEV_ERR_EXTINCT : 0u);
}

__device__ __forceinline__ double br_weight(const BranchArgs& a, double w, int64_t M) {
    return (M == a.N || M == 0) ? w : w * static_cast<double>(M) / static_cast<double>(a.N);
}

template <int NCH>
__global__ void __launch_bounds__(kBr) k_br_collide(MccParams m, BranchArgs a) {
    __shared__ MccLds lds;
    __shared__ int wsum[kBr / 64];
    const XsView X = stage_tables(m, lds);
    const bool sampling = a.step >= a.burn_in;
    float emax = 0.f;
    uint32_t err = 0;
    for (int chunk = blockIdx.x; chunk < a.chunks; chunk += gridDim.x) {
        const int64_t first = static_cast<int64_t>(chunk) * kBr, p = first + threadIdx.x;
        const bool active = p < a.N;
        MccTally<NCH> t{};
        float v[3] = {0.f, 0.f, 0.f};
        bool alive = false;
        if (active) {
            v[0] = a.v[p]; v[1] = a.v[a.N + p]; v[2] = a.v[2 * a.N + p];
            alive = br_electron<NCH>(a, m, X, lds.chan, p, a.step, v, t, emax, err);
        }
        const int ns = active ? (t.nsec < 2 ? t.nsec : 2) : 0;
        // survivors (at most 256) and secondaries (512) in one scan
        int total = 0;
        const int ex = block_scan_int<kBr>((alive ? 1 : 0) | (ns << 16), wsum, total);
        if (threadIdx.x == 0) {
            a.tot[chunk] = total & 0xffff;
            a.tot[a.chunks + chunk] = total >> 16;
        }
        if (alive) {
            const int64_t d = first + (ex & 0xffff);
            a.pre[d] = v[0];
            a.pre[a.N + d] = v[1];
            a.pre[2 * a.N + d] = v[2];
        }
        float* sec = a.sec + 3 * (2 * first + (ex >> 16));
        // both slots unrolled: a runtime index into t.sec would put the
        // tally in scratch memory
#pragma unroll
        for (int k = 0; k < 2; ++k)
            if (k < ns)
#pragma unroll
                for (int d = 0; d < 3; ++d) sec[3 * k + d] = t.sec[k][d];
        if (sampling) {
            unsigned long long cnt[2 + NCH];
            cnt[0] = active ? t.candidates : 0;
            cnt[1] = active ? t.nulls : 0;
#pragma unroll
            for (int c = 0; c < NCH; ++c) cnt[2 + c] = active ? t.chan[c] : 0;
#pragma unroll
            for (int k = 0; k < 2 + NCH; ++k) {
                const unsigned long long x = wave_sum_u64(cnt[k]);
                if ((threadIdx.x & 63) == 0 && x) atomicAdd(a.step_counts + k, x);
            }
        }
    }
    for (int o = 32; o > 0; o >>= 1) {
        emax = fmaxf(emax, __shfl_xor(emax, o, 64));
        err |= __shfl_xor(err, o, 64);
    }
    if ((threadIdx.x & 63) == 0) {
        atomicMax(a.max_energy_bits, __float_as_uint(emax));
        if (err) atomicOr(a.status, err);
    }
}

// One workgroup between a step's collide and resample: the previous step's
// sample sums (fold), then (scan) the chunk totals scanned, the step's checks,
// weight and tallies booked.
__global__ void __launch_bounds__(kBr) k_br_book(BranchArgs a, int blocks, int nch, int fold,
                                                 int scan) {
    __shared__ int wsum[kBr / 64];
    const double n = static_cast<double>(a.N);
    if (fold) {
        double v[2] = {0.0, 0.0};
        for (int b = threadIdx.x; b < blocks; b += kBr) {
            v[0] += a.part[2 * b];
            v[1] += a.part[2 * b + 1];
        }
        const double sum = block_sum<2, kBr>(v);
        const int64_t k = a.step - 1 - a.burn_in;
        if (threadIdx.x < 2) a.samples[threadIdx.x * a.sampling + k] = sum / n;
    }
    if (!scan) return;
    const int64_t A = chunk_offsets<kBr>(a.tot, a.off, a.chunks, wsum);
    const int64_t S = chunk_offsets<kBr>(a.tot + a.chunks, a.off + a.chunks, a.chunks, wsum);
    if (threadIdx.x != 0) return;
    a.pop[0] = A;
    a.pop[1] = S;
    const uint32_t err = br_checks(a, A, S);
    if (err) atomicOr(a.status, err);
    const double w = a.state[0], w_new = br_weight(a, w, A + S);
    a.state[0] = w_new;
    if (a.step >= a.burn_in) {
        a.state[1] += n * w * static_cast<double>(a.dt);
        for (int c = 0; c < nch; ++c) {
            const double k = static_cast<double>(a.step_counts[2 + c]);
            a.state[2 + c] += w * k;
            a.state[10 + c] += w * w * k;
        }
        for (int c = 0; c < 2 + nch; ++c) a.totals[c] += a.step_counts[c];
        a.samples[2 * static_cast<int64_t>(a.sampling) + a.step - a.burn_in] = log(n * w_new);
    }
    for (int c = 0; c < 2 + nch; ++c) a.step_counts[c] = 0;
}

// the chunk holding element x of the scanned totals: the last one whose
// offset does not exceed x
__device__ __forceinline__ int br_chunk_of(const int32_t* off, int chunks, int64_t x) {
    int lo = 0, hi = chunks;          // off[0] = 0 <= x
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (off[mid] <= x) lo = mid; else hi = mid;
    }
    return lo;
}

__global__ void __launch_bounds__(kBr) k_br_resample(BranchArgs a) {
    const int64_t A = a.pop[0], M = A + a.pop[1];
    const double u = br_offset(a, a.step);
    double sums[2] = {0.0, 0.0};
    for (int64_t j = blockIdx.x * static_cast<int64_t>(kBr) + threadIdx.x; j < a.N;
         j += static_cast<int64_t>(gridDim.x) * kBr) {
        if (M == 0) break;                     // extinct: reported by the booking
        const int64_t src = br_source(u, j, M, a.N);
        float vx, vy, vz;
        if (src < A) {
            const int c = br_chunk_of(a.off, a.chunks, src);
            const int64_t d = static_cast<int64_t>(c) * kBr + (src - a.off[c]);
            vx = a.pre[d]; vy = a.pre[a.N + d]; vz = a.pre[2 * a.N + d];
        } else {
            const int32_t* off = a.off + a.chunks;
            const int c = br_chunk_of(off, a.chunks, src - A);
            const float* q = a.sec + 3 * (2 * static_cast<int64_t>(c) * kBr + (src - A - off[c]));
            vx = q[0]; vy = q[1]; vz = q[2];
        }
        a.v[j] = vx;
        a.v[a.N + j] = vy;
        a.v[2 * a.N + j] = vz;
        sums[0] += vx;
        sums[1] += br_energy(a, vx, vy, vz);
    }
    const double r = block_sum<2, kBr>(sums);
    if (threadIdx.x < 2) a.part[2 * blockIdx.x + threadIdx.x] = r;
}

// Steps [a.step, a.step + nsteps) of a population of at most kBrSmall by one
// workgroup.  Thread t owns electrons t, t + T, ...; a step has three
// phases with a barrier after the first two:
//   collide   each wave counts its survivors and secondaries per round
//   place     the (round, wave) counts are scanned by every wave on its own,
//             survivors and secondaries go to their order in pre (LDS;
//             entries past twice the population to the global overflow);
//             wave 0 books the step and the previous step's sample sums
//   resample  each thread reads its electrons' sources
// LDS: v[3][N], pre[3][2N], meta[N].
template <int NCH, int T>
__global__ void __launch_bounds__(T) k_br_small(MccParams m, BranchArgs a, int nsteps,
                                                float* overflow) {
    constexpr int W = T / 64, kRounds = kBrSmall / T;
    extern __shared__ __align__(16) float br_lds[];
    __shared__ MccLds lds;
    __shared__ uint32_t s_wave[kRounds * W];       // survivors | secondaries << 16
    __shared__ uint32_t s_cnt[2][2 + NCH];
    __shared__ double s_red[2][W];
    static_assert(kRounds * W <= 64, "one wave scans the (round, wave) counts");
    const int N = static_cast<int>(a.N), cap = 2 * N;
    float* v = br_lds;
    float* pre = br_lds + 3 * N;
    uint32_t* meta = reinterpret_cast<uint32_t*>(br_lds + 9 * N);
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    const int rounds = (N + T - 1) / T;
    for (int p = tid; p < N; p += T)
        for (int d = 0; d < 3; ++d) v[d * N + p] = a.v[d * a.N + p];
    if (tid < 2 * (2 + NCH)) (&s_cnt[0][0])[tid] = 0u;
    const XsView X = stage_tables(m, lds);         // ends with a barrier
    // wave 0 keeps the running state: w in every lane, lane c its channel's
    // sums and (c < 2 + NCH) counter c
    double w = a.state[0], exposure = a.state[1];
    double weighted = 0.0, squared = 0.0;
    unsigned long long counted = 0;
    if (wid == 0 && lane < NCH) {
        weighted = a.state[2 + lane];
        squared = a.state[10 + lane];
    }
    if (wid == 0 && lane < 2 + NCH) counted = a.totals[lane];
    const double n = static_cast<double>(N);
    double* vel_samples = a.samples;
    double* log_samples = a.samples + 2 * static_cast<int64_t>(a.sampling);
    auto book_sums = [&](int step) {               // the sums of `step`, by wave 0
        if (step < a.burn_in || lane >= 2) return;
        double sum = 0.0;
#pragma unroll
        for (int k = 0; k < W; ++k) sum += s_red[lane][k];
        vel_samples[lane * static_cast<int64_t>(a.sampling) + step - a.burn_in] = sum / n;
    };
    float emax = 0.f;
    uint32_t err = 0;
    for (int it = 0; it < nsteps; ++it) {
        const int step = a.step + it;
        const bool sampling = step >= a.burn_in;
        uint32_t* cnt = s_cnt[it & 1];
        for (int k = 0; k < rounds; ++k) {
            const int p = tid + k * T;
            const bool active = p < N;
            MccTally<NCH> t{};
            bool alive = false;
            if (active) {
                float u[3] = {v[p], v[N + p], v[2 * N + p]};
                alive = br_electron<NCH>(a, m, X, lds.chan, p, step, u, t, emax, err);
                v[p] = u[0];
                v[N + p] = u[1];
                v[2 * N + p] = u[2];
            }
            const int ns = active ? (t.nsec < 2 ? t.nsec : 2) : 0;
#pragma unroll
            for (int q = 0; q < 2; ++q)
                if (q < ns)
#pragma unroll
                    for (int d = 0; d < 3; ++d) a.sec[6 * p + 3 * q + d] = t.sec[q][d];
            const uint64_t ma = __ballot(alive), m1 = __ballot(ns > 0), m2 = __ballot(ns > 1);
            const uint64_t below = (uint64_t{1} << lane) - 1;
            if (active)
                meta[p] = (alive ? 1u : 0u) | (static_cast<uint32_t>(ns) << 1) |
                          (static_cast<uint32_t>(__popcll(ma & below)) << 8) |
                          (static_cast<uint32_t>(__popcll(m1 & below) + __popcll(m2 & below)) << 16);
            if (lane == 0)
                s_wave[k * W + wid] = static_cast<uint32_t>(__popcll(ma)) |
                                      (static_cast<uint32_t>(__popcll(m1) + __popcll(m2)) << 16);
            if (sampling && active && t.candidates) {
                atomicAdd(cnt, t.candidates);
                if (t.nulls) atomicAdd(cnt + 1, t.nulls);
#pragma unroll
                for (int c = 0; c < NCH; ++c)
                    if (t.chan[c]) atomicAdd(cnt + 2 + c, t.chan[c]);
            }
        }
        __syncthreads();
        // at most 2048 survivors and 4096 secondaries: both halves stay below 2^16
        uint32_t x = lane < rounds * W ? s_wave[lane] : 0u, incl = x;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const uint32_t y = __shfl_up(incl, d, 64);
            if (lane >= d) incl += y;
        }
        const uint32_t total = __shfl(incl, 63, 64), excl = incl - x;
        const int A = static_cast<int>(total & 0xffffu), S = static_cast<int>(total >> 16);
        const int M = A + S;
        auto place = [&](int d, float x0, float x1, float x2) {
            if (d < cap) {
                pre[d] = x0;
                pre[cap + d] = x1;
                pre[2 * cap + d] = x2;
            } else {
                overflow[3 * (d - cap)] = x0;
                overflow[3 * (d - cap) + 1] = x1;
                overflow[3 * (d - cap) + 2] = x2;
            }
        };
        for (int k = 0; k < rounds; ++k) {
            const uint32_t base = __shfl(excl, k * W + wid, 64);
            const int p = tid + k * T;
            if (p >= N) continue;
            const uint32_t mt = meta[p];
            if (mt & 1u)
                place(static_cast<int>((base & 0xffffu) + ((mt >> 8) & 0xffu)), v[p], v[N + p],
                      v[2 * N + p]);
            const int ns = static_cast<int>((mt >> 1) & 3u);
            for (int q = 0; q < ns; ++q)
                place(A + static_cast<int>((base >> 16) + (mt >> 16)) + q, a.sec[6 * p + 3 * q],
                      a.sec[6 * p + 3 * q + 1], a.sec[6 * p + 3 * q + 2]);
        }
        if (wid == 0) {
            if (it > 0) book_sums(step - 1);
            err |= br_checks(a, A, S);
            const double w_new = br_weight(a, w, M);
            if (sampling) {
                exposure += n * w * static_cast<double>(a.dt);
                if (lane < NCH) {
                    const double k = static_cast<double>(cnt[2 + lane]);
                    weighted += w * k;
                    squared += w * w * k;
                }
                if (lane < 2 + NCH) counted += cnt[lane];
                // (the logarithm is taken for all steps of the launch at its end)
                if (lane == 0) log_samples[step - a.burn_in] = n * w_new;
            }
            w = w_new;
            wave_lds_fence();   // lane c + 2 clears the counter that lane c has read
            if (lane < 2 + NCH) cnt[lane] = 0u;
        }
        __syncthreads();
        const double u = br_offset(a, step);
        double sums[2] = {0.0, 0.0};
        if (M > 0)                                 // else extinct: reported
            for (int p = tid; p < N; p += T) {
                const int src = static_cast<int>(br_source(u, p, M, N));
                float vx, vy, vz;
                if (src < cap) {
                    vx = pre[src]; vy = pre[cap + src]; vz = pre[2 * cap + src];
                } else {
                    const float* q = overflow + 3 * (src - cap);
                    vx = q[0]; vy = q[1]; vz = q[2];
                }
                v[p] = vx;
                v[N + p] = vy;
                v[2 * N + p] = vz;
                sums[0] += vx;
                sums[1] += br_energy(a, vx, vy, vz);
            }
        if (sampling) {
            const double s0 = wave_sum(sums[0]), s1 = wave_sum(sums[1]);
            if (lane == 0) {
                s_red[0][wid] = s0;
                s_red[1][wid] = s1;
            }
        }
    }
    __syncthreads();
    if (wid == 0) {
        book_sums(a.step + nsteps - 1);
        if (lane == 0) {
            a.state[0] = w;
            a.state[1] = exposure;
        }
        if (lane < NCH) {
            a.state[2 + lane] = weighted;
            a.state[10 + lane] = squared;
        }
        if (lane < 2 + NCH) a.totals[lane] = counted;
    }
    for (int it = tid; it < nsteps; it += T) {
        const int k = a.step + it - a.burn_in;
        if (k >= 0) log_samples[k] = log(log_samples[k]);
    }
    for (int p = tid; p < N; p += T)
        for (int d = 0; d < 3; ++d) a.v[d * a.N + p] = v[d * N + p];
    for (int o = 32; o > 0; o >>= 1) {
        emax = fmaxf(emax, __shfl_xor(emax, o, 64));
        err |= __shfl_xor(err, o, 64);
    }
    if (lane == 0) {
        atomicMax(a.max_energy_bits, __float_as_uint(emax));
        if (err) atomicOr(a.status, err);
    }
}

// block_slope_and_error (Swarm.cpp:136-197)
void block_slope_error(const double* y, int64_t n, double dt, int64_t blocks, double& slope,
                       double& se) {
    const int64_t size = n / blocks;
    std::vector<double> slopes(static_cast<size_t>(blocks));
    for (int64_t b = 0; b < blocks; ++b) {
        const double* x = y + b * size;
        const double mid = 0.5 * static_cast<double>(size - 1);
        double mean = 0.0;
        for (int64_t i = 0; i < size; ++i) mean += x[i];
        mean /= static_cast<double>(size);
        double cov = 0.0, var = 0.0;
        for (int64_t i = 0; i < size; ++i) {
            const double t = static_cast<double>(i) - mid;
            cov += t * (x[i] - mean);
            var += t * t;
        }
        slopes[static_cast<size_t>(b)] = cov / (var * dt);
    }
    block_mean_error(slopes, slope, se);
}

// Queues one k_swarm launch of every admitted, unfinished request (up to
// max_steps steps each) and records the launch's event; steps are booked at
// once, and the requests this launch completes are finalised by
// collect_launch.
void queue_launch(Context& c, SwarmState& s, int64_t max_steps) {
    LaunchBuffers& b = s.buf[s.cur];
    if (b.done) AUR_HIP(hipEventSynchronize(b.done));   // the buffers' previous launch
    const MccParams m = swarm_params(s);
    std::vector<RequestDesc> descs;
    std::vector<WorkItem> items;
    s.finishing.clear();
    for (auto& kv : s.active) {
        RequestState& r = *kv.second;
        const auto& q = r.req;
        const int64_t remaining = q.steps - r.steps_done;
        if (remaining <= 0) continue;
        const int64_t ns = std::min(max_steps, remaining);
        RequestDesc d{};
        const int64_t n = q.particles;
        d.vx = r.v;
        d.vy = r.v + n;
        d.vz = r.v + 2 * n;
        d.dx = r.dx;
        d.moments = r.moments;
        d.part = r.part;
        d.counts = r.counts;
        d.max_energy_bits = r.maxe;
        d.status = r.status;
        d.particles = n;
        const double efield = q.reduced_field_td * kTownsend * s.gas.neutral_density;
        const double accel = -kElementaryCharge * efield / kElectronMass;
        d.half_kick = static_cast<float>(0.5 * accel * q.timestep);
        d.dt = static_cast<float>(q.timestep);
        d.ev_per_v2 = static_cast<float>(0.5 * kElectronMass / kElementaryCharge);
        d.v2_max = v2_ceiling(static_cast<float>(q.max_energy_ev), d.ev_per_v2);
        d.scale_v = static_cast<float>(scales(q).first);
        d.scale_e = static_cast<float>(scales(q).second);
        d.step0 = static_cast<int>(r.steps_done);
        d.nsteps = static_cast<int>(ns);
        d.burn_in = static_cast<int>(q.burn_in);
        d.sampling = static_cast<int>(q.steps - q.burn_in);
        d.blocks = static_cast<int>(q.blocks);
        d.no_candidate = no_candidate_draws(d.dt, m.inv_max_frequency);
        d.seed = q.seed;
        const int ridx = static_cast<int>(descs.size());
        descs.push_back(d);
        for (int64_t ch = 0; ch < r.chunks; ++ch) items.push_back(WorkItem{ridx, static_cast<int>(ch)});
        r.steps_done += ns;
        if (r.steps_done >= q.steps) s.finishing.push_back(kv.first);
    }
    if (items.empty()) return;
    if (b.cap_descs < descs.size()) {
        if (b.h_descs) AUR_HIP(hipHostFree(b.h_descs));
        b.h_descs = nullptr;
        b.cap_descs = descs.size() * 2;
        AUR_HIP(hipHostMalloc(reinterpret_cast<void**>(&b.h_descs),
                              b.cap_descs * sizeof(RequestDesc), hipHostMallocDefault));
        b.descs.alloc(b.cap_descs);
    }
    if (b.cap_items < items.size()) {
        if (b.h_items) AUR_HIP(hipHostFree(b.h_items));
        b.h_items = nullptr;
        b.cap_items = items.size() * 2;
        AUR_HIP(hipHostMalloc(reinterpret_cast<void**>(&b.h_items), b.cap_items * sizeof(WorkItem),
                              hipHostMallocDefault));
        b.items.alloc(b.cap_items);
    }
    if (!b.head.ptr) b.head.alloc(1);
    if (!b.done) AUR_HIP(hipEventCreateWithFlags(&b.done, hipEventDisableTiming));
    std::memcpy(b.h_descs, descs.data(), descs.size() * sizeof(RequestDesc));
    std::memcpy(b.h_items, items.data(), items.size() * sizeof(WorkItem));
    AUR_HIP(hipMemcpyAsync(b.descs.ptr, b.h_descs, descs.size() * sizeof(RequestDesc),
                           hipMemcpyHostToDevice, c.stream));
    AUR_HIP(hipMemcpyAsync(b.items.ptr, b.h_items, items.size() * sizeof(WorkItem),
                           hipMemcpyHostToDevice, c.stream));
    AUR_HIP(hipMemsetAsync(b.head.ptr, 0, sizeof(int), c.stream));
    if (s.blocks_per_cu == 0) {
        // as many workgroups as the CUs hold at once: the kernel pulls
        // chunks from the queue, so more would only wait
        int per_cu = 0;
        with_model(m.nchan, mcc_tables_fit(m), [&]<int NCH, bool LDS>() {
            AUR_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_swarm<NCH, LDS>, kChunk, 0));
        });
        s.blocks_per_cu = per_cu > 0 ? per_cu : 4;
    }
    int64_t grid = static_cast<int64_t>(c.cu_count) * s.blocks_per_cu;
    if (grid > static_cast<int64_t>(items.size())) grid = static_cast<int64_t>(items.size());
    {
        KernelScope ks(c, "swarm");
        with_model(m.nchan, mcc_tables_fit(m), [&]<int NCH, bool LDS>() {
            k_swarm<NCH, LDS><<<static_cast<unsigned>(grid), kChunk, 0, c.stream>>>(
                m, b.descs.ptr, b.items.ptr, static_cast<int>(items.size()), b.head.ptr);
        });
        AUR_HIP(hipGetLastError());
    }
    AUR_HIP(hipEventRecord(b.done, c.stream));
    s.in_flight = true;
    s.cur ^= 1;
}

// Completes the launch in flight: waits for it (wait) or returns while it
// still runs; once done, finalises the requests it completed.
void collect_launch(Context& c, SwarmState& s, bool wait) {
    LaunchBuffers& b = s.buf[s.cur ^ 1];
    if (wait) {
        AUR_HIP(hipEventSynchronize(b.done));
    } else {
        const hipError_t q = hipEventQuery(b.done);
        if (q == hipErrorNotReady) return;
        AUR_HIP(q);
    }
    s.in_flight = false;
    for (int64_t handle : s.finishing) {
        auto it = s.active.find(handle);
        if (it == s.active.end()) continue;
        finalize(c, s, handle, *it->second);
        keep_slab(s, std::move(it->second->slab));
        s.active.erase(it);
    }
    s.finishing.clear();
}

}  // namespace

MccModelHost& swarm_gas_model(Context& c) {
    SwarmState& s = state(c);
    AUR_REQUIRE(s.gas_loaded, AURORA_ERR_INVALID_ARGUMENT, "load the swarm gas first");
    AUR_REQUIRE(s.active.empty(), AURORA_ERR_INVALID_ARGUMENT,
                "the swarm gas cannot change while requests are running");
    return s.gas;
}

void swarm_destroy(Context& c) {
    if (c.swarm) {
        (void)hipStreamSynchronize(c.stream);   // a launch may still read the buffers
        delete static_cast<SwarmState*>(c.swarm);
        c.swarm = nullptr;
    }
}

bool release_spares(Context& c) {
    if (!c.swarm) return false;
    SwarmState& s = *static_cast<SwarmState*>(c.swarm);
    const bool any = !s.spare.empty();
    s.spare.clear();
    s.spare_bytes = 0;
    return any;
}

}  // namespace aurora

using namespace aurora;

extern "C" {

int aurora_hip_swarm_gas(aurora_hip_ctx* h, int nchan, const int* kind, const double* threshold,
                         const int64_t* rows, const double* const* energy,
                         const double* const* sigma, double neutral_density,
                         double max_frequency, int64_t max_candidates, double neutral_mass,
                         double neutral_temperature) {
    return guarded(h, [&](Context& c) {
        SwarmState& s = state(c);
        AUR_REQUIRE(s.active.empty(), AURORA_ERR_INVALID_ARGUMENT,
                    "the swarm gas cannot change while requests are running");
        AUR_REQUIRE(std::isfinite(neutral_temperature) && neutral_temperature >= 0.0,
                    AURORA_ERR_INVALID_ARGUMENT,
                    "swarm neutral_temperature must be finite and non-negative");
        AUR_REQUIRE(std::isfinite(neutral_mass) && neutral_mass > 0.0,
                    AURORA_ERR_INVALID_ARGUMENT, "gas dataset requires positive neutral_mass");
        bool elastic = false;
        for (int k = 0; k < nchan; ++k) elastic = elastic || kind[k] == AURORA_ELASTIC;
        AUR_REQUIRE(elastic, AURORA_ERR_INVALID_ARGUMENT,
                    "electron swarm benchmark requires an elastic channel");
        // model checks and tables (the 1D MCC model loader's)
        MccModelHost& g = s.gas;
        load_mcc_model(g, nchan, kind, threshold, rows, energy, sigma, neutral_density,
                       max_frequency, max_candidates, kElectronMass, neutral_mass,
                       neutral_temperature);
        // energy ceiling of the tables (Swarm.cpp:517-526), eV
        double emax_ev = 1e300;
        for (int k = 0; k < nchan; ++k)
            emax_ev = std::min(emax_ev, energy[k][rows[k] - 1] / kElementaryCharge);
        s.table_max_ev = emax_ev;
        s.gas_loaded = true;
    });
}

uint64_t aurora_hip_swarm_footprint(const aurora_hip_swarm_request* r) {
    return r ? footprint_of(*r) : 0;
}

int aurora_hip_swarm_submit(aurora_hip_ctx* h, const aurora_hip_swarm_request* r,
                            uint64_t hbm_budget, int64_t* handle) {
    return guarded(h, [&](Context& c) {
        SwarmState& s = state(c);
        AUR_REQUIRE(s.gas_loaded, AURORA_ERR_INVALID_ARGUMENT, "load the swarm gas first");
        AUR_REQUIRE(r, AURORA_ERR_INVALID_ARGUMENT, "null request");
        validate_request(s, r);
        for (int k = 0; k < s.gas.nchan; ++k)
            AUR_REQUIRE(s.gas.kind[k] != AURORA_ATTACHMENT, AURORA_ERR_UNSUPPORTED,
                        "fixed-population swarm does not support attachment; use "
                        "population_model = branching_resampled");
        const uint64_t fp = footprint_of(*r);
        if (hbm_budget && s.bytes_in_use + fp > hbm_budget)
            throw Failure{AURORA_ERR_CAPACITY, "swarm request does not fit the HBM budget now"};
        auto st = std::make_unique<RequestState>();
        st->req = *r;
        st->chunks = (r->particles + kChunk - 1) / kChunk;
        const RequestLayout lay(*r, st->chunks);
        // A request holds its footprint, as its admission counts, so that a
        // budget has room for every request whose footprint it has room for.
        // On a context that was never given a budget it may hold up to four
        // times that in a spare slab, and is booked with what it holds.
        s.budgeted = s.budgeted || hbm_budget != 0;
        st->slab = take_spare(s, lay.bytes, s.budgeted ? fp : 4 * fp);
        st->footprint = std::max<uint64_t>(fp, st->slab.count);
        if (hbm_budget) fit_budget(s, st->footprint, hbm_budget);
        if (!st->slab.ptr) st->slab.alloc(lay.bytes);
        uint8_t* base = st->slab.ptr;
        st->part = reinterpret_cast<long long*>(base);
        st->counts = reinterpret_cast<unsigned long long*>(base + lay.counts);
        st->maxe = reinterpret_cast<unsigned*>(base + lay.maxe);
        st->status = reinterpret_cast<uint32_t*>(base + lay.status);
        st->moments = reinterpret_cast<double*>(base + lay.moments);
        st->v = reinterpret_cast<float*>(base + lay.v);
        st->dx = reinterpret_cast<float*>(base + lay.dx);
        AUR_HIP(hipMemsetAsync(base, 0, lay.zeroed, c.stream));
        const double sigma =
            std::sqrt(2.0 * r->initial_mean_energy_ev * kElementaryCharge / (3.0 * kElectronMass));
        const int64_t n = r->particles;
        int64_t g = (n + 255) / 256;
        if (g > 4096) g = 4096;
        k_swarm_init<<<static_cast<unsigned>(g), 256, 0, c.stream>>>(
            st->v, st->v + n, st->v + 2 * n, n, static_cast<float>(sigma), r->seed);
        AUR_HIP(hipGetLastError());
        s.bytes_in_use += st->footprint;
        const int64_t id = s.next_handle++;
        s.active[id] = std::move(st);
        if (handle) *handle = id;
    });
}

int aurora_hip_swarm_launch(aurora_hip_ctx* h, int64_t max_steps, int64_t* active_out) {
    return guarded(h, [&](Context& c) {
        SwarmState& s = state(c);
        AUR_REQUIRE(max_steps > 0, AURORA_ERR_INVALID_ARGUMENT, "max_steps must be positive");
        if (s.in_flight) collect_launch(c, s, true);
        queue_launch(c, s, max_steps);
        if (active_out) *active_out = static_cast<int64_t>(s.active.size());
    });
}

int aurora_hip_swarm_collect(aurora_hip_ctx* h, int wait, int* busy) {
    return guarded(h, [&](Context& c) {
        SwarmState& s = state(c);
        if (s.in_flight) collect_launch(c, s, wait != 0);
        if (busy) *busy = s.in_flight ? 1 : 0;
        flush_timers(c);
    });
}

int aurora_hip_swarm_advance(aurora_hip_ctx* h, int64_t max_steps, int64_t* active_out) {
    return guarded(h, [&](Context& c) {
        SwarmState& s = state(c);
        AUR_REQUIRE(max_steps > 0, AURORA_ERR_INVALID_ARGUMENT, "max_steps must be positive");
        if (s.in_flight) collect_launch(c, s, true);
        queue_launch(c, s, max_steps);
        if (s.in_flight) collect_launch(c, s, true);
        if (active_out) *active_out = static_cast<int64_t>(s.active.size());
        flush_timers(c);
    });
}

int aurora_hip_swarm_poll(aurora_hip_ctx* h, int64_t handle, int* done,
                          aurora_hip_swarm_result* result) {
    return guarded(h, [&](Context& c) {
        SwarmState& s = state(c);
        auto it = s.finished.find(handle);
        if (it != s.finished.end()) {
            if (done) *done = 1;
            if (result) *result = it->second;
            s.finished.erase(it);
            return;
        }
        AUR_REQUIRE(s.active.count(handle), AURORA_ERR_NOT_FOUND, "unknown swarm request handle");
        if (done) *done = 0;
    });
}

int aurora_hip_swarm_branching(aurora_hip_ctx* h, const aurora_hip_swarm_request* r,
                               int64_t population_limit, aurora_hip_swarm_result* result,
                               aurora_hip_swarm_growth* growth) {
    return guarded(h, [&](Context& c) {
        SwarmState& s = state(c);
        AUR_REQUIRE(s.gas_loaded, AURORA_ERR_INVALID_ARGUMENT, "load the swarm gas first");
        AUR_REQUIRE(r && result && growth, AURORA_ERR_INVALID_ARGUMENT, "null argument");
        validate_request(s, r);
        const int64_t N = r->particles, S = r->steps - r->burn_in;
        // Swarm.cpp:327-335, 373-379, 553-557
        AUR_REQUIRE(population_limit > N && population_limit <= 10000000 - N,
                    AURORA_ERR_INVALID_ARGUMENT,
                    "branching swarm population_limit must exceed particles and "
                    "population_limit + particles must not exceed the allocation safety "
                    "limit of 10000000");
        AUR_REQUIRE(S % r->blocks == 0, AURORA_ERR_INVALID_ARGUMENT,
                    "swarm sampling steps must be divisible by uncertainty_blocks");
        AUR_REQUIRE(S / r->blocks >= 2, AURORA_ERR_INVALID_ARGUMENT,
                    "branching swarm requires at least two sampling steps per uncertainty "
                    "block");
        uint32_t attach = 0;
        bool creates = false;
        for (int k = 0; k < s.gas.nchan; ++k) {
            if (s.gas.kind[k] == AURORA_ATTACHMENT) attach |= 1u << k;
            creates = creates || s.gas.kind[k] == AURORA_ATTACHMENT ||
                      s.gas.kind[k] == AURORA_IONIZATION;
        }
        AUR_REQUIRE(creates, AURORA_ERR_INVALID_ARGUMENT,
                    "branching swarm requires an ionization or attachment channel");
        const bool small = N <= kBrSmall;
        const int nch = s.gas.nchan;
        const int chunks = static_cast<int>((N + kBr - 1) / kBr);
        DevBuf<float> v, pre, sec;
        DevBuf<int32_t> ctot, coff;
        DevBuf<long long> pop;
        DevBuf<unsigned long long> counts;     // step counters, then totals
        DevBuf<unsigned> maxe;
        DevBuf<uint32_t> status;
        DevBuf<double> part, st, samples;
        v.alloc(static_cast<size_t>(3 * N));
        // survivors; in the small form the entries past twice the population
        pre.alloc(static_cast<size_t>(3 * N));
        sec.alloc(static_cast<size_t>(6) * chunks * kBr);
        if (!small) {
            ctot.alloc(static_cast<size_t>(2 * chunks));
            coff.alloc(static_cast<size_t>(2 * chunks));
            pop.alloc(2);
        }
        counts.alloc(2 * (kMaxChannels + 2));
        maxe.alloc(1);
        status.alloc(1);
        int64_t g = chunks;
        if (g > static_cast<int64_t>(c.cu_count) * 8) g = static_cast<int64_t>(c.cu_count) * 8;
        part.alloc(static_cast<size_t>(2 * g));
        st.alloc(18);
        samples.alloc(static_cast<size_t>(3 * S));
        AUR_HIP(hipMemsetAsync(counts.ptr, 0, counts.count * 8, c.stream));
        AUR_HIP(hipMemsetAsync(maxe.ptr, 0, 4, c.stream));
        AUR_HIP(hipMemsetAsync(status.ptr, 0, 4, c.stream));
        double st0[18] = {1.0};
        AUR_HIP(hipMemcpyAsync(st.ptr, st0, sizeof st0, hipMemcpyHostToDevice, c.stream));
        const double sigma =
            std::sqrt(2.0 * r->initial_mean_energy_ev * kElementaryCharge / (3.0 * kElectronMass));
        k_swarm_init<<<static_cast<unsigned>(std::min<int64_t>(g, 4096)), 256, 0, c.stream>>>(
            v.ptr, v.ptr + N, v.ptr + 2 * N, N, static_cast<float>(sigma), r->seed);
        AUR_HIP(hipGetLastError());
        BranchArgs a{};
        a.v = v.ptr;
        a.pre = pre.ptr;
        a.sec = sec.ptr;
        a.tot = ctot.ptr;
        a.off = coff.ptr;
        a.pop = pop.ptr;
        a.step_counts = counts.ptr;
        a.totals = counts.ptr + kMaxChannels + 2;
        a.max_energy_bits = maxe.ptr;
        a.status = status.ptr;
        a.part = part.ptr;
        a.state = st.ptr;
        a.samples = samples.ptr;
        a.N = N;
        a.limit = population_limit;
        a.chunks = chunks;
        const double efield = r->reduced_field_td * kTownsend * s.gas.neutral_density;
        a.half_kick = static_cast<float>(0.5 * (-kElementaryCharge * efield / kElectronMass) *
                                         r->timestep);
        a.dt = static_cast<float>(r->timestep);
        a.max_energy_ev = static_cast<float>(r->max_energy_ev);
        a.ev_per_v2 = static_cast<float>(0.5 * kElectronMass / kElementaryCharge);
        a.seed = r->seed;
        a.burn_in = static_cast<int>(r->burn_in);
        a.sampling = static_cast<int>(S);
        a.attach_mask = attach;
        const MccParams m = swarm_params(s);
        auto check = [&]() {
            uint32_t err = 0;
            AUR_HIP(hipMemcpyAsync(&err, status.ptr, 4, hipMemcpyDeviceToHost, c.stream));
            AUR_HIP(hipStreamSynchronize(c.stream));
            if (!err) return;
            const std::string td = std::to_string(r->reduced_field_td);
            if (err & DEV_ERR_POPULATION)
                throw Failure{AURORA_ERR_POPULATION,
                              "branching swarm exceeded population_limit before resampling; "
                              "reduce timestep or raise the limit on an appropriate compute "
                              "host"};
            if (err & DEV_ERR_EXTINCT)
                throw Failure{AURORA_ERR_POPULATION,
                              "branching swarm electron ensemble became extinct; increase "
                              "particles or reduce timestep"};
            if (err & DEV_ERR_ENERGY)
                throw Failure{AURORA_ERR_ENERGY_ABOVE_MAX,
                              "swarm particle energy exceeded max_energy_ev at E/N=" + td +
                                  " Td"};
            if (err & DEV_ERR_RATE)
                throw Failure{AURORA_ERR_RATE_ABOVE_BOUND,
                              "MCC total collision frequency exceeds configured max_frequency"};
            if (err & DEV_ERR_CANDIDATES)
                throw Failure{AURORA_ERR_CANDIDATE_LIMIT,
                              "MCC candidate limit exceeded; reduce dt or increase "
                              "max_candidates_per_particle"};
            if (err & DEV_ERR_PRODUCTS)
                throw Failure{AURORA_ERR_UNSUPPORTED,
                              "more than two ionizations of one electron in one step; reduce "
                              "timestep"};
            throw Failure{AURORA_ERR_INVALID_ARGUMENT, "MCC particle velocity must be finite"};
        };
        {
            KernelScope ks(c, "swarm_branching");
            // errors are looked for every 512 steps (kBrSmallSteps)
            for (int64_t step = 0; small && step < r->steps; step += kBrSmallSteps) {
                a.step = static_cast<int>(step);
                const int k = static_cast<int>(std::min<int64_t>(kBrSmallSteps, r->steps - step));
                const size_t shmem = static_cast<size_t>(10 * N) * sizeof(float);
                with_nchan(m.nchan, [&]<int NCH>() {
                    if (N <= 512)
                        k_br_small<NCH, 512><<<1, 512, shmem, c.stream>>>(m, a, k, pre.ptr);
                    else
                        k_br_small<NCH, 1024><<<1, 1024, shmem, c.stream>>>(m, a, k, pre.ptr);
                });
                AUR_HIP(hipGetLastError());
                if (step + k < r->steps) check();
            }
            for (int64_t step = 0; !small && step < r->steps; ++step) {
                a.step = static_cast<int>(step);
                with_nchan(m.nchan, [&]<int NCH>() {
                    k_br_collide<NCH><<<static_cast<unsigned>(g), kBr, 0, c.stream>>>(m, a);
                });
                k_br_book<<<1, kBr, 0, c.stream>>>(a, static_cast<int>(g), nch,
                                                   step > r->burn_in ? 1 : 0, 1);
                k_br_resample<<<static_cast<unsigned>(g), kBr, 0, c.stream>>>(a);
                AUR_HIP(hipGetLastError());
                if ((step & 511) == 511) check();
            }
            if (!small) {
                // the last step's sample sums
                a.step = static_cast<int>(r->steps);
                k_br_book<<<1, kBr, 0, c.stream>>>(a, static_cast<int>(g), nch, 1, 0);
                AUR_HIP(hipGetLastError());
            }
        }
        check();
        std::vector<double> smp(static_cast<size_t>(3 * S));
        double sv[18];
        unsigned long long tot[kMaxChannels + 2];
        unsigned mx = 0;
        AUR_HIP(hipMemcpy(smp.data(), samples.ptr, smp.size() * 8, hipMemcpyDeviceToHost));
        AUR_HIP(hipMemcpy(sv, st.ptr, sizeof sv, hipMemcpyDeviceToHost));
        AUR_HIP(hipMemcpy(tot, a.totals, sizeof tot, hipMemcpyDeviceToHost));
        AUR_HIP(hipMemcpy(&mx, maxe.ptr, 4, hipMemcpyDeviceToHost));
        // Swarm.cpp:1106-1245 on the samples and tallies
        aurora_hip_swarm_result out{};
        aurora_hip_swarm_growth gr{};
        const int64_t B = r->blocks, len = S / B;
        std::vector<double> vm(static_cast<size_t>(B)), em(static_cast<size_t>(B));
        for (int64_t b = 0; b < B; ++b) {
            double a0 = 0.0, a1 = 0.0;
            for (int64_t i = b * len; i < (b + 1) * len; ++i) {
                a0 += smp[static_cast<size_t>(i)];
                a1 += smp[static_cast<size_t>(S + i)];
            }
            vm[static_cast<size_t>(b)] = a0 / static_cast<double>(len);
            em[static_cast<size_t>(b)] = a1 / static_cast<double>(len);
        }
        double mv, sev, me, see;
        block_mean_error(vm, mv, sev);
        block_mean_error(em, me, see);
        out.drift = -mv;
        out.drift_se = sev;
        out.mean_energy_ev = me;
        out.mean_energy_se = see;
        const double exposure = sv[1];
        out.candidates = tot[0];
        out.nulls = tot[1];
        for (int k = 0; k < nch; ++k) {
            out.collisions[k] = tot[2 + k];
            out.rate[k] = sv[2 + k] / exposure;
            out.rate_se[k] = std::sqrt(sv[10 + k]) / exposure;
            if (s.gas.kind[k] == AURORA_IONIZATION) {
                out.ionization_rate += out.rate[k];
                out.ionization_rate_se = std::hypot(out.ionization_rate_se, out.rate_se[k]);
            } else if (s.gas.kind[k] == AURORA_ATTACHMENT) {
                gr.attachment_rate += out.rate[k];
                gr.attachment_rate_se = std::hypot(gr.attachment_rate_se, out.rate_se[k]);
            }
        }
        float mxf;
        std::memcpy(&mxf, &mx, sizeof mxf);
        out.max_energy_ev = mxf;
        out.status = AURORA_OK;
        gr.initial_weight = static_cast<double>(N);
        gr.final_weight = static_cast<double>(N) * sv[0];
        gr.final_particles = N;
        gr.net_creation_rate = out.ionization_rate - gr.attachment_rate;
        gr.net_creation_rate_se = std::hypot(out.ionization_rate_se, gr.attachment_rate_se);
        block_slope_error(smp.data() + 2 * S, S, r->timestep, B, gr.growth_rate,
                          gr.growth_rate_se);
        if (out.drift > 0.0) {
            const double d = out.drift, de = out.drift_se;
            gr.townsend_available = 1;
            gr.townsend_growth = gr.growth_rate / d;
            gr.townsend_growth_se =
                std::hypot(gr.growth_rate_se / d, gr.growth_rate * de / (d * d));
            gr.townsend_rate_balance = gr.net_creation_rate / d;
            gr.townsend_rate_balance_se =
                std::hypot(gr.net_creation_rate_se / d, gr.net_creation_rate * de / (d * d));
        }
        *result = out;
        *growth = gr;
        flush_timers(c);
    });
}

}  // extern "C"
