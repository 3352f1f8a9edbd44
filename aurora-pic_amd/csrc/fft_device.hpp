// fft_device.hpp - FP64 complex transforms of short lines in LDS, one axis of
// the 2D/3D Poisson solve per kernel.  Two forms with one interface, passed
// to the kernels by value:
//   Pow2Axis<LOG2N>  power-of-two lines up to 1024 points: radix-2 stages,
//                    two or three per LDS pass, sizes known to the compiler
//   MixedAxis        every other length (and 2048): a mixed-radix plan
// Both are decimations in time: element e of a line is stored at slot(e)
// (bit- or digit-reversed), the passes run in place, and the spectrum comes
// out in natural order.  X[k] = sum x[j] e^{-2 pi i jk/n}; the inverse uses
// conjugate twiddles, unscaled (FieldSolver.cpp:171-214).
#pragma once

#include "aurora_internal.hpp"

namespace aurora {

__device__ __forceinline__ double2 cmul(double2 a, double2 b) {
    return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}

// x / d by one high multiply: with m = ceil(2^32 / d) the error m d - 2^32 is
// below d (and 0 for a power of two), so the quotient is exact for
// x < 2^32 / d; the lines and elements divided here stay below 2^21 with
// divisors up to 1024 (2048 is a power of two)
struct FastDiv {
    uint32_t d = 1, m = 0;
    __device__ __forceinline__ int operator()(int x) const {
        return d == 1 ? x : static_cast<int>(__umulhi(static_cast<uint32_t>(x), m));
    }
};
inline FastDiv fast_div(int64_t d) {
    FastDiv f;
    f.d = static_cast<uint32_t>(d);
    f.m = d == 1 ? 0u : static_cast<uint32_t>(((uint64_t{1} << 32) + d - 1) / d);
    return f;
}

// complex elements one block's field buffer holds (20 KiB): lines of N take
// N + N/8 + 1 elements; small buffers let more blocks share a CU
constexpr int kLineLds = 1280;
constexpr int kFftThreads = 256;

// lines per block as a power of two: the LDS budget over the padded line
// length (n + n/8 + 1), at most 64
constexpr int lines_shift(int64_t budget, int64_t n) {
    const int64_t ls = n + n / 8 + 1;
    int l = 0;
    while ((int64_t{2} << l) * ls <= budget && l < 6) ++l;
    return l;
}

// LDS layout: element i of line b at b*LS + i + (i>>3) with LS = N + N/8 + 1.
// The pad after every 8 elements spreads the 8-element register blocks of
// the first pass over the banks, and the odd line stride spreads the column
// accesses of the strided axes.
template <int LOG2N>
struct Pow2Axis {
    static constexpr int N = 1 << LOG2N;
    static constexpr int LS = N + (N >> 3) + 1;
    static constexpr int kPer = 4;        // elements of a line set per thread (B N <= 1024)
    static constexpr int kPerHalf = 3;    // of its half spectrum (B (N/2 + 1) <= 576)
    static constexpr bool kMixed = false;
    __device__ __forceinline__ int n() const { return N; }
    __host__ __device__ __forceinline__ int ls() const { return LS; }
    __host__ __device__ __forceinline__ int twiddles() const { return N / 2; }
    __device__ __forceinline__ int at(int b, int i) const { return b * LS + i + (i >> 3); }
    __device__ __forceinline__ int line(int t) const { return t >> LOG2N; }
    __device__ __forceinline__ int elem(int t, int) const { return t & (N - 1); }
    __device__ __forceinline__ int slot(int e) const {
        return static_cast<int>(__brev(static_cast<unsigned>(e)) >> (32 - LOG2N));
    }

    // The radix-2 stages over `lines` lines, R stages per pass: a thread loads
    // the 2^R elements i0 + k*2^S that stages S .. S+R-1 combine, runs those
    // butterflies in registers (the same twiddles, products and sums as one
    // stage at a time, so the result is the same to the bit) and writes them
    // back -- ceil(LOG2N / R) LDS round trips and barriers instead of LOG2N.
    // The forward x kernels take two stages per pass: a block's B * N / 4 =
    // 256 groups keep all 256 threads busy (8-element groups leave half of
    // them idle) and at 40 VGPRs (67 with three stages, N = 128) a CU holds
    // 8 blocks, the whole 128^3 grid in one round.  The y, last-axis and
    // inverse x kernels keep three (fewer passes measured faster there).
    template <int S, int R>
    __device__ __forceinline__ void pass(double2* __restrict__ lds, int lines,
                                         const double2* __restrict__ s_tw, bool inverse) const {
        constexpr int K = 1 << R, H = 1 << S;
        constexpr int PER_LINE = N / K;
        const int total = lines * PER_LINE;
        for (int t = threadIdx.x; t < total; t += blockDim.x) {
            const int b = t / PER_LINE, q = t & (PER_LINE - 1);
            const int pos = q & (H - 1), grp = q >> S;
            const int i0 = grp * (K * H) + pos;
            double2 v[K];
#pragma unroll
            for (int k = 0; k < K; ++k) v[k] = lds[at(b, i0 + k * H)];
#pragma unroll
            for (int j = 0; j < R; ++j) {
                const int hj = 1 << j;
#pragma unroll
                for (int k = 0; k < K; ++k) {
                    if (k & hj) continue;
                    // position of element k in its stage-(S+j) group of 2 * 2^(S+j)
                    const int posj = pos + (k & (hj - 1)) * H;
                    double2 w = s_tw[posj << (LOG2N - 1 - (S + j))];
                    if (inverse) w.y = -w.y;
                    const double2 u = v[k];
                    const double2 x = cmul(v[k + hj], w);
                    v[k] = make_double2(u.x + x.x, u.y + x.y);
                    v[k + hj] = make_double2(u.x - x.x, u.y - x.y);
                }
            }
#pragma unroll
            for (int k = 0; k < K; ++k) lds[at(b, i0 + k * H)] = v[k];
        }
    }
    template <int S, int MAXR>
    __device__ __forceinline__ void passes(double2* __restrict__ lds, int lines,
                                           const double2* __restrict__ s_tw, bool inverse) const {
        if constexpr (S < LOG2N) {
            constexpr int R = LOG2N - S >= MAXR ? MAXR : LOG2N - S;
            pass<S, R>(lds, lines, s_tw, inverse);
            __syncthreads();
            passes<S + R, MAXR>(lds, lines, s_tw, inverse);
        }
    }
    // MAXR stages per pass (2 or 3); the block's data in LDS on entry and exit
    template <int MAXR>
    __device__ __forceinline__ void transform(double2* __restrict__ lds, int lines,
                                              const double2* __restrict__ s_tw,
                                              bool inverse) const {
        passes<0, MAXR>(lds, lines, s_tw, inverse);
    }
};

// cos and sin of 2 pi m / R for the odd butterflies
template <int R>
struct RootsOf;
template <>
struct RootsOf<3> {
    static constexpr double c[3] = {1.0, -0.5, -0.5};
    static constexpr double s[3] = {0.0, 0.86602540378443864676, -0.86602540378443864676};
};
template <>
struct RootsOf<5> {
    static constexpr double c[5] = {1.0, 0.30901699437494742410, -0.80901699437494742410,
                                    -0.80901699437494742410, 0.30901699437494742410};
    static constexpr double s[5] = {0.0, 0.95105651629515357212, 0.58778525229247312917,
                                    -0.58778525229247312917, -0.95105651629515357212};
};
template <>
struct RootsOf<7> {
    static constexpr double c[7] = {1.0,
                                    0.62348980185873353053,
                                    -0.22252093395631440429,
                                    -0.90096886790241912624,
                                    -0.90096886790241912624,
                                    -0.22252093395631440429,
                                    0.62348980185873353053};
    static constexpr double s[7] = {0.0,
                                    0.78183148246802980871,
                                    0.97492791218182360702,
                                    0.43388373911755812048,
                                    -0.43388373911755812048,
                                    -0.97492791218182360702,
                                    -0.78183148246802980871};
};

// R-point DFT in registers (forward; inverse with sign = -1)
template <int R>
__device__ __forceinline__ void dft_small(double2 (&v)[R], double sign) {
    if constexpr (R == 2) {
        const double2 a = v[0], b = v[1];
        v[0] = make_double2(a.x + b.x, a.y + b.y);
        v[1] = make_double2(a.x - b.x, a.y - b.y);
    } else if constexpr (R == 4) {
        const double2 a = make_double2(v[0].x + v[2].x, v[0].y + v[2].y);
        const double2 b = make_double2(v[0].x - v[2].x, v[0].y - v[2].y);
        const double2 c = make_double2(v[1].x + v[3].x, v[1].y + v[3].y);
        const double2 d = make_double2(sign * (v[1].x - v[3].x), sign * (v[1].y - v[3].y));
        v[0] = make_double2(a.x + c.x, a.y + c.y);
        v[1] = make_double2(b.x + d.y, b.y - d.x);
        v[2] = make_double2(a.x - c.x, a.y - c.y);
        v[3] = make_double2(b.x - d.y, b.y + d.x);
    } else {
        // odd R: sums and differences of the pairs j, R - j
        constexpr int H = R / 2;
        double2 p[H], q[H];
#pragma unroll
        for (int j = 0; j < H; ++j) {
            const double2 a = v[j + 1], b = v[R - 1 - j];
            p[j] = make_double2(a.x + b.x, a.y + b.y);
            q[j] = make_double2(sign * (a.x - b.x), sign * (a.y - b.y));
        }
        const double2 v0 = v[0];
#pragma unroll
        for (int j = 0; j < H; ++j) v[0] = make_double2(v[0].x + p[j].x, v[0].y + p[j].y);
#pragma unroll
        for (int k = 1; k <= H; ++k) {
            double2 e = v0, o = make_double2(0.0, 0.0);
#pragma unroll
            for (int j = 0; j < H; ++j) {
                const double c = RootsOf<R>::c[(j + 1) * k % R];
                const double s = RootsOf<R>::s[(j + 1) * k % R];
                e = make_double2(e.x + p[j].x * c, e.y + p[j].y * c);
                o = make_double2(o.x + q[j].x * s, o.y + q[j].y * s);
            }
            // X_k = e - i o, X_{R-k} = e + i o
            v[k] = make_double2(e.x + o.y, e.y - o.x);
            v[R - k] = make_double2(e.x - o.y, e.y + o.x);
        }
    }
}

// One stage of a mixed-radix plan: groups of r blocks of h elements (h the
// product of the radices before it) become one block of r h.
struct FftStage {
    int r, h;
    int tw_step;           // n / (r h): twiddle table stride of the stage
    FastDiv per_line;      // n / r groups per line
    FastDiv h_div;
};

// A line of any length n <= 2048: radices 4, 2, 3, 5 and 7 in registers, a
// larger prime factor by direct sums over its r inputs.  The plan (stages,
// digit-reversal table) is built once per mesh; its loads are uniform.
struct MixedAxis {
    int N, LS;
    int stages;
    FastDiv n_div;
    const FftStage* stage;
    const uint16_t* rev;      // slot of element e
    static constexpr int kPer = 8;        // B N <= max(1280, 2048)
    static constexpr int kPerHalf = 5;    // B (N/2 + 1) <= 1280
    static constexpr int kDirect = 9;     // two fields' lines with a factor above 7: 2 B N <= 2274
    static constexpr bool kMixed = true;
    __device__ __forceinline__ int n() const { return N; }
    __host__ __device__ __forceinline__ int ls() const { return LS; }
    __host__ __device__ __forceinline__ int twiddles() const { return N; }
    __device__ __forceinline__ int at(int b, int i) const { return b * LS + i + (i >> 3); }
    __device__ __forceinline__ int line(int t) const { return n_div(t); }
    __device__ __forceinline__ int elem(int t, int b) const { return t - b * N; }
    __device__ __forceinline__ int slot(int e) const { return rev[e]; }

    template <int R>
    __device__ __forceinline__ void pass(const FftStage& st, double2* __restrict__ lds, int lines,
                                         const double2* __restrict__ s_tw, bool inverse) const {
        const int per = N / R, total = lines * per, h = st.h;
        const double sign = inverse ? -1.0 : 1.0;
        for (int t = threadIdx.x; t < total; t += blockDim.x) {
            const int b = st.per_line(t), q = t - b * per;
            const int grp = st.h_div(q), pos = q - grp * h;
            const int i0 = grp * (R * h) + pos;
            double2 v[R];
#pragma unroll
            for (int k = 0; k < R; ++k) {
                v[k] = lds[at(b, i0 + k * h)];
                if (k > 0) {
                    double2 w = s_tw[k * pos * st.tw_step];   // k pos < r h: below n
                    if (inverse) w.y = -w.y;
                    v[k] = cmul(v[k], w);
                }
            }
            dft_small<R>(v, sign);
#pragma unroll
            for (int k = 0; k < R; ++k) lds[at(b, i0 + k * h)] = v[k];
        }
    }
    // a prime factor above 7: every thread sums its outputs from the group's r
    // inputs (the twiddle index advances by pos tw_step + k n / r), then all
    // of them replace the inputs
    __device__ __forceinline__ void pass_direct(const FftStage& st, double2* __restrict__ lds,
                                                int lines, const double2* __restrict__ s_tw,
                                                bool inverse) const {
        const int r = st.r, h = st.h, per = N / r, total = lines * N;
        double2 acc[kDirect];
        int where[kDirect];
#pragma unroll
        for (int u = 0; u < kDirect; ++u) {
            const int t = threadIdx.x + u * kFftThreads;
            where[u] = -1;
            acc[u] = make_double2(0.0, 0.0);
            if (t >= total) continue;
            const int b = n_div(t), o = t - b * N;     // o = grp r h + k h + pos
            const int hb = st.h_div(o), pos = o - hb * h;
            const int grp = hb / r, k = hb - grp * r;
            const int i0 = grp * (r * h) + pos;
            const int step = (pos * st.tw_step + k * per) % N;
            int m = 0;
            double sr = 0.0, si = 0.0;
            for (int j = 0; j < r; ++j) {
                double2 w = s_tw[m];
                if (inverse) w.y = -w.y;
                const double2 x = lds[at(b, i0 + j * h)];
                sr += x.x * w.x - x.y * w.y;
                si += x.x * w.y + x.y * w.x;
                m += step;
                if (m >= N) m -= N;
            }
            acc[u] = make_double2(sr, si);
            where[u] = at(b, o);
        }
        __syncthreads();
#pragma unroll
        for (int u = 0; u < kDirect; ++u)
            if (where[u] >= 0) lds[where[u]] = acc[u];
    }
    template <int>
    __device__ __forceinline__ void transform(double2* __restrict__ lds, int lines,
                                              const double2* __restrict__ s_tw,
                                              bool inverse) const {
        for (int s = 0; s < stages; ++s) {
            const FftStage st = stage[s];
            switch (st.r) {
                case 2: pass<2>(st, lds, lines, s_tw, inverse); break;
                case 3: pass<3>(st, lds, lines, s_tw, inverse); break;
                case 4: pass<4>(st, lds, lines, s_tw, inverse); break;
                case 5: pass<5>(st, lds, lines, s_tw, inverse); break;
                case 7: pass<7>(st, lds, lines, s_tw, inverse); break;
                default: pass_direct(st, lds, lines, s_tw, inverse); break;
            }
            __syncthreads();
        }
    }
};

// the block's twiddles, table entries e^{-2 pi i k / n}
template <typename Axis>
__device__ __forceinline__ void stage_twiddles(const Axis& ax, const double2* tw, double2* s_tw) {
    for (int k = threadIdx.x; k < ax.twiddles(); k += blockDim.x) s_tw[k] = tw[k];
}

}  // namespace aurora
