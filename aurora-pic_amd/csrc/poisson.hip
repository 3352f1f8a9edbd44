// poisson.hip - FP64 field solves (FieldSolver.cpp:384-759):
//   1D periodic   spectral solve with continuous k (407-440): FFTs on a power
//                 of two, direct sums on other meshes
//   1D Dirichlet  the tridiagonal solve (733-759) as two prefix sums
//   2D/3D periodic FFT Poisson with spectral E (442-499, 659-731)
// The 2D/3D solve transforms rho forward and the spectral fields back.
// Each spectral field is first projected onto its Hermitian part (zeroing
// the own-axis Nyquist plane of E_a), which leaves its real inverse - the
// quantity the reference keeps - unchanged.  Only the non-negative x
// frequencies of every spectrum are kept (the others are their conjugates);
// the last inverse rebuilds each x line's full spectrum of two real fields,
// (Ex + i Ey) and (Ez + i phi).
#include <algorithm>
#include <cmath>
#include <vector>

#include "fft_device.hpp"
#include "field_device.hpp"

namespace aurora {

namespace {

struct GreenArgs {
    int nx, ny, nz, dim;
    double twopi_over_L[3];
    double eps;
    int want_phi;
};

__device__ __forceinline__ double mode_of(int idx, int n) {
    // Nyquist index counts as +n/2 (FieldSolver.cpp:421, 471, 694)
    return idx <= n / 2 ? static_cast<double>(idx) : -static_cast<double>(n - idx);
}

// The spectral step for one mode (ix, iy, iz) of rho_hat r: phi_hat =
// rho_hat / (eps k^2) with continuous k, E_a = -i k_a phi (FieldSolver.cpp:
// 486-488, 717-720) with the own-axis Nyquist plane removed (Hermitian
// part): E_x, E_y, E_z and phi of the mode (E_z zero outside 3D).  Returned
// by value: no local's address is taken, so every value stays in registers.
struct ModeFields {
    double2 ex, ey, ez, ph;
};

__device__ __forceinline__ ModeFields green_split(const GreenArgs& g, int ix, int iy, int iz,
                                                  double2 r) {
#pragma clang fp contract(off)
    ModeFields f;
    f.ex = f.ey = f.ez = f.ph = make_double2(0.0, 0.0);
    if (ix == 0 && iy == 0 && iz == 0) return f;
    const double kx = g.twopi_over_L[0] * mode_of(ix, g.nx);
    const double ky = g.dim > 1 ? g.twopi_over_L[1] * mode_of(iy, g.ny) : 0.0;
    const double kz = g.dim > 2 ? g.twopi_over_L[2] * mode_of(iz, g.nz) : 0.0;
    double k2 = kx * kx + ky * ky;
    if (g.dim > 2) k2 += kz * kz;
    const double den = g.eps * k2;
    const double pr = r.x / den, pi = r.y / den;
    const bool nyx = (g.nx % 2 == 0) && ix == g.nx / 2;
    const bool nyy = (g.ny % 2 == 0) && iy == g.ny / 2;
    const bool nyz = (g.nz % 2 == 0) && iz == g.nz / 2;
    if (!nyx) f.ex = make_double2(kx * pi, -kx * pr);
    if (!nyy) f.ey = make_double2(ky * pi, -ky * pr);
    if (g.dim > 2 && !nyz) f.ez = make_double2(kz * pi, -kz * pr);
    f.ph = make_double2(pr, pi);
    return f;
}

// 1D periodic: direct spectral sum (FieldSolver.cpp:407-440) in one block.
__global__ void __launch_bounds__(1024) k_spectral_1d(const double* rho, double* phi, double* E,
                                                      float* E32, const double* cs,
                                                      const double* sn, int n, double L,
                                                      double eps) {
    extern __shared__ __align__(16) double sh[];
    __shared__ double mean_s;
    spectral_solve_1d(rho, phi, E, E32, cs, sn, n, L, eps, sh, &mean_s);
}

// 1D Dirichlet Thomas solve (FieldSolver.cpp:733-759)
__global__ void __launch_bounds__(256) k_thomas_1d(const double* rho, double* phi, double* E,
                                                   float* E32, double* s, int n, double dx,
                                                   double eps, double phi_left, double phi_right) {
    dirichlet_solve_1d(rho, [&](int i) { return rho[i]; }, phi, E, E32, s, n, dx, eps, phi_left,
                       phi_right);
}

// ------------------------------------------------------------------------
// The 2D/3D solve in few passes over HBM, on half spectra: rho is real, so
// only x frequencies 0 .. nx/2 are kept (NH = nx/2 + 1 of them), laid out
// [kx][z][y] (node (kx * nz + z) * ny + y; P = ny * nz nodes per kx plane):
//   fwd_x        reads rho (or the species accumulators), forward
//                transform along x, frequencies 0 .. nx/2 written     -> H0
//   rows         forward or inverse transform along y (3D): the lines
//                are contiguous in this layout                   H0 (H1..H3)
//   last         forward transform of the last axis (z in 3D, y in
//                2D), the Green step with the fields kept apart, their
//                inverse transforms of that axis
//                                              -> H0 Ex, H1 Ey, H2 Ez, H3 phi
//   inv_x_c2r    per x line, the full spectrum of (Ex + i Ey) and
//                (Ez + i phi) rebuilt from the halves (frequency n - k
//                is the conjugate of k), inverse transform along x, the
//                outputs (E64, E32, phi) written directly
// Every mesh takes these kernels; each axis has the transform its length
// asks for (Pow2Axis or MixedAxis, fft_device.hpp).  Meshes with a length
// that is no power of two took direct sums, O(n^2) per line with a 64-bit
// remainder per term, in separate passes over full spectra: 210 x 125 nodes
// 560 us per solve, 90 x 75 x 60 670 us, 48^3 480 us, against 25, 69 and
// 46 us.
//
// The kernels run 256 threads; a block stages 2^LB lines, and issues all of
// a thread's global loads into registers before the first LDS store, so the
// loads' latencies overlap instead of adding up; lines are bit- or
// digit-reversed on the way into LDS.  LDS: the twiddles, then the field
// buffer(s).
extern __shared__ __align__(16) double2 fft_lds[];

// LDS bytes of a kernel with `fields` buffers of 2^LB lines
template <typename Axis>
size_t fft_lds_bytes(const Axis& ax, int LB, int fields) {
    return (static_cast<size_t>(fields) * (size_t{1} << LB) * ax.ls() + ax.twiddles()) *
           sizeof(double2);
}

// frequencies 0 .. N/2 of the B lines in LDS to the half layout: element
// kx of x line l at kx * P + l (consecutive threads, consecutive lines)
template <typename Axis>
__device__ __forceinline__ void store_half_x(const Axis& ax, const double2* lds,
                                             double2* __restrict__ out, int64_t line0, int lines,
                                             int LB, int64_t P) {
    const int NH = ax.n() / 2 + 1;
    const int B = 1 << LB;
    for (int t = threadIdx.x; t < B * NH; t += blockDim.x) {
        const int b = t & (B - 1), kx = t >> LB;
        if (b < lines) out[kx * P + line0 + b] = lds[ax.at(b, kx)];
    }
}

template <typename Axis>
__global__ void __launch_bounds__(kFftThreads) k_fwd_x_real(Axis ax, const double* __restrict__ rho,
                                                    double2* __restrict__ out, int64_t nlines,
                                                    int LB, const double2* __restrict__ tw) {
    const int B = 1 << LB, N = ax.n();
    double2* s_tw = fft_lds;
    double2* lds = fft_lds + ax.twiddles();
    stage_twiddles(ax, tw, s_tw);
    const int64_t line0 = static_cast<int64_t>(blockIdx.x) * B;
    const int lines = static_cast<int>(nlines - line0 < B ? nlines - line0 : B);
    double r[Axis::kPer];
#pragma unroll
    for (int u = 0; u < Axis::kPer; ++u) {
        const int t = threadIdx.x + u * kFftThreads;
        if (t < lines * N) r[u] = rho[line0 * N + t];
    }
#pragma unroll
    for (int u = 0; u < Axis::kPer; ++u) {
        const int t = threadIdx.x + u * kFftThreads;
        if (t >= lines * N) continue;
        const int b = ax.line(t);
        lds[ax.at(b, ax.slot(ax.elem(t, b)))] = make_double2(r[u], 0.0);
    }
    __syncthreads();
    ax.template transform<2>(lds, lines, s_tw, false);
    store_half_x(ax, lds, out, line0, lines, LB, nlines);
}

// The step's variant of k_fwd_x_real: the charge density of each node from
// the species accumulators (rho_at, the conversion kernel's operations), the
// accumulators of the next push zeroed on the way.
struct ClearArgs {
    long long* p[kMaxChannels];
    int n;
};

// One 1D step's field solve from the deposit: the charge density from the
// species' fixed-point sums, the next step's accumulators zeroed, then the
// Dirichlet or the periodic solve by workgroup 0 -- one launch where the
// charge conversion, the clears and the solve took one each.  The further
// workgroups fold the species' ledger partials beside it (2.4 us by
// themselves on 64 partials, 7.5 on 2 x 2,210).
__device__ __forceinline__ double rho_node_1d(const RhoArgs& ra, const ClearArgs& cl, double* rho,
                                              int i) {
    const double r = rho_at(ra, i);
    rho[i] = r;
    for (int k = 0; k < cl.n; ++k) cl.p[k][i] = 0;
    return r;
}

__global__ void __launch_bounds__(256) k_thomas_1d_acc(RhoArgs ra, ClearArgs cl, LedgerFolds lf,
                                                       double* rho, double* phi, double* E,
                                                       float* E32, double* s, int n, double dx,
                                                       double eps, double phi_left,
                                                       double phi_right) {
    if (blockIdx.x > 0) {
        fold_ledger(lf.f[blockIdx.x - 1]);
        return;
    }
    dirichlet_solve_1d(rho, [&](int i) { return rho_node_1d(ra, cl, rho, i); }, phi, E, E32, s, n,
                       dx, eps, phi_left, phi_right);
}

__global__ void __launch_bounds__(1024) k_spectral_1d_acc(RhoArgs ra, ClearArgs cl,
                                                          LedgerFolds lf, double* rho,
                                                          double* phi, double* E, float* E32,
                                                          const double* cs, const double* sn,
                                                          int n, double L, double eps) {
    extern __shared__ __align__(16) double sh[];
    __shared__ double mean_s;
    if (blockIdx.x > 0) {
        fold_ledger(lf.f[blockIdx.x - 1]);
        return;
    }
    for (int i = threadIdx.x; i < n; i += blockDim.x) rho_node_1d(ra, cl, rho, i);
    __syncthreads();
    spectral_solve_1d(rho, phi, E, E32, cs, sn, n, L, eps, sh, &mean_s);
}

template <typename Axis>
__global__ void __launch_bounds__(kFftThreads) k_fwd_x_acc(Axis ax, RhoArgs ra, ClearArgs cl,
                                                   double2* __restrict__ out, int64_t nlines,
                                                   int LB, const double2* __restrict__ tw) {
    const int B = 1 << LB, N = ax.n();
    double2* s_tw = fft_lds;
    double2* lds = fft_lds + ax.twiddles();
    stage_twiddles(ax, tw, s_tw);
    const int64_t line0 = static_cast<int64_t>(blockIdx.x) * B;
    const int lines = static_cast<int>(nlines - line0 < B ? nlines - line0 : B);
    double r[Axis::kPer];
#pragma unroll
    for (int u = 0; u < Axis::kPer; ++u) {
        const int t = threadIdx.x + u * kFftThreads;
        if (t < lines * N) r[u] = rho_at(ra, line0 * N + t);
    }
#pragma unroll
    for (int u = 0; u < Axis::kPer; ++u) {
        const int t = threadIdx.x + u * kFftThreads;
        if (t >= lines * N) continue;
        for (int s = 0; s < cl.n; ++s) cl.p[s][line0 * N + t] = 0;
        const int b = ax.line(t);
        lds[ax.at(b, ax.slot(ax.elem(t, b)))] = make_double2(r[u], 0.0);
    }
    __syncthreads();
    ax.template transform<2>(lds, lines, s_tw, false);
    store_half_x(ax, lds, out, line0, lines, LB, nlines);
}

// the half spectra H0 .. H3
struct Halves {
    double2* h[4];
};

// forward or inverse transform of contiguous lines of N (the y lines of the
// half layout), 1 << LB lines per block; blockIdx.y selects the array
template <typename Axis>
__global__ void __launch_bounds__(kFftThreads) k_rows(Axis ax, Halves arr, int64_t nlines, int LB,
                                              const double2* __restrict__ tw, int inverse) {
    // a select, not arr.h[blockIdx.y]: a dynamic index into the argument
    // array would copy it to private (scratch) memory
    const unsigned w = blockIdx.y;
    double2* data = w == 0 ? arr.h[0] : w == 1 ? arr.h[1] : w == 2 ? arr.h[2] : arr.h[3];
    const int B = 1 << LB, N = ax.n();
    double2* s_tw = fft_lds;
    double2* lds = fft_lds + ax.twiddles();
    stage_twiddles(ax, tw, s_tw);
    const int64_t line0 = static_cast<int64_t>(blockIdx.x) * B;
    const int lines = static_cast<int>(nlines - line0 < B ? nlines - line0 : B);
    double2 r[Axis::kPer];
#pragma unroll
    for (int u = 0; u < Axis::kPer; ++u) {
        const int t = threadIdx.x + u * kFftThreads;
        r[u] = t < lines * N ? data[line0 * N + t] : make_double2(0.0, 0.0);
    }
#pragma unroll
    for (int u = 0; u < Axis::kPer; ++u) {
        const int t = threadIdx.x + u * kFftThreads;
        if (t >= lines * N) continue;
        const int b = ax.line(t);
        lds[ax.at(b, ax.slot(ax.elem(t, b)))] = r[u];
    }
    __syncthreads();
    ax.template transform<3>(lds, lines, s_tw, inverse != 0);
    const double scale = inverse ? 1.0 / static_cast<double>(N) : 1.0;
    for (int t = threadIdx.x; t < lines * N; t += blockDim.x) {
        const int b = ax.line(t);
        double2 v = lds[ax.at(b, ax.elem(t, b))];
        v.x *= scale;
        v.y *= scale;
        data[line0 * N + t] = v;
    }
}

// The lines of the last axis: line l is (kx, y) at stride ny in 3D, kx
// alone in 2D (inner 1).
struct LastLines {
    FastDiv inner;       // ny in 3D, 1 in 2D
    int64_t nlines;
    int64_t plane;       // P: nodes per kx
    int dim;
    __device__ __forceinline__ int64_t node(int line, int e) const {
        const int kx = inner(line), y = line - kx * static_cast<int>(inner.d);
        return kx * plane + y + static_cast<int64_t>(e) * inner.d;
    }
};

// forward transform of the last axis of H0, Green step (green_split),
// inverse transforms along the same axis (scaled 1/N) of Ex, Ey, Ez (3D)
// and phi (when wanted) to H0 .. H3.  The fields go two at a time through
// one LDS buffer of 2B lines (field a in lines 0 .. B-1, field b in B ..
// 2B-1), so one set of passes transforms both and keeps every thread
// busy.  A thread keeps only its (at most kPer) elements of rho_hat in
// registers and evaluates the Green step again for each pair (the same
// operations, so the same values).  The fields are written over the
// transformed input once every thread holds its share of rho_hat.
template <typename Axis>
__global__ void __launch_bounds__(kFftThreads) k_last(Axis ax, Halves arr, LastLines p, int LB,
                                              const double2* __restrict__ tw, GreenArgs g,
                                              int want_ez) {
    constexpr int kPer = Axis::kPer;
    const int B = 1 << LB, N = ax.n();
    double2* s_tw = fft_lds;
    double2* X = fft_lds + ax.twiddles();
    stage_twiddles(ax, tw, s_tw);
    const int line0 = static_cast<int>(blockIdx.x) << LB;
    const int nlines = static_cast<int>(p.nlines);
    double2 r[kPer];
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
        const int t = threadIdx.x + u * kFftThreads;
        const int bb = t & (B - 1), e = t >> LB;
        // an unconditional load and selects of the components: a select
        // between a loaded element and a local would go through scratch
        const bool ok = e < N && line0 + bb < nlines;
        const double2 v = arr.h[0][ok ? p.node(line0 + bb, e) : 0];
        r[u] = make_double2(ok ? v.x : 0.0, ok ? v.y : 0.0);
    }
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
        const int t = threadIdx.x + u * kFftThreads;
        const int bb = t & (B - 1), e = t >> LB;
        if (e < N) X[ax.at(bb, ax.slot(e))] = r[u];
    }
    __syncthreads();
    ax.template transform<3>(X, B, s_tw, false);
    double2 rh[kPer];
#pragma unroll
    for (int q = 0; q < kPer; ++q) {
        const int t = threadIdx.x + q * kFftThreads;
        const int tc = t < B * N ? t : 0;
        const int b = ax.line(tc);
        const double2 v = X[ax.at(b, ax.elem(tc, b))];
        const bool ok = t < B * N && line0 + b < nlines;
        rh[q] = make_double2(ok ? v.x : 0.0, ok ? v.y : 0.0);
    }
    // fields FA (and FB >= 0) of every element (0 Ex, 1 Ey, 2 Ez, 3 phi)
    // into X at the reversed slots, inverse transforms written to fa (and fb)
    auto pair = [&]<int FA, int FB>(double2* fa, double2* fb) {
        __syncthreads();
#pragma unroll
        for (int q = 0; q < kPer; ++q) {
            const int t = threadIdx.x + q * kFftThreads;
            if (t >= B * N) continue;
            const int bb = ax.line(t), e = ax.elem(t, bb);
            // lines past the end (rh zero) give zero fields
            const int kx = p.inner(line0 + bb);
            const int y = line0 + bb - kx * static_cast<int>(p.inner.d);
            const ModeFields mf = p.dim == 3 ? green_split(g, kx, y, e, rh[q])
                                             : green_split(g, kx, e, 0, rh[q]);
            const int at = ax.at(bb, ax.slot(e));
            X[at] = FA == 0 ? mf.ex : FA == 1 ? mf.ey : FA == 2 ? mf.ez : mf.ph;
            if constexpr (FB >= 0)
                X[B * ax.ls() + at] = FB == 0 ? mf.ex : FB == 1 ? mf.ey : FB == 2 ? mf.ez : mf.ph;
        }
        __syncthreads();
        constexpr int NF = FB >= 0 ? 2 : 1;
        ax.template transform<3>(X, NF * B, s_tw, true);
        const double scale = 1.0 / static_cast<double>(N);
        for (int t = threadIdx.x; t < NF * B * N; t += blockDim.x) {
            const int f = t >= B * N ? 1 : 0;
            const int tt = t - f * B * N;
            const int bb = tt & (B - 1), e = tt >> LB;
            if (line0 + bb >= nlines) continue;
            double2 v = X[ax.at(f * B + bb, e)];
            v.x *= scale;
            v.y *= scale;
            (f ? fb : fa)[p.node(line0 + bb, e)] = v;
        }
    };
    pair.template operator()<0, 1>(arr.h[0], arr.h[1]);
    if (want_ez && g.want_phi)
        pair.template operator()<2, 3>(arr.h[2], arr.h[3]);
    else if (want_ez)
        pair.template operator()<2, -1>(arr.h[2], nullptr);
    else if (g.want_phi)
        pair.template operator()<3, -1>(arr.h[3], nullptr);
}

// One x line's full spectrum of (a + i b) from the half spectra a_k, b_k
// (k = 0 .. N/2) of two real fields: C_k = a_k + i b_k and C_{N-k} =
// conj(a_k) + i conj(b_k); at k = 0 and k = N/2 of an even N (their own
// conjugates) the real parts.  Stored at the reversed slots of line b.
template <typename Axis>
__device__ __forceinline__ void put_pair(const Axis& ax, double2* lds, int b, int k, double2 a,
                                         double2 v) {
    const int N = ax.n();
    if (k == 0 || 2 * k == N) {
        lds[ax.at(b, ax.slot(k))] = make_double2(a.x, v.x);
        return;
    }
    lds[ax.at(b, ax.slot(k))] = make_double2(a.x - v.y, a.y + v.x);
    lds[ax.at(b, ax.slot(N - k))] = make_double2(a.x + v.y, v.x - a.y);
}

// inverse transform along x: (Ex + i Ey) from H0, H1 and (Ez + i phi) from
// H2, H3 (an absent half reads as zero), scaled 1/N, written as E64 (when
// given), phi (when wanted) and the packed FP32 field
template <typename Axis>
__global__ void __launch_bounds__(kFftThreads) k_inv_x_c2r(Axis ax, Halves arr, int64_t nlines,
                                                   int LB, const double2* __restrict__ tw,
                                                   double* E64, double* phi, float* E32,
                                                   int dim, int want_phi, int64_t nn) {
    const bool use_b = dim == 3 || want_phi;
    const int B = 1 << LB, N = ax.n(), NH = N / 2 + 1;
    double2* s_tw = fft_lds;
    double2* A = fft_lds + ax.twiddles();
    double2* Bb = A + B * ax.ls();
    stage_twiddles(ax, tw, s_tw);
    const int64_t line0 = static_cast<int64_t>(blockIdx.x) * B;
    const int lines = static_cast<int>(nlines - line0 < B ? nlines - line0 : B);
    // every load issued before the first LDS store
    constexpr int kPer = Axis::kPerHalf;
    const double2 zero = make_double2(0.0, 0.0);
    double2 va[kPer], vb[kPer], vc[kPer], vd[kPer];
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
        const int t = threadIdx.x + u * kFftThreads;
        const int b = t & (B - 1), k = t >> LB;
        const bool ok = k < NH && b < lines;
        const int64_t src = k * nlines + line0 + b;
        va[u] = ok ? arr.h[0][src] : zero;
        vb[u] = ok ? arr.h[1][src] : zero;
        vc[u] = ok && dim == 3 ? arr.h[2][src] : zero;
        vd[u] = ok && want_phi ? arr.h[3][src] : zero;
    }
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
        const int t = threadIdx.x + u * kFftThreads;
        const int b = t & (B - 1), k = t >> LB;
        if (k >= NH || b >= lines) continue;
        put_pair(ax, A, b, k, va[u], vb[u]);
        if (use_b) put_pair(ax, Bb, b, k, vc[u], vd[u]);
    }
    __syncthreads();
    // both fields in one set of passes (lines past the end carry no data)
    ax.template transform<3>(A, use_b ? 2 * B : B, s_tw, true);
    const double scale = 1.0 / static_cast<double>(N);
    for (int t = threadIdx.x; t < lines * N; t += blockDim.x) {
        const int64_t i = line0 * N + t;
        const int lb = ax.line(t);
        const int la = ax.at(lb, ax.elem(t, lb));
        double2 a = A[la];
        a.x *= scale;
        a.y *= scale;
        if (E64) {
            E64[i] = a.x;
            E64[nn + i] = a.y;
        }
        if (dim == 3) {
            double2 b = Bb[la];
            b.x *= scale;
            b.y *= scale;
            if (E64) E64[2 * nn + i] = b.x;
            if (want_phi) phi[i] = b.y;
            reinterpret_cast<float4*>(E32)[i] = make_float4(static_cast<float>(a.x),
                                                            static_cast<float>(a.y),
                                                            static_cast<float>(b.x), 0.0f);
        } else {
            if (want_phi) phi[i] = Bb[la].y * scale;
            reinterpret_cast<float2*>(E32)[i] =
                make_float2(static_cast<float>(a.x), static_cast<float>(a.y));
        }
    }
}

// f.operator()<Axis>(axis) with the transform of a mesh axis
template <typename F>
void with_axis(const Context& c, int axis, F&& f) {
    const int64_t n = c.n[axis];
    if ((n & (n - 1)) != 0 || n < 4 || n > 1024) {
        MixedAxis ax{};
        ax.N = static_cast<int>(n);
        ax.LS = ax.N + ax.N / 8 + 1;
        ax.stages = c.fft_stages[axis];
        ax.n_div = fast_div(n);
        ax.stage = reinterpret_cast<const FftStage*>(c.fft_stage[axis].ptr);
        ax.rev = c.fft_rev[axis].ptr;
        f(ax);
        return;
    }
    switch (n) {
        case 4: f(Pow2Axis<2>{}); break;
        case 8: f(Pow2Axis<3>{}); break;
        case 16: f(Pow2Axis<4>{}); break;
        case 32: f(Pow2Axis<5>{}); break;
        case 64: f(Pow2Axis<6>{}); break;
        case 128: f(Pow2Axis<7>{}); break;
        case 256: f(Pow2Axis<8>{}); break;
        case 512: f(Pow2Axis<9>{}); break;
        default: f(Pow2Axis<10>{}); break;
    }
}

// lines per block (log2): what the LDS buffer holds, halved while the launch
// would have fewer blocks than the device has CUs (a small mesh is bound by
// the length of one block's chain)
int lines_per_block(const Context& c, int64_t n, int64_t nlines) {
    int lb = lines_shift(kLineLds, n);
    while (lb > 0 && (nlines >> lb) < c.cu_count) --lb;
    return lb;
}

unsigned line_blocks(int64_t nlines, int lb) {
    return static_cast<unsigned>((nlines + (int64_t{1} << lb) - 1) >> lb);
}

// the half layout's x frequencies (nx/2 + 1) times P = ny * nz nodes
int64_t half_nodes(const Context& c) {
    const int64_t nz = c.dim > 2 ? c.n[2] : 1;
    return (c.n[0] / 2 + 1) * c.n[1] * nz;
}

// from_acc: the first transform reads the species accumulators (the step's
// solve; rho is not written) instead of rho
void solve_periodic(Context& c, const GreenArgs& ga, bool want_phi, bool want_e64,
                    bool from_acc = false) {
    const int64_t nx = c.n[0], ny = c.n[1], nz = c.dim > 2 ? c.n[2] : 1;
    const int64_t P = ny * nz, NH = nx / 2 + 1, half = half_nodes(c);
    Halves H{{c.fa.ptr, c.fa.ptr + half, c.fb.ptr, c.fb.ptr + half}};
    const int LBx = lines_per_block(c, nx, P);
    const unsigned grid_x = line_blocks(P, LBx);
    {
        KernelScope ks(c, "fft_fwd_x");
        if (from_acc) {
            const RhoArgs ra = rho_args(c);
            ClearArgs cl{};
            cl.n = static_cast<int>(c.species.size());
            for (int s = 0; s < cl.n; ++s) {
                Species& sp = c.species[s];
                if (!sp.acc_next.ptr) sp.acc_next.alloc(c.nnodes);
                cl.p[s] = reinterpret_cast<long long*>(sp.acc_next.ptr);
            }
            with_axis(c, 0, [&](auto ax) {
                k_fwd_x_acc<<<grid_x, kFftThreads, fft_lds_bytes(ax, LBx, 1), c.stream>>>(
                    ax, ra, cl, H.h[0], P, LBx, c.tw[0].ptr);
            });
            for (auto& sp : c.species) sp.acc_next_clear = true;
        } else {
            with_axis(c, 0, [&](auto ax) {
                k_fwd_x_real<<<grid_x, kFftThreads, fft_lds_bytes(ax, LBx, 1), c.stream>>>(
                    ax, c.rho.ptr, H.h[0], P, LBx, c.tw[0].ptr);
            });
        }
        AUR_HIP(hipGetLastError());
    }
    // y lines of the half layout (3D): NH * nz contiguous lines of ny
    const int64_t rows = NH * nz;
    auto y_lines = [&](int inverse, unsigned arrays) {
        const int LB = lines_per_block(c, ny, rows * arrays);
        KernelScope ks(c, "fft_axis");
        with_axis(c, 1, [&](auto ax) {
            k_rows<<<dim3(line_blocks(rows, LB), arrays), kFftThreads, fft_lds_bytes(ax, LB, 1),
                     c.stream>>>(ax, H, rows, LB, c.tw[1].ptr, inverse);
        });
        AUR_HIP(hipGetLastError());
    };
    if (c.dim == 3) y_lines(0, 1u);
    {
        // last axis: z lines (kx, y) at stride ny in 3D, y lines (kx) in 2D
        const int last = c.dim - 1;
        LastLines p{};
        p.dim = c.dim;
        p.inner = fast_div(c.dim == 3 ? ny : 1);
        p.nlines = c.dim == 3 ? NH * ny : NH;
        p.plane = P;
        const int LB = lines_per_block(c, c.n[last], p.nlines);
        KernelScope ks(c, "fft_last");
        with_axis(c, last, [&](auto ax) {
            k_last<<<line_blocks(p.nlines, LB), kFftThreads, fft_lds_bytes(ax, LB, 2), c.stream>>>(
                ax, H, p, LB, c.tw[last].ptr, ga, c.dim == 3 ? 1 : 0);
        });
        AUR_HIP(hipGetLastError());
    }
    // inverse y of Ex, Ey, Ez (and phi)
    if (c.dim == 3) y_lines(1, want_phi ? 4u : 3u);
    {
        KernelScope ks(c, "fft_inv_x");
        const int fields = c.dim == 3 || want_phi ? 2 : 1;
        with_axis(c, 0, [&](auto ax) {
            k_inv_x_c2r<<<grid_x, kFftThreads, fft_lds_bytes(ax, LBx, fields), c.stream>>>(
                ax, H, P, LBx, c.tw[0].ptr, want_e64 ? c.E64.ptr : nullptr, c.phi.ptr, c.E32.ptr,
                c.dim, want_phi ? 1 : 0, c.nnodes);
        });
        AUR_HIP(hipGetLastError());
    }
}

// The mixed-radix plan of an axis: factors 4, then 2, 3, 5, 7 and larger
// primes; element e's slot is its digits, most significant stage first.
void plan_mixed(Context& c, int axis) {
    const int n = static_cast<int>(c.n[axis]);
    std::vector<int> radix;
    int m = n;
    while (m % 4 == 0) { radix.push_back(4); m /= 4; }
    for (int f = 2; m > 1; ++f)
        while (m % f == 0) { radix.push_back(f); m /= f; }
    std::vector<FftStage> st;
    int h = 1;
    for (int r : radix) {
        FftStage s{};
        s.r = r;
        s.h = h;
        s.tw_step = n / (r * h);
        s.per_line = fast_div(n / r);
        s.h_div = fast_div(h);
        st.push_back(s);
        h *= r;
    }
    std::vector<uint16_t> rev(static_cast<size_t>(n));
    for (int e = 0; e < n; ++e) {
        int rest = e, block = n, slot = 0;
        for (size_t k = radix.size(); k-- > 0;) {
            block /= radix[k];
            slot += (rest % radix[k]) * block;
            rest /= radix[k];
        }
        rev[static_cast<size_t>(e)] = static_cast<uint16_t>(slot);
    }
    c.fft_stages[axis] = static_cast<int>(st.size());
    c.fft_stage[axis].alloc(st.size() * sizeof(FftStage));
    c.fft_rev[axis].alloc(rev.size());
    AUR_HIP(hipMemcpy(c.fft_stage[axis].ptr, st.data(), st.size() * sizeof(FftStage),
                      hipMemcpyHostToDevice));
    AUR_HIP(hipMemcpy(c.fft_rev[axis].ptr, rev.data(), rev.size() * sizeof(uint16_t),
                      hipMemcpyHostToDevice));
}

}  // namespace

void prepare_solver(Context& c) {
    const double twopi = 6.283185307179586476925286766559;
    if (c.dim == 1 && c.bc == AURORA_PERIODIC) {
        const int n = static_cast<int>(c.n[0]);
        AUR_REQUIRE(n <= 2048, AURORA_ERR_UNSUPPORTED,
                    "1D periodic spectral solve supports at most 2048 nodes");
        std::vector<double> cs(n), sn(n);
        for (int m = 0; m < n; ++m) {
            const double a = twopi * static_cast<double>(m) / static_cast<double>(n);
            cs[m] = std::cos(a);
            sn[m] = std::sin(a);
        }
        c.dft_cos.alloc(n);
        c.dft_sin.alloc(n);
        AUR_HIP(hipMemcpy(c.dft_cos.ptr, cs.data(), n * sizeof(double), hipMemcpyHostToDevice));
        AUR_HIP(hipMemcpy(c.dft_sin.ptr, sn.data(), n * sizeof(double), hipMemcpyHostToDevice));
    } else if (c.dim == 1) {
        // first-difference scratch of the prefix-sum solve
        c.thomas_inv.alloc(static_cast<size_t>(c.n[0]));
    } else if (c.bc == AURORA_PERIODIC) {
        for (int a = 0; a < c.dim; ++a) {
            const int n = static_cast<int>(c.n[a]);
            AUR_REQUIRE(n <= 2048, AURORA_ERR_UNSUPPORTED,
                        "periodic FFT axes longer than 2048 nodes are not supported");
            const bool pow2 = (n & (n - 1)) == 0;
            AUR_REQUIRE(pow2 || n <= 1024, AURORA_ERR_UNSUPPORTED,
                        "non power-of-two FFT axes longer than 1024 are not supported");
            std::vector<double2> tw(n);
            for (int k = 0; k < n; ++k) {
                const double ang = twopi * static_cast<double>(k) / static_cast<double>(n);
                tw[k] = make_double2(std::cos(ang), -std::sin(ang));
            }
            c.tw[a].alloc(n);
            AUR_HIP(hipMemcpy(c.tw[a].ptr, tw.data(), n * sizeof(double2), hipMemcpyHostToDevice));
            plan_mixed(c, a);
        }
        // two half spectra in each buffer
        c.fa.alloc(2 * half_nodes(c));
        c.fb.alloc(2 * half_nodes(c));
    }
}

GreenArgs green_args(const Context& c, bool want_phi) {
    GreenArgs ga{};
    ga.nx = static_cast<int>(c.n[0]);
    ga.ny = static_cast<int>(c.n[1]);
    ga.nz = static_cast<int>(c.n[2]);
    ga.dim = c.dim;
    for (int a = 0; a < 3; ++a) ga.twopi_over_L[a] = 6.283185307179586476925286766559 / c.L[a];
    ga.eps = c.eps;
    ga.want_phi = want_phi ? 1 : 0;
    return ga;
}

// 2D/3D Dirichlet meshes bind, deposit, gather and push; their SOR field
// solve (FieldSolver.cpp:501-657) is not built.
void require_solver(const Context& c) {
    AUR_REQUIRE(c.dim == 1 || c.bc == AURORA_PERIODIC, AURORA_ERR_UNSUPPORTED,
                "2D/3D Dirichlet field solves (SOR) are not part of this build");
}

void solve_step_fields(Context& c, double phi_left, double phi_right) {
    require_solver(c);
    const bool e64 = any_fp64(c);
    if (c.dim >= 2) {
        solve_periodic(c, green_args(c, false), false, e64, true);
        c.rho_valid = false;
        c.phi_valid = false;
        c.e64_valid = e64;
        return;
    }
    {
        // 1D: the charge from the accumulators, the next ones zeroed, the solve
        const RhoArgs ra = rho_args(c);
        ClearArgs cl{};
        cl.n = static_cast<int>(c.species.size());
        for (int s = 0; s < cl.n; ++s) {
            Species& sp = c.species[s];
            if (!sp.acc_next.ptr) sp.acc_next.alloc(c.nnodes);
            cl.p[s] = reinterpret_cast<long long*>(sp.acc_next.ptr);
        }
        const LedgerFolds lf = take_ledger_folds(c);
        const int n = static_cast<int>(c.n[0]);
        if (c.bc == AURORA_PERIODIC) {
            KernelScope ks(c, "solve_spectral_1d");
            const size_t shmem = spectral_1d_lds(n);
            k_spectral_1d_acc<<<1 + lf.n, spectral_1d_threads(n), shmem, c.stream>>>(
                                                            ra, cl, lf, c.rho.ptr, c.phi.ptr,
                                                            c.E64.ptr, c.E32.ptr, c.dft_cos.ptr,
                                                            c.dft_sin.ptr, n, c.L[0], c.eps);
        } else {
            KernelScope ks(c, "solve_thomas_1d");
            k_thomas_1d_acc<<<1 + lf.n, 256, 0, c.stream>>>(ra, cl, lf, c.rho.ptr, c.phi.ptr, c.E64.ptr,
                                                     c.E32.ptr, c.thomas_inv.ptr, n, c.d[0],
                                                     c.eps, phi_left, phi_right);
        }
        AUR_HIP(hipGetLastError());
        for (auto& sp : c.species) sp.acc_next_clear = true;
        c.rho_valid = true;
        c.phi_valid = true;
        c.e64_valid = true;
    }
}

void solve_fields(Context& c, double phi_left, double phi_right, bool want_phi, bool want_e64) {
    require_solver(c);
    if (c.dim == 1) {
        const int n = static_cast<int>(c.n[0]);
        if (c.bc == AURORA_PERIODIC) {
            KernelScope ks(c, "solve_spectral_1d");
            const size_t shmem = spectral_1d_lds(n);
            k_spectral_1d<<<1, spectral_1d_threads(n), shmem, c.stream>>>(c.rho.ptr, c.phi.ptr, c.E64.ptr, c.E32.ptr,
                                                        c.dft_cos.ptr, c.dft_sin.ptr, n, c.L[0],
                                                        c.eps);
        } else {
            KernelScope ks(c, "solve_thomas_1d");
            k_thomas_1d<<<1, 256, 0, c.stream>>>(c.rho.ptr, c.phi.ptr, c.E64.ptr, c.E32.ptr,
                                                 c.thomas_inv.ptr, n, c.d[0], c.eps, phi_left,
                                                 phi_right);
        }
        AUR_HIP(hipGetLastError());
        c.phi_valid = true;
        c.e64_valid = true;
        return;
    }
    solve_periodic(c, green_args(c, want_phi), want_phi, want_e64);
    c.phi_valid = want_phi;
    c.e64_valid = want_e64;
}

}  // namespace aurora
