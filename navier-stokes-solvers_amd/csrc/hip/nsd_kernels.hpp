// nsd_kernels.hpp -- HIP kernels of the pseudospectral vorticity step.
//
// Device data layout (N = nx = ny shown; rectangular grids work the same):
//   state, acc, stage, sfd   compact spectral fields: only the modes kept by
//                            the 2/3 mask (kx <= kxmax, |ky| <= kymax),
//                            [kx][cy] with cy = ky for ky <= kymax and
//                            ky - (ny - nky_keep) for negative ky.
//   mixed[0..3], nl          "mixed" fields, transformed along y only:
//                            [kx][y], kx < nkx_keep, y contiguous.
//   physical                 [y][x] row-major (only for diagnostics/compat).
// Reference layouts (host mirrors, compat staging) are [ky][kx] with
// nkx = nx/2+1 columns (ns_spectral_solver.h:22-68).
//
// Per RK stage two kernels run:
//   k_row_stage : for each pair of rows, inverse x-transform of the four
//                 derivative fields (two complex FFTs per row using the
//                 two-real-signals-in-one-complex trick), the Jacobian
//                 J = psi_x omega_y - psi_y omega_x, the CFL speed max, and
//                 the forward x-transform of J (both rows in one complex FFT).
//   k_col_stage : for each kept kx column, forward y-transform of J, the
//                 normalisation/dealias/negation of spectral_core.c:106-111,
//                 the RK stage update (classic RK4 of
//                 spectral_time_integration.c:50-100 with hyperviscosity and
//                 SFD, or the integrating-factor variant), forcing on the
//                 last stage, then the four derivative spectra of the new
//                 state and their inverse y-transforms.
#pragma once

#include <type_traits>

#include "nsd_fft.hpp"

namespace nsd {

constexpr double kPi = 3.14159265358979323846;

struct Geo {
    int nx, ny, nkx;
    int kxmax, kymax, nkx_keep, nky_keep;
    double Lx, Ly;
};

struct Phys {
    double inv_Re;
    double Re;
    double drag;
    int scheme;  // 0 classic RK4 (reference), 1 integrating factor (Lawson RK4)
    int hv_on;
    int hv_order;
    double hv_coeff, hv_kc, hv_invbw;
    int sfd_on;
    double sfd_strength, sfd_tau;
    int adaptive;
    double cfl, dxmin;
    int force_on;
    int fbx, fby;  // forcing box: kx in [0, fbx), ky in [-fby, fby]
    // adaptive-dt error controller (with `adaptive`; the parameters of
    // AdaptiveTimeParams, include/time_integration.h:16-22, plus tolerances)
    int errctl;
    double err_rtol, err_atol, err_safety, dt_lo, dt_hi;
};

// growth limits of the error controller's step factor
constexpr double kErrFacMin = 0.2, kErrFacMax = 5.0;

struct DevScalars {
    double t;
    double dt;
    unsigned long long umax2_bits;  // max(u^2+v^2) of the stage-1 field, as ordered bits
    unsigned long long fcount;      // forcing generator call counter
    double red[8];                  // reduction outputs (sums)
    unsigned long long redmax[4];   // reduction outputs (max, as ordered bits)
    int status;                     // 0 ok, 2 diverged (SolverStatus values)
    int pad_;
    // adaptive-dt error controller
    double dt_err;                  // step the last judged error allows next
    double err;                     // last judged error norm (1 = tolerance)
    unsigned long long n_acc, n_rej;  // judged steps accepted / rejected
    int pending;                    // a candidate step waits to be judged
    int redo;                       // this step restores the last accepted state
    int errparts;                   // workgroup partials the candidate left
    int pad2_;
};

// ---------------------------------------------------------------- helpers

__device__ __forceinline__ double kx_of(const Geo& g, int i) { return 2.0 * kPi * i / g.Lx; }
__device__ __forceinline__ int band_of(const Geo& g, int j) { return j <= g.ny / 2 ? j : j - g.ny; }
__device__ __forceinline__ double ky_of(const Geo& g, int j) {
    return 2.0 * kPi * band_of(g, j) / g.Ly;
}
// spectral_initialization.c:46-49
__device__ __forceinline__ bool kept(const Geo& g, int i, int j) {
    const int b = band_of(g, j);
    return i <= g.kxmax && (b < 0 ? -b : b) <= g.kymax;
}
__device__ __forceinline__ int compact_y(const Geo& g, int j) {
    return j <= g.kymax ? j : j - (g.ny - g.nky_keep);
}

template <typename T>
__device__ __forceinline__ T powi(T x, int n) {
    T r = T(1);
    for (int i = 0; i < n; ++i) r *= x;
    return r;
}

// hyperviscosity.c:90-101
__device__ __forceinline__ double hv_weight(const Phys& p, double kmag) {
    if (!p.hv_on || kmag <= p.hv_kc) return 0.0;
    return p.hv_coeff * powi((kmag - p.hv_kc) * p.hv_invbw, p.hv_order);
}
// hyperviscosity.c:124-136
__device__ __forceinline__ double sfd_weight(const Phys& p, double kmag) {
    if (!p.sfd_on || p.hv_invbw <= 0.0 || kmag <= p.hv_kc) return 0.0;
    double s = (kmag - p.hv_kc) * p.hv_invbw;
    s = s < 0.0 ? 0.0 : (s > 1.0 ? 1.0 : s);
    return p.sfd_strength * powi(s, p.hv_order);
}

// band_of for a column of compile-time length LC (= ny): with TPL = LC / P
// the sign of the band of slot s is then known at compile time for all but
// one slot.  LC = 0 reads ny from the geometry.
template <int LC>
__device__ __forceinline__ int col_band(const Geo& g, int j) {
    if constexpr (LC > 0) return j <= LC / 2 ? j : j - LC;
    else return band_of(g, j);
}

// -1/k^2 of a nonzero wavenumber, for psi_hat = -omega_hat / k^2
// (spectral_core.c:17-20): FP32 through the hardware reciprocal (1 ulp, where
// a correctly rounded division takes about ten instructions), FP64 divides.
template <typename T>
__device__ __forceinline__ T neg_inv_k2(T k2) {
    if constexpr (sizeof(T) == 4) return -__builtin_amdgcn_rcpf(k2);
    else return T(-1) / k2;
}

// x^n (n >= 0) by repeated squaring: log2(n) steps for a runtime n.  n is
// uniform over the grid; the exponents of the usual even hyperviscous orders
// (2 to 8, halved) take straight products, the same ones the loop forms, so
// the results are identical and no lane selects between squarings.
template <typename T>
__device__ __forceinline__ T powi_sq(T x, int n) {
    if (n == 4) {
        const T x2 = x * x;
        return x2 * x2;
    }
    if (n == 1) return x;
    if (n == 2) return x * x;
    if (n == 3) return x * (x * x);
    T r = T(1);
    for (; n > 0; n >>= 1) {
        if (n & 1) r *= x;
        x *= x;
    }
    return r;
}

// The same weights evaluated at the working precision of the stage kernels,
// from k^2.  With the usual cutoff kc = 0 and an even order 2m the
// hyperviscous weight is c (k^2 / bw^2)^m, which needs no square root.
template <typename T>
__device__ __forceinline__ T hv_weight_t(const Phys& p, T k2) {
    if (!p.hv_on) return T(0);
    if (p.hv_kc == 0.0 && (p.hv_order & 1) == 0)
        return T(p.hv_coeff) * powi_sq(k2 * T(p.hv_invbw * p.hv_invbw), p.hv_order >> 1);
    const T kmag = sqrt(k2);
    if (kmag <= T(p.hv_kc)) return T(0);
    return T(p.hv_coeff) * powi_sq((kmag - T(p.hv_kc)) * T(p.hv_invbw), p.hv_order);
}
template <typename T>
__device__ __forceinline__ T sfd_weight_t(const Phys& p, T k2) {
    if (!p.sfd_on || p.hv_invbw <= 0.0) return T(0);
    const T kmag = sqrt(k2);
    if (kmag <= T(p.hv_kc)) return T(0);
    T s = (kmag - T(p.hv_kc)) * T(p.hv_invbw);
    s = s < T(0) ? T(0) : (s > T(1) ? T(1) : s);
    return T(p.sfd_strength) * powi_sq(s, p.hv_order);
}

// expm1(x) at the working precision, for the integrating-factor exponents
// L h / 2 (L <= 0 for valid parameters).  FP32: the Taylor series to x^7 for
// |x| < 0.35, whose truncation is below 0.35^7 / 8! = 1.6e-8 of |x|, and
// exp(x) - 1 from the hardware exp elsewhere, where |expm1(x)| > 0.29 bounds
// the cancellation: 2.6 ulp at most in an FP32 emulation over [-100, 0] (the
// library expm1f: ~1 ulp, at twice the instructions).  Positive x, which only
// invalid parameters give, stays within 4e-6 relative up to x = 80.  FP64
// keeps the library function.
template <typename T>
__device__ __forceinline__ T expm1_t(T x) {
    if constexpr (sizeof(T) == 4) {
        if (x < -18.f) return -1.f;  // e^x < 2^-25: -1 is expm1 correctly rounded
        const float p =
            x * (1.f + x * (0.5f + x * (1.f / 6 + x * (1.f / 24 + x * (1.f / 120 +
                 x * (1.f / 720 + x * (1.f / 5040)))))));
        const float e = __expf(x) - 1.f;
        return fabsf(x) < 0.35f ? p : e;
    } else {
        // e^x < 2^-54 for x < -40, so -1 is expm1 correctly rounded: the modes that
        // the hyperviscous factor damps completely (most of the high
        // wavenumbers) skip the library call
        if (x < -40.0) return -1.0;
        return expm1(x);
    }
}

// spectral_time_integration.c:22-28 with MIN_DT/MAX_DT of common_types.h:32-33
__device__ __forceinline__ double cfl_dt(const Phys& p, double umax) {
    const double dt_cfl = p.cfl * p.dxmin / (umax + 1e-12);
    const double dt_visc = 0.5 * p.Re * p.dxmin * p.dxmin;
    double dt = fmin(dt_cfl, dt_visc);
    dt = fmax(dt, 1e-8);
    dt = fmin(dt, 0.1);
    return dt;
}

__device__ __forceinline__ unsigned long long ordered_bits(double x) {
    return (unsigned long long)__double_as_longlong(x);
}

template <typename T>
__device__ __forceinline__ T wave_max(T v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        T w = __shfl_xor(v, o, 64);
        v = w > v ? w : v;
    }
    return v;
}
template <typename T>
__device__ __forceinline__ T wave_sum(T v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// Block-wide max of non-negative doubles folded into *dst with one atomic per
// workgroup (non-negative doubles order like their bit patterns; NaN and Inf
// order above every finite value, so divergence is never lost).
__device__ __forceinline__ void block_max_to(double v, unsigned long long* dst, double* red_lds) {
    v = wave_max(v);
    const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
    __syncthreads();
    if (l == 0) red_lds[w] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        double m = red_lds[0];
        for (int i = 1; i < (int)(blockDim.x >> 6); ++i) m = red_lds[i] > m ? red_lds[i] : m;
        if (m != m) m = __longlong_as_double(0x7ff8000000000000LL);
        atomicMax(dst, ordered_bits(m));
    }
}

// Running maximum of squared speeds u^2 + v^2.  Every value is a sum of
// squares (+0, positive, +inf) or a NaN; for those the unsigned order of the
// FP32 bit patterns is the numeric order with every NaN above +inf, so one
// integer max per value does the NaN test and the compare-select at once.  A
// NaN reads back as +inf: a diverged field still wins the max (and drives the
// CFL dt to its floor).  FP64 has no 64-bit integer max, so it compares.
template <typename T>
struct SpeedMax {
    T m = T(0);
    __device__ __forceinline__ void add(T s) {
        if (s != s) s = T(__builtin_inf());
        m = s > m ? s : m;
    }
    __device__ __forceinline__ T value() const { return m; }
};
template <>
struct SpeedMax<float> {
    unsigned m = 0u;
    __device__ __forceinline__ void add(float s) { m = max(m, __float_as_uint(s)); }
    __device__ __forceinline__ float value() const {
        const float f = __uint_as_float(m);
        return f != f ? __builtin_inff() : f;
    }
};

// Speeds of two rows transformed together: a holds psi_x, b holds psi_y of
// rows y0 (real parts) and y0 + 1 (imaginary parts); u = psi_y, v = -psi_x
// (spectral_core.c:30-31).
template <typename T>
__device__ __forceinline__ void add_speeds(SpeedMax<T>& um, const cx<T>* a, const cx<T>* b) {
#pragma unroll
    for (int s = 0; s < P; ++s) {
        um.add(a[s].x * a[s].x + b[s].x * b[s].x);
        um.add(a[s].y * a[s].y + b[s].y * b[s].y);
    }
}

__device__ __forceinline__ void block_sum_to(double v, double* dst, double* red_lds) {
    v = wave_sum(v);
    const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
    __syncthreads();
    if (l == 0) red_lds[w] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        double s = 0.0;
        for (int i = 0; i < (int)(blockDim.x >> 6); ++i) s += red_lds[i];
        atomicAdd(dst, s);
    }
}

template <typename T>
__device__ __forceinline__ cx<T> ld(const cx<T>* p, size_t i) {
    return p[i];
}
template <typename T>
__device__ __forceinline__ cx<T> ld_ref(const double* p, size_t i) {  // interleaved FP64
    return mk(T(p[2 * i]), T(p[2 * i + 1]));
}
template <typename T>
__device__ __forceinline__ void st_ref(double* p, size_t i, cx<T> v) {
    p[2 * i] = double(v.x);
    p[2 * i + 1] = double(v.y);
}

// line transform of compile-time length LC (> 0) or runtime length g.L
template <int DIR, int LC, typename T>
__device__ __forceinline__ void fft_any(cx<T> (&v)[P], cx<T>* lds, int j, const Line& g,
                                        const cx<T>* __restrict__ tw) {
    if constexpr (LC > 0) line_fft_c<DIR, LC>(v, lds, j, tw);
    else line_fft<DIR>(v, lds, j, g, tw);
}
template <int DIR, int LC, typename T>
__device__ __forceinline__ void fft_any(cx<T> (&v)[P], cx<T>* lds, int j, const Line&,
                                        const TwRegs<LC, T>& tw) {
    line_fft_c<DIR, LC>(v, lds, j, tw);
}
// wave-split transform, wave-strided pattern in (a pointwise
// product of ws_a outputs), standard pattern out; the region is free again
// only after a workgroup barrier
template <int DIR, int LC, typename T>
__device__ __forceinline__ void fft_any(cx<T> (&v)[P], cx<T>* lds, int j, const Line&,
                                        const TwWs<LC, T>& tw) {
    cx<T>(*const vv[1])[P] = {&v};
    cx<T>* const ll[1] = {lds};
    ws_b<DIR, 1, (sizeof(T) == 8)>(vv, ll, j, tw);  // 16-byte rows at FP64
    __syncthreads();
}

// Element i of a mixed field at (workgroup-uniform) base F, addressed as the
// base plus a 32-bit byte offset: the loads then take the scalar base and one
// 32-bit offset register per slot.  A mixed field is at most 2731 x 8192
// FP64 complex values (358 MB), well inside 32 bits.
// Element (k, y) of a mixed field (column k, row y): k ny + y through the
// full-rate 24-bit multiply (k and ny are below 2^24; the 32-bit multiply
// issues at a quarter of the rate).
__device__ __forceinline__ unsigned col_elem(int k, int ny, int y) {
    return __umul24((unsigned)k, (unsigned)ny) + (unsigned)y;
}

// Element (k, y) of J in 2 x 2 blocks: columns k, k ^ 1 and rows y, y ^ 1 in
// 32 contiguous bytes at FP32, ordered (k even: y even, y odd; k odd: ...).
// The row stage then stores one row pair's two values of a column as one
// 16-byte piece next to its neighbour column's (a lane pair fills the block),
// so no line leaves L2 half written; the column stage reads 8 of each 16
// bytes.  The buffer holds an even number of columns.
__device__ __forceinline__ unsigned jblock_elem(int k, int ny, int y) {
    return ((__umul24((unsigned)(k >> 1), (unsigned)(ny >> 1)) + (unsigned)(y >> 1)) << 2) +
           ((unsigned)(k & 1) << 1) + (unsigned)(y & 1);
}

// Element (k, y) of a mixed field in row-pair tiles: ROWPAIR_TY rows of all K
// buffer columns in one run, column by column, (y - y % TY) K + TY k + y % TY.
// With TY = 2 (FP64, 32 bytes per column) a row pair's elements are one
// contiguous run and ROWPAIR_CPL = 4 columns share a 128-byte line.
constexpr int ROWPAIR_TY = 2;
constexpr int ROWPAIR_CPL = 128 / (ROWPAIR_TY * 16);
__device__ __forceinline__ unsigned rowpair_elem(int k, int K, int y) {
    constexpr unsigned TY = ROWPAIR_TY;
    return __umul24((unsigned)y & ~(TY - 1), (unsigned)K) + TY * (unsigned)k +
           ((unsigned)y & (TY - 1));
}

// This thread's slots of one line of a mixed field: slot s at element
// e0 + s es.
struct SlotElems {
    unsigned e0, es;
};
// Row stage, rows y, y + 1 (y even): slot s is column j + s LC/P.
template <int LC>
__device__ __forceinline__ SlotElems row_slots(int j, int ny, int K, int y, bool tiles) {
    if (tiles) return {rowpair_elem(j, K, y), (unsigned)ROWPAIR_TY * (LC / P)};
    return {col_elem(j, ny, y), (unsigned)ny * (LC / P)};
}
// Column stage, column k: slot s is row j + s LC/P (LC / P a multiple of
// ROWPAIR_TY).
template <int LC>
__device__ __forceinline__ SlotElems col_slots(int k, int j, int ny, int K, bool tiles) {
    static_assert((LC / P) % ROWPAIR_TY == 0, "slots step by whole tiles");
    if (tiles) return {rowpair_elem(k, K, j), (unsigned)K * (LC / P)};
    return {col_elem(k, ny, j), (unsigned)(LC / P)};
}

template <typename T>
__device__ __forceinline__ const cx<T>* at32(const cx<T>* F, unsigned i) {
    return reinterpret_cast<const cx<T>*>(reinterpret_cast<const char*>(F) +
                                          i * (unsigned)sizeof(cx<T>));
}
template <typename T>
__device__ __forceinline__ cx<T>* at32(cx<T>* F, unsigned i) {
    return reinterpret_cast<cx<T>*>(reinterpret_cast<char*>(F) + i * (unsigned)sizeof(cx<T>));
}

// Kept bands of the 2/3 rule (spectral_initialization.c:46-48) for lines of
// compile-time length LC: last kept kx of a row of length LC and last kept
// |ky| of a column of length LC.  slot_kind classifies register slot s of
// the standard pattern (indices s*TPL .. s*TPL+TPL-1): 1 = always in the
// positive kept band, 2 = always in the negative (mirrored) kept band,
// 0 = never kept, 3 = straddles a band edge (decided per lane).
template <int LC>
struct Band {
    static constexpr int kxm = (2 * (LC / 2 + 1)) / 3;
    static constexpr int kym = (2 * LC) / 6;
};

// Whether the time-step kernels run their inverse transforms two at a time
// (needs two line regions per line in LDS): when the workgroup's two regions stay
// within 80 KB, so that two workgroups share a CU.
// FP32 lines of 8192 are paired as well (147 KB, one workgroup of 16 waves per
// CU): one region leaves room for no second workgroup either, and the
// wave-split pairs took k_row at 8192^2 from 926 to 537 us and k_col from 527
// to 450 us (per-pair layout).  FP64 lines of 2048 are not, though two regions
// would fit: they run wave-split in a field at a time like those of 4096
// (ws_lines64; 2048^2 FP64 step 351 -> 311 us).
template <typename T, int LC, int NT = threads_for(LC)>
constexpr bool paired_lines() {
    if (LC <= 0) return false;
    if (sizeof(T) == 4 && LC == 8192) return true;
    if (sizeof(T) == 8 && LC == 2048) return false;
    return 2 * (LC + LC / 16) * (int)sizeof(cx<T>) * (NT * P / LC) <= 80 * 1024;
}
template <typename T, int LC, int NT = threads_for(LC)>
constexpr int line_regions() {
    return paired_lines<T, LC, NT>() ? 2 : 1;
}

// FP64 lines of 2048 and 4096 (two workgroups or one per CU): wave-split
// transforms with a second line region.  The row stage stages each field in
// one region and runs the cross-wave rows in the other, so staging the next
// field needs no barrier of its own; the column stage transposes back to the
// standard pattern through the second region, so consecutive transforms need
// none between them.
template <typename T, int LC, int NT = threads_for(LC)>
constexpr bool ws_lines64() {
    return sizeof(T) == 8 && (LC == 2048 || LC == 4096) && NT * P == LC &&
           !paired_lines<T, LC, NT>();
}


constexpr int slot_kind(int s, int L, int km) {
    const int tpl = L / P, lo = s * tpl, hi = lo + tpl - 1;
    if (hi <= km) return 1;
    if (lo >= L - km && lo > 0) return 2;
    if (lo > km && hi < L - km) return 0;
    return 3;
}

// ---------------------------------------------------------------- forcing

__device__ __forceinline__ unsigned long long splitmix64_at(unsigned long long seed,
                                                            unsigned long long k) {
    // k-th output (k >= 1) of the SplitMix64 stream of forcing.c:11-16
    unsigned long long z = seed + k * 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}
__device__ __forceinline__ double uniform_at(unsigned long long seed, unsigned long long k) {
    return (double)(splitmix64_at(seed, k) >> 11) * (1.0 / 9007199254740992.0);
}

// Forcing draws (forcing.c:117-184 semantics through the counter form of the
// SplitMix64 stream: on call c with A active modes, mode rank a uses
// uniforms 2(cA+a)+1 and 2(cA+a)+2), then the build-defined application:
// Hermitian projection of the kx = 0 column, mask, and scaling to the
// injection rate.
struct ForceArgs {
    Geo geo;
    int A;
    const int* modes;    // reference index j*nkx + i per active mode (reference order)
    const int* partner;  // rank of the (0, ny-j) partner for kx = 0 modes, else -1
    unsigned long long seed;
    int colored;
    double tau, energy_target, rate;
    double* ou;          // colored state per active rank (interleaved complex)
    double* work;        // 5 A doubles
    int fbx, fby;
    int box_T;           // 1: box in FP32, 0: FP64
    void* fbox;
    DevScalars* sc;
    const unsigned long long* m_seed;  // per-member seeds of a batch (else seed)
    int skip_on_redo;                  // error controller: no draw on a restoring step
};

// Sums over the modes are formed over 256 lanes, whatever the workgroup, with the
// products' roundings written out, so that a draw's bits do not depend on the launch
// that makes it: lane v adds the modes v, v + 256, ..., and the four waves' sums are
// added in order.
constexpr int kForceLanes = 256;
// those that have modes, in whole waves
__device__ __forceinline__ int force_lanes(int A) { return min(kForceLanes, (A + 63) & ~63); }

// value(r) for the modes r < A, which also stores it where load(r) finds it, and
// add(sum, value) over them, the waves' sums in red[0 .. 3]; every thread of a workgroup
// of whole waves calls it.  ALL: the values by all threads of a larger workgroup, then
// summed from memory; else by the lanes of the sums.
template <bool ALL, typename V, typename L, typename F>
__device__ __forceinline__ void force_sum(int A, double* red, V&& value, L&& load, F&& add) {
    if constexpr (ALL) {
        for (int r = threadIdx.x; r < A; r += blockDim.x) (void)value(r);
        __syncthreads();
    }
    for (int v = threadIdx.x; v < force_lanes(A); v += blockDim.x) {
        double part = 0.0;
        int r = v;
        if constexpr (ALL) {
            constexpr int N = 8;  // loads in flight
            for (; r + (N - 1) * kForceLanes < A; r += N * kForceLanes) {
                decltype(load(0)) x[N];
#pragma unroll
                for (int i = 0; i < N; ++i) x[i] = load(r + i * kForceLanes);
#pragma unroll
                for (int i = 0; i < N; ++i) part = add(part, x[i]);
            }
            for (; r < A; r += kForceLanes) part = add(part, load(r));
        } else {
            for (; r < A; r += kForceLanes) part = add(part, value(r));
        }
        part = wave_sum(part);
        if ((v & 63) == 0) red[v >> 6] = part;
    }
    __syncthreads();
}
__device__ __forceinline__ double force_total(int A, const double* red) {
    double t = 0.0;
    for (int i = 0; i < force_lanes(A) / 64; ++i) t += red[i];
    return t;
}

// The draw for member mb, by one workgroup; red: kForceRed doubles of LDS.
constexpr int kForceRed = kForceLanes / 64 + 1;
template <bool ALL>
__device__ __forceinline__ void force_draw(const ForceArgs& a, int mb, double* red) {
    const Geo& G = a.geo;
    // member mb of a batch: its own generator, OU state, box and scalars
    const size_t box0 = (size_t)a.fbx * (2 * a.fby + 1) * mb;
    DevScalars* const dsc = a.sc + mb;
    double* const ou = a.ou + (size_t)mb * 2 * a.A;
    double* const work = a.work + (size_t)mb * 5 * a.A;
    float* const box32 = reinterpret_cast<float*>(a.fbox) + 2 * box0;
    double* const box64 = reinterpret_cast<double*>(a.fbox) + 2 * box0;
    const unsigned long long seed = a.m_seed ? a.m_seed[mb] : a.seed;
    const unsigned long long c = dsc->fcount;
    const double dt = dsc->dt;
    double& s_scale = red[kForceLanes / 64];
    double alpha = 0.0, beta = 1.0;
    if (a.colored) {
        const double tau = fmax(a.tau, 1e-6);
        alpha = exp(-dt / tau);
        beta = sqrt(fmax(1.0 - alpha * alpha, 0.0));
    }
    auto draw = [&](int r) {
        const unsigned long long k = 2ull * (c * (unsigned long long)a.A + r) + 1ull;
        double u1 = uniform_at(seed, k), u2 = uniform_at(seed, k + 1);
        u1 = fmax(u1, 2.2250738585072014e-308);
        const double rad = sqrt(-2.0 * log(u1));
        const double th = 2.0 * kPi * u2;
        double vr = rad * cos(th), vi = rad * sin(th);
        if (a.colored) {
            vr = alpha * ou[2 * r] + beta * vr;
            vi = alpha * ou[2 * r + 1] + beta * vi;
        }
        work[2 * r] = vr;
        work[2 * r + 1] = vi;
        return mk(vr, vi);
    };
    force_sum<ALL>(
        a.A, red, draw, [&](int r) { return mk(work[2 * r], work[2 * r + 1]); },
        [](double t, cx<double> f) { return fma(f.x, f.x, fma(f.y, f.y, t)); });
    if (threadIdx.x == 0) s_scale = sqrt(a.energy_target / fmax(force_total(a.A, red), 1e-16));
    __syncthreads();
    const double sc = s_scale;
    for (int r = threadIdx.x; r < a.A; r += blockDim.x) {
        work[2 * r] *= sc;
        work[2 * r + 1] *= sc;
        if (a.colored) {
            ou[2 * r] = work[2 * r];
            ou[2 * r + 1] = work[2 * r + 1];
        }
    }
    __syncthreads();
    // Hermitian projection + mask, rate of the projected field
    double* const pr = work + 2 * a.A;  // projected values
    double* const er = work + 4 * a.A;  // and the rates that they inject
    auto project = [&](int r) {
        const int idx = a.modes[r];
        const int jy = idx / G.nkx, i = idx % G.nkx;
        double fr = work[2 * r], fi = work[2 * r + 1];
        if (i == 0 || 2 * i == G.nx) {
            const int p = a.partner[r];
            if (p >= 0) {
                fr = 0.5 * (fr + work[2 * p]);
                fi = 0.5 * (fi - work[2 * p + 1]);
            } else if (jy == 0 || 2 * jy == G.ny) {
                fi = 0.0;
            }
        }
        const double kx = kx_of(G, i), ky = ky_of(G, jy);
        const double k2 = kx * kx + ky * ky;
        if (!kept(G, i, jy) || k2 <= 1e-12) fr = fi = 0.0;
        pr[2 * r] = fr;
        pr[2 * r + 1] = fi;
        const double wt = (i == 0 || 2 * i == G.nx) ? 1.0 : 2.0;
        const double e = k2 > 1e-12 ? 0.5 * wt * fma(fr, fr, fi * fi) / k2 : 0.0;
        if constexpr (ALL) er[r] = e;
        return e;
    };
    force_sum<ALL>(
        a.A, red, project, [&](int r) { return er[r]; }, [](double t, double e) { return t + e; });
    if (threadIdx.x == 0) {
        const double t = force_total(a.A, red);
        s_scale = (t > 0.0 && a.rate > 0.0) ? sqrt(a.rate / t) : 0.0;
    }
    __syncthreads();
    const double s2 = s_scale;
    const int boxn = a.fbx * (2 * a.fby + 1);
    for (int e = threadIdx.x; e < boxn; e += blockDim.x) {
        if (a.box_T) box32[2 * e] = box32[2 * e + 1] = 0.f;
        else box64[2 * e] = box64[2 * e + 1] = 0.0;
    }
    __syncthreads();
    for (int r = threadIdx.x; r < a.A; r += blockDim.x) {
        const int idx = a.modes[r];
        const int jy = idx / G.nkx, i = idx % G.nkx;
        const int b = band_of(G, jy);
        if (i >= a.fbx || b < -a.fby || b > a.fby) continue;
        const int e = i * (2 * a.fby + 1) + (b + a.fby);
        if (a.box_T) {
            box32[2 * e] = float(s2 * pr[2 * r]);
            box32[2 * e + 1] = float(s2 * pr[2 * r + 1]);
        } else {
            box64[2 * e] = s2 * pr[2 * r];
            box64[2 * e + 1] = s2 * pr[2 * r + 1];
        }
    }
    if (threadIdx.x == 0) dsc->fcount = c + 1;
}

// ------------------------------------------------------------ column side

enum ColMode { COL_STAGE = 0, COL_PRIME = 1, COL_FWD = 2, COL_INV = 3 };

// Field operations applied in spectral space before an inverse y-transform
// (COL_INV), derived from the reference's spectral_core.c:8-34,62-99.
enum FieldOp {
    OP_ID0 = 0,   // in0
    OP_ID1 = 1,   // in1
    OP_DX0 = 2,   // i kx in0
    OP_DY0 = 3,   // i ky in0
    OP_DX1 = 4,   // i kx in1
    OP_DY1 = 5,   // i ky in1
    OP_PSI0 = 6,  // psi_hat = -in0/k^2 (quirk: sign of spectral_core.c:18)
    OP_U0 = 7,    // u_hat = i ky psi_hat(in0)
    OP_V0 = 8,    // v_hat = -i kx psi_hat(in0)
};

template <typename T>
struct ColArgs {
    Geo geo;
    Phys phys;
    int mode;
    int stage;       // 0..3 for COL_STAGE
    int nout;        // number of mixed outputs (COL_INV)
    int ops[4];      // FieldOp per output (COL_INV)
    int in_ref;      // COL_INV inputs / COL_FWD output in FP64 reference layout
    double fwd_scale;  // COL_FWD: factor applied with the 1/(nx ny) normalisation
    const cx<T>* tw;  // twiddles for length ny
    const cx<T>* nl;  // mixed input (COL_STAGE, COL_FWD)
    cx<T>* mixed[4];  // mixed outputs
    int pairs;        // COL_STAGE, COL_PRIME: write them in the stage layout (stage_layout)
    int jblocks;      // COL_STAGE, COL_FWD: J in 2 x 2 blocks (square pair-layout grids)
    cx<T>* state;     // compact state (read; written on the last stage)
    cx<T>* acc;       // compact RK accumulator
    cx<T>* stagebuf;  // compact stage state (classic scheme)
    cx<T>* sfd;       // compact SFD filter state (classic scheme, if on)
    const cx<T>* fbox;  // forcing box [fbx][2 fby + 1], already scaled to the injection rate
    const double* in0_ref;
    const double* in1_ref;
    const cx<T>* in0;  // compact inputs for COL_INV (if !in_ref)
    double* out_ref;   // COL_FWD output, FP64 reference layout, all nkx columns
    DevScalars* sc;
    // batches: member blockIdx.y works on fields offset by these element
    // strides, on scalars sc[blockIdx.y] and, if set, its own 1/Re
    size_t bm, bc, bf;
    const double* m_inv_re;
    cx<T>* out_c;      // COL_FWD: compact output of the kept modes (instead of out_ref)
    const cx<T>* src;  // COL_STAGE: compact source added to the nonlinear term
    int nbat;          // members along grid y for the transform modes (0 = 1)
    // error controller (COL_STAGE, ERR): state before the step, midpoint
    // solution, per-workgroup {sum w |y4 - y2|^2, sum w |y4|^2} (stride bp
    // per member); finalize: stage 0 only restores a rejected step
    cx<T>* prev;
    cx<T>* ymid;
    double* errpart;
    size_t bp;
    int finalize;
    double kxs, kys, norm;  // 2 pi / Lx, 2 pi / Ly, 1 / (nx ny) (field-parallel kernels)
};

template <typename T>
__device__ __forceinline__ cx<T> apply_op(int op, cx<T> a, cx<T> b, T kx, T ky, T k2) {
    switch (op) {
    case OP_ID0: return a;
    case OP_ID1: return b;
    case OP_DX0: return mul_i(a, kx);
    case OP_DY0: return mul_i(a, ky);
    case OP_DX1: return mul_i(b, kx);
    case OP_DY1: return mul_i(b, ky);
    default: break;
    }
    const cx<T> psi = k2 > T(1e-12) ? neg_inv_k2(k2) * a : mk(T(0), T(0));
    if (op == OP_PSI0) return psi;
    if (op == OP_U0) return mul_i(psi, ky);
    return mul_i(psi, -kx);  // OP_V0
}

// (1 + em1) * w with em1 = factor - 1, rounded once per component
template <typename T>
__device__ __forceinline__ cx<T> grow(cx<T> w, T em1) {
    return mk(fma(em1, w.x, w.x), fma(em1, w.y, w.y));
}

// occupancy floor handed to the register allocator: waves per SIMD
// Pair layout of the stage kernels' mixed fields (FP32, 2048- and 4096-point lines):
// (psi_x, psi_y) interleaved per (kx, y) in the buffer of psi_x and psi_y,
// (omega_x, omega_y) likewise in that of omega_x and omega_y; pair element e
// = kx ny + y of member m sits at 2 (m M + e) of the pair's buffer (M = kept
// kx times ny).  A row pair's two 16-byte gathers of one pair then fall in
// one 64-byte line, where the per-field layout puts a field's row pair in a
// line of its own: half the L1 misses of the row kernel's gathers, whose
// address path otherwise waits on the cache for about half of its cycles.
// k_col still writes whole lines (one 16-byte store per lane and pair).
// It is a property of the instantiation: the paired wave-split transforms of
// square FP32 2048^2, 4096^2 and (in row-pair tiles, pairtile_layout) 8192^2
// grids (the gather-ahead k_row path reads it, the paired k_col path writes
// it).  The host selects it per launch (ColArgs/RowArgs::pairs) when the row and
// column instantiations it launches both hold it (stage_variant_pairs); the
// transform modes keep the per-field layout.  At 2048 it came with the
// wave-split transforms (2048^2 FP32: k_row 29.2 -> 24.7 us, k_col 23.5 -> 24.1,
// step 194 -> 180 us); at 64..1024, with Stockham lines, it measured slower
// (256-member ensemble 92k -> 86k member-steps/s).
template <typename T, int LC, int NT>
constexpr bool pair_layout() {
    return sizeof(T) == 4 && (LC == 2048 || LC == 4096 || LC == 8192) && NT * P == LC &&
           paired_lines<T, LC, NT>();
}

// Row-pair tiles of the mixed fields (rowpair_elem): the FP64 stage kernels
// of 2048 and 4096 (ws_lines64), selected per launch like the pair layout.  A row
// pair's gathers of one field then read one contiguous run of 32 bytes per
// kept column, neighbouring columns adjacent (2 KB per wave instruction),
// where the per-field layout puts every lane in a 64 KB column of its own and
// a row pair's gathers span the fields' whole 358 MB; k_col writes 32-byte
// runs, ROWPAIR_CPL columns to a 128-byte line (xcd_group_remap keeps them on
// one XCD, one after the other).  J stays [kx][y]: in tiles of 2, 4 or 8
// rows the column stage's reads of it cost more than the row stage's stores
// gained.
template <typename T, int LC, int NT>
constexpr bool rowpair_layout() {
    return ws_lines64<T, LC, NT>();
}

// Row-pair tiles of the pair buffers: FP32 lines of 8192.  Element (kx, y) of
// member m of a pair at 4 ((y / 2) K + kx) + 2 (y mod 2) + m (pairtile_elem):
// both rows of both fields are 32 bytes per column and a row pair's gather of
// a pair buffer is one contiguous run, as in the FP64 tiles above; four
// columns share a 128-byte line.  The 716 MB of mixed fields at 8192^2 lie
// beyond the MALL and the reach of the address translation, as the FP64
// 4096^2 ones do: against the pair layout k_row takes 423 us instead of 537
// and k_col 499 instead of 450 (8192^2 step 3.93 -> 3.65 ms; at the start of
// both, with Stockham lines in one region and the per-field layout, 5.81 ms).
// What bounds them now: about 16 us of VALU issue in the 26 us of a row pair,
// with one workgroup per CU whose waves wait at the same barriers.  A
// persistent row stage that gathered the next row pair's psi fields under J's
// transform took 477 us (96 bytes of scratch).
template <typename T, int LC, int NT>
constexpr bool pairtile_layout() {
    return LC == 8192 && pair_layout<T, LC, NT>();
}
__device__ __forceinline__ unsigned pairtile_elem(int k, int K, int y) {
    return 4u * (__umul24((unsigned)y >> 1, (unsigned)K) + (unsigned)k) + 2u * ((unsigned)y & 1u);
}

// the stage kernels' own layout of the mixed fields, if any (RowArgs and
// ColArgs::pairs select it per launch)
template <typename T, int LC, int NT>
constexpr bool stage_layout() {
    return pair_layout<T, LC, NT>() || rowpair_layout<T, LC, NT>();
}

// line regions of the stage kernels
template <typename T, int LC, int NT = threads_for(LC)>
constexpr int stage_regions() {
    return ws_lines64<T, LC, NT>() ? 2 : line_regions<T, LC, NT>();
}
// stage kernels that run wave-split transforms (their line regions hold
// WS_REGION elements; staged lines in them are unpadded)
template <typename T, int LC, int NT = threads_for(LC)>
constexpr bool ws_stage() {
    return pair_layout<T, LC, NT>() || ws_lines64<T, LC, NT>();
}
// elements of one line region of a stage kernel (compile-time lengths)
template <typename T, int LC, int NT = threads_for(LC)>
constexpr int region_elems() {
    return ws_stage<T, LC, NT>() ? ws_region(LC) : LC + LC / 16;
}

// store (first, second) at pair element e of pair buffer B (one 16 bytes)
__device__ __forceinline__ void store_pair(cx<float>* B, size_t e, cx<float> first,
                                           cx<float> second) {
    *reinterpret_cast<float4*>(B + 2 * e) = make_float4(first.x, first.y, second.x, second.y);
}

// a thread's slots (first, second) of column k into row-pair tiles of pair
// buffer B: rows j + s LC / P
template <int LC>
__device__ __forceinline__ void store_pair_tiles(cx<float>* B, int k, int K, int j,
                                                 const cx<float> (&first)[P],
                                                 const cx<float> (&second)[P]) {
    static_assert((LC / P) % 2 == 0, "slots step by whole tiles");
    const unsigned e0 = pairtile_elem(k, K, j), es = 2u * (unsigned)(LC / P) * (unsigned)K;
#pragma unroll
    for (int s = 0; s < P; ++s)
        *reinterpret_cast<float4*>(at32(B, e0 + (unsigned)s * es)) =
            make_float4(first[s].x, first[s].y, second[s].x, second[s].y);
}

template <typename T>
constexpr int min_waves() { return sizeof(T) == 4 ? 4 : 2; }

// Twiddle source of a kernel's compile-time transforms: registers (REG) or
// the table in global memory.
template <bool REG, int L, typename T>
struct TwSource {
    using type = const cx<T>*;
};
template <int L, typename T>
struct TwSource<true, L, T> {
    using type = TwRegs<L, T>;
};

// MW: occupancy floor handed to the register allocator (waves per SIMD)
template <typename T, int NT, int MODE, int SCHEME, int LC, bool ERR = false,
          int MW = min_waves<T>()>
__global__ __launch_bounds__(NT, MW) void k_col(ColArgs<T> a) {
    static_assert(!pair_layout<T, LC, NT>() || paired_lines<T, LC, NT>(),
                  "the pair layout is written by the paired k_col path");
    extern __shared__ __align__(16) unsigned char smem_raw[];
    cx<T>* smem = reinterpret_cast<cx<T>*>(smem_raw);
    const Geo& G = a.geo;
    // member blockIdx.y of a batch: its fields, scalars and 1/Re (the
    // argument block itself stays untouched, in constant kernarg memory)
    const size_t mb = blockIdx.y;
    const cx<T>* const nl = a.nl + mb * a.bm;
    cx<T>* const state = a.state + mb * a.bc;
    cx<T>* const acc = a.acc + mb * a.bc;
    cx<T>* const stagebuf = a.stagebuf + mb * a.bc;
    cx<T>* const sfd = a.sfd + mb * a.bc;
    const cx<T>* const fbox = a.fbox + mb * a.bf;
    DevScalars* const sc = a.sc + mb;
    const cx<T>* const src = a.src ? a.src + mb * a.bc : nullptr;
    const size_t mixed_off = mb * a.bm;
    // Error controller: a step that restores a rejected candidate runs only
    // its stage-0 column pass, which writes the restored state and its
    // derivative fields; a finalize pass does the same, and nothing when the
    // last candidate was accepted.  (`redo` is uniform over the grid.)
    int redo = 0;
    if constexpr (ERR && MODE == COL_STAGE) {
        redo = sc->redo;
        if (redo ? a.stage > 0 : a.finalize != 0) return;
    }
    cx<T>* const prev = ERR ? a.prev + mb * a.bc : nullptr;
    cx<T>* const ymid = ERR ? a.ymid + mb * a.bc : nullptr;
    Phys ph = a.phys;
    if (a.m_inv_re) {
        ph.inv_Re = a.m_inv_re[mb];
        ph.Re = 1.0 / ph.inv_Re;
    }
    const Line g = make_line(LC > 0 ? LC : G.ny);
    const int TPL = LC > 0 ? LC / P : g.TPL;
    const int Ll = LC > 0 ? LC : g.L;
    const int lines = NT / TPL;
    const int m = threadIdx.x / TPL, j = threadIdx.x - m * TPL;
    constexpr int NB = stage_regions<T, LC, NT>();
    const int RE = LC > 0 ? region_elems<T, LC, NT>() : Ll + Ll / 16;
    cx<T>* lds = smem + m * NB * RE;
    cx<T>* lds2 = lds + (NB - 1) * RE;
    constexpr bool WS = ws_lines64<T, LC, NT>();
    // forward transform through ws_c as well (two line regions free for it)
    constexpr bool WSF = WS || pairtile_layout<T, LC, NT>();
    // pair-layout kernels read J in 2 x 2 blocks: columns k and k ^ 1 share
    // lines; row-pair tiles put ROWPAIR_CPL columns in one line
    constexpr int XG = pairtile_layout<T, LC, NT>()   ? 4
                       : pair_layout<T, LC, NT>()    ? 2
                       : rowpair_layout<T, LC, NT>() ? ROWPAIR_CPL
                                                         : 1;
    const int kxi = xcd_group_remap<XG>(blockIdx.x, gridDim.x) * lines + m;
    const int ncols = (MODE == COL_FWD) ? G.nkx : G.nkx_keep;
    // The stage launches cover exactly the kept columns (launch_col_fused);
    // with one column per workgroup every workgroup has one, and the
    // compiler drops the zero fills and masks of an idle column.  Taken for
    // the prime pass and the integrating-factor stage up to 4096 points: in
    // the classic scheme with the error controller, and at 8192, the freed
    // schedule costs the compiler registers it then spills; up to 512 points
    // one column per workgroup is a launch variant, which has to round as the
    // others do.
    constexpr bool ALL_KEPT = (MODE == COL_PRIME || (MODE == COL_STAGE && SCHEME == 1)) &&
                              LC > 512 && LC <= 4096 && NT * P / LC == 1;
    const bool active = ALL_KEPT || kxi < ncols;
    const bool has_data = ALL_KEPT || (active && kxi < G.nkx_keep);
    const T kx = T(kxi) * T(2.0 * kPi / G.Lx);
    const size_t mbase = (size_t)kxi * G.ny;
    const cx<T> zero = mk(T(0), T(0));

    cx<T> v[P];
    cx<T> w[P];

    // y-band of the 2/3 mask: compile-time for compile-time column lengths
    const int kym = LC > 0 ? Band<LC>::kym : G.kymax;
    const int ncy = LC > 0 ? 2 * Band<LC>::kym + 1 : G.nky_keep;
    // Paired stage columns of compile-time length: the state and accumulator
    // values of this column are loaded ahead of the forward transform, which
    // runs while they arrive (its twiddles in registers, loaded first, so that
    // it has no global load of its own to wait behind them).
    constexpr bool PF = MODE == COL_STAGE && LC >= 64 &&
                        (paired_lines<T, LC, NT>() || (sizeof(T) == 8 && NT <= 512));
    cx<T> pw0[P], pacc[P];
    // The smallest FP32 workgroups (launches with few waves): dt and the modes'
    // factors before the transform of J, which waits a memory latency anyway.
    // 256^2 step 58.8 -> 58.2 us, 128^2 54.4 -> 53.5 us.
    constexpr bool EARLY = PF && sizeof(T) == 4 && NT == 64 && !ERR;
    T el[P], es[P];  // el: L or E - 1, es: the SFD weight or E2 - 1
    double dt = 0.0, u2 = 0.0;
    auto pick_dt = [&]() {
        dt = cfl_dt(ph, sqrt(u2));
        // the error controller's step limit, within [dt_min, dt_max]
        if constexpr (ERR) dt = fmin(fmax(fmin(dt, sc->dt_err), ph.dt_lo), ph.dt_hi);
        if (blockIdx.x == 0 && threadIdx.x == 0 && !redo) {
            sc->dt = dt;
            if (!(u2 <= 1.0e300)) sc->status = 2;  // SOLVER_DIVERGED
        }
    };
    if constexpr (EARLY) {
        if (a.stage == 0 && ph.adaptive) u2 = __longlong_as_double((long long)sc->umax2_bits);
        else dt = sc->dt;
    }

    // ---- forward y-transform of the mixed nonlinear field
    if constexpr (PF) {
        std::conditional_t<WSF, TwWs<LC, T>, TwRegs<LC, T>> tw;
        if constexpr (WSF) load_tw_ws(tw, j, a.tw);
        else load_tw_regs<LC, 0>(tw, j, a.tw);
        if constexpr (pair_layout<T, LC, NT>()) {
            // J in 2 x 2 blocks: jblock_elem(kxi, ny, y), y = j + s TPL (TPL
            // even), is a column base, the lane's offset j + (j & ~1), and
            // 2 TPL per slot; [kx][y] on rectangular grids, whose row stage
            // has another length and writes that
            const bool jb = a.jblocks != 0;
            const unsigned jb0 = jb ? __umul24((unsigned)(kxi & ~1), (unsigned)G.ny) +
                                          2u * (unsigned)(kxi & 1) + (unsigned)(j + (j & ~1))
                                    : col_elem(kxi, G.ny, j);
            const unsigned jbs = jb ? 2u * (unsigned)TPL : (unsigned)TPL;
#pragma unroll
            for (int s = 0; s < P; ++s)
                v[s] = has_data ? *at32(nl, jb0 + (unsigned)s * jbs) : zero;
        } else if constexpr (rowpair_layout<T, LC, NT>()) {
            // J's last reader, whole columns: non-temporal loads, which leave
            // the caches to the mixed fields written next (FP64 4096^2:
            // k_col 177.1 -> 174.0 us); every column of the grid is kept
            // (COL_STAGE launches nkx_keep of them), so the loads are in bounds
            typedef T t2 __attribute__((ext_vector_type(2)));
#pragma unroll
            for (int s = 0; s < P; ++s) {
                const t2 q = __builtin_nontemporal_load(
                    reinterpret_cast<const t2*>(nl + mbase + j + s * TPL));
                v[s] = has_data ? mk(q.x, q.y) : zero;
            }
        } else {
#pragma unroll
            for (int s = 0; s < P; ++s) v[s] = has_data ? nl[mbase + j + s * TPL] : zero;
        }
        // the accumulator only from stage 1 on, where the update reads it (a
        // uniform branch around whole loads, which a select would split)
        const bool with_acc = a.stage > 0;
#pragma unroll
        for (int s = 0; s < P; ++s) {
            const int kind = slot_kind(s, LC, Band<LC>::kym);
            const int jy = j + s * TPL;
            if (kind == 0 || !has_data) continue;
            const bool pos = kind == 1 || (kind == 3 && jy <= kym);
            if (kind == 3 && !pos && jy < Ll - kym) continue;
            const size_t ci = (size_t)kxi * ncy + (pos ? jy : jy - (Ll - ncy));
            pw0[s] = state[ci];
            pacc[s] = zero;
            if (with_acc) pacc[s] = acc[ci];
        }
        if constexpr (EARLY) {
            if (a.stage == 0 && ph.adaptive) pick_dt();
#pragma unroll
            for (int s = 0; s < P; ++s) {
                if (slot_kind(s, LC, Band<LC>::kym) == 0) continue;
                const T ky = T(col_band<LC>(G, j + s * TPL)) * T(2.0 * kPi / G.Ly);
                const T k2 = kx * kx + ky * ky;
                const T L = -(k2 * T(ph.inv_Re) + T(ph.drag) + hv_weight_t<T>(ph, k2));
                if constexpr (SCHEME == 0) {
                    el[s] = L;
                    es[s] = sfd_weight_t<T>(ph, k2);
                } else {
                    es[s] = expm1_t(L * (T(0.5) * T(dt)));
                    el[s] = es[s] * (T(2) + es[s]);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (WSF) {
            cx<T>(*const vv[1])[P] = {&v};
            cx<T>* const r1[1] = {lds};
            cx<T>* const t1[1] = {lds2};
            ws_c<-1, 1, WS>(vv, r1, t1, j, tw);
        } else {
            fft_any<-1, LC>(v, lds, j, g, tw);
        }
        // nothing that uses the values loaded above may be scheduled into
        // the transform (it would wait there for them)
        __builtin_amdgcn_sched_barrier(0);
    } else if constexpr (MODE == COL_STAGE || MODE == COL_FWD) {
        if (MODE == COL_FWD && a.jblocks) {
#pragma unroll
            for (int s = 0; s < P; ++s)
                v[s] = has_data ? *at32(nl, jblock_elem(kxi, G.ny, j + s * TPL)) : zero;
        } else {
#pragma unroll
            for (int s = 0; s < P; ++s) v[s] = has_data ? nl[mbase + j + s * TPL] : zero;
        }
        fft_any<-1, LC>(v, lds, j, g, a.tw);
    }

    if constexpr (MODE == COL_FWD) {
        // spectral_transforms.c:13-21: x 1/(nx ny), then zero outside the mask
        const T norm = T(a.fwd_scale / ((double)G.nx * (double)G.ny));
#pragma unroll
        for (int s = 0; s < P; ++s) {
            const int jy = j + s * TPL;
            const bool k = has_data && kept(G, kxi, jy);
            cx<T> r = k ? norm * v[s] : zero;
            if (a.out_c) {  // compact layout of the kept modes
                if (k) a.out_c[mb * a.bc + (size_t)kxi * G.nky_keep + compact_y(G, jy)] = r;
            } else if (active) {
                st_ref(a.out_ref, (size_t)jy * G.nkx + kxi, r);
            }
        }
        return;
    }

    // ---- spectral state of this column after the stage (or as is)
    if constexpr (MODE == COL_STAGE && !EARLY) {
        if (a.stage == 0 && ph.adaptive) {
            u2 = __longlong_as_double((long long)sc->umax2_bits);
            pick_dt();
        } else {
            dt = sc->dt;
        }
    }
    const T h = T(dt);
    const T norm = T(1.0 / ((double)G.nx * (double)G.ny));
    const double sfd_alpha = (ph.sfd_tau > 0.0) ? fmin(fmax(dt / ph.sfd_tau, 0.0), 1.0) : 0.0;
    const T sqh = T(sqrt(dt));
    // error controller, last stage: this thread's sum w |y4 - y2|^2 and
    // sum w |y4|^2 (FP64)
    double esum = 0.0, ssum = 0.0;

#pragma unroll
    for (int s = 0; s < P; ++s) {
        const int kind = LC > 0 ? slot_kind(s, LC, Band<LC>::kym) : 3;
        const int jy = j + s * TPL;
        w[s] = zero;
        if (kind == 0 || !has_data) continue;
        const bool pos = kind == 1 || (kind == 3 && jy <= kym);
        if (kind == 3 && !pos && jy < Ll - kym) continue;
        const size_t ci = (size_t)kxi * ncy + (pos ? jy : jy - (Ll - ncy));
        const T ky = T(pos ? jy : jy - Ll) * T(2.0 * kPi / G.Ly);
        if constexpr (MODE == COL_PRIME) {
            w[s] = state[ci];
            continue;
        }
        if constexpr (MODE == COL_INV) {
            w[s] = a.in_ref ? ld_ref<T>(a.in0_ref, (size_t)jy * G.nkx + kxi) : a.in0[mb * a.bc + ci];
            continue;
        }
        if constexpr (ERR && MODE == COL_STAGE) {
            if (redo) {  // the state of the last accepted step comes back
                w[s] = prev[ci];
                state[ci] = w[s];
                continue;
            }
        }
        // COL_STAGE: N = -norm * FFT(J) (spectral_core.c:106-111)
        cx<T> N = (-norm) * v[s];
        if (src) N = N + src[ci];  // learned subgrid tendency, frozen over the step
        const cx<T> w0 = PF ? pw0[s] : state[ci];
        if constexpr (ERR) {
            if (a.stage == 0) prev[ci] = w0;
        }
        const T k2 = kx * kx + ky * ky;
        cx<T> wn;
        if constexpr (SCHEME == 0) {
            // classic RK4 (spectral_time_integration.c:50-100) with
            // hyperviscosity_apply (hyperviscosity.c:104-150) and drag
            const cx<T> ws = (a.stage == 0) ? w0 : stagebuf[ci];
            const T lin = EARLY ? el[s] : -(k2 * T(ph.inv_Re) + T(ph.drag) + hv_weight_t<T>(ph, k2));
            cx<T> ks = N + lin * ws;
            const T sw = EARLY ? es[s] : sfd_weight_t<T>(ph, k2);
            if (sw > T(0)) ks = ks - sw * (ws - sfd[ci]);
            if (a.stage == 0) {
                acc[ci] = w0 + (h / T(6)) * ks;
                wn = w0 + (T(0.5) * h) * ks;
            } else if (a.stage == 1) {
                acc[ci] = (PF ? pacc[s] : acc[ci]) + (h / T(3)) * ks;
                wn = w0 + (T(0.5) * h) * ks;
                if constexpr (ERR) ymid[ci] = w0 + h * ks;  // explicit midpoint solution
            } else if (a.stage == 2) {
                acc[ci] = (PF ? pacc[s] : acc[ci]) + (h / T(3)) * ks;
                wn = w0 + h * ks;
            } else {
                wn = (PF ? pacc[s] : acc[ci]) + (h / T(6)) * ks;
                if (ph.sfd_on && ph.sfd_tau > 0.0) {  // hyperviscosity.c:152-178
                    const T al = T(sfd_alpha);
                    sfd[ci] = (T(1) - al) * sfd[ci] + al * wn;
                }
            }
            if (a.stage < 3) stagebuf[ci] = wn;
        } else {
            // integrating factor, L = -(k^2/Re + w_hv + mu).  The factors are
            // carried as E - 1 (expm1): near k = 0 the per-step decay L h is
            // ~1e-5, which 1 + (E - 1) keeps to full relative precision while
            // E itself, rounded to FP32, would lose ~0.3 % of it every step.
            const T L = -(k2 * T(ph.inv_Re) + T(ph.drag) + hv_weight_t<T>(ph, k2));
            // E2 - 1, E2 = exp(L h / 2), and E - 1, E = E2^2
            const T e2 = EARLY ? es[s] : expm1_t(L * (T(0.5) * h));
            const T e1 = EARLY ? el[s] : e2 * (T(2) + e2);
            if (a.stage == 0) {
                acc[ci] = grow(w0, e1) + (h / T(6)) * grow(N, e1);
                wn = grow(w0 + (T(0.5) * h) * N, e2);
            } else if (a.stage == 1) {
                acc[ci] = (PF ? pacc[s] : acc[ci]) + (h / T(3)) * grow(N, e2);
                wn = grow(w0, e2) + (T(0.5) * h) * N;
                // Lawson midpoint solution E w0 + h E2 N(b)
                if constexpr (ERR) ymid[ci] = grow(w0, e1) + h * grow(N, e2);
            } else if (a.stage == 2) {
                acc[ci] = (PF ? pacc[s] : acc[ci]) + (h / T(3)) * grow(N, e2);
                wn = grow(w0, e1) + h * grow(N, e2);
            } else {
                wn = (PF ? pacc[s] : acc[ci]) + (h / T(6)) * N;
            }
        }
        if (a.stage == 3) {
            if constexpr (ERR) {  // embedded estimate, before the forcing kick
                const cx<T> e = wn - ymid[ci];
                const double wt = kxi == 0 ? 1.0 : 2.0;
                esum += wt * ((double)e.x * (double)e.x + (double)e.y * (double)e.y);
                ssum += wt * ((double)wn.x * (double)wn.x + (double)wn.y * (double)wn.y);
            }
            if (ph.force_on && kxi < ph.fbx) {
                const int b = band_of(G, jy);
                if (b >= -ph.fby && b <= ph.fby)
                    wn = wn + sqh * fbox[kxi * (2 * ph.fby + 1) + (b + ph.fby)];
            }
            state[ci] = wn;
        }
        w[s] = wn;
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        if (MODE == COL_STAGE && a.stage == 3) {
            sc->t += dt;
            sc->umax2_bits = 0ull;
        } else if (MODE == COL_STAGE && redo) {
            sc->umax2_bits = 0ull;  // stage 3 does not run on a restoring step
        } else if (MODE == COL_PRIME) {
            sc->umax2_bits = 0ull;
            sc->pending = 0;  // a new state: nothing waits to be judged
            sc->redo = 0;
        }
    }
    if constexpr (ERR && MODE == COL_STAGE) {
        if (a.stage == 3) {
            // workgroup sums in a fixed order (wave butterflies, then the
            // waves in index order): the judge adds the partials in index
            // order, so the decision is reproducible bit for bit
            __shared__ double ered[2 * (NT / 64)];
            esum = wave_sum(esum);
            ssum = wave_sum(ssum);
            const int wv = threadIdx.x >> 6;
            if ((threadIdx.x & 63) == 0) {
                ered[2 * wv] = esum;
                ered[2 * wv + 1] = ssum;
            }
            __syncthreads();
            if (threadIdx.x == 0) {
                double e = 0.0, z = 0.0;
                for (int i = 0; i < NT / 64; ++i) {
                    e += ered[2 * i];
                    z += ered[2 * i + 1];
                }
                double* part = a.errpart + mb * a.bp + 2 * (size_t)blockIdx.x;
                part[0] = e;
                part[1] = z;
                if (blockIdx.x == 0) {
                    sc->pending = 1;
                    sc->errparts = (int)gridDim.x;
                }
            }
        }
    }

    // ---- derivative spectra and inverse y-transforms
    const T kys = T(2.0 * kPi / G.Ly);
    if constexpr (MODE == COL_INV) {
        for (int f = 0; f < a.nout; ++f) {
#pragma unroll
            for (int s = 0; s < P; ++s) {
                const int jy = j + s * TPL;
                const T ky = T(col_band<LC>(G, jy)) * kys;
                const T k2 = kx * kx + ky * ky;
                cx<T> b = zero;
                if (a.in1_ref && has_data && kept(G, kxi, jy))
                    b = ld_ref<T>(a.in1_ref, (size_t)jy * G.nkx + kxi);
                v[s] = apply_op(a.ops[f], w[s], b, kx, ky, k2);
            }
            fft_any<+1, LC>(v, lds, j, g, a.tw);
            if (has_data) {
                cx<T>* out = a.mixed[f] + mixed_off;
#pragma unroll
                for (int s = 0; s < P; ++s) out[mbase + j + s * TPL] = v[s];
            }
        }
    } else if constexpr (paired_lines<T, LC, NT>()) {
        // outputs 0 psi_x, 1 psi_y, 2 omega_x, 3 omega_y (spectral_core.c:62-99),
        // transformed two at a time: (omega_y, omega_x), then w becomes
        // psi_hat = -w/k^2 in place and (psi_y, psi_x)
        cx<T> v2[P];
        if constexpr (LC >= 64) {
            // Unrolled: the twiddles of the second pair go into
            // registers before the first pair's stores are issued, so that
            // its transform does not wait for those stores to retire (the
            // vector-memory counter retires stores and loads in order).
#pragma unroll
            for (int s = 0; s < P; ++s) {
                const T ky = T(col_band<LC>(G, j + s * TPL)) * kys;
                v[s] = mul_i(w[s], ky);
                v2[s] = mul_i(w[s], kx);
            }
            // FP32 2048 to 8192 (pair layout): wave-split transforms, standard
            // pattern in and out (ws_c), transposing back in the same regions
            constexpr bool WSC = pair_layout<T, LC, NT>();
            std::conditional_t<WSC, TwWs<LC, T>, TwRegs<LC, T>> tw;
            cx<T>(*const vv[2])[P] = {&v, &v2};
            cx<T>* const rr[2] = {lds, lds2};
            if constexpr (WSC) {
                load_tw_ws(tw, j, a.tw);
                renew_tw(tw);
                __syncthreads();  // the forward transform's last reads are done
                ws_c<+1, 2>(vv, rr, rr, j, tw);  // omega_y, omega_x
            } else {
                line_fft2_c<+1, LC>(v, v2, lds, lds2, j, a.tw);  // omega_y, omega_x
                load_tw_regs<LC, 0>(tw, j, a.tw);
            }
            if (has_data) {
                if constexpr (pair_layout<T, LC, NT>()) {
                    if (a.pairs) {  // (omega_x, omega_y)
                        cx<T>* pb = a.mixed[2] + 2 * mixed_off;
                        if constexpr (pairtile_layout<T, LC, NT>()) {
                            store_pair_tiles<LC>(pb, kxi, (G.nkx_keep + 1) & ~1, j, v2, v);
                        } else {
#pragma unroll
                            for (int s = 0; s < P; ++s)
                                store_pair(pb, mbase + j + s * TPL, v2[s], v[s]);
                        }
                    }
                }
                if (!(pair_layout<T, LC, NT>() && a.pairs)) {
                    cx<T>* o1 = a.mixed[3] + mixed_off;
                    cx<T>* o2 = a.mixed[2] + mixed_off;
#pragma unroll
                    for (int s = 0; s < P; ++s) {
                        o1[mbase + j + s * TPL] = v[s];
                        o2[mbase + j + s * TPL] = v2[s];
                    }
                }
            }
#pragma unroll
            for (int s = 0; s < P; ++s) {
                const T ky = T(col_band<LC>(G, j + s * TPL)) * kys;
                const T k2 = kx * kx + ky * ky;
                const cx<T> psi = k2 > T(1e-12) ? neg_inv_k2(k2) * w[s] : zero;
                v[s] = mul_i(psi, ky);
                v2[s] = mul_i(psi, kx);
            }
            if constexpr (WSC) {
                __syncthreads();  // others may still read the transposed first pair
                renew_tw(tw);
                ws_c<+1, 2>(vv, rr, rr, j, tw);  // psi_y, psi_x
            } else {
                line_fft2_c<+1, LC>(v, v2, lds, lds2, j, tw);  // psi_y, psi_x
            }
            if (has_data) {
                if constexpr (pair_layout<T, LC, NT>()) {
                    if (a.pairs) {  // (psi_x, psi_y)
                        cx<T>* pb = a.mixed[0] + 2 * mixed_off;
                        if constexpr (pairtile_layout<T, LC, NT>()) {
                            store_pair_tiles<LC>(pb, kxi, (G.nkx_keep + 1) & ~1, j, v2, v);
                        } else {
#pragma unroll
                            for (int s = 0; s < P; ++s)
                                store_pair(pb, mbase + j + s * TPL, v2[s], v[s]);
                        }
                    }
                }
                if (!(pair_layout<T, LC, NT>() && a.pairs)) {
                    cx<T>* o1 = a.mixed[1] + mixed_off;
                    cx<T>* o2 = a.mixed[0] + mixed_off;
#pragma unroll
                    for (int s = 0; s < P; ++s) {
                        o1[mbase + j + s * TPL] = v[s];
                        o2[mbase + j + s * TPL] = v2[s];
                    }
                }
            }
            return;
        }
#pragma unroll 1
        for (int f = 3; f >= 1; f -= 2) {
            if (f == 1) {
#pragma unroll
                for (int s = 0; s < P; ++s) {
                    const T ky = T(col_band<LC>(G, j + s * TPL)) * kys;
                    const T k2 = kx * kx + ky * ky;
                    w[s] = k2 > T(1e-12) ? neg_inv_k2(k2) * w[s] : zero;
                }
            }
#pragma unroll
            for (int s = 0; s < P; ++s) {
                const T ky = T(col_band<LC>(G, j + s * TPL)) * kys;
                v[s] = mul_i(w[s], ky);
                v2[s] = mul_i(w[s], kx);
            }
            line_fft2_c<+1, LC>(v, v2, lds, lds2, j, a.tw);
            if (has_data) {
                cx<T>* o1 = a.mixed[f] + mixed_off;
                cx<T>* o2 = a.mixed[f - 1] + mixed_off;
#pragma unroll
                for (int s = 0; s < P; ++s) {
                    o1[mbase + j + s * TPL] = v[s];
                    o2[mbase + j + s * TPL] = v2[s];
                }
            }
        }
    } else if constexpr (WS) {
        // FP64 columns of 2048 and 4096: the four outputs one at a time through ws_c
        // (spectral_core.c:62-99), swizzled rows in lds, the transposing
        // exchange in lds2: two barriers per transform
        TwWs<LC, T> tw;
        load_tw_ws(tw, j, a.tw);
        cx<T>(*const vv[1])[P] = {&v};
        cx<T>* const r1[1] = {lds};
        cx<T>* const t1[1] = {lds2};
        // the outputs in row-pair tiles or per field ([kx][y])
        const SlotElems se = col_slots<LC>(kxi, j, G.ny, (G.nkx_keep + 1) & ~1, a.pairs != 0);
#pragma unroll 1
        for (int f = 3; f >= 0; --f) {
            if (f == 1) {
#pragma unroll
                for (int s = 0; s < P; ++s) {
                    const T ky = T(col_band<LC>(G, j + s * TPL)) * kys;
                    const T k2 = kx * kx + ky * ky;
                    w[s] = k2 > T(1e-12) ? neg_inv_k2(k2) * w[s] : zero;
                }
            }
#pragma unroll
            for (int s = 0; s < P; ++s) {
                const T ky = T(col_band<LC>(G, j + s * TPL)) * kys;
                v[s] = mul_i(w[s], (f & 1) ? ky : kx);
            }
            ws_c<+1, 1, true>(vv, r1, t1, j, tw);
            if (has_data) {
                cx<T>* out = a.mixed[f] + mixed_off;
#pragma unroll
                for (int s = 0; s < P; ++s) *at32(out, se.e0 + (unsigned)s * se.es) = v[s];
            }
        }
    } else {
        // outputs 0 psi_x, 1 psi_y, 2 omega_x, 3 omega_y (spectral_core.c:62-99);
        // the omega-based pair first, then w becomes psi_hat = -w/k^2 in place.
        // FP64 stage columns take their twiddles from registers, so that no
        // transform waits for the previous field's stores to retire.
        constexpr bool REG = PF && sizeof(T) == 8;
        typename TwSource<REG, (LC > 0 ? LC : 16), T>::type tws;
        if constexpr (REG) load_tw_regs<LC, 0>(tws, j, a.tw);
        else tws = a.tw;
#pragma unroll 1
        for (int f = 3; f >= 0; --f) {
            if (f == 1) {
#pragma unroll
                for (int s = 0; s < P; ++s) {
                    const T ky = T(col_band<LC>(G, j + s * TPL)) * kys;
                    const T k2 = kx * kx + ky * ky;
                    w[s] = k2 > T(1e-12) ? neg_inv_k2(k2) * w[s] : zero;
                }
            }
#pragma unroll
            for (int s = 0; s < P; ++s) {
                const T ky = T(col_band<LC>(G, j + s * TPL)) * kys;
                v[s] = mul_i(w[s], (f & 1) ? ky : kx);
            }
            fft_any<+1, LC>(v, lds, j, g, tws);
            if (has_data) {
                cx<T>* out = a.mixed[f] + mixed_off;
#pragma unroll
                for (int s = 0; s < P; ++s) out[mbase + j + s * TPL] = v[s];
            }
        }
    }
}

// --------------------------------------------------------------- row side

enum RowMode { ROW_STAGE = 0, ROW_C2R = 1, ROW_R2C = 2 };

template <typename T>
struct RowArgs {
    Geo geo;
    int mode;
    int nfields;           // ROW_C2R: number of mixed fields to transform
    int track_umax;        // ROW_STAGE: fold max(u^2+v^2) into sc->umax2_bits
    const cx<T>* tw;       // twiddles for length nx
    const cx<T>* mixed[4];
    cx<T>* nl;             // ROW_STAGE / ROW_R2C output (mixed)
    double* out_ref[4];    // ROW_C2R outputs (FP64 [ny][nx]) if non-null
    T* out[4];             // ROW_C2R outputs (T [ny][nx]) otherwise
    int minus1;            // ROW_C2R: out_ref[1] negated
    const double* in_ref;  // ROW_R2C input (FP64 [ny][nx])
    const T* in_t;         // ROW_R2C input at the working precision (instead of in_ref)
    DevScalars* sc;
    size_t bm;             // batches: mixed-field stride of member blockIdx.y
    size_t br;             // batches: physical-field stride (ROW_C2R out, ROW_R2C in_t)
    int nbat;              // members along grid y for the transform modes (0 = 1)
    int stagger_lo;        // ROW_STAGE: first-round workgroups [lo, hi) start late
    int stagger_hi;
    unsigned short* out_bf16;  // ROW_C2R: field 0 as bf16, times out_bf16_scale (if non-null)
    float out_bf16_scale;
    int pairs;                 // ROW_STAGE: mixed fields in the stage layout (stage_layout)
    int jblocks;               // ROW_STAGE: write J in 2 x 2 blocks (square pair-layout grids)
    int skip_on_redo;          // ROW_STAGE, ERR: idle when the step restores a rejected one
    // ROW_STAGE, FORCE: the step's forcing draw, made by workgroup 0 beside the
    // row pairs of the others (stage 1: dt is known since stage 0, the box is
    // read in stage 3)
    ForceArgs force;
};

// Build the Hermitian extension of Z = A + iB in LDS for one row y from
// the kept mixed columns (c2r convention: imaginary parts of the kx = 0
// values are ignored, as FFTW's c2r does), then read the standard pattern.
template <int LC, typename T>
__device__ __forceinline__ void build_row_pair(cx<T> (&v)[P], cx<T>* lds, int j, const Line& g,
                                               const Geo& G, const cx<T>* A, const cx<T>* B,
                                               int y, bool active) {
    const int TPL = LC > 0 ? LC / P : g.TPL;
    const int Ll = LC > 0 ? LC : g.L;
    const cx<T> zero = mk(T(0), T(0));
    __syncthreads();
#pragma unroll
    for (int s = 0; s < P; ++s) {
        const int k = j + s * TPL;
        if (k <= G.kxmax) {
            cx<T> a = zero, b = zero;
            if (active) {
                a = A ? A[(size_t)k * G.ny + y] : zero;
                b = B ? B[(size_t)k * G.ny + y] : zero;
            }
            if (k == 0) {
                a.y = T(0);
                b.y = T(0);
            }
            lds[pad(k)] = mk(a.x - b.y, a.y + b.x);
            if (k > 0) lds[pad(Ll - k)] = mk(a.x + b.y, b.x - a.y);
        } else if (k < Ll - G.kxmax) {
            lds[pad(k)] = zero;
        }
    }
    __syncthreads();
    if constexpr (LC > 0) lds_read_c<LC>(v, lds, j);
    else lds_read_std(v, lds, j, TPL);
}

// Same Hermitian extension for Z = F(., y) + i F(., y+1): the two rows of one
// field, fetched with a single 2-element load per column (the rows are
// adjacent in the [kx][y] mixed layout).
template <int LC, typename T>
__device__ __forceinline__ void stage_two_rows(cx<T>* lds, int j, const Line& g, const Geo& G,
                                               const cx<T>* F, int y, bool active) {
    const int TPL = LC > 0 ? LC / P : g.TPL;
    const int Ll = LC > 0 ? LC : g.L;
    const int kxm = LC > 0 ? Band<LC>::kxm : G.kxmax;
    const cx<T> zero = mk(T(0), T(0));
#pragma unroll
    for (int s = 0; s < P; ++s) {
        const int kind = LC > 0 ? slot_kind(s, LC, Band<LC>::kxm) : 3;
        const int k = j + s * TPL;
        if (kind == 2) continue;  // written by the owner of Ll - k
        if (kind == 0) {
            lds[pad(k)] = zero;
            continue;
        }
        if (kind == 1 || k <= kxm) {
            cx<T> a = zero, b = zero;
            if (active) {
                const cx<T>* src = F + (size_t)k * G.ny + y;
                a = src[0];
                b = src[1];
            }
            if (k == 0) {
                a.y = T(0);
                b.y = T(0);
            }
            lds[pad(k)] = mk(a.x - b.y, a.y + b.x);
            if (k > 0) lds[pad(Ll - k)] = mk(a.x + b.y, b.x - a.y);
        } else if (k < Ll - kxm) {
            lds[pad(k)] = zero;
        }
    }
}

template <int LC, typename T>
__device__ __forceinline__ void build_two_rows(cx<T> (&v)[P], cx<T>* lds, int j, const Line& g,
                                               const Geo& G, const cx<T>* F, int y,
                                               bool active) {
    __syncthreads();
    stage_two_rows<LC>(lds, j, g, G, F, y, active);
    __syncthreads();
    if constexpr (LC > 0) lds_read_c<LC>(v, lds, j);
    else lds_read_std(v, lds, j, g.TPL);
}

// both fields F1, F2 for rows y, y+1 into two line regions
template <int LC, typename T>
__device__ __forceinline__ void build_two_rows2(cx<T> (&v1)[P], cx<T> (&v2)[P], cx<T>* lds1,
                                                cx<T>* lds2, int j, const Line& g, const Geo& G,
                                                const cx<T>* F1, const cx<T>* F2, int y,
                                                bool active) {
    __syncthreads();
    stage_two_rows<LC>(lds1, j, g, G, F1, y, active);
    stage_two_rows<LC>(lds2, j, g, G, F2, y, active);
    __syncthreads();
    lds_read_c<LC>(v1, lds1, j);
    lds_read_c<LC>(v2, lds2, j);
}


// Forward x-transform of two real rows packed as v = ra + i rb, then
// separation of the two half spectra and store of the kept columns into
// the mixed layout at rows y and y+1.
template <int LC, typename T, typename TW, bool JB = false>
__device__ __forceinline__ void fwd_rows_store(cx<T> (&v)[P], cx<T>* lds, int j, const Line& g,
                                               const Geo& G, const TW& tw, cx<T>* out, int y,
                                               bool active, int jblocks = 0) {
    const int TPL = LC > 0 ? LC / P : g.TPL;
    const int Ll = LC > 0 ? LC : g.L;
    const int kxm = LC > 0 ? Band<LC>::kxm : G.kxmax;
    fft_any<-1, LC>(v, lds, j, g, tw);
    // after a wave-split transform the line goes unpadded (only unit-stride
    // accesses follow)
    constexpr bool PADL = !std::is_same<TW, TwWs<(LC > 0 ? LC : 4096), T>>::value;
    auto at = [](int i) { return PADL ? pad(i) : i; };
    if constexpr (LC > 0) {
        // the separation below reads kept columns k and their partners
        // Ll - k only, never a slot inside the dealiased band (kind 0)
        if constexpr (LC / P % 16 == 0) {
            cx<T>* b = lds + at(j);
#pragma unroll
            for (int s = 0; s < P; ++s)
                if (slot_kind(s, LC, Band<LC>::kxm) != 0) b[PADL ? padc(s * TPL) : s * TPL] = v[s];
        } else {
            lds_write_c<LC>(v, lds, j);
        }
    } else {
        lds_write_std(v, lds, j, TPL);
    }
    __syncthreads();
#pragma unroll
    for (int s = 0; s < P; ++s) {
        const int kind = LC > 0 ? slot_kind(s, LC, Band<LC>::kxm) : 3;
        if (kind == 0 || kind == 2) continue;
        const int k = j + s * TPL;
        if ((kind == 1 || k <= kxm) && active) {
            const cx<T> zk = lds[at(k)];
            const cx<T> zm = lds[at((Ll - k) & (Ll - 1))];
            const cx<T> ja = mk(T(0.5) * (zk.x + zm.x), T(0.5) * (zk.y - zm.y));
            const cx<T> jb = mk(T(0.5) * (zk.y + zm.y), T(0.5) * (zm.x - zk.x));
            if constexpr (JB) {
                // jblock_elem(k, ny, y) for even y: (k & ~1) ny + 2 (k & 1) + 2 y;
                // [kx][y] where the column stage has another length
                static_assert(sizeof(T) == 4, "J blocks are an FP32 layout");
                const unsigned e = jblocks ? __umul24((unsigned)(k & ~1), (unsigned)G.ny) +
                                                 2u * (unsigned)((k & 1) + y)
                                           : col_elem(k, G.ny, y);
                *reinterpret_cast<float4*>(at32(out, e)) = float4{ja.x, ja.y, jb.x, jb.y};
            } else {
                cx<T>* dst = at32(out, col_elem(k, G.ny, y));
                dst[0] = ja;
                dst[1] = jb;
            }
        }
    }
}

// Standard-pattern read of a line staged with SKIP0: its kind-0 slots are
// zero in registers, known to the compiler, so the first butterflies fold
// them away, and they cost no LDS read.
template <int LC, bool PAD = true, typename T>
__device__ __forceinline__ void lds_read_kept(cx<T> (&v)[P], const cx<T>* lds, int j) {
    constexpr int TPL = LC / P;
    static_assert(TPL % 16 == 0, "compile-time offsets need TPL % 16 == 0");
    const cx<T>* b = lds + (PAD ? pad(j) : j);
#pragma unroll
    for (int s = 0; s < P; ++s)
        v[s] = slot_kind(s, LC, Band<LC>::kxm) == 0 ? mk(T(0), T(0))
                                                    : b[PAD ? padc(s * TPL) : s * TPL];
}

template <int LC, bool KEPT, typename T>
__device__ __forceinline__ void lds_read_any(cx<T> (&v)[P], const cx<T>* lds, int j) {
    if constexpr (KEPT) lds_read_kept<LC>(v, lds, j);
    else lds_read_c<LC>(v, lds, j);
}

// Kept columns of one field at rows y, y + 1 (the two rows of one packed
// line) for this thread's slots, held in registers from the gather to the
// LDS staging.  Zero for an inactive line.
template <typename T>
struct RowPairRegs {
    cx<T> a[P], b[P];
};

template <int LC, typename T>
__device__ __forceinline__ void gather_two_rows(RowPairRegs<T>& r, int j, const Geo& G,
                                                const cx<T>* F, int y, bool active) {
    constexpr int kxm = Band<LC>::kxm;
#pragma unroll
    for (int s = 0; s < P; ++s) {
        const int kind = slot_kind(s, LC, kxm);
        const int k = j + s * (LC / P);
        if (kind == 1 || (kind == 3 && k <= kxm)) {
            if (active) {
                const cx<T>* src = at32(F, col_elem(k, G.ny, y));
                r.a[s] = src[0];
                r.b[s] = src[1];
            } else {
                r.a[s] = mk(T(0), T(0));
                r.b[s] = mk(T(0), T(0));
            }
        }
    }
}

// The same from slot elements (row_slots), rows y and y + 1 adjacent: the per-field
// layout, or row-pair tiles.  In tiles no other row pair reads these bytes, and the
// stage reads each field once, so they need not displace from L2 and the MALL the J
// values and compact fields that k_col reads next: non-temporal loads there (FP64
// 4096^2 step 1.368 -> 1.346 ms: k_row +3.7 us, k_col -9.7 us).  The per-field layout
// (rectangles, large batches) shares each line among four row pairs: ordinary loads
// (non-temporal ones took k_row at 2048 x 4096 from 84 to 144 us).  The FP32 pair
// layout keeps ordinary loads as well (gather_pair_rows): 76 against 137 us.
template <int LC, bool TILES, typename T>
__device__ __forceinline__ void gather_two_rows(RowPairRegs<T>& r, int j, const cx<T>* F,
                                                SlotElems se) {
    typedef T t2 __attribute__((ext_vector_type(2)));
    constexpr int kxm = Band<LC>::kxm;
    auto load = [](const t2* p) { return TILES ? __builtin_nontemporal_load(p) : *p; };
#pragma unroll
    for (int s = 0; s < P; ++s) {
        const int kind = slot_kind(s, LC, kxm);
        const int k = j + s * (LC / P);
        if (kind == 1 || (kind == 3 && k <= kxm)) {
            const t2* src = reinterpret_cast<const t2*>(at32(F, se.e0 + (unsigned)s * se.es));
            const t2 a = load(src), b = load(src + 1);
            r.a[s] = mk(a.x, a.y);
            r.b[s] = mk(b.x, b.y);
        }
    }
}

// Both fields of a pair-layout buffer at rows y, y + 1 (f0: first, f1:
// second): two 16-byte loads per slot from one 64-byte line.
template <int LC>
__device__ __forceinline__ void gather_pair_rows(RowPairRegs<float>& f0, RowPairRegs<float>& f1,
                                                 int j, const Geo& G, const cx<float>* B, int y,
                                                 bool active) {
    constexpr int kxm = Band<LC>::kxm;
#pragma unroll
    for (int s = 0; s < P; ++s) {
        const int kind = slot_kind(s, LC, kxm);
        const int k = j + s * (LC / P);
        if (kind == 1 || (kind == 3 && k <= kxm)) {
            if (active) {
                const float4* src = reinterpret_cast<const float4*>(at32(B, 2 * col_elem(k, G.ny, y)));
                const float4 r0 = src[0], r1 = src[1];  // rows y, y + 1
                f0.a[s] = mk(r0.x, r0.y);
                f1.a[s] = mk(r0.z, r0.w);
                f0.b[s] = mk(r1.x, r1.y);
                f1.b[s] = mk(r1.z, r1.w);
            } else {
                f0.a[s] = f1.a[s] = f0.b[s] = f1.b[s] = mk(0.f, 0.f);
            }
        }
    }
}

// The same from row-pair tiles of the pair buffers: 32 contiguous bytes per
// column, read by this row pair only (non-temporal, as in the FP64 tiles).
template <int LC>
__device__ __forceinline__ void gather_pair_tiles(RowPairRegs<float>& f0, RowPairRegs<float>& f1,
                                                  int j, const cx<float>* B, int K, int y) {
    typedef float f4 __attribute__((ext_vector_type(4)));
    constexpr int kxm = Band<LC>::kxm;
    const unsigned e0 = pairtile_elem(j, K, y);
#pragma unroll
    for (int s = 0; s < P; ++s) {
        const int kind = slot_kind(s, LC, kxm);
        const int k = j + s * (LC / P);
        if (kind == 1 || (kind == 3 && k <= kxm)) {
            const f4* src = reinterpret_cast<const f4*>(at32(B, e0 + (unsigned)(4 * s * (LC / P))));
            const f4 r0 = __builtin_nontemporal_load(src), r1 = __builtin_nontemporal_load(src + 1);
            f0.a[s] = mk(r0.x, r0.y);
            f1.a[s] = mk(r0.z, r0.w);
            f0.b[s] = mk(r1.x, r1.y);
            f1.b[s] = mk(r1.z, r1.w);
        }
    }
}

// The LDS image of stage_two_rows, from gathered registers.  SKIP0: the
// slots that lie inside the dealiased band for every thread (kind 0) are
// left unwritten, for a reader that takes them as zero (lds_read_kept).
// PAD: the line's one-in-sixteen padding, which the Stockham passes need;
// a line read back only in the standard pattern goes unpadded (every access
// to it is at unit stride).
template <int LC, bool SKIP0 = false, bool PAD = true, typename T>
__device__ __forceinline__ void stage_two_rows_regs(cx<T>* lds, int j, const RowPairRegs<T>& r) {
    constexpr int TPL = LC / P, kxm = Band<LC>::kxm;
    const cx<T> zero = mk(T(0), T(0));
    auto at = [](int i) { return PAD ? pad(i) : i; };
#pragma unroll
    for (int s = 0; s < P; ++s) {
        const int kind = slot_kind(s, LC, kxm);
        const int k = j + s * TPL;
        if (kind == 2) continue;  // written by the owner of LC - k
        if (kind == 0) {
            if (!SKIP0) lds[at(k)] = zero;
            continue;
        }
        if (kind == 1 || k <= kxm) {
            cx<T> a = r.a[s], b = r.b[s];
            if (k == 0) {
                a.y = T(0);
                b.y = T(0);
            }
            lds[at(k)] = mk(a.x - b.y, a.y + b.x);
            if (k > 0) lds[at(LC - k)] = mk(a.x + b.y, b.x - a.y);
        } else if (k < LC - kxm) {
            lds[at(k)] = zero;
        }
    }
}

// both fields of a pair buffer, in row-pair tiles (TILES) or pair by pair
template <int LC, bool TILES>
__device__ __forceinline__ void gather_pair(RowPairRegs<float>& f0, RowPairRegs<float>& f1, int j,
                                            const Geo& G, const cx<float>* B, int y, bool active) {
    if constexpr (TILES) gather_pair_tiles<LC>(f0, f1, j, B, (G.nkx_keep + 1) & ~1, y);
    else gather_pair_rows<LC>(f0, f1, j, G, B, y, active);
}

// Paired row stages that issue the omega gathers ahead of the psi
// transforms: every compile-time length at FP32, and at FP64 all but 1024,
// whose closing radix-2 pass (four butterflies per thread) pushes that
// schedule past the 256-register budget into 44 bytes of scratch.  FP32 rows
// of 1024 spill 8-20 bytes with it and still run faster than without it
// (256-member mixed-size ensemble: 87.0k -> 90.4k member-steps/s).
template <typename T, int LC>
constexpr bool row_prefetch() {
    return LC >= 64 && (LC != 1024 || sizeof(T) == 4);
}

// FORCE: workgroup 0 makes the forcing draw; TILES (ws_lines64): the inputs are in
// row-pair tiles, else per field ([kx][y])
template <typename T, int NT, int MODE, int LC, bool ERR = false,
          int MW = min_waves<T>(), bool FORCE = false, bool TILES = true>
__global__ __launch_bounds__(NT, MW) void k_row(RowArgs<T> a) {
    static_assert(!pair_layout<T, LC, NT>() ||
                      (paired_lines<T, LC, NT>() && row_prefetch<T, LC>()),
                  "the pair layout is read by the paired gather-ahead k_row path");
    // error controller: stages 1-3 of a step that restores a rejected
    // candidate have nothing to do (uniform over the grid)
    if constexpr (ERR && MODE == ROW_STAGE) {
        if (a.skip_on_redo && a.sc[blockIdx.y].redo) return;
    }
    extern __shared__ __align__(16) unsigned char smem_raw[];
    cx<T>* smem = reinterpret_cast<cx<T>*>(smem_raw);
    __shared__ double red[NT / 64];
    const Geo& G = a.geo;
    const Line g = make_line(LC > 0 ? LC : G.nx);
    const int TPL = LC > 0 ? LC / P : g.TPL;
    const int Ll = LC > 0 ? LC : g.L;
    const int lines = NT / TPL;
    const int m = threadIdx.x / TPL, j = threadIdx.x - m * TPL;
    constexpr int NB = stage_regions<T, LC, NT>();
    const int RE = LC > 0 ? region_elems<T, LC, NT>() : Ll + Ll / 16;
    cx<T>* lds = smem + m * NB * RE;
    cx<T>* lds2 = lds + (NB - 1) * RE;
    if constexpr (FORCE) {
        if (blockIdx.x == 0) {
            force_draw<(NT > kForceLanes)>(a.force, blockIdx.y, reinterpret_cast<double*>(smem_raw));
            return;
        }
    }
    const int bx = (int)blockIdx.x - (FORCE ? 1 : 0);
    const int blk = xcd_remap(bx, gridDim.x - (FORCE ? 1 : 0));
    const int item = blk * lines + m;  // row pair (STAGE, R2C) or row (C2R)
    // Staggered start.  The dispatcher gives every compute unit one workgroup
    // before it gives any a second (the host checks this on the device when a
    // context is created and passes an empty range otherwise), so blocks
    // [ncu, 2 ncu) of member 0 are the second residents; they start about 12k
    // cycles late.  The two workgroups of a CU then reach their gather phases
    // at different times, each loading under the other's transforms, and keep
    // that offset for the whole launch (a freed slot is refilled at once).  At
    // 4096 (FP32, two resident workgroups per CU, wave-split transforms) this
    // takes a launch from 72.9 to 71.8 us; 16k cycles (the best delay for the
    // Stockham form, which waited at 27 barriers) measures 72.9 again and 24k
    // cycles 75.6.
    if constexpr (MODE == ROW_STAGE && LC == 4096 && sizeof(T) == 4) {
        if (blockIdx.y == 0 && bx >= a.stagger_lo && bx < a.stagger_hi) {
            __builtin_amdgcn_s_sleep(63);
            __builtin_amdgcn_s_sleep(63);
            __builtin_amdgcn_s_sleep(63);
        }
    }
    cx<T> v[P];
    // member blockIdx.y of a batch (ROW_STAGE only)
    // member blockIdx.y of a batch (mixed fields, physical fields)
    const size_t moff = blockIdx.y * a.bm, roff = blockIdx.y * a.br;

    if constexpr (MODE == ROW_C2R) {
        const int y = item;
        const bool active = y < G.ny;
        for (int f = 0; f < a.nfields; f += 2) {
            const cx<T>* B = (f + 1 < a.nfields) ? a.mixed[f + 1] + moff : nullptr;
            build_row_pair<LC>(v, lds, j, g, G, a.mixed[f] + moff, B, y, active);
            fft_any<+1, LC>(v, lds, j, g, a.tw);
            if (active) {
#pragma unroll
                for (int s = 0; s < P; ++s) {
                    const size_t o = (size_t)y * G.nx + j + s * TPL;
                    if (a.out_ref[f]) a.out_ref[f][o] = double(v[s].x);
                    else if (f == 0 && a.out_bf16)  // round to nearest even
                        a.out_bf16[roff + o] = __builtin_bit_cast(
                            unsigned short, (__bf16)(a.out_bf16_scale * v[s].x));
                    else a.out[f][roff + o] = v[s].x;
                    if (B) {
                        if (a.out_ref[f + 1])
                            a.out_ref[f + 1][o] = double(f == 0 && a.minus1 ? -v[s].y : v[s].y);
                        else a.out[f + 1][roff + o] = v[s].y;
                    }
                }
            }
        }
        return;
    }

    const int y0 = 2 * item;
    const bool active = y0 < G.ny;

    if constexpr (MODE == ROW_R2C) {
#pragma unroll
        for (int s = 0; s < P; ++s) {
            const int x = j + s * TPL;
            if (!active) v[s] = mk(T(0), T(0));
            else if (a.in_t) v[s] = mk(a.in_t[roff + (size_t)y0 * G.nx + x], a.in_t[roff + (size_t)(y0 + 1) * G.nx + x]);
            else v[s] = mk(T(a.in_ref[(size_t)y0 * G.nx + x]), T(a.in_ref[(size_t)(y0 + 1) * G.nx + x]));
        }
        fwd_rows_store<LC>(v, lds, j, g, G, a.tw, a.nl + moff, y0, active);
        return;
    }

    // ROW_STAGE: J = psi_x omega_y - psi_y omega_x (spectral_core.c:101-104).
    // Each field is transformed for both rows at once (f(y0) + i f(y0+1)),
    // in the order psi_x, psi_y, omega_x, omega_y, so that only two packed
    // accumulators live across transforms.
    cx<T> X[P], Jp[P];
    SpeedMax<T> um;
    if constexpr (pair_layout<T, LC, NT>()) {
        // FP32 rows of 2048 to 8192, one to a workgroup: the paired gather-ahead schedule
        // below with wave-split transforms (ws_a for the four fields, whose
        // outputs are in the wave-strided pattern, ws_b for J, which takes
        // that pattern back to the standard one): 11 workgroup barriers per
        // row pair instead of 27 (at 4096).
        TwWs<LC, T> tw;
        load_tw_ws(tw, j, a.tw);
        if (blk * lines < G.ny / 2) {
            // one line per workgroup: inside this branch its row pair exists,
            // and the gathers need no zero fill for an inactive one
            static_assert(NT * P / LC == 1, "one row pair per workgroup");
            constexpr bool live = true;
            constexpr bool PT = pairtile_layout<T, LC, NT>();
            RowPairRegs<T> r0, r1, q0, q1;
            const bool pl = a.pairs != 0;
            if (pl) gather_pair<LC, PT>(r0, r1, j, G, a.mixed[0] + 2 * moff, y0, live);
            else {
                gather_two_rows<LC>(r0, j, G, a.mixed[0] + moff, y0, live);
                gather_two_rows<LC>(r1, j, G, a.mixed[1] + moff, y0, live);
            }
            stage_two_rows_regs<LC, true, false>(lds, j, r0);
            stage_two_rows_regs<LC, true, false>(lds2, j, r1);
            if (pl) gather_pair<LC, PT>(q0, q1, j, G, a.mixed[2] + 2 * moff, y0, live);
            else {
                gather_two_rows<LC>(q0, j, G, a.mixed[2] + moff, y0, live);
                gather_two_rows<LC>(q1, j, G, a.mixed[3] + moff, y0, live);
            }
            __syncthreads();
            cx<T> v2[P];
            cx<T>(*const vv[2])[P] = {&v, &v2};
            cx<T>* const ll[2] = {lds, lds2};
            lds_read_kept<LC, false>(v, lds, j);
            lds_read_kept<LC, false>(v2, lds2, j);
            __syncthreads();
            ws_a<+1, 2>(vv, ll, j, tw);  // psi_x, psi_y
            renew_tw(tw);
            if (a.track_umax) add_speeds(um, v, v2);
#pragma unroll
            for (int s = 0; s < P; ++s) {
                X[s] = v[s];
                Jp[s] = v2[s];
            }
            __syncthreads();
            stage_two_rows_regs<LC, true, false>(lds, j, q0);
            stage_two_rows_regs<LC, true, false>(lds2, j, q1);
            __syncthreads();
            lds_read_kept<LC, false>(v, lds, j);
            lds_read_kept<LC, false>(v2, lds2, j);
            __syncthreads();
            ws_a<+1, 2>(vv, ll, j, tw);  // omega_x, omega_y
            renew_tw(tw);
#pragma unroll
            for (int s = 0; s < P; ++s)
                v[s] = mk(X[s].x * v2[s].x - Jp[s].x * v[s].x, X[s].y * v2[s].y - Jp[s].y * v[s].y);
            fwd_rows_store<LC, T, TwWs<LC, T>, true>(v, lds, j, g, G, tw, a.nl + moff, y0, active,
                                                     a.jblocks);
        }
        if (a.track_umax) block_max_to(active ? double(um.value()) : 0.0, &a.sc[blockIdx.y].umax2_bits, red);
        return;
    }
    if constexpr (paired_lines<T, LC, NT>() && row_prefetch<T, LC>()) {
        // Twiddles first, then the psi gathers, then the omega gathers,
        // which stay in flight while the psi fields are transformed: with
        // the twiddles in registers the transforms issue no global loads
        // that would have to wait behind the gathers.
        TwRegs<LC, T> tw;
        load_tw_regs<LC, 0>(tw, j, a.tw);
        // slots inside the dealiased band neither staged nor read back
        constexpr bool KEPT = LC / P % 16 == 0;
        // (always true: the grid holds no idle workgroup; as a branch it keeps
        // the compiler's schedule of the loads above within 128 VGPRs)
        if (blk * lines < G.ny / 2) {
            RowPairRegs<T> r0, r1, q0, q1;
            gather_two_rows<LC>(r0, j, G, a.mixed[0] + moff, y0, active);
            gather_two_rows<LC>(r1, j, G, a.mixed[1] + moff, y0, active);
            stage_two_rows_regs<LC, KEPT>(lds, j, r0);
            stage_two_rows_regs<LC, KEPT>(lds2, j, r1);
            gather_two_rows<LC>(q0, j, G, a.mixed[2] + moff, y0, active);
            gather_two_rows<LC>(q1, j, G, a.mixed[3] + moff, y0, active);
            __syncthreads();
            cx<T> v2[P];
            lds_read_any<LC, KEPT>(v, lds, j);
            lds_read_any<LC, KEPT>(v2, lds2, j);
            line_fft2_c<+1, LC>(v, v2, lds, lds2, j, tw);  // psi_x, psi_y
            if (a.track_umax) add_speeds(um, v, v2);
#pragma unroll
            for (int s = 0; s < P; ++s) {
                X[s] = v[s];
                Jp[s] = v2[s];
            }
            __syncthreads();
            stage_two_rows_regs<LC, KEPT>(lds, j, q0);
            stage_two_rows_regs<LC, KEPT>(lds2, j, q1);
            __syncthreads();
            lds_read_any<LC, KEPT>(v, lds, j);
            lds_read_any<LC, KEPT>(v2, lds2, j);
            line_fft2_c<+1, LC>(v, v2, lds, lds2, j, tw);  // omega_x, omega_y
#pragma unroll
            for (int s = 0; s < P; ++s)
                v[s] = mk(X[s].x * v2[s].x - Jp[s].x * v[s].x, X[s].y * v2[s].y - Jp[s].y * v[s].y);
            fwd_rows_store<LC, T, TwRegs<LC, T>>(v, lds, j, g, G, tw, a.nl + moff, y0, active);
        }
        if (a.track_umax) block_max_to(active ? double(um.value()) : 0.0, &a.sc[blockIdx.y].umax2_bits, red);
        return;
    }
    if constexpr (paired_lines<T, LC, NT>()) {
        // FP64 rows of 1024: gathers at their use
        cx<T> v2[P];
        build_two_rows2<LC>(v, v2, lds, lds2, j, g, G, a.mixed[0] + moff, a.mixed[1] + moff, y0, active);
        line_fft2_c<+1, LC>(v, v2, lds, lds2, j, a.tw);  // psi_x, psi_y
        if (a.track_umax) add_speeds(um, v, v2);
#pragma unroll
        for (int s = 0; s < P; ++s) {
            X[s] = v[s];
            Jp[s] = v2[s];
        }
        build_two_rows2<LC>(v, v2, lds, lds2, j, g, G, a.mixed[2] + moff, a.mixed[3] + moff, y0, active);
        line_fft2_c<+1, LC>(v, v2, lds, lds2, j, a.tw);  // omega_x, omega_y
#pragma unroll
        for (int s = 0; s < P; ++s)
            v[s] = mk(X[s].x * v2[s].x - Jp[s].x * v[s].x, X[s].y * v2[s].y - Jp[s].y * v[s].y);
        fwd_rows_store<LC>(v, lds, j, g, G, a.tw, a.nl + moff, y0, active);
        if (a.track_umax) block_max_to(active ? double(um.value()) : 0.0, &a.sc[blockIdx.y].umax2_bits, red);
        return;
    }
    if constexpr (ws_lines64<T, LC, NT>()) {
        // FP64 rows of 2048 and 4096: one field at a time, each gather in flight while
        // the previous field is transformed (as below), with wave-split
        // transforms whose cross-wave rows live in lds2.  Every read of the
        // staged line in lds precedes the barrier inside ws_a, so the next
        // field is staged without one: 10 barriers per row pair instead of 45.
        TwWs<LC, T> tw;
        load_tw_ws(tw, j, a.tw);
        if (blk * lines < G.ny / 2) {
            cx<T>(*const vv[1])[P] = {&v};
            cx<T>* const rr[1] = {lds2};
            // one line per workgroup, whose row pair exists inside this branch
            static_assert(NT * P / LC == 1, "one row pair per workgroup");
            // (pairs is set where TILES is; as a run-time value it keeps a schedule of the
            // gathers that is 1.5 % faster: FP64 4096^2 162.5 -> 159.5 us)
            const SlotElems se =
                row_slots<LC>(j, G.ny, (G.nkx_keep + 1) & ~1, y0, TILES && a.pairs != 0);
            RowPairRegs<T> r;
            gather_two_rows<LC, TILES>(r, j, a.mixed[0] + moff, se);
            stage_two_rows_regs<LC, true, false>(lds, j, r);
            gather_two_rows<LC, TILES>(r, j, a.mixed[1] + moff, se);
            __syncthreads();
            lds_read_kept<LC, false>(v, lds, j);
            ws_a<+1, 1, true>(vv, rr, j, tw);  // psi_x
#pragma unroll
            for (int s = 0; s < P; ++s) X[s] = v[s];
            __builtin_amdgcn_sched_barrier(0);
            stage_two_rows_regs<LC, true, false>(lds, j, r);
            gather_two_rows<LC, TILES>(r, j, a.mixed[2] + moff, se);
            __syncthreads();
            lds_read_kept<LC, false>(v, lds, j);
            ws_a<+1, 1, true>(vv, rr, j, tw);  // psi_y
            if (a.track_umax) add_speeds(um, X, v);
#pragma unroll
            for (int s = 0; s < P; ++s) Jp[s] = v[s];
            __builtin_amdgcn_sched_barrier(0);
            stage_two_rows_regs<LC, true, false>(lds, j, r);
            gather_two_rows<LC, TILES>(r, j, a.mixed[3] + moff, se);
            __syncthreads();
            lds_read_kept<LC, false>(v, lds, j);
            ws_a<+1, 1, true>(vv, rr, j, tw);  // omega_x
#pragma unroll
            for (int s = 0; s < P; ++s) Jp[s] = mk(-Jp[s].x * v[s].x, -Jp[s].y * v[s].y);
            __builtin_amdgcn_sched_barrier(0);
            stage_two_rows_regs<LC, true, false>(lds, j, r);
            __syncthreads();
            lds_read_kept<LC, false>(v, lds, j);
            ws_a<+1, 1, true>(vv, rr, j, tw);  // omega_y
#pragma unroll
            for (int s = 0; s < P; ++s)
                v[s] = mk(Jp[s].x + X[s].x * v[s].x, Jp[s].y + X[s].y * v[s].y);
            // J: ws_b in lds, whose rows nobody reads any more
            fwd_rows_store<LC, T, TwWs<LC, T>>(v, lds, j, g, G, tw, a.nl + moff, y0, active);
        }
        if (a.track_umax) block_max_to(active ? double(um.value()) : 0.0, &a.sc[blockIdx.y].umax2_bits, red);
        return;
    }
    if constexpr (LC >= 2048 && NT <= 512) {
        // Long rows, one line region (FP64): each field's gather is in flight
        // while the previous field is transformed (twiddles in registers, as
        // in the paired path above).  Not for the 1024-thread workgroups of
        // the longest rows, whose 128-register budget it would overflow.
        TwRegs<LC, T> tw;
        load_tw_regs<LC, 0>(tw, j, a.tw);
        // (always true; as a branch it keeps the schedule of the loads above
        // within the register budget)
        if (blk * lines < G.ny / 2) {
            RowPairRegs<T> r;
            gather_two_rows<LC>(r, j, G, a.mixed[0] + moff, y0, active);
            stage_two_rows_regs<LC>(lds, j, r);
            gather_two_rows<LC>(r, j, G, a.mixed[1] + moff, y0, active);
            __syncthreads();
            lds_read_c<LC>(v, lds, j);
            line_fft_c<+1, LC>(v, lds, j, tw);  // psi_x
#pragma unroll
            for (int s = 0; s < P; ++s) X[s] = v[s];
            __builtin_amdgcn_sched_barrier(0);
            __syncthreads();
            stage_two_rows_regs<LC>(lds, j, r);
            gather_two_rows<LC>(r, j, G, a.mixed[2] + moff, y0, active);
            __syncthreads();
            lds_read_c<LC>(v, lds, j);
            line_fft_c<+1, LC>(v, lds, j, tw);  // psi_y
            if (a.track_umax) add_speeds(um, X, v);
#pragma unroll
            for (int s = 0; s < P; ++s) Jp[s] = v[s];
            __builtin_amdgcn_sched_barrier(0);
            __syncthreads();
            stage_two_rows_regs<LC>(lds, j, r);
            gather_two_rows<LC>(r, j, G, a.mixed[3] + moff, y0, active);
            __syncthreads();
            lds_read_c<LC>(v, lds, j);
            line_fft_c<+1, LC>(v, lds, j, tw);  // omega_x
#pragma unroll
            for (int s = 0; s < P; ++s) Jp[s] = mk(-Jp[s].x * v[s].x, -Jp[s].y * v[s].y);
            __builtin_amdgcn_sched_barrier(0);
            __syncthreads();
            stage_two_rows_regs<LC>(lds, j, r);
            __syncthreads();
            lds_read_c<LC>(v, lds, j);
            line_fft_c<+1, LC>(v, lds, j, tw);  // omega_y
#pragma unroll
            for (int s = 0; s < P; ++s)
                v[s] = mk(Jp[s].x + X[s].x * v[s].x, Jp[s].y + X[s].y * v[s].y);
            fwd_rows_store<LC>(v, lds, j, g, G, tw, a.nl + moff, y0, active);
        }
        if (a.track_umax) block_max_to(active ? double(um.value()) : 0.0, &a.sc[blockIdx.y].umax2_bits, red);
        return;
    }
    build_two_rows<LC>(v, lds, j, g, G, a.mixed[0] + moff, y0, active);  // psi_x
    fft_any<+1, LC>(v, lds, j, g, a.tw);
#pragma unroll
    for (int s = 0; s < P; ++s) X[s] = v[s];
    build_two_rows<LC>(v, lds, j, g, G, a.mixed[1] + moff, y0, active);  // psi_y
    fft_any<+1, LC>(v, lds, j, g, a.tw);
    if (a.track_umax) add_speeds(um, X, v);
#pragma unroll
    for (int s = 0; s < P; ++s) Jp[s] = v[s];  // psi_y, folded with omega_x next
    build_two_rows<LC>(v, lds, j, g, G, a.mixed[2] + moff, y0, active);  // omega_x
    fft_any<+1, LC>(v, lds, j, g, a.tw);
#pragma unroll
    for (int s = 0; s < P; ++s) Jp[s] = mk(-Jp[s].x * v[s].x, -Jp[s].y * v[s].y);
    build_two_rows<LC>(v, lds, j, g, G, a.mixed[3] + moff, y0, active);  // omega_y
    fft_any<+1, LC>(v, lds, j, g, a.tw);
#pragma unroll
    for (int s = 0; s < P; ++s)
        v[s] = mk(Jp[s].x + X[s].x * v[s].x, Jp[s].y + X[s].y * v[s].y);
    fwd_rows_store<LC>(v, lds, j, g, G, a.tw, a.nl + moff, y0, active);
    if (a.track_umax) block_max_to(active ? double(um.value()) : 0.0, &a.sc[blockIdx.y].umax2_bits, red);
}

}  // namespace nsd
