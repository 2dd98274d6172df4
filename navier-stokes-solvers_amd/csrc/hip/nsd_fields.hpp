// nsd_fields.hpp -- field-parallel stage kernels: small FP64 grids, and any grid of up
// to 1024 points a side by name (stage_variant_default has the rule).
//
// The stage kernels of nsd_kernels.hpp give a line to one group of L / 8
// threads, which takes a row pair through its four inverse transforms and the
// transform of J one after the other (two at a time in lock-step).  That is the
// least work per launch, and where a launch has many lines the waves of other
// lines fill the waits.  A launch with few lines has nothing to fill them with:
// at 1024^2 the 512 row pairs are one wave per SIMD, and its time is the length
// of that chain.  Here a row pair (or a column) is a unit of four groups of
// L / 8 threads, one per derivative field: the four transforms of a unit run
// side by side, the chain is one inverse and one forward transform, and the
// launch has four times the waves.  The pointwise work (the per-mode update, the
// separation of J's two rows) is spread over all four groups.  A line of up to
// 512 points stays inside one wave, so its exchanges through LDS need no
// workgroup barrier.
//
// Same layouts and the same formulas as the kernels of nsd_kernels.hpp:
// per-field mixed fields and J, both [kx][y].
#pragma once

#include "nsd_kernels.hpp"

namespace nsd {

// ------------------------------------------------------------------ lines

// All twiddles of a line's passes in registers: W^k of the full-radix passes
// (powers by squaring, as TwRegs) and the table values of the closing radix-2
// or radix-4 pass, so that no load sits inside a transform.
template <int L, typename T>
struct TwAll {
    static constexpr int R = CLine<L>::rem;
    static constexpr int QN = R > 1 ? P / R : 1, EN = R == 4 ? 2 : 1;
    cx<T> w[CLine<L>::passes];
    cx<T> tail[QN][EN];
    template <int L2, int PASS>
    __device__ __forceinline__ cx<T> get(int q, int e, int) const {
        if constexpr (CLine<L>::radix(PASS) == P) {
            cx<T> r = w[PASS];
            for (int i = 0; i < e; ++i) r = cmul(r, r);
            return r;
        } else {
            return tail[q][e];
        }
    }
};

template <int L, int PASS, typename T>
__device__ __forceinline__ void load_tw_all(TwAll<L, T>& t, int j, const cx<T>* __restrict__ tw) {
    if constexpr (PASS < CLine<L>::passes) {
        using G = CLine<L>;
        constexpr int Ns = G::stride(PASS), R = G::radix(PASS);
        if constexpr (Ns > 1 && R == P) {
            t.w[PASS] = tw[(j & (Ns - 1)) * (L / (Ns * P))];
        } else if constexpr (Ns > 1) {
#pragma unroll
            for (int q = 0; q < P / R; ++q)
#pragma unroll
                for (int e = 0; e < (R == 4 ? 2 : 1); ++e)
                    t.tail[q][e] = tw[(((j + q * G::TPL) & (Ns - 1)) << e) * (L / (Ns * R))];
        }
        load_tw_all<L, PASS + 1>(t, j, tw);
    }
}

// the powers that one transform formed are not kept for the next (renew)
template <int L, typename T>
__device__ __forceinline__ void renew_tw_all(TwAll<L, T>& t) {
#pragma unroll
    for (int p = 1; p < CLine<L>::nP; ++p) renew(t.w[p]);
}

// threads of a unit (four lines side by side)
template <int L>
constexpr int unit_threads() { return L / 2; }

// Exchanges between the threads of one line, and of one unit: inside a wave
// only the compiler has to be held back.  NTH threads in aligned groups.
template <int NTH>
__device__ __forceinline__ void group_sync() {
    if constexpr (NTH <= 64) wave_lds_fence();
    else __syncthreads();
}
template <int L>
__device__ __forceinline__ void line_sync() { group_sync<L / P>(); }
template <int L>
__device__ __forceinline__ void unit_sync() { group_sync<unit_threads<L>()>(); }

// The transform of one line by its L / 8 threads, standard pattern in and out.
// `act`: this line has one (uniform over its threads); every thread takes the
// barriers.  The region must be free on entry; the line's threads may still
// read it on return.
template <int DIR, int L, int PASS = 0, typename T>
__device__ __forceinline__ void line_fft_act(cx<T> (&v)[P], cx<T>* lds, int j,
                                             const TwAll<L, T>& tw, bool act) {
    if constexpr (PASS < CLine<L>::passes) {
        if constexpr (PASS > 0) {
            line_sync<L>();  // the previous pass is written
            if (act) lds_read_c<L>(v, lds, j);
            if constexpr (PASS + 1 < CLine<L>::passes) line_sync<L>();
        }
        if (act) cpass<DIR, L, PASS>(v, j, tw, lds);
        line_fft_act<DIR, L, PASS + 1>(v, lds, j, tw, act);
    }
}

// Lines of 1024 points (two waves): wave-split transforms (ws_a, ws_b), one
// barrier each where the Stockham passes take six.
template <int L>
constexpr bool ws_unit() { return L > 512; }
// elements of a line region
template <int L>
constexpr int unit_region() { return ws_unit<L>() ? ws_region(L) : L + L / 16; }
template <int L, typename T>
using UnitTw = std::conditional_t<ws_unit<L>(), TwWs<(L > 512 ? L : 1024), T>, TwAll<L, T>>;

template <int L, typename T>
__device__ __forceinline__ void load_unit_tw(UnitTw<L, T>& t, int j, const cx<T>* __restrict__ tw) {
    if constexpr (ws_unit<L>()) load_tw_ws(t, j, tw);
    else load_tw_all<L, 0>(t, j, tw);
}

// ws_a and ws_b of one line, for the lines that have one (`act`)
template <int DIR, int L, typename T>
__device__ __forceinline__ void ws_a_act(cx<T> (&v)[P], cx<T>* lds, int j, const TwWs<L, T>& tw,
                                         bool act) {
    constexpr int W = ws_waves(L), Q = 8 / W;
    constexpr bool SWZ = sizeof(T) == 8;
    const int l = j & 63;
    cx<T>* const row[1] = {lds + (j >> 6) * WS_ROW};
    if (act) {
        ws_cross<DIR, W, true>(v, tw.wj);
        cx<T>* o = lds + ws_pos<SWZ>(j);
#pragma unroll
        for (int r = 0; r < W; ++r)
#pragma unroll
            for (int h = 0; h < Q; ++h) o[r * WS_ROW + ws_off<SWZ>(W * h)] = v[h + Q * r];
    }
    __syncthreads();
    if (act) {
        const cx<T>* i = row[0] + ws_pos<SWZ>(l);
#pragma unroll
        for (int s = 0; s < 8; ++s) v[s] = i[ws_off<SWZ>(s)];
        wave_lds_fence();
        cx<T>(*const vv[1])[P] = {&v};
        ws_local<DIR, 1, SWZ>(vv, row, l, tw);
    }
}
template <int DIR, int L, typename T>
__device__ __forceinline__ void ws_b_act(cx<T> (&v)[P], cx<T>* lds, int j, const TwWs<L, T>& tw,
                                         bool act) {
    constexpr int W = ws_waves(L), Q = 8 / W;
    constexpr bool SWZ = sizeof(T) == 8;
    const int l = j & 63;
    cx<T>* const row[1] = {lds + (j >> 6) * WS_ROW};
    if (act) {
        cx<T>(*const vv[1])[P] = {&v};
        ws_local<DIR, 1, SWZ>(vv, row, l, tw);
        cx<T>* o = row[0] + ws_pos<SWZ>(l);
#pragma unroll
        for (int s = 0; s < 8; ++s) o[ws_off<SWZ>(s)] = v[s];
    }
    __syncthreads();
    if (act) {
        const cx<T>* i = lds + ws_pos<SWZ>(j);
#pragma unroll
        for (int r = 0; r < W; ++r)
#pragma unroll
            for (int h = 0; h < Q; ++h) v[h + Q * r] = i[r * WS_ROW + ws_off<SWZ>(W * h)];
        ws_cross<DIR, W, false>(v, tw.wj);
    }
}
// the wave-strided pattern's element of slot s is ws_index(j) + s L / 8, as the
// standard pattern's is j + s L / 8
template <int L>
__device__ __forceinline__ int ws_index(int j) { return ws_waves(L) * (j & 63) + (j >> 6); }

// ---------------------------------------------------------------- row stage

// One row pair (rows y, y + 1) of the row stage: inverse x-transforms of the
// four fields, J, the forward x-transform of J, kept columns stored.  r: this
// thread of the unit; lds: the unit's four line regions.
template <typename T, int L>
__device__ __forceinline__ void row_unit(cx<T>* lds, int r, const Geo& G, const cx<T>* F, cx<T>* nl,
                                         int y, bool active, UnitTw<L, T>& tw, bool track,
                                         SpeedMax<T>& um) {
    constexpr int TPL = L / P, RE = unit_region<L>(), kxm = Band<L>::kxm;
    constexpr bool KEPT = TPL % 16 == 0, WS = ws_unit<L>();
    auto at = [](int i) { return WS ? i : pad(i); };
    const int f = r / TPL, j = r - f * TPL;
    cx<T>* const own = lds + f * RE;
    cx<T> v[P];
    {
        RowPairRegs<T> q;
#pragma unroll
        for (int s = 0; s < P; ++s) {
            const int kind = slot_kind(s, L, kxm), k = j + s * TPL;
            if (kind == 1 || (kind == 3 && k <= kxm)) {
                if (active) {
                    const cx<T>* src = at32(F, col_elem(k, G.ny, y));
                    q.a[s] = src[0];
                    q.b[s] = src[1];
                } else {
                    q.a[s] = mk(T(0), T(0));
                    q.b[s] = mk(T(0), T(0));
                }
            }
        }
        stage_two_rows_regs<L, KEPT, !WS>(own, j, q);
    }
    line_sync<L>();
    if constexpr (WS) lds_read_kept<L, false>(v, own, j);
    else lds_read_any<L, KEPT>(v, own, j);
    line_sync<L>();
    // the exchange area of a thread: its slots of the line, or (wave-split) of
    // its wave's own row
    const int x0 = WS ? (j >> 6) * WS_ROW + (j & 63) : pad(j);
    auto xo = [](int s) { return WS ? 64 * s : TPL % 16 == 0 ? padc(s * TPL) : 0; };
    auto put = [&](cx<T>* o) {
        if constexpr (WS || TPL % 16 == 0) {
#pragma unroll
            for (int s = 0; s < P; ++s) o[x0 + xo(s)] = v[s];
        } else {
            lds_write_c<L>(v, o, j);
        }
    };
    auto get = [&](cx<T> (&d)[P], const cx<T>* o) {
        if constexpr (WS || TPL % 16 == 0) {
#pragma unroll
            for (int s = 0; s < P; ++s) d[s] = o[x0 + xo(s)];
        } else {
            lds_read_c<L>(d, o, j);
        }
    };
    if constexpr (WS) {
        ws_a_act<+1, L>(v, own, j, tw, true);
    } else {
        line_fft_act<+1, L>(v, own, j, tw, true);
        line_sync<L>();
    }
    // psi_y, omega_x, omega_y to the threads that hold psi_x
    if (f > 0) put(own);
    unit_sync<L>();
    const bool first = f == 0;
    if (first) {
        // J = psi_x omega_y - psi_y omega_x (spectral_core.c:101-104), in two
        // sweeps so that few values are held at once
        cx<T> b[P], c[P];
        get(b, lds + RE);
        get(c, lds + 2 * RE);
        if (track) add_speeds(um, v, b);
#pragma unroll
        for (int s = 0; s < P; ++s) b[s] = mk(b[s].x * c[s].x, b[s].y * c[s].y);
        __builtin_amdgcn_sched_barrier(0);
        get(c, lds + 3 * RE);
#pragma unroll
        for (int s = 0; s < P; ++s)
            v[s] = mk(v[s].x * c[s].x - b[s].x, v[s].y * c[s].y - b[s].y);
    }
    if constexpr (WS) {
        renew(tw.wj);
        renew(tw.w8);
        renew(tw.w64);
        ws_b_act<-1, L>(v, lds, j, tw, first);
    } else {
        renew_tw_all(tw);
        line_fft_act<-1, L>(v, lds, j, tw, first);
    }
    line_sync<L>();
    if (first) {
        // the slots that the separation reads (as fwd_rows_store)
        if constexpr (KEPT) {
            cx<T>* b = lds + at(j);
#pragma unroll
            for (int s = 0; s < P; ++s)
                if (slot_kind(s, L, kxm) != 0) b[WS ? s * TPL : padc(s * TPL)] = v[s];
        } else {
            lds_write_c<L>(v, lds, j);
        }
    }
    unit_sync<L>();
    // separation of the two rows, one kept column per thread
    constexpr int UT = unit_threads<L>();
#pragma unroll
    for (int k0 = 0; k0 <= kxm; k0 += UT) {
        const int k = k0 + r;
        if (k <= kxm && active) {
            const cx<T> zk = lds[at(k)];
            const cx<T> zm = lds[at((L - k) & (L - 1))];
            cx<T>* dst = at32(nl, col_elem(k, G.ny, y));
            dst[0] = mk(T(0.5) * (zk.x + zm.x), T(0.5) * (zk.y - zm.y));
            dst[1] = mk(T(0.5) * (zk.y + zm.y), T(0.5) * (zm.x - zk.x));
        }
    }
}

// U row pairs per workgroup (ERR: under the error controller, idle in the later stages
// of a step that restores a rejected one)
template <typename T, int L, int U, int MW, bool FORCE, bool ERR>
__global__ __launch_bounds__(U * L / 2, MW) void k_row_fields(RowArgs<T> a) {
    static_assert(!(FORCE && ERR), "the controller's draw is a kernel of its own");
    extern __shared__ __align__(16) unsigned char smem_raw[];
    if constexpr (ERR) {
        if (a.skip_on_redo && a.sc[blockIdx.y].redo) return;
    }
    if constexpr (FORCE) {  // workgroup 0 makes the step's forcing draw
        if (blockIdx.x == 0) {
            force_draw<(U * L / 2 > kForceLanes)>(a.force, blockIdx.y, reinterpret_cast<double*>(smem_raw));
            return;
        }
    }
    const int bx = (int)blockIdx.x - (FORCE ? 1 : 0);
    __shared__ double red[U * L / 2 > 64 ? U * L / 128 : 1];
    constexpr int UT = unit_threads<L>(), RE = unit_region<L>();
    const int u = threadIdx.x / UT, r = threadIdx.x - u * UT;
    const int f = r / (L / P), j = r - f * (L / P);
    const Geo& G = a.geo;
    const int y = 2 * (xcd_remap(bx, gridDim.x - (FORCE ? 1 : 0)) * U + u);
    const size_t moff = blockIdx.y * a.bm;
    UnitTw<L, T> tw;
    load_unit_tw<L>(tw, j, a.tw);
    const cx<T>* F = f < 2 ? (f == 0 ? a.mixed[0] : a.mixed[1]) : (f == 2 ? a.mixed[2] : a.mixed[3]);
    SpeedMax<T> um;
    row_unit<T, L>(reinterpret_cast<cx<T>*>(smem_raw) + u * 4 * RE, r, G, F + moff,
                              a.nl + moff, y, y < G.ny, tw, a.track_umax != 0, um);
    if (a.track_umax) block_max_to(double(um.value()), &a.sc[blockIdx.y].umax2_bits, red);
}

// ------------------------------------------------------------- column stage

// What a mode's stage update needs beside the fields, formed while they arrive:
// classic scheme a = L = -(k^2/Re + drag + w_hv), b the SFD weight; integrating
// factor a = E - 1, b = E2 - 1 (k_col has the reason), E2 = exp(L h / 2).
template <typename T>
struct ModeFactors {
    T a, b;
};
template <typename T, int SCHEME>
__device__ __forceinline__ ModeFactors<T> mode_factors(const Phys& ph, T h, T k2) {
    ModeFactors<T> m;
    const T lin = -(k2 * T(ph.inv_Re) + T(ph.drag) + hv_weight_t<T>(ph, k2));
    if constexpr (SCHEME == 0) {
        m.a = lin;
        m.b = sfd_weight_t<T>(ph, k2);
    } else {
        m.b = expm1_t(lin * (T(0.5) * h));
        m.a = m.b * (T(2) + m.b);  // E = E2^2
    }
    return m;
}

// One mode's stage update: N (with the closure's source), the state at the
// step's start w0, the accumulator av (from stage 1 on) and, in the classic
// scheme, the stage field ws and the SFD state fs; h6 = h / 6, h3 = h / 3.
// Returns the new stage field and leaves the accumulator in av (stages 0..2) and
// the SFD state in fs; ERR: in stage 1 also the midpoint solution, in mid.
template <typename T, int SCHEME, bool ERR>
__device__ __forceinline__ cx<T> mode_update(const Phys& ph, int stage, T h, T h6, T h3, double dt,
                                             ModeFactors<T> m, cx<T> N, cx<T> w0, cx<T>& av,
                                             cx<T> ws, cx<T>& fs, cx<T>& mid) {
    cx<T> wn;
    if constexpr (SCHEME == 0) {
        // classic RK4 (spectral_time_integration.c:50-100) with
        // hyperviscosity_apply (hyperviscosity.c:104-150) and drag
        cx<T> ks = N + m.a * ws;
        if (m.b > T(0)) ks = ks - m.b * (ws - fs);
        if (stage == 0) {
            av = w0 + h6 * ks;
            wn = w0 + (T(0.5) * h) * ks;
        } else if (stage == 1) {
            av = av + h3 * ks;
            wn = w0 + (T(0.5) * h) * ks;
            if constexpr (ERR) mid = w0 + h * ks;
        } else if (stage == 2) {
            av = av + h3 * ks;
            wn = w0 + h * ks;
        } else {
            wn = av + h6 * ks;
            if (ph.sfd_on && ph.sfd_tau > 0.0) {  // hyperviscosity.c:152-178
                const T al = T(fmin(fmax(dt / ph.sfd_tau, 0.0), 1.0));
                fs = (T(1) - al) * fs + al * wn;
            }
        }
    } else {
        const T e1 = m.a, e2 = m.b;
        if (stage == 0) {
            av = grow(w0, e1) + h6 * grow(N, e1);
            wn = grow(w0 + (T(0.5) * h) * N, e2);
        } else if (stage == 1) {
            av = av + h3 * grow(N, e2);
            wn = grow(w0, e2) + (T(0.5) * h) * N;
            if constexpr (ERR) mid = grow(w0, e1) + h * grow(N, e2);
        } else if (stage == 2) {
            av = av + h3 * grow(N, e2);
            wn = grow(w0, e1) + h * grow(N, e2);
        } else {
            wn = av + h6 * N;
        }
    }
    return wn;
}

// Kept modes of a column per thread of its unit (2 L / 3 over L / 2 threads)
constexpr int kUnitModes = 2;

// Inverse y-transforms of the derivative fields of one column's stage field,
// whose kept modes lie in region w of the unit (in order; padded unless
// wave-split): field f of this thread's group into out.  Outputs 0 psi_x, 1 psi_y, 2 omega_x,
// 3 omega_y (spectral_core.c:62-99).
template <typename T, int L>
__device__ __forceinline__ void col_unit_out(cx<T>* lds, const cx<T>* w, int r, const Geo& G,
                                             int kxi, T kx, T kys, cx<T>* out, bool active,
                                             const UnitTw<L, T>& tw) {
    constexpr int TPL = L / P, RE = unit_region<L>(), kym = Band<L>::kym;
    const int f = r / TPL, j = r - f * TPL;
    constexpr bool WS = ws_unit<L>();
    const int ji = WS ? ws_index<(L > 512 ? L : 1024)>(j) : j;  // input pattern
    cx<T> v[P];
#pragma unroll
    for (int s = 0; s < P; ++s) {
        const int kind = slot_kind(s, L, kym), jy = ji + s * TPL;
        v[s] = mk(T(0), T(0));
        if (kind == 0) continue;
        const cx<T> m = w[WS ? jy : pad(jy)];
        if (kind != 3 || jy <= kym || jy >= L - kym) v[s] = m;
    }
    unit_sync<L>();  // the modes are read: the transforms may use their region
    if (f < 2) {  // psi_hat = -omega_hat / k^2
#pragma unroll
        for (int s = 0; s < P; ++s) {
            if (slot_kind(s, L, kym) == 0) continue;
            const T ky = T(col_band<L>(G, ji + s * TPL)) * kys;
            const T k2 = kx * kx + ky * ky;
            v[s] = k2 > T(1e-12) ? neg_inv_k2(k2) * v[s] : mk(T(0), T(0));
        }
    }
#pragma unroll
    for (int s = 0; s < P; ++s) {
        const T ky = T(col_band<L>(G, ji + s * TPL)) * kys;
        v[s] = mul_i(v[s], (f & 1) ? ky : kx);
    }
    if constexpr (WS) ws_b_act<+1, L>(v, lds + f * RE, j, tw, true);
    else line_fft_act<+1, L>(v, lds + f * RE, j, tw, true);
    if (active) {
        cx<T>* o = out + (size_t)kxi * G.ny + j;
#pragma unroll
        for (int s = 0; s < P; ++s) o[s * TPL] = v[s];
    }
}

// U columns per workgroup, one stage (ERR: under the error controller, as k_col: the
// state kept before a candidate, the midpoint solution, the sums of the estimate, and
// the restoring pass of a rejected candidate)
template <typename T, int L, int SCHEME, int U, int MW, bool ERR>
__global__ __launch_bounds__(U * L / 2, MW) void k_col_fields(ColArgs<T> a) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    constexpr int UT = unit_threads<L>(), TPL = L / P, RE = unit_region<L>();
    constexpr int kym = Band<L>::kym, ncy = 2 * kym + 1;
    static_assert(ncy <= kUnitModes * UT, "kept modes per thread");
    const int u = threadIdx.x / UT, r = threadIdx.x - u * UT;
    const int f = r / TPL, j = r - f * TPL;
    cx<T>* const lds = reinterpret_cast<cx<T>*>(smem_raw) + u * 4 * RE;
    const Geo& G = a.geo;
    const size_t mb = blockIdx.y;
    DevScalars* const sc = a.sc + mb;
    int redo = 0;  // uniform over the grid
    if constexpr (ERR) {
        redo = sc->redo;
        if (redo ? a.stage > 0 : a.finalize != 0) return;
    }
    Phys ph = a.phys;
    if (a.m_inv_re) {
        ph.inv_Re = a.m_inv_re[mb];
        ph.Re = 1.0 / ph.inv_Re;
    }
    const int kxi = blockIdx.x * U + u;
    const bool active = kxi < G.nkx_keep;
    // wavenumber steps and 1 / (nx ny) from the host: no division on the way
    const T kx = T(kxi) * T(a.kxs), kys = T(a.kys);
    const cx<T> zero = mk(T(0), T(0));
    // The step's dt first, then everything that needs no field: a launch this
    // small waits one memory latency for J, and what the wave works out in that
    // time costs nothing (64^2 FP64 step 47.1 -> 46.5 us, 512-point columns of
    // 2048 x 512 134.2 -> 132.2 us).
    const bool pick = a.stage == 0 && ph.adaptive;
    const double u2 = pick ? __longlong_as_double((long long)sc->umax2_bits) : 0.0;
    double dt = pick ? 0.0 : sc->dt;
    UnitTw<L, T> tw;
    load_unit_tw<L>(tw, j, a.tw);
    // J by the first group
    cx<T> v[P];
    const bool first = f == 0;
    if (first) {
        const cx<T>* nl = a.nl + mb * a.bm + (size_t)kxi * G.ny + j;
#pragma unroll
        for (int s = 0; s < P; ++s) v[s] = active ? nl[s * TPL] : zero;
    }
    const size_t c0 = mb * a.bc + (size_t)kxi * ncy;
    cx<T> w0[kUnitModes], av[kUnitModes], ws[kUnitModes], fs[kUnitModes];
#pragma unroll
    for (int q = 0; q < kUnitModes; ++q) {
        const int c = r + q * UT;
        w0[q] = av[q] = ws[q] = fs[q] = zero;
        if (c < ncy && active) {
            w0[q] = a.state[c0 + c];
            if (a.stage > 0) av[q] = a.acc[c0 + c];
            if constexpr (SCHEME == 0) {
                ws[q] = a.stage == 0 ? w0[q] : a.stagebuf[c0 + c];
                if (ph.sfd_on) fs[q] = a.sfd[c0 + c];
            }
        }
    }
    constexpr bool WS = ws_unit<L>();
    auto at = [](int i) { return WS ? i : pad(i); };
    if (pick) {
        dt = cfl_dt(ph, sqrt(u2));
        if constexpr (ERR) dt = fmin(fmax(fmin(dt, sc->dt_err), ph.dt_lo), ph.dt_hi);
        if (blockIdx.x == 0 && threadIdx.x == 0 && !redo) {
            sc->dt = dt;
            if (!(u2 <= 1.0e300)) sc->status = 2;  // SOLVER_DIVERGED
        }
    }
    const T h = T(dt), norm = T(a.norm), sqh = T(sqrt(dt));
    const T h6 = h / T(6), h3 = h / T(3);
    ModeFactors<T> mf[kUnitModes];
#pragma unroll
    for (int q = 0; q < kUnitModes; ++q) {
        const int c = r + q * UT;
        const T ky = T(c <= kym ? c : c - ncy) * kys;
        mf[q] = mode_factors<T, SCHEME>(ph, h, kx * kx + ky * ky);
    }
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (WS) ws_a_act<-1, L>(v, lds, j, tw, first);
    else line_fft_act<-1, L>(v, lds, j, tw, first);
    __builtin_amdgcn_sched_barrier(0);
    // J's spectrum in order: region 0, or (wave-split, whose rows other waves may
    // still read there) region 1; the updated modes go to the next region
    cx<T>* const jh = lds + (WS ? RE : 0);
    cx<T>* const wh = jh + RE;
    if constexpr (WS) {
        if (first) {
            cx<T>* o = jh + ws_index<(L > 512 ? L : 1024)>(j);
#pragma unroll
            for (int s = 0; s < P; ++s) o[s * TPL] = v[s];
        }
    } else {
        line_sync<L>();
        if (first) lds_write_c<L>(v, jh, j);
    }
    unit_sync<L>();
    double esum = 0.0, ssum = 0.0;  // sums w |y4 - y2|^2 and w |y4|^2 of this thread
#pragma unroll
    for (int q = 0; q < kUnitModes; ++q) {
        const int c = r + q * UT;
        if (c >= ncy || !active) continue;
        const int jy = c <= kym ? c : c + (L - ncy);
        if constexpr (ERR) {
            if (redo) {  // the state of the last accepted step comes back
                const cx<T> back = a.prev[c0 + c];
                a.state[c0 + c] = back;
                wh[at(jy)] = back;
                continue;
            }
            if (a.stage == 0) a.prev[c0 + c] = w0[q];
        }
        // N = -norm FFT(J) (spectral_core.c:106-111)
        cx<T> N = (-norm) * jh[at(jy)];
        if (a.src) N = N + a.src[c0 + c];
        cx<T> mid = zero;
        cx<T> wn = mode_update<T, SCHEME, ERR>(ph, a.stage, h, h6, h3, dt, mf[q], N, w0[q], av[q],
                                               ws[q], fs[q], mid);
        if constexpr (ERR) {
            if (a.stage == 1) a.ymid[c0 + c] = mid;
            if (a.stage == 3) {  // embedded estimate, before the forcing kick
                const cx<T> e = wn - a.ymid[c0 + c];
                const double wt = kxi == 0 ? 1.0 : 2.0;
                esum += wt * ((double)e.x * (double)e.x + (double)e.y * (double)e.y);
                ssum += wt * ((double)wn.x * (double)wn.x + (double)wn.y * (double)wn.y);
            }
        }
        if (a.stage < 3) {
            a.acc[c0 + c] = av[q];
            if constexpr (SCHEME == 0) a.stagebuf[c0 + c] = wn;
        } else {
            if constexpr (SCHEME == 0) {
                if (ph.sfd_on && ph.sfd_tau > 0.0) a.sfd[c0 + c] = fs[q];
            }
            if (ph.force_on && kxi < ph.fbx) {
                const int b = c <= kym ? jy : jy - L;
                if (b >= -ph.fby && b <= ph.fby)
                    wn = wn + sqh * a.fbox[mb * a.bf + kxi * (2 * ph.fby + 1) + (b + ph.fby)];
            }
            a.state[c0 + c] = wn;
        }
        wh[at(jy)] = wn;
    }
    if (blockIdx.x == 0 && threadIdx.x == 0 && a.stage == 3) {
        sc->t += dt;
        sc->umax2_bits = 0ull;
    }
    if constexpr (ERR) {
        // stage 3 does not run on a restoring step
        if (blockIdx.x == 0 && threadIdx.x == 0 && redo) sc->umax2_bits = 0ull;
        if (a.stage == 3) {  // workgroup sums in a fixed order
            constexpr int NW = U * L / 128;
            __shared__ double ered[2 * NW];
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
                for (int i = 0; i < NW; ++i) {
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
    unit_sync<L>();
    cx<T>* out = f < 2 ? (f == 0 ? a.mixed[0] : a.mixed[1]) : (f == 2 ? a.mixed[2] : a.mixed[3]);
    col_unit_out<T, L>(lds, wh, r, G, kxi, kx, kys, out + mb * a.bm, active, tw);
}

// The derivative fields of the state as it is (COL_PRIME), through the output passes
// of the stage kernel: a state that was uploaded, restored or primed again after
// other transforms steps on with the bits of a run that kept its fields.
template <typename T, int L, int U, int MW>
__global__ __launch_bounds__(U * L / 2, MW) void k_col_fields_prime(ColArgs<T> a) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    constexpr int UT = unit_threads<L>(), TPL = L / P, RE = unit_region<L>();
    constexpr int kym = Band<L>::kym, ncy = 2 * kym + 1;
    constexpr bool WS = ws_unit<L>();
    const int u = threadIdx.x / UT, r = threadIdx.x - u * UT;
    const int f = r / TPL, j = r - f * TPL;
    cx<T>* const lds = reinterpret_cast<cx<T>*>(smem_raw) + u * 4 * RE;
    const Geo& G = a.geo;
    const size_t mb = blockIdx.y;
    const int kxi = blockIdx.x * U + u;
    const bool active = kxi < G.nkx_keep;
    UnitTw<L, T> tw;
    load_unit_tw<L>(tw, j, a.tw);
    cx<T>* const wh = lds + (WS ? 2 * RE : RE);
#pragma unroll
    for (int q = 0; q < kUnitModes; ++q) {
        const int c = r + q * UT;
        if (c >= ncy || !active) continue;
        const int jy = c <= kym ? c : c + (L - ncy);
        wh[WS ? jy : pad(jy)] = a.state[mb * a.bc + (size_t)kxi * ncy + c];
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        DevScalars* const sc = a.sc + mb;
        sc->umax2_bits = 0ull;
        sc->pending = 0;  // a new state: nothing waits to be judged
        sc->redo = 0;
    }
    unit_sync<L>();
    cx<T>* out = f < 2 ? (f == 0 ? a.mixed[0] : a.mixed[1]) : (f == 2 ? a.mixed[2] : a.mixed[3]);
    col_unit_out<T, L>(lds, wh, r, G, kxi, T(kxi) * T(a.kxs), T(a.kys), out + mb * a.bm, active,
                       tw);
}

}  // namespace nsd
