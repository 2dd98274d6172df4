// nsd_stage.hip -- time-step kernels instantiated for every supported
// transform length, so that all LDS addresses and strides are compile-time
// constants.  Compiled once per precision with -DNSD_T=float / double.
//
// Lengths of up to 1024 (the ensemble sizes) also get launch variants: 1, 2 and 4
// are variant 0's code in workgroups of one wave, of twice and of half the threads,
// 3 the field-parallel kernels of nsd_fields.hpp.
#include "nsd_stage.hpp"

#ifndef NSD_T
#error "NSD_T must be float or double"
#endif

namespace nsd {

namespace {

template <int L>
constexpr int nt_for() {
    return L / P > 256 ? L / P : 256;
}

// variant V of length L: threads per workgroup
template <int L, int V>
constexpr int var_nt() {
    return V == kSmallVariant ? 64 : V == 2 ? 2 * nt_for<L>() : V == 4 ? nt_for<L>() / 2 : nt_for<L>();
}
template <int L, int V>
constexpr bool var_ok() {
    return V == 0 || (V == kSmallVariant ? L / P <= 64 : L >= 64 && L <= 1024);
}

// the stage kernels' LDS (FP64 lines of 4096 take a second line region)
template <typename T, int L, int V>
size_t stage_lds() {
    constexpr int NT = var_nt<L, V>();
    constexpr int lines = NT * P / L;
    constexpr int PR = -1;
    return (size_t)lines * stage_regions<T, L, NT, PR>() * region_elems<T, L, NT, PR>() *
           sizeof(cx<T>);
}

// ERR: the error controller's instantiations (launch variant 0 only)
template <typename T, int LOG, int V, bool ERR = false>
void row_stage_LV(const RowArgs<T>& a, int items, int members, hipStream_t st,
                  bool force = false) {
    constexpr int L = 1 << LOG;
    if constexpr (V == kFieldsVariant) {
        if constexpr (L <= kFieldsMax) launch_row_fields<T>(a, L, items, members, st, force);
    } else if constexpr (var_ok<L, V>()) {
        constexpr int NT = var_nt<L, V>();
        constexpr int PR = -1;
        constexpr int lines = NT * P / L;
        const int blocks = (items + lines - 1) / lines;
        const size_t lds = stage_lds<T, L, V>();
        if constexpr (!ERR) {
            if (force) {
                hipLaunchKernelGGL((k_row<T, NT, ROW_STAGE, L, PR, false, min_waves<T>(), true>),
                                   dim3(blocks + 1, members), dim3(NT), lds, st, a);
                return;
            }
        }
        hipLaunchKernelGGL((k_row<T, NT, ROW_STAGE, L, PR, ERR>), dim3(blocks, members), dim3(NT),
                           lds, st, a);
    }
}

template <typename T, int LOG, int V, bool ERR = false>
void col_fused_LV(const ColArgs<T>& a, int ncols, int members, hipStream_t st) {
    constexpr int L = 1 << LOG;
    if constexpr (V == kFieldsVariant) {
        if constexpr (L <= kFieldsMax) launch_col_fields<T>(a, L, ncols, members, st);
    } else if constexpr (var_ok<L, V>()) {
        constexpr int NT = var_nt<L, V>();
        constexpr int PR = -1;
        constexpr int lines = NT * P / L;
        const int blocks = (ncols + lines - 1) / lines;
        const dim3 grid(blocks, members);
        const size_t lds = stage_lds<T, L, V>();
        if (a.mode == COL_PRIME)
            hipLaunchKernelGGL((k_col<T, NT, COL_PRIME, 0, L, PR>), grid, dim3(NT), lds, st, a);
        else if (a.phys.scheme == 0)
            hipLaunchKernelGGL((k_col<T, NT, COL_STAGE, 0, L, PR, ERR>), grid, dim3(NT), lds, st,
                               a);
        else
            hipLaunchKernelGGL((k_col<T, NT, COL_STAGE, 1, L, PR, ERR>), grid, dim3(NT), lds, st,
                               a);
    }
}

template <typename K>
void lds_attr(K kernel, int bytes) {
    (void)hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                              bytes);
}

template <typename T, int LOG, int V>
void limits_LV(int bytes) {
    constexpr int L = 1 << LOG;
    if constexpr (var_ok<L, V>() && V != kFieldsVariant) {
        constexpr int NT = var_nt<L, V>();
        constexpr int PR = -1;
        lds_attr(k_row<T, NT, ROW_STAGE, L, PR>, bytes);
        lds_attr(k_row<T, NT, ROW_STAGE, L, PR, false, min_waves<T>(), true>, bytes);
        lds_attr(k_col<T, NT, COL_PRIME, 0, L, PR>, bytes);
        lds_attr(k_col<T, NT, COL_STAGE, 0, L, PR>, bytes);
        lds_attr(k_col<T, NT, COL_STAGE, 1, L, PR>, bytes);
        if constexpr (V == 0) {
            lds_attr(k_row<T, NT, ROW_STAGE, L, PR, true>, bytes);
            lds_attr(k_col<T, NT, COL_STAGE, 0, L, PR, true>, bytes);
            lds_attr(k_col<T, NT, COL_STAGE, 1, L, PR, true>, bytes);
        }
    }
}

template <typename T, int LOG, int V>
int var_pairs() {
    constexpr int L = 1 << LOG;
    if constexpr (V != kFieldsVariant && var_ok<L, V>()) return stage_layout<T, L, var_nt<L, V>(), -1>() ? 1 : 0;
    return 0;
}

// -1: no such variant, 0: transforms one at a time, 1: in lock-step pairs, 2: field-parallel
template <typename T, int LOG, int V>
int var_rounding() {
    constexpr int L = 1 << LOG;
    if constexpr (V == kFieldsVariant) return L <= kFieldsMax ? 2 : -1;
    else if constexpr (var_ok<L, V>()) return paired_lines<T, L, var_nt<L, V>(), -1>() ? 1 : 0;
    return -1;
}

template <typename T, int LOG, int V>
int var_valid(int maxlds) {
    constexpr int L = 1 << LOG;
    if constexpr (V == kFieldsVariant) return fields_fits<T>(L, maxlds) ? 1 : 0;
    else if constexpr (var_ok<L, V>())
        return stage_lds<T, L, V>() <= (size_t)maxlds ? 1 : 0;
    return 0;
}

template <typename T, int LOG, int V>
int row_threads() {
    constexpr int L = 1 << LOG;
    if constexpr (V == kFieldsVariant) return row_fields_threads(L);
    else if constexpr (var_ok<L, V>()) return var_nt<L, V>();
    return 0;
}

int log2i(int L) {
    int l = 0;
    while ((1 << l) < L) ++l;
    return l;
}

}  // namespace

#define NSD_FOR_LOGS(X) X(4) X(5) X(6) X(7) X(8) X(9) X(10) X(11) X(12) X(13)
#define NSD_FOR_VARS(X, n) X(n, 0) X(n, 1) X(n, 2) X(n, 3) X(n, 4)

template <typename T>
void launch_row_stage(const RowArgs<T>& a, int L, int items, int members, int variant,
                      hipStream_t st, bool errctl, bool force) {
    const int lg = log2i(L);
    if (errctl) {
#define E_(n) \
    if (lg == n) return row_stage_LV<T, n, 0, true>(a, items, members, st);
        NSD_FOR_LOGS(E_)
#undef E_
        return;
    }
#define V_(n, v) \
    if (lg == n && variant == v) return row_stage_LV<T, n, v>(a, items, members, st, force);
#define X(n) NSD_FOR_VARS(V_, n)
    NSD_FOR_LOGS(X)
#undef X
#undef V_
}

template <typename T>
void launch_col_fused(const ColArgs<T>& a, int L, int ncols, int members, int variant,
                      hipStream_t st, bool errctl) {
    const int lg = log2i(L);
    if (errctl && a.mode == COL_STAGE) {
#define E_(n) \
    if (lg == n) return col_fused_LV<T, n, 0, true>(a, ncols, members, st);
        NSD_FOR_LOGS(E_)
#undef E_
        return;
    }
#define V_(n, v) \
    if (lg == n && variant == v) return col_fused_LV<T, n, v>(a, ncols, members, st);
#define X(n) NSD_FOR_VARS(V_, n)
    NSD_FOR_LOGS(X)
#undef X
#undef V_
}

template <typename T>
int stage_variant_valid(int L, int variant, int maxlds) {
    const int lg = log2i(L);
#define V_(n, v) \
    if (lg == n && variant == v) return var_valid<T, n, v>(maxlds);
#define X(n) NSD_FOR_VARS(V_, n)
    NSD_FOR_LOGS(X)
#undef X
#undef V_
    return 0;
}

template <typename T>
int stage_variant_pairs(int L, int variant) {
    const int lg = log2i(L);
#define V_(n, v) \
    if (lg == n && variant == v) return var_pairs<T, n, v>();
#define X(n) NSD_FOR_VARS(V_, n)
    NSD_FOR_LOGS(X)
#undef X
#undef V_
    return 0;
}

template <typename T>
int stage_variant_rounding(int L, int variant) {
    const int lg = log2i(L);
#define V_(n, v) \
    if (lg == n && variant == v) return var_rounding<T, n, v>();
#define X(n) NSD_FOR_VARS(V_, n)
    NSD_FOR_LOGS(X)
#undef X
#undef V_
    return -1;
}
template int stage_variant_rounding<NSD_T>(int, int);

template <typename T>
int row_stage_threads(int L, int variant) {
    const int lg = log2i(L);
#define V_(n, v) \
    if (lg == n && variant == v) return row_threads<T, n, v>();
#define X(n) NSD_FOR_VARS(V_, n)
    NSD_FOR_LOGS(X)
#undef X
#undef V_
    return 0;
}
template int row_stage_threads<NSD_T>(int, int);

template <typename T>
void stage_lds_limits(int bytes) {
#define V_(n, v) limits_LV<T, n, v>(bytes);
#define X(n) NSD_FOR_VARS(V_, n)
    NSD_FOR_LOGS(X)
#undef X
#undef V_
    fields_lds_limits<T>(bytes);
}

template void launch_row_stage<NSD_T>(const RowArgs<NSD_T>&, int, int, int, int, hipStream_t,
                                      bool, bool);
template void launch_col_fused<NSD_T>(const ColArgs<NSD_T>&, int, int, int, int, hipStream_t,
                                      bool);

// workgroups of the default column launch over ncols columns of length L
// (the number of partials the error controller's last stage leaves)
template <typename T>
int col_fused_blocks(int L, int ncols) {
    const int NT = L / P > 256 ? L / P : 256;
    const int lines = NT * P / L;
    return (ncols + lines - 1) / lines;
}
template int col_fused_blocks<NSD_T>(int, int);
// Variant a context starts with, for `lines` lines (row pairs, kind 0, or kept
// columns, kind 1, times batch members) of length L on a grid whose longer side is
// `side`.  `waves`: what variant 0 would launch (the device holds 1024 SIMDs).
//
// Launches that leave at most one wave per SIMD take the field-parallel kernels
// or, on FP32 grids below 512^2, variant 0's own code in the smallest workgroups.
// us per RK4 step of one field, variant 0 -> smallest workgroups -> field-parallel:
//   64^2 FP64 72 -> 56 -> 49, 512^2 FP64 120 -> - -> 69, 1024^2 FP64 188 -> 172 -> 149,
//   256^2 FP32 98 -> 81 -> 67, 512^2 FP32 103 -> 85 -> 71, 1024^2 FP32 140 -> 130 -> 124.
// The small FP32 grids keep variant 0's code because its rounding is theirs: a
// step's difference of one FP32 rounding grows to 2e-5 of the field within 400
// forced steps at 256^2, and runs, batch members and restarts of these sizes are
// compared with one another bit for bit.  Lines of 2048 stay with variant 0: a
// unit is 1024 threads there, one to a compute unit at FP64, and 256 row pairs
// take 22.0 us against 20.9 us.
//
// Larger launches (us per step; 0, fields, 4: variant 0, field-parallel, half-size
// workgroups, of the rows or columns named, variant 0 for the others):
//   FP64 rows: 512 x 16 members 0 310.5, fields 288.9, 4 303.2; 1024 x 24 2073, 1801,
//     1985; 256 x 100 442.6, 439.3, 418.5; 128 x 300 318.0, 343.2, 308.7.
//   FP64 columns: 128 x 300 318.0, 297.5, 320.2; 256 x 300 1249, 1185, 1210; 512 x 80
//     1411, 1346, 1356; 2048 x 1024 grid, classic scheme 233.0, 261.5, 219.0,
//     integrating factor 226.5, 226.5, 212.2; 4096 x 1024 473.7, 511.3, 465.1.
//   FP32 rows: 1024 x 4 192.6, 189.7, 190.1; 1024 x 8 311.0, 321.9, 311.2; 512 x 8
//     129.9, 133.2, 132.2.
//   FP32 columns: 512 x 8 129.9, 116.0, 126.4; 512 x 24 217.6, 211.5, 209.2; 1024 x 2
//     154.6, 149.1, 146.5; 1024 x 16 566.8, 632.5, 552.6.
//   FP32 below 512^2, both with variant 4: 256 x 32 126.8 -> 121.0, 128 x 120 121.9 -> 114.7.
template <typename T>
int stage_variant_default(int kind, int L, long lines, int side, int maxlds) {
    const long waves = lines * (L / P) / 64;
    if (L > kFieldsMax) return 0;
    const bool many = waves > 1024;
    if (L < 64 && many) return 0;
    const int half = stage_variant_valid<T>(L, 4, maxlds) ? 4 : 0;
    if (sizeof(T) == 4 && side < 512) return many ? half : kSmallVariant;
    bool fields;
    if (sizeof(T) == 8) fields = !many || (kind == 0 ? L >= 512 : L <= 512);
    else fields = waves <= (kind == 0 ? (L == 1024 ? 4096 : 1024) : (L == 512 ? 2048 : 1024));
    if (fields) return fields_fits<T>(L, maxlds) ? kFieldsVariant : 0;
    return sizeof(T) == 8 || kind == 1 ? half : 0;
}
template int stage_variant_default<NSD_T>(int, int, long, int, int);
template int stage_variant_valid<NSD_T>(int, int, int);
template int stage_variant_pairs<NSD_T>(int, int);
template void stage_lds_limits<NSD_T>(int);

}  // namespace nsd
