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

// the stage kernels' LDS (FP64 lines of 2048 and 4096 take a second line region)
template <typename T, int L, int V>
size_t stage_lds() {
    constexpr int NT = var_nt<L, V>();
    constexpr int lines = NT * P / L;
    return (size_t)lines * stage_regions<T, L, NT>() * region_elems<T, L, NT>() *
           sizeof(cx<T>);
}

// ERR: the error controller's instantiations (variants 0 and 3)
template <typename T, int LOG, int V, bool ERR = false>
void row_stage_LV(const RowArgs<T>& a, int items, int members, hipStream_t st,
                  bool force = false) {
    constexpr int L = 1 << LOG;
    if constexpr (V == kFieldsVariant) {
        if constexpr (L <= kFieldsMax) launch_row_fields<T>(a, L, items, members, st, ERR, force);
    } else if constexpr (var_ok<L, V>()) {
        constexpr int NT = var_nt<L, V>();
        constexpr int lines = NT * P / L;
        const int blocks = (items + lines - 1) / lines;
        const size_t lds = stage_lds<T, L, V>();
        const dim3 grid(blocks + (force && !ERR ? 1 : 0), members), nt(NT);
        auto go = [&](auto tiles) {
            constexpr bool TI = decltype(tiles)::value;
            constexpr int MW = min_waves<T>();
            if constexpr (!ERR) {
                if (force) {
                    hipLaunchKernelGGL((k_row<T, NT, ROW_STAGE, L, false, MW, true, TI>), grid, nt,
                                       lds, st, a);
                    return;
                }
            }
            hipLaunchKernelGGL((k_row<T, NT, ROW_STAGE, L, ERR, MW, false, TI>), grid, nt, lds, st,
                               a);
        };
        // kernels of their own: as branches of one the tiles' loads lose their hint, or
        // the step 0.5 % (FP64 4096^2)
        if constexpr (ws_lines64<T, L, NT>()) {
            if (!a.pairs) return go(std::false_type{});
        }
        go(std::true_type{});
    }
}

template <typename T, int LOG, int V, bool ERR = false>
void col_fused_LV(const ColArgs<T>& a, int ncols, int members, hipStream_t st) {
    constexpr int L = 1 << LOG;
    if constexpr (V == kFieldsVariant) {
        if constexpr (L <= kFieldsMax) launch_col_fields<T>(a, L, ncols, members, st, ERR);
    } else if constexpr (var_ok<L, V>()) {
        constexpr int NT = var_nt<L, V>();
        constexpr int lines = NT * P / L;
        const int blocks = (ncols + lines - 1) / lines;
        const dim3 grid(blocks, members);
        const size_t lds = stage_lds<T, L, V>();
        if (a.mode == COL_PRIME)
            hipLaunchKernelGGL((k_col<T, NT, COL_PRIME, 0, L>), grid, dim3(NT), lds, st, a);
        else if (a.phys.scheme == 0)
            hipLaunchKernelGGL((k_col<T, NT, COL_STAGE, 0, L, ERR>), grid, dim3(NT), lds, st,
                               a);
        else
            hipLaunchKernelGGL((k_col<T, NT, COL_STAGE, 1, L, ERR>), grid, dim3(NT), lds, st,
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
        constexpr int MW = min_waves<T>();
        lds_attr(k_row<T, NT, ROW_STAGE, L>, bytes);
        lds_attr(k_row<T, NT, ROW_STAGE, L, false, MW, true>, bytes);
        if constexpr (ws_lines64<T, L, NT>()) {
            lds_attr(k_row<T, NT, ROW_STAGE, L, false, MW, false, false>, bytes);
            lds_attr(k_row<T, NT, ROW_STAGE, L, false, MW, true, false>, bytes);
            lds_attr(k_row<T, NT, ROW_STAGE, L, true, MW, false, false>, bytes);
        }
        lds_attr(k_col<T, NT, COL_PRIME, 0, L>, bytes);
        lds_attr(k_col<T, NT, COL_STAGE, 0, L>, bytes);
        lds_attr(k_col<T, NT, COL_STAGE, 1, L>, bytes);
        if constexpr (V == 0) {
            lds_attr(k_row<T, NT, ROW_STAGE, L, true>, bytes);
            lds_attr(k_col<T, NT, COL_STAGE, 0, L, true>, bytes);
            lds_attr(k_col<T, NT, COL_STAGE, 1, L, true>, bytes);
        }
    }
}

template <typename T, int LOG, int V>
int var_pairs() {
    constexpr int L = 1 << LOG;
    if constexpr (V != kFieldsVariant && var_ok<L, V>()) return stage_layout<T, L, var_nt<L, V>()>() ? 1 : 0;
    return 0;
}

// -1: no such variant, 0: transforms one at a time, 1: in lock-step pairs, 2: field-parallel
template <typename T, int LOG, int V>
int var_rounding() {
    constexpr int L = 1 << LOG;
    if constexpr (V == kFieldsVariant) return L <= kFieldsMax ? 2 : -1;
    else if constexpr (var_ok<L, V>()) return paired_lines<T, L, var_nt<L, V>()>() ? 1 : 0;
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
    if (lg == n && variant == kFieldsVariant) \
        return row_stage_LV<T, n, kFieldsVariant, true>(a, items, members, st); \
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
    if (lg == n && variant == kFieldsVariant) \
        return col_fused_LV<T, n, kFieldsVariant, true>(a, ncols, members, st); \
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

// Variant a context starts with, for `members` times `lines` lines (row pairs, kind 0,
// or kept columns, kind 1) of length L.
//
// Whether the field-parallel kernels or variant 0's code (in one workgroup size or
// another) run a grid decides its rounding, so it follows the grid and the precision
// alone: batch members have the bits of a single run.  FP64 takes the field-parallel
// kernels where one field's launch leaves at most one wave per SIMD (`one`, the waves of
// variant 0; the device holds 1024 SIMDs), and where they are the faster ones past that.
// us per RK4 step, variant 0 / its fastest workgroups / field-parallel, FP64 members of
//   64^2: 1 member 70 / 54 / 41, 64 76 / 67 / 55, 260 113 / 108 / 116
//   128^2: 1 91 / 64 / 49, 60 125 / 119 / 121, 200 254 / 201 / 226
//   256^2: 1 100 / 69 / 50, 64 290 / 260 / 262, 200 875 / 835 / 876
//   512^2: 1 116 / 82 / 61, 8 190 / 172 / 165, 64 1171 / 1061 / 1026
//   1024^2: 1 180 / 167 / 139, 8 664 / 603 / 555, 24 2078 / 1879 / 1709
// and rows of one field: 1024 x 2048 209 / 209 / 193, 512 x 4096 201 / 201 / 196, 256 x 8192
// 411 / 411 / 422; columns: 2048 x 1024 225 / 211 / 225, 4096 x 512 217 / 209 / 218.  Lines of
// 2048 stay with variant 0: a unit is 1024 threads there, one to a compute unit, and 256
// row pairs take 22.0 us against 20.9 us.
//
// FP32 does without them.  A single field would gain (512^2 82 / 63 / 49, 1024^2 118 / 110 /
// 96), but batches lose against variant 0 (512^2 x 16 160 / 151 / 168, x 64 471 / 457 / 534;
// 1024^2 x 16 544 / 531 / 659), and one rounding grows to 2e-5 of the field within 400
// forced steps at 256^2.
//
// Workgroups of variant 0's code (us per step, one-wave ones, half-size from 1024 points):
//   FP32 both kinds, 32^2 x 600 members 81 -> 61, 64^2 x 16 57 -> 47, x 260 76 -> 78, x 2000
//     219 -> 199, 128^2 x 200 147 -> 128, 256^2 x 200 369 -> 337;
//   columns of 512 512^2 x 24 214 -> 195, 4096 x 512 152 -> 144; of 1024 1024^2 x 64 2321 ->
//     2245, 8192 x 1024 396 -> 385, FP64 2048 x 1024 225 -> 211;
//   rows of 512 512^2 x 1 82 -> 76, x 8 128 -> 132, 512 x 4096 145 -> 162; of 1024 1024^2 x 1
//     118 -> 116, x 64 2321 -> 2374, 1024 x 4096 213 -> 219: up to one wave per SIMD;
//   shorter rows of tall grids 64 x 1024 74 -> 59 (with its columns), 128 x 8192 170 -> 175,
//     256 x 8192 197 -> 212: up to half a wave per SIMD from one field.
template <typename T>
int stage_variant_default(int kind, int L, long lines, int members, int maxlds) {
    const long one = lines * (L / P) / 64;
    if (L > kFieldsMax) return 0;
    if (sizeof(T) == 8) {
        if ((one <= 1024 || (kind == 0 ? L >= 512 : L <= 512)) && fields_fits<T>(L, maxlds))
            return kFieldsVariant;
        return kind == 1 && L == 1024 ? 4 : 0;
    }
    if (kind == 0 && (L >= 512 ? one * members > 1024 : one > 512)) return 0;
    return L == 1024 ? 4 : kSmallVariant;
}
template int stage_variant_default<NSD_T>(int, int, long, int, int);
template int stage_variant_valid<NSD_T>(int, int, int);
template int stage_variant_pairs<NSD_T>(int, int);
template void stage_lds_limits<NSD_T>(int);

}  // namespace nsd
