// nsd_fields.hip -- launches of the field-parallel stage kernels for every line
// length they take.  Compiled once per precision with -DNSD_T=float / double.
#include "nsd_fields.hpp"

#include "nsd_stage.hpp"

#ifndef NSD_T
#error "NSD_T must be float or double"
#endif

namespace nsd {

namespace {

// whole units of L / 2 threads in workgroups of 256 where they fit
template <int L>
constexpr int fields_units() { return row_fields_threads(L) / (L / 2); }
// occupancy floor (waves per SIMD): what the lines' LDS leaves room for, and at
// FP64 the register budget that the rows of up to 512 points need
template <typename T, int L>
constexpr int fields_mw() { return sizeof(T) == 8 && L <= 512 ? 3 : 4; }
template <typename T, int L>
constexpr size_t fields_lds() {
    return (size_t)fields_units<L>() * 4 * unit_region<L>() * sizeof(cx<T>);
}

template <typename T, int L>
void row_fields(const RowArgs<T>& a, int items, int members, hipStream_t st, bool errctl,
                bool force) {
    constexpr int U = fields_units<L>();
    constexpr int MW = fields_mw<T, L>();
    const dim3 grid((items + U - 1) / U + (force ? 1 : 0), members), nt(U * L / 2);
    const size_t lds = fields_lds<T, L>();
    if (errctl)
        hipLaunchKernelGGL((k_row_fields<T, L, U, MW, false, true>), grid, nt, lds, st, a);
    else if (force)
        hipLaunchKernelGGL((k_row_fields<T, L, U, MW, true, false>), grid, nt, lds, st, a);
    else
        hipLaunchKernelGGL((k_row_fields<T, L, U, MW, false, false>), grid, nt, lds, st, a);
}

template <typename T, int L>
void col_fields(const ColArgs<T>& a, int ncols, int members, hipStream_t st, bool errctl) {
    constexpr int U = fields_units<L>(), MW = fields_mw<T, L>();
    const dim3 grid((ncols + U - 1) / U, members), nt(U * L / 2);
    const size_t lds = fields_lds<T, L>();
    if (a.mode == COL_PRIME)
        hipLaunchKernelGGL((k_col_fields_prime<T, L, U, MW>), grid, nt, lds, st, a);
    else if (errctl && a.phys.scheme == 0)
        hipLaunchKernelGGL((k_col_fields<T, L, 0, U, MW, true>), grid, nt, lds, st, a);
    else if (errctl)
        hipLaunchKernelGGL((k_col_fields<T, L, 1, U, MW, true>), grid, nt, lds, st, a);
    else if (a.phys.scheme == 0)
        hipLaunchKernelGGL((k_col_fields<T, L, 0, U, MW, false>), grid, nt, lds, st, a);
    else
        hipLaunchKernelGGL((k_col_fields<T, L, 1, U, MW, false>), grid, nt, lds, st, a);
}

template <typename K>
void lds_attr(K kernel, int bytes) {
    (void)hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                              bytes);
}

template <typename T, int L>
void limits(int bytes) {
    constexpr int U = fields_units<L>(), MW = fields_mw<T, L>();
    lds_attr(k_row_fields<T, L, U, MW, false, false>, bytes);
    lds_attr(k_row_fields<T, L, U, MW, true, false>, bytes);
    lds_attr(k_row_fields<T, L, U, MW, false, true>, bytes);
    lds_attr(k_col_fields_prime<T, L, U, MW>, bytes);
    lds_attr(k_col_fields<T, L, 0, U, MW, false>, bytes);
    lds_attr(k_col_fields<T, L, 1, U, MW, false>, bytes);
    lds_attr(k_col_fields<T, L, 0, U, MW, true>, bytes);
    lds_attr(k_col_fields<T, L, 1, U, MW, true>, bytes);
}

}  // namespace

#define NSD_FOR_FIELDS(X) X(16) X(32) X(64) X(128) X(256) X(512) X(1024)
static_assert(kFieldsMax == 1024, "the lengths above");

template <typename T>
void launch_row_fields(const RowArgs<T>& a, int L, int items, int members, hipStream_t st,
                       bool errctl, bool force) {
#define X(n) \
    if (L == n) return row_fields<T, n>(a, items, members, st, errctl, force);
    NSD_FOR_FIELDS(X)
#undef X
}

template <typename T>
void launch_col_fields(const ColArgs<T>& a, int L, int ncols, int members, hipStream_t st,
                       bool errctl) {
#define X(n) \
    if (L == n) return col_fields<T, n>(a, ncols, members, st, errctl);
    NSD_FOR_FIELDS(X)
#undef X
}

template <typename T>
bool fields_fits(int L, int maxlds) {
#define X(n) \
    if (L == n) return fields_lds<T, n>() <= (size_t)maxlds;
    NSD_FOR_FIELDS(X)
#undef X
    return false;
}

template <typename T>
void fields_lds_limits(int bytes) {
#define X(n) limits<T, n>(bytes);
    NSD_FOR_FIELDS(X)
#undef X
}

template void launch_row_fields<NSD_T>(const RowArgs<NSD_T>&, int, int, int, hipStream_t, bool,
                                       bool);
template void launch_col_fields<NSD_T>(const ColArgs<NSD_T>&, int, int, int, hipStream_t, bool);
template bool fields_fits<NSD_T>(int, int);
template void fields_lds_limits<NSD_T>(int);

}  // namespace nsd
