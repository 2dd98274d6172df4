// nsd_stage.hpp -- launchers of the time-step kernels, instantiated per
// transform length (compile-time lines) and launch variant in nsd_stage.hip.
#pragma once

#include "nsd_kernels.hpp"

namespace nsd {

// number of launch variants per length (variant 0 is the default shape)
constexpr int kStageVariants = 5;
// the field-parallel kernels (nsd_fields.hpp), lines of up to kFieldsMax points
constexpr int kFieldsVariant = 3;
constexpr int kFieldsMax = 1024;
// workgroups of one wave, lines of up to 512 points
constexpr int kSmallVariant = 1;

// k_row in ROW_STAGE mode for rows of length L (power of two, 16..8192),
// `members` batch members along grid y
// (errctl: the error controller's instantiation, of the field-parallel kernels and of
// variant 0, which stands for its other workgroup sizes; force: one more workgroup
// per member makes the forcing draw a.force, not with errctl)
template <typename T>
void launch_row_stage(const RowArgs<T>& a, int L, int items, int members, int variant,
                      hipStream_t st, bool errctl = false, bool force = false);
// k_col in COL_STAGE (scheme from a.phys.scheme) or COL_PRIME mode, length L
template <typename T>
void launch_col_fused(const ColArgs<T>& a, int L, int ncols, int members, int variant,
                      hipStream_t st, bool errctl = false);
// variant that a context starts with for `lines` lines (kind 0: row pairs, 1: columns)
// of each member
template <typename T>
int stage_variant_default(int kind, int L, long lines, int members, int maxlds);
// threads of a workgroup of that row launch
template <typename T>
int row_stage_threads(int L, int variant);
// 1 if `variant` exists for length L and fits `maxlds` bytes of LDS
template <typename T>
int stage_variant_valid(int L, int variant, int maxlds);
// Variants of one length with equal values here contract the same products and give
// the same bits; -1: no such variant
template <typename T>
int stage_variant_rounding(int L, int variant);
// 1 if the stage kernels of `variant` at length L read (k_row) and write
// (k_col) the mixed fields in a layout of their own (stage_layout)
template <typename T>
int stage_variant_pairs(int L, int variant);
// the field-parallel launches (nsd_fields.hip): L <= kFieldsMax
template <typename T>
void launch_row_fields(const RowArgs<T>& a, int L, int items, int members, hipStream_t st,
                       bool errctl, bool force);
template <typename T>
void launch_col_fields(const ColArgs<T>& a, int L, int ncols, int members, hipStream_t st,
                       bool errctl);
// threads of a workgroup of theirs
constexpr int row_fields_threads(int L) { return L <= 512 ? 256 : L / 2; }
// whether they take lines of length L with `maxlds` bytes of LDS
template <typename T>
bool fields_fits(int L, int maxlds);
template <typename T>
void fields_lds_limits(int bytes);
// raise the dynamic-LDS limit of every instantiation above
template <typename T>
void stage_lds_limits(int bytes);

}  // namespace nsd
