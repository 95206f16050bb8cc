// The column kernels' (mgg_kernels.hip) table range, slots and walk over a
// row's pixels, in one place for the device and for the host code that checks
// that no index leaves the table.
#pragma once

#include <type_traits>

#ifdef __HIP__
#include <hip/hip_runtime.h>
#define MGG_HD __host__ __device__ __forceinline__
#else
#define MGG_HD inline
#endif

namespace mgg {

enum : int { COL_BACK = 0, COL_ADJOINT = 1 };

// Index range [ct_lo, ct_hi) of the pair table.  Over all frames the pixels of
// the lists reach -563 to 1,187 for columns of up to six slab voxels and -785
// to 1,401 for up to ten transposed ones; longer columns clamp (col_clamps).
MGG_HD constexpr int ct_lo(int mode) { return mode == COL_BACK ? -576 : -800; }
MGG_HD constexpr int ct_hi(int mode) { return mode == COL_BACK ? 1200 : 1416; }

// Voxels per column (slots) for a column extent len along its axis.
MGG_HD int col_slots(int mode, float len)
{
    if (mode == COL_BACK) return len < 5.f ? 5 : len < 6.f ? 6 : 7;
    return len < 6.f ? 6 : len < 8.f ? 8 : len < 10.f ? 10 : 14;
}
MGG_HD constexpr bool col_clamps(int mode, int slots) { return mode == COL_BACK ? slots == 7 : slots > 10; }
// The same for slots looked up one by one (lanes at a half-integer index): of
// an even number the last lies 125 entries below the last pair's.
MGG_HD constexpr bool col_clamps_single(int mode, int slots) { return slots % 2 == 0 || col_clamps(mode, slots); }

// A pixel offset is listed while its distance from the column along a cross
// axis (frame components u, v) is at most this.
MGG_HD float col_list_reach(float u, float v)
{
    return 2.02f + 0.5f * (__builtin_fabsf(u) + __builtin_fabsf(v));
}

// The cnt pixels of a row from its first one on, each once and no other: up to
// six in groups of three (head, from values loaded before), then in pairs, the
// last by itself where it has no partner (tail).  The groups' sizes are types.
template <class Head, class Tail>
MGG_HD void col_row(int cnt, Head &&head, Tail &&tail)
{
    using One = std::integral_constant<int, 1>;
    using Two = std::integral_constant<int, 2>;
    using Three = std::integral_constant<int, 3>;
    using First = std::integral_constant<int, 0>;
    if (cnt >= 3) head(First{}, Three{});
    else if (cnt == 2) head(First{}, Two{});
    else if (cnt == 1) head(First{}, One{});
    if (cnt >= 6) head(Three{}, Three{});
    else if (cnt == 5) head(Three{}, Two{});
    else if (cnt == 4) head(Three{}, One{});
    for (int e = 6; e < cnt; e += 2) {
        if (e + 1 < cnt) tail(e, Two{});
        else tail(e, One{});
    }
}

}  // namespace mgg
