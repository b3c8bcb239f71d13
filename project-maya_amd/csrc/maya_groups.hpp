// maya_groups.hpp - which entries a workgroup's group holds.  Over any argument structure with the grouping's fields
// (maya_moe_args, maya_exl3_args) and any pointer-like types in it, so that a host program can run it over checked ones.
#pragma once

#include <stdint.h>

namespace maya {

struct GroupRef {
    uint64_t blob;
    int e0, ne;          // entries [e0, e0 + ne) of grp_ent (or the single entry e0 when grp_ptr is null)
};
// A launch has a column of workgroups for every group there can be (tokens * k); how many there are, only the device knows.
// A caller's arrays may end with its groups (grp_ptr [groups], grp_start [groups + 1]), so the count is compared first and
// the group's words wait for it.  WHOLE: the arrays have a word for every entry (grp_ptr [tokens * k], grp_start
// [tokens * k + 1] - a layer's own workspace), all is asked for at once and what lies behind the last group is dropped.
template <bool WHOLE, typename Args>
__device__ __forceinline__ bool group_of(const Args& a, int g, GroupRef& r) {
    if (a.skip && *a.skip) return false;
    if (a.grp_ptr) {
        if constexpr (WHOLE) {
            const int ng = *a.n_groups, end = a.grp_start[g + 1];
            r.blob = a.grp_ptr[g];
            r.e0 = a.grp_start[g];
            r.ne = end - r.e0;
            if (g >= ng) return false;
        } else {
            if (g >= *a.n_groups) return false;
            r.blob = a.grp_ptr[g];
            r.e0 = a.grp_start[g];
            r.ne = a.grp_start[g + 1] - r.e0;
        }
    } else {
        if (g >= a.n_tokens * a.k) return false;
        r.blob = a.plan_ptr[g];
        r.e0 = g;
        r.ne = 1;
    }
    return r.blob != 0ull && r.ne > 0;
}
template <typename Args> __device__ __forceinline__ int entry_of(const Args& a, const GroupRef& r, int i) {
    return a.grp_ptr ? a.grp_ent[r.e0 + i] : r.e0;
}

}  // namespace maya
