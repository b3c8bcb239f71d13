"""How a workgroup finds its group (csrc/maya_groups.hpp), run on the host over pointers that stop at the first index out of range."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <stdio.h>
#include <stdlib.h>
#include <vector>
#define __device__
#define __forceinline__ inline
#include "maya_groups.hpp"

template <typename T> struct Checked {   // a pointer to n words
    const T* p = nullptr;
    int n = 0;
    const char* what = "";
    explicit operator bool() const { return p != nullptr; }
    const T& operator[](int i) const {
        if (i < 0 || i >= n) { printf("%s[%d] of %d\n", what, i, n); exit(1); }
        return p[i];
    }
    const T& operator*() const { return (*this)[0]; }
};
struct Args {
    int n_tokens, k;
    Checked<uint64_t> plan_ptr, grp_ptr;
    Checked<int> grp_start, grp_ent, n_groups, skip;
};
template <typename T> Checked<T> of(const std::vector<T>& v, const char* what) { return Checked<T>{v.data(), (int) v.size(), what}; }

// n_tokens x k entries, entry e on expert e % experts; entries with e % 7 == 3 on none
template <bool WHOLE> int check(int n_tokens, int k, int experts) {
    const int n = n_tokens * k;
    std::vector<uint64_t> plan(n), ptr;
    std::vector<int> start, ent, ng(1);
    for (int e = 0; e < n; ++e) plan[e] = e % 7 == 3 ? 0 : 4096 * (1 + e % experts);
    for (int x = 0; x < experts; ++x) {
        const size_t before = ent.size();
        for (int e = 0; e < n; ++e)
            if (plan[e] == 4096ull * (1 + x)) ent.push_back(e);
        if (ent.size() > before) ptr.push_back(4096 * (1 + x)), start.push_back((int) before);
    }
    start.push_back((int) ent.size());
    ng[0] = (int) ptr.size();
    const std::vector<uint64_t> want = ptr;
    const std::vector<int> first = start;
    ent.resize(n, -1);
    if (WHOLE) ptr.resize(n, 0xdead), start.resize(n + 1, -7);   // (else: arrays that end with the groups)
    Args a{n_tokens, k, of(plan, "plan_ptr"), of(ptr, "grp_ptr"), of(start, "grp_start"), of(ent, "grp_ent"), of(ng, "n_groups"), {}};
    for (int g = 0; g < n; ++g) {   // a column of the launch each
        maya::GroupRef r;
        const bool there = maya::group_of<WHOLE>(a, g, r);
        if (there != (g < ng[0])) { printf("group %d of %d: %d\n", g, ng[0], there); return 1; }
        if (there && (r.blob != want[g] || r.e0 != first[g] || r.ne != first[g + 1] - first[g])) { printf("group %d\n", g); return 1; }
        for (int i = 0; there && i < r.ne; ++i)
            if (plan[maya::entry_of(a, r, i)] != r.blob) { printf("group %d entry %d\n", g, i); return 1; }
    }
    a.grp_ptr = {};   // no groups: an entry each
    for (int g = 0; g < n + 3; ++g) {
        maya::GroupRef r;
        const bool there = maya::group_of<WHOLE>(a, g, r);
        if (there != (g < n && plan[g] != 0)) { printf("entry %d\n", g); return 1; }
    }
    return 0;
}
int main() {
    for (int t : {1, 2, 5, 16})
        for (int k : {1, 3, 16})
            for (int x : {1, 2, 11, 300})
                if (check<false>(t, k, x) || check<true>(t, k, x)) return 1;
    return 0;
}
"""


def test_no_word_outside_the_callers_arrays(tmp_path):
    """grp_ptr [groups] and grp_start [groups + 1] suffice (maya_moe_args, maya_exl3_args); a layer's own whole arrays do too."""
    src, exe = tmp_path / "groups.cpp", str(tmp_path / "groups")
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", os.path.join(ROOT, "project-maya_amd", "csrc"), str(src), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
