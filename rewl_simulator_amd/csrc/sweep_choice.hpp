// Which contexts the sixteen-lanes-a-walker sweep of integer energies
// (sweep_tree.hpp) takes from the kernels with one lane per walker.  No HIP, so
// that a host compiler can test it.
#pragma once

namespace rewl {

// Walkers of a context up to which it may take a system; four are a workgroup,
// 1024 of which are four per CU.  More share the CU's four SIMDs, its time per
// attempt grows with them, and the kernels with one lane per walker still have
// room.  Measured, cycles per attempt, this kernel against one lane:
//  * sizes with an unrolled row: L = 64 Ising 124 / 160 at 4096 walkers, 152 /
//    164 at 5120, 246 / 168 at 6144; L = 16 172 / 176, 24 161 / 168, 48 148 / 168
//    at 5120; Ashkin-Teller 159-201 / 194-218 at 5120, 236 / 198 at 6144.  L = 32
//    Ising, the shortest rows that meet their producer after every one, 124 /
//    162 at 4096 and 164 / 163 at 4352.
//  * other sizes: 225 / 500 at L = 42 with 8192, at L = 10 481 / 517 (Ashkin-
//    Teller 581 / 586) with 12288.  The fewer a row's blocks, the more of the time
//    is the row's own: L = 9 461 / 521 (547 / 597) with 10240, 530 / 521 (644 /
//    597) with 12288; L = 5 346 / 565 (448 / 681) with 6144, 588 / 565 (743 / 680)
//    with 7168.
//  * observables: the sums take the LDS of the walkers that would share a CU.
//    L = 16 Ashkin-Teller, moments, 688 / 810 at 4096 and 858 / 845 at 5120.
inline int tree_walker_limit(int planes, int L, int observables, bool unrolled) {
    if (observables) return 4096;
    if (unrolled) return planes == 1 && L == 32 ? 4096 : 5120;
    return L >= 10 ? 12288 : L >= 7 ? 10240 : 6144;
}

// How many workgroups of so many bytes of LDS a CU holds, and in how many
// rounds the chip takes `groups` of them.
inline long long workgroups_per_cu(long long lds, long long lds_max) {
    return lds > 0 && lds < lds_max ? lds_max / lds : 1;
}
inline long long workgroup_rounds(long long groups, long long lds, long long lds_max, int cus) {
    const long long at_once = cus * workgroups_per_cu(lds, lds_max);
    return (groups + at_once - 1) / at_once;
}

// Whether it is the faster one for systems with an unrolled row, when windows
// are so wide that LDS decides how many workgroups run at once.  A round of it
// takes about 3/4 of the time of one lane's, with moments 3/5, with correlators
// 1/3; of workgroups that have their CU to themselves 2/3, 1/2, 1/3.  Measured,
// cycles per attempt, this kernel against one lane, by rounds: L = 64
// Ashkin-Teller, 540 bins, 4096 walkers 260 / 190 (2 to 1); L = 64 Ising, 1171
// bins 220 / 319 (2 to 2); with moments 217 bins 322 / 268 (2 to 1) and 586 bins
// 539 / 871 (4 to 3, alone), L = 32 Ashkin-Teller 69 bins 784 / 709 (2 to 1);
// with correlators 217 bins 412 / 640 (2 to 1).
inline bool tree_pays(int observables, long long tree_rounds, bool alone, long long lane_rounds) {
    const int lane[2][3] = {{4, 5, 3}, {3, 2, 3}}, tree[2][3] = {{3, 3, 1}, {2, 1, 1}};
    return tree_rounds * tree[alone][observables] <= lane_rounds * lane[alone][observables];
}

}  // namespace rewl
