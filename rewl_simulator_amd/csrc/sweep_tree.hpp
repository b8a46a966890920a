// Wang-Landau sweep, Philox mode, integer energies, a few thousand walkers at
// most: sixteen lanes per walker.
//
// Same chain, same draws and the same FP64 ln g arithmetic as k_sweep (the
// reference's wang_landau_update, wang_landau.hpp:49-93).  With one lane per
// walker the chip is mostly idle and a walker's time per attempt is the length
// of one wavefront's instruction stream plus an LDS read on its dependency
// chain (158 cycles an attempt at L = 64).  Here a walker has a row of sixteen
// lanes and takes four attempts at a time: the outcomes of four successive
// attempts are a binary tree of fifteen decisions, each lane makes one of
// them under the hypothesis that the attempts before it ended as its place in
// the tree says, and the walk from the root along the decisions gives what
// the four attempts in order give.  One LDS read latency and one state
// hand-over are paid per four attempts instead of per attempt.
//
// A lane's node n (heap order: root 1, children 2n and 2n + 1) has depth t =
// 0..3; bit a_i of n's path is the assumed outcome of attempt i < t.
//
//  * Row prologue: lane j of a walker's row takes block j (sites 4j..4j+3) of
//    the lattice row, whose neighbours above, below and to the right are
//    final (held in registers), and writes the energy changes of its four sites as signed bytes,
//    for the left neighbour as it stands and flipped.  The lattice is kept in
//    LDS as one nibble per byte, so a block is a byte.
//  * A node picks its path's four bytes with one v_perm_b32 and gets its
//    current and proposed state with one v_dot4_i32_i8 each: the state u is
//    the LDS byte offset of ln g at the walker's energy (energy x pitch / bin,
//    so the bin's slot is u with the low bits masked).
//  * The increments of the path's earlier attempts are applied to the two
//    ln g values in registers: one masked add of ln f for each earlier state
//    in the same bin (the adds are all of the same ln f, so their order does
//    not matter and the sums round as in sequence).
//  * Guard bins hold ln g = +inf and reach four proposals beyond the window,
//    so every hypothetical state is a valid slot, and one outside the window
//    is rejected by the comparison itself.
//  * The lanes on the walked path add ln f and a count to the bin after their
//    attempt; the last one hands the state and the step's flips over to its
//    row through an LDS word per block.
//
// With observables the hand-over carries the magnetisations too, a node gets
// its own by two more dot products, and the lanes on the path add their moments
// to the bin's sums in LDS (added to HBM after the launch).  A correlator sample
// (every 1000th update of a bin) is queued by its lane and taken at the end of
// the row by the whole wavefront, one lattice row per lane.
//
// The acceptance bounds come from a producer wavefront (accept_bound.hpp), a
// segment of rows ahead, one barrier per segment.
//
// What bounds it: the instruction stream of one wavefront (about 5 cycles an
// instruction when it has its SIMD to itself) and two LDS round trips per four
// attempts.  Of the 440 cycles of a step the sixteen instructions of the
// increments take 85, the FP64 atomic 50 and the count 25; a row adds 320.
// Measured, cycles per attempt per walker, one lane a walker -> this kernel:
// L = 64 Ising, 2048 walkers 158 -> 110 (270 -> 190 ms per 1000 sweeps); L = 16,
// 8 walkers 253 -> 130; L = 42, 256 walkers (row kernel) 493 -> 112; L = 32
// Ashkin-Teller, 512 walkers 196 -> 128.  A workgroup has one walker wavefront:
// two (four) behind one barrier wait for each other and cost 114 at 2048 (137
// at 4096) where one costs 110 (123); a second producer gained nothing.  With the
// four, steps of three attempts cost 107 by the same count and of two 126.  With observables = 1, one lane a walker -> this
// kernel: L = 64 Ising 273 -> 157 with 2048 walkers; L = 30 1012 -> 163; L = 32
// Ashkin-Teller 798 -> 298.  With 2: L = 64 Ising 620 -> 197 (the samples 23 of
// 172 with 256 walkers), L = 30 2700 -> 191, Ashkin-Teller L = 32
// 1256 -> 353, L = 20 4200 -> 381.  The spin flips as an LDS exclusive-or on the path
// and the state hand-over before the updates measured no better.
#pragma once
#include <type_traits>

#include "accept_bound.hpp"
#include "device.hpp"
#include "sweep_tuned.hpp"

namespace rewl {

constexpr int kTreeLanes = 16;      // lanes per walker
constexpr int kTreePerWave = 4;     // walkers per wavefront
constexpr int kTreeMaxDepth = 4;    // attempts per step
constexpr int kTreeMinL = 5;        // the first and the last block of a row differ

// Byte scale of one system's states and energy changes (host: tree_scale).
struct TreeScale {
    int32_t pitch;   // bytes of one ln g bin row in LDS (power of two, >= the bin size)
    int32_t g;       // every energy change is a multiple of g
    int32_t m;       // stored byte = energy change / g * m
    int32_t w;       // state bytes per stored unit: w m = pitch g / bin
    int32_t guard;   // guard bins on each side
};

// LDS of one workgroup: four walkers (offsets in bytes).
struct TreeLds {
    int32_t rowb, lat, ring, ringw, rec, queue, cnt, lng, sums, total;
};

// Per walker: 16 records of a row's blocks and the last one's alternative,
// then 16 state words, one per block, and a sink of the same size for the lanes
// that do not end a step; 8 bytes each, with observables 16.
template <bool OBS>
struct TreeRow {
    static constexpr int kWord = OBS ? 16 : 8;
    static constexpr int kAlt = 16 * kWord, kState = 17 * kWord, kSink = 33 * kWord, kBytes = 49 * kWord;
};

constexpr __host__ __device__ int tree_blocks(int L) { return (L + 3) / 4; }
// rows per segment of bounds: at least 32 attempts between barriers
constexpr __host__ __device__ int tree_seg_rows(int L) { return L >= 32 ? 1 : (32 + L - 1) / L; }

// `obs`: observables (0, 1, 2), `values` of them per update
__host__ __device__ inline TreeLds tree_lds(int planes, int L, int nbins, int pitch, int guard, int obs, int values) {
    constexpr int S = kTreePerWave;
    TreeLds t;
    t.rowb = (tree_blocks(L) + 3) & ~3;                    // a row of nibbles
    t.lat = 0;                                             // [walker][plane][row]
    t.ringw = 2 * tree_seg_rows(L) * L * 8 + 32;           // bounds of one walker
    t.ring = (t.lat + S * (planes * L * t.rowb + 4) + 15) & ~15;
    t.rec = t.ring + S * t.ringw;                          // [walker] kTreeRow bytes, see there
    t.queue = t.rec + S * (obs ? TreeRow<true>::kBytes : TreeRow<false>::kBytes);
    const int other = t.queue + (obs == 2 ? S * 4 * tree_blocks(L) * 8 : 0);
    const int nb = nbins + 2 * guard;
    // ln g at twice the offset of the counts, so that a count's address is
    // half its ln g's
    int cb = other > nb * pitch / 2 ? other : nb * pitch / 2;
    cb = (cb + pitch - 1) & ~(pitch - 1);
    t.cnt = cb;
    t.lng = 2 * cb;
    t.sums = t.lng + nb * pitch;                           // [bin][walker][value], no guard bins
    t.total = t.sums + (obs ? nbins * pitch * values : 0);
    return t;
}

typedef uint32_t u32x2v __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) u32x2v lds_u32x2_t;
typedef __attribute__((address_space(3))) uint8_t lds_u8_t;
__device__ __forceinline__ u32x2v lds_u32x2(uint32_t addr) { return *(lds_u32x2_t*)(uintptr_t)addr; }
__device__ __forceinline__ void lds_store_u32x2(uint32_t addr, u32x2v v) { *(lds_u32x2_t*)(uintptr_t)addr = v; }
__device__ __forceinline__ uint32_t lds_u8(uint32_t addr) { return *(lds_u8_t*)(uintptr_t)addr; }
__device__ __forceinline__ void lds_store_u8(uint32_t addr, uint32_t v) { *(lds_u8_t*)(uintptr_t)addr = (uint8_t)v; }

// bit i of a nibble to bit 8 i
__device__ __forceinline__ uint32_t spread_nibble(uint32_t x) { return __umul24(x, 0x204081u) & 0x01010101u; }

// x + f if c, else x, rounded once (f finite)
__device__ __forceinline__ double add_if(bool c, double f, double x) {
    return __builtin_fma(__hiloint2double(c ? 0x3ff00000 : 0, 0), f, x);
}

// What a lane keeps for its node.
struct TreeLane {
    uint32_t sel0;              // v_perm selector of its path's bytes (left of the block's first site as it stands)
    int wC, wN, w1, w2;         // byte weights: current state, proposal, states after the first and second attempt
    double f1, f2, f3;          // ln f where that earlier state exists, else 0
    uint32_t mlo, mhi;          // its ancestors' bits of the decision mask
    uint32_t want, want_tail;   // their outcomes on its path (all ones: never on the path)
    uint32_t out0, out1;        // outcomes word if its attempt is rejected, accepted: flips << 4, 4 if the last site flipped
    uint32_t l8;                // its walker's column of ln g
    double lnf;
    int t;                      // its depth: the path's attempts before its own
    int mC, mN;                 // with observables: byte weights of the flips, before and with its attempt
    uint32_t sums;              // with observables: a bin's sums are at ln g's offset x values + this
};

struct TreeState {
    uint32_t u;      // LDS offset of ln g at the walker's energy
    uint32_t out;    // outcomes of the step before: bit 2 its last site flipped, bits 4..7 its sites' flips
    int m, mb;       // with observables: magnetisation of the plane being flipped, of the product plane
};

// The states of a node and their slots: C, N = u + dv.w (signed bytes) and the
// states after the path's first and second attempt, then each slot = (state &
// mask) | l8.  One block, because the result of a dot product may be read by
// another VALU instruction only three instructions later, which this order
// keeps (and because the three-operand form leaves u where it is).
__device__ __forceinline__ void node_slots(const TreeLane& c, uint32_t dv, uint32_t u, uint32_t mask, uint32_t& C,
                                           uint32_t& N, uint32_t& sC, uint32_t& sN, uint32_t& s1, uint32_t& s2) {
    asm("v_dot4_i32_i8 %[C], %[dv], %[wC], %[u]\n\t"
        "v_dot4_i32_i8 %[N], %[dv], %[wN], %[u]\n\t"
        "v_dot4_i32_i8 %[s1], %[dv], %[w1], %[u]\n\t"
        "v_dot4_i32_i8 %[s2], %[dv], %[w2], %[u]\n\t"
        "v_and_or_b32 %[sC], %[C], %[mask], %[l8]\n\t"
        "v_and_or_b32 %[sN], %[N], %[mask], %[l8]\n\t"
        "v_and_or_b32 %[s1], %[s1], %[mask], %[l8]\n\t"
        "v_and_or_b32 %[s2], %[s2], %[mask], %[l8]"
        : [C] "=&v"(C), [N] "=&v"(N), [sC] "=&v"(sC), [sN] "=&v"(sN), [s1] "=&v"(s1), [s2] "=&v"(s2)
        : [dv] "v"(dv), [wC] "v"(c.wC), [wN] "v"(c.wN), [w1] "v"(c.w1), [w2] "v"(c.w2), [u] "v"(u), [mask] "s"(mask),
          [l8] "v"(c.l8));
}

template <int OBS>
struct TreeInput {
    u32x2v rec;   // energy-change bytes of the block's sites, left neighbour as it stands / flipped
    u32x2v mag;   // with observables: magnetisation-change bytes, of the plane and of the product plane
    double B;     // acceptance bound of this lane's attempt
    __device__ __forceinline__ void read(uint32_t addr) {
        if constexpr (OBS) {
            const u32x4v v = lds_u32x4(addr);
            rec = u32x2v{v.x, v.y};
            mag = u32x2v{v.z, v.w};
        } else {
            rec = lds_u32x2(addr);
        }
    }
};

// Update counts with observables = 2.  A sample is due at the updates whose
// bin had 0, 1000, 2000, ... before them: a count word's low ten bits are 24 + t
// mod 1000, or 0 where t mod 1000 = 0 (what the plain increment of 1023 leaves),
// and the due update adds 24 more; so "due" is ten zero bits.
__device__ __forceinline__ uint32_t cycle_word(uint32_t t) {
    const uint32_t r = t % 1000u;
    return r ? r + 24u : 0u;
}
__device__ __forceinline__ uint32_t cycle_count(uint32_t w) {
    const uint32_t r = w & 1023u;
    return (w >> 10) * 1000u + (r ? r - 24u : 0u);
}

// What the walker wavefront keeps beside its state with observables.
struct TreeObs {
    int N;
    int other;             // magnetisation of the plane not being flipped (two planes)
    bool second;           // the plane being flipped is the second one
    uint32_t queue, due;   // samples due in this row: LDS queue, how many
};

// Four attempts (or, TAIL, the row's last r < 5: lanes of deeper nodes have
// want_tail = never).  `in` is the block's input on entry; the next block's,
// read from next_rec and next_B while this one's ln g are in flight, on exit.
// The state goes to word K from au (the row's words for the lane that ends the
// step, else the sink) and is read back from word K from ust by the whole row.
// With observables every lane on the path adds its moments to the bin's sums;
// with observables = 2 it also looks whether its update is due for a sample,
// and then queues the bin, its walker, the block and the block's flips so far
// for the end of the row (`block`: the block's number).
template <int MODEL, int OBS, bool TAIL, int K>
__device__ __forceinline__ void tree_block(const TreeLane& c, TreeState& st, TreeInput<OBS>& in, TreeObs& ob,
                                           uint32_t next_rec, uint32_t next_B, uint32_t mask, uint32_t au, uint32_t ust,
                                           uint32_t block) {
    using Mdl = Model<MODEL>;
    constexpr int AT = K * TreeRow<OBS != 0>::kWord;
    const uint32_t dv = __builtin_amdgcn_perm(in.rec.y, in.rec.x, c.sel0 | (st.out & 4u));
    uint32_t C, N, sC, sN, s1, s2;
    node_slots(c, dv, st.u, mask, C, N, sC, sN, s1, s2);
    double lc = lds_f64(sC), ln = lds_f64(sN);
    uint32_t tC = 0, tN = 0;
    if constexpr (OBS == 2) {
        tC = lds_u32_at(sC >> 1);
        tN = lds_u32_at(sN >> 1);
    }
    const double B = in.B;
    int mC = 0, mN = 0, bC = 0, bN = 0;
    if constexpr (OBS != 0) {
        mC = __builtin_amdgcn_sdot4((int)in.mag.x, c.mC, st.m, false);
        mN = __builtin_amdgcn_sdot4((int)in.mag.x, c.mN, st.m, false);
        if constexpr (Mdl::kPlanes > 1) {
            bC = __builtin_amdgcn_sdot4((int)in.mag.y, c.mC, st.mb, false);
            bN = __builtin_amdgcn_sdot4((int)in.mag.y, c.mN, st.mb, false);
        }
    }
    if (!TAIL) {
        in.read(next_rec);
        in.B = lds_f64(next_B);
    }
    lc = add_if(sC == s1, c.f1, lc);
    ln = add_if(sN == s1, c.f1, ln);
    lc = add_if(sC == s2, c.f2, lc);
    ln = add_if(sN == s2, c.f2, ln);
    lc = lc + c.f3;
    ln = add_if(sN == sC, c.f3, ln);
    const bool acc = (ln - lc) < B;
    const uint64_t M = __builtin_amdgcn_ballot_w64(acc);
    const uint32_t pv = ((uint32_t)M & c.mlo) | ((uint32_t)(M >> 32) & c.mhi);
    const uint64_t path = __builtin_amdgcn_ballot_w64(pv == (TAIL ? c.want_tail : c.want));
    const uint32_t sF = acc ? sN : sC;
    const uint32_t cF = sF >> 1, one = 1u;
    // The last lane of the path hands the state over to its row; the lanes on
    // the path add ln f and a count.  (Stores and atomics without return;
    // every lane is active here.)
    if constexpr (OBS == 0) {
        u32x2v uf;
        uf.x = acc ? N : C;
        uf.y = acc ? c.out1 : c.out0;
        asm volatile("s_mov_b64 exec, %[path]\n\t"
                     "ds_write_b64 %[au], %[uf] offset:%[at]\n\t"
                     "ds_add_f64 %[sF], %[lnf]\n\t"
                     "ds_add_u32 %[cF], %[one]\n\t"
                     "s_mov_b64 exec, -1"
                     :
                     : [path] "s"(path), [au] "v"(au), [uf] "v"(uf), [at] "n"(AT), [sF] "v"(sF), [lnf] "v"(c.lnf),
                       [cF] "v"(cF), [one] "v"(one)
                     : "memory");
        const u32x2v s = lds_u32x2(ust + AT);
        st.u = s.x;
        st.out = s.y;
    } else {
        u32x4v uf;
        uf.x = acc ? N : C;
        uf.y = acc ? c.out1 : c.out0;
        uf.z = (uint32_t)(acc ? mN : mC);
        uf.w = (uint32_t)(acc ? bN : bC);
        constexpr int NV = Mdl::kValues;
        int m[3] = {(int)uf.z, 0, 0};
        if constexpr (Mdl::kPlanes > 1) {
            m[0] = ob.second ? ob.other : (int)uf.z;
            m[1] = ob.second ? (int)uf.z : ob.other;
            m[2] = (int)uf.w;
        }
        double v[NV];
        const uint32_t sum = __umul24(sF, (uint32_t)NV) + c.sums;
        u32x4v s;
        if constexpr (NV == 3) {
            // the adds of the moments run while the state comes back: one block,
            // whose wait, for all but the last five LDS operations, is for that
            // read (LDS operations end in order)
            Mdl::values(ob.N, m, v);
            asm volatile("s_mov_b64 exec, %[path]\n\t"
                         "ds_write_b128 %[au], %[uf] offset:%[at]\n\t"
                         "s_mov_b64 exec, -1\n\t"
                         "ds_read_b128 %[s], %[ust] offset:%[at]\n\t"
                         "s_mov_b64 exec, %[path]\n\t"
                         "ds_add_f64 %[sF], %[lnf]\n\t"
                         "ds_add_u32 %[cF], %[one]\n\t"
                         "ds_add_f64 %[sum], %[v0]\n\t"
                         "ds_add_f64 %[sum], %[v1] offset:8\n\t"
                         "ds_add_f64 %[sum], %[v2] offset:16\n\t"
                         "s_mov_b64 exec, -1\n\t"
                         "s_waitcnt lgkmcnt(5)"
                         : [s] "=&v"(s)
                         : [path] "s"(path), [au] "v"(au), [uf] "v"(uf), [at] "n"(AT), [ust] "v"(ust), [sF] "v"(sF),
                           [lnf] "v"(c.lnf), [cF] "v"(cF), [one] "v"(one), [sum] "v"(sum), [v0] "v"(v[0]), [v1] "v"(v[1]),
                           [v2] "v"(v[2])
                         : "memory");
        } else {
            asm volatile("s_mov_b64 exec, %[path]\n\t"
                         "ds_write_b128 %[au], %[uf] offset:%[at]\n\t"
                         "s_mov_b64 exec, -1\n\t"
                         "ds_read_b128 %[s], %[ust] offset:%[at]\n\t"
                         "s_mov_b64 exec, %[path]\n\t"
                         "ds_add_f64 %[sF], %[lnf]\n\t"
                         "ds_add_u32 %[cF], %[one]\n\t"
                         "s_mov_b64 exec, -1\n\t"
                         "s_waitcnt lgkmcnt(2)"
                         : [s] "=&v"(s)
                         : [path] "s"(path), [au] "v"(au), [uf] "v"(uf), [at] "n"(AT), [ust] "v"(ust), [sF] "v"(sF),
                           [lnf] "v"(c.lnf), [cF] "v"(cF), [one] "v"(one)
                         : "memory");
            Mdl::values(ob.N, m, v);
#pragma unroll
            for (int i = 0; i < NV; i += 3)
                asm volatile("s_mov_b64 exec, %[path]\n\t"
                             "ds_add_f64 %[sum], %[v0] offset:%[o0]\n\t"
                             "ds_add_f64 %[sum], %[v1] offset:%[o1]\n\t"
                             "ds_add_f64 %[sum], %[v2] offset:%[o2]\n\t"
                             "s_mov_b64 exec, -1"
                             :
                             : [path] "s"(path), [sum] "v"(sum), [v0] "v"(v[i]), [v1] "v"(v[i + 1]), [v2] "v"(v[i + 2]),
                               [o0] "n"(8 * i), [o1] "n"(8 * i + 8), [o2] "n"(8 * i + 16)
                             : "memory");
        }
        st.u = s.x;
        st.out = s.y;
        st.m = (int)s.z;
        st.mb = (int)s.w;
        if constexpr (OBS == 2) {
            // counts as they were before the step; the path's earlier updates of
            // the same bin bring at most three more (told by the depth: ln f is 0
            // while a refinement samples)
            const uint32_t t = acc ? tN : tC;
            if (__builtin_amdgcn_ballot_w64(((t + 3u) & 1023u) < 4u) & path) {
                const uint32_t before = (c.t >= 2 && sF == s1 ? 1u : 0u) + (c.t >= 3 && sF == s2 ? 1u : 0u) +
                                        (c.t >= 1 && sF == sC ? 1u : 0u);
                const uint64_t due = __builtin_amdgcn_ballot_w64(((t + before) & 1023u) == 0u) & path;
                const int lane = threadIdx.x & 63;
                if ((due >> lane) & 1ull) {
                    lds_add_u32(cF, 24u);
                    const uint32_t k = ob.due + (uint32_t)__popcll(due & ((1ull << lane) - 1ull));
                    lds_store_u32x2(ob.queue + 8u * k, u32x2v{sF, (uf.y & 0xf0u) | (uint32_t)(lane >> 4) | (block << 8)});
                }
                ob.due += (uint32_t)__popcll(due);
            }
        }
    }
}

// x of the lane that the DPP control names (every lane active)
template <int CTRL>
__device__ __forceinline__ double dpp_f64(double x) {
    return __hiloint2double(__builtin_amdgcn_mov_dpp(__double2hiint(x), CTRL, 0xf, 0xf, false),
                            __builtin_amdgcn_mov_dpp(__double2loint(x), CTRL, 0xf, 0xf, false));
}
__device__ __forceinline__ double lane_f64(double x, int lane) {
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(x), lane),
                            __builtin_amdgcn_readlane(__double2loint(x), lane));
}
// A double's sum over the wavefront: pairs, quads, halves of a row of sixteen,
// rows, then the four rows.
__device__ __forceinline__ double wave_sum(double x) {
    x += dpp_f64<0xb1>(x);    // quad_perm 1 0 3 2
    x += dpp_f64<0x4e>(x);    // quad_perm 2 3 0 1
    x += dpp_f64<0x141>(x);   // row_half_mirror
    x += dpp_f64<0x140>(x);   // row_mirror
    return (lane_f64(x, 0) + lane_f64(x, 16)) + (lane_f64(x, 32) + lane_f64(x, 48));
}

// G(qmin) of the +-1 field whose row y is lane y's w (bit 1 = -1; lanes and
// bits from L on are zero), lane k holding cos and sin of qmin k
// (fourier_correlator.hpp:65-118): row sums are popcounts, column sums ballots.
__device__ __forceinline__ double tree_fourier(int L, int lane, uint64_t w, double co, double si) {
    int col = 0;
    auto columns = [&](uint32_t v, int first) {
#pragma unroll
        for (int x = 0; x < 32; ++x) {
            const int k = (int)__popcll(__builtin_amdgcn_ballot_w64((v & (1u << x)) != 0u));
            col = lane == first + x ? k : col;
        }
    };
    columns((uint32_t)w, 0);
    if (L > 32) columns((uint32_t)(w >> 32), 32);
    const bool in = lane < L;
    const double R = in ? (double)(L - 2 * (int)__popcll(w)) : 0.0, Cx = in ? (double)(L - 2 * col) : 0.0;
    const double f[4] = {wave_sum(R * co), wave_sum(R * si), wave_sum(Cx * co), wave_sum(Cx * si)};
    return fourier_g(L, f);
}

// The samples due in row y (observables = 2, update_qmin_correlator,
// ising2d_hamiltonian.hpp:247-252): for each, the lattice as it was after its
// update, a row per lane.  The row in LDS is as it was before its sweep; the
// state words hold the flips of its blocks.
template <int MODEL>
__device__ __forceinline__ void tree_samples(const KArgs& a, const DevGroup& G, const DevSystem& S, const TreeScale& T,
                                          const TreeLds& o, int lane, int y, const TreeObs& ob, double co, double si,
                                          int fl) {
    using Mdl = Model<MODEL>;
    constexpr int NP = Mdl::kPlanes;
    using Row = TreeRow<true>;
    const int L = S.L;
    for (uint32_t k = 0; k < ob.due; ++k) {
        const u32x2v e = lds_u32x2(ob.queue + 8u * k);
        const uint32_t slot = (uint32_t)__builtin_amdgcn_readfirstlane((int)e.x);
        const uint32_t what = (uint32_t)__builtin_amdgcn_readfirstlane((int)e.y);
        const int j = (int)(what & 15u), block = (int)(what >> 8);
        const int pf = Mdl::flip_plane(__builtin_amdgcn_readlane(fl, 16 * j));
        const uint32_t words = (uint32_t)(o.rec + j * Row::kBytes + Row::kState + 4);
        uint32_t fl_lo = 0, fl_hi = 0;   // every block's flips; the row's before `block`
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const uint32_t f = (lds_u32_at(words + (uint32_t)(Row::kWord * i)) >> 4) & 15u;
            if (i < 8) fl_lo |= f << (4 * i);
            else fl_hi |= f << (4 * i - 32);
        }
        const uint64_t fw = ((((uint64_t)fl_hi << 32) | fl_lo) & ((1ull << (4 * block)) - 1ull)) |
                            (uint64_t)((what >> 4) & 15u) << (4 * block);
        uint64_t w[NP];
        const uint64_t sites = L == 64 ? ~0ull : (1ull << L) - 1ull;
#pragma unroll
        for (int q = 0; q < NP; ++q) {
            w[q] = 0;
            const uint32_t src = (uint32_t)(o.lat + j * (NP * L * o.rowb + 4) + (q * L + min(lane, L - 1)) * o.rowb);
#pragma unroll
            for (int i = 0; i < 4; ++i) {   // past a short row: cut off below
                const uint32_t v = lds_u32_at(src + 4u * (uint32_t)i);
                w[q] |= (uint64_t)((v & 0xfu) | ((v >> 4) & 0xf0u) | ((v >> 8) & 0xf00u) | ((v >> 12) & 0xf000u)) << (16 * i);
            }
            if (q == pf && lane == y) w[q] ^= fw;
            w[q] &= lane < L ? sites : 0ull;
        }
        const double gs = tree_fourier(L, lane, w[0], co, si);
        const double gb = Mdl::kBaxterCorrelator ? tree_fourier(L, lane, w[0] ^ w[NP - 1], co, si) : 0.;
        if (lane == 0) {
            const int b = (int)((slot - (uint32_t)o.lng) >> __builtin_ctz((unsigned)T.pitch)) - T.guard;
            double* p = a.obs + (G.hist_base + j + (int64_t)b * kLanes) * a.nobs;
            Mdl::add_correlators([&](int s, double g) { obs_add(p + s, g); }, gs, gb);
        }
    }
}

// The walker wavefront: four walkers.
template <int MODEL, int OBS>
__device__ __forceinline__ void sweep_walkers_tree(const KArgs& a, const DevGroup& G, const DevSystem& S,
                                                   const TreeScale& T, const TreeLds& o, int nsweeps) {
    using Mdl = Model<MODEL>;
    constexpr int NP = Mdl::kPlanes;
    constexpr int NPASS = Mdl::kPasses;
    constexpr bool KQ = Mdl::kProductCoupling;
    using Row = TreeRow<OBS != 0>;
    constexpr uint32_t WB = Row::kWord;
    const int tid = threadIdx.x & 63;
    const int n = tid & 15, j = tid >> 4;
    const bool active = j < G.nwalkers;
    const int g = G.first_walker + (active ? j : 0);
    const DevWindow Wn = a.win[a.w_window[g]];
    const double lnf = a.win_lnf[a.w_window[g]];
    const int L = S.L, nblk = tree_blocks(L), tail = L - 4 * (nblk - 1);
    const uint32_t mask = ~(uint32_t)(T.pitch - 1);
    const int bshift = Wn.shift;                                  // log2 of the bin size
    const int pshift = 31 - __builtin_clz((unsigned)T.pitch);
    const uint32_t u0 = (uint32_t)(o.lng + T.guard * T.pitch);    // energy = window minimum

    // ---- the lane's node -----------------------------------------------------
    TreeLane c;
    {
        const int t = n < 2 ? 0 : n < 4 ? 1 : n < 8 ? 2 : 3;
        uint32_t anc = 0, want = 0, sel = 0x03020100u;
        int wC = 0, w1 = 0, w2 = 0, mC = 0;
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            if (i >= t) continue;
            const int k = t - i;              // the ancestor that decides attempt i is n >> k
            const int ai = (n >> (k - 1)) & 1;
            anc |= 1u << (n >> k);
            want |= (uint32_t)ai << (n >> k);
            if (ai) {
                wC |= T.w << (8 * i);
                mC |= 1 << (8 * i);
                if (i < 1 && t >= 2) w1 |= T.w << (8 * i);
                if (i < 2 && t >= 3) w2 |= T.w << (8 * i);
                sel |= 4u << (8 * (i + 1));   // the site after a flip sees its left neighbour flipped
            }
        }
        c.t = t;
        c.sel0 = sel;
        c.wC = wC;
        c.wN = wC | (T.w << (8 * t));
        c.w1 = w1;
        c.w2 = w2;
        c.f1 = t >= 2 ? lnf : 0.0;
        c.f2 = t >= 3 ? lnf : 0.0;
        c.f3 = t >= 1 ? lnf : 0.0;
        const uint32_t sh = 16u * (j & 1);
        const bool on = active && n > 0;
        c.mlo = on && j < 2 ? anc << sh : 0u;
        c.mhi = on && j >= 2 ? anc << sh : 0u;
        c.want = on ? want << sh : 0xffffffffu;
        c.want_tail = on && t < tail ? want << sh : 0xffffffffu;
        uint32_t flips = 0;
#pragma unroll
        for (int i = 0; i < 3; ++i)
            if (i < t) flips |= (uint32_t)((n >> (t - i - 1)) & 1) << (4 + i);
        c.out0 = flips;
        c.out1 = flips | (1u << (4 + t)) | 4u;
        c.l8 = (uint32_t)(j * 8);
        c.lnf = lnf;
        c.mC = mC;
        c.mN = mC | (1 << (8 * t));
        c.sums = (uint32_t)(o.sums - (o.lng + T.guard * T.pitch) * Mdl::kValues);
    }
    const uint32_t latw = (uint32_t)(o.lat + j * (NP * L * o.rowb + 4));
    const uint32_t recw = (uint32_t)(o.rec + j * Row::kBytes);
    // where the lane leaves a step's state: the row's word if it ends the step
    const uint32_t au = recw + (uint32_t)(c.t == 3 ? Row::kState : Row::kSink);
    const uint32_t au_tail = recw + (uint32_t)(c.t == tail - 1 ? Row::kState : Row::kSink);
    const uint32_t ringw = (uint32_t)(o.ring + j * o.ringw + c.t * 8);
    // energy change bytes by the number of disagreeing neighbours; with two
    // couplings biased by 64 each, so that the bytes add without carries, and
    // made signed afterwards
    uint32_t tj_lo = 0, tj_hi = 0, tk_lo = 0, tk_hi = 0;
    {
        auto entry = [&](int two, int k) { return (uint32_t)((two * (4 - 2 * k) / T.g) * T.m + (KQ ? 64 : 0)) & 255u; };
        for (int k = 0; k < 4; ++k) {
            tj_lo |= entry(S.twoJ, k) << (8 * k);
            if (KQ) tk_lo |= entry(S.twoK, k) << (8 * k);
        }
        tj_hi = entry(S.twoJ, 4);
        if (KQ) tk_hi = entry(S.twoK, 4);
    }
    int fl = a.w_flavor[g];
    // the walker is inside its window (rewl_adjust_to_range); the clamp keeps
    // its slot in bounds regardless
    const int e0 = min(max((int)a.w_E[g] - Wn.imin, 0), (Wn.nbins << bshift) - 1);
    TreeState st{u0 + (uint32_t)(e0 << (pshift - bshift)), 0u, 0, 0};
    // an absent walker's row never writes its state words
    if (n < nblk) lds_store_u32x2(recw + (uint32_t)Row::kState + WB * (uint32_t)n, u32x2v{st.u, 0u});
    TreeObs ob{L * L, 0, false, (uint32_t)o.queue, 0u};
    // observables = 2: lane k has cos and sin of qmin k
    double co = 0.0, si = 0.0;
    if constexpr (OBS == 2) {
        const double qmin = 2. * acos(-1.) / (double)L;
        co = cos(qmin * (double)tid);
        si = sin(qmin * (double)tid);
    }

    // the lane's block of a row and its neighbours in the row
    const int b = n < nblk ? n : nblk - 1;
    const int bl = b == 0 ? nblk - 1 : b - 1, br = b == nblk - 1 ? 0 : b + 1;
    const int topl = bl == nblk - 1 ? tail - 1 : 3, top = b == nblk - 1 ? tail - 1 : 3;
    // Counts of disagreeing neighbours below and beside, by site of the lane's
    // block: [right neighbour of the row's last site as it stands, flipped]
    // [left neighbour as it stands, flipped]; the product plane's too.
    struct Beside {
        uint32_t p[2][2], q[2][2];
    } bs{};
    uint32_t up = 0, cur = 0, dn = 0;   // the lane's nibbles: the row above as rewritten, this row, the row below
    uint32_t qcu = 0;                   // product coupling: other plane's disagreement with the row above
    uint32_t qc = 0;                    // and its nibble
    uint32_t lat = 0, latq = 0;         // the plane this pass flips, the other one
    struct Bytes {
        uint32_t dn, l, r, qc, qu, qd, ql, qr;
    };
    // row y's bytes around the lane's block (its own nibble aside)
    auto read_row = [&](int y) {
        const int yd = y == L - 1 ? 0 : y + 1;
        Bytes v{};
        v.dn = lds_u8(lat + (uint32_t)(yd * o.rowb + b));
        v.l = lds_u8(lat + (uint32_t)(y * o.rowb + bl));
        v.r = lds_u8(lat + (uint32_t)(y * o.rowb + br));
        if constexpr (KQ) {
            const int yu = y == 0 ? L - 1 : y - 1;
            v.qc = lds_u8(latq + (uint32_t)(y * o.rowb + b));
            v.qu = lds_u8(latq + (uint32_t)(yu * o.rowb + b));
            v.qd = lds_u8(latq + (uint32_t)(yd * o.rowb + b));
            v.ql = lds_u8(latq + (uint32_t)(y * o.rowb + bl));
            v.qr = lds_u8(latq + (uint32_t)(y * o.rowb + br));
        }
        return v;
    };
    // disagreements of nibble p with the site to the right, to the left
    auto right_of = [&](uint32_t p, uint32_t r) { return p ^ ((p >> 1) | ((r & 1u) << top)); };
    auto left_of = [&](uint32_t p, uint32_t l) { return (p ^ ((p << 1) | ((l >> topl) & 1u))) & 15u; };
    auto beside = [&](uint32_t p, const Bytes& v) {
        const uint32_t rt = right_of(p, v.r), lf = left_of(p, v.l), d = p ^ v.dn;
        auto sums = [&](uint32_t dd, uint32_t rr, uint32_t ll, uint32_t (&out)[2][2]) {
            const uint32_t s = spread_nibble(dd), r0 = spread_nibble(rr), r1 = r0 ^ (1u << (8 * top));
            const uint32_t l0 = spread_nibble(ll), l1 = l0 ^ 0x01010101u;
            out[0][0] = s + r0 + l0;
            out[0][1] = s + r0 + l1;
            out[1][0] = s + r1 + l0;
            out[1][1] = s + r1 + l1;
        };
        sums(d, rt, lf, bs.p);
        if constexpr (KQ) {
            sums(d ^ v.qc ^ v.qd, rt ^ right_of(v.qc, v.qr), lf ^ left_of(v.qc, v.ql), bs.q);
            qcu = v.qc ^ v.qu;
            qc = v.qc;
        }
        dn = v.dn;
    };
    const bool last_block = n >= nblk - 1;
    const int seg_rows = tree_seg_rows(L);
    const int nrows = nsweeps * NPASS * L;
    int y = 0, in_seg = 0, slot = 0;
    __syncthreads();   // LDS loaded, first segment of bounds ready
    if constexpr (OBS != 0) {
        // magnetisations: a lane counts rows n, n + 16, ... of each plane
        int ps[NP] = {}, px = 0;
        for (int yy = n; yy < L; yy += 16)
            for (int k = 0; k < o.rowb; k += 4) {
                uint32_t x = 0;
#pragma unroll
                for (int q = 0; q < NP; ++q) {
                    const uint32_t v = lds_u32_at(latw + (uint32_t)((q * L + yy) * o.rowb + k));
                    ps[q] += (int)__popc(v);
                    x ^= v;
                }
                px += (int)__popc(x);
            }
        auto row_sum = [&](int x) {
#pragma unroll
            for (int k = 8; k >= 1; k >>= 1) x += __shfl_xor(x, k, 64);
            return L * L - 2 * x;
        };
        // the plane that the first pass flips, and the other one
        const int pf = Mdl::flip_plane(fl);
        st.m = row_sum(plane_pick(ps, pf));
        if constexpr (NP > 1) {
            ob.other = row_sum(plane_pick(ps, NP - 1 - pf));
            st.mb = row_sum(px);
        }
    }
    for (int r = 0; r < nrows; ++r) {
        if (y == 0 && (NPASS > 1 || r == 0)) {
            const int pf = Mdl::flip_plane(fl), qf = NP - 1 - pf;
            if constexpr (OBS != 0 && NP > 1) {
                if (r > 0) {
                    const int m = st.m;
                    st.m = ob.other;
                    ob.other = m;
                }
                ob.second = pf != 0;
            }
            lat = latw + (uint32_t)(pf * L * o.rowb);
            latq = latw + (uint32_t)(qf * L * o.rowb);
            up = lds_u8(lat + (uint32_t)((L - 1) * o.rowb + b));
            cur = lds_u8(lat + b);
            beside(cur, read_row(0));
        }
        const uint32_t ring = ringw + (uint32_t)(slot * L * 8);
        TreeInput<OBS> in;
        in.B = lds_f64(ring);
        // ---- energy changes of the row: lane n takes block n; only the row
        // above is new, the rest was prepared during the row before ------------
        const uint32_t su = spread_nibble(cur ^ up);
        uint32_t sq = 0;
        if constexpr (KQ) sq = spread_nibble(cur ^ up ^ qcu);
        u32x2v mag{0u, 0u};
        if constexpr (OBS != 0) {
            // a flip takes -1 to +1 (bit 1) or back
            mag.x = __builtin_amdgcn_perm(0u, 0x02feu, spread_nibble(cur));
            if constexpr (NP > 1) mag.y = __builtin_amdgcn_perm(0u, 0x02feu, spread_nibble(cur ^ qc));
        }
        auto record = [&](int alt) {
            u32x2v v;
            v.x = __builtin_amdgcn_perm(tj_hi, tj_lo, su + bs.p[alt][0]);
            v.y = __builtin_amdgcn_perm(tj_hi, tj_lo, su + bs.p[alt][1]);
            if constexpr (KQ) {
                v.x += __builtin_amdgcn_perm(tk_hi, tk_lo, sq + bs.q[alt][0]);
                v.y += __builtin_amdgcn_perm(tk_hi, tk_lo, sq + bs.q[alt][1]);
                v ^= 0x80808080u;
            }
            return v;
        };
        auto store_record = [&](uint32_t at, u32x2v v) {
            if constexpr (OBS != 0) *(lds_u32x4_t*)(uintptr_t)at = u32x4v{v.x, v.y, mag.x, mag.y};
            else lds_store_u32x2(at, v);
        };
        {
            const u32x2v v = record(0);
            if (n < nblk) store_record(recw + WB * (uint32_t)n, v);
            // the first block's: lane 0's, to its row
            in.rec.x = (uint32_t)__builtin_amdgcn_mov_dpp((int)v.x, 0x150, 0xf, 0xf, false);
            in.rec.y = (uint32_t)__builtin_amdgcn_mov_dpp((int)v.y, 0x150, 0xf, 0xf, false);
            if constexpr (OBS != 0) {
                in.mag.x = (uint32_t)__builtin_amdgcn_mov_dpp((int)mag.x, 0x150, 0xf, 0xf, false);
                in.mag.y = (uint32_t)__builtin_amdgcn_mov_dpp((int)mag.y, 0x150, 0xf, 0xf, false);
            }
        }
        const Bytes nx = read_row(y == L - 1 ? 0 : y + 1);
        // ---- the row's blocks --------------------------------------------------
        st.out = 0u;   // left of site 0 is site L - 1, as it stands
        ob.due = 0u;
        const uint32_t nlast = (uint32_t)(nblk - 1);
        // blocks q4 + k, k = 0..3, in fours from q4 = 0
        uint32_t x = recw, rg = ring, aq = au;   // addresses at block q4
        asm("" : "+v"(x), "+v"(rg), "+v"(aq));
        // block q4 + K, the next one's record at xr
        auto block = [&](auto k, uint32_t q4, uint32_t xr) {
            constexpr int K = decltype(k)::value;
            tree_block<MODEL, OBS, false, K>(c, st, in, ob, xr, rg + (uint32_t)(32 * (K + 1)), mask, aq,
                                             x + (uint32_t)Row::kState, q4 + (uint32_t)K);
        };
        using std::integral_constant;
        block(integral_constant<int, 0>{}, 0u, x + WB);
        if (n == nblk - 1) store_record(recw + (uint32_t)Row::kAlt, record(1));
        const uint32_t own = cur;
        cur = dn;
        beside(cur, nx);   // for the next row
        // the last block's last site sees site 0 as it is now
        const uint32_t rec_last = (st.out & 16u) ? recw + (uint32_t)Row::kAlt : recw + WB * nlast;
        auto next_rec = [&](uint32_t i, uint32_t xr) { return i == nlast ? rec_last : xr; };
        if (nlast > 1u) block(integral_constant<int, 1>{}, 0u, next_rec(2u, x + 2u * WB));
        if (nlast > 2u) block(integral_constant<int, 2>{}, 0u, next_rec(3u, x + 3u * WB));
        if (nlast > 3u) block(integral_constant<int, 3>{}, 0u, next_rec(4u, x + 4u * WB));
        uint32_t i = 4u;
        x += 4u * WB;
        rg += 128u;
        aq += 4u * WB;
        for (; i + 4u <= nlast; i += 4u) {
            // opaque, so that every address of the four is one of these plus
            // an offset of its instruction
            asm("" : "+v"(x), "+v"(rg), "+v"(aq));
            block(integral_constant<int, 0>{}, i, x + WB);
            block(integral_constant<int, 1>{}, i, x + 2u * WB);
            block(integral_constant<int, 2>{}, i, x + 3u * WB);
            block(integral_constant<int, 3>{}, i, next_rec(i + 4u, x + 4u * WB));
            x += 4u * WB;
            rg += 128u;
            aq += 4u * WB;
        }
        if (i < nlast) {
            asm("" : "+v"(x), "+v"(rg), "+v"(aq));
            block(integral_constant<int, 0>{}, i, next_rec(i + 1u, x + WB));
            if (i + 1u < nlast) block(integral_constant<int, 1>{}, i, next_rec(i + 2u, x + 2u * WB));
            if (i + 2u < nlast) block(integral_constant<int, 2>{}, i, next_rec(i + 3u, x + 3u * WB));
        }
        if (nlast == 1u) in.read(rec_last);   // read before the first block was decided
        // ---- the row as rewritten: the state words hold the blocks' flips ----
        const uint32_t word = lds_u32x2(recw + (uint32_t)Row::kState + WB * (uint32_t)b).y;
        tree_block<MODEL, OBS, true, 0>(c, st, in, ob, 0u, 0u, mask, au_tail + WB * nlast,
                                        recw + WB * nlast + (uint32_t)Row::kState, nlast);
        if constexpr (OBS == 2) {
            if (ob.due) tree_samples<MODEL>(a, G, S, T, o, tid, y, ob, co, si, fl);
        }
        up = own ^ (((last_block ? st.out : word) >> 4) & 15u);
        if (n < nblk) lds_store_u8(lat + (uint32_t)(y * o.rowb + n), up);
        if (++y == L) {
            y = 0;
            fl = Mdl::next_flavour(fl);   // flavour switches after site N - 1
        }
        if (++slot == 2 * seg_rows) slot = 0;
        if (++in_seg == seg_rows) {
            in_seg = 0;
            __syncthreads();   // this segment's bounds consumed, the next one's written
        }
    }
    if (in_seg) __syncthreads();
    if (active && n == 0) {
        a.w_E[g] = (double)((int)((st.u - u0) >> (pshift - bshift)) + Wn.imin);
        a.w_flavor[g] = fl;
    }
}

// Producer side, one wavefront: the bounds of the rows [r0, r0 + count) (rows of
// the launch, counted over its passes and sweeps) for every walker of the
// group, one Philox block (up to four bounds) per lane.  A walker's ring of ringw bytes
// holds `slots` rows of rowb bytes.
template <int MODEL>
__device__ __forceinline__ void tree_fill(const DevGroup& G, const DevSystem& S, int ring, int ringw, int rowb, int slots,
                                          int lane, uint64_t sweep_base, int r0, int count, const BoundEntry* tab) {
    const int L = S.L, per_sweep = Model<MODEL>::kPasses * L;
    const uint64_t blocks = (uint64_t)((S.ndof + 3) / 4);   // Philox blocks per sweep
    const int nbb = (L & 3) ? L / 4 + 2 : L / 4;            // blocks that a row can touch
    const int total = count * nbb * kTreePerWave;
    for (int i = lane; i < total; i += kLanes) {
        const int j = i & (kTreePerWave - 1);
        const int rest = i / kTreePerWave;
        const int k = rest / nbb, bb = rest - k * nbb;
        if (j >= G.nwalkers) continue;
        const int r = r0 + k;
        const int s = r / per_sweep;
        const int p0 = (r - s * per_sweep) * L;             // attempt position of the row's first site in its sweep
        const int blk = (p0 >> 2) + bb;
        const int x0 = 4 * blk - p0;
        if (x0 >= L) continue;
        const uint64_t bi = (sweep_base + (uint64_t)s) * blocks + (uint64_t)blk;
        const uint32_t walker = (uint32_t)(G.first_walker - S.first_walker + j);
        const u32x4 w = philox4x32_10(u32x4{(uint32_t)bi, (uint32_t)(bi >> 32), DOMAIN_SWEEP, walker}, S.k0, S.k1);
        const double v[4] = {accept_bound(w.x, tab), accept_bound(w.y, tab), accept_bound(w.z, tab),
                             accept_bound(w.w, tab)};
        const uint32_t dst = (uint32_t)(ring + j * ringw + (r % slots) * rowb);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int x = x0 + q;
            if (x >= 0 && x < L) lds_store_f64(dst + 8u * (uint32_t)x, v[q]);
        }
    }
}

// One workgroup = one walker wavefront (four walkers) + one producer.  The grid has
// one for every group of the list; the loop is for a smaller one.
template <int MODEL, int OBS>
__global__ void __launch_bounds__(2 * kLanes) k_sweep_tree(KArgs a, const TreeScale* scale, const int32_t* groups,
                                                           int ngroups, int nsweeps, uint64_t sweep_base) {
    using Mdl = Model<MODEL>;
    constexpr int NP = Mdl::kPlanes;
    constexpr int SW = kTreePerWave;
    constexpr int nth = 2 * kLanes;
    const int tid = threadIdx.x;
    const bool walkers = __builtin_amdgcn_readfirstlane(tid) < kLanes;
    const BoundEntry* tab = static_cast<const BoundEntry*>(a.bound_tab);
    if (walkers) __builtin_amdgcn_s_setprio(3);
    for (int gi = blockIdx.x; gi < ngroups; gi += gridDim.x) {
        const DevGroup G = a.grp[groups[gi]];
        const DevSystem S = a.sys[G.sys];
        const TreeScale T = scale[G.sys];
        const int L = S.L;
        const TreeLds o = tree_lds(NP, L, G.nbins, T.pitch, T.guard, OBS, Mdl::kValues);
        // ---- load (LDS addresses are offsets: the kernel has no static LDS):
        // histograms (guard bins and absent walkers: +inf), lattice --
        const int nb = G.nbins + 2 * T.guard;
        // a thread loads one walker's bins, eight at a time in flight
        const int jw = tid & (SW - 1), bins = jw < G.nwalkers ? a.win[a.w_window[G.first_walker + jw]].nbins : 0;
        const int64_t h0 = G.hist_base + jw;
        constexpr int STEP = nth / SW;
        for (int b0 = tid / SW; b0 < nb; b0 += 8 * STEP) {
            double lng[8];
            uint32_t cnt[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                const int b = b0 + k * STEP - T.guard;
                const bool in = b >= 0 && b < bins;
                const int64_t h = h0 + (int64_t)b * kLanes;
                lng[k] = in ? a.lng[h] : __builtin_inf();
                cnt[k] = !in ? 0u : OBS == 2 ? a.obs_tot[h] : a.cnt[h];
            }
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                const int b = b0 + k * STEP;
                if (b >= nb) continue;
                const uint32_t at = (uint32_t)(b * T.pitch + jw * 8);
                lds_store_f64((uint32_t)o.lng + at, lng[k]);
                lds_store_u32((uint32_t)o.cnt + at / 2, OBS == 2 ? cycle_word(cnt[k]) : cnt[k]);
            }
        }
        if constexpr (OBS != 0)
            for (int i = tid; i < (o.total - o.sums) / 8; i += nth) lds_store_f64((uint32_t)(o.sums + 8 * i), 0.0);
        for (int i = tid; i < NP * L * SW; i += nth) {
            const int j = i & (SW - 1), qy = i / SW;
            const uint64_t w = j < G.nwalkers ? a.lat[G.lat_base + j + (int64_t)qy * kLanes] : 0ull;
            const uint32_t dst = (uint32_t)(o.lat + j * (NP * L * o.rowb + 4) + qy * o.rowb);
            for (int k = 0; k < o.rowb / 4; ++k) {
                const uint32_t x = (uint32_t)(w >> (16 * k)) & 0xffffu;
                lds_store_u32(dst + 4u * (uint32_t)k,
                              (x & 0xfu) | ((x & 0xf0u) << 4) | ((x & 0xf00u) << 8) | ((x & 0xf000u) << 12));
            }
        }
        if (walkers) {
            sweep_walkers_tree<MODEL, OBS>(a, G, S, T, o, nsweeps);
        } else {
            const int nrows = nsweeps * Mdl::kPasses * L, seg = tree_seg_rows(L);
            auto fill = [&](int r, int count) {
                tree_fill<MODEL>(G, S, o.ring, o.ringw, 8 * L, 2 * seg, tid - kLanes, sweep_base, r, count, tab);
            };
            fill(0, min(seg, nrows));
            __syncthreads();   // pairs with the walkers' barrier after the load
            for (int r = 0; r < nrows; r += seg) {
                const int next = r + seg;
                if (next < nrows) fill(next, min(seg, nrows - next));
                __syncthreads();   // pairs with the walkers' end-of-segment barrier
            }
        }
        __syncthreads();   // the walkers' last updates are in LDS
        // ---- store -----------------------------------------------------------
        for (int b = tid / SW; b < bins; b += STEP) {
            const int64_t h = h0 + (int64_t)b * kLanes;
            const uint32_t at = (uint32_t)((b + T.guard) * T.pitch + jw * 8);
            a.lng[h] = lds_f64((uint32_t)o.lng + at);
            const uint32_t cw = lds_u32_at((uint32_t)o.cnt + at / 2);
            if constexpr (OBS == 2) {
                const uint32_t t0 = a.obs_tot[h], updates = cycle_count(cw) - t0 % 1000u;
                a.obs_tot[h] = t0 + updates;
                a.cnt[h] += updates;
            } else {
                a.cnt[h] = cw;
            }
            if constexpr (OBS != 0) {
                // sums of bins without an update are zero
                double* p = a.obs + h * a.nobs;
                const uint32_t sum = (uint32_t)(o.sums + (b * T.pitch + jw * 8) * Mdl::kValues);
#pragma unroll
                for (int k = 0; k < Mdl::kValues; ++k) {
                    const double v = lds_f64(sum + 8u * (uint32_t)k);
                    if (v != 0.0) obs_add(p + (k / 3) * (OBS == 2 ? 4 : 3) + k % 3, v);
                }
            }
        }
        for (int i = tid; i < NP * L * SW; i += nth) {
            const int j = i & (SW - 1), qy = i / SW;
            if (j >= G.nwalkers) continue;
            const uint32_t src = (uint32_t)(o.lat + j * (NP * L * o.rowb + 4) + qy * o.rowb);
            uint64_t w = 0;
            for (int k = 0; k < o.rowb / 4; ++k) {
                const uint32_t v = lds_u32_at(src + 4u * (uint32_t)k);
                w |= (uint64_t)((v & 0xfu) | ((v >> 4) & 0xf0u) | ((v >> 8) & 0xf00u) | ((v >> 12) & 0xf000u)) << (16 * k);
            }
            a.lat[G.lat_base + j + (int64_t)qy * kLanes] = w;
        }
        __syncthreads();   // LDS is reused by the next group
    }
}

}  // namespace rewl
