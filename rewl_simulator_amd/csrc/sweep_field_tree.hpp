// Wang-Landau sweep, Philox mode, FP64 energies (random-field Ising,
// random-strain Ashkin-Teller, couplings off the integers): sixteen lanes per
// walker.
//
// Same chain, same draws and the same FP64 arithmetic as k_sweep and
// k_sweep_field (the reference's wang_landau_update, wang_landau.hpp:49-93).
// As in k_sweep_tree (sweep_tree.hpp, whose node numbering, decision masks and
// LDS hand-over are used here) four attempts are a binary tree of fifteen
// decisions, one lane each.  What differs is the energy, a sum that rounds at
// every step:
//
//  * E' = (E + a) + b with the model's terms a, b (Model::energy_terms), which
//    depend on the site's neighbours only.  A producer wavefront computes them
//    a row ahead, for every site and each value that the neighbours still to be
//    decided can take: the spin above (decided while the producer works) and
//    the left neighbour flipped or not; for the row's last site also with its
//    right neighbour, site 0, flipped.
//  * A node adds the terms of the attempts that its path accepts, in order:
//    fma(m, a, E) with m = 1 or 0 is E + a or E, rounded as in sequence.
//  * The bin of an energy is a function of the energy alone; every node
//    computes the bins of its path's states.  The quotient is a product with
//    1 / bin unless one lies so near an integer that it could truncate
//    differently (kBinMargin); then the wavefront divides.
//  * Two producer wavefronts: one computes the terms, the other the bounds
//    (accept_bound.hpp).
//  * A proposal outside the window reads a slot that holds ln g = +inf.
//
// What bounds it: the instruction stream of one wavefront (about 100 a step, a
// third of them FP64) and two LDS round trips per four attempts, 650 cycles;
// rows of up to four blocks wait for their producers, 2400-3000 cycles a row.
// Measured, one lane a walker -> this kernel: random-field Ising L = 30, 64
// walkers, 612 -> 184 cycles per attempt (a check cycle of 200 sweeps with its
// queries 45.8 -> 17.4 ms); 256 random-strain Ashkin-Teller systems of L = 16 to
// 48, 8192 walkers, 50 sweeps 73.9 -> 25.8 ms.  LDS for four workgroups per CU
// matters there: at 41 KB each three fit, 30.2 ms.  Reading the state back
// before the increments measured no better than after.
#pragma once
#include <type_traits>

#include "accept_bound.hpp"
#include "device.hpp"
#include "sweep_tree.hpp"

namespace rewl {

// LDS of one workgroup: four walkers (offsets in bytes).
struct FieldTreeLds {
    int32_t lat;           // [walker][plane][row] 64-bit words
    int32_t ring, ringw;   // acceptance bounds of two rows per walker
    int32_t rec, recw;     // energy terms of two rows per walker
    int32_t field;         // the field on one row
    int32_t state;         // [walker] state word and a sink
    int32_t hist, rowb;    // per bin: four ln g, four counts
    int32_t total;
};

// bytes of a site's terms for one case of its neighbours
constexpr __host__ __device__ int field_term_bytes(int terms) { return 8 * terms; }
// a row's records: four cases for each site of its blocks, then the last
// site's with site 0 flipped
constexpr __host__ __device__ int field_row_bytes(int terms, int L) {
    return (4 * tree_blocks(L) + 1) * 4 * field_term_bytes(terms);
}

__host__ __device__ inline FieldTreeLds field_tree_lds(int planes, int terms, int L, int nbins) {
    FieldTreeLds t;
    t.lat = 0;
    t.ring = kTreePerWave * planes * L * 8;
    t.ringw = 2 * 8 * (4 * tree_blocks(L)) + 16;
    t.rec = (t.ring + kTreePerWave * t.ringw + 15) & ~15;
    t.recw = 2 * field_row_bytes(terms, L) + 16;
    t.field = t.rec + kTreePerWave * t.recw;
    t.state = t.field + 8 * (L + (L & 1));
    t.hist = t.state + kTreePerWave * 32;
    t.rowb = kTreePerWave * 12;
    t.total = t.hist + (nbins + 1) * t.rowb;   // the last row: ln g = +inf
    return t;
}

// One case's terms.
template <int TERMS>
struct EnergyTerms {
    double a, b;
};
template <int TERMS>
__device__ __forceinline__ EnergyTerms<TERMS> lds_terms(uint32_t addr) {
    EnergyTerms<TERMS> t;
    if constexpr (TERMS == 1) {
        t.a = t.b = lds_f64(addr);
    } else {
        const f64x2 v = lds_f64x2(addr);
        t.a = v.x;
        t.b = v.y;
    }
    return t;
}
// E + a + b where m = 1, E where m = 0
template <int TERMS>
__device__ __forceinline__ double add_terms(const EnergyTerms<TERMS>& t, double m, double E) {
    return __builtin_fma(m, t.b, __builtin_fma(m, t.a, E));
}
// x if c, else y, both in registers (a choice between the members of a struct
// would be made between their addresses, and the struct kept in memory)
__device__ __forceinline__ double pick_f64(bool c, double x, double y) {
    return __hiloint2double(c ? __double2hiint(x) : __double2hiint(y), c ? __double2loint(x) : __double2loint(y));
}
template <int TERMS>
__device__ __forceinline__ EnergyTerms<TERMS> pick_terms(bool c, EnergyTerms<TERMS> x, EnergyTerms<TERMS> y) {
    EnergyTerms<TERMS> t;
    t.a = pick_f64(c, x.a, y.a);
    t.b = TERMS == 1 ? t.a : pick_f64(c, x.b, y.b);
    return t;
}

// What a lane keeps for its node (t: its depth; see TreeLane).
struct FieldTreeLane {
    int t;
    double m0, m1, m2;          // 1 where its path's first, second, third attempt flipped, else 0
    double f1, f2, f3;          // ln f where that earlier state exists, else 0
    uint32_t c1, c2, c3;        // offsets from a block's records: second site, third site, its own site
    uint32_t d3;                // from its own site's record to the one after a flip of the step before (root only)
    uint32_t mlo, mhi, want, want_tail, out0, out1;
};

// A block's input: the terms of the path's first three sites and of the lane's
// own site (y: the step before flipped its last site), its bound.
template <int TERMS>
struct FieldTreeInput {
    EnergyTerms<TERMS> s0x, s0y, s1, s2, s3x, s3y;
    double B;
};

// Addresses that a lane reads from, of the first of four blocks.
struct FieldTreePtr {
    uint32_t a0, a1, a2, a3;   // records: the block's first three sites, the lane's own
    uint32_t bound;
    uint32_t up;               // spins above the block's sites, from bit 0
};

// Block NB from p; a3 is p.a3 or, for the row's last block, past it.
template <int TERMS, int NB>
__device__ __forceinline__ void field_tree_read(const FieldTreeLane& c, FieldTreeInput<TERMS>& in, const FieldTreePtr& p,
                                                uint32_t a3) {
    constexpr uint32_t TB = field_term_bytes(TERMS), AT = NB * 16 * TB;
    constexpr int US = TERMS == 1 ? 4 : 5;   // log2(2 TB)
    const uint32_t x0 = p.a0 + (__builtin_amdgcn_ubfe(p.up, 4 * NB, 1) << US);
    const uint32_t x1 = p.a1 + (__builtin_amdgcn_ubfe(p.up, 4 * NB + 1, 1) << US);
    const uint32_t x2 = p.a2 + (__builtin_amdgcn_ubfe(p.up, 4 * NB + 2, 1) << US);
    const uint32_t x3 = a3 + (__builtin_amdgcn_ubfe(p.up, c.t + 4 * NB, 1) << US);
    in.s0x = lds_terms<TERMS>(x0 + AT);
    in.s0y = lds_terms<TERMS>(x0 + (AT + TB));
    in.s1 = lds_terms<TERMS>(x1 + AT);
    in.s2 = lds_terms<TERMS>(x2 + AT);
    in.s3x = lds_terms<TERMS>(x3 + AT);
    in.s3y = lds_terms<TERMS>(x3 + c.d3 + AT);
    in.B = lds_f64(p.bound + 32u * NB);
}

// An energy's bin is trunc(RN(x / bs)), x = RN(E - window minimum), clamped to
// the window.  z = RN(E inv + zero), with inv = RN(1 / bs) and zero = RN(margin
// - minimum inv), truncates to the same bin if its fraction is at least twice
// the margin: with M the larger of the window's bounds over bs, z - margin and
// x / bs differ by less than 8 M 2^-53, the margin is at least M 2^-48 and at
// least 2^-32, so x / bs and its rounding lie strictly between floor(z) and
// floor(z) + 1 (below zero either clamps to bin 0).
__device__ __forceinline__ double bin_margin(double emin, double emax, double bs) {
    return fmax(0x1p-32, fmax(fabs(emin), fabs(emax)) / bs * 0x1p-48);
}

// trunc(x) as v_cvt_u32_f64 does it: negative and NaN to 0, too large to 2^32 - 1
__device__ __forceinline__ uint32_t u32_of(double x) {
    uint32_t r;
    asm("v_cvt_u32_f64 %0, %1" : "=v"(r) : "v"(x));
    return r;
}

struct FieldTreeWindow {
    double emin, bs, inv, zero, near, lnf;   // near: twice the margin
    int plo, span;               // range test
    uint32_t last, none;         // last bin, the row of +inf
    uint32_t base;               // LDS address of bin 0's ln g
    uint32_t cnt;                // from a bin's ln g to its count
    uint32_t au, au_tail, state; // where the lane leaves a step's state, where its row reads it
    uint64_t lanes, lanes_tail;  // lanes of present walkers (that a row's last block uses)
};

typedef uint32_t u32x3v __attribute__((ext_vector_type(3)));
typedef __attribute__((address_space(3))) u32x3v lds_u32x3_t;

struct FieldTreeState {
    double E;
    uint32_t out;   // the step's flips, bit 31: its last site flipped
};

// Four attempts (or, TAIL, the row's last r < 5: lanes of deeper nodes have
// want_tail = never).  `in` is the block's input on entry, the next block's on
// exit, which is number NB from p.
template <int TERMS, bool TAIL, int NB>
__device__ __forceinline__ void field_tree_step(const FieldTreeLane& c, const FieldTreeWindow& w, FieldTreeState& st,
                                                FieldTreeInput<TERMS>& in, const FieldTreePtr& p, uint32_t a3) {
    const bool left = (int32_t)st.out < 0;
    const double E1 = add_terms(pick_terms(left, in.s0y, in.s0x), c.m0, st.E);
    const double E2 = add_terms(in.s1, c.m1, E1);
    const double C = add_terms(in.s2, c.m2, E2);
    const EnergyTerms<TERMS> t3 = pick_terms(left, in.s3y, in.s3x);
    const double N = (C + t3.a) + t3.b;
    const double B = in.B;
    // ---- bins ------------------------------------------------------------------
    double z1 = __builtin_fma(E1, w.inv, w.zero), z2 = __builtin_fma(E2, w.inv, w.zero);
    double zC = __builtin_fma(C, w.inv, w.zero), zN = __builtin_fma(N, w.inv, w.zero);
    // E1 and E2 are proposals, or the state, of lanes above this one
    const double nearest = fmin(__builtin_amdgcn_fract(zC), __builtin_amdgcn_fract(zN));
    if (__builtin_amdgcn_ballot_w64(nearest < w.near) & (TAIL ? w.lanes_tail : w.lanes)) {
        z1 = (E1 - w.emin) / w.bs;
        z2 = (E2 - w.emin) / w.bs;
        zC = (C - w.emin) / w.bs;
        zN = (N - w.emin) / w.bs;
    }
    const bool inside = (uint32_t)(trunc_half(N) - w.plo) < (uint32_t)w.span;
    const uint32_t b1 = min(u32_of(z1), w.last), b2 = min(u32_of(z2), w.last), bC = min(u32_of(zC), w.last);
    uint32_t bN = min(u32_of(zN), w.last);
    asm("" : "+v"(bN));   // a choice below, not a branch around the conversion
    bN = inside ? bN : w.none;
    constexpr uint32_t rowb = kTreePerWave * 12;
    const uint32_t sC = __umul24(bC, rowb) + w.base, sN = __umul24(bN, rowb) + w.base;
    double lc = lds_f64(sC), ln = lds_f64(sN);
    // the next block's reads go out while these are in flight
    if (!TAIL) field_tree_read<TERMS, NB>(c, in, p, a3);
    __builtin_amdgcn_sched_barrier(0);
    // ---- the decision: increments of the path's earlier attempts ---------------
    lc = add_if(bC == b1, c.f1, lc);
    ln = add_if(bN == b1, c.f1, ln);
    lc = add_if(bC == b2, c.f2, lc);
    ln = add_if(bN == b2, c.f2, ln);
    lc = lc + c.f3;
    ln = add_if(bN == bC, c.f3, ln);
    const bool acc = (ln - lc) < B;
    const uint64_t M = __builtin_amdgcn_ballot_w64(acc);
    const uint32_t pv = ((uint32_t)M & c.mlo) | ((uint32_t)(M >> 32) & c.mhi);
    const uint64_t path = __builtin_amdgcn_ballot_w64(pv == (TAIL ? c.want_tail : c.want));
    const double F = acc ? N : C;
    u32x3v uf;
    uf.x = (uint32_t)__double2loint(F);
    uf.y = (uint32_t)__double2hiint(F);
    uf.z = acc ? c.out1 : c.out0;
    const uint32_t sF = acc ? sN : sC;
    const uint32_t cF = sF + w.cnt, one = 1u;
    const uint32_t au = TAIL ? w.au_tail : w.au;
    // The last lane of the path hands the state over to its row, which reads
    // it back; the lanes on the path add ln f and a count, which nothing waits
    // for.  (One block: its wait, for all but the last two LDS operations of
    // the wavefront, is for the read, as LDS operations end in order.  Every
    // lane is active here.)
    u32x3v s;
    asm volatile("s_mov_b64 exec, %[path]\n\t"
                 "ds_write_b96 %[au], %[uf]\n\t"
                 "s_mov_b64 exec, -1\n\t"
                 "ds_read_b96 %[s], %[state]\n\t"
                 "s_mov_b64 exec, %[path]\n\t"
                 "ds_add_f64 %[sF], %[lnf]\n\t"
                 "ds_add_u32 %[cF], %[one]\n\t"
                 "s_mov_b64 exec, -1\n\t"
                 "s_waitcnt lgkmcnt(2)"
                 : [s] "=&v"(s)
                 : [path] "s"(path), [au] "v"(au), [uf] "v"(uf), [state] "v"(w.state), [sF] "v"(sF), [lnf] "v"(w.lnf),
                   [cF] "v"(cF), [one] "v"(one)
                 : "memory");
    st.E = f64_of(s.x, s.y);
    st.out = s.z;
}

// The walker wavefront: four walkers.
template <int MODEL>
__device__ __forceinline__ void sweep_walkers_field_tree(const KArgs& a, const DevGroup& G, const DevSystem& S,
                                                         const FieldTreeLds& o, int nsweeps) {
    using Mdl = Model<MODEL>;
    constexpr int NP = Mdl::kPlanes;
    constexpr int TERMS = Mdl::kEnergyTerms;
    constexpr uint32_t TB = field_term_bytes(TERMS), SB = 4 * TB;   // bytes of a case, of a site
    const int tid = threadIdx.x & 63;
    const int n = tid & 15, j = tid >> 4;
    const bool active = j < G.nwalkers;
    const int g = G.first_walker + (active ? j : 0);
    const DevWindow Wn = a.win[a.w_window[g]];
    const int L = S.L, nblk = tree_blocks(L), tail = L - 4 * (nblk - 1);

    FieldTreeLane c;
    FieldTreeWindow w;
    w.lnf = a.win_lnf[a.w_window[g]];
    const int t = n < 2 ? 0 : n < 4 ? 1 : n < 8 ? 2 : 3;
    {
        uint32_t anc = 0, want = 0, flips = 0;
        uint32_t act[3] = {0u, 0u, 0u};   // the path's outcomes
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            if (i >= t) continue;
            const int k = t - i;          // the ancestor that decides attempt i is n >> k
            act[i] = (uint32_t)(n >> (k - 1)) & 1u;
            anc |= 1u << (n >> k);
            want |= act[i] << (n >> k);
            flips |= act[i] << i;
        }
        c.t = t;
        c.m0 = act[0] ? 1.0 : 0.0;
        c.m1 = act[1] ? 1.0 : 0.0;
        c.m2 = act[2] ? 1.0 : 0.0;
        c.c1 = SB + TB * act[0];
        c.c2 = 2u * SB + TB * act[1];
        const uint32_t before = t == 0 ? 0u : t == 1 ? act[0] : t == 2 ? act[1] : act[2];
        c.c3 = (uint32_t)t * SB + TB * before;
        c.d3 = t == 0 ? TB : 0u;
        c.f1 = t >= 2 ? w.lnf : 0.0;
        c.f2 = t >= 3 ? w.lnf : 0.0;
        c.f3 = t >= 1 ? w.lnf : 0.0;
        const uint32_t sh = 16u * (uint32_t)(j & 1);
        const bool on = active && n > 0;
        c.mlo = on && j < 2 ? anc << sh : 0u;
        c.mhi = on && j >= 2 ? anc << sh : 0u;
        c.want = on ? want << sh : 0xffffffffu;
        c.want_tail = on && t < tail ? want << sh : 0xffffffffu;
        c.out0 = flips;
        c.out1 = flips | (1u << t) | 0x80000000u;
        w.lanes = __builtin_amdgcn_ballot_w64(on);
        w.lanes_tail = __builtin_amdgcn_ballot_w64(on && t < tail);
    }
    w.emin = Wn.emin;
    w.bs = Wn.bs;
    w.inv = 1.0 / Wn.bs;
    const double margin = bin_margin(Wn.emin, Wn.emax, Wn.bs);
    w.zero = margin - Wn.emin * w.inv;
    w.near = 2.0 * margin;
    w.plo = Wn.phi_lo;
    w.span = Wn.phi_hi - Wn.phi_lo;
    w.last = (uint32_t)(Wn.nbins - 1);
    w.none = (uint32_t)G.nbins;
    w.base = (uint32_t)(o.hist + 8 * j);
    w.cnt = (uint32_t)(8 * kTreePerWave - 4 * j);
    w.state = (uint32_t)(o.state + 32 * j);
    w.au = w.state + (t == 3 ? 0u : 16u);
    w.au_tail = w.state + (t == tail - 1 ? 0u : 16u);
    const uint32_t latw = (uint32_t)(o.lat + j * NP * L * 8);
    const uint32_t recw = (uint32_t)(o.rec + j * o.recw), rowrec = (uint32_t)field_row_bytes(TERMS, L);
    const uint32_t ringw = (uint32_t)(o.ring + j * o.ringw + 8 * t), rowring = 32u * (uint32_t)nblk;
    // to the last site's terms with site 0 flipped, for the lanes that decide it
    const uint32_t alt = t == tail - 1 ? SB * (uint32_t)(4 - t) : 0u;
    int fl = a.w_flavor[g];
    FieldTreeState st{a.w_E[g], 0u};
    // an absent walker's row never writes its state word
    if (n == 0) {
        u32x4v s;
        s.x = (uint32_t)__double2loint(st.E);
        s.y = (uint32_t)__double2hiint(st.E);
        s.z = s.w = 0u;
        *(lds_u32x4_t*)(uintptr_t)w.state = s;
    }
    const int nrows = nsweeps * Mdl::kPasses * L;
    const uint32_t nlast = (uint32_t)(nblk - 1);
    const int unused = 64 - 4 * nblk;   // bits of a row's flips below its first site, see fw
    int y = 0;
    uint32_t buf = 0;
    __syncthreads();   // LDS loaded
    u32x2v up = lds_u32x2(latw + 8u * (uint32_t)(Mdl::flip_plane(fl) * L + L - 1));   // the row above as rewritten
    __syncthreads();   // the first row's terms and bounds ready
    for (int r = 0; r < nrows; ++r) {
        const uint32_t at = latw + 8u * (uint32_t)(Mdl::flip_plane(fl) * L + y);
        const u32x2v cur = lds_u32x2(at);
        const uint32_t recs = recw + (buf ? rowrec : 0u);
        FieldTreePtr p{recs, recs + c.c1, recs + c.c2, recs + c.c3, ringw + (buf ? rowring : 0u), up.x};
        // opaque, so that every address of four blocks is one of these plus an
        // offset of its instruction
        auto hold = [&]() { asm("" : "+v"(p.a0), "+v"(p.a1), "+v"(p.a2), "+v"(p.a3), "+v"(p.bound)); };
        FieldTreeInput<TERMS> in;
        hold();
        field_tree_read<TERMS, 0>(c, in, p, p.a3);
        st.out = 0u;        // left of site 0 is site L - 1, as it stands
        u32x2v fw{0u, 0u};  // flips of the blocks done, the latest on top
        uint32_t past = 0;  // from the lane's own site in the last block to its record
        auto flips = [&]() {
            fw.x = __builtin_amdgcn_alignbit(fw.y, fw.x, 4);
            fw.y = __builtin_amdgcn_alignbit(st.out, fw.y, 4);
        };
        // block i + NB - 1; the next may be the last one
        auto block = [&](auto nb, uint32_t i) {
            constexpr int NB = decltype(nb)::value;
            field_tree_step<TERMS, false, NB>(c, w, st, in, p, p.a3 + (i + NB == nlast ? past : 0u));
            flips();
        };
        using std::integral_constant;
        block(integral_constant<int, 1>{}, 0u);
        past = (st.out & 1u) ? alt : 0u;   // site 0 as it is now
        // with two blocks the second's input was read before the first was decided
        if (nlast == 1u) field_tree_read<TERMS, 1>(c, in, p, p.a3 + past);
        if (nlast > 1u) block(integral_constant<int, 2>{}, 0u);
        if (nlast > 2u) block(integral_constant<int, 3>{}, 0u);
        if (nlast > 3u) block(integral_constant<int, 4>{}, 0u);
        uint32_t i = 0;
        auto next_four = [&]() {
            i += 4u;
            p.a0 += 16u * SB;
            p.a1 += 16u * SB;
            p.a2 += 16u * SB;
            p.a3 += 16u * SB;
            p.bound += 128u;
            up.x = __builtin_amdgcn_alignbit(up.y, up.x, 16);
            up.y >>= 16;
            p.up = up.x;
            hold();
        };
        next_four();
        for (; i + 4u <= nlast; next_four()) {
            block(integral_constant<int, 1>{}, i);
            block(integral_constant<int, 2>{}, i);
            block(integral_constant<int, 3>{}, i);
            block(integral_constant<int, 4>{}, i);
        }
        if (i < nlast) block(integral_constant<int, 1>{}, i);
        if (i + 1u < nlast) block(integral_constant<int, 2>{}, i);
        if (i + 2u < nlast) block(integral_constant<int, 3>{}, i);
        field_tree_step<TERMS, true, 0>(c, w, st, in, p, 0u);
        flips();
        const uint64_t f = (((uint64_t)fw.y << 32) | fw.x) >> unused;
        up.x = cur.x ^ (uint32_t)f;
        up.y = cur.y ^ (uint32_t)(f >> 32);
        if (n == 0) lds_store_u32x2(at, up);
        if (++y == L) {
            y = 0;
            fl = Mdl::next_flavour(fl);   // flavour switches after site N - 1
        }
        buf ^= 1u;
        __syncthreads();   // this row's terms and bounds consumed, the next row's written
    }
    if (active && n == 0) {
        a.w_E[g] = st.E;
        a.w_flavor[g] = fl;
    }
}

// Producer side: the energy terms of row r (rows of the launch, counted over
// its passes and sweeps) for every walker of the group, one wavefront.  A lane
// takes sites of one walker, whose flavour at the start of the launch is fl0; h
// is the field on the row's site `lane`.  The row above may be being decided, in the plane that it
// flips: that plane's spins are not used.
template <int MODEL>
__device__ __forceinline__ void field_tree_terms(const DevGroup& G, const DevSystem& S, const FieldTreeLds& o, int lane,
                                                 int r, int fl0, double h) {
    using Mdl = Model<MODEL>;
    constexpr int NP = Mdl::kPlanes;
    constexpr int TERMS = Mdl::kEnergyTerms;
    constexpr uint32_t TB = field_term_bytes(TERMS);
    const int L = S.L, j = lane & (kTreePerWave - 1);
    if (lane < L) lds_store_f64((uint32_t)(o.field + 8 * lane), h);
    if (j >= G.nwalkers) return;
    const int pass = r / L, y = r - pass * L;
    const int yu = y == 0 ? L - 1 : y - 1, yd = y == L - 1 ? 0 : y + 1;
    int fl = fl0, before = fl0;
    for (int k = 0; k < pass % Mdl::kPasses; ++k) fl = Mdl::next_flavour(fl);
    for (int k = 0; k < (pass + Mdl::kPasses - 1) % Mdl::kPasses; ++k) before = Mdl::next_flavour(before);
    const int pf = Mdl::flip_plane(fl);
    const int pu = y == 0 && r > 0 ? Mdl::flip_plane(before) : pf;   // the plane that the row above flipped
    const uint32_t lat = (uint32_t)(o.lat + j * NP * L * 8);
    const uint32_t dst = (uint32_t)(o.rec + j * o.recw) + ((r & 1) ? (uint32_t)field_row_bytes(TERMS, L) : 0u);
    for (int x = lane / kTreePerWave; x <= L; x += kLanes / kTreePerWave) {
        const bool again = x == L;   // the last site once more, with site 0 flipped
        const int xs = again ? L - 1 : x, xl = xs == 0 ? L - 1 : xs - 1, xr = xs == L - 1 ? 0 : xs + 1;
        const double hx = lds_f64((uint32_t)(o.field + 8 * xs));
        auto spin = [&](int q, int row, int col) {
            const uint32_t v = lds_u32_at(lat + 8u * (uint32_t)(q * L + row) + (col >= 32 ? 4u : 0u));
            return __hiloint2double((int)(0x3ff00000u | (((v >> (col & 31)) & 1u) << 31)), 0);
        };
        double own[NP], nb[NP][4], left[NP];
#pragma unroll
        for (int q = 0; q < NP; ++q) {
            own[q] = spin(q, y, xs);
            nb[q][0] = spin(q, yu, xs);
            left[q] = nb[q][1] = spin(q, y, xl);
            nb[q][2] = spin(q, y, xr);
            if (again && q == pf) nb[q][2] = -nb[q][2];
            nb[q][3] = spin(q, yd, xs);
        }
        const uint32_t at = dst + 4u * TB * (uint32_t)(again ? 4 * tree_blocks(L) : x);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
#pragma unroll
            for (int q = 0; q < NP; ++q) {
                if (q == pu) nb[q][0] = (k & 2) ? -1.0 : 1.0;
                nb[q][1] = (k & 1) && q == pf ? -left[q] : left[q];
            }
            double ta, tb;
            Mdl::energy_terms(S.J, S.K, S.has_field, hx, own, nb, fl, ta, tb);
            if constexpr (TERMS == 1) lds_store_f64(at + TB * (uint32_t)k, ta);
            else lds_store_f64x2(at + TB * (uint32_t)k, f64x2{ta, tb});
        }
    }
}

// One workgroup = one walker wavefront (four walkers) + two producers.  The grid
// has one for every group of the list; the loop is for a smaller one.
template <int MODEL>
__global__ void __launch_bounds__(3 * kLanes, 3)
    k_sweep_field_tree(KArgs a, const int32_t* groups, int ngroups, int nsweeps, uint64_t sweep_base) {
    using Mdl = Model<MODEL>;
    constexpr int NP = Mdl::kPlanes;
    constexpr int SW = kTreePerWave;
    constexpr int nth = 3 * kLanes;
    const int tid = threadIdx.x;
    const BoundEntry* tab = static_cast<const BoundEntry*>(a.bound_tab);
    if (tid < 64) __builtin_amdgcn_s_setprio(3);
    for (int gi = blockIdx.x; gi < ngroups; gi += gridDim.x) {
        const DevGroup G = a.grp[groups[gi]];
        const DevSystem S = a.sys[G.sys];
        const int L = S.L;
        const FieldTreeLds o = field_tree_lds(NP, Mdl::kEnergyTerms, L, G.nbins);
        // ---- load (LDS addresses are offsets: the kernel has no static LDS):
        // histograms, lattice; zeros where a row's last block has no site ------
        // a thread loads one walker's bins, four at a time in flight
        const int jw = tid & (SW - 1);
        const bool there = jw < G.nwalkers;
        const int64_t h0 = G.hist_base + jw;
        constexpr int STEP = nth / SW;
        for (int b0 = tid / SW; b0 <= G.nbins; b0 += 4 * STEP) {
            double lng[4];
            uint32_t cnt[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int b = b0 + k * STEP;
                const bool in = there && b < G.nbins;
                const int64_t h = h0 + (int64_t)b * kLanes;
                lng[k] = in ? a.lng[h] : __builtin_inf();
                cnt[k] = in ? a.cnt[h] : 0u;
            }
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int b = b0 + k * STEP;
                if (b > G.nbins) continue;
                const uint32_t at = (uint32_t)(o.hist + b * o.rowb);
                lds_store_f64(at + 8u * (uint32_t)jw, lng[k]);
                lds_store_u32(at + 8u * SW + 4u * (uint32_t)jw, cnt[k]);
            }
        }
        for (int i = tid; i < NP * L * SW; i += nth) {
            const int j = i & (SW - 1), qy = i / SW;
            const uint64_t v = j < G.nwalkers ? a.lat[G.lat_base + j + (int64_t)qy * kLanes] : 0ull;
            lds_store_u32x2((uint32_t)(o.lat + (j * NP * L + qy) * 8), u32x2v{(uint32_t)v, (uint32_t)(v >> 32)});
        }
        for (int i = tid; i < SW * o.recw / 8; i += nth) lds_store_f64((uint32_t)(o.rec + 8 * i), 0.0);
        if (tid < 64) {
            sweep_walkers_field_tree<MODEL>(a, G, S, o, nsweeps);
        } else {
            const int nrows = nsweeps * Mdl::kPasses * L, lane = tid & (kLanes - 1), j = lane & (SW - 1);
            const int fl0 = a.w_flavor[G.first_walker + (j < G.nwalkers ? j : 0)];
            const bool terms = tid < 2 * kLanes;
            auto field = [&](int r) { return lane < L ? field_at(S, r % L * L + lane) : 0.0; };
            double h = terms ? field(0) : 0.0;
            auto fill = [&](int r) {
                if (r >= nrows) return;
                if (terms) {
                    const double hr = h;
                    h = field(r + 1);   // arrives before the next row needs it
                    field_tree_terms<MODEL>(G, S, o, lane, r, fl0, hr);
                } else {
                    tree_fill<MODEL>(G, S, o.ring, o.ringw, 32 * tree_blocks(L), 2, lane, sweep_base, r, 1, tab);
                }
            };
            __syncthreads();   // LDS loaded
            fill(0);
            __syncthreads();   // pairs with the walkers' second barrier
            for (int r = 0; r < nrows; ++r) {
                fill(r + 1);
                __syncthreads();   // pairs with the walkers' end-of-row barrier
            }
        }
        __syncthreads();   // the walkers' last updates are in LDS
        // ---- store -----------------------------------------------------------
        for (int b = tid / SW; there && b < G.nbins; b += STEP) {
            const int64_t h = h0 + (int64_t)b * kLanes;
            const uint32_t at = (uint32_t)(o.hist + b * o.rowb);
            a.lng[h] = lds_f64(at + 8u * (uint32_t)jw);
            a.cnt[h] = lds_u32_at(at + 8u * SW + 4u * (uint32_t)jw);
        }
        for (int i = tid; i < NP * L * SW; i += nth) {
            const int j = i & (SW - 1), qy = i / SW;
            if (j >= G.nwalkers) continue;
            const u32x2v v = lds_u32x2((uint32_t)(o.lat + (j * NP * L + qy) * 8));
            a.lat[G.lat_base + j + (int64_t)qy * kLanes] = ((uint64_t)v.y << 32) | v.x;
        }
        __syncthreads();   // LDS is reused by the next group
    }
}

}  // namespace rewl
