// Set-up, replica-exchange, flatness/averaging and thermodynamics kernels.
#pragma once
#include "device.hpp"

namespace rewl {

__device__ __forceinline__ const DevSystem& sys_of(const KArgs& a, int g) { return a.sys[a.win[a.w_window[g]].sys]; }

__device__ __forceinline__ bool win_in_range(const DevWindow& W, double e) {
    const int t = trunc_half(e);
    return t >= W.phi_lo && t < W.phi_hi;
}
__device__ __forceinline__ int win_bin(const DevWindow& W, double e) {
    const int b = (int)((e - W.emin) / W.bs);
    return b < 0 ? 0 : (b >= W.nbins ? W.nbins - 1 : b);
}

// Ising2d::recalculate_state / Ashkin_Teller2d::recalculate_state
// (ising2d_hamiltonian.hpp:190-210, ashkin_teller2d_hamiltonian.hpp:193-217):
// the per-site terms of the model summed over the sites in order.
template <int M>
__device__ double recalc_energy(const DevSystem& S, const uint64_t* lat, int64_t base) {
    double E = 0.;
    for (int i = 0; i < S.N; ++i) {
        double own[Model<M>::kPlanes], nb[Model<M>::kPlanes][4];
        site_spins_mem<M>(S, lat, base, i, own, nb);
        E = Model<M>::add_site_energy(E, S.J, S.K, S.has_field, field_at(S, i), own, nb);
    }
    return E;
}

__global__ void k_recalc(KArgs a) {
    const int g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= a.num_walkers) return;
    const DevSystem& S = sys_of(a, g);
    a.w_E[g] = with_model(S.model, [&](auto m) { return recalc_energy<decltype(m)::value>(S, a.lat, a.w_lat[g]); });
}

// REWL_Walker::adjust_state_to_range (rewl_walker.hpp:71-115): one draw picks
// the starting site, then sites are scanned in order, accepting flips that move
// the energy toward the window.  Each proposal is change_state's (FP64, the
// reference's order); the flavour of a model with several advances at the
// wrap to site 0 and, with mode 0, also after site N-1 as change_state does
// (mode 1 keeps only the toggle at the wrap, so sigma and tau passes alternate).
template <int M>
__device__ void adjust_walker(const DevWindow& W, const DevSystem& S, uint64_t* lat, int64_t base, double& E,
                              int& fl, double u, uint64_t max_steps, int mode, int32_t* err) {
    uint64_t site = (uint64_t)(u * S.N);
    bool in = win_in_range(W, E);
    uint64_t steps = 0;
    while (!in) {
        if (++steps > max_steps) { atomicOr(err, 2); break; }
        ++site;
        if (site == (uint64_t)S.N) { site = 0; fl = Model<M>::next_flavour(fl); }
        const int plane = Model<M>::flip_plane(fl);
        const double En = proposal_energy_mem<M>(S, lat, base, (int)site, fl, E);
        if (mode == 0 && site == (uint64_t)(S.N - 1)) fl = Model<M>::next_flavour(fl);
        const bool low = trunc_half(E) < W.phi_lo, high = trunc_half(E) >= W.phi_hi;
        if ((low && En > E) || (!low && high && En <= E)) {
            const int x = (int)site % S.L, y = (int)site / S.L;
            lat[base + (int64_t)(plane * S.L + y) * kLanes] ^= (1ull << x);
            E = En;
        }
        in = win_in_range(W, E);
    }
}

template <bool REPLAY>
__global__ void k_adjust(KArgs a, uint64_t max_steps, int mode) {
    const int g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= a.num_walkers) return;
    const DevWindow W = a.win[a.w_window[g]];
    const DevSystem& S = a.sys[W.sys];
    double E = a.w_E[g];
    int fl = a.w_flavor[g];
    double u;
    if (REPLAY) {
        uint64_t c = a.w_cursor[g];
        if (c < a.ring_filled[g]) u = canonical_from_u64(a.ring[(int64_t)g * (int64_t)a.ring_cap + (int64_t)(c & (a.ring_cap - 1))]);
        else { u = 0.0; atomicOr(a.err, 1); }
        a.w_cursor[g] = c + 1;
    } else {
        u = canonical_from_u64(philox_u64(S.k0, S.k1, DOMAIN_INIT, (uint32_t)a.w_local[g], 0ull));
    }
    with_model(S.model, [&](auto m) {
        adjust_walker<decltype(m)::value>(W, S, a.lat, a.w_lat[g], E, fl, u, max_steps, mode, a.err);
        return 0;
    });
    a.w_E[g] = E;
    a.w_flavor[g] = fl;
}

// ---- std::shuffle restated for the exchange partner draw ------------------
// libstdc++ (GCC 11) shuffles n elements with a 64-bit engine by drawing swap
// positions in pairs from one uniform_int_distribution call, each call using
// Lemire's nearly divisionless reduction with a 128-bit product.
struct ExchStream {
    bool replay;
    const uint64_t* ring;
    uint64_t cap, filled;
    uint32_t k0, k1, walker;
    uint64_t cursor;
    int32_t* err;
    __device__ uint64_t next() {
        uint64_t c = cursor++;
        if (replay) {
            if (c < filled) return ring[c & (cap - 1)];
            atomicOr(err, 1);
            return ~0ull;   // ends any rejection loop below
        }
        return philox_u64(k0, k1, DOMAIN_EXCH, walker, c);
    }
    // uniform integer in [0, range) (Lemire 2019)
    __device__ uint64_t below(uint64_t range) {
        uint64_t x = next();
        uint64_t lo = x * range, hi = __umul64hi(x, range);
        if (lo < range) {
            const uint64_t threshold = (0ull - range) % range;
            for (int guard = 0; lo < threshold && guard < 4096; ++guard) {
                x = next();
                lo = x * range;
                hi = __umul64hi(x, range);
            }
        }
        return hi;
    }
};

__device__ void shuffle_partners(int* v, int n, ExchStream& st) {
    int i = 1;
    if (n <= 1) return;
    if ((n % 2) == 0) {
        const int j = (int)st.below(2);
        const int t = v[i]; v[i] = v[j]; v[j] = t;
        ++i;
    }
    while (i != n) {
        const uint64_t r = (uint64_t)i + 1;
        const uint64_t x = st.below(r * (r + 1));
        const int p1 = (int)(x / (r + 1)), p2 = (int)(x % (r + 1));
        int t = v[i]; v[i] = v[p1]; v[p1] = t; ++i;
        t = v[i]; v[i] = v[p2]; v[p2] = t; ++i;
    }
}

// The same shuffle of v[k] = first + k, k < n, by a wavefront.  The draws do
// not depend on one another unless one is rejected, so each lane takes its own
// and the swap positions that follow from it; swap i then puts v[p] at i and
// first + i, which nothing has moved yet, at p.  A draw that might be rejected
// (or lie beyond a replay stream) sends lane 0 through them in order.  v, pos:
// LDS, n ints each; the cursor is lane 0's.
__device__ __forceinline__ void wave_shuffle(int* v, int* pos, int n, int first, ExchStream& st, int lane) {
    if (n < 2) return;   // no draw
    const int odd = n & 1, draws = n / 2;   // n even: the first draw makes one swap
    bool in_order = false;
    for (int d = lane; d < draws; d += kLanes) {
        const uint64_t c = st.cursor + (uint64_t)d;
        const int i = odd ? 2 * d + 1 : 2 * d;
        const uint32_t r = (uint32_t)i + 1u;
        const uint64_t range = i ? (uint64_t)r * (r + 1u) : 2u;
        const bool there = !st.replay || c < st.filled;
        const uint64_t x = !there ? 0ull : st.replay ? st.ring[c & (st.cap - 1)]
                                                     : philox_u64(st.k0, st.k1, DOMAIN_EXCH, st.walker, c);
        in_order = in_order || !there || x * range < range;
        const uint32_t k = (uint32_t)__umul64hi(x, range);
        if (i) {
            pos[i] = (int)(k / (r + 1u));
            pos[i + 1] = (int)(k % (r + 1u));
        } else {
            pos[1] = (int)k;
        }
    }
    // the lanes read one another's positions: the compiler keeps the order of the
    // LDS operations, which end in order within a wavefront
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    if (__builtin_amdgcn_ballot_w64(in_order)) {
        if (lane == 0) shuffle_partners(v, n, st);
        return;
    }
    st.cursor += (uint64_t)draws;
    if (n <= kLanes) {
        // one entry per lane
        const int p = lane < n && lane > 0 ? pos[lane] : 0;
        int e = first + lane;
        for (int i = 1; i < n; ++i) {
            const int pi = __builtin_amdgcn_readlane(p, i), moved = __builtin_amdgcn_readlane(e, pi);
            e = lane == i ? moved : e;
            e = lane == pi ? first + i : e;
        }
        if (lane < n) v[lane] = e;
    } else if (lane == 0) {
        for (int i = 1; i < n; ++i) {
            const int pi = pos[i];
            v[i] = v[pi];
            v[pi] = first + i;
        }
    }
}

__device__ __forceinline__ ExchStream exch_stream(const KArgs& a, int g, bool replay) {
    const DevSystem& S = sys_of(a, g);
    ExchStream st;
    st.replay = replay;
    st.ring = replay ? a.ring + (int64_t)g * (int64_t)a.ring_cap : nullptr;
    st.cap = a.ring_cap;
    st.filled = replay ? a.ring_filled[g] : 0ull;
    st.k0 = S.k0; st.k1 = S.k1; st.walker = (uint32_t)a.w_local[g];
    st.cursor = a.w_cursor[g];
    st.err = a.err;
    return st;
}

constexpr int kMaxReplicas = 256;

// One replica-exchange phase for one pair of adjacent windows
// (rewl_simulation.hpp:228-346): replica 0 of the lower window shuffles the
// upper replicas into a random bijection, each pair accepts with
// p = exp(min(0, dlng_lower)) * exp(min(0, dlng_upper)) against a float
// uniform of the lower walker, accepted pairs swap energy and lattice, and
// every paired walker then increments its histogram at its current bin.
//
// Bound by latency: the shuffle, then a load behind each of several others.  A
// workgroup has a wavefront per replica pair (up to sixteen), which share out
// the lattices to swap and, with observables, the walkers to measure (a row per
// lane).  Measured, 31 pairs of windows of 64 replicas at L = 64, one wavefront
// with the shuffle on one lane -> this: 24.0 -> 11.2 us.
__global__ void __launch_bounds__(16 * kLanes) k_exchange(KArgs a, const int32_t* pairs, int npairs, int replay) {
    __shared__ int shuffled[kMaxReplicas];
    __shared__ int accept[kMaxReplicas];   // the shuffle's swap positions before
    __shared__ double s_cs[128];   // cos/sin(qmin k), k < L <= 64, for the correlators
    const int pi = blockIdx.x;
    if (pi >= npairs) return;
    const int lw = pairs[pi], uw = lw + 1;
    const DevWindow WL = a.win[lw], WU = a.win[uw];
    const DevSystem& S = a.sys[WL.sys];
    const int R = WL.R;
    const int tid = threadIdx.x, lane = tid & (kLanes - 1);
    const int wave = tid / kLanes, waves = (int)blockDim.x / kLanes;
    if (a.obs_corr) {
        const double qmin = 2. * acos(-1.) / (double)S.L;
        for (int k = tid; k < S.L; k += blockDim.x) {
            s_cs[k] = cos(qmin * (double)k);
            s_cs[S.L + k] = sin(qmin * (double)k);
        }
    }
    for (int k = tid; k < R; k += blockDim.x) shuffled[k] = R + k;
    __syncthreads();
    if (tid < kLanes) {
        ExchStream st = exch_stream(a, WL.first_walker, replay != 0);
        wave_shuffle(shuffled, accept, R, R, st, lane);
        if (tid == 0) a.w_cursor[WL.first_walker] = st.cursor;
    }
    __syncthreads();
    for (int r = tid; r < R; r += blockDim.x) {
        const int ga = WL.first_walker + r, gb = WU.first_walker + shuffled[r] - R;
        const double Ea = a.w_E[ga], Eb = a.w_E[gb];
        const int64_t ha = a.w_hist[ga], hb = a.w_hist[gb];
        double pa = 0., pb = 0.;
        if (win_in_range(WL, Eb))
            pa = exp(fmin(0., a.lng[ha + (int64_t)win_bin(WL, Ea) * kLanes] - a.lng[ha + (int64_t)win_bin(WL, Eb) * kLanes]));
        if (win_in_range(WU, Ea))
            pb = exp(fmin(0., a.lng[hb + (int64_t)win_bin(WU, Eb) * kLanes] - a.lng[hb + (int64_t)win_bin(WU, Ea) * kLanes]));
        const double p = pa * pb;
        int acc = 0;
        if (p != 0.) {
            ExchStream st = exch_stream(a, ga, replay != 0);
            const float u = (float)canonical_from_u64(st.next());
            a.w_cursor[ga] = st.cursor;
            acc = u < p;
        }
        accept[r] = acc;
        if (acc) {
            a.w_E[ga] = Eb;
            a.w_E[gb] = Ea;
            atomicAdd(a.exch_accepted, 1ull);
        }
    }
    __syncthreads();
    const int words = with_model(S.model, [](auto m) { return Model<decltype(m)::value>::kPlanes; }) * S.L;
    for (int r = wave; r < R; r += waves) {
        if (!accept[r]) continue;
        const int ga = WL.first_walker + r, gb = WU.first_walker + shuffled[r] - R;
        const int64_t la = a.w_lat[ga], lb = a.w_lat[gb];
        for (int k = lane; k < words; k += kLanes) {
            const uint64_t t = a.lat[la + (int64_t)k * kLanes];
            a.lat[la + (int64_t)k * kLanes] = a.lat[lb + (int64_t)k * kLanes];
            a.lat[lb + (int64_t)k * kLanes] = t;
        }
    }
    __syncthreads();
    const double fl = a.win_lnf[lw], fu = a.win_lnf[uw];
    for (int r = tid; r < R; r += blockDim.x) {
        const int ga = WL.first_walker + r, gb = WU.first_walker + shuffled[r] - R;
        const int64_t ia = a.w_hist[ga] + (int64_t)win_bin(WL, a.w_E[ga]) * kLanes;
        const int64_t ib = a.w_hist[gb] + (int64_t)win_bin(WU, a.w_E[gb]) * kLanes;
        a.cnt[ia] += 1u;
        a.lng[ia] += fl;
        a.cnt[ib] += 1u;
        a.lng[ib] += fu;
    }
    if (!a.obs) return;
    // the paired walkers' observables: a wavefront per walker
    for (int i = wave; i < 2 * R; i += waves) {
        const int r = i >> 1;
        const bool upper = (i & 1) != 0;
        const int g = upper ? WU.first_walker + shuffled[r] - R : WL.first_walker + r;
        const DevWindow& W = upper ? WU : WL;
        const int64_t h = a.w_hist[g] + (int64_t)win_bin(W, a.w_E[g]) * kLanes;
        const uint64_t* lt = a.lat + a.w_lat[g];
        with_model(S.model, [&](auto mt) {
            constexpr int M = decltype(mt)::value;
            constexpr int NP = Model<M>::kPlanes;
            // sums of plane 0, the last plane and their product
            // (lattice_magnetisations)
            const uint64_t s0 = lane < S.L ? lt[(int64_t)lane * kLanes] : 0ull;
            const uint64_t s1 = lane < S.L ? lt[(int64_t)((NP - 1) * S.L + lane) * kLanes] : 0ull;
            int m[3] = {(int)__popcll(s0), (int)__popcll(s1), (int)__popcll(s0 ^ s1)};
#pragma unroll
            for (int q = 0; q < 3; ++q) {
#pragma unroll
                for (int k = kLanes / 2; k >= 1; k >>= 1) m[q] += __shfl_xor(m[q], k, kLanes);
                m[q] = S.N - 2 * m[q];
            }
            if (lane == 0) {
                update_observables<M>(a.obs + h * a.nobs, S.N, m, a.obs_corr != 0);
                if (Model<M>::kDensities && a.dens) update_density(a.dens, h, S.N, m);
                if (a.obs_corr) {
                    const uint32_t t = a.obs_tot[h];
                    a.obs_tot[h] = t + 1u;
                    if (t % 1000u == 0u) add_correlators<M>(a.obs + h * a.nobs, lt, S.L, -1, nullptr, s_cs);
                }
            }
            return 0;
        });
    }
}

// ---- flatness, averaging, reset and ln f schedule, one wavefront per window --
template <typename T>
__device__ __forceinline__ T wave_min(T v) {
    for (int o = 32; o > 0; o >>= 1) { T w = __shfl_xor(v, o); v = w < v ? w : v; }
    return v;
}
template <typename T>
__device__ __forceinline__ T wave_max(T v) {
    for (int o = 32; o > 0; o >>= 1) { T w = __shfl_xor(v, o); v = w > v ? w : v; }
    return v;
}
template <typename T>
__device__ __forceinline__ T wave_sum(T v) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    return v;
}

constexpr int kMaxCheckBins = 8192;   // largest window the visited-support flatness test handles

// The sum of v(0) ... v(R-1) over a window's replicas, associated as the
// reference's MPI_Allreduce(SUM) over the window communicator associates it
// (rewl_simulation.hpp:383, 416-429) under MPICH's recursive doubling: with
// pof2 the largest power of two <= R and rem = R - pof2, the first 2 rem
// values are added in pairs, then the pof2 partial values are added as a
// balanced binary tree in rank order.  The tree is built left to right with
// a carry stack (one partial sum per level).
template <class F>
__device__ __forceinline__ double replica_sum(int R, F v) {
    int pof2 = 1, top = 0;
    while (pof2 * 2 <= R) { pof2 *= 2; ++top; }
    const int rem = R - pof2;
    double st[9];
    for (int k = 0; k < pof2; ++k) {
        double x = k < rem ? v(2 * k) + v(2 * k + 1) : v(k + rem);
        int lv = 0;
        while ((k >> lv) & 1) { x = st[lv] + x; ++lv; }
        st[lv] = x;
    }
    return st[top];
}

struct CheckParams {
    int32_t flatness_mode;
    int32_t schedule;
    int32_t reduce_logdos;
    int32_t average_mode;
    double flatness;
    double lnf_final;
    int64_t pending_sweeps;
};

// check_if_window_is_flat + average_and_redistribute_window + reset_counts +
// the ln f schedule (rewl_simulation.hpp:458-470, 361-454, 541-598;
// rewl_histograms.hpp:83-95, 115-152).
__global__ void __launch_bounds__(kLanes) k_check(KArgs a, CheckParams cp, int32_t* flat_out, int32_t* done_out) {
    const int wi = blockIdx.x;
    if (wi >= a.num_windows) return;
    const int lane = threadIdx.x;
    if (!a.win_active[wi]) {   // a retired system: state kept as it was
        if (lane == 0) {
            flat_out[wi] = 0;
            done_out[wi] = a.win_done[wi];
        }
        return;
    }
    const DevWindow W = a.win[wi];
    const int R = W.R, nb = W.nbins;
    const uint8_t* ex = a.exclude + W.excl_off;
    const bool oot_on = cp.schedule == 1 && a.win_oot[wi];

    // mode 3: bins that no replica of the window has ever visited are left out
    __shared__ uint8_t unseen[kMaxCheckBins];
    if (cp.flatness_mode == 3) {
        for (int b = lane; b < nb; b += kLanes) {
            bool seen = false;
            for (int r = 0; r < R && !seen; ++r) {
                const int64_t i = a.w_hist[W.first_walker + r] + (int64_t)b * kLanes;
                seen = (a.visits[i] + a.cnt[i]) != 0ull;
            }
            unseen[b] = seen ? 0 : 1;
        }
        __syncthreads();
    }
    bool flat = true;
    if (!oot_on) {
        for (int r = 0; r < R && flat; ++r) {
            const int64_t h = a.w_hist[W.first_walker + r];
            uint32_t mn = 0xFFFFFFFFu, mx = 0u;
            unsigned long long sum = 0ull;
            int ne = 0, zero = 0;
            for (int b = lane; b < nb; b += kLanes) {
                if (ex[b]) continue;
                if (cp.flatness_mode == 3 && unseen[b]) continue;
                const uint32_t c = a.cnt[h + (int64_t)b * kLanes];
                mn = c < mn ? c : mn;
                mx = c > mx ? c : mx;
                sum += c;
                ++ne;
                zero |= (c == 0u);
            }
            mn = wave_min(mn); mx = wave_max(mx); sum = wave_sum(sum); ne = wave_sum(ne); zero = wave_max(zero);
            bool f;
            if (ne == 0) f = true;
            else if (cp.flatness_mode == 0) f = !zero;
            else if (cp.flatness_mode == 1)
                f = (mn != 0u ? (static_cast<float>(mx - mn) / static_cast<float>(mn)) : 3.402823466e+38f) <= (float)cp.flatness;
            else f = (mn != 0u) && ((double)mn >= cp.flatness * ((double)sum / (double)ne));
            flat = flat && f;
        }
    }

    if (flat) {
        if (R > 1 && cp.average_mode == 1) {
            const double wgt = 1. / static_cast<double>(R);
            for (int b = lane; b < nb; b += kLanes) {
                const double acc = replica_sum(R, [&](int r) {
                    return wgt * a.lng[a.w_hist[W.first_walker + r] + (int64_t)b * kLanes];
                });
                for (int r = 0; r < R; ++r) a.lng[a.w_hist[W.first_walker + r] + (int64_t)b * kLanes] = acc;
            }
        } else if (R > 1) {
            for (int b = lane; b < nb; b += kLanes) {
                unsigned long long tot = 0ull;
                for (int r = 0; r < R; ++r) tot += a.cnt[a.w_hist[W.first_walker + r] + (int64_t)b * kLanes];
                if (tot == 0ull) continue;
                const double acc = replica_sum(R, [&](int r) {
                    const int64_t i = a.w_hist[W.first_walker + r] + (int64_t)b * kLanes;
                    return (static_cast<double>(a.cnt[i]) / static_cast<double>(tot)) * a.lng[i];
                });
                for (int r = 0; r < R; ++r) a.lng[a.w_hist[W.first_walker + r] + (int64_t)b * kLanes] = acc;
            }
        }
        __syncthreads();
        for (int r = 0; r < R; ++r) {
            const int64_t h = a.w_hist[W.first_walker + r];
            const double reducer = -a.lng[h] + 0.0;
            __syncthreads();
            for (int b = lane; b < nb; b += kLanes) {
                const int64_t i = h + (int64_t)b * kLanes;
                a.visits[i] += a.cnt[i];
                a.cnt[i] = 0u;
                if (cp.reduce_logdos) a.lng[i] += reducer;
            }
            __syncthreads();
        }
    }
    if (lane == 0) {
        int64_t sw = a.win_sweeps[wi] + cp.pending_sweeps;
        if (flat) {
            int64_t it = a.win_iter[wi];
            double lnf = a.win_lnf[wi];
            int oot = a.win_oot[wi];
            const double t = static_cast<double>(sw * it);
            if (cp.schedule == 1 && !oot) oot = (lnf <= 1. / t);
            const bool on = cp.schedule == 1 && oot;
            lnf = on ? (0.5 * lnf) * 0.0 + 1. / t : (0.5 * lnf);
            a.win_lnf[wi] = lnf;
            a.win_oot[wi] = oot;
            a.win_done[wi] = !(lnf >= cp.lnf_final);
            a.win_iter[wi] = it + 1;
            sw = 0;
        }
        a.win_sweeps[wi] = sw;
        flat_out[wi] = flat ? 1 : 0;
        done_out[wi] = a.win_done[wi];
    }
}

// Final intra-window average weighted by all-time visits
// (rewl_simulation.hpp:687 with simulation_incomplete == false), or by 1/R.
__global__ void __launch_bounds__(kLanes) k_finalize(KArgs a, int average_mode) {
    const int wi = blockIdx.x;
    if (wi >= a.num_windows) return;
    const DevWindow W = a.win[wi];
    const int R = W.R;
    if (R == 1) return;
    for (int b = threadIdx.x; b < W.nbins; b += kLanes) {
        if (average_mode == 1) {
            const double wgt = 1. / static_cast<double>(R);
            const double acc = replica_sum(R, [&](int r) {
                return wgt * a.lng[a.w_hist[W.first_walker + r] + (int64_t)b * kLanes];
            });
            for (int r = 0; r < R; ++r) a.lng[a.w_hist[W.first_walker + r] + (int64_t)b * kLanes] = acc;
            continue;
        }
        auto updates = [&](int r) {
            const int64_t i = a.w_hist[W.first_walker + r] + (int64_t)b * kLanes;
            return (double)(a.visits[i] + a.cnt[i]);
        };
        const double tot = replica_sum(R, updates);
        if (tot == 0.) continue;
        const double acc = replica_sum(R, [&](int r) {
            return (updates(r) / tot) * a.lng[a.w_hist[W.first_walker + r] + (int64_t)b * kLanes];
        });
        for (int r = 0; r < R; ++r) a.lng[a.w_hist[W.first_walker + r] + (int64_t)b * kLanes] = acc;
    }
}

// ---- multicanonical refinement (no counterpart in the reference) -------------
// Every (bin, walker) histogram entry of the context: visits and counts
// cleared (a fill kernel, not a memset, so that the step can be captured), or
// counts rolled into visits.
__global__ void k_hist_clear(KArgs a, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        a.visits[i] = 0ull;
        a.cnt[i] = 0u;
    }
}
__global__ void k_hist_roll(KArgs a, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        a.visits[i] += a.cnt[i];
        a.cnt[i] = 0u;
    }
}

// After sampling with fixed weights 1/g (ln f = 0) the histogram of a window
// is H(b) proportional to g(b) / g_est(b): ln g_est(b) + ln H(b) estimates
// ln g(b) up to the window's constant.  H sums the window's replicas; bins no
// replica visited keep their ln g.  One wavefront per window, lanes over bins;
// every replica receives the corrected curve (replica 0's ln g, which the
// preceding average made common to all replicas).
__global__ void __launch_bounds__(kLanes) k_refine(KArgs a) {
    const int wi = blockIdx.x;
    if (wi >= a.num_windows) return;
    const DevWindow W = a.win[wi];
    for (int b = threadIdx.x; b < W.nbins; b += kLanes) {
        unsigned long long H = 0ull;
        for (int r = 0; r < W.R; ++r) {
            const int64_t i = a.w_hist[W.first_walker + r] + (int64_t)b * kLanes;
            H += a.visits[i] + a.cnt[i];
        }
        if (H == 0ull) continue;
        const double v = a.lng[a.w_hist[W.first_walker] + (int64_t)b * kLanes] + log((double)H);
        for (int r = 0; r < W.R; ++r) a.lng[a.w_hist[W.first_walker + r] + (int64_t)b * kLanes] = v;
    }
}

// ---- canonical averages --------------------------------------------------------
// Thermodynamics::calculate_thermodynamics, trapezoid rule (thermodynamics.hpp:
// 77-236): at every temperature the bins' weights exp(ln g - E/T - max) and
// their sums, taken from the top bin down in FP64 as the reference takes them.
//
// A lane is a temperature and a workgroup of four wavefronts has 64 of them:
// chunks of 64 bins, whose weights the wavefronts compute a quarter each into
// LDS, and whose sums they then share out by sum, so that every sum still runs
// over the bins in the reference's order.  One thread per temperature for
// everything left the chip with less than one wavefront per SIMD, waiting on
// its own exp and two FP64 divisions per bin.  At 50 000 temperatures and the
// 2049 bins of an L = 64 curve: energy part 0.81 -> 0.34 ms, three
// observables 1.15 -> 0.41 ms (with the exp, about 40 FP64 instructions, on the
// half of the weights that are not zero; nearly FP64-issue bound).
constexpr int kThermoT = 64;       // temperatures per workgroup
constexpr int kThermoWaves = 4;
constexpr int kThermoChunk = 64;   // bins per chunk
constexpr int kThermoMaxObs = 16;

// E/T as the division rounds it: TAME (every energy and temperature an
// ordinary number, thermo_tame on the host) as a product with 1/T and one
// correction, whose residual is exact; else the division.
template <bool TAME>
struct ThermoT {
    double T, r;
    __device__ explicit ThermoT(double t) : T(t), r(1.0 / t) {}
    __device__ __forceinline__ double over(double E) const {
        if (!TAME) return E / T;
        const double q = E * r;
        return fma(fma(-q, T, E), r, q);
    }
};

// Largest of ln g - E/T over the bins; NaN where the top bin's is (the
// reference starts from it and moves on only to a larger value).
template <bool TAME>
__device__ __forceinline__ double thermo_max(const double* E, const double* lng, int nb, const ThermoT<TAME>& t,
                                             int wave, int lane, double (*part)[kThermoT]) {
    double m = -__builtin_inf();
#pragma unroll 4
    for (int b = wave; b < nb; b += kThermoWaves) {
        const double v = lng[b] - t.over(E[b]);
        m = m < v ? v : m;
    }
    part[wave][lane] = m;
    __syncthreads();
    const double top = lng[nb - 1] - t.over(E[nb - 1]);
    double mx = top;
    for (int w = 0; w < kThermoWaves; ++w) mx = mx < part[w][lane] ? part[w][lane] : mx;
    return mx;
}

// The weights of bins top, top - 1, ..., top - n + 1 into ws[0 .. n): a
// quarter per wavefront.  A weight below exp(-746) is zero; a wavefront whose
// temperatures all have it so does not compute it.
template <bool TAME>
__device__ __forceinline__ void thermo_weights(const double* E, const double* lng, int top, int n, const ThermoT<TAME>& t,
                                               double mx, int wave, int lane, double (*ws)[kThermoT]) {
#pragma unroll 2
    for (int i = wave; i < n; i += kThermoWaves) {
        const double x = (lng[top - i] - t.over(E[top - i])) - mx;
        double w = 0.;
        if (__builtin_amdgcn_ballot_w64(!(x < -746.))) w = exp(x);
        ws[i][lane] = w;
    }
}

template <bool TAME>
__global__ void __launch_bounds__(kThermoT* kThermoWaves) k_thermo(const double* E, const double* lng, int nb, int N,
                                                                   double tmin, double dT, int nT, double* out) {
    __shared__ double ws[kThermoChunk][kThermoT];
    __shared__ double part[kThermoWaves][kThermoT];
    const int lane = threadIdx.x & (kThermoT - 1);
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x / kThermoT);
    const int k = blockIdx.x * kThermoT + lane;   // a lane beyond the last temperature repeats it
    const double T = tmin + dT * (double)min(k, nT - 1);
    const ThermoT<TAME> t(T);
    const double mx = thermo_max(E, lng, nb, t, wave, lane, part);
    double s = 0.;   // wavefront 0: partition function, 1: U, 2: U^2, 3: S
    for (int top = nb - 1; top >= 0; top -= kThermoChunk) {
        const int n = min(kThermoChunk, top + 1);
        __syncthreads();   // the chunk before is summed
        thermo_weights(E, lng, top, n, t, mx, wave, lane, ws);
        __syncthreads();
        auto sum = [&](auto term) {
#pragma unroll 8
            for (int i = 0; i < n; ++i) {
                const int cb = top - i;
                s += term(cb, ws[i][lane], cb == 0 || cb == nb - 1);
            }
        };
        if (wave == 0) sum([&](int, double w, bool end) { return end ? w : 2. * w; });
        else if (wave == 1) sum([&](int cb, double w, bool end) { return end ? 0.5 * E[cb] * w : E[cb] * w; });
        else if (wave == 2) sum([&](int cb, double w, bool end) { return end ? 0.5 * E[cb] * E[cb] * w : E[cb] * E[cb] * w; });
        else sum([&](int cb, double w, bool end) { return end ? 0.5 * lng[cb] * w : lng[cb] * w; });
    }
    __syncthreads();
    part[wave][lane] = s;
    __syncthreads();
    if (wave != 0 || k >= nT) return;
    const double Z = 0.5 * part[0][lane];
    double U = part[1][lane], U2 = part[2][lane], Sx = part[3][lane];
    double* o = out + 5 * (size_t)k;
    o[0] = -T * (mx + log(Z)) / (double)N;
    U /= ((double)N * Z);
    U2 /= ((double)N * (double)N * Z);
    Sx /= ((double)N * Z);
    o[1] = U; o[2] = U2; o[3] = Sx;
    o[4] = (double)N * (U2 - U * U) / (T * T);
}

// Canonical averages of per-bin observables (the observable part of
// Thermodynamics::calculate_thermodynamics, thermodynamics.hpp:156-236):
// <O>(T) = sum_b t_b O_b w_b / Z, t_b = 1/2 at the two end bins and 1 inside,
// Z the trapezoid partition function.  Observable o is summed by wavefront
// o mod 4, Z by the last.
template <bool TAME>
__global__ void __launch_bounds__(kThermoT* kThermoWaves) k_thermo_obs(const double* E, const double* lng,
                                                                       const double* obs, int nb, int nobs, double tmin,
                                                                       double dT, int nT, double* out) {
    __shared__ double ws[kThermoChunk][kThermoT];
    __shared__ double part[kThermoWaves][kThermoT];
    const int lane = threadIdx.x & (kThermoT - 1);
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x / kThermoT);
    const int k = blockIdx.x * kThermoT + lane;
    const ThermoT<TAME> t(tmin + dT * (double)min(k, nT - 1));
    const double mx = thermo_max(E, lng, nb, t, wave, lane, part);
    constexpr int kMine = kThermoMaxObs / kThermoWaves;
    double Z = 0., acc[kMine];
#pragma unroll
    for (int j = 0; j < kMine; ++j) acc[j] = 0.;
    for (int top = nb - 1; top >= 0; top -= kThermoChunk) {
        const int n = min(kThermoChunk, top + 1);
        __syncthreads();   // the chunk before is summed
        thermo_weights(E, lng, top, n, t, mx, wave, lane, ws);
        __syncthreads();
        if (wave == kThermoWaves - 1) {   // the wavefront with the fewest observables
#pragma unroll 8
            for (int i = 0; i < n; ++i) Z += (top - i == 0 || top - i == nb - 1) ? ws[i][lane] : 2. * ws[i][lane];
        }
#pragma unroll
        for (int j = 0; j < kMine; ++j) {
            const int ob = wave + kThermoWaves * j;
            if (ob >= nobs) break;
#pragma unroll 8
            for (int i = 0; i < n; ++i) {
                const int cb = top - i;
                const double ov = obs[(size_t)cb * nobs + ob];
                acc[j] += (cb == 0 || cb == nb - 1) ? 0.5 * ov * ws[i][lane] : ov * ws[i][lane];
            }
        }
    }
    if (wave == kThermoWaves - 1) part[0][lane] = 0.5 * Z;   // the maxima were read before the first chunk
    __syncthreads();
    if (k >= nT) return;
    Z = part[0][lane];
#pragma unroll
    for (int j = 0; j < kMine; ++j)
        if (wave + kThermoWaves * j < nobs) out[(size_t)k * nobs + wave + kThermoWaves * j] = acc[j] / Z;
}

}  // namespace rewl
