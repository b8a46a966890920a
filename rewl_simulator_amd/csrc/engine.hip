// Host side of the REWL engine: the C ABI declared in include/rewl_c.h.
//
// One rewl_ctx owns every walker of one or more REWL systems on one GPU.  The
// host builds the windows (glazier EQUAL_WINDOWS, glazier.hpp:69-115), packs
// walkers into wavefront groups, uploads the tables, and then drives the
// device with four kinds of launch that replace the reference's per-rank loop
// and its MPI traffic: sweep (sixteen lanes per walker, or one), exchange (up to
// sixteen wavefronts per adjacent window pair), check (one wavefront per
// window) and finalize.
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <limits>
#include <memory>
#include <mutex>
#include <new>
#include <numeric>
#include <random>
#include <string>
#include <vector>

#include "../../include/rewl_c.h"
#include "aux_kernels.hpp"
#include "replay_fill.hpp"
#include "sweep_choice.hpp"
#include "sweep.hpp"
#include "sweep_fast.hpp"
#include "sweep_field.hpp"
#include "sweep_tuned.hpp"
#include "sweep_tree.hpp"
#include "sweep_field_tree.hpp"
#include "anneal.hpp"

namespace rewl {
// tuned_kernels.hip
const void* tuned_kernel(int model, int L, bool simple, int spec, int obs);
}  // namespace rewl

static_assert(REWL_ISING2D == 0 && REWL_ASHKIN_TELLER2D == 1, "the C ABI's model index is Model<M>'s M");

using namespace rewl;

namespace {

thread_local std::string g_err;

int fail(int code, const std::string& msg) {
    g_err = msg;
    return code;
}

#define HIP_TRY(expr)                                                                      \
    do {                                                                                   \
        hipError_t e_ = (expr);                                                            \
        if (e_ != hipSuccess)                                                              \
            return fail(REWL_ERR_DEVICE, std::string(#expr) + ": " + hipGetErrorString(e_)); \
    } while (0)

template <typename T>
struct DevBuf {
    T* p = nullptr;
    size_t n = 0;
    hipError_t alloc(size_t count) {
        n = count;
        if (count == 0) return hipSuccess;
        return hipMalloc((void**)&p, count * sizeof(T));
    }
    void release() {
        if (p) (void)hipFree(p);
        p = nullptr;
        n = 0;
    }
};

struct HostWindow {
    double emin, emax, bs;
    int nbins;
    int sys, first_walker, R;
};

struct HostSystem {
    rewl_system_desc d;
    int N, ndof;
    bool intpath;
    int twoJ, twoK;
    bool has_field;
    std::vector<double> field;
    std::vector<uint64_t> walker_seeds;
    int first_walker, first_window;
    std::vector<uint8_t> exclude;
};

// glazier::construct_windows, EQUAL_WINDOWS variant (glazier.hpp:69-115):
// equal widths, each window start snapped onto the previous window's bin grid,
// the end capped at the global maximum; windows are half-open [min, max).
std::vector<HostWindow> make_windows(const rewl_system_desc& d) {
    std::vector<HostWindow> out((size_t)d.num_windows);
    const double denom = 1 + (double)(d.num_windows - 1) * (1 - d.overlap);
    const double size = (d.e_max - d.e_min) / denom;
    for (int k = 0; k < d.num_windows; ++k) {
        double lo = d.e_min + (double)k * (1 - d.overlap) * size;
        double hi = lo + size;
        if (k != 0) {
            const double prev = out[k - 1].emin;
            lo = prev + d.bin_size * (double)((size_t)((lo - prev) / d.bin_size));
        }
        const size_t nb = (size_t)std::ceil((hi - lo) / d.bin_size);
        hi = lo + d.bin_size * (double)nb;
        while (hi > d.e_max) hi -= d.bin_size;
        out[k].emin = lo;
        out[k].emax = hi;
        out[k].bs = d.bin_size;
        out[k].nbins = (int)(size_t)((hi - lo) / d.bin_size);
    }
    return out;
}

bool integral(double v) { return std::isfinite(v) && std::floor(v) == v && std::fabs(v) < 1e9; }

// k_sweep_field_tree takes the FP64 systems of a context as long as their
// walkers, each counted as its system's degrees of freedom over the largest
// system's, are at most this many: 1024 workgroups, four per CU (registers and
// LDS allow no more).  A second round of them takes as long as the kernel with
// one lane per walker.  Measured, cycles per attempt, tree against lane: L = 30
// random-field Ising 198 / 570 at 1024 walkers, 212 / 571 at 2048, 260 / 573 at
// 4096, 643 / 570 at 8192; L = 32 186 / 441, 197 / 443, 243 / 442, 629 / 445;
// L = 48 random-strain Ashkin-Teller 173 / 687, 222 / 687, 271 / 690, 615 / 693.
// 8192 walkers of four sizes (16 to 48, 3698 counted so): 25.8 ms per 50 sweeps
// against 73.9.
constexpr int kFieldTreeMaxWalkers = 4096;

constexpr int kTunedL[5] = {16, 24, 32, 48, 64};
int tuned_index(int L) {
    for (int i = 0; i < 5; ++i)
        if (kTunedL[i] == L) return i;
    return -1;
}

// Whether the reference's range test on a system's integer energies is plainly
// min <= E < max: E = -1 collides with E = 0 in its +0.5 truncation, which
// matters only if E = -1 is reachable and a window bound is 0.
bool simple_range(const HostSystem& S, const std::vector<HostWindow>& win) {
    const ModelInfo mi = model_info(S.d.model);
    const long long g = mi.energy_step(S.twoJ, S.twoK);
    const long long e0 = mi.ground_energy(S.N, S.twoJ, S.twoK);
    bool zero_bound = false;
    for (int k = 0; k < S.d.num_windows; ++k)
        zero_bound = zero_bound || win[S.first_window + k].emin == 0.0 || win[S.first_window + k].emax == 0.0;
    const bool m1_reachable = g == 0 ? (e0 == -1) : (((-1 - e0) % g) == 0);
    return !(zero_bound && m1_reachable);
}

}  // namespace

struct rewl_ctx {
    rewl_params p{};
    std::vector<HostSystem> sys;
    std::vector<HostWindow> win;
    std::vector<DevGroup> groups;
    std::vector<int> w_window, w_local, w_group, w_lane;
    std::vector<int64_t> w_hist, w_lat;
    int num_walkers = 0;
    size_t hist_total = 0, lat_total = 0;
    // group lists per launch class: index = model * 2 + intpath
    std::vector<int32_t> class_groups[4];
    int class_maxbins[4] = {0, 0, 0, 0};
    bool class_packed[4] = {false, false, false, false};
    bool class_simple[4] = {true, true, true, true};   // plain [min, max) range test is exact
    int class_maxlanes[4] = {0, 0, 0, 0};
    int class_maxL[4] = {0, 0, 0, 0};
    bool class_field[4] = {false, false, false, false};   // FP64 class swept by k_sweep_field
    size_t class_field_lds[4] = {0, 0, 0, 0};             // its largest group's LDS
    int nprod = 1;                                      // producer wavefronts of the fast path
    DevBuf<int32_t> d_class_groups[4];
    // row-unrolled kernel: group lists per (model, lattice size kTunedL[i])
    std::vector<int32_t> tuned_groups[2][5];
    int tuned_maxbins[2][5] = {};
    int tuned_maxlanes[2][5] = {};
    bool tuned_simple[2][5] = {{true, true, true, true, true}, {true, true, true, true, true}};
    int tuned_guard[2][5] = {};                          // guard bins each side: max |Delta E| / bin size
    int tuned_nprod = 2;
    DevBuf<int32_t> d_tuned_groups[2][5];
    // sixteen-lanes-a-walker kernels (sweep_tree.hpp, sweep_field_tree.hpp):
    // group lists per model and energies (2 model + 1: FP64)
    std::vector<int32_t> tree_groups[4], tree_groups_all[4];
    DevBuf<int32_t> d_tree_groups[4];
    DevBuf<TreeScale> d_tree_scale;                      // per system
    size_t tree_lds_bytes[4] = {0, 0, 0, 0};             // the largest group's LDS
    std::vector<int32_t> pairs_even, pairs_odd;
    DevBuf<int32_t> d_pairs_even, d_pairs_odd;

    DevBuf<DevSystem> d_sys;
    DevBuf<DevWindow> d_win;
    DevBuf<DevGroup> d_grp;
    DevBuf<int32_t> d_w_window, d_w_local, d_w_flavor, d_err;
    DevBuf<int64_t> d_w_hist, d_w_lat, d_win_iter, d_win_sweeps;
    DevBuf<double> d_w_E, d_win_lnf, d_fields;
    DevBuf<uint64_t> d_w_cursor, d_lat, d_visits, d_ring, d_ring_filled;
    DevBuf<int32_t> d_win_oot, d_win_done, d_win_active;
    std::vector<uint8_t> sys_retired;   // rewl_params.retire: systems whose windows are all done
    // the lists before any retirement (rewl_refine runs every system again)
    std::vector<int32_t> class_groups_all[4], tuned_groups_all[2][5], pairs_even_all, pairs_odd_all;
    DevBuf<uint8_t> d_exclude;
    DevBuf<double> d_lng;
    DevBuf<uint32_t> d_cnt;
    DevBuf<unsigned long long> d_exch;
    DevBuf<BoundEntry> d_bound_tab;
    DevBuf<double> d_obs;       // observable sums (observables on)
    DevBuf<double> d_stage;     // rewl_set_logdos: one walker's ln g, copied linearly, then scattered
    // Pinned host memory that kernels write query results into (fetch), and
    // the flat / done flags of rewl_check: [2 * windows]
    std::mutex fetch_mu;
    void* h_fetch = nullptr;
    size_t h_fetch_bytes = 0;
    int32_t* h_check = nullptr;
    DevBuf<uint32_t> d_obs_tot; // updates so far per (bin, walker) (observables with correlators)
    DevBuf<uint32_t> d_dens;    // AT sigma-tau density counts [(hist index) * 1024 + cell] (densities on)
    int nobs = 0;

    // replay streams
    std::vector<std::mt19937_64> engines;
    std::vector<uint64_t> filled;
    uint64_t ring_cap = 0;
    uint64_t replay_left = 0;   // every stream holds at least this many words not consumed

    hipStream_t stream = nullptr;
    int lds_max = 65536;
    int flush_every = 1;
    uint64_t sweep_index = 0;
    int64_t pending_sweeps = 0;
    int exchange_waves = 1;   // of a k_exchange workgroup: the most replicas of a window, at most sixteen
    bool direction_even = true;
    bool in_windows = false;   // every walker inside its window (rewl_adjust_to_range ran)
    bool refining = false;     // between rewl_refine_begin and rewl_refine_end
    int64_t refine_since_exchange = 0;
    rewl_stats stats{};
    std::vector<std::pair<hipEvent_t, hipEvent_t>> ev_sweep;
    std::vector<hipEvent_t> ev_free;   // at most as many as ev_sweep has held: 2 x 257
    std::vector<int32_t> done_host;
    KArgs args{};
};

namespace {

void destroy_ctx(rewl_ctx* c) {
    if (!c) return;
    for (auto& e : c->ev_sweep) { (void)hipEventDestroy(e.first); (void)hipEventDestroy(e.second); }
    c->ev_sweep.clear();
    for (auto& e : c->ev_free) (void)hipEventDestroy(e);
    c->ev_free.clear();
    for (auto* b : {&c->d_w_window, &c->d_w_local, &c->d_w_flavor, &c->d_err, &c->d_win_oot, &c->d_win_done,
                    &c->d_win_active,
                    &c->d_pairs_even, &c->d_pairs_odd})
        b->release();
    for (auto& b : c->d_class_groups) b.release();
    for (auto& row : c->d_tuned_groups)
        for (auto& b : row) b.release();
    for (auto& b : c->d_tree_groups) b.release();
    c->d_tree_scale.release();
    c->d_w_hist.release(); c->d_w_lat.release(); c->d_win_iter.release(); c->d_win_sweeps.release();
    c->d_w_E.release(); c->d_win_lnf.release(); c->d_fields.release();
    c->d_w_cursor.release(); c->d_lat.release(); c->d_visits.release(); c->d_ring.release(); c->d_ring_filled.release();
    c->d_exclude.release(); c->d_lng.release(); c->d_cnt.release(); c->d_exch.release(); c->d_bound_tab.release(); c->d_obs.release(); c->d_obs_tot.release(); c->d_dens.release(); c->d_stage.release();
    c->d_sys.release(); c->d_win.release(); c->d_grp.release();
    if (c->h_fetch) (void)hipHostFree(c->h_fetch);
    if (c->h_check) (void)hipHostFree(c->h_check);
    if (c->stream) (void)hipStreamDestroy(c->stream);
    delete c;
}

template <typename T>
int upload(DevBuf<T>& b, const std::vector<T>& v, hipStream_t s) {
    HIP_TRY(b.alloc(v.size()));
    if (!v.empty()) HIP_TRY(hipMemcpyAsync(b.p, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice, s));
    return REWL_OK;
}

// New contents of a buffer no larger than its allocation (a list that shrank)
template <typename T>
int overwrite(DevBuf<T>& b, const std::vector<T>& v, hipStream_t s) {
    if (v.size() > b.n) return fail(REWL_ERR_INVALID, "internal: list grew beyond its buffer");
    if (!v.empty()) HIP_TRY(hipMemcpyAsync(b.p, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice, s));
    return REWL_OK;
}

// Query results.  A walker's column of a histogram is one element (or `width`)
// per row of 64 lanes; copied by hipMemcpy2D every element is a copy of its
// own (1.6 ms for the 236 doubles of an L = 64 window, 0.45 ms for 64 rows of
// spins), and even one value copied to pageable memory costs 29 us.  A gather
// kernel that writes into pinned memory of the context and one stream
// synchronisation take about 15 us for any of them.
template <typename T>
__global__ void k_gather(T* dst, const T* src, int64_t stride, int rows, int width) {
    const int n = rows * width;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
        dst[i] = src[(int64_t)(i / width) * stride + i % width];
}

// Room for `bytes` in the pinned buffer (fetch_mu held).
int reserve_fetch(rewl_ctx* c, size_t bytes) {
    if (bytes <= c->h_fetch_bytes) return REWL_OK;
    if (c->h_fetch) (void)hipHostFree(c->h_fetch);
    c->h_fetch = nullptr;
    c->h_fetch_bytes = 0;
    const size_t want = std::max<size_t>(bytes, 16384);
    HIP_TRY(hipHostMalloc(&c->h_fetch, want, hipHostMallocDefault));
    c->h_fetch_bytes = want;
    return REWL_OK;
}

// out[r * width + i] = src[r * stride + i] for r < rows, i < width, after all
// work queued on the context's stream.
template <typename T>
int fetch(rewl_ctx* c, const T* src, int64_t stride, int rows, int width, T* out) {
    std::lock_guard<std::mutex> lock(c->fetch_mu);
    const size_t n = (size_t)rows * (size_t)width;
    int rc;
    if ((rc = reserve_fetch(c, n * sizeof(T)))) return rc;
    const unsigned grid = (unsigned)std::min<size_t>(256, (n + 255) / 256);
    hipLaunchKernelGGL(k_gather<T>, dim3(grid), dim3(256), 0, c->stream, static_cast<T*>(c->h_fetch), src, stride, rows,
                       width);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipStreamSynchronize(c->stream));
    std::memcpy(out, c->h_fetch, n * sizeof(T));
    return REWL_OK;
}

// The changing part of a window's record, written to pinned memory.
struct WindowState {
    double lnf;
    int64_t iteration, sweeps;
    int32_t done, one_over_t;
};
__global__ void k_window_state(KArgs a, int wi, WindowState* out) {
    out->lnf = a.win_lnf[wi];
    out->iteration = a.win_iter[wi];
    out->sweeps = a.win_sweeps[wi];
    out->done = a.win_done[wi];
    out->one_over_t = a.win_oot[wi];
}

int resolve_sweep_events(rewl_ctx* c) {
    for (auto& e : c->ev_sweep) {
        HIP_TRY(hipEventSynchronize(e.second));
        float ms = 0.f;
        HIP_TRY(hipEventElapsedTime(&ms, e.first, e.second));
        c->stats.kernel_ms_sweep += ms;
        c->stats.sweep_launches += 1;
        c->ev_free.push_back(e.first);
        c->ev_free.push_back(e.second);
    }
    c->ev_sweep.clear();
    return REWL_OK;
}

int check_err_flag(rewl_ctx* c) {
    int32_t e = 0;
    int rc;
    if ((rc = fetch(c, c->d_err.p, 1, 1, 1, &e))) return rc;
    if (e & 1) return fail(REWL_ERR_REPLAY, "replay stream exhausted");
    if (e & 2) return fail(REWL_ERR_RANGE, "a walker could not be brought into its window");
    return REWL_OK;
}

int clear_err_bits(rewl_ctx* c, int32_t bits) {
    int32_t e = 0;
    int rc;
    if ((rc = fetch(c, c->d_err.p, 1, 1, 1, &e))) return rc;
    if (!(e & bits)) return REWL_OK;
    e &= ~bits;
    HIP_TRY(hipMemcpyAsync(c->d_err.p, &e, sizeof(int32_t), hipMemcpyHostToDevice, c->stream));
    HIP_TRY(hipStreamSynchronize(c->stream));
    return REWL_OK;
}

// Make sure every replay stream holds the `need` words that the next launch
// can consume at most.  The cursors are read, and the streams filled up, only
// when what earlier launches can have consumed leaves fewer (replay_left): with
// a read, a copy per walker and a wait for each, a fill takes longer than the
// five sweeps of an L = 12 launch.
int replay_topup(rewl_ctx* c, uint64_t need) {
    if (c->p.rng_mode != REWL_RNG_REPLAY) return REWL_OK;
    if (c->replay_left >= need) {
        c->replay_left -= need;
        return REWL_OK;
    }
    const int W = c->num_walkers;
    std::vector<uint64_t> cur((size_t)W);
    HIP_TRY(hipMemcpyAsync(cur.data(), c->d_w_cursor.p, (size_t)W * sizeof(uint64_t), hipMemcpyDeviceToHost, c->stream));
    HIP_TRY(hipStreamSynchronize(c->stream));
    const uint64_t C = c->ring_cap;
    const uint64_t room = std::min(replay_lack(W, cur.data(), c->filled.data(), C), kReplayStage);
    const std::unique_ptr<uint64_t[]> stage(new (std::nothrow) uint64_t[room]);
    if (!stage) return fail(REWL_ERR_DEVICE, "no host memory for the replay streams");
    hipError_t e = hipSuccess;
    const bool filled = replay_fill(
        W, cur.data(), c->filled.data(), C, stage.get(), room, [&](int g) { return c->engines[g](); },
        [&](int g, uint64_t pos, const uint64_t* w, uint64_t n) {
            e = hipMemcpyAsync(c->d_ring.p + (size_t)g * C + pos, w, n * sizeof(uint64_t), hipMemcpyHostToDevice,
                               c->stream);
            return e == hipSuccess;
        },
        [&] {
            e = hipStreamSynchronize(c->stream);
            return e == hipSuccess;
        });
    if (filled)
        e = hipMemcpyAsync(c->d_ring_filled.p, c->filled.data(), (size_t)W * sizeof(uint64_t), hipMemcpyHostToDevice,
                           c->stream);
    const hipError_t waited = hipStreamSynchronize(c->stream);   // stage goes
    HIP_TRY(e);
    HIP_TRY(waited);
    c->replay_left = C - std::min(need, C);
    return REWL_OK;
}

// Philox mode on the integer path: the throughput kernel (sweep_fast.hpp).
template <int MODEL, int NPROD>
void* fast_kernel(bool simple) {
    return simple ? (void*)k_sweep_fast<MODEL, true, NPROD> : (void*)k_sweep_fast<MODEL, false, NPROD>;
}

template <int MODEL>
int launch_sweep_fast(rewl_ctx* c, int cls, int nsweeps) {
    const int ng = (int)c->class_groups[cls].size();
    const int nb = c->class_maxbins[cls];
    const int np = c->nprod;
    const size_t lanes = (size_t)c->class_maxlanes[cls];
    const size_t lds = (size_t)nb * lanes * (sizeof(double) + sizeof(uint32_t)) +
                       (np ? 2 * (size_t)c->class_maxL[cls] * lanes * sizeof(float) : 0);
    const bool simple = c->class_simple[cls];
    void* kern = np == 0 ? fast_kernel<MODEL, 0>(simple) : np == 1 ? fast_kernel<MODEL, 1>(simple)
               : np == 2 ? fast_kernel<MODEL, 2>(simple) : fast_kernel<MODEL, 3>(simple);
    HIP_TRY(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    KArgs args = c->args;
    const int32_t* gl = c->d_class_groups[cls].p;
    uint64_t base = c->sweep_index;
    void* kargs[] = {&args, (void*)&gl, (void*)&ng, (void*)&nsweeps, (void*)&base};
    HIP_TRY(hipLaunchKernel((const void*)kern, dim3((unsigned)ng), dim3(kLanes * (1 + np)), kargs, lds, c->stream));
    HIP_TRY(hipGetLastError());
    return REWL_OK;
}

// Philox mode, FP64 energies (field models): sweep_field.hpp.
constexpr int kFieldProducers = 3;

// LDS of one k_sweep_field group: ln g and counts, the field, the bound ring.
size_t field_group_lds(int nbins, int nwalkers, int N, int L) {
    return (((size_t)nbins * nwalkers * 12 + 15) & ~(size_t)15) + (size_t)N * 8 + (2 * (size_t)L + 1) * nwalkers * 8;
}

size_t field_lds(const rewl_ctx* c, int cls) { return c->class_field_lds[cls]; }

template <int MODEL>
int launch_sweep_field(rewl_ctx* c, int cls, int nsweeps) {
    const int ng = (int)c->class_groups[cls].size();
    const size_t lds = field_lds(c, cls);
    // without observables the row-unrolled walker serves L in {16, 24, 32, 48}
    const void* kern = c->p.observables ? (const void*)k_sweep_field<MODEL, kFieldProducers, true>
                                        : (const void*)k_sweep_field<MODEL, kFieldProducers, false, true>;
    HIP_TRY(hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    KArgs args = c->args;
    const int32_t* gl = c->d_class_groups[cls].p;
    uint64_t base = c->sweep_index;
    void* kargs[] = {&args, (void*)&gl, (void*)&ng, (void*)&nsweeps, (void*)&base};
    HIP_TRY(hipLaunchKernel(kern, dim3((unsigned)ng), dim3(kLanes * (1 + kFieldProducers)), kargs, lds, c->stream));
    HIP_TRY(hipGetLastError());
    return REWL_OK;
}

// LDS bytes per (bin, walker) of the row-unrolled kernel's observable sums:
// with observables on, the moment sums stay in LDS for the launch
// (sweep_tuned.hpp); otherwise none.
size_t tuned_obs_bytes(int model, int observables) {
    return observables >= 1 ? 8 * (size_t)model_info(model).values : 0;
}

// A system in the row-unrolled kernel: guard bins (|Delta E| <= 4 (2J) (+ 4
// (2K)) on the integer path), LDS of a walker, walkers of a workgroup.
struct TunedShape {
    int guard, walkers;
    size_t per_walker;
};
TunedShape tuned_shape(const rewl_ctx* c, const HostSystem& S, int maxbins) {
    TunedShape t;
    const long long maxde =
        4LL * std::abs(S.twoJ) + (model_info(S.d.model).product_coupling ? 4LL * std::abs(S.twoK) : 0LL);
    const long long bs = (long long)c->win[S.first_window].bs;
    t.guard = (int)((maxde + bs - 1) / bs) + 1;
    t.per_walker = (size_t)(maxbins + 2 * t.guard) * kTunedSlot + (size_t)tuned_ring_stride(S.d.L) +
                   (size_t)maxbins * tuned_obs_bytes(S.d.model, c->p.observables);
    // observables = 2: the cos/sin table of the correlator after the rings
    const size_t room = (size_t)c->lds_max - (c->p.observables == 2 ? 16 * (size_t)S.d.L : 0);
    t.walkers = std::min(kLanes, (int)(room / t.per_walker));
    return t;
}

// Philox mode, integer path, L in kTunedL: the row-unrolled kernel (sweep_tuned.hpp).
template <int MODEL, int L>
int launch_sweep_tuned(rewl_ctx* c, int li, int nsweeps) {
    const auto& list = c->tuned_groups[MODEL][li];
    const int ng = (int)list.size();
    if (ng == 0) return REWL_OK;
    const size_t lanes = (size_t)c->tuned_maxlanes[MODEL][li];
    const int guard = c->tuned_guard[MODEL][li];
    const size_t lds = ((size_t)c->tuned_maxbins[MODEL][li] + 2 * guard) * lanes * kTunedSlot +
                       (size_t)tuned_ring_stride(L) * lanes + (c->p.observables == 2 ? 16 * (size_t)L : 0) +
                       (size_t)c->tuned_maxbins[MODEL][li] * lanes * tuned_obs_bytes(MODEL, c->p.observables);
    const bool simple = c->tuned_simple[MODEL][li];
    const int np = c->tuned_nprod;
    // sweep_kernel 2: no speculation, 3 (and auto): next slot for both outcomes,
    // 4: that and the next ln g read ahead
    const int sk = c->p.sweep_kernel;
    const int spec = sk == 2 ? 0 : sk == 4 ? 2 : 1;
    const void* kern = tuned_kernel(MODEL, L, simple, spec, spec == 1 ? c->p.observables : 0);
    if (!kern) return fail(REWL_ERR_INVALID, "internal: no row-unrolled kernel of this form");
    HIP_TRY(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    KArgs args = c->args;
    const int32_t* gl = c->d_tuned_groups[MODEL][li].p;
    uint64_t base = c->sweep_index;
    int guard_arg = guard;
    void* kargs[] = {&args, (void*)&gl, (void*)&ng, (void*)&nsweeps, (void*)&base, (void*)&guard_arg};
    HIP_TRY(hipLaunchKernel((const void*)kern, dim3((unsigned)ng), dim3(kLanes * (1 + np)), kargs, lds, c->stream));
    HIP_TRY(hipGetLastError());
    return REWL_OK;
}

// Events around a launch of sweeps (stats: kernel_ms_sweep), taken from a
// pool.  Recorded by themselves they are packets of their own before and after
// the kernel; when the launch is one kernel they ride on it.
struct SweepEvents {
    hipEvent_t start, stop;
    bool one_kernel;
};

int take_event(rewl_ctx* c, hipEvent_t* e) {
    if (c->ev_free.empty()) {
        HIP_TRY(hipEventCreate(e));
        return REWL_OK;
    }
    *e = c->ev_free.back();
    c->ev_free.pop_back();
    return REWL_OK;
}

template <int MODEL>
int launch_sweep_tree(rewl_ctx* c, int nsweeps, const SweepEvents& ev) {
    constexpr int list = 2 * MODEL;
    const int ng = (int)c->tree_groups[list].size();
    if (ng == 0) return REWL_OK;
    const size_t lds = c->tree_lds_bytes[list];
    void (*const kern)(KArgs, const TreeScale*, const int32_t*, int, int, uint64_t) =
        c->p.observables == 2 ? k_sweep_tree<MODEL, 2> : c->p.observables ? k_sweep_tree<MODEL, 1> : k_sweep_tree<MODEL, 0>;
    HIP_TRY(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    KArgs args = c->args;
    const TreeScale* scale = c->d_tree_scale.p;
    const int32_t* gl = c->d_tree_groups[list].p;
    int ngroups = ng;
    uint64_t base = c->sweep_index;
    void* kargs[] = {&args, (void*)&scale, (void*)&gl, &ngroups, &nsweeps, &base};
    HIP_TRY(hipExtLaunchKernel((const void*)kern, dim3((unsigned)ng), dim3(2 * kLanes), kargs, lds, c->stream,
                               ev.one_kernel ? ev.start : nullptr, ev.one_kernel ? ev.stop : nullptr, 0));
    HIP_TRY(hipGetLastError());
    return REWL_OK;
}

template <int MODEL>
int launch_sweep_field_tree(rewl_ctx* c, int nsweeps, const SweepEvents& ev) {
    constexpr int list = 2 * MODEL + 1;
    const int ng = (int)c->tree_groups[list].size();
    if (ng == 0) return REWL_OK;
    const size_t lds = c->tree_lds_bytes[list];
    HIP_TRY(hipFuncSetAttribute((const void*)k_sweep_field_tree<MODEL>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                (int)lds));
    KArgs args = c->args;
    const int32_t* gl = c->d_tree_groups[list].p;
    int ngroups = ng;
    uint64_t base = c->sweep_index;
    void* kargs[] = {&args, (void*)&gl, &ngroups, &nsweeps, &base};
    HIP_TRY(hipExtLaunchKernel((const void*)k_sweep_field_tree<MODEL>, dim3((unsigned)ng), dim3(3 * kLanes), kargs, lds,
                               c->stream, ev.one_kernel ? ev.start : nullptr, ev.one_kernel ? ev.stop : nullptr, 0));
    HIP_TRY(hipGetLastError());
    return REWL_OK;
}

template <int MODEL>
int launch_tuned_all(rewl_ctx* c, int nsweeps) {
    int rc;
    if ((rc = launch_sweep_tuned<MODEL, 16>(c, 0, nsweeps))) return rc;
    if ((rc = launch_sweep_tuned<MODEL, 24>(c, 1, nsweeps))) return rc;
    if ((rc = launch_sweep_tuned<MODEL, 32>(c, 2, nsweeps))) return rc;
    if ((rc = launch_sweep_tuned<MODEL, 48>(c, 3, nsweeps))) return rc;
    return launch_sweep_tuned<MODEL, 64>(c, 4, nsweeps);
}

template <int MODEL, bool INTP>
int launch_sweep_class(rewl_ctx* c, int cls, int nsweeps) {
    const int ng = (int)c->class_groups[cls].size();
    if (ng == 0) return REWL_OK;
    const bool obs = c->p.observables != 0;
    const bool corr = c->p.observables == 2;
    if (INTP && c->p.rng_mode == REWL_RNG_PHILOX && !obs) return launch_sweep_fast<MODEL>(c, cls, nsweeps);
    if (!INTP && c->class_field[cls]) return launch_sweep_field<MODEL>(c, cls, nsweeps);
    const bool packed = c->class_packed[cls];
    const int nb = c->class_maxbins[cls];
    // with correlators: ln g, counts and update counts at the group's stride, then the cos/sin table
    const size_t lds = corr ? (((size_t)nb * c->class_maxlanes[cls] * 16 + 15) & ~(size_t)15) +
                                  16 * (size_t)c->class_maxL[cls]
                            : (size_t)nb * kLanes * sizeof(double) +
                                  (packed ? (size_t)((nb + 1) / 2) : (size_t)nb) * kLanes * sizeof(uint32_t);
    const bool replay = c->p.rng_mode == REWL_RNG_REPLAY;
    const dim3 grid((unsigned)ng), block(kLanes);
    const int32_t* gl = c->d_class_groups[cls].p;
    const int fe = c->flush_every;
    void (*kern)(KArgs, const int32_t*, int, int, uint64_t, int);
    if (corr) {
        kern = replay ? k_sweep<MODEL, INTP, true, false, 2> : k_sweep<MODEL, INTP, false, false, 2>;
    } else if (obs) {
        if (replay) kern = packed ? k_sweep<MODEL, INTP, true, true, 1> : k_sweep<MODEL, INTP, true, false, 1>;
        else kern = packed ? k_sweep<MODEL, INTP, false, true, 1> : k_sweep<MODEL, INTP, false, false, 1>;
    } else {
        if (replay) kern = packed ? k_sweep<MODEL, INTP, true, true, 0> : k_sweep<MODEL, INTP, true, false, 0>;
        else kern = packed ? k_sweep<MODEL, INTP, false, true, 0> : k_sweep<MODEL, INTP, false, false, 0>;
    }
    HIP_TRY(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL(kern, grid, block, lds, c->stream, c->args, gl, ng, nsweeps, c->sweep_index, fe);
    HIP_TRY(hipGetLastError());
    return REWL_OK;
}

int launch_sweep_kernels(rewl_ctx* c, int nsweeps, SweepEvents& ev) {
    int rc;
    int others = 0, trees = 0;
    for (const auto& l : c->class_groups) others += l.empty() ? 0 : 1;
    for (const auto& m : c->tuned_groups)
        for (const auto& l : m) others += l.empty() ? 0 : 1;
    for (const auto& l : c->tree_groups) trees += l.empty() ? 0 : 1;
    ev.one_kernel = others == 0 && trees == 1;
    if (!ev.one_kernel) HIP_TRY(hipEventRecord(ev.start, c->stream));
    if ((rc = launch_sweep_class<0, false>(c, 0, nsweeps))) return rc;
    if ((rc = launch_sweep_class<0, true>(c, 1, nsweeps))) return rc;
    if ((rc = launch_sweep_class<1, false>(c, 2, nsweeps))) return rc;
    if ((rc = launch_sweep_class<1, true>(c, 3, nsweeps))) return rc;
    if ((rc = launch_tuned_all<0>(c, nsweeps))) return rc;
    if ((rc = launch_tuned_all<1>(c, nsweeps))) return rc;
    if ((rc = launch_sweep_tree<0>(c, nsweeps, ev))) return rc;
    if ((rc = launch_sweep_tree<1>(c, nsweeps, ev))) return rc;
    if ((rc = launch_sweep_field_tree<0>(c, nsweeps, ev))) return rc;
    if ((rc = launch_sweep_field_tree<1>(c, nsweeps, ev))) return rc;
    if (!ev.one_kernel) HIP_TRY(hipEventRecord(ev.stop, c->stream));
    return REWL_OK;
}

int launch_sweeps(rewl_ctx* c, int nsweeps) {
    SweepEvents ev{};
    int rc = take_event(c, &ev.start);
    if (rc == REWL_OK) rc = take_event(c, &ev.stop);
    if (rc == REWL_OK) rc = launch_sweep_kernels(c, nsweeps, ev);
    if (rc != REWL_OK) {
        if (ev.start) c->ev_free.push_back(ev.start);
        if (ev.stop) c->ev_free.push_back(ev.stop);
        return rc;
    }
    c->ev_sweep.emplace_back(ev.start, ev.stop);
    if (c->ev_sweep.size() > 256) return resolve_sweep_events(c);
    return REWL_OK;
}

// Byte scale of a system's states and energy changes in k_sweep_tree, and
// whether that kernel takes the system: the state is energy x pitch / bin,
// stored energy changes are signed bytes and their weight too.
bool tree_scale(const rewl_system_desc& d, int twoJ, int twoK, TreeScale* out) {
    const bool kq = model_info(d.model).product_coupling;
    const long long bin = (long long)d.bin_size;
    if (bin < 1 || bin > 256) return false;
    const long long aJ = std::abs((long long)twoJ), aK = kq ? std::abs((long long)twoK) : 0;
    if (aJ > 1000000 || aK > 1000000) return false;
    const long long g = std::gcd(2 * aJ, 2 * aK);   // energy changes: twoJ (4 - 2 k) + twoK (4 - 2 q)
    if (g == 0) return false;
    TreeScale t{};
    const long long pitch = std::max<long long>(8 * kTreePerWave, bin);
    const long long unit = pitch / bin * g;
    long long m = 1;
    while (unit / m > 127 && unit % (2 * m) == 0) m *= 2;
    if (unit / m > 127) return false;
    const long long most = kq ? 63 : 127;
    if (4 * aJ / g * m > most || 4 * aK / g * m > most) return false;
    // four proposals ahead of a state inside the window
    const long long reach = 4 * (4 * aJ + 4 * aK);
    t.pitch = (int)pitch;
    t.g = (int)g;
    t.m = (int)m;
    t.w = (int)(unit / m);
    t.guard = (int)((reach + bin - 1) / bin) + 1;
    *out = t;
    return true;
}

int max_ndof(const rewl_ctx* c) {
    int m = 1;
    for (auto& s : c->sys) m = std::max(m, s.ndof);
    return m;
}

// A launch has one workgroup per group and the dispatcher starts them in
// list order: the longest first (attempts per sweep, DoF of the system),
// so that when a batch has more groups than the chip holds, the groups
// that start last are short ones (longest-processing-time order).
void longest_first(const rewl_ctx* c, std::vector<int32_t>& list) {
    std::stable_sort(list.begin(), list.end(), [&](int32_t x, int32_t y) {
        return c->sys[(size_t)c->groups[(size_t)x].sys].ndof > c->sys[(size_t)c->groups[(size_t)y].sys].ndof;
    });
}

// The rows of the four-walker groups' lattices and histograms.  A row is kLanes
// wide and sixteen consecutive groups share it: with rows of their own they
// took sixteen times the memory, which creation and the passes over all
// walkers went through (512 Ashkin-Teller walkers with observables 2 created in
// 1.38 ms instead of 0.91; 256 replicas in 16 windows at L = 64 finalized in
// 669 us instead of 555).  Workgroups go to the eight XCDs in turn, and a line that
// two XCDs write costs (a sweep and exchange of 2048 walkers at L = 64 1.2 %
// when neighbours on the list shared rows), so the list takes groups of eight
// rows in turn: the sixteen of a row run on one XCD.  Fewer than 128 groups
// of a size are spread over eight rows likewise.
void place_tree_groups(rewl_ctx* c) {
    constexpr size_t kXcds = 8, kSides = kLanes / kTreePerWave;
    for (auto& list : c->tree_groups) {
        longest_first(c, list);
        auto ndof = [&](size_t i) { return c->sys[(size_t)c->groups[(size_t)list[i]].sys].ndof; };
        std::vector<int32_t> order(list.size());
        for (size_t first = 0, n; first < list.size(); first += n) {
            for (n = 1; n < kXcds * kSides && first + n < list.size() && ndof(first + n) == ndof(first);) ++n;
            size_t next = first;   // groups of rows 0, 1, ... one after the other
            for (size_t x = 0; x < std::min(kXcds, n); ++x) {
                const size_t sides = n / kXcds + (x < n % kXcds ? 1 : 0);
                size_t nb = 0;
                for (size_t side = 0; side < sides; ++side) {
                    const int32_t gid = list[next + side];
                    DevGroup& G = c->groups[(size_t)gid];
                    G.hist_base = (int64_t)(c->hist_total + side * kTreePerWave);
                    G.lat_base = (int64_t)(c->lat_total + side * kTreePerWave);
                    for (int j = 0; j < G.nwalkers; ++j) {
                        c->w_hist[(size_t)(G.first_walker + j)] = G.hist_base + j;
                        c->w_lat[(size_t)(G.first_walker + j)] = G.lat_base + j;
                    }
                    nb = std::max(nb, (size_t)G.nbins);
                    order[first + x + side * kXcds] = gid;
                }
                const HostSystem& S = c->sys[(size_t)c->groups[(size_t)list[next]].sys];
                c->hist_total += nb * kLanes;
                c->lat_total += (size_t)model_info(S.d.model).planes * (size_t)S.d.L * kLanes;
                next += sides;
            }
        }
        list.swap(order);
    }
}

// Device buffers of one rewl_anneal call, released on every return path.
struct AnnealBuffers {
    DevBuf<DevSystem> sys;
    DevBuf<double> fields, beta, ebuf, emin, efin;
    DevBuf<uint64_t> lat;
    DevBuf<unsigned long long> sweeps;
    ~AnnealBuffers() {
        sys.release(); fields.release(); beta.release(); ebuf.release(); emin.release(); efin.release();
        lat.release(); sweeps.release();
    }
};

}  // namespace

extern "C" {

const char* rewl_last_error(void) { return g_err.c_str(); }
const char* rewl_version(void) { return "rewl-mi355x 0.1"; }

int rewl_device_count(int* count) {
    int n = 0;
    hipError_t e = hipGetDeviceCount(&n);
    if (e != hipSuccess) n = 0;
    if (count) *count = n;
    return REWL_OK;
}

int rewl_create(const rewl_system_desc* systems, int32_t num_systems, const rewl_params* params, rewl_ctx** out) {
    if (!systems || num_systems <= 0 || !params || !out) return fail(REWL_ERR_INVALID, "null argument");
    *out = nullptr;
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0)
        return fail(REWL_ERR_NO_DEVICE, "no HIP device visible: the REWL engine runs only on the GPU");
    const rewl_params& P = *params;
    if (P.sweeps_per_check <= 0 || P.sweeps_per_exchange <= 0 || P.lnf_initial <= 0 ||
        (P.flatness_mode < 0 || P.flatness_mode > 3) || (P.schedule < 0 || P.schedule > 1) ||
        (P.rng_mode < 0 || P.rng_mode > 1) || (P.adjust_mode < 0 || P.adjust_mode > 1) || (P.average_mode < 0 || P.average_mode > 1) || (P.sweep_kernel < 0 || P.sweep_kernel > 4) || (P.observables < 0 || P.observables > 2) || (P.retire < 0 || P.retire > 1) || P.walkers_per_group < 0 || P.walkers_per_group > kLanes ||
        (P.densities < 0 || P.densities > 1))
        return fail(REWL_ERR_INVALID, "invalid rewl_params");
    if (P.densities && !P.observables)
        return fail(REWL_ERR_INVALID, "densities are recorded with the observables: set observables >= 1");

    rewl_ctx* c = new rewl_ctx();
    c->p = P;
    auto bail = [&](int code) { destroy_ctx(c); return code; };

    // ---- systems and windows ------------------------------------------------
    int walker = 0;
    for (int si = 0; si < num_systems; ++si) {
        const rewl_system_desc& d = systems[si];
        if (d.model != REWL_ISING2D && d.model != REWL_ASHKIN_TELLER2D) return bail(fail(REWL_ERR_INVALID, "unknown model"));
        if (d.L < 2 || d.L > 64) return bail(fail(REWL_ERR_INVALID, "L must lie in [2, 64]"));
        if (d.num_windows < 1 || d.replicas_per_window < 1 || d.replicas_per_window > kMaxReplicas)
            return bail(fail(REWL_ERR_INVALID, "num_windows >= 1 and 1 <= replicas_per_window <= 256 required"));
        if (!(d.bin_size > 0) || !(d.e_max > d.e_min) || d.overlap < 0 || d.overlap >= 1)
            return bail(fail(REWL_ERR_INVALID, "bad energy range, bin size or overlap"));
        HostSystem S;
        S.d = d;
        S.N = d.L * d.L;
        S.ndof = model_info(d.model).planes * S.N;
        if (d.field) S.field.assign(d.field, d.field + S.N);
        S.d.field = nullptr;
        S.has_field = d.field != nullptr || d.h != 0.0;
        const double tJ = 2 * d.J, tK = 2 * d.K;
        S.twoJ = (int)tJ;
        S.twoK = (int)tK;
        auto wins = make_windows(d);
        bool ip = !S.has_field && integral(tJ) && (!model_info(d.model).product_coupling || integral(tK));
        for (auto& w : wins) {
            if (w.nbins < 1) return bail(fail(REWL_ERR_INVALID, "a window has no bins"));
            if (P.flatness_mode == REWL_FLAT_MIN_OVER_MEAN_VISITED && w.nbins > kMaxCheckBins)
                return bail(fail(REWL_ERR_INVALID, "visited-support flatness handles at most 8192 bins per window"));
            const double lb = std::log2(w.bs);
            ip = ip && integral(w.emin) && integral(w.emax) && integral(w.bs) && integral(lb);
        }
        S.intpath = ip;
        S.first_walker = walker;
        S.first_window = (int)c->win.size();
        const size_t gbins = (size_t)std::llround((d.e_max - d.e_min) / d.bin_size) + 1;
        S.exclude.assign(gbins, 0);
        if (d.exclude_bins)
            for (size_t b = 0; b + 1 < gbins; ++b) S.exclude[b] = d.exclude_bins[b];
        if (d.walker_seeds) S.walker_seeds.assign(d.walker_seeds, d.walker_seeds + (size_t)d.num_windows * d.replicas_per_window);
        for (int k = 0; k < d.num_windows; ++k) {
            HostWindow w = wins[k];
            w.sys = si;
            w.R = d.replicas_per_window;
            w.first_walker = walker + k * d.replicas_per_window;
            c->win.push_back(w);
        }
        for (int k = 0; k < d.num_windows; ++k)
            for (int r = 0; r < d.replicas_per_window; ++r) {
                c->w_window.push_back(S.first_window + k);
                c->w_local.push_back(k * d.replicas_per_window + r);
            }
        walker += d.num_windows * d.replicas_per_window;
        c->sys.push_back(std::move(S));
    }
    c->num_walkers = walker;
    for (const HostSystem& S : c->sys)
        c->exchange_waves = std::max(c->exchange_waves, std::min<int>(S.d.replicas_per_window, 16));
    const int W = walker;

    // ---- device limits ------------------------------------------------------
    int dev = 0;
    (void)hipGetDevice(&dev);
    int lds = 0;
    if (hipDeviceGetAttribute(&lds, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) == hipSuccess && lds > 0)
        c->lds_max = lds;
    if (hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) != hipSuccess)
        return bail(fail(REWL_ERR_DEVICE, "hipStreamCreate failed"));

    // ---- systems swept with sixteen lanes a walker -------------------------------
    // When the caller asks for no particular kernel or launch shape and the
    // context has few enough walkers (sweep_choice.hpp, kFieldTreeMaxWalkers).
    std::vector<uint8_t> tree_sys(c->sys.size(), 0);
    std::vector<TreeScale> tree_scales(c->sys.size());
    {
        int cus = 0;
        if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus < 1) cus = 256;
        const bool shape_free = P.rng_mode == REWL_RNG_PHILOX && P.sweep_kernel == 0 && P.producers == 0 &&
                                P.walkers_per_group == 0 && !P.densities;
        auto max_bins = [&](const HostSystem& S) {
            int nb = 1;
            for (int k = 0; k < S.d.num_windows; ++k) nb = std::max(nb, c->win[S.first_window + k].nbins);
            return nb;
        };
        // bytes of LDS of a workgroup, 0 if the kernel does not take the system
        auto group_lds = [&](const HostSystem& S, TreeScale* t) -> size_t {
            if (!tree_scale(S.d, S.twoJ, S.twoK, t)) return 0;
            const int nb = max_bins(S);
            const long long bytes = (long long)(nb + 2 * t->guard) * t->pitch * 2;
            if (bytes > 4LL * c->lds_max) return 0;   // keeps the sums below in range
            const ModelInfo m = model_info(S.d.model);
            const size_t lds = (size_t)tree_lds(m.planes, S.d.L, nb, t->pitch, t->guard, P.observables, m.values).total;
            return lds <= (size_t)c->lds_max ? lds : 0;
        };
        // Of a model's systems with an unrolled row: workgroups and largest LDS
        // here and, by lattice side, with one lane per walker.
        struct Launch {
            long long groups = 0, lds = 0;
        } tree_launch[2], lane_launch[2][5];
        for (size_t si = 0; shape_free && si < c->sys.size(); ++si) {
            const HostSystem& S = c->sys[si];
            const int li = tuned_index(S.d.L), walkers = S.d.num_windows * S.d.replicas_per_window;
            if (W > tree_walker_limit(model_info(S.d.model).planes, S.d.L, P.observables, li >= 0)) continue;
            if (!S.intpath || S.d.L < kTreeMinL || !simple_range(S, c->win)) continue;
            const size_t lds = group_lds(S, &tree_scales[si]);
            tree_sys[si] = lds > 0;
            if (!lds || li < 0) continue;
            const TunedShape t = tuned_shape(c, S, max_bins(S));
            if (t.walkers < 1) continue;
            auto add = [&](Launch& l, int per, size_t bytes) {
                l.groups += (walkers + per - 1) / per;
                l.lds = std::max(l.lds, (long long)bytes);
            };
            add(tree_launch[S.d.model], kTreePerWave, lds);
            add(lane_launch[S.d.model][li], t.walkers, (size_t)t.walkers * t.per_walker);
        }
        for (int m = 0; m < 2; ++m) {
            long long lane_rounds = 0;
            for (const Launch& l : lane_launch[m]) lane_rounds += workgroup_rounds(l.groups, l.lds, c->lds_max, cus);
            const Launch& l = tree_launch[m];
            if (tree_pays(P.observables, workgroup_rounds(l.groups, l.lds, c->lds_max, cus),
                          workgroups_per_cu(l.lds, c->lds_max) == 1, lane_rounds))
                continue;
            for (size_t si = 0; si < c->sys.size(); ++si)
                if (c->sys[si].d.model == m && tuned_index(c->sys[si].d.L) >= 0) tree_sys[si] = 0;
        }
        int64_t attempts = 0, largest = 1;   // of the FP64 systems, per sweep: all walkers', one walker's at most
        for (const HostSystem& S : c->sys) {
            if (S.intpath) continue;
            attempts += (int64_t)S.ndof * S.d.num_windows * S.d.replicas_per_window;
            largest = std::max<int64_t>(largest, S.ndof);
        }
        const bool few = attempts <= largest * kFieldTreeMaxWalkers;
        for (size_t si = 0; shape_free && !P.observables && few && si < c->sys.size(); ++si) {
            const HostSystem& S = c->sys[si];
            if (S.intpath || S.d.L < kTreeMinL) continue;
            const int nb = max_bins(S);
            if ((long long)nb * 12 * kTreePerWave > c->lds_max) continue;   // keeps the sum below in range
            const ModelInfo m = model_info(S.d.model);
            if (field_tree_lds(m.planes, m.energy_terms, S.d.L, nb).total <= c->lds_max) tree_sys[si] = 1;
        }
    }

    // ---- wavefront groups -----------------------------------------------------
    c->w_group.assign(W, 0);
    c->w_lane.assign(W, 0);
    c->w_hist.assign(W, 0);
    c->w_lat.assign(W, 0);
    for (int si = 0; si < (int)c->sys.size(); ++si) {
        const HostSystem& S = c->sys[si];
        const int nw = S.d.num_windows * S.d.replicas_per_window;
        const int planes = model_info(S.d.model).planes;
        int maxbins = 1;
        for (int k = 0; k < S.d.num_windows; ++k) maxbins = std::max(maxbins, c->win[S.first_window + k].nbins);
        // The throughput kernel keeps FP64 ln g and u32 counts of every walker
        // of the group in LDS with the bin stride equal to the group size, so
        // a window of many bins gets fewer walkers per wavefront.
        // observables on: every class runs k_sweep, which tracks the magnetisations
        const bool obs = P.observables != 0;
        const bool fast = S.intpath && P.rng_mode == REWL_RNG_PHILOX && !obs;
        // field models in Philox mode: k_sweep_field (sweep_kernel 1 or producers < 0 keep k_sweep)
        const bool field_fast = !S.intpath && P.rng_mode == REWL_RNG_PHILOX && P.producers >= 0 &&
                                P.sweep_kernel != 1 && (!obs || (P.observables == 1 && !P.densities));
        c->nprod = P.producers < 0 ? 0 : (P.producers == 0 ? 1 : std::min<int>(P.producers, 3));
        c->tuned_nprod = P.producers == 0 ? 7 : std::min<int>(std::max<int>(P.producers, 1), 7);
        const int li = tuned_index(S.d.L);
        // observables (without densities) also run on the row-unrolled kernel, in its default form
        const bool tuned_obs = P.observables >= 1 && !P.densities && P.sweep_kernel != 2 && P.sweep_kernel != 4;
        const bool tree = tree_sys[(size_t)si] != 0;
        const bool tuned = !tree && S.intpath && P.rng_mode == REWL_RNG_PHILOX && (!obs || tuned_obs) && P.producers >= 0 &&
                           li >= 0 && P.sweep_kernel != 1;
        if (P.sweep_kernel >= 2 && !tuned)
            return bail(fail(REWL_ERR_INVALID, "the row-unrolled kernel needs the Philox integer path, producers >= 0 "
                                               "and L in {16, 24, 32, 48, 64}; with observables, sweep_kernel 0 or 3 "
                                               "and no densities"));
        const bool field_tree = tree && !S.intpath;
        int wpg = tree ? kTreePerWave : kLanes;
        int guard = 0;
        if (tuned) {
            const TunedShape t = tuned_shape(c, S, maxbins);
            guard = t.guard;
            wpg = t.walkers;
        }
        else if (fast && !tree)
            wpg = std::min(kLanes, (int)((size_t)c->lds_max /
                                         ((size_t)(maxbins + 1) * 12 + (c->nprod ? 8 * (size_t)S.d.L : 0))));
        else if (field_fast && !tree) {
            const long long room = (long long)c->lds_max - 16 - 8LL * S.N;
            wpg = room <= 0 ? 0 : std::min<long long>(kLanes, room / (12LL * maxbins + 16LL * S.d.L));
        } else if (!tree && P.observables == 2) {
            // ln g, counts and update counts per (bin, walker), plus the cos/sin table
            const long long room = (long long)c->lds_max - 16 - 16LL * S.d.L;
            wpg = room <= 0 ? 0 : std::min<long long>(kLanes, room / (16LL * maxbins));
        }
        // a system's windows are accepted or refused whichever kernel takes them
        // (the walkers of the context decide that): with moments, off the
        // unrolled-row sizes, those that the generic kernel holds
        if (tree && P.observables == 1 && li < 0 &&
            ((size_t)maxbins * 8 + (size_t)((maxbins + 1) / 2) * 4) * kLanes > (size_t)c->lds_max)
            wpg = 0;
        if (P.walkers_per_group > 0) wpg = std::min(wpg, (int)P.walkers_per_group);
        if (wpg < 1) return bail(fail(REWL_ERR_INVALID, "window too wide for LDS: " + std::to_string(maxbins) + " bins"));
        if (!tree) {
            const bool simple = simple_range(S, c->win);
            if (tuned) {
                if (!simple) c->tuned_simple[S.d.model][li] = false;
                c->tuned_maxlanes[S.d.model][li] = std::max(c->tuned_maxlanes[S.d.model][li], wpg);
                c->tuned_guard[S.d.model][li] = std::max(c->tuned_guard[S.d.model][li], guard);
            } else {
                const int cls = S.d.model * 2 + (S.intpath ? 1 : 0);
                if (!simple) c->class_simple[cls] = false;
                c->class_maxlanes[cls] = std::max(c->class_maxlanes[cls], wpg);
                c->class_maxL[cls] = std::max(c->class_maxL[cls], S.d.L);
                if (field_fast) c->class_field[cls] = true;
            }
        }
        for (int off = 0; off < nw; off += wpg) {
            DevGroup G{};
            G.sys = si;
            G.first_walker = S.first_walker + off;
            G.nwalkers = std::min(wpg, nw - off);
            int nb = 0;
            for (int j = 0; j < G.nwalkers; ++j) nb = std::max(nb, c->win[c->w_window[G.first_walker + j]].nbins);
            G.nbins = nb;
            if (!tree) {   // else place_tree_groups
                G.hist_base = (int64_t)c->hist_total;
                G.lat_base = (int64_t)c->lat_total;
                c->hist_total += (size_t)nb * kLanes;
                c->lat_total += (size_t)planes * S.d.L * kLanes;
            }
            const int gid = (int)c->groups.size();
            for (int j = 0; j < G.nwalkers; ++j) {
                const int g = G.first_walker + j;
                c->w_group[g] = gid;
                c->w_lane[g] = j;
                c->w_hist[g] = G.hist_base + j;
                c->w_lat[g] = G.lat_base + j;
            }
            if (tree) {
                const int list = 2 * S.d.model + (field_tree ? 1 : 0);
                c->tree_groups[list].push_back(gid);
                const TreeScale& t = tree_scales[(size_t)si];
                const int terms = model_info(S.d.model).energy_terms;
                const int bytes = field_tree ? field_tree_lds(planes, terms, S.d.L, nb).total
                                             : tree_lds(planes, S.d.L, nb, t.pitch, t.guard, P.observables,
                                                        model_info(S.d.model).values).total;
                c->tree_lds_bytes[list] = std::max(c->tree_lds_bytes[list], (size_t)bytes);
            } else if (tuned) {
                c->tuned_groups[S.d.model][li].push_back(gid);
                c->tuned_maxbins[S.d.model][li] = std::max(c->tuned_maxbins[S.d.model][li], nb);
            } else {
                const int cls = S.d.model * 2 + (S.intpath ? 1 : 0);
                c->class_groups[cls].push_back(gid);
                c->class_maxbins[cls] = std::max(c->class_maxbins[cls], nb);
                if (field_fast)
                    c->class_field_lds[cls] = std::max(c->class_field_lds[cls], field_group_lds(nb, G.nwalkers, S.N, S.d.L));
            }
            c->groups.push_back(G);
        }
    }
    for (int cls = 0; cls < 4; ++cls) {
        const int nb = c->class_maxbins[cls];
        const size_t full = (size_t)nb * kLanes * 12;
        const size_t packed = (size_t)nb * kLanes * 8 + (size_t)((nb + 1) / 2) * kLanes * 4;
        if (c->class_groups[cls].empty()) continue;
        if (c->class_field[cls]) {
            if (field_lds(c, cls) > (size_t)c->lds_max)
                return bail(fail(REWL_ERR_INVALID, "field systems of this batch do not fit LDS together"));
            continue;
        }
        if (P.observables == 2) {
            c->class_packed[cls] = false;
            if (((((size_t)nb * c->class_maxlanes[cls] * 16) + 15) & ~(size_t)15) + 16 * (size_t)c->class_maxL[cls] >
                (size_t)c->lds_max)
                return bail(fail(REWL_ERR_INVALID, "window too wide for LDS with correlators"));
            continue;
        }
        if ((cls & 1) && P.rng_mode == REWL_RNG_PHILOX && !P.observables) {
            // throughput kernel: u32 counts, stride = group size (checked above)
            if ((size_t)nb * c->class_maxlanes[cls] * 12 +
                    (c->nprod ? 8 * (size_t)c->class_maxL[cls] * c->class_maxlanes[cls] : 0) > (size_t)c->lds_max)
                return bail(fail(REWL_ERR_INVALID, "group too wide for LDS"));
            continue;
        }
        if (full <= (size_t)c->lds_max) c->class_packed[cls] = false;
        else if (packed <= (size_t)c->lds_max) c->class_packed[cls] = true;
        else return bail(fail(REWL_ERR_INVALID, "window too wide for LDS: " + std::to_string(nb) + " bins"));
    }
    place_tree_groups(c);
    c->flush_every = std::max(1, 65535 / (max_ndof(c) + 1));

    // ---- exchange pair lists ---------------------------------------------------
    for (auto& S : c->sys)
        for (int k = 0; k + 1 < S.d.num_windows; ++k)
            (k % 2 == 0 ? c->pairs_even : c->pairs_odd).push_back(S.first_window + k);

    // ---- device tables ------------------------------------------------------
    int rc;
    std::vector<double> fields;
    std::vector<DevSystem> ds;
    std::vector<size_t> field_off;
    for (auto& S : c->sys) {
        field_off.push_back(fields.size());
        fields.insert(fields.end(), S.field.begin(), S.field.end());
    }
    if ((rc = upload(c->d_fields, fields, c->stream))) return bail(rc);
    std::vector<uint8_t> excl;
    std::vector<DevWindow> dw;
    for (int si = 0; si < (int)c->sys.size(); ++si) {
        const HostSystem& S = c->sys[si];
        DevSystem D{};
        D.model = S.d.model; D.L = S.d.L; D.N = S.N; D.ndof = S.ndof;
        D.intpath = S.intpath; D.twoJ = S.twoJ; D.twoK = S.twoK; D.has_field = S.has_field;
        D.J = S.d.J; D.K = S.d.K; D.h = S.d.h;
        D.field = S.field.empty() ? nullptr : c->d_fields.p + field_off[si];
        D.k0 = (uint32_t)S.d.seed; D.k1 = (uint32_t)(S.d.seed >> 32);
        D.first_walker = S.first_walker; D.first_window = S.first_window;
        D.W = S.d.num_windows; D.R = S.d.replicas_per_window;
        ds.push_back(D);
        for (int k = 0; k < S.d.num_windows; ++k) {
            const HostWindow& w = c->win[S.first_window + k];
            DevWindow x{};
            x.emin = w.emin; x.emax = w.emax; x.bs = w.bs; x.nbins = w.nbins;
            x.sys = si; x.first_walker = w.first_walker; x.R = w.R;
            x.phi_lo = (int)(w.emin + 0.5);
            x.phi_hi = (int)(w.emax + 0.5);
            if (S.intpath) {
                x.imin = (int)w.emin;
                x.shift = (int)std::llround(std::log2(w.bs));
            }
            x.excl_off = (int64_t)excl.size();
            const size_t off = (size_t)std::llround((w.emin - S.d.e_min) / S.d.bin_size);
            for (int b = 0; b < w.nbins; ++b) excl.push_back(off + b < S.exclude.size() ? S.exclude[off + b] : 0);
            dw.push_back(x);
        }
    }
    if ((rc = upload(c->d_sys, ds, c->stream))) return bail(rc);
    if ((rc = upload(c->d_win, dw, c->stream))) return bail(rc);
    if ((rc = upload(c->d_grp, c->groups, c->stream))) return bail(rc);
    if ((rc = upload(c->d_exclude, excl, c->stream))) return bail(rc);
    if ((rc = upload(c->d_w_window, c->w_window, c->stream))) return bail(rc);
    if ((rc = upload(c->d_w_local, c->w_local, c->stream))) return bail(rc);
    if ((rc = upload(c->d_w_hist, c->w_hist, c->stream))) return bail(rc);
    if ((rc = upload(c->d_w_lat, c->w_lat, c->stream))) return bail(rc);
    for (int cls = 0; cls < 4; ++cls) longest_first(c, c->class_groups[cls]);
    for (int m = 0; m < 4; ++m)
        if ((rc = upload(c->d_tree_groups[m], c->tree_groups[m], c->stream))) return bail(rc);
    if ((rc = upload(c->d_tree_scale, tree_scales, c->stream))) return bail(rc);
    for (int cls = 0; cls < 4; ++cls)
        if ((rc = upload(c->d_class_groups[cls], c->class_groups[cls], c->stream))) return bail(rc);
    for (int m = 0; m < 2; ++m)
        for (int i = 0; i < 5; ++i) {
            if (c->tuned_groups[m][i].empty()) continue;
            const size_t need = ((size_t)c->tuned_maxbins[m][i] + 2 * c->tuned_guard[m][i]) * c->tuned_maxlanes[m][i] *
                                    kTunedSlot + (size_t)tuned_ring_stride(kTunedL[i]) * c->tuned_maxlanes[m][i] +
                                (P.observables == 2 ? 16 * (size_t)kTunedL[i] : 0) +
                                (size_t)c->tuned_maxbins[m][i] * c->tuned_maxlanes[m][i] * tuned_obs_bytes(m, P.observables);
            if (need > (size_t)c->lds_max) return bail(fail(REWL_ERR_INVALID, "group too wide for LDS"));
            if ((rc = upload(c->d_tuned_groups[m][i], c->tuned_groups[m][i], c->stream))) return bail(rc);
        }
    if ((rc = upload(c->d_pairs_even, c->pairs_even, c->stream))) return bail(rc);
    if ((rc = upload(c->d_pairs_odd, c->pairs_odd, c->stream))) return bail(rc);

    const size_t nwin = c->win.size();
    std::vector<double> lnf(nwin, P.lnf_initial);
    std::vector<int64_t> iter(nwin, 1), zeros64(nwin, 0);
    std::vector<int32_t> zeros32(nwin, 0), flav(W, 0);
    std::vector<double> E0(W, 0.0);
    std::vector<uint64_t> cur0(W, 0);
    if ((rc = upload(c->d_win_lnf, lnf, c->stream))) return bail(rc);
    if ((rc = upload(c->d_win_iter, iter, c->stream))) return bail(rc);
    if ((rc = upload(c->d_win_sweeps, zeros64, c->stream))) return bail(rc);
    if ((rc = upload(c->d_win_oot, zeros32, c->stream))) return bail(rc);
    if ((rc = upload(c->d_win_done, zeros32, c->stream))) return bail(rc);
    if ((rc = upload(c->d_win_active, std::vector<int32_t>(nwin, 1), c->stream))) return bail(rc);
    c->sys_retired.assign(c->sys.size(), 0);
    for (int cls = 0; cls < 4; ++cls) c->class_groups_all[cls] = c->class_groups[cls];
    for (int m = 0; m < 2; ++m)
        for (int i = 0; i < 5; ++i) c->tuned_groups_all[m][i] = c->tuned_groups[m][i];
    for (int m = 0; m < 4; ++m) c->tree_groups_all[m] = c->tree_groups[m];
    c->pairs_even_all = c->pairs_even;
    c->pairs_odd_all = c->pairs_odd;
    if ((rc = upload(c->d_w_flavor, flav, c->stream))) return bail(rc);
    if ((rc = upload(c->d_w_E, E0, c->stream))) return bail(rc);
    if ((rc = upload(c->d_w_cursor, cur0, c->stream))) return bail(rc);
    if ((rc = upload(c->d_err, std::vector<int32_t>(1, 0), c->stream))) return bail(rc);
    if ((rc = upload(c->d_exch, std::vector<unsigned long long>(1, 0ull), c->stream))) return bail(rc);
    c->done_host.assign(nwin, 0);
    if (hipHostMalloc((void**)&c->h_check, 2 * nwin * sizeof(int32_t), hipHostMallocDefault) != hipSuccess)
        return bail(fail(REWL_ERR_DEVICE, "hipHostMalloc failed"));

    if (c->d_lat.alloc(c->lat_total) != hipSuccess || c->d_lng.alloc(c->hist_total) != hipSuccess ||
        c->d_cnt.alloc(c->hist_total) != hipSuccess || c->d_visits.alloc(c->hist_total) != hipSuccess)
        return bail(fail(REWL_ERR_DEVICE, "hipMalloc failed for lattice/histograms"));
    if (hipMemsetAsync(c->d_lat.p, 0, c->lat_total * 8, c->stream) != hipSuccess ||
        hipMemsetAsync(c->d_lng.p, 0, c->hist_total * 8, c->stream) != hipSuccess ||
        hipMemsetAsync(c->d_cnt.p, 0, c->hist_total * 4, c->stream) != hipSuccess ||
        hipMemsetAsync(c->d_visits.p, 0, c->hist_total * 8, c->stream) != hipSuccess)
        return bail(fail(REWL_ERR_DEVICE, "hipMemset failed"));
    if (P.observables) {
        bool any_at = false, any_ising = false;
        for (const auto& S : c->sys) {
            any_at = any_at || S.d.model == REWL_ASHKIN_TELLER2D;
            any_ising = any_ising || S.d.model == REWL_ISING2D;
        }
        const bool corr = P.observables == 2;
        c->nobs = any_at ? (corr ? REWL_NUM_OBS_AT_CORR : REWL_NUM_OBS_AT)
                         : (corr ? REWL_NUM_OBS_ISING_CORR : REWL_NUM_OBS_ISING);
        const size_t n = c->hist_total * (size_t)c->nobs;
        if (c->d_obs.alloc(n) != hipSuccess) return bail(fail(REWL_ERR_DEVICE, "hipMalloc failed for observables"));
        if (hipMemsetAsync(c->d_obs.p, 0, n * 8, c->stream) != hipSuccess)
            return bail(fail(REWL_ERR_DEVICE, "hipMemset failed"));
        if (corr) {
            if (c->d_obs_tot.alloc(c->hist_total) != hipSuccess)
                return bail(fail(REWL_ERR_DEVICE, "hipMalloc failed for observables"));
            if (hipMemsetAsync(c->d_obs_tot.p, 0, c->hist_total * 4, c->stream) != hipSuccess)
                return bail(fail(REWL_ERR_DEVICE, "hipMemset failed"));
        }
        if (P.densities) {
            if (any_ising)
                return bail(fail(REWL_ERR_INVALID, "densities are an Ashkin-Teller observable (every system must be AT)"));
            const size_t nd = c->hist_total * (size_t)REWL_DENSITY_CELLS;
            if (c->d_dens.alloc(nd) != hipSuccess) return bail(fail(REWL_ERR_DEVICE, "hipMalloc failed for densities"));
            if (hipMemsetAsync(c->d_dens.p, 0, nd * 4, c->stream) != hipSuccess)
                return bail(fail(REWL_ERR_DEVICE, "hipMemset failed"));
        }
    }

    // ---- replay streams ---------------------------------------------------------
    if (P.rng_mode == REWL_RNG_REPLAY) {
        uint64_t need = (uint64_t)max_ndof(c) * 16 + 8 * kMaxReplicas + 1024;
        uint64_t C = 1;
        while (C < 2 * need) C <<= 1;
        c->ring_cap = C;
        if (c->d_ring.alloc((size_t)W * C) != hipSuccess) return bail(fail(REWL_ERR_DEVICE, "hipMalloc replay ring"));
        c->engines.resize(W);
        c->filled.assign(W, 0);
        for (auto& S : c->sys)
            for (int j = 0; j < S.d.num_windows * S.d.replicas_per_window; ++j)
                c->engines[S.first_walker + j].seed(S.walker_seeds.empty() ? (uint64_t)1 : S.walker_seeds[j]);
        if ((rc = upload(c->d_ring_filled, c->filled, c->stream))) return bail(rc);
    } else {
        c->ring_cap = 1;
        if ((rc = upload(c->d_ring_filled, std::vector<uint64_t>(1, 0), c->stream))) return bail(rc);
        if (c->d_ring.alloc(1) != hipSuccess) return bail(fail(REWL_ERR_DEVICE, "hipMalloc"));
    }

    {
        std::vector<BoundEntry> tab(kBoundTabN);
        build_bound_table(tab.data());
        if ((rc = upload(c->d_bound_tab, tab, c->stream))) return bail(rc);
    }

    KArgs& a = c->args;
    a.sys = c->d_sys.p; a.win = c->d_win.p; a.grp = c->d_grp.p;
    a.w_window = c->d_w_window.p; a.w_local = c->d_w_local.p; a.w_hist = c->d_w_hist.p; a.w_lat = c->d_w_lat.p;
    a.w_E = c->d_w_E.p; a.w_flavor = c->d_w_flavor.p; a.w_cursor = c->d_w_cursor.p;
    a.win_lnf = c->d_win_lnf.p; a.win_iter = c->d_win_iter.p; a.win_sweeps = c->d_win_sweeps.p;
    a.win_oot = c->d_win_oot.p; a.win_done = c->d_win_done.p; a.win_active = c->d_win_active.p;
    a.exclude = c->d_exclude.p;
    a.lat = c->d_lat.p; a.lng = c->d_lng.p; a.cnt = c->d_cnt.p; a.visits = c->d_visits.p;
    a.obs = c->d_obs.p; a.nobs = c->nobs; a.obs_tot = c->d_obs_tot.p; a.obs_corr = P.observables == 2 ? 1 : 0;
    a.dens = c->d_dens.p;
    a.ring = c->d_ring.p; a.ring_filled = c->d_ring_filled.p; a.ring_cap = c->ring_cap;
    a.err = c->d_err.p; a.exch_accepted = c->d_exch.p; a.bound_tab = c->d_bound_tab.p;
    a.num_walkers = W; a.num_windows = (int)nwin; a.num_groups = (int)c->groups.size();

    // initial energies of the all-up lattices (recalculate_state)
    hipLaunchKernelGGL(k_recalc, dim3((W + 63) / 64), dim3(64), 0, c->stream, c->args);
    if (hipGetLastError() != hipSuccess) return bail(fail(REWL_ERR_DEVICE, "k_recalc launch failed"));
    if (hipStreamSynchronize(c->stream) != hipSuccess) return bail(fail(REWL_ERR_DEVICE, "stream sync failed"));
    c->stats.num_walkers = W;
    *out = c;
    return REWL_OK;
}

int rewl_destroy(rewl_ctx* c) {
    if (c) {
        (void)hipStreamSynchronize(c->stream);
        destroy_ctx(c);
    }
    return REWL_OK;
}

int rewl_adjust_to_range(rewl_ctx* c) {
    if (!c) return fail(REWL_ERR_INVALID, "null context");
    int rc;
    // a failed earlier adjustment left the range bit set; it describes that
    // attempt only (the replay-exhausted bit stays: the streams are spent)
    if ((rc = clear_err_bits(c, 2))) return rc;
    if ((rc = replay_topup(c, 1))) return rc;
    uint64_t steps = (uint64_t)max_ndof(c) * 4096ull;
    const int mode = c->p.adjust_mode;
    if (c->p.rng_mode == REWL_RNG_REPLAY)
        hipLaunchKernelGGL(k_adjust<true>, dim3((c->num_walkers + 63) / 64), dim3(64), 0, c->stream, c->args, steps,
                           mode);
    else
        hipLaunchKernelGGL(k_adjust<false>, dim3((c->num_walkers + 63) / 64), dim3(64), 0, c->stream, c->args, steps,
                           mode);
    HIP_TRY(hipGetLastError());
    rc = check_err_flag(c);
    c->in_windows = rc == REWL_OK;
    return rc;
}

int rewl_sweeps(rewl_ctx* c, int32_t n) {
    if (!c || n < 0) return fail(REWL_ERR_INVALID, "bad arguments");
    // the sweep kernels index a walker's histogram by its current energy
    if (!c->in_windows)
        return fail(REWL_ERR_RANGE, "walkers are not inside their windows: call rewl_adjust_to_range first");
    int rc;
    int done = 0;
    const int chunk = c->p.rng_mode == REWL_RNG_REPLAY
                          ? (int)std::max<uint64_t>(1, (c->ring_cap - 8 * kMaxReplicas - 1024) / (uint64_t)max_ndof(c))
                          : n;
    while (done < n) {
        const int k = std::min(chunk, n - done);
        if ((rc = replay_topup(c, (uint64_t)k * (uint64_t)max_ndof(c)))) return rc;
        if ((rc = launch_sweeps(c, k))) return rc;
        c->sweep_index += (uint64_t)k;
        done += k;
    }
    c->pending_sweeps += n;
    c->stats.sweeps += (uint64_t)n;
    uint64_t att = 0;
    for (size_t si = 0; si < c->sys.size(); ++si) {
        if (c->sys_retired[si]) continue;
        const HostSystem& S = c->sys[si];
        att += (uint64_t)S.ndof * (uint64_t)S.d.num_windows * (uint64_t)S.d.replicas_per_window;
    }
    c->stats.attempts += att * (uint64_t)n;
    if (c->p.rng_mode == REWL_RNG_REPLAY) return check_err_flag(c);
    return REWL_OK;
}

int rewl_exchange(rewl_ctx* c) {
    if (!c) return fail(REWL_ERR_INVALID, "null context");
    int rc;
    // a draw per swap pair of the shuffle (at most kMaxReplicas / 2, rejections
    // are one in 2^48) and one for the decision
    if ((rc = replay_topup(c, kMaxReplicas))) return rc;
    const bool even = c->direction_even;
    const std::vector<int32_t>& pl = even ? c->pairs_even : c->pairs_odd;
    if (!pl.empty()) {
        const int32_t* dp = even ? c->d_pairs_even.p : c->d_pairs_odd.p;
        hipLaunchKernelGGL(k_exchange, dim3((unsigned)pl.size()), dim3((unsigned)(kLanes * c->exchange_waves)), 0, c->stream, c->args, dp,
                           (int)pl.size(), c->p.rng_mode == REWL_RNG_REPLAY ? 1 : 0);
        HIP_TRY(hipGetLastError());
    }
    c->direction_even = !c->direction_even;
    c->stats.exchange_calls += 1;
    if (c->p.rng_mode == REWL_RNG_REPLAY) return check_err_flag(c);
    return REWL_OK;
}

// rewl_params.retire: systems whose windows are all done leave the group
// lists of the sweep kernels, the exchange pair lists and the check.
static int retire_done_systems(rewl_ctx* c) {
    bool changed = false;
    for (size_t si = 0; si < c->sys.size(); ++si) {
        if (c->sys_retired[si]) continue;
        const HostSystem& S = c->sys[si];
        bool all = true;
        for (int k = 0; k < S.d.num_windows; ++k) all = all && c->done_host[(size_t)(S.first_window + k)] != 0;
        if (all) { c->sys_retired[si] = 1; changed = true; }
    }
    if (!changed) return REWL_OK;
    auto keep = [&](std::vector<int32_t>& groups) {
        std::vector<int32_t> out;
        for (int32_t gid : groups)
            if (!c->sys_retired[(size_t)c->groups[(size_t)gid].sys]) out.push_back(gid);
        groups.swap(out);
    };
    int rc;
    for (int cls = 0; cls < 4; ++cls) {
        keep(c->class_groups[cls]);
        if ((rc = overwrite(c->d_class_groups[cls], c->class_groups[cls], c->stream))) return rc;
    }
    for (int m = 0; m < 2; ++m)
        for (int i = 0; i < 5; ++i) {
            keep(c->tuned_groups[m][i]);
            if ((rc = overwrite(c->d_tuned_groups[m][i], c->tuned_groups[m][i], c->stream))) return rc;
        }
    for (int m = 0; m < 4; ++m) {
        keep(c->tree_groups[m]);
        if ((rc = overwrite(c->d_tree_groups[m], c->tree_groups[m], c->stream))) return rc;
    }
    auto keep_pairs = [&](std::vector<int32_t>& pl) {
        std::vector<int32_t> out;
        for (int32_t w : pl)
            if (!c->sys_retired[(size_t)c->win[(size_t)w].sys]) out.push_back(w);
        pl.swap(out);
    };
    keep_pairs(c->pairs_even);
    keep_pairs(c->pairs_odd);
    if ((rc = overwrite(c->d_pairs_even, c->pairs_even, c->stream))) return rc;
    if ((rc = overwrite(c->d_pairs_odd, c->pairs_odd, c->stream))) return rc;
    std::vector<int32_t> active(c->win.size(), 1);
    for (size_t k = 0; k < c->win.size(); ++k) active[k] = c->sys_retired[(size_t)c->win[k].sys] ? 0 : 1;
    if ((rc = overwrite(c->d_win_active, active, c->stream))) return rc;
    HIP_TRY(hipStreamSynchronize(c->stream));
    return REWL_OK;
}

// Every system back in the lists (after retirements)
static int unretire_all(rewl_ctx* c) {
    bool any = false;
    for (uint8_t r : c->sys_retired) any = any || r;
    if (!any) return REWL_OK;
    int rc;
    for (int cls = 0; cls < 4; ++cls) {
        c->class_groups[cls] = c->class_groups_all[cls];
        if ((rc = overwrite(c->d_class_groups[cls], c->class_groups[cls], c->stream))) return rc;
    }
    for (int m = 0; m < 2; ++m)
        for (int i = 0; i < 5; ++i) {
            c->tuned_groups[m][i] = c->tuned_groups_all[m][i];
            if ((rc = overwrite(c->d_tuned_groups[m][i], c->tuned_groups[m][i], c->stream))) return rc;
        }
    for (int m = 0; m < 4; ++m) {
        c->tree_groups[m] = c->tree_groups_all[m];
        if ((rc = overwrite(c->d_tree_groups[m], c->tree_groups[m], c->stream))) return rc;
    }
    c->pairs_even = c->pairs_even_all;
    c->pairs_odd = c->pairs_odd_all;
    if ((rc = overwrite(c->d_pairs_even, c->pairs_even, c->stream))) return rc;
    if ((rc = overwrite(c->d_pairs_odd, c->pairs_odd, c->stream))) return rc;
    if ((rc = overwrite(c->d_win_active, std::vector<int32_t>(c->win.size(), 1), c->stream))) return rc;
    c->sys_retired.assign(c->sys.size(), 0);
    HIP_TRY(hipStreamSynchronize(c->stream));
    return REWL_OK;
}

int rewl_check(rewl_ctx* c) {
    if (!c) return fail(REWL_ERR_INVALID, "null context");
    CheckParams cp{};
    cp.flatness_mode = c->p.flatness_mode;
    cp.schedule = c->p.schedule;
    cp.reduce_logdos = c->p.reduce_logdos;
    cp.average_mode = c->p.average_mode;
    cp.flatness = c->p.flatness;
    cp.lnf_final = c->p.lnf_final;
    cp.pending_sweeps = c->pending_sweeps;
    const int nwin = (int)c->win.size();
    // the kernel writes each window's flat and done flags to pinned memory
    int32_t* const flat = c->h_check;
    int32_t* const done = c->h_check + nwin;
    hipLaunchKernelGGL(k_check, dim3((unsigned)nwin), dim3(kLanes), 0, c->stream, c->args, cp, flat, done);
    HIP_TRY(hipGetLastError());
    c->pending_sweeps = 0;
    HIP_TRY(hipStreamSynchronize(c->stream));
    std::copy(done, done + nwin, c->done_host.begin());
    int all = 1;
    for (int k = 0; k < nwin; ++k) {
        all &= c->done_host[k] ? 1 : 0;
        c->stats.flat_events += flat[k] ? 1 : 0;
    }
    c->stats.all_done = all;
    c->stats.checks += 1;
    if (c->p.retire) return retire_done_systems(c);
    return REWL_OK;
}

int rewl_run(rewl_ctx* c, int64_t max_checks) {
    if (!c) return fail(REWL_ERR_INVALID, "null context");
    const int per_check = c->p.sweeps_per_check / c->p.sweeps_per_exchange;
    int rc;
    for (int64_t k = 0; k < max_checks; ++k) {
        for (int u = 0; u < per_check; ++u) {
            if ((rc = rewl_sweeps(c, c->p.sweeps_per_exchange))) return rc;
            if (c->p.exchange && (rc = rewl_exchange(c))) return rc;
        }
        if ((rc = rewl_check(c))) return rc;
        if (c->stats.all_done) return REWL_OK;
    }
    return fail(REWL_ERR_ITER_CAP, "not converged after max_checks check cycles");
}

int rewl_finalize(rewl_ctx* c) {
    if (!c) return fail(REWL_ERR_INVALID, "null context");
    hipLaunchKernelGGL(k_finalize, dim3((unsigned)c->win.size()), dim3(kLanes), 0, c->stream, c->args,
                       (int)c->p.average_mode);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipStreamSynchronize(c->stream));
    return REWL_OK;
}

int rewl_refine_begin(rewl_ctx* c) {
    if (!c) return fail(REWL_ERR_INVALID, "null context");
    if (!c->in_windows)
        return fail(REWL_ERR_RANGE, "walkers are not inside their windows: call rewl_adjust_to_range first");
    int rc;
    // every system takes part (retired ones too); the replicas' common
    // curve, then fixed weights: ln f = 0 in every window
    if ((rc = unretire_all(c))) return rc;
    if ((rc = rewl_finalize(c))) return rc;
    if ((rc = overwrite(c->d_win_lnf, std::vector<double>(c->win.size(), 0.0), c->stream))) return rc;
    const int64_t n = (int64_t)c->hist_total;
    const unsigned grid = (unsigned)std::min<int64_t>(4096, (n + 255) / 256);
    hipLaunchKernelGGL(k_hist_clear, dim3(grid), dim3(256), 0, c->stream, c->args, n);
    HIP_TRY(hipGetLastError());
    c->refining = true;
    c->refine_since_exchange = 0;
    return REWL_OK;
}

int rewl_refine_sweeps(rewl_ctx* c, int64_t sweeps, int32_t sweeps_per_exchange) {
    if (!c || sweeps < 0 || sweeps_per_exchange < 1) return fail(REWL_ERR_INVALID, "bad arguments");
    if (!c->refining) return fail(REWL_ERR_INVALID, "rewl_refine_sweeps outside rewl_refine_begin / rewl_refine_end");
    const int64_t n = (int64_t)c->hist_total;
    const unsigned grid = (unsigned)std::min<int64_t>(4096, (n + 255) / 256);
    int rc;
    // launches of at most 1000 sweeps keep a bin's u32 count far below 2^32;
    // an exchange after every sweeps_per_exchange sweeps, counted across calls
    int64_t done = 0;
    while (done < sweeps) {
        const int k = (int)std::min<int64_t>(
            {1000, (int64_t)sweeps_per_exchange - c->refine_since_exchange, sweeps - done});
        if ((rc = rewl_sweeps(c, k))) return rc;
        done += k;
        c->refine_since_exchange += k;
        if (c->refine_since_exchange >= sweeps_per_exchange) {
            if (c->p.exchange && (rc = rewl_exchange(c))) return rc;
            c->refine_since_exchange = 0;
        }
        hipLaunchKernelGGL(k_hist_roll, dim3(grid), dim3(256), 0, c->stream, c->args, n);
        HIP_TRY(hipGetLastError());
    }
    HIP_TRY(hipStreamSynchronize(c->stream));
    return REWL_OK;
}

int rewl_refine_end(rewl_ctx* c) {
    if (!c) return fail(REWL_ERR_INVALID, "null context");
    if (!c->refining) return fail(REWL_ERR_INVALID, "rewl_refine_end without rewl_refine_begin");
    hipLaunchKernelGGL(k_refine, dim3((unsigned)c->win.size()), dim3(kLanes), 0, c->stream, c->args);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipStreamSynchronize(c->stream));
    c->refining = false;
    return REWL_OK;
}

int rewl_refine(rewl_ctx* c, int64_t sweeps, int32_t sweeps_per_exchange) {
    if (!c || sweeps < 1 || sweeps_per_exchange < 1) return fail(REWL_ERR_INVALID, "bad arguments");
    int rc;
    if ((rc = rewl_refine_begin(c))) return rc;
    if ((rc = rewl_refine_sweeps(c, sweeps, sweeps_per_exchange))) return rc;
    return rewl_refine_end(c);
}

int rewl_synchronize(rewl_ctx* c) {
    if (!c) return fail(REWL_ERR_INVALID, "null context");
    HIP_TRY(hipStreamSynchronize(c->stream));
    return REWL_OK;
}

int rewl_num_walkers(const rewl_ctx* c, int32_t* n) {
    if (!c || !n) return fail(REWL_ERR_INVALID, "null argument");
    *n = c->num_walkers;
    return REWL_OK;
}

int rewl_num_windows(const rewl_ctx* c, int32_t* n) {
    if (!c || !n) return fail(REWL_ERR_INVALID, "null argument");
    *n = (int32_t)c->win.size();
    return REWL_OK;
}

int rewl_get_window_info(rewl_ctx* c, int32_t wi, rewl_window_info* o) {
    if (!c || !o || wi < 0 || wi >= (int32_t)c->win.size()) return fail(REWL_ERR_INVALID, "bad window index");
    const HostWindow& w = c->win[wi];
    o->system = w.sys;
    o->window = wi - c->sys[w.sys].first_window;
    o->first_walker = w.first_walker;
    o->num_bins = w.nbins;
    o->e_min = w.emin; o->e_max = w.emax; o->bin_size = w.bs;
    std::lock_guard<std::mutex> lock(c->fetch_mu);
    int rc;
    if ((rc = reserve_fetch(c, sizeof(WindowState)))) return rc;
    hipLaunchKernelGGL(k_window_state, dim3(1), dim3(1), 0, c->stream, c->args, (int)wi,
                       static_cast<WindowState*>(c->h_fetch));
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipStreamSynchronize(c->stream));
    WindowState s;
    std::memcpy(&s, c->h_fetch, sizeof(s));
    o->lnf = s.lnf;
    o->iteration = s.iteration;
    o->sweeps_in_iteration = s.sweeps + c->pending_sweeps;
    o->done = s.done;
    o->one_over_t = s.one_over_t;
    return REWL_OK;
}

int rewl_get_stats(rewl_ctx* c, rewl_stats* o) {
    if (!c || !o) return fail(REWL_ERR_INVALID, "null argument");
    int rc;
    if ((rc = resolve_sweep_events(c))) return rc;
    unsigned long long acc = 0;
    if ((rc = fetch(c, c->d_exch.p, 1, 1, 1, &acc))) return rc;
    c->stats.exchanges_accepted = acc;
    *o = c->stats;
    return REWL_OK;
}

static int walker_ok(const rewl_ctx* c, int32_t g) { return c && g >= 0 && g < c->num_walkers; }

int rewl_get_logdos(rewl_ctx* c, int32_t g, double* out, int32_t n) {
    if (!walker_ok(c, g) || !out) return fail(REWL_ERR_INVALID, "bad walker");
    const int nb = c->win[c->w_window[g]].nbins;
    if (n < nb) return fail(REWL_ERR_INVALID, "output buffer too small");
    return fetch(c, c->d_lng.p + c->w_hist[g], kLanes, nb, 1, out);
}

int rewl_get_counts(rewl_ctx* c, int32_t g, uint32_t* out, int32_t n) {
    if (!walker_ok(c, g) || !out) return fail(REWL_ERR_INVALID, "bad walker");
    const int nb = c->win[c->w_window[g]].nbins;
    if (n < nb) return fail(REWL_ERR_INVALID, "output buffer too small");
    return fetch(c, c->d_cnt.p + c->w_hist[g], kLanes, nb, 1, out);
}

int rewl_get_visits(rewl_ctx* c, int32_t g, uint64_t* out, int32_t n) {
    if (!walker_ok(c, g) || !out) return fail(REWL_ERR_INVALID, "bad walker");
    const int nb = c->win[c->w_window[g]].nbins;
    if (n < nb) return fail(REWL_ERR_INVALID, "output buffer too small");
    return fetch(c, c->d_visits.p + c->w_hist[g], kLanes, nb, 1, out);
}

int rewl_get_observables(rewl_ctx* c, int32_t g, double* sums, int32_t n, int32_t nobs) {
    if (!walker_ok(c, g) || !sums) return fail(REWL_ERR_INVALID, "bad walker");
    if (!c->d_obs.p) return fail(REWL_ERR_INVALID, "observables are off (rewl_params.observables)");
    const HostSystem& S = c->sys[c->win[c->w_window[g]].sys];
    const bool corr = c->p.observables == 2;
    // groups of three moments, each followed by a correlator slot with corr
    const int want = model_info(S.d.model).values / 3 * (corr ? 4 : 3);
    if (nobs != want) return fail(REWL_ERR_INVALID, "nobs does not match the walker's model");
    const int nb = c->win[c->w_window[g]].nbins;
    if (n < nb) return fail(REWL_ERR_INVALID, "output buffer too small");
    return fetch(c, c->d_obs.p + c->w_hist[g] * c->nobs, (int64_t)kLanes * c->nobs, nb, nobs, sums);
}

int rewl_get_densities(rewl_ctx* c, int32_t g, uint32_t* out, int32_t n) {
    if (!walker_ok(c, g) || !out) return fail(REWL_ERR_INVALID, "bad walker");
    if (!c->d_dens.p) return fail(REWL_ERR_INVALID, "densities are off (rewl_params.densities)");
    const int nb = c->win[c->w_window[g]].nbins;
    if (n < nb) return fail(REWL_ERR_INVALID, "output buffer too small");
    const size_t row = (size_t)REWL_DENSITY_CELLS * sizeof(uint32_t);
    HIP_TRY(hipMemcpy2DAsync(out, row, c->d_dens.p + c->w_hist[g] * REWL_DENSITY_CELLS, row * kLanes, row, (size_t)nb,
                             hipMemcpyDeviceToHost, c->stream));
    HIP_TRY(hipStreamSynchronize(c->stream));
    return REWL_OK;
}

int rewl_get_spins(rewl_ctx* c, int32_t g, int8_t* out, int32_t n) {
    if (!walker_ok(c, g) || !out) return fail(REWL_ERR_INVALID, "bad walker");
    const HostSystem& S = c->sys[c->win[c->w_window[g]].sys];
    if (n < S.ndof) return fail(REWL_ERR_INVALID, "output buffer too small");
    const int planes = model_info(S.d.model).planes, L = S.d.L;
    std::vector<uint64_t> words((size_t)planes * L);
    int rc;
    if ((rc = fetch(c, c->d_lat.p + c->w_lat[g], kLanes, (int)words.size(), 1, words.data()))) return rc;
    for (int i = 0; i < S.N; ++i) {
        const int x = i % L, y = i / L;
        for (int q = 0; q < planes; ++q) {
            const int8_t v = ((words[(size_t)q * L + y] >> x) & 1ull) ? -1 : 1;
            out[planes == 1 ? i : 2 * i + q] = v;
        }
    }
    return REWL_OK;
}

int rewl_get_energy(rewl_ctx* c, int32_t g, double* e) {
    if (!walker_ok(c, g) || !e) return fail(REWL_ERR_INVALID, "bad walker");
    return fetch(c, c->d_w_E.p + g, 1, 1, 1, e);
}

int rewl_get_flavor(rewl_ctx* c, int32_t g, int32_t* f) {
    if (!walker_ok(c, g) || !f) return fail(REWL_ERR_INVALID, "bad walker");
    return fetch(c, c->d_w_flavor.p + g, 1, 1, 1, f);
}

int rewl_get_rng_cursor(rewl_ctx* c, int32_t g, uint64_t* cur) {
    if (!walker_ok(c, g) || !cur) return fail(REWL_ERR_INVALID, "bad walker");
    return fetch(c, c->d_w_cursor.p + g, 1, 1, 1, cur);
}

// One walker's ln g column ([bin][lane] layout) from a linear staging copy.
__global__ void k_scatter_column(double* dst, const double* src, int n) {
    const int b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b < n) dst[(int64_t)b * kLanes] = src[b];
}

int rewl_set_logdos(rewl_ctx* c, int32_t g, const double* lng, int32_t n) {
    if (!walker_ok(c, g) || !lng) return fail(REWL_ERR_INVALID, "bad walker");
    const int nb = c->win[c->w_window[g]].nbins;
    if (n != nb) return fail(REWL_ERR_INVALID, "ln g length must equal the window's bin count");
    // a strided copy of single doubles takes milliseconds per walker; a
    // linear copy into a staging buffer and one scatter launch, microseconds
    if (c->d_stage.n < (size_t)nb) {
        c->d_stage.release();
        const hipError_t e = c->d_stage.alloc((size_t)nb);
        if (e != hipSuccess) {
            c->d_stage.release();
            return fail(REWL_ERR_DEVICE, std::string("staging buffer: ") + hipGetErrorString(e));
        }
    }
    HIP_TRY(hipMemcpyAsync(c->d_stage.p, lng, (size_t)nb * sizeof(double), hipMemcpyHostToDevice, c->stream));
    hipLaunchKernelGGL(k_scatter_column, dim3((nb + 255) / 256), dim3(256), 0, c->stream, c->d_lng.p + c->w_hist[g],
                       (const double*)c->d_stage.p, nb);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipStreamSynchronize(c->stream));
    return REWL_OK;
}

int rewl_set_window_lnf(rewl_ctx* c, int32_t wi, double lnf) {
    if (!c || wi < 0 || wi >= (int32_t)c->win.size() || !(lnf > 0)) return fail(REWL_ERR_INVALID, "bad window or ln f");
    HIP_TRY(hipMemcpyAsync(c->d_win_lnf.p + wi, &lnf, sizeof(double), hipMemcpyHostToDevice, c->stream));
    HIP_TRY(hipStreamSynchronize(c->stream));
    return REWL_OK;
}

// Bit-packed rows (plane-major, bit x of row y = site y*L+x, 1 = spin -1) of a
// configuration given in the reference's DoF layout.
static std::vector<uint64_t> pack_rows(const HostSystem& S, const int8_t* spins) {
    const int planes = model_info(S.d.model).planes, L = S.d.L;
    std::vector<uint64_t> words((size_t)planes * L, 0ull);
    for (int i = 0; i < S.N; ++i) {
        const int x = i % L, y = i / L;
        for (int q = 0; q < planes; ++q) {
            const int8_t v = spins[planes == 1 ? i : 2 * i + q];
            if (v < 0) words[(size_t)q * L + y] |= (1ull << x);
        }
    }
    return words;
}

static int upload_rows(rewl_ctx* c, int32_t g, const std::vector<uint64_t>& words) {
    HIP_TRY(hipMemcpy2DAsync(c->d_lat.p + c->w_lat[g], kLanes * sizeof(uint64_t), words.data(), sizeof(uint64_t),
                             sizeof(uint64_t), words.size(), hipMemcpyHostToDevice, c->stream));
    return REWL_OK;
}

// Energies of every walker from its lattice, then the walkers count as
// outside their windows until the next rewl_adjust_to_range.
static int recalc_all(rewl_ctx* c) {
    hipLaunchKernelGGL(k_recalc, dim3((c->num_walkers + 63) / 64), dim3(64), 0, c->stream, c->args);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipStreamSynchronize(c->stream));
    c->in_windows = false;   // the new state may lie outside the window
    return REWL_OK;
}

int rewl_set_spins(rewl_ctx* c, int32_t g, const int8_t* spins, int32_t n) {
    if (!walker_ok(c, g) || !spins) return fail(REWL_ERR_INVALID, "bad walker");
    const HostSystem& S = c->sys[c->win[c->w_window[g]].sys];
    if (n != S.ndof) return fail(REWL_ERR_INVALID, "spin array length must equal the number of degrees of freedom");
    int rc;
    if ((rc = upload_rows(c, g, pack_rows(S, spins)))) return rc;
    return recalc_all(c);
}

int rewl_set_system_spins(rewl_ctx* c, int32_t si, const int8_t* spins, int32_t n) {
    if (!c || si < 0 || si >= (int32_t)c->sys.size() || !spins) return fail(REWL_ERR_INVALID, "bad system");
    const HostSystem& S = c->sys[si];
    if (n != S.ndof) return fail(REWL_ERR_INVALID, "spin array length must equal the number of degrees of freedom");
    const std::vector<uint64_t> words = pack_rows(S, spins);
    int rc;
    for (int32_t g = 0; g < c->num_walkers; ++g)
        if (c->win[c->w_window[g]].sys == si && (rc = upload_rows(c, g, words))) return rc;
    return recalc_all(c);
}

// ---- results path -------------------------------------------------------------
// Derivative of a tabulated function as numerical_derivatives.hpp:46-70 takes
// it: one-sided at the ends, second-order next to them, fourth-order inside.
static double tab_deriv(size_t i, const std::vector<double>& f, const std::vector<double>& e) {
    const size_t n = f.size();
    if (i == 0) return (f[1] - f[0]) / (e[1] - e[0]);
    if (i == n - 1) return (f[i] - f[i - 1]) / (e[i] - e[i - 1]);
    if (i == 1 || i == n - 2) return (f[i + 1] - f[i - 1]) / (2. * (e[i] - e[i - 1]));
    return (-f[i + 2] + 8. * f[i + 1] - 8. * f[i - 1] + f[i - 2]) / (12. * (e[i] - e[i - 1]));
}

// |x| as the reference evaluates it: its unqualified abs() on a double binds
// to int abs(int), truncating toward zero (vector_matching.hpp:107, 116).
static double int_abs(double v) { return (double)std::abs((int)v); }

int rewl_stitch(rewl_ctx* c, int32_t si, double states_per_site, double* energies, double* logdos, int32_t capacity,
                int32_t* n_out) {
    if (!c || si < 0 || si >= (int32_t)c->sys.size() || !n_out) return fail(REWL_ERR_INVALID, "bad system");
    const HostSystem& S = c->sys[si];
    const int nw = S.d.num_windows;
    std::vector<std::vector<double>> et(nw), lt(nw);
    for (int k = 0; k < nw; ++k) {
        const HostWindow& w = c->win[S.first_window + k];
        lt[k].resize(w.nbins);
        int rc = rewl_get_logdos(c, w.first_walker, lt[k].data(), w.nbins);
        if (rc) return rc;
        // bin energies on the system's global grid: the same value for the same
        // bin in every window (emin + bs b equals it whenever bs is dyadic, as in
        // the reference's integer bins; with other bin sizes the per-window sums
        // round differently and the reference's exact match would fail)
        const long long g0 = std::llround((w.emin - S.d.e_min) / S.d.bin_size);
        for (int b = 0; b < w.nbins; ++b) et[k].push_back(S.d.e_min + S.d.bin_size * (double)(g0 + b));
    }
    // concatenate_tables_multiple_overlap (concatenate_rewl_tables.hpp:167-305)
    std::vector<double> fe = et[0], fl = lt[0];
    double shifter = 0.;
    for (int k = 1; k < nw; ++k) {
        long start = -1;
        for (long i = (long)fe.size() - 1; i >= 0; --i)
            if (fe[i] == et[k].front()) { start = i; break; }
        if (start < 0) return fail(REWL_ERR_INVALID, "adjacent windows do not overlap");
        const size_t nl = fl.size();
        double bd = int_abs(tab_deriv((size_t)start, fl, fe) - tab_deriv(0, lt[k], et[k]));
        size_t join = (size_t)start;
        for (size_t j = 1; j != nl - (size_t)start; ++j) {
            const double t = int_abs(tab_deriv((size_t)start + j, fl, fe) - tab_deriv(j, lt[k], et[k]));
            if (t + 0.5 < bd + 0.5) { bd = t; join = (size_t)start + j; }
        }
        size_t r = 0;
        for (size_t i = (size_t)start; i < fe.size(); ++i) {
            r = i - (size_t)start;
            if (i == join) shifter = fl[i] - lt[k][r];
            else if (i > join) fl[i] = lt[k][r] + shifter;
        }
        for (size_t j = r + 1; j < et[k].size(); ++j) { fe.push_back(et[k][j]); fl.push_back(lt[k][j] + shifter); }
    }
    // normalize_logDoS (array_shift.hpp:15-43)
    if (states_per_site > 0) {
        double mx = 0.;
        for (double v : fl) mx = mx * (double)(mx > v) + v * (double)(mx <= v);
        double sum = 0.;
        for (double v : fl) sum += exp(-(mx - v));
        sum = log(sum) + mx;
        const double sh = (double)S.N * log(states_per_site) - sum - log(2.) * (double)(S.d.e_max == 0.);
        for (double& v : fl) v += sh;
    }
    *n_out = (int32_t)fl.size();
    for (size_t i = 0; i < fl.size() && (int32_t)i < capacity; ++i) {
        if (energies) energies[i] = fe[i];
        if (logdos) logdos[i] = fl[i];
    }
    return REWL_OK;
}

// Every energy below 1e100 and every temperature between 1e-100 and 1e100 in
// size: E/T can be taken as a corrected product (ThermoT).
static bool thermo_tame(const double* E, int32_t nb, double tmin, double tmax) {
    const double lo = std::min(tmin, tmax), hi = std::max(tmin, tmax);
    if (!(lo > 1e-100 && hi < 1e100) && !(hi < -1e-100 && lo > -1e100)) return false;
    for (int32_t b = 0; b < nb; ++b)
        if (!(std::fabs(E[b]) < 1e100)) return false;
    return true;
}

static void launch_thermo(bool tame, const double* dE, const double* dl, int nb, int N, double tmin, double dT, int nT,
                          double* dout) {
    hipLaunchKernelGGL(tame ? k_thermo<true> : k_thermo<false>, dim3((unsigned)((nT + kThermoT - 1) / kThermoT)),
                       dim3(kThermoT * kThermoWaves), 0, nullptr, dE, dl, nb, N, tmin, dT, nT, dout);
}

int rewl_thermodynamics(const double* E, const double* lng, int32_t nb, int32_t N, double tmin, double tmax, int32_t nT,
                        double* out) {
    if (!E || !lng || !out || nb < 2 || nT < 1 || N < 1) return fail(REWL_ERR_INVALID, "bad arguments");
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0) return fail(REWL_ERR_NO_DEVICE, "no HIP device");
    double *dE = nullptr, *dl = nullptr, *dout = nullptr;
    HIP_TRY(hipMalloc((void**)&dE, (size_t)nb * sizeof(double)));
    HIP_TRY(hipMalloc((void**)&dl, (size_t)nb * sizeof(double)));
    HIP_TRY(hipMalloc((void**)&dout, (size_t)nT * 5 * sizeof(double)));
    HIP_TRY(hipMemcpy(dE, E, (size_t)nb * sizeof(double), hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(dl, lng, (size_t)nb * sizeof(double), hipMemcpyHostToDevice));
    const double dT = (tmax - tmin) / (double)nT;
    launch_thermo(thermo_tame(E, nb, tmin, tmax), dE, dl, nb, N, tmin, dT, nT, dout);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipMemcpy(out, dout, (size_t)nT * 5 * sizeof(double), hipMemcpyDeviceToHost));
    (void)hipFree(dE);
    (void)hipFree(dl);
    (void)hipFree(dout);
    return REWL_OK;
}

// ---- rewl_thermodynamics without allocation ------------------------------------
// The staging buffers of rewl_thermodynamics (the two input curves and the
// output table) live in one static device array instead of hipMalloc'd
// memory.  Each GPU holds its own copy of `scratch` at its own address, which
// hipGetSymbolAddress returns once per device with that device current; host
// code uses only that pointer.  Every call on a GPU shares its copy: the
// inputs are copied in and the output is written in full by every call, so
// nothing needs clearing, and calls that overlap on one GPU race.
constexpr int kStaticThermoMaxBins = 16384;
constexpr int kStaticThermoMaxTemps = 65536;
constexpr size_t kStaticThermoDoubles = 2 * (size_t)kStaticThermoMaxBins + 5 * (size_t)kStaticThermoMaxTemps;
static __device__ __align__(256) double scratch[kStaticThermoDoubles];   // 2.75 MiB per GPU

namespace {
constexpr int kMaxScratchDevices = 64;
std::mutex g_scratch_mu;
double* g_scratch_ptr[kMaxScratchDevices] = {};

// scratch's address on the current device (looked up on the first call there)
int scratch_on_current_device(double** out) {
    int dev = 0;
    HIP_TRY(hipGetDevice(&dev));
    if (dev < 0 || dev >= kMaxScratchDevices) return fail(REWL_ERR_DEVICE, "device index beyond the scratch table");
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void* p = nullptr;
        HIP_TRY(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        if (!p) return fail(REWL_ERR_DEVICE, "hipGetSymbolAddress returned no address for the scratch array");
        g_scratch_ptr[dev] = static_cast<double*>(p);
    }
    *out = g_scratch_ptr[dev];
    return REWL_OK;
}
}  // namespace

int rewl_thermodynamics_noalloc(const double* E, const double* lng, int32_t nb, int32_t N, double tmin, double tmax,
                                int32_t nT, double* out) {
    if (!E || !lng || !out || nb < 2 || nT < 1 || N < 1) return fail(REWL_ERR_INVALID, "bad arguments");
    if (nb > kStaticThermoMaxBins || nT > kStaticThermoMaxTemps)
        return fail(REWL_ERR_INVALID, "rewl_thermodynamics_noalloc: at most 16384 bins and 65536 temperatures "
                                      "(the size of its static device scratch)");
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0) return fail(REWL_ERR_NO_DEVICE, "no HIP device");
    double* base = nullptr;
    int rc;
    if ((rc = scratch_on_current_device(&base))) return rc;
    double* dE = base;
    double* dl = base + kStaticThermoMaxBins;
    double* dout = base + 2 * (size_t)kStaticThermoMaxBins;
    HIP_TRY(hipMemcpy(dE, E, (size_t)nb * sizeof(double), hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(dl, lng, (size_t)nb * sizeof(double), hipMemcpyHostToDevice));
    const double dT = (tmax - tmin) / (double)nT;
    launch_thermo(thermo_tame(E, nb, tmin, tmax), dE, dl, nb, N, tmin, dT, nT, dout);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipMemcpy(out, dout, (size_t)nT * 5 * sizeof(double), hipMemcpyDeviceToHost));
    return REWL_OK;
}

int rewl_thermo_observables(const double* E, const double* lng, const double* obs, int32_t nb, int32_t nobs,
                            double tmin, double tmax, int32_t nT, double* out) {
    if (!E || !lng || !obs || !out || nb < 2 || nT < 1 || nobs < 1 || nobs > kThermoMaxObs)
        return fail(REWL_ERR_INVALID, "bad arguments");
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0) return fail(REWL_ERR_NO_DEVICE, "no HIP device");
    double *dE = nullptr, *dl = nullptr, *dobs = nullptr, *dout = nullptr;
    auto release = [&]() { (void)hipFree(dE); (void)hipFree(dl); (void)hipFree(dobs); (void)hipFree(dout); };
    if (hipMalloc((void**)&dE, (size_t)nb * sizeof(double)) != hipSuccess ||
        hipMalloc((void**)&dl, (size_t)nb * sizeof(double)) != hipSuccess ||
        hipMalloc((void**)&dobs, (size_t)nb * nobs * sizeof(double)) != hipSuccess ||
        hipMalloc((void**)&dout, (size_t)nT * nobs * sizeof(double)) != hipSuccess) {
        release();
        return fail(REWL_ERR_DEVICE, "hipMalloc failed");
    }
    hipError_t e = hipMemcpy(dE, E, (size_t)nb * sizeof(double), hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(dl, lng, (size_t)nb * sizeof(double), hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(dobs, obs, (size_t)nb * nobs * sizeof(double), hipMemcpyHostToDevice);
    if (e == hipSuccess) {
        const double dT = (tmax - tmin) / (double)nT;
        hipLaunchKernelGGL(thermo_tame(E, nb, tmin, tmax) ? k_thermo_obs<true> : k_thermo_obs<false>,
                           dim3((unsigned)((nT + kThermoT - 1) / kThermoT)), dim3(kThermoT * kThermoWaves), 0, nullptr,
                           (const double*)dE, (const double*)dl, (const double*)dobs, (int)nb, (int)nobs, tmin, dT, (int)nT,
                           dout);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipMemcpy(out, dout, (size_t)nT * nobs * sizeof(double), hipMemcpyDeviceToHost);
    release();
    if (e != hipSuccess) return fail(REWL_ERR_DEVICE, std::string("rewl_thermo_observables: ") + hipGetErrorString(e));
    return REWL_OK;
}

int rewl_stitch_overlap(rewl_ctx* c, int32_t si, double states_per_site, double* energies, double* logdos,
                        int32_t capacity, int32_t* n_out) {
    if (!c || si < 0 || si >= (int32_t)c->sys.size() || !n_out) return fail(REWL_ERR_INVALID, "bad system");
    const HostSystem& S = c->sys[si];
    const int nw = S.d.num_windows;
    // the system's global bin grid; unvisited bins stay NaN
    int nb_total = 0;
    std::vector<long long> g0(nw);
    for (int k = 0; k < nw; ++k) {
        const HostWindow& w = c->win[S.first_window + k];
        g0[k] = std::llround((w.emin - S.d.e_min) / S.d.bin_size);
        nb_total = std::max<int>(nb_total, (int)(g0[k] + w.nbins));
    }
    std::vector<double> lng((size_t)nb_total, std::nan(""));
    std::vector<char> vis((size_t)nb_total, 0);
    for (int k = 0; k < nw; ++k) {
        const HostWindow& w = c->win[S.first_window + k];
        std::vector<double> lk(w.nbins);
        std::vector<uint32_t> ck(w.nbins);
        std::vector<uint64_t> vk(w.nbins), vsum(w.nbins, 0);
        int rc = rewl_get_logdos(c, w.first_walker, lk.data(), w.nbins);
        if (rc) return rc;
        for (int r = 0; r < w.R; ++r) {
            if ((rc = rewl_get_counts(c, w.first_walker + r, ck.data(), w.nbins))) return rc;
            if ((rc = rewl_get_visits(c, w.first_walker + r, vk.data(), w.nbins))) return rc;
            for (int b = 0; b < w.nbins; ++b) vsum[b] += vk[b] + ck[b];
        }
        if (k == 0) {
            for (int b = 0; b < w.nbins; ++b)
                if (vsum[b]) { lng[(size_t)(g0[k] + b)] = lk[b]; vis[(size_t)(g0[k] + b)] = 1; }
            continue;
        }
        // shift onto the curve so far: mean difference over the bins both visited
        double sum = 0.;
        std::vector<long long> common;
        for (int b = 0; b < w.nbins; ++b) {
            const size_t i = (size_t)(g0[k] + b);
            if (vsum[b] && vis[i]) { sum += lng[i] - lk[b]; common.push_back((long long)i); }
        }
        if (common.empty()) return fail(REWL_ERR_INVALID, "adjacent windows share no visited bin");
        const double shift = sum / (double)common.size();
        const long long from = common[common.size() / 2];   // take over from the middle of the common stretch
        for (int b = 0; b < w.nbins; ++b) {
            const long long i = g0[k] + b;
            if (vsum[b] && i >= from) { lng[(size_t)i] = lk[b] + shift; vis[(size_t)i] = 1; }
        }
    }
    // normalise over the visited bins as normalize_logDoS does (array_shift.hpp:15-43)
    if (states_per_site > 0) {
        double mx = -INFINITY;
        for (size_t i = 0; i < lng.size(); ++i) if (vis[i]) mx = std::max(mx, lng[i]);
        double sum = 0.;
        for (size_t i = 0; i < lng.size(); ++i) if (vis[i]) sum += exp(lng[i] - mx);
        const double sh = (double)S.N * log(states_per_site) - (log(sum) + mx) - log(2.) * (double)(S.d.e_max == 0.);
        for (size_t i = 0; i < lng.size(); ++i) if (vis[i]) lng[i] += sh;
    }
    *n_out = nb_total;
    for (int i = 0; i < nb_total && i < capacity; ++i) {
        if (energies) energies[i] = S.d.e_min + S.d.bin_size * (double)i;
        if (logdos) logdos[i] = lng[(size_t)i];
    }
    return REWL_OK;
}

int rewl_anneal(const rewl_system_desc* systems, int32_t num_systems, const rewl_anneal_params* params,
                double* min_energy, double* final_energy, uint64_t* sweeps, int8_t* final_spins) {
    if (!systems || num_systems < 1 || !params || !min_energy || !final_energy || !sweeps)
        return fail(REWL_ERR_INVALID, "bad argument");
    const rewl_anneal_params& P = *params;
    if (!(P.initial_temperature > 0) || !(P.final_temperature > 0) || P.num_temperatures < 1 || P.block_size < 1 ||
        P.max_blocks < 1 || P.chains < 1 || !(P.stdev_tolerance >= 0))
        return fail(REWL_ERR_INVALID, "invalid rewl_anneal_params");
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0)
        return fail(REWL_ERR_NO_DEVICE, "no HIP device visible: the annealer runs only on the GPU");
    const int gps = (P.chains + kLanes - 1) / kLanes;
    const size_t ngroups = (size_t)num_systems * (size_t)gps;
    const size_t ebuf_n = ngroups * (size_t)P.block_size * kLanes;
    if (ebuf_n * sizeof(double) > ((size_t)16 << 30))
        return fail(REWL_ERR_INVALID, "block energies of all chains exceed 16 GiB: fewer chains or a smaller block");
    std::vector<DevSystem> ds((size_t)num_systems);
    std::vector<double> fields;
    std::vector<size_t> foff((size_t)num_systems, (size_t)-1);
    for (int si = 0; si < num_systems; ++si) {
        const rewl_system_desc& d = systems[si];
        if (d.model != REWL_ISING2D && d.model != REWL_ASHKIN_TELLER2D) return fail(REWL_ERR_INVALID, "unknown model");
        if (d.L < 2 || d.L > 64) return fail(REWL_ERR_INVALID, "L must lie in [2, 64]");
        DevSystem& D = ds[(size_t)si];
        D.model = d.model; D.L = d.L; D.N = d.L * d.L; D.ndof = model_info(d.model).planes * D.N;
        D.has_field = d.field != nullptr || d.h != 0.0;
        D.J = d.J; D.K = d.K; D.h = d.h;
        D.k0 = (uint32_t)d.seed; D.k1 = (uint32_t)(d.seed >> 32);
        if (d.field) {
            foff[(size_t)si] = fields.size();
            fields.insert(fields.end(), d.field, d.field + D.N);
        }
    }
    // the temperature schedule on the host, as calculate_temperature computes it
    std::vector<double> beta((size_t)P.num_temperatures + 1);
    for (int k = 0; k <= P.num_temperatures; ++k) {
        const double T = P.initial_temperature * pow(P.final_temperature / P.initial_temperature,
                                                      (double)k / (double)P.num_temperatures);
        beta[(size_t)k] = 1. / T;
    }
    AnnealBuffers B;
    const hipStream_t st = nullptr;
    int rc;
    if ((rc = upload(B.fields, fields, st))) return rc;
    for (int si = 0; si < num_systems; ++si)
        if (foff[(size_t)si] != (size_t)-1) ds[(size_t)si].field = B.fields.p + foff[(size_t)si];
    if ((rc = upload(B.sys, ds, st))) return rc;
    if ((rc = upload(B.beta, beta, st))) return rc;
    const size_t nout = (size_t)num_systems * (size_t)P.chains;
    HIP_TRY(B.lat.alloc(ngroups * (size_t)kAnnealGroupWords));
    HIP_TRY(B.ebuf.alloc(ebuf_n));
    HIP_TRY(B.emin.alloc(nout));
    HIP_TRY(B.efin.alloc(nout));
    HIP_TRY(B.sweeps.alloc(nout));
    AnnealArgs a{};
    a.sys = B.sys.p; a.lat = B.lat.p; a.ebuf = B.ebuf.p; a.beta = B.beta.p;
    a.num_temps = P.num_temperatures; a.block_size = P.block_size; a.max_blocks = P.max_blocks;
    a.chains = P.chains; a.groups_per_sys = gps;
    a.tol = P.stdev_tolerance; a.frozen = P.frozen_criterion;
    a.min_energy = B.emin.p; a.final_energy = B.efin.p; a.sweeps = B.sweeps.p;
    bool has_model[2] = {false, false};
    size_t lds = 0;   // the largest per-site field, staged in LDS by each workgroup
    for (int si = 0; si < num_systems; ++si) {
        has_model[ds[(size_t)si].model] = true;
        if (systems[si].field) lds = std::max(lds, (size_t)ds[(size_t)si].N * sizeof(double));
    }
    if (has_model[REWL_ISING2D]) {
        hipLaunchKernelGGL(k_anneal<REWL_ISING2D>, dim3((unsigned)ngroups), dim3(kLanes), lds, st, a);
        HIP_TRY(hipGetLastError());
    }
    if (has_model[REWL_ASHKIN_TELLER2D]) {
        hipLaunchKernelGGL(k_anneal<REWL_ASHKIN_TELLER2D>, dim3((unsigned)ngroups), dim3(kLanes), lds, st, a);
        HIP_TRY(hipGetLastError());
    }
    HIP_TRY(hipStreamSynchronize(st));
    HIP_TRY(hipMemcpy(min_energy, B.emin.p, nout * sizeof(double), hipMemcpyDeviceToHost));
    HIP_TRY(hipMemcpy(final_energy, B.efin.p, nout * sizeof(double), hipMemcpyDeviceToHost));
    HIP_TRY(hipMemcpy(sweeps, B.sweeps.p, nout * sizeof(uint64_t), hipMemcpyDeviceToHost));
    if (final_spins) {
        std::vector<uint64_t> lat(ngroups * (size_t)kAnnealGroupWords);
        HIP_TRY(hipMemcpy(lat.data(), B.lat.p, lat.size() * sizeof(uint64_t), hipMemcpyDeviceToHost));
        int8_t* o = final_spins;
        for (int si = 0; si < num_systems; ++si) {
            const DevSystem& D = ds[(size_t)si];
            const int planes = model_info(D.model).planes;
            for (int ch = 0; ch < P.chains; ++ch) {
                const uint64_t* g = lat.data() + ((size_t)si * gps + (size_t)(ch / kLanes)) * kAnnealGroupWords;
                const int lane = ch % kLanes;
                for (int i = 0; i < D.N; ++i)
                    for (int q = 0; q < planes; ++q) {
                        const uint64_t w = g[(size_t)(q * D.L + i / D.L) * kLanes + (size_t)lane];
                        *o++ = ((w >> (i % D.L)) & 1ull) ? -1 : 1;
                    }
            }
        }
    }
    return REWL_OK;
}

int rewl_random_field(uint64_t seed, int32_t distribution, double strength, int32_t num_sites, double* out) {
    if (!out || num_sites < 0) return fail(REWL_ERR_INVALID, "rewl_random_field: bad argument");
    if (distribution != REWL_DISORDER_UNIFORM && distribution != REWL_DISORDER_GAUSSIAN)
        return fail(REWL_ERR_INVALID, "rewl_random_field: unknown distribution");
    std::mt19937_64 gen(seed);
    std::uniform_real_distribution<double> u_real(0., 1.);
    const double eps = std::numeric_limits<double>::epsilon();
    const double two_pi = 2.0 * std::acos(-1.0);
    auto draw = [&]() -> double {
        if (distribution == REWL_DISORDER_UNIFORM) return 2. * strength * (-1. + 2. * u_real(gen));
        double u = u_real(gen), v = u_real(gen);
        while (u <= eps) { u = u_real(gen); v = u_real(gen); }
        const double magnitude = strength * std::sqrt(-2.0 * std::log(u));
        const double z0 = magnitude * std::cos(two_pi * v) + 0.;
        const double z1 = magnitude * std::sin(two_pi * v) + 0.;
        const bool return_cos = u_real(gen) < 0.5;
        return z0 * return_cos + z1 * (!return_cos);
    };
    for (int32_t i = 0; i < num_sites; ++i) {
        double h = 0.;
        for (int k = 0; k < 20; ++k) h = draw();   // WAIT_BETWEEN_FIELD_GENERATION (random_fields.hpp:12)
        h = draw();
        out[i] = h;
    }
    return REWL_OK;
}

// LDS read bandwidth: every thread reads 16 B per iteration from a 16 KiB LDS
// buffer, consecutive lanes at consecutive 16-byte slots (no bank conflict),
// eight independent reads in flight per thread; the values are folded into a
// result that is stored only if it equals a constant it never takes, which
// keeps the reads live without any global traffic in the loop.
constexpr int kLdsProbeSlots = 1024;   // 16-byte slots = 16 KiB per workgroup
__global__ void __launch_bounds__(256) k_lds_probe(int iters, uint32_t* sink) {
    __shared__ uint4 buf[kLdsProbeSlots];
    const int t = threadIdx.x;
    for (int i = t; i < kLdsProbeSlots; i += 256) buf[i] = make_uint4(i, 3 * i, 5 * i, 7 * i);
    __syncthreads();
    uint32_t a0 = 0, a1 = 0, a2 = 0, a3 = 0;
    for (int k = 0; k < iters; k += 8) {
        // the slots repeat with a period of a few iterations: an opaque base
        // keeps the compiler from proving the reads loop-invariant and
        // hoisting them out of the loop;
        int base = t + k * 128;
        asm volatile("" : "+v"(base));
        // eight distinct slots per thread and iteration (offsets j * 128 of
        // 1024), so that no two reads of an iteration can be merged
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const uint4 v = buf[(base + j * 128) & (kLdsProbeSlots - 1)];
            a0 ^= v.x; a1 += v.y; a2 ^= v.z; a3 += v.w;
        }
    }
    if ((a0 ^ a1 ^ a2 ^ a3) == 0x9e3779b9u) sink[blockIdx.x] = 1u;
}

int rewl_selfcheck(int32_t what, double* out) {
    if ((what < 0 || what > 2) || !out) return fail(REWL_ERR_INVALID, "unknown self-check");
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0) return fail(REWL_ERR_NO_DEVICE, "no HIP device");
    if (what == 2) {
        int dev = 0, cus = 0;
        HIP_TRY(hipGetDevice(&dev));
        HIP_TRY(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
        const int blocks = cus * 8, iters = 1 << 16;
        uint32_t* sink = nullptr;
        HIP_TRY(hipMalloc((void**)&sink, (size_t)blocks * sizeof(uint32_t)));
        hipEvent_t e0 = nullptr, e1 = nullptr;
        hipError_t e = hipEventCreate(&e0);
        if (e == hipSuccess) e = hipEventCreate(&e1);
        float best = 0.f;
        for (int rep = 0; rep < 4 && e == hipSuccess; ++rep) {   // the first launch warms the clocks
            e = hipEventRecord(e0, nullptr);
            if (e == hipSuccess) {
                hipLaunchKernelGGL(k_lds_probe, dim3(blocks), dim3(256), 0, nullptr, iters, sink);
                e = hipGetLastError();
            }
            if (e == hipSuccess) e = hipEventRecord(e1, nullptr);
            if (e == hipSuccess) e = hipEventSynchronize(e1);
            float ms = 0.f;
            if (e == hipSuccess) e = hipEventElapsedTime(&ms, e0, e1);
            if (e == hipSuccess && rep > 0 && (best == 0.f || ms < best)) best = ms;
        }
        if (e0) (void)hipEventDestroy(e0);
        if (e1) (void)hipEventDestroy(e1);
        (void)hipFree(sink);
        if (e != hipSuccess) return fail(REWL_ERR_DEVICE, std::string("rewl_selfcheck: ") + hipGetErrorString(e));
        const double bytes = (double)blocks * 256.0 * 16.0 * (double)iters;
        *out = bytes / (best * 1e-3) / 1e9;   // GB/s
        return REWL_OK;
    }
    if (what == 1) {
        // device acceptance bounds (device log) against the same function on the
        // host (glibc log) for 2^24 sampled words and the extreme words
        const uint32_t n = 1u << 24;
        std::vector<uint32_t> ks(n);
        for (uint32_t i = 0; i < n; ++i) ks[i] = i * 257u + 12345u;
        ks[0] = 0u;
        ks[1] = 1u;
        ks[2] = 0xffffffffu;
        ks[3] = 0xfffffffeu;
        std::vector<BoundEntry> tab(kBoundTabN);
        build_bound_table(tab.data());
        uint32_t* dk = nullptr;
        double* db = nullptr;
        BoundEntry* dt = nullptr;
        HIP_TRY(hipMalloc((void**)&dk, n * sizeof(uint32_t)));
        hipError_t e = hipMalloc((void**)&db, n * sizeof(double));
        if (e == hipSuccess) e = hipMalloc((void**)&dt, kBoundTabN * sizeof(BoundEntry));
        if (e == hipSuccess) e = hipMemcpy(dk, ks.data(), n * sizeof(uint32_t), hipMemcpyHostToDevice);
        if (e == hipSuccess) e = hipMemcpy(dt, tab.data(), kBoundTabN * sizeof(BoundEntry), hipMemcpyHostToDevice);
        if (e == hipSuccess) {
            hipLaunchKernelGGL(k_selfcheck_bounds, dim3(4096), dim3(256), 0, nullptr, dk, n, dt, db);
            e = hipGetLastError();
        }
        std::vector<double> got(n);
        if (e == hipSuccess) e = hipMemcpy(got.data(), db, n * sizeof(double), hipMemcpyDeviceToHost);
        (void)hipFree(dk);
        (void)hipFree(db);
        (void)hipFree(dt);
        if (e != hipSuccess) return fail(REWL_ERR_DEVICE, std::string("rewl_selfcheck: ") + hipGetErrorString(e));
        uint64_t bad = 0;
        for (uint32_t i = 0; i < n; ++i) bad += double_bits(got[i]) != double_bits(accept_bound(ks[i], tab.data()));
        *out = (double)bad;
        return REWL_OK;
    }
    unsigned long long* d = nullptr;
    HIP_TRY(hipMalloc((void**)&d, sizeof(unsigned long long)));
    hipError_t e = hipMemset(d, 0, sizeof(unsigned long long));
    // all 2^32 words in 4 launches of 2^30
    for (uint32_t q = 0; q < 4 && e == hipSuccess; ++q) {
        hipLaunchKernelGGL(k_selfcheck_neglog, dim3(4096), dim3(256), 0, nullptr, q << 30, 1u << 30, d);
        e = hipGetLastError();
    }
    unsigned long long bits = 0;
    if (e == hipSuccess) e = hipMemcpy(&bits, d, sizeof(bits), hipMemcpyDeviceToHost);
    (void)hipFree(d);
    if (e != hipSuccess) return fail(REWL_ERR_DEVICE, std::string("rewl_selfcheck: ") + hipGetErrorString(e));
    double v;
    std::memcpy(&v, &bits, sizeof(v));
    *out = v;
    return REWL_OK;
}

}  // extern "C"

// ---- warm-start MLP (include/rewl_mlp.h) ---------------------------------------------
#include "../../include/rewl_mlp.h"
#include "mlp.hpp"

static_assert(rewl::mlp::NP == REWL_MLP_NUM_PARAMS, "parameter count");

struct rewl_mlp {
    int device = 0;
    hipStream_t stream = nullptr;
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    float* theta = nullptr;     // FP32 master
    float* adam_m = nullptr;
    float* adam_v = nullptr;
    uint16_t* wq = nullptr;     // bf16 copies
    float* grad = nullptr;      // NPART
    float* part = nullptr;      // part_rows x NPART
    int part_rows = 0;
    float* dx = nullptr;        // data on the device
    float* dt = nullptr;
    float* dw = nullptr;
    float* dy = nullptr;
    int64_t data_cap = 0;
    int64_t adam_t = 0;
    double last_ms = 0.0;
};

namespace {

constexpr int kMlpMaxGrid = 512;

void mlp_free_data(rewl_mlp* m) {
    for (float** p : {&m->dx, &m->dt, &m->dw, &m->dy})
        if (*p) {
            (void)hipFree(*p);
            *p = nullptr;
        }
    m->data_cap = 0;
}

int mlp_reserve(rewl_mlp* m, int64_t n) {
    if (n <= m->data_cap) return REWL_OK;
    mlp_free_data(m);
    HIP_TRY(hipMalloc((void**)&m->dx, (size_t)n * rewl::mlp::NIN * sizeof(float)));
    HIP_TRY(hipMalloc((void**)&m->dt, (size_t)n * sizeof(float)));
    HIP_TRY(hipMalloc((void**)&m->dw, (size_t)n * sizeof(float)));
    HIP_TRY(hipMalloc((void**)&m->dy, (size_t)n * sizeof(float)));
    m->data_cap = n;
    return REWL_OK;
}

int mlp_grid(int64_t npts) {
    const int64_t tiles = (npts + rewl::mlp::TILE - 1) / rewl::mlp::TILE;
    return (int)std::max<int64_t>(1, std::min<int64_t>(tiles, kMlpMaxGrid));
}

// uploads x (and t, w when given); w == nullptr means unit weights
int mlp_upload(rewl_mlp* m, const float* x, const float* t, const float* w, int64_t n, double* wsum) {
    for (int64_t i = 0; i < (int64_t)n * rewl::mlp::NIN; ++i)
        if (!std::isfinite(x[i])) return fail(REWL_ERR_NONFINITE, "rewl_mlp: non-finite input feature");
    int rc = mlp_reserve(m, n);
    if (rc) return rc;
    HIP_TRY(hipMemcpyAsync(m->dx, x, (size_t)n * rewl::mlp::NIN * sizeof(float), hipMemcpyHostToDevice, m->stream));
    if (t) {
        for (int64_t i = 0; i < n; ++i)
            if (!std::isfinite(t[i])) return fail(REWL_ERR_NONFINITE, "rewl_mlp: non-finite target");
        HIP_TRY(hipMemcpyAsync(m->dt, t, (size_t)n * sizeof(float), hipMemcpyHostToDevice, m->stream));
        double s = 0.0;
        if (w) {
            for (int64_t i = 0; i < n; ++i) {
                if (!(w[i] >= 0.f) || !std::isfinite(w[i]))
                    return fail(REWL_ERR_INVALID, "rewl_mlp: weights must be finite and >= 0");
                s += w[i];
            }
            HIP_TRY(hipMemcpyAsync(m->dw, w, (size_t)n * sizeof(float), hipMemcpyHostToDevice, m->stream));
        } else {
            s = (double)n;
        }
        if (!(s > 0.0)) return fail(REWL_ERR_INVALID, "rewl_mlp: weights sum to zero");
        if (wsum) *wsum = s;
    }
    return REWL_OK;
}

rewl::mlp::Args mlp_args(const rewl_mlp* m, int64_t n, bool weighted) {
    rewl::mlp::Args a{};
    a.theta = m->theta;
    a.wq = m->wq;
    a.x = m->dx;
    a.t = m->dt;
    a.w = weighted ? m->dw : nullptr;
    a.n = n;
    a.npts = n;
    return a;
}

int mlp_ensure_part(rewl_mlp* m, int rows) {
    if (rows <= m->part_rows) return REWL_OK;
    if (m->part) (void)hipFree(m->part);
    m->part = nullptr;
    m->part_rows = 0;
    HIP_TRY(hipMalloc((void**)&m->part, (size_t)rows * rewl::mlp::NPART * sizeof(float)));
    m->part_rows = rows;
    return REWL_OK;
}

int mlp_check(const rewl_mlp* m) {
    if (!m) return fail(REWL_ERR_INVALID, "rewl_mlp: null handle");
    HIP_TRY(hipSetDevice(m->device));
    return REWL_OK;
}

}  // namespace

extern "C" {

int rewl_mlp_create(uint64_t seed, rewl_mlp** out) {
    using namespace rewl::mlp;
    if (!out) return fail(REWL_ERR_INVALID, "rewl_mlp_create: null output");
    *out = nullptr;
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0)
        return fail(REWL_ERR_NO_DEVICE, "no HIP device visible: the warm-start MLP runs only on the GPU");
    // He-uniform weights from a splitmix64 stream, zero biases
    std::vector<float> th(NP, 0.f);
    uint64_t st = seed;
    auto uni = [&st]() {
        uint64_t z = (st += 0x9E3779B97F4A7C15ull);
        z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
        z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
        z ^= z >> 31;
        return (double)(z >> 11) * 0x1p-53;
    };
    auto fill = [&](int off, int count, int fan_in) {
        const double a = std::sqrt(6.0 / fan_in);
        for (int i = 0; i < count; ++i) th[off + i] = (float)((2.0 * uni() - 1.0) * a);
    };
    fill(O_W1, H * NIN, NIN);
    fill(O_W2, H * H, H);
    fill(O_W3, H * H, H);
    fill(O_W4, H, 4 * H);
    auto* m = new rewl_mlp();
    int rc = REWL_OK;
    auto body = [&]() -> int {
        HIP_TRY(hipGetDevice(&m->device));
        HIP_TRY(hipStreamCreate(&m->stream));
        HIP_TRY(hipEventCreate(&m->ev0));
        HIP_TRY(hipEventCreate(&m->ev1));
        HIP_TRY(hipMalloc((void**)&m->theta, NP * sizeof(float)));
        HIP_TRY(hipMalloc((void**)&m->adam_m, NP * sizeof(float)));
        HIP_TRY(hipMalloc((void**)&m->adam_v, NP * sizeof(float)));
        HIP_TRY(hipMalloc((void**)&m->wq, NQ * sizeof(uint16_t)));
        HIP_TRY(hipMalloc((void**)&m->grad, NPART * sizeof(float)));
        return REWL_OK;
    };
    rc = body();
    if (rc == REWL_OK) rc = rewl_mlp_set_params(m, th.data(), NP);
    if (rc != REWL_OK) {
        std::string keep = g_err;
        rewl_mlp_destroy(m);
        g_err = keep;
        return rc;
    }
    *out = m;
    return REWL_OK;
}

int rewl_mlp_destroy(rewl_mlp* m) {
    if (!m) return REWL_OK;
    (void)hipSetDevice(m->device);
    if (m->stream) (void)hipStreamSynchronize(m->stream);
    mlp_free_data(m);
    for (float* p : {m->theta, m->adam_m, m->adam_v, m->grad, m->part})
        if (p) (void)hipFree(p);
    if (m->wq) (void)hipFree(m->wq);
    if (m->ev0) (void)hipEventDestroy(m->ev0);
    if (m->ev1) (void)hipEventDestroy(m->ev1);
    if (m->stream) (void)hipStreamDestroy(m->stream);
    delete m;
    return REWL_OK;
}

int rewl_mlp_get_params(const rewl_mlp* m, float* theta, int64_t n) {
    int rc = mlp_check(m);
    if (rc) return rc;
    if (!theta || n != rewl::mlp::NP) return fail(REWL_ERR_INVALID, "rewl_mlp_get_params: need REWL_MLP_NUM_PARAMS values");
    HIP_TRY(hipMemcpyAsync(theta, m->theta, (size_t)n * sizeof(float), hipMemcpyDeviceToHost, m->stream));
    HIP_TRY(hipStreamSynchronize(m->stream));
    return REWL_OK;
}

int rewl_mlp_set_params(rewl_mlp* m, const float* theta, int64_t n) {
    using namespace rewl::mlp;
    int rc = mlp_check(m);
    if (rc) return rc;
    if (!theta || n != NP) return fail(REWL_ERR_INVALID, "rewl_mlp_set_params: need REWL_MLP_NUM_PARAMS values");
    for (int64_t i = 0; i < n; ++i)
        if (!std::isfinite(theta[i])) return fail(REWL_ERR_NONFINITE, "rewl_mlp_set_params: non-finite parameter");
    HIP_TRY(hipMemcpyAsync(m->theta, theta, NP * sizeof(float), hipMemcpyHostToDevice, m->stream));
    HIP_TRY(hipMemsetAsync(m->adam_m, 0, NP * sizeof(float), m->stream));
    HIP_TRY(hipMemsetAsync(m->adam_v, 0, NP * sizeof(float), m->stream));
    hipLaunchKernelGGL(k_mlp_quantise, dim3((NP + 255) / 256), dim3(256), 0, m->stream, m->theta, m->wq);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipStreamSynchronize(m->stream));
    m->adam_t = 0;
    return REWL_OK;
}

int rewl_mlp_forward(rewl_mlp* m, const float* x, int64_t n, float* y) {
    using namespace rewl::mlp;
    int rc = mlp_check(m);
    if (rc) return rc;
    if (!x || !y || n <= 0) return fail(REWL_ERR_INVALID, "rewl_mlp_forward: empty input");
    rc = mlp_upload(m, x, nullptr, nullptr, n, nullptr);
    if (rc) return rc;
    Args a = mlp_args(m, n, false);
    a.y = m->dy;
    HIP_TRY(hipEventRecord(m->ev0, m->stream));
    hipLaunchKernelGGL(k_mlp<false>, dim3(mlp_grid(n)), dim3(256), 0, m->stream, a);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipEventRecord(m->ev1, m->stream));
    HIP_TRY(hipMemcpyAsync(y, m->dy, (size_t)n * sizeof(float), hipMemcpyDeviceToHost, m->stream));
    HIP_TRY(hipStreamSynchronize(m->stream));
    float ms = 0.f;
    HIP_TRY(hipEventElapsedTime(&ms, m->ev0, m->ev1));
    m->last_ms = ms;
    return REWL_OK;
}

int rewl_mlp_gradient(rewl_mlp* m, const float* x, const float* t, const float* w, int64_t n, float* grad,
                      double* loss) {
    using namespace rewl::mlp;
    int rc = mlp_check(m);
    if (rc) return rc;
    if (!x || !t || !grad || n <= 0) return fail(REWL_ERR_INVALID, "rewl_mlp_gradient: empty input");
    double wsum = 0.0;
    rc = mlp_upload(m, x, t, w, n, &wsum);
    if (rc) return rc;
    const int G = mlp_grid(n);
    rc = mlp_ensure_part(m, G);
    if (rc) return rc;
    Args a = mlp_args(m, n, w != nullptr);
    a.inv_wsum = (float)(1.0 / wsum);
    a.part = m->part;
    HIP_TRY(hipEventRecord(m->ev0, m->stream));
    hipLaunchKernelGGL(k_mlp<true>, dim3(G), dim3(256), 0, m->stream, a);
    HIP_TRY(hipGetLastError());
    hipLaunchKernelGGL(k_mlp_reduce, dim3((NPART + 63) / 64), dim3(64), 0, m->stream, m->part, G, m->grad);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipEventRecord(m->ev1, m->stream));
    std::vector<float> g(NPART);
    HIP_TRY(hipMemcpyAsync(g.data(), m->grad, NPART * sizeof(float), hipMemcpyDeviceToHost, m->stream));
    HIP_TRY(hipStreamSynchronize(m->stream));
    std::copy(g.begin(), g.begin() + NP, grad);
    if (loss) *loss = (double)g[NP] / wsum;
    float ms = 0.f;
    HIP_TRY(hipEventElapsedTime(&ms, m->ev0, m->ev1));
    m->last_ms = ms;
    return REWL_OK;
}

int rewl_mlp_train(rewl_mlp* m, const float* x, const float* t, const float* w, int64_t n,
                   const rewl_mlp_train_params* p, float* loss_history) {
    using namespace rewl::mlp;
    int rc = mlp_check(m);
    if (rc) return rc;
    if (!x || !t || !p || n <= 0) return fail(REWL_ERR_INVALID, "rewl_mlp_train: empty input");
    if (n >= (int64_t)1 << 32) return fail(REWL_ERR_INVALID, "rewl_mlp_train: at most 2^32 - 1 points");
    if (p->steps < 0 || p->batch <= 0 || !(p->lr > 0.0) || !(p->lr_final >= 0.0) || !(p->beta1 >= 0.0 && p->beta1 < 1.0) ||
        !(p->beta2 >= 0.0 && p->beta2 < 1.0) || !(p->eps > 0.0) || p->warmup < 0)
        return fail(REWL_ERR_INVALID, "rewl_mlp_train: bad hyper-parameters");
    double wsum = 0.0;
    rc = mlp_upload(m, x, t, w, n, &wsum);
    if (rc) return rc;
    const int G = mlp_grid(p->batch);
    rc = mlp_ensure_part(m, G);
    if (rc) return rc;
    Args a = mlp_args(m, n, w != nullptr);
    a.npts = p->batch;
    a.sample = 1;
    a.k0 = (uint32_t)p->seed;
    a.k1 = (uint32_t)(p->seed >> 32);
    // minibatch loss: sum_k w_k (y_k - t_k)^2 / (batch * mean weight)
    a.inv_wsum = (float)(1.0 / ((double)p->batch * (wsum / (double)n)));
    a.part = m->part;
    float* dloss = nullptr;
    if (loss_history && p->steps > 0) HIP_TRY(hipMalloc((void**)&dloss, (size_t)p->steps * sizeof(float)));
    HIP_TRY(hipEventRecord(m->ev0, m->stream));
    for (int64_t s = 0; s < p->steps; ++s) {
        a.step = (uint64_t)s;
        hipLaunchKernelGGL(k_mlp<true>, dim3(G), dim3(256), 0, m->stream, a);
        m->adam_t += 1;
        double lr = p->lr_final + 0.5 * (p->lr - p->lr_final) * (1.0 + std::cos(M_PI * (double)s / (double)std::max<int64_t>(1, p->steps)));
        if (s < p->warmup) lr *= (double)(s + 1) / (double)p->warmup;
        const double bc1 = 1.0 - std::pow(p->beta1, (double)m->adam_t);
        const double bc2 = 1.0 - std::pow(p->beta2, (double)m->adam_t);
        hipLaunchKernelGGL(k_mlp_step, dim3((NPART + 63) / 64), dim3(64), 0, m->stream, (const float*)m->part, G, m->theta,
                           m->adam_m, m->adam_v, (float)lr, (float)p->beta1, (float)p->beta2, (float)p->eps, (float)bc1,
                           (float)bc2, m->wq, dloss ? dloss + s : nullptr);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) {
            if (dloss) (void)hipFree(dloss);
            return fail(REWL_ERR_DEVICE, std::string("rewl_mlp_train launch: ") + hipGetErrorString(e));
        }
    }
    HIP_TRY(hipEventRecord(m->ev1, m->stream));
    HIP_TRY(hipStreamSynchronize(m->stream));
    float ms = 0.f;
    HIP_TRY(hipEventElapsedTime(&ms, m->ev0, m->ev1));
    m->last_ms = ms;
    if (dloss) {
        std::vector<float> h((size_t)p->steps);
        hipError_t e = hipMemcpy(h.data(), dloss, h.size() * sizeof(float), hipMemcpyDeviceToHost);
        (void)hipFree(dloss);
        if (e != hipSuccess) return fail(REWL_ERR_DEVICE, std::string("rewl_mlp_train: ") + hipGetErrorString(e));
        for (int64_t s = 0; s < p->steps; ++s) loss_history[s] = h[(size_t)s] * a.inv_wsum;
    }
    return REWL_OK;
}

int rewl_mlp_last_ms(const rewl_mlp* m, double* ms) {
    if (!m || !ms) return fail(REWL_ERR_INVALID, "rewl_mlp_last_ms: null argument");
    *ms = m->last_ms;
    return REWL_OK;
}

}  // extern "C"
