// The instances of the row-unrolled sweep kernel (sweep_tuned.hpp), in a
// translation unit of their own: they take most of the build's time, and the
// engine is compiled beside them.
#include <hip/hip_runtime.h>

#include "sweep_tuned.hpp"

namespace rewl {

const void* tuned_kernel(int model, int L, bool simple, int spec, int obs);

namespace {

template <int MODEL, int L, bool SIMPLE>
const void* of_form(int spec, int obs) {
    if (spec == 0) return (const void*)k_sweep_tuned<MODEL, L, SIMPLE, 0>;
    if (spec == 2) return (const void*)k_sweep_tuned<MODEL, L, SIMPLE, 2>;
    if (obs == 2) return (const void*)k_sweep_tuned<MODEL, L, SIMPLE, 1, 2>;
    if (obs) return (const void*)k_sweep_tuned<MODEL, L, SIMPLE, 1, 1>;
    return (const void*)k_sweep_tuned<MODEL, L, SIMPLE, 1>;
}

template <int MODEL, int L>
const void* of_size(bool simple, int spec, int obs) {
    return simple ? of_form<MODEL, L, true>(spec, obs) : of_form<MODEL, L, false>(spec, obs);
}

template <int MODEL>
const void* of_model(int L, bool simple, int spec, int obs) {
    switch (L) {
        case 16: return of_size<MODEL, 16>(simple, spec, obs);
        case 24: return of_size<MODEL, 24>(simple, spec, obs);
        case 32: return of_size<MODEL, 32>(simple, spec, obs);
        case 48: return of_size<MODEL, 48>(simple, spec, obs);
        case 64: return of_size<MODEL, 64>(simple, spec, obs);
        default: return nullptr;
    }
}

}  // namespace

// The kernel of one model, lattice side, range test (simple: plainly min <= E
// < max), speculation (0 none, 1 next slot, 2 next read) and observables (0,
// 1, 2; spec 1 only); null if there is none.
const void* tuned_kernel(int model, int L, bool simple, int spec, int obs) {
    return model == 0 ? of_model<0>(L, simple, spec, obs) : of_model<1>(L, simple, spec, obs);
}

}  // namespace rewl
