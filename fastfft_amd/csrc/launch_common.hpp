// Shared helpers of the launch_*.hip translation units.
#pragma once

#include <cstdlib>
#include <type_traits>
#include <typeinfo>
#include <utility>

#include "launch.hpp"
#include "line_kernels.hpp"

namespace fastfft_amd {

static_assert(kTwiddleTableN == kTwiddleN + 2 * kTwiddleN, "host and device twiddle table lengths differ");

inline LineMap to_device(const HostLineMap& m) {
    LineMap d;
    d.s1 = m.s1;
    d.s2 = m.s2;
    d.es = m.es;
    d.n2 = m.n2;
    return d;
}

// Calls f(std::integral_constant<int, P>) for the runtime sub-transform size P.
template <class F>
hipError_t dispatch_P(int P, F&& f) {
    switch ( P ) {
        case 2: return f(std::integral_constant<int, 2>{ });
        case 4: return f(std::integral_constant<int, 4>{ });
        case 8: return f(std::integral_constant<int, 8>{ });
        case 16: return f(std::integral_constant<int, 16>{ });
        case 32: return f(std::integral_constant<int, 32>{ });
        case 64: return f(std::integral_constant<int, 64>{ });
        case 128: return f(std::integral_constant<int, 128>{ });
        case 256: return f(std::integral_constant<int, 256>{ });
        case 512: return f(std::integral_constant<int, 512>{ });
        case 1024: return f(std::integral_constant<int, 1024>{ });
        case 2048: return f(std::integral_constant<int, 2048>{ });
        case 4096: return f(std::integral_constant<int, 4096>{ });
        case 8192: return f(std::integral_constant<int, 8192>{ });
        default: return hipErrorInvalidValue;
    }
}

// Grid and LDS of a line stage, with the dynamic-LDS attribute raised above 64 KiB.
template <int P, class K>
hipError_t prepare_launch(K kernel, int nlines, dim3& grid, dim3& block, size_t& lds) {
    using S = LineShape<P>;
    lds     = sizeof(float2) * (size_t)S::LDS;
    grid    = dim3((unsigned)((nlines + S::G - 1) / S::G));
    block   = dim3(S::BLOCK);
    if ( lds > 65536 ) {
        hipError_t e = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if ( e != hipSuccess )
            return e;
    }
    return hipSuccess;
}

inline int twiddle_stride(int N) { return kTwiddleN / N; }

// Integer value of a tuning environment variable (dflt when unset).  Read on
// every call so that tests can switch kernels within one process; getenv is
// cheap next to a kernel launch.
inline int env_int(const char* name, int dflt) {
    const char* v = std::getenv(name);
    return (v && v[0]) ? std::atoi(v) : dflt;
}

// Calls f(N, PPW) for the pair-row kernels (pair_rows.hpp): rows of N points, PPW pairs per
// workgroup, at most FASTFFT_PAIR_GROUP; not supported where pair_rows_pay (plan.hpp) says no.
// Four pairs make 64-byte segments (workgroups of 1024 threads at N = 4096; 8192-point rows fit
// two).  The group is halved below 160 workgroups' worth of pairs, which keeps CUs busy.  Whole 2-D
// transforms, us with one, two and four pairs: 509 whole rows of 4096 points forward 15.8, 16.0 and
// 19.8, inverse 16.1, 17.6 and 22.2; 809 rows 24.1, 21.8, 25.6 and 23.6, 22.5, 27.1; 1281 rows 29.5, 29.6,
// 29.3 and 27.4, 26.5, 28.7; 4091 rows 66.1, 62.1, 53.4 and 61.9, 58.1, 57.9; 1281 rows of 2048 points cut to
// 509 values 19.8, 18.9 and 18.2.  8192-point rows keep single pairs up to 512 of them, which are all in
// flight at once, two to a CU: 509 rows inverse 27.4 with one and 33.5 with two, 1024 rows forward 38.4 and
// 38.8, inverse 34.4 and 37.1; 2045 rows 64.4 and 60.0, 60.4 and 59.4.
template <class F>
hipError_t pair_rows_dispatch(int N, int nrows, int min_pairs, F&& f) {
    const int npairs = (nrows + 1) / 2, cap = env_int("FASTFFT_PAIR_GROUP", 4);
    if ( ! pair_rows_pay(N, nrows, min_pairs) )
        return hipErrorNotSupported;
    int       g      = N < 8192 ? 4 : npairs > 512 ? 2 : 1;
    while ( g > 1 && (g > cap || (N < 8192 && npairs < 160 * g)) )
        g /= 2;
    auto by_n = [&](auto nc) -> hipError_t {
        constexpr int NN = decltype(nc)::value;
        if constexpr ( NN <= 4096 )
            if ( g == 4 )
                return f(nc, std::integral_constant<int, 4>{ });
        return g >= 2 ? f(nc, std::integral_constant<int, 2>{ }) : f(nc, std::integral_constant<int, 1>{ });
    };
    switch ( N ) {
        case 1024: return by_n(std::integral_constant<int, 1024>{ });
        case 2048: return by_n(std::integral_constant<int, 2048>{ });
        case 4096: return by_n(std::integral_constant<int, 4096>{ });
        case 8192: return by_n(std::integral_constant<int, 8192>{ });
        default: return hipErrorNotSupported;
    }
}

// A type whose mangled name spells out the kernel K with its template arguments.
template <auto K>
struct KernelTag { };

// K<<<grid, block, lds, st>>>(a...), named on stderr first when FASTFFT_LOG is set.
template <auto K, class... A>
inline void launch_kernel(dim3 grid, dim3 block, size_t lds, hipStream_t st, A&&... a) {
    if ( log_enabled( ) )
        log_launch(typeid(KernelTag<K>).name( ), grid, block, lds);
    K<<<grid, block, lds, st>>>(std::forward<A>(a)...);
}

} // namespace fastfft_amd
