// Forward line stages: R2C x-pass (real input) and C2C y/z passes.
#include <cstdint>

#include "full_wave.hpp"
#include "launch_common.hpp"
#include "pair_rows.hpp"
#include "rows_packed.hpp"
#include "rows_wave.hpp"

namespace fastfft_amd {

template <int P, typename TIn, bool REAL, typename TOut>
static hipError_t go_fwd(const Stage& s, const StageIO& io, const float2* tw, hipStream_t st) {
    dim3       grid, block;
    size_t     lds;
    hipError_t e = prepare_launch<P>(k_fwd<P, TIn, REAL, TOut>, s.nlines, grid, block, lds);
    if ( e != hipSuccess )
        return e;
    launch_kernel<k_fwd<P, TIn, REAL, TOut>>(grid, block, lds, st, static_cast<const TIn*>(io.src), to_device(s.im), s.L,
                                                        static_cast<TOut*>(io.dst), to_device(s.om), s.N, s.Q, s.nout,
                                                        s.nlines, io.scale, tw, twiddle_stride(s.N));
    return hipGetLastError( );
}

// R2C rows with P in {256, 512, 1024}: one block per row, one wave per sub-transform.
template <int P, int Q, typename TIn>
static hipError_t go_r2c_wave(const Stage& s, const StageIO& io, const float2* tw, hipStream_t st) {
    launch_kernel<k_r2c_rows_wave<P, Q, TIn>>(dim3((unsigned)s.nlines), dim3(64 * Q), 0, st,
            static_cast<const TIn*>(io.src), to_device(s.im), s.L, static_cast<float2*>(io.dst), to_device(s.om), s.nout,
            s.nlines, io.scale, tw, nullptr);
    return hipGetLastError( );
}

template <int P, int Q, typename TIn>
static hipError_t go_r2c_wave_batch(const Stage& s, const RowBatchItem* items, int n, int max_rows, float pre,
                                    const float2* tw, hipStream_t st) {
    launch_kernel<k_r2c_rows_wave<P, Q, TIn>>(dim3((unsigned)max_rows, (unsigned)n), dim3(64 * Q), 0, st,
            nullptr, to_device(s.im), s.L, nullptr, to_device(s.om), s.nout, max_rows, pre, tw, items);
    return hipGetLastError( );
}

// R2C rows of 512 or 1024 real points, one wave per row (rows_packed.hpp); the
// batched form takes its per-template in, pitch, L and row count from items.
static bool r2c_packed_covers(const Stage& s) {
    return s.kind == StageKind::fwd_real && (s.N == 512 || s.N == 1024) && s.nout >= 1 && s.nout <= s.N / 2 + 1 &&
           s.L >= 0 && s.L <= s.N && ! env_int("FASTFFT_NO_PACKED_ROWS", 0);
}

template <int P, typename TIn>
static hipError_t go_r2c_packed(const Stage& s, const void* src, void* dst, int nrows, float pre, const float2* tw,
                                const RowBatchItem* items, int n, hipStream_t st) {
    const dim3 grid((unsigned)((nrows + kPackedRows - 1) / kPackedRows), (unsigned)n);
    launch_kernel<k_r2c_rows_packed<P, TIn>>(grid, dim3(64 * kPackedRows), 0, st, static_cast<const TIn*>(src), to_device(s.im), s.L,
                                                                      static_cast<float2*>(dst), to_device(s.om), s.nout,
                                                                      nrows, pre, tw, items);
    return hipGetLastError( );
}

static hipError_t launch_r2c_packed(const Stage& s, const void* src, void* dst, RealT rt, int nrows, float pre,
                                    const float2* tw, const RowBatchItem* items, int n, hipStream_t st) {
    if ( ! r2c_packed_covers(s) || nrows < 1 || n < 1 )
        return hipErrorNotSupported;
    if ( s.N == 512 )
        return rt == RealT::f32 ? go_r2c_packed<256, float>(s, src, dst, nrows, pre, tw, items, n, st)
                                : go_r2c_packed<256, __half>(s, src, dst, nrows, pre, tw, items, n, st);
    return rt == RealT::f32 ? go_r2c_packed<512, float>(s, src, dst, nrows, pre, tw, items, n, st)
                            : go_r2c_packed<512, __half>(s, src, dst, nrows, pre, tw, items, n, st);
}

// The stage with sub-transforms of at least 256 points: shorter ones run no faster per point,
// and no row kernel takes them (128 of 2048 points: the whole correlation 40 us on the generic
// line kernel).
static Stage r2c_at_least_256(const Stage& s) {
    Stage r = s;
    if ( r.P < 256 && r.N >= 256 ) {
        r.P = 256;
        r.Q = r.N / 256;
    }
    return r;
}

// (P, Q) of an R2C row stage that k_r2c_rows_wave covers
static bool r2c_rows_shape(const Stage& s) {
    return (s.P == 256 || s.P == 512 || s.P == 1024) && (s.Q == 1 || s.Q == 2 || s.Q == 4 || s.Q == 8 || s.Q == 16) &&
           s.P * s.Q <= kTwiddleN;
}

// Column-major batch output: row r at r, element k at k * es (es even, every column
// holding whole groups of kCmRows rows).
static bool r2c_cm_output(const Stage& s) {
    return s.om.n2 == 1 && s.om.s1 == 1 && s.om.es > 1 && s.om.es % 2 == 0 &&
           s.om.es >= (s.nlines + kCmRows - 1) / kCmRows * kCmRows;
}

bool r2c_rows_batch_covers(const Stage& s) {
    if ( r2c_cm_output(s) )
        return r2c_packed_covers(s) && s.im.n2 == 1 && s.im.es == 1;
    // one template per grid row: single-index lines, unit-stride row-major output with even leading dimension
    return (r2c_rows_shape(s) || r2c_packed_covers(s)) && s.im.n2 == 1 && s.im.es == 1 && s.om.n2 == 1 && s.om.es == 1 &&
           s.om.s1 % 2 == 0;
}

template <int P, typename TIn>
static hipError_t go_r2c_packed_cm(const Stage& s, const RowBatchItem* items, int n, int max_rows, float pre,
                                   const float2* tw, hipStream_t st) {
    const dim3 grid((unsigned)((max_rows + kCmRows - 1) / kCmRows), (unsigned)n);
    // non-zero registers of a row's packed input: ceil(L / 128) for the longest template row
    constexpr int E  = P / 64;
    const int     nz = (s.L + 127) / 128;
    auto          go = [&](auto zc) {
        launch_kernel<k_r2c_rows_packed_cm<P, TIn, decltype(zc)::value>>(grid, dim3(64 * kCmWaves), 0, st, s.om.es, s.nout, pre, tw,
                                                                                               items);
        return hipGetLastError( );
    };
    if ( nz <= 1 )
        return go(std::integral_constant<int, 1>{ });
    if ( nz <= 2 )
        return go(std::integral_constant<int, 2>{ });
    if ( nz <= 3 && E > 3 )
        return go(std::integral_constant<int, (E > 3 ? 3 : E)>{ });
    if ( nz <= 4 && E > 4 )
        return go(std::integral_constant<int, (E > 4 ? 4 : E)>{ });
    return go(std::integral_constant<int, E>{ });
}

hipError_t launch_r2c_rows_batch(const Stage& s, const void* items, int n, int max_rows, RealT in_rt, float pre,
                                 const float2* tw, hipStream_t st) {
    if ( ! r2c_rows_batch_covers(s) )
        return hipErrorNotSupported;
    const auto* it = static_cast<const RowBatchItem*>(items);
    if ( r2c_cm_output(s) ) {
        if ( max_rows < 1 || n < 1 )
            return hipErrorNotSupported;
        if ( s.N == 512 )
            return in_rt == RealT::f32 ? go_r2c_packed_cm<256, float>(s, it, n, max_rows, pre, tw, st)
                                       : go_r2c_packed_cm<256, __half>(s, it, n, max_rows, pre, tw, st);
        return in_rt == RealT::f32 ? go_r2c_packed_cm<512, float>(s, it, n, max_rows, pre, tw, st)
                                   : go_r2c_packed_cm<512, __half>(s, it, n, max_rows, pre, tw, st);
    }
    {
        hipError_t e = launch_r2c_packed(s, nullptr, nullptr, in_rt, max_rows, pre, tw, it, n, st);
        if ( e != hipErrorNotSupported )
            return e;
    }
    auto by_p = [&](auto pc) -> hipError_t {
        constexpr int P  = decltype(pc)::value;
        auto          go = [&](auto qc) -> hipError_t {
            constexpr int Q = decltype(qc)::value;
            if constexpr ( P * Q > kTwiddleN )
                return hipErrorNotSupported;
            else
                return in_rt == RealT::f32 ? go_r2c_wave_batch<P, Q, float>(s, it, n, max_rows, pre, tw, st)
                                           : go_r2c_wave_batch<P, Q, __half>(s, it, n, max_rows, pre, tw, st);
        };
        switch ( s.Q ) {
            case 1: return go(std::integral_constant<int, 1>{ });
            case 2: return go(std::integral_constant<int, 2>{ });
            case 4: return go(std::integral_constant<int, 4>{ });
            case 8: return go(std::integral_constant<int, 8>{ });
            case 16: return go(std::integral_constant<int, 16>{ });
            default: return hipErrorNotSupported;
        }
    };
    if ( s.P == 256 )
        return by_p(std::integral_constant<int, 256>{ });
    if ( s.P == 512 )
        return by_p(std::integral_constant<int, 512>{ });
    return by_p(std::integral_constant<int, 1024>{ });
}

template <typename TIn>
static hipError_t try_r2c_wave(const Stage& s, const StageIO& io, const float2* tw, hipStream_t st) {
    auto by_p = [&](auto pc) -> hipError_t {
        constexpr int P = decltype(pc)::value;
        switch ( s.Q ) {
            case 1: return go_r2c_wave<P, 1, TIn>(s, io, tw, st);
            case 2: return go_r2c_wave<P, 2, TIn>(s, io, tw, st);
            case 4: return go_r2c_wave<P, 4, TIn>(s, io, tw, st);
            case 8: return go_r2c_wave<P, 8, TIn>(s, io, tw, st);
            case 16:
                if constexpr ( P * 16 <= kTwiddleN )
                    return go_r2c_wave<P, 16, TIn>(s, io, tw, st);
                return hipErrorNotSupported;
            default: return hipErrorNotSupported;
        }
    };
    if ( s.P == 256 )
        return by_p(std::integral_constant<int, 256>{ });
    if ( s.P == 512 )
        return by_p(std::integral_constant<int, 512>{ });
    if ( s.P == 1024 )
        return by_p(std::integral_constant<int, 1024>{ });
    return hipErrorNotSupported;
}

// Lines of 256 <= N <= 8192 points with L <= N non-zero inputs: one workgroup per
// line, P = 512 (256 for N = 256) and Q = N / P.
template <int P, int Q, typename TIn, bool REAL, typename TOut>
static hipError_t go_full_wave_t(const Stage& s, const StageIO& io, const float2* tw, hipStream_t st) {
    auto go = [&](auto pad) {
        launch_kernel<k_fwd_full_wave<P, Q, TIn, REAL, TOut, decltype(pad)::value>>(dim3((unsigned)s.nlines), dim3(64 * Q), 0, st,
                static_cast<const TIn*>(io.src), to_device(s.im), s.L, static_cast<TOut*>(io.dst), to_device(s.om), s.nout,
                s.nlines, io.scale, tw);
        return hipGetLastError( );
    };
    return s.L < s.N ? go(std::true_type{ }) : go(std::false_type{ });
}

template <int P, int Q>
static hipError_t go_full_wave(const Stage& s, const StageIO& io, const float2* tw, hipStream_t st) {
    if ( io.src_real ) {
        if ( io.dst_ct != CpxT::c64 )
            return hipErrorNotSupported;
        return io.src_rt == RealT::f32 ? go_full_wave_t<P, Q, float, true, float2>(s, io, tw, st)
                                       : go_full_wave_t<P, Q, __half, true, float2>(s, io, tw, st);
    }
    // (the planner's complex forward stages read FP32 intermediates)
    if ( io.src_ct != CpxT::c64 )
        return hipErrorNotSupported;
    return io.dst_ct == CpxT::c64 ? go_full_wave_t<P, Q, float2, false, float2>(s, io, tw, st)
                                  : go_full_wave_t<P, Q, float2, false, __half2>(s, io, tw, st);
}

// Real rows of 1024 .. 8192 points into a transposed spectrum, two rows as one complex
// line (pair_rows.hpp), PPW pairs per workgroup.
template <int N, int PPW, typename TIn, bool PAD>
static hipError_t go_pair_rows_t(const Stage& s, const StageIO& io, const float2* tw, hipStream_t st) {
    const dim3 grid((unsigned)(((s.nlines + 1) / 2 + PPW - 1) / PPW)), block(N / kPairE * PPW);
    launch_kernel<k_r2c_pair_rows<N, PPW, TIn, PAD>>(grid, block, 0, st, static_cast<const TIn*>(io.src), to_device(s.im), s.L,
            static_cast<float2*>(io.dst), to_device(s.om), s.nout, s.nlines, io.scale, tw);
    return hipGetLastError( );
}

template <int N, int PPW>
static hipError_t go_pair_rows(const Stage& s, const StageIO& io, const float2* tw, hipStream_t st) {
    if ( io.src_rt == RealT::f32 )
        return s.L < s.N ? go_pair_rows_t<N, PPW, float, true>(s, io, tw, st) : go_pair_rows_t<N, PPW, float, false>(s, io, tw, st);
    return s.L < s.N ? go_pair_rows_t<N, PPW, __half, true>(s, io, tw, st) : go_pair_rows_t<N, PPW, __half, false>(s, io, tw, st);
}

static hipError_t try_pair_rows(const Stage& s, const StageIO& io, const float2* tw, hipStream_t st) {
    if ( s.N < 1024 || s.kind != StageKind::fwd_real || ! io.src_real || io.dst_real || io.dst_ct != CpxT::c64 || s.nlines < 1 ||
         s.L > s.N || s.nout < 1 || s.nout > s.N / 2 + 1 || s.im.n2 != 1 || s.im.es != 1 || s.om.n2 != 1 || s.om.s1 != 1 ||
         s.om.es % 2 != 0 || s.om.es < s.nlines ||
         reinterpret_cast<std::uintptr_t>(io.dst) % 16 != 0 || env_int("FASTFFT_NO_PAIR_LINES", 0) )
        return hipErrorNotSupported;
    return pair_rows_dispatch(s.N, s.nlines, kPairMinForward, [&](auto nc, auto gc) {
        return go_pair_rows<decltype(nc)::value, decltype(gc)::value>(s, io, tw, st);
    });
}

static hipError_t try_full_wave(const Stage& s, const StageIO& io, const float2* tw, hipStream_t st) {
    if ( s.L > s.N || io.dst_real || s.nout > s.N )
        return hipErrorNotSupported;
    switch ( s.N ) {
        case 256: return go_full_wave<256, 1>(s, io, tw, st);
        case 512: return go_full_wave<512, 1>(s, io, tw, st);
        case 1024: return go_full_wave<512, 2>(s, io, tw, st);
        case 2048: return go_full_wave<512, 4>(s, io, tw, st);
        case 4096: return go_full_wave<512, 8>(s, io, tw, st);
        case 8192: return go_full_wave<512, 16>(s, io, tw, st);
        default: return hipErrorNotSupported;
    }
}

hipError_t launch_fwd(const Stage& s, const StageIO& io, const float2* tw, hipStream_t st) {
    // a unit-stride output row is written two values at a time: even line offsets, aligned base
    const std::uintptr_t pair_bytes = io.dst_ct == CpxT::c64 ? 16 : 8;
    const bool           rows_ok    = s.om.es != 1 || (s.om.s1 % 2 == 0 && s.om.s2 % 2 == 0 &&
                                          reinterpret_cast<std::uintptr_t>(io.dst) % pair_bytes == 0);
    const bool           full_lines = rows_ok && ! env_int("FASTFFT_NO_WAVE_ROWS", 0) && ! env_int("FASTFFT_NO_FULL_LINES", 0);
    // real rows of 1024 points and up into a transposed spectrum (1024^2: 14.6 us with the
    // one-wave packed rows, 13.3-13.8 here; 384^2 templates' row-major rows do not come here)
    if ( full_lines ) {
        hipError_t e = try_pair_rows(s, io, tw, st);
        if ( e != hipErrorNotSupported )
            return e;
    }
    // lines of 64 to 512 points: C2C passes, and real rows into a transposed spectrum
    if ( (s.kind == StageKind::fwd_cpx || (s.kind == StageKind::fwd_real && s.om.es != 1)) &&
         ! env_int("FASTFFT_NO_WAVE_ROWS", 0) ) {
        hipError_t e = launch_lines(s, io, tw, st);
        if ( e != hipErrorNotSupported )
            return e;
    }
    if ( io.src_real && ! io.dst_real && io.dst_ct == CpxT::c64 && ! env_int("FASTFFT_NO_WAVE_ROWS", 0) ) {
        hipError_t e = launch_r2c_packed(s, io.src, io.dst, io.src_rt, s.nlines, io.scale, tw, nullptr, 1, st);
        if ( e != hipErrorNotSupported )
            return e;
    }
    if ( full_lines && s.L == s.N ) {
        hipError_t e = try_full_wave(s, io, tw, st);
        if ( e != hipErrorNotSupported )
            return e;
    }
    // padded lines left: unit-stride complex lines, and real rows that no sub-transform kernel takes
    if ( full_lines && s.L < s.N && (io.src_real ? ! r2c_rows_shape(r2c_at_least_256(s)) : s.im.es == 1 && s.om.es == 1) ) {
        hipError_t e = try_full_wave(s, io, tw, st);
        if ( e != hipErrorNotSupported )
            return e;
    }
    if ( io.src_real && ! io.dst_real && io.dst_ct == CpxT::c64 && rows_ok && ! env_int("FASTFFT_NO_WAVE_ROWS", 0) ) {
        const Stage r = r2c_at_least_256(s);
        hipError_t  e = io.src_rt == RealT::f32 ? try_r2c_wave<float>(r, io, tw, st) : try_r2c_wave<__half>(r, io, tw, st);
        if ( e != hipErrorNotSupported )
            return e;
    }
    return dispatch_P(s.P, [&](auto pc) -> hipError_t {
        constexpr int P = decltype(pc)::value;
        if ( io.src_real ) {
            if ( io.dst_real || io.dst_ct != CpxT::c64 )
                return hipErrorInvalidValue;
            if ( io.src_rt == RealT::f32 )
                return go_fwd<P, float, true, float2>(s, io, tw, st);
            return go_fwd<P, __half, true, float2>(s, io, tw, st);
        }
        if ( io.src_ct != CpxT::c64 || io.dst_real )
            return hipErrorInvalidValue;
        if ( io.dst_ct == CpxT::c64 )
            return go_fwd<P, float2, false, float2>(s, io, tw, st);
        return go_fwd<P, float2, false, __half2>(s, io, tw, st);
    });
}

size_t stage_lds_bytes(int P) {
    size_t out = 0;
    (void)dispatch_P(P, [&](auto pc) -> hipError_t {
        out = sizeof(float2) * (size_t)LineShape<decltype(pc)::value>::LDS;
        return hipSuccess;
    });
    return out;
}

} // namespace fastfft_amd
