// Line transforms of 64 to 512 points (lines.hpp): the passes of the 3-D transforms and
// the 256- and 512-point passes of the 2-D ones.
#include <cstdint>

#include "launch_common.hpp"
#include "lines.hpp"

namespace fastfft_amd {

template <int N, int LT, int DIR, typename TIn, bool HERM, typename TOut, bool IX, bool OX>
static hipError_t go_lines_t(const Stage& s, const StageIO& io, const float2* tw, hipStream_t st, int M, int o, int per,
                             int tiles) {
    // bit 0: XCD-contiguous workgroups, measured faster where more rows are written than read (a
    // forward that pads) and slower for reading passes; FASTFFT_TILE_FLAGS overrides it
    const int flags = env_int("FASTFFT_TILE_FLAGS", (IX || OX) && DIR < 0 && M > s.L ? 1 : 0) & 1;
    launch_kernel<k_lines<N, LT, DIR, TIn, HERM, TOut, IX, OX>>(dim3((unsigned)(s.nlines / per * tiles)),
            dim3(LT * N / line_values(N, is_real_element<TIn>)), 0, st, static_cast<const TIn*>(io.src), to_device(s.im), DIR < 0 ? s.L : N,
            static_cast<TOut*>(io.dst), to_device(s.om), M, o, s.nlines, io.scale, tw, flags);
    return hipGetLastError( );
}

// Lines per workgroup: 16 (tiles), or 256 threads' worth of unit-stride lines, where that leaves at
// least FASTFFT_LINES_MIN workgroups, else a quarter.  128 workgroups, half the CUs.  Transforms in a
// graph, us with the large workgroups alone, with the small ones and by the rule: 64^2 padded to 512^2 8.1, 6.8
// and 6.8, 512^2 inverse 10.2, 8.2 and 8.1, 64^3 forward 9.4, 9.9 and 9.0, 64^3 padded to 256^3 31.6, 36.8 and
// 31.7, 512^3 cut to 128^3 171, 235 and 171.
template <int N, int DIR, typename TIn, bool HERM, typename TOut, bool IX, bool OX>
static hipError_t go_lines(const Stage& s, const StageIO& io, const float2* tw, hipStream_t st, int M, int o) {
    constexpr int ROWS = HERM ? 2 : 1, BIG = IX || OX ? kTileLines : 256 * line_values(N, is_real_element<TIn>) / N, SMALL = BIG / 4;
    const int     per = s.im.n2 > 1 ? s.im.n2 : s.nlines;
    auto          tiles = [&](int lt) { return (per + lt * ROWS - 1) / (lt * ROWS); };
    if ( s.nlines / per * tiles(BIG) >= env_int("FASTFFT_LINES_MIN", 128) )
        return go_lines_t<N, BIG, DIR, TIn, HERM, TOut, IX, OX>(s, io, tw, st, M, o, per, tiles(BIG));
    return go_lines_t<N, SMALL, DIR, TIn, HERM, TOut, IX, OX>(s, io, tw, st, M, o, per, tiles(SMALL));
}

// lines next to each other (unit stride between lines, inside one group of a two-index map)
// with far-apart elements
static bool across_map(const HostLineMap& m) {
    return (m.n2 == 1 ? m.s1 == 1 : m.s2 == 1) && m.es >= kTileLines;
}

static bool row_map(const HostLineMap& m) { return m.es == 1; }

// whole groups of lines, offsets of a workgroup's elements within 32 bits
static bool line_groups(const Stage& s, const HostLineMap& m) {
    const long step = m.n2 > 1 ? m.s2 : m.s1;
    return m.n2 == s.im.n2 && m.n2 >= 1 && (m.n2 == 1 || s.nlines % m.n2 == 0) && step >= 0 &&
           (long)s.N * m.es + 256 * step < (1L << 28);
}

// Few 256-point lines of a 2-D pass: the kernels of one wave per line (k_fwd_full_wave, k_inv_full_wave,
// k_inv_window_rows) fill more of the chip.  2-D transforms, us here and there: 256^2 forward 7.5 and 6.7, inverse 7.6
// and 6.9, cut to 61 x 59 7.1 and 6.4; 256 rows of 64 values in 256 x 1024 8.5 and 8.0.  Rows: a tie at 512 (256 x 512
// forward 7.9 and 7.9), behind at 682 (8.8 and 9.4, 191 values each in 256 x 1024).  Unit-stride complex lines, inverse:
// 513 of 1024 x 256 cut to 253 x 59 8.9 and 8.5, 1025 of 2048 x 256 9.8 and 9.6, 2049 of 4096 x 256 11.9 and 12.0;
// forward: 513 of 1024 x 256 8.5 and 9.0.
static bool few_lines(const Stage& s) {
    if ( s.N != 256 || s.im.n2 != 1 || s.om.n2 != 1 )
        return false;
    return s.kind == StageKind::inv_c2r || s.kind == StageKind::fwd_real ? s.nlines <= 256
                                                                         : s.im.es == 1 && s.om.es == 1 &&
                                                                                   s.nlines <= (s.kind == StageKind::fwd_cpx ? 300 : 1100);
}

bool lines_cover(const Stage& s) {
    if ( ! (s.N == 64 || s.N == 128 || s.N == 256 || s.N == 512) || s.nlines <= 0 || few_lines(s) || ! line_groups(s, s.im) ||
         ! line_groups(s, s.om) )
        return false;
    if ( s.kind == StageKind::inv_c2r )
        return across_map(s.im) && row_map(s.om);
    if ( s.kind == StageKind::fwd_real ) // real rows in, transposed spectrum rows out
        return row_map(s.im) && across_map(s.om) && s.nout <= s.N;
    if ( s.kind == StageKind::xcorr )
        return s.im.n2 == 1 && line_groups(s, s.gm) && across_map(s.im) && across_map(s.om) && across_map(s.gm) && s.L <= s.N &&
               s.M >= 1 && s.M <= s.N;
    return (across_map(s.im) && across_map(s.om)) || (row_map(s.im) && row_map(s.om));
}

hipError_t launch_lines(const Stage& s, const StageIO& io, const float2* tw, hipStream_t st) {
    if ( ! lines_cover(s) || env_int("FASTFFT_NO_TILE_LINES", 0) )
        return hipErrorNotSupported;
    const bool r2c = s.kind == StageKind::fwd_real;
    const bool fwd = s.kind == StageKind::fwd_cpx || r2c, c2r = s.kind == StageKind::inv_c2r;
    const int  M = fwd ? s.nout : s.M, o = fwd ? 0 : ((s.o % s.N) + s.N) % s.N;
    if ( M < 1 || M > s.N || io.src_real != r2c || io.dst_real != c2r )
        return hipErrorNotSupported;
    auto go = [&](auto nc) -> hipError_t {
        constexpr int N = decltype(nc)::value;
        if ( s.kind == StageKind::xcorr ) {
            auto xc = [&](auto img) {
                using TImg = decltype(img);
                launch_kernel<k_lines_xcorr<N, TImg>>(dim3((unsigned)((s.nlines + kTileLines - 1) / kTileLines)),
                        dim3(kTileLines * N / line_values(N, false)), 0, st, static_cast<const float2*>(io.src), to_device(s.im), s.L,
                        static_cast<const TImg*>(io.img), to_device(s.gm), static_cast<float2*>(io.dst), to_device(s.om),
                        s.M, o, s.nlines, io.scale, tw);
                return hipGetLastError( );
            };
            return io.img_ct == CpxT::c64 ? xc(float2{ }) : xc(__half2{ });
        }
        if ( r2c ) {
            if ( io.dst_ct != CpxT::c64 )
                return hipErrorNotSupported;
            return io.src_rt == RealT::f32 ? go_lines<N, -1, float, false, float2, false, true>(s, io, tw, st, M, o)
                                           : go_lines<N, -1, __half, false, float2, false, true>(s, io, tw, st, M, o);
        }
        if ( c2r ) {
            if ( io.src_ct != CpxT::c64 )
                return hipErrorNotSupported;
            return io.dst_rt == RealT::f32 ? go_lines<N, +1, float2, true, float, true, false>(s, io, tw, st, M, o)
                                           : go_lines<N, +1, float2, true, __half, true, false>(s, io, tw, st, M, o);
        }
        const bool across = across_map(s.im) && across_map(s.om);
        auto       types  = [&](auto ac) -> hipError_t {
            constexpr bool X = decltype(ac)::value;
            if ( fwd ) {
                if ( io.src_ct != CpxT::c64 )
                    return hipErrorNotSupported;
                return io.dst_ct == CpxT::c64 ? go_lines<N, -1, float2, false, float2, X, X>(s, io, tw, st, M, o)
                                              : go_lines<N, -1, float2, false, __half2, X, X>(s, io, tw, st, M, o);
            }
            if ( io.dst_ct != CpxT::c64 )
                return hipErrorNotSupported;
            return io.src_ct == CpxT::c64 ? go_lines<N, +1, float2, false, float2, X, X>(s, io, tw, st, M, o)
                                          : go_lines<N, +1, __half2, false, float2, X, X>(s, io, tw, st, M, o);
        };
        return across ? types(std::true_type{ }) : types(std::false_type{ });
    };
    switch ( s.N ) {
        case 64: return go(std::integral_constant<int, 64>{ });
        case 128: return go(std::integral_constant<int, 128>{ });
        case 256: return go(std::integral_constant<int, 256>{ });
        default: return go(std::integral_constant<int, 512>{ });
    }
}

} // namespace fastfft_amd
