// Line transforms of N = 64 .. 512 points: the passes of the 3-D transforms (the
// reference's strided 3-D kernels, block_fft_kernel_C2C_INCREASE / C2C_NONE_XYZ /
// C2C_DECREASE / C2R_DECREASE with the XZ/XYZ permutes, src/fastfft/FastFFT.cu and
// include/detail/memory_addressing.h:25-104) and the 256- and 512-point passes of the
// 2-D ones.
//
// T = N / E threads per line, E = 16 or 8 values per thread (line_values; thread t holds
// elements t + T i), radix-E Stockham passes: at most two LDS exchanges.
//   IN_X / OUT_X: the lines lie next to each other and their elements far apart (a
//     z-pass, the transposed side of an x-pass): consecutive lanes take consecutive
//     lines, so that the 16 lines of a workgroup are one 128-byte segment per element,
//     loaded into and stored from registers without passing through LDS;
//   else the lanes run along the line (unit stride).
// The first exchange also turns the one arrangement into the other.
//   HERM:     rows holding X[0 .. N/2] of a Hermitian sequence, real outputs (C2R): two
//             rows A, B as one complex line Z[k] = A[k] + i B[k], Z[N-k] = conj A[k] +
//             i conj B[k], whose inverse is a + i b.  The imaginary parts of k = 0 and
//             N/2 are dropped, as the real part of the Hermitian extension's inverse
//             drops them.
//   forward (DIR = -1): X[k] = sum_{n < L} x[n] W_N^{n k}, k < M (window origin 0)
//   inverse (DIR = +1): y[j] = sum_k X[k] W_N^{-k (o + j)}, j < M
#pragma once

#include <type_traits>

#include "rows_wave.hpp"

namespace fastfft_amd {

// Values per thread: 8, and 16 for real rows of 256 points (5,084 of them 6.9 us with 16, 8.7 with 8).
// Twice the threads of a line outweigh the exchange that 16 values save at 64, 128 and 256 points (128^2
// forward 8.2 us with 16, 6.6 with 8, inverse 9.2 and 7.0; fused z-pass of 256^3 35.3 and 30.4, its C2R rows 9.6
// and 8.6), and at 512 points 16 values need as many exchanges (512^3 cut to 128^3: 143 + 48 us and 118 + 42).
constexpr int line_values(int N, bool real_in) { return N == 256 && real_in ? 16 : 8; }
template <typename T>
constexpr bool is_real_element = std::is_same<T, float>::value || std::is_same<T, __half>::value;
constexpr int kTileLines = 16; // transforms of a workgroup whose lanes run across lines

// LDS slot of element k of a line: one pad slot per E values, and 2 more per line, so that the
// scatters and gathers of both arrangements are free of bank conflicts but for single lanes.
template <int E>
__device__ __forceinline__ int line_slot(int k) {
    return k + k / E;
}
template <int E>
constexpr int line_step(int k) { return k + k / E; }
template <int N, int E>
constexpr int line_pitch = N + N / E + 2;

// The Stockham twiddles of the passes after the first, pass by pass, [r - 1][j] within a pass
// of stride Ns and radix R: W_{Ns R}^{j r}.  Copied into LDS once per workgroup: read from
// memory, one load per value per thread, they took as long as the data (512-point lines of
// a 512^3 inverse: 147 us against 124).
template <int N, int E>
constexpr int line_table_size( ) {
    int n = 0;
    for ( int ns = E; ns < N; ns *= E )
        n += ns * ((N / ns < E ? N / ns : E) - 1);
    return n;
}

// Index of table entry g in the multi-resolution twiddle table.
template <int N, int E, int Ns = E>
__device__ __forceinline__ int line_table_index(int g) {
    constexpr int R = N / Ns < E ? N / Ns : E, SZ = Ns * (R - 1);
    if constexpr ( Ns * R < N ) {
        if ( g >= SZ )
            return line_table_index<N, E, Ns * R>(g - SZ);
    }
    return Ns * R + (g & (Ns - 1)) * (1 + g / Ns);
}

// Fills the table with NT threads: load() issues the thread's loads, store() writes them.
template <int N, int E, int NT>
struct LineTable {
    static constexpr int SIZE = line_table_size<N, E>( ), ROWS = (SIZE + NT - 1) / NT;
    bits_t<float2>       w[ROWS];
    __device__ __forceinline__ void load(const float2* __restrict__ twm) {
#pragma unroll
        for ( int r = 0; r < ROWS; r++ ) {
            const int g = threadIdx.x + NT * r;
            if ( g < SIZE )
                w[r] = load_bits(as_global(twm) + line_table_index<N, E>(g));
        }
    }
    __device__ __forceinline__ void store(float2* tab) const {
#pragma unroll
        for ( int r = 0; r < ROWS; r++ ) {
            const int g = threadIdx.x + NT * r;
            if ( g < SIZE )
                tab[g] = bits_value(w[r]);
        }
    }
};

// Orders the exchange of a workgroup whose lines span waves; a line within one wave needs
// no barrier.
template <bool WG>
__device__ __forceinline__ void line_sync( ) {
    if constexpr ( WG )
        __syncthreads( );
    else
        wave_lds_fence( );
}

// Stockham passes from stride Ns on.  A thread holds elements tw + T i of the line at bw on
// entry; from the first exchange on those tr + T i of the line at br.  tab: the twiddles of
// the pass (of the next one for Ns = 1).  FIRST: the first exchange also orders the table.
template <int N, int E, int Ns, int DIR, bool WG, bool FIRST>
__device__ __forceinline__ void line_passes(float2 (&v)[E], float2* bw, int tw, float2* br, int tr,
                                            const float2* tab) {
    constexpr int  T = N / E, R = N / Ns < E ? N / Ns : E, B = E / R;
    constexpr bool LAST = Ns * R == N;
#pragma unroll
    for ( int m = 0; m < B; m++ ) {
        const int j = (tw + T * m) & (Ns - 1);
        float2    u[R];
#pragma unroll
        for ( int r = 0; r < R; r++ )
            u[r] = v[m + B * r];
        if constexpr ( Ns > 1 ) {
#pragma unroll
            for ( int r = 1; r < R; r++ ) {
                const float2 w = tab[(r - 1) * Ns + j];
                u[r]           = DIR < 0 ? cmul(u[r], w) : cmulc(u[r], w);
            }
        }
        SmallDFT<R, DIR>::run(u);
#pragma unroll
        for ( int r = 0; r < R; r++ )
            v[m + B * r] = u[r];
    }
    if constexpr ( ! LAST ) {
        if constexpr ( Ns > 1 )
            line_sync<WG>( ); // the previous exchange's readers are done
#pragma unroll
        for ( int m = 0; m < B; m++ ) {
            const int b = tw + T * m, j = b & (Ns - 1);
            float2*   dst = bw + line_slot<E>((b - j) * R + j); // element (b - j) R + j + r Ns for r < R
#pragma unroll
            for ( int r = 0; r < R; r++ )
                dst[Ns == 1 ? r : r * line_step<E>(Ns)] = v[m + B * r];
        }
        line_sync<WG || FIRST>( );
#pragma unroll
        for ( int i = 0; i < E; i++ ) {
            if constexpr ( T % E == 0 )
                v[i] = br[line_slot<E>(tr) + i * line_step<E>(T)];
            else
                v[i] = br[line_slot<E>(tr + T * i)];
        }
        line_passes<N, E, Ns * R, DIR, WG, false>(v, br, tr, br, tr, tab + (Ns > 1 ? Ns * (R - 1) : 0));
    }
}

// The lines of one workgroup: `per` lines of each group of a two-index map (all lines of a
// single-index one) are cut into tiles of LT, the last one partly filled.
struct LineTile {
    int line0, count; // first line, lines that exist
    __device__ __forceinline__ LineTile(int tile, int per, int lt) {
        const int tpg = (per + lt - 1) / lt, g = tile / tpg, y0 = (tile - g * tpg) * lt;
        line0 = g * per + y0;
        count = min(lt, per - y0);
    }
};

// element-index step between neighbouring lines of a tile
__device__ __forceinline__ unsigned line_stride(const LineMap& m) { return (unsigned)(m.n2 > 1 ? m.s2 : m.s1); }

// Grid: groups x ceil(per / LT) workgroups of LT N / line_values threads
// (HERM: two rows per transform).  flags bit 0: workgroups in XCD-contiguous ranges.
template <int N, int LT, int DIR, typename TIn, bool HERM, typename TOut, bool IN_X, bool OUT_X>
__global__ void __launch_bounds__(LT* N / line_values(N, is_real_element<TIn>))
        k_lines(const TIn* __restrict__ in, LineMap im, int L, TOut* __restrict__ out, LineMap om, int M, int o, int nlines,
                float scale, const float2* __restrict__ tw, int flags) {
    constexpr int  E = line_values(N, is_real_element<TIn>), T = N / E, H = N / 2;
    constexpr bool WG       = (IN_X || OUT_X) && LT * T > 64;
    constexpr bool REAL_OUT = is_real_element<TOut>, REAL_IN = is_real_element<TIn>;
    static_assert(HERM == REAL_OUT, "real outputs come from Hermitian rows, two at a time");
    constexpr int     ROWS = HERM ? 2 : 1;
    __shared__ float2 s_x[LT * line_pitch<N, E>];
    __shared__ float2 s_tw[line_table_size<N, E>( )];
    LineTable<N, E, LT * T> table;
    table.load(multi_twiddles(tw));
    const LineTile    tile((flags & 1) ? xcd_row(blockIdx.x, gridDim.x) : (int)blockIdx.x, im.n2 > 1 ? im.n2 : nlines,
                           LT * ROWS);
    const int         li = IN_X ? threadIdx.x % LT : threadIdx.x / T, ti = IN_X ? threadIdx.x / LT : threadIdx.x % T;
    const int         lo = OUT_X ? threadIdx.x % LT : threadIdx.x / T, to = OUT_X ? threadIdx.x / LT : threadIdx.x % T;
    float2            v[E];
    {
        const auto*    ip = as_global(in) + im.base(tile.line0);
        const unsigned es = (unsigned)im.es, ls = line_stride(im), row = ROWS * li;
        const bool     ha = (int)row < tile.count;
        // every load of the thread in flight before the first value is used
        bits_t<TIn> a[E], b[HERM ? E : 1];
#pragma unroll
        for ( int i = 0; i < E; i++ ) {
            const int n = ti + T * i;
            a[i]        = bits_t<TIn>{ };
            if constexpr ( HERM ) {
                const unsigned at = (unsigned)(n <= H ? n : N - n) * es + row * ls;
                b[i]              = bits_t<TIn>{ };
                if ( ha )
                    a[i] = load_bits(at_bytes(ip, (unsigned)sizeof(TIn) * at));
                if ( (int)row + 1 < tile.count )
                    b[i] = load_bits(at_bytes(ip, (unsigned)sizeof(TIn) * (at + ls)));
            }
            else if ( ha && n < L ) {
                a[i] = load_bits(at_bytes(ip, (unsigned)sizeof(TIn) * ((unsigned)n * es + row * ls)));
            }
        }
#pragma unroll
        for ( int i = 0; i < E; i++ ) {
            if constexpr ( HERM ) {
                const int n  = ti + T * i;
                float2    za = bits_value(a[i]), zb = bits_value(b[i]);
                if ( n == 0 || n == H )
                    za.y = zb.y = 0.f;
                v[i] = n <= H ? make_float2(za.x - zb.y, za.y + zb.x) : make_float2(za.x + zb.y, zb.x - za.y);
            }
            else if constexpr ( REAL_IN ) {
                v[i] = make_float2(bits_value(a[i]), 0.f);
            }
            else {
                v[i] = bits_value(a[i]);
            }
        }
    }
    table.store(s_tw);
    line_passes<N, E, 1, DIR, WG, (LT * T > 64)>(v, s_x + li * line_pitch<N, E>, ti, s_x + lo * line_pitch<N, E>, to, s_tw);
    auto*          op = as_global(out) + om.base(tile.line0);
    const unsigned es = (unsigned)om.es, ls = line_stride(om), row = ROWS * lo;
    if ( (int)row >= tile.count )
        return;
#pragma unroll
    for ( int i = 0; i < E; i++ ) {
        // value n of the transform is output j = (n - o) mod N, kept when j < M
        const int j = (to + T * i - o) & (N - 1);
        if ( j < M ) {
            const unsigned at = (unsigned)j * es + row * ls;
            if constexpr ( REAL_OUT ) {
                store_real(at_bytes(op, (unsigned)sizeof(TOut) * at), 0, v[i].x * scale);
                if ( (int)row + 1 < tile.count )
                    store_real(at_bytes(op, (unsigned)sizeof(TOut) * (at + ls)), 0, v[i].y * scale);
            }
            else {
                store_cpx(at_bytes(op, (unsigned)sizeof(TOut) * at), 0, cscale(v[i], scale));
            }
        }
    }
}

// The fused z-pass of a 3-D FwdImageInvFFT (the reference's
// block_fft_kernel_C2C_FWD_INCREASE_OP_INV_NONE, src/fastfft/FastFFT.cu:20-56, on strided
// lines): forward of L template values, image x conj, inverse, M outputs from lag o.
// Template, image and output lines all lie next to each other.
template <int N, typename TImg>
__global__ void __launch_bounds__(kTileLines* N / line_values(N, false))
        k_lines_xcorr(const float2* __restrict__ a, LineMap am, int L, const TImg* __restrict__ img, LineMap gm,
                      float2* __restrict__ out, LineMap om, int M, int o, int nlines, float scale,
                      const float2* __restrict__ tw) {
    constexpr int     E = line_values(N, false), T = N / E, LT = kTileLines;
    constexpr bool    WG = LT * T > 64;
    __shared__ float2 s_x[LT * line_pitch<N, E>];
    __shared__ float2 s_tw[line_table_size<N, E>( )];
    LineTable<N, E, LT * T> table;
    table.load(multi_twiddles(tw));
    const LineTile    tile(blockIdx.x, nlines, LT);
    const int         l = threadIdx.x % LT, t = threadIdx.x / LT;
    const bool        mine = l < tile.count;
    float2*           buf  = s_x + l * line_pitch<N, E>;
    float2            v[E];
    const auto*       ap = as_global(a) + am.base(tile.line0);
#pragma unroll
    for ( int i = 0; i < E; i++ ) {
        const int n = t + T * i;
        v[i]        = make_float2(0.f, 0.f);
        if ( mine && n < L )
            v[i] = load_cpx(at_bytes(ap, 8u * ((unsigned)n * (unsigned)am.es + (unsigned)l)), 0);
    }
    table.store(s_tw);
    line_passes<N, E, 1, -1, WG, (LT * T > 64)>(v, buf, t, buf, t, s_tw);
    const auto* gp = as_global(img) + gm.base(tile.line0);
    bits_t<TImg> g[E];
#pragma unroll
    for ( int i = 0; i < E; i++ ) {
        g[i] = bits_t<TImg>{ };
        if ( mine )
            g[i] = load_bits(at_bytes(gp, (unsigned)sizeof(TImg) * ((unsigned)(t + T * i) * (unsigned)gm.es + (unsigned)l)));
    }
#pragma unroll
    for ( int i = 0; i < E; i++ )
        v[i] = cmulc(bits_value(g[i]), v[i]);
    line_sync<WG>( ); // the forward's last exchange is read before the inverse writes its first
    line_passes<N, E, 1, +1, WG, false>(v, buf, t, buf, t, s_tw);
    if ( ! mine )
        return;
    auto* op = as_global(out) + om.base(tile.line0);
#pragma unroll
    for ( int i = 0; i < E; i++ ) {
        const int j = (t + T * i - o) & (N - 1);
        if ( j < M )
            store_cpx(at_bytes(op, 8u * ((unsigned)j * (unsigned)om.es + (unsigned)l)), 0, cscale(v[i], scale));
    }
}

} // namespace fastfft_amd
