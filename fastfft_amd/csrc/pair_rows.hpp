// Real rows of N = 1024 .. 8192 points against a transposed spectrum, two rows as one
// complex line: the R2C x-pass of a FwdFFT (any non-zero length L <= N) and the C2R
// x-pass of an InvFFT (any window), the reference's block_fft_kernel_R2C_NONE_XY,
// R2C_INCREASE_XY, C2R_NONE_XY and C2R_DECREASE_XY (src/fastfft/FastFFT.cu:1055-1166,
// :1641-1692), which transform one real row as a complex line each.
//
//   z = a + i b,  Z = FFT_N(z):  A[k] = (Z[k] + conj Z[N-k]) / 2,  B[k] = -i (Z[k] - conj Z[N-k]) / 2
//   Z[k] = A[k] + i B[k],  Z[N-k] = conj A[k] + i conj B[k]:       z = IFFT_N(Z), a = Re z, b = Im z
//
// The spectrum is stored A[kx][y]: the 2 PPW rows of a workgroup are one 16 PPW-byte
// segment of every kx, moved 16 bytes per lane; the rows themselves are unit stride.
// 16 values per thread in registers (T = N / 16 threads per pair), loaded and stored
// directly, and radix-16 Stockham passes.  The exchanges of a workgroup of 1024 threads move the
// real and then the imaginary parts through one LDS buffer of N floats per pair.  That halves
// the LDS of a pair, and immediate offsets keep the addresses out of the registers (64 at most),
// so two such workgroups share a CU and one loads or stores while the other computes.
// Bound by arithmetic and memory about alike: 4096^2 (134 MB) takes 29.9 us forward and
// 29.7 us inverse, 4.5 TB/s, where complex exchanges with one workgroup per CU took
// 38.6 us forward and one row per workgroup with 8-byte gathers 51.7 us inverse.
#pragma once

#include <type_traits>

#include "rows_wave.hpp"

namespace fastfft_amd {

constexpr int kPairE = 16; // values per thread

// Workgroups of at most 512 threads (8192 points) move whole complex values through LDS: two of
// them still fit a CU, and half the barriers matter where a launch has few workgroups per CU.
// 2-D transforms: 2048^2 forward 27.3 -> 26.4 us, inverse 27.0 -> 26.2; 512 rows of 4096 points
// 17.5 -> 16.9 and 17.5 -> 17.0; 512 rows of 8192 points 30.1 -> 28.6.
template <int N, int PPW>
constexpr bool pair_whole = N * PPW <= 8192;
template <int N, int PPW>
using PairWord = std::conditional_t<pair_whole<N, PPW>, float2, float>;

// Calls f(part) for every exchange of a pair: the real and the imaginary parts in turn, or whole values.
template <bool WHOLE, class F>
__device__ __forceinline__ void for_parts(F&& f) {
    if constexpr ( ! WHOLE ) {
        f([](auto& z) -> auto& { return z.x; });
        f([](auto& z) -> auto& { return z.y; });
    }
    else {
        f([](auto& z) -> auto& { return z; });
    }
}

// Exchange slot of element k: one pad word per 16, so that the scatters of the radix-16
// passes (lane strides 16 and 256) and the unit-stride gathers fall on distinct banks.
// Slots 16 m elements apart lie 17 m words apart: one address and immediate offsets.
__device__ __forceinline__ int pair_slot(int k) { return k + (k >> 4); }
constexpr int                  pair_step(int k) { return k + k / 16; }
// Floats per pair (slot N, a copy of element 0 beside the mirrored element N - k, included):
// PPW consecutive pairs start 64 / PPW banks apart, so that the lanes of
// the segment accesses (PPW pairs, 64 / PPW consecutive k) fall on distinct banks as well.
template <int N, int PPW>
constexpr int pair_pitch = N + N / 16 + (pair_whole<N, PPW> ? 32 : 64) / PPW;

// A pair of one wave needs no workgroup barrier in its own exchanges.
template <int T>
__device__ __forceinline__ void pair_sync( ) {
    if constexpr ( T == 64 )
        wave_lds_fence( );
    else
        __syncthreads( );
}

// The second pass's twiddles W_256^{j r}, [r - 1][j], copied into LDS once per workgroup of NT
// threads (read from memory at their use instead, 4096^2 takes 59.0 us forward and 33.9 us cut
// to 1001 x 900, here 57.2 and 32.4): load() issues the thread's loads, store() writes them.
constexpr int kPairTable = 15 * 16;
template <int NT>
struct PairTable {
    static constexpr int ROWS = (kPairTable + NT - 1) / NT;
    bits_t<float2>       w[ROWS]; // (bits: as float2 the compiler waits for the load before it issues the rows')
    __device__ __forceinline__ void load(const float2* __restrict__ twm) {
#pragma unroll
        for ( int r = 0; r < ROWS; r++ ) {
            const int g = threadIdx.x + NT * r;
            if ( g < kPairTable )
                w[r] = load_bits(as_global(twm) + 256 + (g & 15) * (1 + (g >> 4)));
        }
    }
    __device__ __forceinline__ void store(float2* tab) const {
#pragma unroll
        for ( int r = 0; r < ROWS; r++ ) {
            const int g = threadIdx.x + NT * r;
            if ( g < kPairTable )
                tab[g] = bits_value(w[r]);
        }
    }
};

// Twiddles W_{Ns R}^{j r} of one thread's butterflies in the later passes, where a load's 64
// addresses spread over 4 r cache lines: r = 4 a + b kept as the factors of 4 a and b (six
// values for R = 16) and multiplied in one after the other.  (A table with every r's twiddles
// contiguous in j measured 2-3 % slower, with the same errors against 64 bits.)
template <int R, int B>
struct PairTwiddles {
    static constexpr int NB = R < 4 ? R : 4, NA = R / NB;
    float2               lo[B][NB > 1 ? NB - 1 : 1], hi[B][NA > 1 ? NA - 1 : 1];

    template <int Ns, int T>
    __device__ __forceinline__ void load(int t, const float2* __restrict__ twm) {
        const auto* tab = as_global(twm) + Ns * R;
#pragma unroll
        for ( int m = 0; m < B; m++ ) {
            const int j = (t + T * m) & (Ns - 1);
#pragma unroll
            for ( int b = 1; b < NB; b++ )
                lo[m][b - 1] = load_cpx(at_bytes(tab, 8u * (unsigned)(j * b)), 0);
#pragma unroll
            for ( int a = 1; a < NA; a++ )
                hi[m][a - 1] = load_cpx(at_bytes(tab, 8u * (unsigned)(j * NB * a)), 0);
        }
    }

    template <int DIR>
    __device__ __forceinline__ void apply(float2 (&u)[R], int m) const {
#pragma unroll
        for ( int r = 1; r < R; r++ ) {
            const int a = r / NB, b = r % NB;
            if ( a )
                u[r] = DIR < 0 ? cmul(u[r], hi[m][a - 1]) : cmulc(u[r], hi[m][a - 1]);
            if ( b )
                u[r] = DIR < 0 ? cmul(u[r], lo[m][b - 1]) : cmulc(u[r], lo[m][b - 1]);
        }
    }
};

// Stockham passes from stride Ns on: register i of thread t holds element t + T i on entry
// and on return (natural order).  buf: the pair's exchange buffer of N words.
template <int N, int PPW, int Ns, int DIR>
__device__ __forceinline__ void pair_passes(float2 (&v)[kPairE], PairWord<N, PPW>* __restrict__ buf, int t,
                                            const float2* tab, const float2* __restrict__ twm) {
    constexpr int  T = N / kPairE, R = N / Ns < kPairE ? N / Ns : kPairE, B = kPairE / R;
    constexpr bool LAST = Ns * R == N;
    PairTwiddles<R, B> w;
    if constexpr ( Ns > 16 )
        w.template load<Ns, T>(t, twm);
#pragma unroll
    for ( int m = 0; m < B; m++ ) {
        float2 u[R];
#pragma unroll
        for ( int r = 0; r < R; r++ )
            u[r] = v[m + B * r];
        if constexpr ( Ns == 16 ) {
#pragma unroll
            for ( int r = 1; r < R; r++ ) {
                const float2 w2 = tab[(r - 1) * 16 + (t & 15)];
                u[r]            = DIR < 0 ? cmul(u[r], w2) : cmulc(u[r], w2);
            }
        }
        else if constexpr ( Ns > 16 )
            w.template apply<DIR>(u, m);
        SmallDFT<R, DIR>::run(u);
#pragma unroll
        for ( int r = 0; r < R; r++ )
            v[m + B * r] = u[r];
    }
    if constexpr ( ! LAST ) {
        for_parts<pair_whole<N, PPW>>([&](auto part) {
            pair_sync<T>( ); // the buffer's readers are done
#pragma unroll
            for ( int m = 0; m < B; m++ ) {
                const int b = t + T * m, j = b & (Ns - 1);
                auto*     dst = buf + pair_slot((b - j) * R + j); // element (b - j) R + j + r Ns for r < R
#pragma unroll
                for ( int r = 0; r < R; r++ )
                    dst[Ns == 1 ? r : r * pair_step(Ns)] = part(v[m + B * r]);
            }
            pair_sync<T>( );
#pragma unroll
            for ( int i = 0; i < kPairE; i++ )
                part(v[i]) = buf[pair_slot(t) + i * pair_step(T)];
        });
        pair_passes<N, PPW, Ns * R, DIR>(v, buf, t, tab, twm);
    }
}

// R2C: rows 0 .. nlines - 1 of L real values (im.es = 1) into out[k om.es + row], k < nout
// <= N/2 + 1; om.s1 = 1, om.es even, out 16-byte aligned, and om.es leaves room for an even
// row count.  Grid: ceil(ceil(nlines / 2) / PPW) workgroups of T PPW threads.
// PAD: L < N.  Whole rows load without a branch per value, which matters where a CU has few
// workgroups to hide a wait: 2048 x 256 forward 10.2 -> 9.8 us, 2048 x 1024 16.9 -> 16.4.
template <int N, int PPW, typename TIn, bool PAD>
__global__ void __launch_bounds__(N / kPairE * PPW, N / kPairE * PPW == 1024 ? 8 : 4)
        k_r2c_pair_rows(const TIn* __restrict__ in, LineMap im, int L, float2* __restrict__ out, LineMap om, int nout,
                        int nlines, float pre_scale, const float2* __restrict__ tw) {
    constexpr int T = N / kPairE, NT = T * PPW, H = N / 2, ITER = H / T + 1;
    __shared__ PairWord<N, PPW> s_x[PPW * pair_pitch<N, PPW>];
    __shared__ float2           s_tw[kPairTable];
    PairTable<NT>               table;
    table.load(multi_twiddles(tw));
    const int     h     = PPW > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x / T) : 0;
    const int     t     = threadIdx.x % T;
    // single pairs' 16-byte segments meet in one L2; wider ones store as fast from any XCD, and some counts faster (2731
    // rows of 2048 points in groups of four 27.0 us, 28.1 in ranges)
    const int     pair0 = (PPW == 1 ? xcd_range(blockIdx.x, gridDim.x) : xcd_row(blockIdx.x, gridDim.x)) * PPW;
    const int     row   = 2 * (pair0 + h);
    auto*         buf   = s_x + h * pair_pitch<N, PPW>;
    float2        v[kPairE];
    {
        const bool  hb = row + 1 < nlines;
        const auto* la = as_global(in) + im.base(row < nlines ? row : 0); // (a row past the last one: any row, not stored)
        const auto* lb = as_global(in) + im.base(hb ? row + 1 : 0);
        // every load of the thread in flight before the first value is used
        bits_t<TIn> a[kPairE], b[kPairE];
#pragma unroll
        for ( int i = 0; i < kPairE; i++ ) {
            const int n = t + T * i;
            if constexpr ( PAD ) {
                a[i] = b[i] = bits_t<TIn>{ };
                if ( n < L ) {
                    a[i] = load_bits(at_bytes(la, (unsigned)sizeof(TIn) * (unsigned)n));
                    b[i] = load_bits(at_bytes(lb, (unsigned)sizeof(TIn) * (unsigned)n));
                }
            }
            else {
                a[i] = load_bits(at_bytes(la, (unsigned)sizeof(TIn) * (unsigned)n));
                b[i] = load_bits(at_bytes(lb, (unsigned)sizeof(TIn) * (unsigned)n));
            }
        }
#pragma unroll
        for ( int i = 0; i < kPairE; i++ )
            v[i] = make_float2(bits_value(a[i]) * pre_scale, hb ? bits_value(b[i]) * pre_scale : 0.f);
    }
    table.store(s_tw);
    __syncthreads( );
    pair_passes<N, PPW, 1, -1>(v, buf, t, s_tw, multi_twiddles(tw));
    // Z in natural order through LDS: item (k, g) takes A[k] and B[k] of the workgroup's pair g,
    // 16 bytes of the segment of k
    const int   g  = threadIdx.x % PPW, k0 = threadIdx.x / PPW; // k = k0 + T c
    const auto *zk = s_x + g * pair_pitch<N, PPW> + pair_slot(k0), *zn = s_x + g * pair_pitch<N, PPW> + pair_slot(N - k0);
    auto*       op = as_global(out) + 2 * pair0;
    const bool  rows = 2 * (pair0 + g) < nlines;
    auto        spread = [&](auto part) {
        __syncthreads( );
#pragma unroll
        for ( int i = 0; i < kPairE; i++ )
            buf[pair_slot(t) + i * pair_step(T)] = part(v[i]);
        if ( t == 0 )
            buf[pair_step(N)] = part(v[0]);
        __syncthreads( );
    };
    // a = (Re A[k], Im A[k]) and b of item c
    auto store = [&](int c, float2 a, float2 b) {
        const int k = k0 + T * c;
        if ( k < nout && rows && (c + 1 < ITER || k0 == 0) )
            store_cpx_pair(at_bytes(op, 8u * (unsigned)k * (unsigned)om.es + 16u * (unsigned)g), 0, a, b);
    };
    if constexpr ( ! pair_whole<N, PPW> ) { // real parts first
        float ax[ITER], by[ITER];
        spread([](float2 z) { return z.x; });
#pragma unroll
        for ( int c = 0; c < ITER; c++ )
            if ( c + 1 < ITER || k0 == 0 ) {
                ax[c] = 0.5f * (zk[c * pair_step(T)] + zn[-c * pair_step(T)]);
                by[c] = 0.5f * (zn[-c * pair_step(T)] - zk[c * pair_step(T)]);
            }
        spread([](float2 z) { return z.y; });
#pragma unroll
        for ( int c = 0; c < ITER; c++ )
            if ( c + 1 < ITER || k0 == 0 ) {
                const float yk = zk[c * pair_step(T)], yn = zn[-c * pair_step(T)];
                store(c, make_float2(ax[c], 0.5f * (yk - yn)), make_float2(0.5f * (yk + yn), by[c]));
            }
    }
    else {
        spread([](float2 z) { return z; });
#pragma unroll
        for ( int c = 0; c < ITER; c++ )
            if ( c + 1 < ITER || k0 == 0 ) {
                const float2 a = zk[c * pair_step(T)], b = zn[-c * pair_step(T)];
                store(c, make_float2(0.5f * (a.x + b.x), 0.5f * (a.y - b.y)), make_float2(0.5f * (a.y + b.y), 0.5f * (b.x - a.x)));
            }
    }
}

// C2R: in[k im.es + row], k <= N/2 (im.s1 = 1, im.es even, in 16-byte aligned), to the
// window y[(o + j) mod N], j < M, of every row (om.es = 1).  The imaginary parts of
// k = 0 and N/2 are dropped, as the real part of the Hermitian extension's inverse drops
// them.  Grid as above.
template <int N, int PPW, typename TOut>
__global__ void __launch_bounds__(N / kPairE * PPW, N / kPairE * PPW == 1024 ? 8 : 4)
        k_c2r_pair_rows(const float2* __restrict__ in, LineMap im, TOut* __restrict__ out, LineMap om, int M, int o,
                        int nlines, float post_scale, const float2* __restrict__ tw) {
    constexpr int T = N / kPairE, NT = T * PPW, H = N / 2, ITER = H / T + 1;
    __shared__ PairWord<N, PPW> s_x[PPW * pair_pitch<N, PPW>];
    __shared__ float2           s_tw[kPairTable];
    PairTable<NT>               table;
    table.load(multi_twiddles(tw));
    const int     h     = PPW > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x / T) : 0;
    const int     t     = threadIdx.x % T;
    const int     pair0 = xcd_range(blockIdx.x, gridDim.x) * PPW, row = 2 * (pair0 + h);
    auto*         buf   = s_x + h * pair_pitch<N, PPW>;
    float2        v[kPairE];
    {
        const auto* ip   = as_global(in) + 2 * pair0;
        const int   g    = threadIdx.x % PPW, k0 = threadIdx.x / PPW; // k = k0 + T c
        const bool  ha   = 2 * (pair0 + g) < nlines, hb = 2 * (pair0 + g) + 1 < nlines;
        float4      u[ITER];
#pragma unroll
        for ( int c = 0; c < ITER; c++ ) {
            const int k = k0 + T * c;
            u[c]        = make_float4(0.f, 0.f, 0.f, 0.f);
            if ( ha && (c + 1 < ITER || k0 == 0) )
                u[c] = load_cpx_pair(at_bytes(ip, 8u * (unsigned)k * (unsigned)im.es + 16u * (unsigned)g), 0);
        }
#pragma unroll
        for ( int c = 0; c < ITER; c++ ) {
            if ( ! hb ) // past the last row: whatever the buffer holds
                u[c].z = u[c].w = 0.f;
            if ( (c == 0 || c + 1 == ITER) && k0 == 0 )
                u[c].y = u[c].w = 0.f;
        }
        auto *zk = s_x + g * pair_pitch<N, PPW> + pair_slot(k0), *zn = s_x + g * pair_pitch<N, PPW> + pair_slot(N - k0);
        table.store(s_tw);
        auto   spread = [&](auto lo, auto hi) {
#pragma unroll
            for ( int c = 0; c < ITER; c++ )
                if ( c + 1 < ITER || k0 == 0 ) { // (element N / 2 is its own mirror, and lo = hi there)
                    zk[c * pair_step(T)]  = lo(u[c]);
                    zn[-c * pair_step(T)] = hi(u[c]);
                }
            __syncthreads( );
        };
        auto gather = [&](auto part) {
#pragma unroll
            for ( int i = 0; i < kPairE; i++ )
                part(v[i]) = buf[pair_slot(t) + i * pair_step(T)];
        };
        if constexpr ( ! pair_whole<N, PPW> ) {
            spread([](float4 z) { return z.x - z.w; }, [](float4 z) { return z.x + z.w; });
            gather([](float2& z) -> float& { return z.x; });
            __syncthreads( );
            spread([](float4 z) { return z.z + z.y; }, [](float4 z) { return z.z - z.y; });
            gather([](float2& z) -> float& { return z.y; });
        }
        else {
            spread([](float4 z) { return make_float2(z.x - z.w, z.z + z.y); },
                   [](float4 z) { return make_float2(z.x + z.w, z.z - z.y); });
            gather([](float2& z) -> float2& { return z; });
        }
    }
    __syncthreads( ); // (the first exchange of a one-wave pair orders its own wave only)
    pair_passes<N, PPW, 1, +1>(v, buf, t, s_tw, multi_twiddles(tw));
    if ( row >= nlines )
        return;
    const bool hb = row + 1 < nlines;
    auto*      oa = as_global(out) + om.base(row);
    auto*      ob = as_global(out) + om.base(hb ? row + 1 : row);
#pragma unroll
    for ( int i = 0; i < kPairE; i++ ) {
        const int j = (t + T * i - o) & (N - 1);
        if ( j < M ) {
            store_real(at_bytes(oa, (unsigned)sizeof(TOut) * (unsigned)j), 0, v[i].x * post_scale);
            if ( hb )
                store_real(at_bytes(ob, (unsigned)sizeof(TOut) * (unsigned)j), 0, v[i].y * post_scale);
        }
    }
}

} // namespace fastfft_amd
