// Forward line transforms of any non-zero length L <= N with one workgroup of Q
// wavefronts per line: the C2C y-pass of a FwdFFT, padded or not, and the R2C x-pass
// of rows too short for the pair kernel (the reference's block_fft_kernel_R2C_NONE_XY,
// R2C_INCREASE_XY, C2C_NONE and C2C_INCREASE, src/fastfft/FastFFT.cu:1055-1166,
// :1348-1367).
//
// N = P*Q is split decimation-in-frequency style:
//   y_q[m]      = sum_s x[s P + m] W_Q^{s q}          (radix-Q pass over the line in LDS)
//   X[Q k' + q] = FFT_P( y_q[m] W_N^{m q} )[k']         (wave q, register Stockham)
// The line is read with coalesced loads into LDS, zeros from L on (PAD: L < N; whole lines
// load without a branch per value, 2048^2 forward y-pass 10.0 us, 10.5 with it): a padded line costs
// the arithmetic of a whole one but reads L values only, and the stores of the N outputs
// bound it.  The generic line kernel, which runs one P-point transform per output residue
// (P >= L) in turn, took 17.3 us for 257 lines of 64 in 512 points and 79 us for 2049 of
// 2750 in 4096 (here about 4 and 21 us).  A unit-stride output line is
// written through LDS with 16-byte stores; a strided one (the transposed x-pass
// output) one value per output line, with each XCD owning a contiguous range
// of lines so that the partial lines meet in one L2.
#pragma once

#include "rows_wave.hpp"

namespace fastfft_amd {

template <int P, int Q, typename TIn, bool REAL, typename TOut, bool PAD>
__global__ void __launch_bounds__(64 * Q)
        k_fwd_full_wave(const TIn* __restrict__ in, LineMap im, int L, TOut* __restrict__ out, LineMap om, int nout, int nlines,
                        float pre_scale, const float2* __restrict__ tw) {
    constexpr int T = 64, E = P / T, N = P * Q, NT = T * Q;
    using FFT       = WaveFFT<P>;
    static_assert(Q * FFT::SLOTS >= N, "a line must fit the exchange buffers");
    static_assert(P % NT == 0 || NT % P == 0, "whole groups of the radix-Q pass per thread");
    __shared__ float2 lds[Q * FFT::SLOTS];
    __shared__ float2 s_twp[P];
    __shared__ float2 s_twn[NT];
    __shared__ float  s_real[REAL ? N : 1];
    const int     q    = __builtin_amdgcn_readfirstlane(threadIdx.x / T);
    const int     t    = threadIdx.x % T;
    const int     line = xcd_row(blockIdx.x, nlines);
    const float2* twm  = multi_twiddles(tw);
    // ---- the line into LDS (natural order), every load of the thread in
    // flight before its LDS writes
    {
        RowTwiddleStage<P, Q> tws;
        tws.load(twm);
        const auto* lp = as_global(in) + im.base(line);
        float2      z[N / NT];
#pragma unroll
        for ( int r = 0; r < N / NT; r++ ) {
            const int n = threadIdx.x + NT * r;
            z[r]        = make_float2(0.f, 0.f);
            if ( ! PAD || n < L ) {
                if constexpr ( REAL )
                    z[r].x = load_real(lp, n * im.es);
                else
                    z[r] = load_cpx(lp, n * im.es);
            }
        }
        tws.store(s_twp, s_twn);
#pragma unroll
        for ( int r = 0; r < N / NT; r++ ) {
            const int n = threadIdx.x + NT * r;
            if constexpr ( REAL )
                s_real[n] = z[r].x * pre_scale;
            else
                lds[n] = make_float2(z[r].x * pre_scale, z[r].y * pre_scale);
        }
    }
    __syncthreads( );
    // ---- radix-Q pass: thread m holds x[s P + m], s < Q, and leaves y_q[m] at q P + m
    for ( int m = threadIdx.x; m < P; m += NT ) {
        float2 u[Q];
#pragma unroll
        for ( int s = 0; s < Q; s++ ) {
            if constexpr ( REAL )
                u[s] = make_float2(s_real[s * P + m], 0.f);
            else
                u[s] = lds[s * P + m];
        }
        SmallDFT<Q, -1>::run(u);
#pragma unroll
        for ( int s = 0; s < Q; s++ )
            lds[s * P + m] = u[s];
    }
    __syncthreads( );
    FFT fft;
    fft.init_pt(t, s_twp);
    const float2 lw = lane_twiddle(s_twn, t, q); // W_N^{t q}
    float2       v[E];
#pragma unroll
    for ( int i = 0; i < E; i++ )
        v[i] = cmul(cmul(lds[q * P + t + T * i], twm[N + ((T * i * q) & (N - 1))]), lw);
    __syncthreads( );
    fft.template run<-1>(v, lds + q * FFT::SLOTS, t);
    auto* op = as_global(out) + om.base(line);
    if ( om.es == 1 ) {
        // natural order through LDS, then pair stores (op aligned to two values)
        __syncthreads( );
#pragma unroll
        for ( int i = 0; i < E; i++ )
            lds[dec_slot<P, Q>(Q * (t + T * i) + q)] = v[i];
        __syncthreads( );
        for ( int m = threadIdx.x; 2 * m < nout; m += NT ) {
            const float2 u0 = lds[dec_slot<P, Q>(2 * m)];
            if ( 2 * m + 1 < nout ) {
                const float2 u1 = lds[dec_slot<P, Q>(2 * m + 1)];
                store_cpx_pair(op, m, u0, u1);
            }
            else {
                store_cpx(op, 2 * m, u0);
            }
        }
    }
    else {
#pragma unroll
        for ( int i = 0; i < E; i++ ) {
            const int k = Q * (t + T * i) + q;
            if ( k < nout )
                store_cpx(op, k * om.es, v[i]);
        }
    }
}

// Full-length inverse line transforms (M = N outputs from 0): the C2C inverse
// passes and the C2R x-pass of an InvFFT without size change (the reference's
// block_fft_kernel_C2C_NONE inverse and C2R_NONE_XY, FastFFT.cu:1369-1403,
// :1641-1660).  With N = P*Q, decimation in time:
//   U_q[m]      = IFFT_P( X[Q k' + q] )[m]                       (wave q)
//   y[m + P s]  = sum_q W_Q^{-s q} ( W_N^{-m q} U_q[m] )         (radix-Q pass in LDS)
// HERM: the input line holds X[0 .. N/2] of a Hermitian sequence (X[N-k] =
// conj X[k] above) and only the real part of y is stored (REAL_OUT).
template <int P, int Q, typename TIn, bool HERM, typename TOut, bool REAL_OUT>
__global__ void __launch_bounds__(64 * Q)
        k_inv_full_wave(const TIn* __restrict__ in, LineMap im, TOut* __restrict__ out, LineMap om, int nlines,
                        float post_scale, const float2* __restrict__ tw) {
    constexpr int T = 64, E = P / T, N = P * Q, NT = T * Q, H = N / 2;
    using FFT       = WaveFFT<P>;
    static_assert(Q * FFT::SLOTS >= N, "a line must fit the exchange buffers");
    __shared__ float2 lds[Q * FFT::SLOTS];
    __shared__ float2 s_twp[P];
    __shared__ float2 s_twn[NT];
    const int     q    = __builtin_amdgcn_readfirstlane(threadIdx.x / T);
    const int     t    = threadIdx.x % T;
    const int     line = xcd_row(blockIdx.x, nlines);
    const float2* twm  = multi_twiddles(tw);
    // ---- unit-stride complex lines of up to 4 waves: every wave reads its decimated values from
    // memory, as in window_rows.hpp (1024^2 inverse 13.0 -> 12.4 us, 2048^2 26.2 -> 25.1)
    FFT    fft;
    float2 v[E];
    bool   direct = false;
    if constexpr ( ! HERM && std::is_same_v<TIn, float2> && Q <= 4 )
        direct = im.es == 1;
    if ( direct ) {
        RowTwiddleStage<P, Q> tws;
        tws.load(twm);
        const auto* lp = as_global(in) + im.base(line);
#pragma unroll
        for ( int i = 0; i < E; i++ )
            v[i] = load_cpx(at_bytes(lp, (unsigned)sizeof(TIn) * (unsigned)(Q * (t + T * i) + q)), 0);
        tws.store(s_twp, s_twn);
        __syncthreads( );
        fft.init_pt(t, s_twp);
    }
    // ---- else the input line into LDS, decimated by Q, two values per lane (the
    // decimated layout is conflict-free for pairs), every load of the thread
    // in flight before its LDS writes
    else {
        RowTwiddleStage<P, Q> tws;
        tws.load(twm);
        const auto*   lp = as_global(in) + im.base(line);
        constexpr int KN = HERM ? H + 1 : N;
        constexpr int MR = (KN + 2 * NT - 1) / (2 * NT);
        float2        u[MR][2];
#pragma unroll
        for ( int r = 0; r < MR; r++ ) {
            const int m = threadIdx.x + NT * r;
            u[r][0]     = 2 * m < KN ? load_cpx(lp, (long)(2 * m) * im.es) : make_float2(0.f, 0.f);
            u[r][1]     = 2 * m + 1 < KN ? load_cpx(lp, (long)(2 * m + 1) * im.es) : make_float2(0.f, 0.f);
        }
        tws.store(s_twp, s_twn);
#pragma unroll
        for ( int r = 0; r < MR; r++ ) {
            const int m = threadIdx.x + NT * r;
            if ( 2 * m < KN )
                lds[dec_slot<P, Q>(2 * m)] = u[r][0];
            if ( 2 * m + 1 < KN )
                lds[dec_slot<P, Q>(2 * m + 1)] = u[r][1];
        }
        __syncthreads( );
        fft.init_pt(t, s_twp);
#pragma unroll
        for ( int i = 0; i < E; i++ ) {
            const int k = Q * (t + T * i) + q;
            if constexpr ( HERM ) {
                const bool lo = k <= H;
                float2     z  = lds[dec_slot<P, Q>(lo ? k : N - k)];
                v[i]          = lo ? z : make_float2(z.x, -z.y);
            }
            else {
                v[i] = lds[dec_slot<P, Q>(k)];
            }
        }
        __syncthreads( );
    }
    float2* wl = lds + q * FFT::SLOTS;
    fft.template run<+1>(v, wl, t);
    // conj(W_N^{m q}) U_q[m], m = t + 64 i, into LDS at q P + m
    const float2 lw = lane_twiddle(s_twn, t, q);
    __syncthreads( );
#pragma unroll
    for ( int i = 0; i < E; i++ ) {
        const float2 w = cmul(lw, twm[N + ((T * i * q) & (N - 1))]);
        lds[q * P + t + T * i] = cmulc(v[i], w);
    }
    __syncthreads( );
    TOut* op = out + om.base(line);
    for ( int m = threadIdx.x; m < P; m += NT ) {
        float2 u[Q];
#pragma unroll
        for ( int s = 0; s < Q; s++ )
            u[s] = lds[s * P + m];
        SmallDFT<Q, +1>::run(u);
#pragma unroll
        for ( int s = 0; s < Q; s++ ) {
            const long j = (long)(m + P * s) * om.es;
            if constexpr ( REAL_OUT )
                store_real(op, j, u[s].x * post_scale);
            else
                store_cpx(op, j, make_float2(u[s].x * post_scale, u[s].y * post_scale));
        }
    }
}

} // namespace fastfft_amd
