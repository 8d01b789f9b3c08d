// Fused correlation pass of one template with one workgroup of Q wavefronts per column
// (FwdImageInvFFT's second axis; the reference's block_fft_kernel_C2C_FWD_INCREASE_OP_INV_NONE /
// _FWD_NONE_INV_DECREASE_ConjMul, src/fastfft/FastFFT.cu:20-56, :1295-1344): any template
// length L <= N, any window of M <= N outputs from any origin o.
//
// For a column of full length N = P*Q, wave q computes
//   X[Q k' + q] = FFT_P( W_N^{m q} sum_s a[s P + m] W_Q^{s q} )[k'],   m < P, s P + m < L
//   U_q         = IFFT_P( img[Q k' + q] conj(X[Q k' + q]) )
// and leaves U_q in LDS; each output takes y[o + j] = sum_q W_N^{-(o + j) q} U_q[(o + j) mod P]
// in log2 Q steps (share_sum): no product per value of the sub-transforms, and nothing of the
// window in their registers.  (Windows of over a quarter of the column take one radix-Q pass
// instead, which costs less there.)  The image values are loaded
// before the template's transform and the Stockham twiddles are read from LDS at their use,
// which leaves 76 registers, three workgroups of 8 waves per CU.  No unit is saturated: 4096^2 with
// a 384^2 template and a 512^2 window (82 MB) keeps the VALU busy 65 % of its 30.9 us, the address
// units 60 % (the waves' image values share their lines) and the LDS 34 %, and waves wait for
// data and for their turn alike; the form with a product per value and 128 registers took 33.6 us.
// Capped at 64 registers 11 spill (39.5 us).
//
// DC and Nyquist columns (0 and last_line of a real transform): workgroup 0 takes both as one
// complex column, as described in xcorr_col.hpp.
#pragma once

#include <type_traits>

#include "rows_wave.hpp"

namespace fastfft_amd {

// WaveFFT<P>'s transform with the twiddles read from the pass table at their use instead of
// being held in registers.
template <int P, int DIR, int Ns = 1, int OFF = 0>
__device__ __forceinline__ void wave_passes(float2 (&v)[P / 64], float2* __restrict__ lds, int t, const float2* tab) {
    constexpr int  T = 64, E = P / T, R = (P / Ns) < E ? (P / Ns) : E, B = E / R;
    constexpr bool LAST = Ns * R == P;
    using Layout        = ExchangeLayout<P, E>;
#pragma unroll
    for ( int m = 0; m < B; m++ ) {
        const int b = t + T * m, j = b & (Ns - 1);
        float2    u[R];
#pragma unroll
        for ( int r = 0; r < R; r++ )
            u[r] = v[m + B * r];
        if constexpr ( Ns > 1 ) {
#pragma unroll
            for ( int r = 1; r < R; r++ ) {
                const float2 w = tab[OFF + (r - 1) * Ns + j];
                u[r]           = DIR < 0 ? cmul(u[r], w) : cmulc(u[r], w);
            }
        }
        SmallDFT<R, DIR>::run(u);
#pragma unroll
        for ( int r = 0; r < R; r++ ) {
            if constexpr ( LAST )
                v[m + B * r] = u[r];
            else
                lds[Layout::slot((b - j) * R + j + r * Ns)] = u[r];
        }
    }
    if constexpr ( ! LAST ) {
        wave_lds_fence( );
#pragma unroll
        for ( int i = 0; i < E; i++ )
            v[i] = lds[Layout::slot(t + T * i)];
        wave_lds_fence( );
        wave_passes<P, DIR, Ns * R, OFF + (Ns > 1 ? Ns * (R - 1) : 0)>(v, lds, t, tab);
    }
}

// sum_q W^q u[q PITCH], q < Q, with w[l] = conj W^{2^l}: the two halves' sums and one product, log2 Q
// products deep.  (Horner's rule in W, Q - 1 deep, puts a rounding of the whole sum at each step: rel-L2 error
// against 64 bits of small windows of 4096^2 2.8e-7, here 2.65e-7; of 1024 x 8192 with sixteen shares 3.1e-7, with
// eight 2.8e-7, here 2.65e-7.)
template <int Q, int PITCH, int LQ>
__device__ __forceinline__ float2 share_sum(const float2* u, const float2 (&w)[LQ]) {
    if constexpr ( Q == 1 )
        return u[0];
    else
        return cadd(share_sum<Q / 2, PITCH>(u, w), cmulc(share_sum<Q / 2, PITCH>(u + Q / 2 * PITCH, w), w[__builtin_ctz(Q / 2)]));
}

// Grid: nlines - 1 workgroups when pack_ends (columns 0 and last_line share workgroup 0), else
// nlines.  Element n of template column c is a[c lda + n a_es], of image column c img[c ldg + n],
// output j out[c ldo + j o_es]; 0 <= o < N.
template <int P, int Q, typename TImg>
__global__ void __launch_bounds__(64 * Q) __attribute__((amdgpu_waves_per_eu(P == 1024 ? 4 : 6)))
        k_xcorr_one(const float2* __restrict__ a, long lda, long a_es, int L, const TImg* __restrict__ img, long ldg,
                    float2* __restrict__ out, long ldo, long o_es, int M, int o, float scale, const float2* __restrict__ tw,
                    int last_line, int pack_ends) {
    constexpr int T = 64, E = P / T, N = P * Q, NT = T * Q, LQ = Q > 1 ? __builtin_ctz(Q) : 1;
    using FFT       = WaveFFT<P>;
    static_assert(FFT::SLOTS == P, "the workgroup's regions hold a whole column");
    __shared__ float2 lds[Q * P];
    __shared__ float2 s_twp[FFT::PT];
    const int     q    = __builtin_amdgcn_readfirstlane(threadIdx.x / T);
    const int     t    = threadIdx.x % T;
    const long    col  = xcd_row(blockIdx.x, gridDim.x);
    const bool    ends = pack_ends && col == 0;
    const float2* twm  = multi_twiddles(tw);
    float2*       wl   = lds + q * P;
    float2        pt[FFT::template pass_table_rows<NT>];
    FFT::template load_pass_table<NT>(pt, twm, threadIdx.x);
    const float2 lw = load_cpx(as_global(twm) + N, t * q); // W_N^{t q}
    auto         body = [&](auto ends_c) {
        constexpr bool ENDS = decltype(ends_c)::value;
        bits_t<TImg>   g[ENDS ? 1 : E];
        const auto*    ac = as_global(a) + col * lda;
        const auto*    a1 = as_global(a) + (long)last_line * lda;
        for ( int n = threadIdx.x; n < L; n += NT )
            lds[n] = ENDS ? make_float2(load_cpx(ac, n * a_es).x, load_cpx(a1, n * a_es).x) : load_cpx(ac, n * a_es);
        if constexpr ( ! ENDS ) {
            const auto* gc = as_global(img) + col * ldg;
#pragma unroll
            for ( int i = 0; i < E; i++ )
                g[i] = load_bits(at_bytes(gc, (unsigned)sizeof(TImg) * (unsigned)(Q * (t + T * i) + q)));
        }
        FFT::template store_pass_table<NT>(s_twp, pt, threadIdx.x);
        __syncthreads( );
        float2 v[E];
#pragma unroll
        for ( int i = 0; i < E; i++ )
            v[i] = t + T * i < L ? lds[t + T * i] : make_float2(0.f, 0.f);
        if constexpr ( Q > 1 ) {
            for ( int s = 1; s * P < L; s++ ) {
                const float2 c = twm[Q + ((s * q) & (Q - 1))]; // W_Q^{s q}, wave-uniform
#pragma unroll
                for ( int i = 0; i < E; i++ ) {
                    const int n = s * P + t + T * i;
                    if ( n < L )
                        v[i] = cadd(v[i], cmul(lds[n], c));
                }
            }
            if ( q != 0 ) { // wave-uniform
#pragma unroll
                for ( int i = 0; i < E; i++ )
                    v[i] = cmul(v[i], cmul(twm[N + ((T * i * q) & (N - 1))], lw));
            }
        }
        __syncthreads( ); // the template column is read before its slots become exchange regions
        wave_passes<P, -1>(v, wl, t, s_twp);
        if constexpr ( ! ENDS ) {
#pragma unroll
            for ( int i = 0; i < E; i++ )
                v[i] = cmulc(bits_value(g[i]), v[i]);
        }
        else {
            // Z[-k] for k = Q k' + q lies in the region of wave (Q - q) mod Q
#pragma unroll
            for ( int i = 0; i < E; i++ )
                wl[t + T * i] = v[i];
            __syncthreads( );
            const int   qp = (Q - q) % Q;
            const auto* g0 = as_global(img);
            const auto* g1 = as_global(img) + (long)last_line * ldg;
#pragma unroll
            for ( int i = 0; i < E; i++ ) {
                const int    kp  = t + T * i;
                const int    kpp = q == 0 ? (P - kp) & (P - 1) : P - 1 - kp;
                const float2 zm  = lds[qp * P + kpp];
                const int    k = Q * kp + q, km = (N - k) & (N - 1);
                const float2 i0 = load_cpx(g0, k), i0m = load_cpx(g0, km);
                const float2 i1 = load_cpx(g1, k), i1m = load_cpx(g1, km);
                const float2 h0 = make_float2(i0.x + i0m.x, i0.y - i0m.y); // 2 H_0[k]
                const float2 h1 = make_float2(i1.x + i1m.x, i1.y - i1m.y); // 2 H_1[k]
                const float2 d = csub(h0, h1), sm = cadd(h0, h1);
                const float2 r = cadd(cmul(make_float2(v[i].x, -v[i].y), d), cmul(zm, sm));
                v[i]           = make_float2(0.25f * r.x, 0.25f * r.y);
                // one value's loads at a time: this workgroup's registers bound every workgroup's
                __builtin_amdgcn_sched_barrier(0);
            }
            __syncthreads( );
        }
        wave_passes<P, +1>(v, wl, t, s_twp);
        auto* to    = as_global(out);
        auto  store = [&](int j, float2 y) {
            if constexpr ( ! ENDS ) {
                store_cpx(to, col * ldo + j * o_es, cscale(y, scale));
            }
            else {
                store_cpx(to, j * o_es, make_float2(y.x * scale, 0.f));
                store_cpx(to, (long)last_line * ldo + j * o_es, make_float2(y.y * scale, 0.f));
            }
        };
        if ( 4 * M > N ) {
            // a large part of the column: every output by one radix-Q pass,
            // y[m + P s] = sum_q W_Q^{-s q} ( W_N^{-m q} U_q[m] ) (exact for an impulse, as a whole
            // inverse's passes are)
#pragma unroll
            for ( int i = 0; i < E; i++ )
                wl[t + T * i] = Q > 1 ? cmulc(v[i], cmul(twm[N + ((T * i * q) & (N - 1))], lw)) : v[i];
            __syncthreads( );
            for ( int m = threadIdx.x; m < P; m += NT ) {
                float2 u[Q];
#pragma unroll
                for ( int s = 0; s < Q; s++ )
                    u[s] = lds[s * P + m];
                SmallDFT<Q, +1>::run(u);
#pragma unroll
                for ( int s = 0; s < Q; s++ ) {
                    const int j = (m + P * s - o) & (N - 1);
                    if ( j < M )
                        store(j, u[s]);
                }
            }
            return;
        }
#pragma unroll
        for ( int i = 0; i < E; i++ )
            wl[t + T * i] = v[i];
        __syncthreads( );
        for ( int j = threadIdx.x; j < M; j += NT ) {
            const int x = (o + j) & (N - 1);
            float2    w[LQ];
            // W_N^{x 2^l}: two entries W_{N / 2^l}^x of the table, then squares (all from the table, 1 % more accurate, takes
            // 2 % more of 4096^2 with 1021^2 and 1019^2: the loads' addresses)
#pragma unroll
            for ( int l = 0; l < LQ; l++ ) {
                if ( l < 2 )
                    w[l] = load_cpx(as_global(twm) + (N >> l), x & ((N >> l) - 1));
                else
                    w[l] = make_float2(fmaf(w[l - 1].x, w[l - 1].x, -w[l - 1].y * w[l - 1].y), 2.f * w[l - 1].x * w[l - 1].y);
            }
            store(j, share_sum<Q, P>(lds + (x & (P - 1)), w));
        }
    };
    if ( ends )
        body(std::true_type{ });
    else
        body(std::false_type{ });
}

} // namespace fastfft_amd
