// fbp.hip - the row filter of the DBT FBP: cosine weight and FFT convolution
// in LDS.
//
// The filter is a convolution along detector x (the tube-motion direction)
// with odd-length centred taps, samples off the detector 0:
//   q[a][i][j] = sum_i' taps[i' - i + c] pw[a][i'][j],  c = (ntaps - 1) / 2,
// pw the cosine-weighted views. Only taps with |i' - i| <= nbx - 1 meet data,
// so with L the power of two >= 2 nbx - 1 the sum is exactly the circular
// convolution of the zero-padded column with
//   H[m mod L] = taps[c - m],  |m| <= nbx - 1 (0 elsewhere),
// q = IFFT(FFT(pw column) FFT(H)). Two real columns ride in one complex
// sequence (column j real, j + 1 imaginary): H is real, so the convolution
// keeps them apart. Per column pair a forward and an inverse radix-2 FFT
// (L/2 log2 L butterflies each) replace the 2 nbx^2 multiply-adds of the
// direct sum.
//
// fbp_spectrum_kernel (one group) forms FFT(H) / L and the twiddle table
// exp(-2 pi i k / L), k < L/2, rounded from double; the filter kernels give
// each group SEQ column pairs of one view: they take them weighted and in
// bit-reversed order, run the decimation-in-time forward transform (natural
// order out), multiply by the spectrum, run the decimation-in-frequency
// inverse with conjugate twiddles (bit-reversed order out) and store rows
// i < nbx from their bit-reversed positions, so no reordering pass is needed.
// From L = 1024 on (there with many groups) fbp_filter_reg_kernel holds 16 points
// per thread and sequence in registers through up to four radix-2 stages between
// LDS exchanges; otherwise fbp_filter_kernel passes over LDS two stages at a time.
// Both make the same operations.
#include <type_traits>

#include "ostr_internal.h"

namespace ostr {

namespace {

constexpr int FFT_THREADS = 256;

__device__ __forceinline__ float2 cmul(float2 a, float2 b) {
    return make_float2(fmaf(a.x, b.x, -(a.y * b.y)), fmaf(a.x, b.y, a.y * b.x));
}
__device__ __forceinline__ float2 cadd(float2 a, float2 b) {
    return make_float2(a.x + b.x, a.y + b.y);
}
__device__ __forceinline__ float2 csub(float2 a, float2 b) {
    return make_float2(a.x - b.x, a.y - b.y);
}
__device__ __forceinline__ unsigned bitrev(unsigned i, int logl) {
    return __builtin_bitreverse32(i) >> (32 - logl);
}

// Forward transform, bit-reversed order in, natural order out, on the seq
// sequences of L = 2^logl elements at buf + s L. Radix-2 decimation in time,
// two stages at a time: the quadruple (i0, i0 + m, i0 + 2m, i0 + 3m) of stage
// half-size m goes through both radix-2 butterflies in registers (the same
// operations, one LDS round trip and barrier instead of two); an odd first
// stage runs alone. Ends with a barrier.
__device__ void fft_dit(float2* buf, int seq, int logl, const float2* tw) {
    const int L = 1 << logl;
    int lg = 0;
    if (logl & 1) {
        __syncthreads();
        for (int b = threadIdx.x; b < L / 2; b += FFT_THREADS) {
            const int i0 = b << 1;
            for (int s = 0; s < seq; ++s) {
                float2* a = buf + s * L;
                const float2 u = a[i0], o = cmul(a[i0 + 1], tw[0]);
                a[i0] = cadd(u, o);
                a[i0 + 1] = csub(u, o);
            }
        }
        lg = 1;
    }
    for (; lg < logl; lg += 2) {
        const int m = 1 << lg;
        __syncthreads();
        for (int b = threadIdx.x; b < L / 4; b += FFT_THREADS) {
            const int k = b & (m - 1);
            const int i0 = ((b >> lg) << (lg + 2)) | k;
            const float2 w = tw[k << (logl - 1 - lg)];
            const float2 w4a = tw[k << (logl - 2 - lg)];
            const float2 w4b = tw[(k + m) << (logl - 2 - lg)];
            for (int s = 0; s < seq; ++s) {
                float2* a = buf + s * L;
                const float2 e0 = a[i0], e1 = a[i0 + m], e2 = a[i0 + 2 * m], e3 = a[i0 + 3 * m];
                const float2 o1 = cmul(e1, w), o3 = cmul(e3, w);
                const float2 A0 = cadd(e0, o1), A1 = csub(e0, o1);
                const float2 A2 = cadd(e2, o3), A3 = csub(e2, o3);
                const float2 p2 = cmul(A2, w4a), p3 = cmul(A3, w4b);
                a[i0] = cadd(A0, p2);
                a[i0 + 2 * m] = csub(A0, p2);
                a[i0 + m] = cadd(A1, p3);
                a[i0 + 3 * m] = csub(A1, p3);
            }
        }
    }
    __syncthreads();
}

// Inverse transform without the 1/L, natural order in, bit-reversed order out:
// radix-2 decimation in frequency with conjugate twiddles, two stages at a
// time (the quadruple (i0, i0 + M/2, i0 + M, i0 + 3M/2) of stage half-size M
// through both butterflies in registers); an odd last stage runs alone.
__device__ void fft_dif_inverse(float2* buf, int seq, int logl, const float2* tw) {
    const int L = 1 << logl;
    auto ctw = [&](int i) {
        const float2 t = tw[i];
        return make_float2(t.x, -t.y);
    };
    int lg = logl - 1;
    for (; lg >= 1; lg -= 2) {
        const int M = 1 << lg, h = M >> 1;
        __syncthreads();
        for (int b = threadIdx.x; b < L / 4; b += FFT_THREADS) {
            const int k = b & (h - 1);
            const int i0 = ((b >> (lg - 1)) << (lg + 1)) | k;
            const float2 wk = ctw(k << (logl - 1 - lg));
            const float2 wh = ctw((k + h) << (logl - 1 - lg));
            const float2 v = ctw(k << (logl - lg));
            for (int s = 0; s < seq; ++s) {
                float2* a = buf + s * L;
                const float2 e0 = a[i0], e1 = a[i0 + h], e2 = a[i0 + M], e3 = a[i0 + M + h];
                const float2 A0 = cadd(e0, e2), A2 = cmul(csub(e0, e2), wk);
                const float2 A1 = cadd(e1, e3), A3 = cmul(csub(e1, e3), wh);
                a[i0] = cadd(A0, A1);
                a[i0 + h] = cmul(csub(A0, A1), v);
                a[i0 + M] = cadd(A2, A3);
                a[i0 + M + h] = cmul(csub(A2, A3), v);
            }
        }
    }
    if (lg == 0) {
        __syncthreads();
        for (int b = threadIdx.x; b < L / 2; b += FFT_THREADS) {
            const int i0 = b << 1;
            const float2 w = ctw(0);
            for (int s = 0; s < seq; ++s) {
                float2* a = buf + s * L;
                const float2 u = a[i0], v = a[i0 + 1];
                a[i0] = cadd(u, v);
                a[i0 + 1] = cmul(csub(u, v), w);
            }
        }
    }
    __syncthreads();
}

// ---- 16 points per thread in registers --------------------------------------
// L = 2^LOGL points, T = L / 16 threads. Pass p covers the radix-2 stages
// 4p .. 4p + S - 1, S = min(4, LOGL - 4p): a thread holds 16 >> S whole groups of
// 2^S points whose positions differ in those S bits only, so its stages need no
// exchange. Between passes the points go through LDS; a thread writes where it
// read in the pass before, so one barrier per exchange suffices. Positions are
// swizzled (fft_swz) so that the 32 lanes of an 8-byte LDS access fall on
// different banks in every pass (plain positions of pass 0 lie 128 bytes apart,
// 16 lanes to a bank).
template <int LOGL>
struct FftPlan {
    static constexpr int T = 1 << (LOGL - 4), PASSES = (LOGL + 3) / 4;
    // column pairs of a filter group; at 8192 points two would take all 160 KB of LDS
    static constexpr int SEQ = LOGL < 13 ? 2 : 1;
    static constexpr int stages(int p) { return LOGL - 4 * p < 4 ? LOGL - 4 * p : 4; }
};
__device__ __forceinline__ int fft_swz(int i) { return i ^ ((i >> 4) & 31); }

// Position of point q of group gg of thread t in pass P.
template <int LOGL, int P>
__device__ __forceinline__ int fft_pos(int t, int gg, int q) {
    constexpr int S = FftPlan<LOGL>::stages(P), LG = 4 * P;
    const int g = t + FftPlan<LOGL>::T * gg;
    return ((g >> LG) << (LG + S)) | (q << LG) | (g & ((1 << LG) - 1));
}

// b times a twiddle (w or, conjugated, its mirror): index j of stage s of a group
// at k = 0 is exp(-pi i j / 2^s), 1 for j = 0 and -i for j = 2^(s-1), for which
// nothing is multiplied (the table holds these exactly, so the bits are the
// same).
template <bool INVERSE>
__device__ __forceinline__ float2 fft_twiddle(float2 b, float2 w, int s, int j, bool at0) {
    if (at0 && j == 0) return b;
    if (at0 && 2 * j == (1 << s))
        return INVERSE ? make_float2(-b.y, b.x) : make_float2(b.y, -b.x);
    return cmul(b, w);
}

// Stages of pass P on the thread's points of SEQ sequences, e[seq][gg 2^S + q];
// the twiddles are read once for all sequences. In pass 0 the group's k is 0.
template <int LOGL, int SEQ, int P, bool INVERSE>
__device__ __forceinline__ void fft_pass(float2 (&e)[SEQ][16], int t, const float2* tw) {
    constexpr int S = FftPlan<LOGL>::stages(P), LG = 4 * P, N = 1 << S;
#pragma unroll
    for (int gg = 0; gg < 16 / N; ++gg) {
        const int k = (t + FftPlan<LOGL>::T * gg) & ((1 << LG) - 1);
        float2 w[N];  // stage s, index j at (1 << s) + j
#pragma unroll
        for (int s = 0; s < S; ++s)
#pragma unroll
            for (int j = 0; j < (1 << s); ++j) {
                const float2 v = tw[(k + (j << LG)) << (LOGL - 1 - LG - s)];
                w[(1 << s) + j] = INVERSE ? make_float2(v.x, -v.y) : v;
            }
#pragma unroll
        for (int c = 0; c < SEQ; ++c) {
            float2* a = e[c] + gg * N;
#pragma unroll
            for (int u = 0; u < S; ++u) {
                const int s = INVERSE ? S - 1 - u : u;
#pragma unroll
                for (int q = 0; q < N; ++q) {
                    if (q & (1 << s)) continue;
                    const int j = q & ((1 << s) - 1);
                    float2 &x = a[q], &y = a[q + (1 << s)];
                    const float2 ws = w[(1 << s) + j];
                    if (INVERSE) {
                        const float2 d = csub(x, y);
                        x = cadd(x, y);
                        y = fft_twiddle<true>(d, ws, s, j, P == 0);
                    } else {
                        const float2 o = fft_twiddle<false>(y, ws, s, j, P == 0);
                        y = csub(x, o);
                        x = cadd(x, o);
                    }
                }
            }
        }
    }
}

// The points from pass P's positions to pass Q's, through buf (SEQ L float2).
template <int LOGL, int SEQ, int P, int Q>
__device__ __forceinline__ void fft_exchange(float2 (&e)[SEQ][16], int t, float2* buf) {
    constexpr int L = 1 << LOGL;
    constexpr int NP = 1 << FftPlan<LOGL>::stages(P), NQ = 1 << FftPlan<LOGL>::stages(Q);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int at = fft_swz(fft_pos<LOGL, P>(t, i / NP, i % NP));
#pragma unroll
        for (int c = 0; c < SEQ; ++c) buf[c * L + at] = e[c][i];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int at = fft_swz(fft_pos<LOGL, Q>(t, i / NQ, i % NQ));
#pragma unroll
        for (int c = 0; c < SEQ; ++c) e[c][i] = buf[c * L + at];
    }
}

// Forward transform from pass 0's positions (bit-reversed order in) to the last
// pass' positions (natural order out); the inverse goes back the same way.
template <int LOGL, int SEQ, int P = 0>
__device__ __forceinline__ void fft_forward(float2 (&e)[SEQ][16], int t, float2* buf,
                                            const float2* tw) {
    fft_pass<LOGL, SEQ, P, false>(e, t, tw);
    if constexpr (P + 1 < FftPlan<LOGL>::PASSES) {
        fft_exchange<LOGL, SEQ, P, P + 1>(e, t, buf);
        fft_forward<LOGL, SEQ, P + 1>(e, t, buf, tw);
    }
}
template <int LOGL, int SEQ, int P = FftPlan<LOGL>::PASSES - 1>
__device__ __forceinline__ void fft_inverse(float2 (&e)[SEQ][16], int t, float2* buf,
                                            const float2* tw) {
    fft_pass<LOGL, SEQ, P, true>(e, t, tw);
    if constexpr (P > 0) {
        fft_exchange<LOGL, SEQ, P, P - 1>(e, t, buf);
        fft_inverse<LOGL, SEQ, P - 1>(e, t, buf, tw);
    }
}

// One group: the twiddles tw (global, L/2) and hs = FFT(H) / L (global, L).
// LDS: L + L/2 float2.
__global__ __launch_bounds__(FFT_THREADS) void fbp_spectrum_kernel(const float* __restrict__ taps,
                                                                   int ntaps, int nbx, int logl,
                                                                   float2* __restrict__ tw_out,
                                                                   float2* __restrict__ hs) {
    extern __shared__ float2 lds[];
    const int L = 1 << logl, c = (ntaps - 1) / 2;
    float2* tw = lds;
    float2* a = lds + L / 2;
    for (int k = threadIdx.x; k < L / 2; k += FFT_THREADS) {
        double sn, cs;
        sincospi(-2.0 * (double)k / (double)L, &sn, &cs);
        const float2 w = make_float2((float)cs, (float)sn);
        tw[k] = w;
        tw_out[k] = w;
    }
    for (int p = threadIdx.x; p < L; p += FFT_THREADS) {
        const int m = p < L / 2 ? p : p - L;
        const int t = c - m;
        const bool on = m >= -(nbx - 1) && m <= nbx - 1 && t >= 0 && t < ntaps;
        a[bitrev((unsigned)p, logl)] = make_float2(on ? taps[t] : 0.0f, 0.0f);
    }
    fft_dit(a, 1, logl, tw);
    const float inv = 1.0f / (float)L;  // a power of two: exact
    for (int p = threadIdx.x; p < L; p += FFT_THREADS)
        hs[p] = make_float2(a[p].x * inv, a[p].y * inv);
}

// fbp_spectrum_kernel with 16 points per thread in registers (L / 16 threads).
// The twiddles come from the first octant, the rest by symmetry: in double,
// one CU's share of 2048 sine and cosine pairs took longer than the transform.
template <int LOGL>
__global__ __launch_bounds__(FftPlan<LOGL>::T) void fbp_spectrum_reg_kernel(
    const float* __restrict__ taps, int ntaps, int nbx, float2* __restrict__ tw_out,
    float2* __restrict__ hs) {
    extern __shared__ float2 lds[];
    constexpr int L = 1 << LOGL, T = FftPlan<LOGL>::T, LAST = FftPlan<LOGL>::PASSES - 1;
    float2* tw = lds;
    float2* buf = lds + L / 2;
    const int t = threadIdx.x, c = (ntaps - 1) / 2;
    float2 e[1][16];
#pragma unroll
    for (int m = 0; m < 16; ++m) {
        const int pos = (int)bitrev((unsigned)(16 * t + m), LOGL);
        const int k = pos < L / 2 ? pos : pos - L;
        const int i = c - k;
        const bool on = k >= -(nbx - 1) && k <= nbx - 1 && i >= 0 && i < ntaps;
        e[0][m] = make_float2(on ? taps[i] : 0.0f, 0.0f);
    }
    for (int k = t; k <= L / 8; k += T) {
        double sn, cs;
        sincospi(2.0 * (double)k / (double)L, &sn, &cs);
        const float x = (float)cs, y = (float)sn;
        tw[k] = make_float2(x, -y);
        tw[L / 4 - k] = make_float2(y, -x);
        tw[L / 4 + k] = make_float2(-y, -x);
        if (k) tw[L / 2 - k] = make_float2(-x, -y);
    }
    __syncthreads();
    for (int k = t; k < L / 2; k += T) tw_out[k] = tw[k];
    fft_forward<LOGL, 1>(e, t, buf, tw);
    const float inv = 1.0f / (float)L;  // a power of two: exact
#pragma unroll
    for (int m = 0; m < 16; ++m) {
        constexpr int N = 1 << FftPlan<LOGL>::stages(LAST);
        hs[fft_pos<LOGL, LAST>(t, m / N, m % N)] = make_float2(e[0][m].x * inv, e[0][m].y * inv);
    }
}

// Group b of an n-group launch runs on XCD b % 8; hand each XCD one contiguous
// range of task indices so that neighbouring column chunks, which share cache
// lines of every detector row, meet in the same L2.
__device__ __forceinline__ int xcd_contiguous(int b, int n) {
    const int x = b & 7, q = n >> 3, r = n & 7;
    return x * q + (x < r ? x : r) + (b >> 3);
}

// Group = SEQ column pairs (2 SEQ columns from j0) of one slot. LDS: L/2 + SEQ L
// float2. p is [slot][nbx][nby] from slot a0, q the same or, with rows,
// detector-row-major [slot][nby][nbx]; vec: nby % 4 == 0 and p, q 16-byte
// aligned (float4 row loads and stores).
__global__ __launch_bounds__(FFT_THREADS) void fbp_filter_kernel(
    DevGeom g, const ViewTab* __restrict__ views, int a0, int n_slots, int n_chunks, int logl,
    const float2* __restrict__ tw_g, const float2* __restrict__ hs, const float* __restrict__ p,
    float* __restrict__ q, int vec, int rows) {
    constexpr int SEQ = 2;
    extern __shared__ float2 lds[];
    const int L = 1 << logl;
    float2* tw = lds;
    float2* buf = lds + L / 2;
    const int task = xcd_contiguous((int)blockIdx.x, n_chunks * n_slots);
    const int slot = task / n_chunks;
    const int j0 = (task % n_chunks) * 2 * SEQ;
    const int nbx = g.nbx, nby = g.nby;
    const ViewTab v = views[a0 + slot];
    const float D = v.z0 + g.det_r;
    float dy[2 * SEQ];
#pragma unroll
    for (int c = 0; c < 2 * SEQ; ++c) {
        const float ey = (float)((double)g.y_d0 + ((double)(j0 + c) + 0.5) * (double)g.dby);
        dy[c] = ey - g.src_y;
    }
    const int64_t base = (int64_t)slot * nbx * nby + j0;

    for (int k = threadIdx.x; k < L / 2; k += FFT_THREADS) tw[k] = tw_g[k];
    for (int i = threadIdx.x; i < L; i += FFT_THREADS) {
        float val[2 * SEQ];
#pragma unroll
        for (int c = 0; c < 2 * SEQ; ++c) val[c] = 0.0f;
        if (i < nbx) {
            const float ex = (float)((double)g.x_d0 + ((double)i + 0.5) * (double)g.dbx);
            const float dx = ex - v.x0;
            const float* row = p + base + (int64_t)i * nby;
            if (vec) {
                const float4 r4 = *(const float4*)row;
                val[0] = r4.x;
                val[1] = r4.y;
                val[2] = r4.z;
                val[3] = r4.w;
            } else {
#pragma unroll
                for (int c = 0; c < 2 * SEQ; ++c) val[c] = j0 + c < nby ? row[c] : 0.0f;
            }
#pragma unroll
            for (int c = 0; c < 2 * SEQ; ++c)
                val[c] *= D / sqrtf(fmaf(dx, dx, fmaf(dy[c], dy[c], D * D)));
        }
        const unsigned r = bitrev((unsigned)i, logl);
#pragma unroll
        for (int s = 0; s < SEQ; ++s) buf[s * L + r] = make_float2(val[2 * s], val[2 * s + 1]);
    }
    fft_dit(buf, SEQ, logl, tw);
    for (int f = threadIdx.x; f < L; f += FFT_THREADS) {
        const float2 h = hs[f];
#pragma unroll
        for (int s = 0; s < SEQ; ++s) buf[s * L + f] = cmul(buf[s * L + f], h);
    }
    fft_dif_inverse(buf, SEQ, logl, tw);
    if (rows) {  // a detector row is contiguous: whole lines
        const int64_t row0 = ((int64_t)slot * nby + j0) * nbx;
        for (int i = threadIdx.x; i < nbx; i += FFT_THREADS) {
            const unsigned r = bitrev((unsigned)i, logl);
#pragma unroll
            for (int s = 0; s < SEQ; ++s) {
                const float2 y = buf[s * L + r];
                if (j0 + 2 * s < nby) q[row0 + (int64_t)(2 * s) * nbx + i] = y.x;
                if (j0 + 2 * s + 1 < nby) q[row0 + (int64_t)(2 * s + 1) * nbx + i] = y.y;
            }
        }
        return;
    }
    for (int i = threadIdx.x; i < nbx; i += FFT_THREADS) {
        const unsigned r = bitrev((unsigned)i, logl);
        float val[2 * SEQ];
#pragma unroll
        for (int s = 0; s < SEQ; ++s) {
            const float2 y = buf[s * L + r];
            val[2 * s] = y.x;
            val[2 * s + 1] = y.y;
        }
        float* row = q + base + (int64_t)i * nby;
        if (vec) {
            *(float4*)row = make_float4(val[0], val[1], val[2], val[3]);
        } else {
#pragma unroll
            for (int c = 0; c < 2 * SEQ; ++c)
                if (j0 + c < nby) row[c] = val[c];
        }
    }
}

// fbp_filter_kernel with 16 points per thread and sequence in registers: same
// task and buffers, L / 16 threads. The forward transform's last pass, the
// spectrum and the inverse's first pass work on the same points, so 4 LDS
// exchanges at L = 4096 (one more for ROWS, detector-row-major q) replace 14
// passes over LDS. Bound by VALU issue (two waves per SIMD, 245 VGPRs) and the
// 16-byte pieces of p. 9 views of 2048x1664 bins:
// 365 us in passes, 174 here (ROWS 179); 25 of 1106x777 460, 253 (ROWS 210).
template <int LOGL, bool ROWS>
__global__ __launch_bounds__(FftPlan<LOGL>::T) __attribute__((amdgpu_waves_per_eu(2)))
void fbp_filter_reg_kernel(
    DevGeom g, const ViewTab* __restrict__ views, int a0, int n_slots, int n_chunks,
    const float2* __restrict__ tw_g, const float2* __restrict__ hs, const float* __restrict__ p,
    float* __restrict__ q, int vec) {
    extern __shared__ float2 lds[];
    constexpr int L = 1 << LOGL, T = FftPlan<LOGL>::T, LAST = FftPlan<LOGL>::PASSES - 1;
    constexpr int SEQ = FftPlan<LOGL>::SEQ;
    float2* tw = lds;
    float2* buf = lds + L / 2;
    const int t = threadIdx.x;
    const int task = xcd_contiguous((int)blockIdx.x, n_chunks * n_slots);
    const int slot = task / n_chunks;
    const int j0 = (task % n_chunks) * 2 * SEQ;
    const int nbx = g.nbx, nby = g.nby;
    const ViewTab v = views[a0 + slot];
    const float D = v.z0 + g.det_r;
    float dy[2 * SEQ];
#pragma unroll
    for (int c = 0; c < 2 * SEQ; ++c) {
        const float ey = (float)((double)g.y_d0 + ((double)(j0 + c) + 0.5) * (double)g.dby);
        dy[c] = ey - g.src_y;
    }
    const int64_t base = (int64_t)slot * nbx * nby + j0;
    // the column pairs' rows in bit-reversed order, all loads first
    float2 e[SEQ][16];
#pragma unroll
    for (int m = 0; m < 16; ++m) {
        const int i = (int)bitrev((unsigned)(16 * t + m), LOGL);
        float val[2 * SEQ];
#pragma unroll
        for (int c = 0; c < 2 * SEQ; ++c) val[c] = 0.0f;
        if (i < nbx) {
            const float* row = p + base + (int64_t)i * nby;
            if (SEQ == 2 && vec) {
                const float4 r4 = *(const float4*)row;
                val[0] = r4.x;
                val[1] = r4.y;
                val[2 * SEQ - 2] = r4.z;
                val[2 * SEQ - 1] = r4.w;
            } else {
#pragma unroll
                for (int c = 0; c < 2 * SEQ; ++c) val[c] = j0 + c < nby ? row[c] : 0.0f;
            }
        }
#pragma unroll
        for (int c = 0; c < SEQ; ++c) e[c][m] = make_float2(val[2 * c], val[2 * c + 1]);
    }
    for (int k = t; k < L / 2; k += T) tw[k] = tw_g[k];
#pragma unroll
    for (int m = 0; m < 16; ++m) {
        const int i = (int)bitrev((unsigned)(16 * t + m), LOGL);
        if (i >= nbx) continue;
        const float ex = (float)((double)g.x_d0 + ((double)i + 0.5) * (double)g.dbx);
        const float dx = ex - v.x0;
#pragma unroll
        for (int c = 0; c < SEQ; ++c) {
            e[c][m].x *= D / sqrtf(fmaf(dx, dx, fmaf(dy[2 * c], dy[2 * c], D * D)));
            e[c][m].y *= D / sqrtf(fmaf(dx, dx, fmaf(dy[2 * c + 1], dy[2 * c + 1], D * D)));
        }
    }
    __syncthreads();
    fft_forward<LOGL, SEQ>(e, t, buf, tw);
#pragma unroll
    for (int m = 0; m < 16; ++m) {
        constexpr int N = 1 << FftPlan<LOGL>::stages(LAST);
        const float2 h = hs[fft_pos<LOGL, LAST>(t, m / N, m % N)];
#pragma unroll
        for (int c = 0; c < SEQ; ++c) e[c][m] = cmul(e[c][m], h);
    }
    fft_inverse<LOGL, SEQ>(e, t, buf, tw);
    if (ROWS) {
        // through LDS once more, so that a wave writes whole lines of a row;
        // positions swizzled for the bit-reversed writes (8 lanes to a bank)
        __syncthreads();
        auto swz = [](int i) { return i ^ ((i >> 3) & 31); };
#pragma unroll
        for (int m = 0; m < 16; ++m) {
            const int i = (int)bitrev((unsigned)(16 * t + m), LOGL);
#pragma unroll
            for (int c = 0; c < SEQ; ++c) buf[c * L + swz(i)] = e[c][m];
        }
        __syncthreads();
        float* row = q + ((int64_t)slot * nby + j0) * nbx;
        for (int i = t; i < nbx; i += T) {
#pragma unroll
            for (int c = 0; c < SEQ; ++c) {
                const float2 y = buf[c * L + swz(i)];
                if (j0 + 2 * c < nby) row[(int64_t)(2 * c) * nbx + i] = y.x;
                if (j0 + 2 * c + 1 < nby) row[(int64_t)(2 * c + 1) * nbx + i] = y.y;
            }
        }
        return;
    }
#pragma unroll
    for (int m = 0; m < 16; ++m) {
        const int i = (int)bitrev((unsigned)(16 * t + m), LOGL);
        if (i >= nbx) continue;
        float* row = q + base + (int64_t)i * nby;
        if (SEQ == 2 && vec) {
            *(float4*)row =
                make_float4(e[0][m].x, e[0][m].y, e[SEQ - 1][m].x, e[SEQ - 1][m].y);
        } else {
#pragma unroll
            for (int c = 0; c < 2 * SEQ; ++c)
                if (j0 + c < nby) row[c] = (c & 1) ? e[c / 2][m].y : e[c / 2][m].x;
        }
    }
}

// Dynamic LDS beyond 64 KiB per group needs the kernel's opt-in.
hipError_t allow_lds(const void* kernel, size_t bytes) {
    if (bytes <= 65536) return hipSuccess;
    return hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
}

}  // namespace

int fbp_fft_log2(int nbx) {
    int logl = 1;
    while ((1 << logl) < 2 * nbx - 1) ++logl;
    return logl;
}

hipError_t launch_fbp_filter(const DevGeom& g, const ViewTab* views, int a0, int a1,
                             const float* taps, int ntaps, const float* p, float2* spec,
                             float* q, int rows, int lds_limit, hipStream_t st) {
    const int n_slots = a1 - a0;
    if (n_slots <= 0) return hipSuccess;
    const int logl = fbp_fft_log2(g.nbx);
    const int L = 1 << logl;
    if (logl > 13) return hipErrorInvalidValue;
    float2* tw = spec;        // L/2
    float2* hs = spec + L / 2;  // L
    const size_t spec_lds = (size_t)(L + L / 2) * sizeof(float2);
    const int seq = logl < 13 ? 2 : 1;  // column pairs per group (FftPlan::SEQ)
    const size_t lds = (size_t)(L / 2 + seq * L) * sizeof(float2);
    if (lds > (size_t)lds_limit || spec_lds > (size_t)lds_limit) return hipErrorInvalidValue;
    const int vec = (g.nby % 4 == 0) && ((uintptr_t)p % 16 == 0) && ((uintptr_t)q % 16 == 0);
    const int n_chunks = (g.nby + 2 * seq - 1) / (2 * seq);
    const dim3 grid((unsigned)(n_chunks * n_slots));
    // at most 1024 points; 256 threads, which one wave of 16 points each is slower than
    auto spectrum_by_passes = [&] {
        hipLaunchKernelGGL(fbp_spectrum_kernel, dim3(1), dim3(FFT_THREADS), spec_lds, st, taps,
                           ntaps, g.nbx, logl, tw, hs);
        return hipGetLastError();
    };
    auto in_registers = [&](auto logl_c) {
        constexpr int LOGL = decltype(logl_c)::value;
        const auto kernel = rows ? fbp_filter_reg_kernel<LOGL, true>
                                 : fbp_filter_reg_kernel<LOGL, false>;
        hipError_t err = allow_lds((const void*)kernel, lds);
        if (err != hipSuccess) return err;
        if constexpr (LOGL > 10) {
            const auto spectrum = fbp_spectrum_reg_kernel<LOGL>;
            if ((err = allow_lds((const void*)spectrum, spec_lds)) != hipSuccess) return err;
            hipLaunchKernelGGL(spectrum, dim3(1), dim3(FftPlan<LOGL>::T), spec_lds, st, taps,
                               ntaps, g.nbx, tw, hs);
            if ((err = hipGetLastError()) != hipSuccess) return err;
        } else if ((err = spectrum_by_passes()) != hipSuccess) {
            return err;
        }
        hipLaunchKernelGGL(kernel, grid, dim3(FftPlan<LOGL>::T), lds, st, g, views, a0, n_slots,
                           n_chunks, tw, hs, p, q, vec);
        return hipGetLastError();
    };
    switch (logl) {
        // one wave per 1024 points: faster where the groups are more than two per
        // CU (9 views of 300x300 bins, 675 groups, 21.4 us in passes and 19.2; 25
        // of 512x1200, 7500 groups, 128 and 91), slower where a group's latency
        // is the launch's (one view of 512x222 16.6 and 19.3, 5 of 512x400, 500
        // groups, 18.9 and 20.5)
        case 10:
            if (grid.x > 512) return in_registers(std::integral_constant<int, 10>());
            break;
        case 11: return in_registers(std::integral_constant<int, 11>());
        case 12: return in_registers(std::integral_constant<int, 12>());
        case 13: return in_registers(std::integral_constant<int, 13>());
    }
    // passes over LDS: fewer than 64 threads of 16 points, or few groups
    const hipError_t e = spectrum_by_passes();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(fbp_filter_kernel, grid, dim3(FFT_THREADS), lds, st, g, views, a0,
                       n_slots, n_chunks, logl, tw, hs, p, q, vec, rows);
    return hipGetLastError();
}

}  // namespace ostr
