// Router: logits (fp32 products, fp64 accumulation) -> top-k (ties to the lower expert id) ->
// softmax over the k selected logits.  Arithmetic follows the reference CPU path
// (src/run.cpp:321-404, 628-642); the GPU functions replaced are gemm_router
// (src/hip/gemms/gemm_router.hip:184), topk (src/hip/topk.hip:59) and softmax (src/hip/softmax.hip:46).
#include <type_traits>

#include "common.h"
#include "kernels.h"
#include "topk.h"

namespace moe {

// ---------------------------------------------------------------------------------------------
// Partial dot products.  One lane = one token, one wave = EG experts over one k-segment, so every
// accumulator walks its segment in ascending k exactly like the reference loop; with one segment
// the fp64 sum is bit-identical to src/run.cpp:348-351.  The four waves of a block share a
// transposed activation chunk of KC k-values in LDS (row stride 65 floats: conflict-free for the transposing
// store and for the lane-per-token read); weights are wave-uniform 16-byte loads issued one group
// of eight elements ahead (scalar registers: no vector ALU work to unpack them).
// grid = (ceil(T/64), ceil(E/(4*EG)), S), block = 256.
// partial layout: [S][T][E] fp64.
// ---------------------------------------------------------------------------------------------
template <int EG, int KC>
__global__ __launch_bounds__(256) void router_partial_kernel(const float* __restrict__ x,
                                                             const uint16_t* __restrict__ w,
                                                             double* __restrict__ partial,
                                                             uint16_t* __restrict__ x_bf16, int T, int H,
                                                             int E, int seg_len) {
    constexpr int NF = KC / 16;  // float4 loads per thread and chunk
    __shared__ float xs[KC][65];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int t0 = blockIdx.x * 64;
    const int e0 = (blockIdx.y * 4 + wave) * EG;  // first expert of the wave
    const int s = blockIdx.z;
    const int kbeg = s * seg_len;
    const int kend = min(H, kbeg + seg_len);

    // the blocks of the first expert group also emit the bf16 copy of the activations that the
    // expert GEMMs consume (every (token tile, segment) pair is visited exactly once by them)
    const bool write_bf16 = x_bf16 != nullptr && blockIdx.y == 0;

    double acc[EG];
#pragma unroll
    for (int j = 0; j < EG; ++j) acc[j] = 0.0;

    // chunk c+1 is fetched into registers while chunk c is consumed from LDS
    float4 xr[NF];
    auto fetch = [&](int k0) {
        const int kc = min(KC, kend - k0);  // multiple of 8
        const int q4 = kc >> 2;
#pragma unroll
        for (int it = 0; it < NF; ++it) {
            const int i = threadIdx.x + 256 * it;
            const int tl = i / q4;
            const int c = i - tl * q4;
            const int tok = t0 + tl;
            xr[it] = make_float4(0.f, 0.f, 0.f, 0.f);
            if (i < 64 * q4 && tok < T) xr[it] = *reinterpret_cast<const float4*>(x + (size_t)tok * H + k0 + 4 * c);
        }
    };
    auto stash = [&](int k0) {
        const int kc = min(KC, kend - k0);
        const int q4 = kc >> 2;
#pragma unroll
        for (int it = 0; it < NF; ++it) {
            const int i = threadIdx.x + 256 * it;
            if (i < 64 * q4) {
                const int tl = i / q4;
                const int c = i - tl * q4;
                if (write_bf16 && t0 + tl < T) {
                    uint2 o;
                    o.x = pack_bf16x2(xr[it].x, xr[it].y);
                    o.y = pack_bf16x2(xr[it].z, xr[it].w);
                    *reinterpret_cast<uint2*>(x_bf16 + (size_t)(t0 + tl) * H + k0 + 4 * c) = o;
                }
                xs[4 * c + 0][tl] = xr[it].x;
                xs[4 * c + 1][tl] = xr[it].y;
                xs[4 * c + 2][tl] = xr[it].z;
                xs[4 * c + 3][tl] = xr[it].w;
            }
        }
    };
    // weights: wave-uniform addresses (scalar loads), fetched one group of eight ahead
    const uint16_t* wrow[EG];
#pragma unroll
    for (int j = 0; j < EG; ++j) wrow[j] = w + (size_t)min(e0 + j, E - 1) * H;
    uint4 wv[EG], wn[EG];
#pragma unroll
    for (int j = 0; j < EG; ++j) wn[j] = *reinterpret_cast<const uint4*>(wrow[j] + min(kbeg, H - 8));
    if (kbeg < kend) fetch(kbeg);
    for (int k0 = kbeg; k0 < kend; k0 += KC) {
        const int kc = min(KC, kend - k0);
        stash(k0);
        __syncthreads();
        if (k0 + KC < kend) fetch(k0 + KC);
        if (e0 < E) {
            for (int kk = 0; kk < kc; kk += 8) {
#pragma unroll
                for (int j = 0; j < EG; ++j) {
                    wv[j] = wn[j];
                    wn[j] = *reinterpret_cast<const uint4*>(wrow[j] + min(k0 + kk + 8, H - 8));
                }
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const float xv = xs[kk + i][lane];
#pragma unroll
                    for (int j = 0; j < EG; ++j) {
                        const uint32_t word = (i < 2) ? wv[j].x : (i < 4) ? wv[j].y : (i < 6) ? wv[j].z : wv[j].w;
                        const float wf = (i & 1) ? __uint_as_float(word & 0xFFFF0000u)
                                                 : __uint_as_float(word << 16);
                        acc[j] += (double)__fmul_rn(wf, xv);
                    }
                }
            }
        }
        __syncthreads();
    }
    const int tok = t0 + lane;
    if (tok < T) {
#pragma unroll
        for (int j = 0; j < EG; ++j) {
            const int e = e0 + j;
            if (e < E) partial[((size_t)s * T + tok) * E + e] = acc[j];
        }
    }
}

// ---------------------------------------------------------------------------------------------
// Few tokens (a handful of token tiles): every block is latency bound, so it handles one segment
// of at most KS k-values in a single pass: all loads of the activation tile and of the four
// experts' weight segments are issued together, both land in LDS (weights widened to fp32), and
// each wave then walks its expert's segment in ascending k.  Same grid and partial layout as
// router_partial_kernel<1, *>.
// ---------------------------------------------------------------------------------------------
constexpr int kSmallSeg = 192;


__global__ __launch_bounds__(256) void router_partial_small_kernel(const float* __restrict__ x,
                                                                   const uint16_t* __restrict__ w,
                                                                   double* __restrict__ partial,
                                                                   uint16_t* __restrict__ x_bf16, int T, int H,
                                                                   int E, int seg_len) {
    constexpr int KS = kSmallSeg;
    constexpr int NF = KS / 16;
    __shared__ float xs[KS][65];
    __shared__ __align__(16) float wsh[4][KS];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int t0 = blockIdx.x * 64;
    const int e = blockIdx.y * 4 + wave;
    const int s = blockIdx.z;
    const int kbeg = s * seg_len;
    const int kc = min(H, kbeg + seg_len) - kbeg;  // multiple of 8, may be <= 0 for a trailing segment
    const bool write_bf16 = x_bf16 != nullptr && blockIdx.y == 0;
    double acc = 0.0;
    if (kc > 0) {
        const int q4 = kc >> 2;
        const int q8 = kc >> 3;
        float4 xr[NF];
#pragma unroll
        for (int it = 0; it < NF; ++it) {
            const int i = threadIdx.x + 256 * it;
            const int tl = i / q4;
            const int c = i - tl * q4;
            xr[it] = make_float4(0.f, 0.f, 0.f, 0.f);
            if (i < 64 * q4 && t0 + tl < T)
                xr[it] = *reinterpret_cast<const float4*>(x + (size_t)(t0 + tl) * H + kbeg + 4 * c);
        }
        // weights: thread i < 4*q8 loads eight bf16 of expert (blockIdx.y*4 + i/q8)
        uint4 wr = make_uint4(0, 0, 0, 0);
        const int wj = threadIdx.x / q8, wc = threadIdx.x - wj * q8;
        const bool wload = threadIdx.x < 4 * q8;
        if (wload)
            wr = *reinterpret_cast<const uint4*>(w + (size_t)min(blockIdx.y * 4 + wj, E - 1) * H + kbeg + 8 * wc);
#pragma unroll
        for (int it = 0; it < NF; ++it) {
            const int i = threadIdx.x + 256 * it;
            if (i < 64 * q4) {
                const int tl = i / q4;
                const int c = i - tl * q4;
                if (write_bf16 && t0 + tl < T) {
                    uint2 o;
                    o.x = pack_bf16x2(xr[it].x, xr[it].y);
                    o.y = pack_bf16x2(xr[it].z, xr[it].w);
                    *reinterpret_cast<uint2*>(x_bf16 + (size_t)(t0 + tl) * H + kbeg + 4 * c) = o;
                }
                xs[4 * c + 0][tl] = xr[it].x;
                xs[4 * c + 1][tl] = xr[it].y;
                xs[4 * c + 2][tl] = xr[it].z;
                xs[4 * c + 3][tl] = xr[it].w;
            }
        }
        if (wload) {
            float4 lo, hi;
            lo.x = __uint_as_float(wr.x << 16);
            lo.y = __uint_as_float(wr.x & 0xFFFF0000u);
            lo.z = __uint_as_float(wr.y << 16);
            lo.w = __uint_as_float(wr.y & 0xFFFF0000u);
            hi.x = __uint_as_float(wr.z << 16);
            hi.y = __uint_as_float(wr.z & 0xFFFF0000u);
            hi.z = __uint_as_float(wr.w << 16);
            hi.w = __uint_as_float(wr.w & 0xFFFF0000u);
            *reinterpret_cast<float4*>(&wsh[wj][8 * wc]) = lo;
            *reinterpret_cast<float4*>(&wsh[wj][8 * wc + 4]) = hi;
        }
        __syncthreads();
        if (e < E) {
            for (int kk = 0; kk < kc; kk += 8) {
                const float4 wa = *reinterpret_cast<const float4*>(&wsh[wave][kk]);
                const float4 wb = *reinterpret_cast<const float4*>(&wsh[wave][kk + 4]);
                acc += (double)__fmul_rn(wa.x, xs[kk + 0][lane]);
                acc += (double)__fmul_rn(wa.y, xs[kk + 1][lane]);
                acc += (double)__fmul_rn(wa.z, xs[kk + 2][lane]);
                acc += (double)__fmul_rn(wa.w, xs[kk + 3][lane]);
                acc += (double)__fmul_rn(wb.x, xs[kk + 4][lane]);
                acc += (double)__fmul_rn(wb.y, xs[kk + 5][lane]);
                acc += (double)__fmul_rn(wb.z, xs[kk + 6][lane]);
                acc += (double)__fmul_rn(wb.w, xs[kk + 7][lane]);
            }
        }
    }
    const int tok = t0 + lane;
    if (tok < T && e < E) partial[((size_t)s * T + tok) * E + e] = acc;
}

// ---------------------------------------------------------------------------------------------
// Finalise: one wave per token.  score[e] = float(sum_s partial[s][t][e]) + bias[e]
// (src/run.cpp:352, 635-637), then K rounds of wave-wide argmax ordered by (value desc, index
// asc), then the softmax of src/run.cpp:321-339 on the K selected values.
// When `partial` is NULL the scores are read from `scores_in` instead.
// grid = ceil(T/4), block = 256, dynamic LDS = 4*E floats.
// ---------------------------------------------------------------------------------------------

__global__ __launch_bounds__(256) void router_finalize_kernel(const double* __restrict__ partial, int S,
                                                              const float* __restrict__ scores_in,
                                                              const uint16_t* __restrict__ bias,
                                                              float* __restrict__ scores_out,
                                                              float* __restrict__ topk_v,
                                                              int* __restrict__ topk_i, int T, int E,
                                                              int K, int do_topk, int do_softmax) {
    extern __shared__ float sc[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int t = blockIdx.x * 4 + wave;
    if (t >= T) return;  // no block-wide barrier below
    float* my = sc + (size_t)wave * E;

    auto store = [&](int e, float v) {
        my[e] = v;
        if (scores_out) scores_out[(size_t)t * E + e] = v;
    };
    // summed in segment order, all loads in flight.  The number of segments is a constant of the loop: sixteen loads whatever it is
    // cost short rows more than the sums do (moe_gemm_router, us, so : a constant: 7 tokens, rows of 64, 512 experts 11.4 : 8.9; 64 tokens, rows
    // of 320, 512 experts 13.4 : 10.7; 4096 tokens, rows of 320, 128 experts 32.4 : 29.4).
    auto sums = [&](auto n) {
        constexpr int N = decltype(n)::value;
        const double* from = partial + (size_t)t * E;
        const size_t segment = (size_t)T * E;
        for (int e = lane; e < E; e += 64) {
            double sum = 0.0;
            double part[N];
#pragma unroll
            for (int s = 0; s < N; ++s) part[s] = from[s * segment + e];
#pragma unroll
            for (int s = 0; s < N; ++s) sum += part[s];
            store(e, (float)sum + bf16_bits_to_f32(bias[e]));
        }
    };
    if (!partial) {
        for (int e = lane; e < E; e += 64) store(e, scores_in[(size_t)t * E + e]);
    } else if (S == 16) {  // router_segments: a power of two up to 16
        sums(std::integral_constant<int, 16>{});
    } else if (S == 8) {
        sums(std::integral_constant<int, 8>{});
    } else if (S == 4) {
        sums(std::integral_constant<int, 4>{});
    } else if (S == 2) {
        sums(std::integral_constant<int, 2>{});
    } else {
        sums(std::integral_constant<int, 1>{});
    }
    if (!do_topk) return;
    __builtin_amdgcn_wave_barrier();

    float my_v;
    int my_i;
    select_topk(my, E, K, lane, my_v, my_i);
    write_topk(my_v, my_i, K, lane, do_softmax, topk_v + (size_t)t * K, topk_i + (size_t)t * K);
}

// ---------------------------------------------------------------------------------------------
// First pass of the two-pass router: approximate logits of ALL experts on the matrix cores.
// Every activation is split into two bf16 pieces, x = hi + lo + r with |r| <= 2^-16 |x|, and both
// pieces are multiplied with the bf16 router weights (products of two bf16 are exact in fp32) and
// accumulated in fp32 by v_mfma_f32_16x16x32_bf16.  Taking every fp32 addition inside the matrix
// unit and every accumulation to be good to one unit in the last place, a partial over a segment
// of n k-steps is within (33 + 2n) * 2^-23 * sum|w_k x_k| of the products it adds up.
// A wave owns 16 tokens (MFMA rows) and NE tiles of 16 experts (MFMA columns) over one k-segment.
// The same pass writes the bf16 copy of the activations (the hi pieces) for the expert GEMMs, the
// squared norm of every token's segment (xn2 [S][T]) and, in the blocks of the first token tile,
// of every router row's segment (wn2 [S][E]).  partial is [S][T][E] fp32.
// The four waves of a block share the router rows of their segment through LDS.
// grid = (ceil(T/64), ceil(E/(16*NE)), S), block = 256, dynamic LDS = 16*NE*(seg_len+8)*2 bytes;
// seg_len % 32 == 0, H % 32 == 0.
// ---------------------------------------------------------------------------------------------
// D: k-steps whose activation loads are in flight together (the kernel is a chain of memory round
// trips: one for the router rows, then one per D k-steps of its segment).
template <int NE, int D>
__global__ __launch_bounds__(256) void router_screen_kernel(const float* __restrict__ x,
                                                            const uint16_t* __restrict__ w,
                                                            float* __restrict__ partial, float* __restrict__ wn2,
                                                            float* __restrict__ xn2, uint16_t* __restrict__ x_bf16,
                                                            int T, int H, int E, int seg_len) {
    extern __shared__ __attribute__((aligned(16))) uint16_t wl[];  // [16*NE][seg_len + 8]
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane & 15, g = lane >> 4;
    const int t0 = blockIdx.x * 64 + wave * 16;
    const int e_base = blockIdx.y * 16 * NE;
    const int s = blockIdx.z;
    const int kbeg = s * seg_len;
    const int kend = min(H, kbeg + seg_len);  // kend - kbeg is a positive multiple of 32
    const int ldw = seg_len + 8;              // row stride 16 bytes off a multiple of 64: rows r, r+1 land 4 banks apart
    const bool first_group = blockIdx.y == 0;

    // activations first: D k-steps (32 values each) per request group, the next group in flight
    // while the current one is converted and multiplied
    const int tok = min(t0 + r, T - 1);
    const bool tok_ok = t0 + r < T;
    const float* xrow = x + (size_t)tok * H + 8 * g;
    float4 xa[D][2];
    auto load_group = [&](int k0) {
#pragma unroll
        for (int d = 0; d < D; ++d) {
            const int k = min(k0 + 32 * d, kend - 32);
            xa[d][0] = *reinterpret_cast<const float4*>(xrow + k);
            xa[d][1] = *reinterpret_cast<const float4*>(xrow + k + 4);
        }
    };
    load_group(kbeg);

    // this block's router rows over the segment -> LDS, shared by the four waves
    {
        const int cpr = (kend - kbeg) >> 3;  // 16-byte chunks per row
        for (int idx = threadIdx.x; idx < 16 * NE * cpr; idx += 256) {
            const int row = idx / cpr, c = idx - row * cpr;
            const int e = min(e_base + row, E - 1);
            *reinterpret_cast<u32x4*>(wl + row * ldw + 8 * c) =
                *reinterpret_cast<const u32x4*>(w + (size_t)e * H + kbeg + 8 * c);
        }
    }
    __syncthreads();

    if (blockIdx.x == 0) {  // block-uniform: squared norms of this block's router rows
        for (int i = wave; i < 16 * NE; i += 4) {
            const int e = e_base + i;
            if (e >= E) break;
            float q = 0.f;
            for (int k = lane; k < kend - kbeg; k += 64) {
                const float wf = bf16_bits_to_f32(wl[i * ldw + k]);
                q = fmaf(wf, wf, q);
            }
            q = wave_sum(q);
            if (lane == 0) wn2[(size_t)s * E + e] = q;
        }
    }
    if (t0 >= T) return;  // wave-uniform; no block-wide barrier below

    f32x4 acc[NE];
#pragma unroll
    for (int n = 0; n < NE; ++n) acc[n] = f32x4{0.f, 0.f, 0.f, 0.f};
    float x2 = 0.f;
    const int wfrag = r * ldw + 8 * g - kbeg;  // element index of this lane's fragment at k = 0

    for (int k0 = kbeg; k0 < kend; k0 += 32 * D) {
        float4 cur[D][2];
#pragma unroll
        for (int d = 0; d < D; ++d) {
            cur[d][0] = xa[d][0];
            cur[d][1] = xa[d][1];
        }
        if (k0 + 32 * D < kend) load_group(k0 + 32 * D);
#pragma unroll
        for (int d = 0; d < D; ++d) {
            const int k = k0 + 32 * d;
            if (k < kend) {  // wave-uniform
                const float v[8] = {cur[d][0].x, cur[d][0].y, cur[d][0].z, cur[d][0].w,
                                    cur[d][1].x, cur[d][1].y, cur[d][1].z, cur[d][1].w};
                u32x4 hi, lo;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const uint32_t h2 = pack_bf16x2(v[2 * i], v[2 * i + 1]);
                    hi[i] = h2;
                    lo[i] = pack_bf16x2(v[2 * i] - __uint_as_float(h2 << 16),
                                        v[2 * i + 1] - __uint_as_float(h2 & 0xFFFF0000u));
                    x2 = fmaf(v[2 * i], v[2 * i], x2);
                    x2 = fmaf(v[2 * i + 1], v[2 * i + 1], x2);
                }
                if (first_group && tok_ok && x_bf16)
                    *reinterpret_cast<u32x4*>(x_bf16 + (size_t)tok * H + 8 * g + k) = hi;
#pragma unroll
                for (int n = 0; n < NE; ++n) {
                    const u32x4 b = *reinterpret_cast<const u32x4*>(wl + (wfrag + 16 * n * ldw + k));
                    acc[n] = mfma_16x16x32(hi, b, acc[n]);
                    acc[n] = mfma_16x16x32(lo, b, acc[n]);
                }
            }
        }
    }
    // accumulator layout: lane holds tokens t0 + 4g + i (i = 0..3) for expert e_base + 16n + r
#pragma unroll
    for (int n = 0; n < NE; ++n) {
        const int e = e_base + 16 * n + r;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int t = t0 + 4 * g + i;
            if (e < E && t < T) partial[((size_t)s * T + t) * E + e] = acc[n][i];
        }
    }
    if (first_group) {
        x2 += __shfl_xor(x2, 16, 64);
        x2 += __shfl_xor(x2, 32, 64);
        if (g == 0 && tok_ok) xn2[(size_t)s * T + tok] = x2;
    }
}

// Exact logits of NE experts for one token, by one wave: fp32 products, fp64 sums
// (src/run.cpp:341-354).  Lane l takes float4 number l, l + 64, ... of the token's activations in
// ascending order; the lanes' sums are combined by wave_sum's fixed tree, so a logit does not depend
// on NE or on which other experts share the call.  The trip count is the same for every lane, so that
// the loads of several iterations can be in flight together: a lane past the end re-reads the row's last
// values and multiplies zeros in place of both (either may be an infinity), which leave its sum unchanged.
// Every lane returns all NE totals.
template <int NE, int UNROLL>
MOE_DEVICE void exact_dots(const float* __restrict__ x_row, const uint16_t* __restrict__ w, const int (&e)[NE], int H,
                           int lane, double (&total)[NE]) {
    const int n4 = H >> 2;
    const int trips = ceil_div(n4, 64);
    const float4* xrow = reinterpret_cast<const float4*>(x_row);
    const uint2* wrow[NE];
    double acc[NE];
#pragma unroll
    for (int i = 0; i < NE; ++i) {
        wrow[i] = reinterpret_cast<const uint2*>(w + (size_t)e[i] * H);
        acc[i] = 0.0;
    }
#pragma unroll UNROLL
    for (int j = 0; j < trips; ++j) {
        const bool live = lane + 64 * j < n4;
        const int i4 = min(lane + 64 * j, n4 - 1);
        float4 xv = xrow[i4];
        uint2 wb[NE];
#pragma unroll
        for (int i = 0; i < NE; ++i) wb[i] = wrow[i][i4];
        if (!live) xv = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
        for (int i = 0; i < NE; ++i) {
            if (!live) wb[i] = make_uint2(0u, 0u);
            acc[i] += (double)__fmul_rn(__uint_as_float(wb[i].x << 16), xv.x);
            acc[i] += (double)__fmul_rn(__uint_as_float(wb[i].x & 0xFFFF0000u), xv.y);
            acc[i] += (double)__fmul_rn(__uint_as_float(wb[i].y << 16), xv.z);
            acc[i] += (double)__fmul_rn(__uint_as_float(wb[i].y & 0xFFFF0000u), xv.w);
        }
    }
#pragma unroll
    for (int i = 0; i < NE; ++i) total[i] = wave_sum(acc[i]);
}

// The same for one expert and a row of up to 256 TRIPS values that the wave holds in registers (row_load): all of the router row's
// loads are in flight together.
template <int TRIPS>
MOE_DEVICE void row_load(const float* __restrict__ x_row, int H, int lane, float4 (&xv)[TRIPS]) {
#pragma unroll
    for (int j = 0; j < TRIPS; ++j) xv[j] = reinterpret_cast<const float4*>(x_row)[min(lane + 64 * j, (H >> 2) - 1)];
}
template <int TRIPS>
MOE_DEVICE double exact_dot_held(const float4 (&xv)[TRIPS], const uint16_t* __restrict__ w_row, int H, int lane) {
    const int n4 = H >> 2;
    uint2 wb[TRIPS];
#pragma unroll
    for (int j = 0; j < TRIPS; ++j) wb[j] = reinterpret_cast<const uint2*>(w_row)[min(lane + 64 * j, n4 - 1)];
    double acc = 0.0;
#pragma unroll
    for (int j = 0; j < TRIPS; ++j) {
        if (64 * j >= n4) break;  // wave-uniform
        float4 v = xv[j];
        if (lane + 64 * j >= n4) {
            v = make_float4(0.f, 0.f, 0.f, 0.f);
            wb[j] = make_uint2(0u, 0u);
        }
        acc += (double)__fmul_rn(__uint_as_float(wb[j].x << 16), v.x);
        acc += (double)__fmul_rn(__uint_as_float(wb[j].x & 0xFFFF0000u), v.y);
        acc += (double)__fmul_rn(__uint_as_float(wb[j].y << 16), v.z);
        acc += (double)__fmul_rn(__uint_as_float(wb[j].y & 0xFFFF0000u), v.w);
    }
    return wave_sum(acc);
}

// ---------------------------------------------------------------------------------------------
// Scores only, for a handful of tokens whose top-k is left to the gate/up kernel (experts_small.hip): a wave per (token, expert), so
// that the router rows come through many compute units instead of one.  Block of 1 token, E = 32, us, whole router before : this
// kernel 7.9 : 4.4; E = 128 11.8 : 4.4.
// grid = (ceil(E / 4), T), block = 256.
// ---------------------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void router_scores_kernel(const float* __restrict__ x, const uint16_t* __restrict__ w,
                                                            const uint16_t* __restrict__ bias, uint16_t* __restrict__ x_bf16,
                                                            float* __restrict__ scores, int H, int E) {
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int t = blockIdx.y;
    const int n4 = H >> 2;
    const float4* xr = reinterpret_cast<const float4*>(x + (size_t)t * H);
    if (blockIdx.x == 0)
        for (int c = threadIdx.x; c < n4; c += 256) {
            const float4 v = xr[c];
            reinterpret_cast<uint2*>(x_bf16 + (size_t)t * H)[c] = make_uint2(pack_bf16x2(v.x, v.y), pack_bf16x2(v.z, v.w));
        }
    const int e[1] = {(int)blockIdx.x * 4 + wave};
    if (e[0] >= E) return;
    double total[1];
    exact_dots<1, 12>(x + (size_t)t * H, w, e, H, lane, total);
    if (lane == 0) scores[(size_t)t * E + e[0]] = (float)total[0] + bf16_bits_to_f32(bias[e[0]]);
}

// ---------------------------------------------------------------------------------------------
// Whole router in one launch for batches too small for the two-pass router to pay: one block per
// token.  The block stages the token's activation row in LDS (and writes its row of the bf16 copy
// that the expert GEMMs consume); wave w scores experts NE*w .. NE*w + NE-1 (then NE*(w + waves) ..,
// if there are more) with the arithmetic and the order of additions of exact_dots — the same logits, bit for bit,
// as the exact pass of the two-pass router — and leaves them in LDS; wave 0 then runs top-k and
// softmax and writes the score row if the caller wants it.
// All loads of a wave's first pass (the activation piece it stages, its two router rows) are issued
// before anything waits, so a block costs one memory round trip plus the arithmetic.
// grid = T, block = 64 * waves, dynamic LDS = (256 * kFusedTrips + E) floats; H <= 256 * kFusedTrips.  NE experts per
// wave and pass: two with up to 16 waves (128 registers per lane hold the loads of two rows), four
// with up to 8 waves.
// ---------------------------------------------------------------------------------------------
constexpr int kFusedTrips = 12;  // rows of up to 3072 values

template <int NE>
__global__ __launch_bounds__(NE == 2 ? 1024 : 512) void router_fused_kernel(const float* __restrict__ x, const uint16_t* __restrict__ w,
                                                            const uint16_t* __restrict__ bias,
                                                            uint16_t* __restrict__ x_bf16,
                                                            float* __restrict__ scores_out, float* __restrict__ topk_v,
                                                            int* __restrict__ topk_i, int H, int E, int K,
                                                            int do_softmax) {
    extern __shared__ __attribute__((aligned(16))) float fused_lds[];
    float4* xs = reinterpret_cast<float4*>(fused_lds);  // [64 * kFusedTrips], zeros past the row
    float* sc = fused_lds + 256 * kFusedTrips;           // [E]
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n_waves = blockDim.x >> 6;
    const int t = blockIdx.x;
    const int n4 = H >> 2;
    const float4* xr = reinterpret_cast<const float4*>(x + (size_t)t * H);
    const int n_groups = ceil_div(E, NE);

    // activation row: thread i stages float4 number i, i + blockDim, ...
    constexpr int STG = NE == 2 ? 1 : 2;  // enough for a full-size block; smaller blocks take the loops below
    float4 xv_st[STG];
#pragma unroll
    for (int i = 0; i < STG; ++i) {
        const int c = threadIdx.x + i * blockDim.x;
        xv_st[i] = xr[min(c, n4 - 1)];
    }
    // per-lane element index of trip j, clamped into the row; as 32-bit byte offsets next to
    // wave-uniform row bases the loads need no per-lane 64-bit addresses
    uint32_t idx[kFusedTrips];
#pragma unroll
    for (int j = 0; j < kFusedTrips; ++j) idx[j] = (uint32_t)min(lane + 64 * j, n4 - 1);
    uint2 wb[kFusedTrips][NE];
    auto load_rows = [&](int grp) {
#pragma unroll
        for (int i = 0; i < NE; ++i) {
            const char* wrow = reinterpret_cast<const char*>(w + (size_t)min(grp * NE + i, E - 1) * H);
#pragma unroll
            for (int j = 0; j < kFusedTrips; ++j) wb[j][i] = *reinterpret_cast<const uint2*>(wrow + (size_t)(idx[j] * 8u));
        }
    };
    if (wave < n_groups) load_rows(wave);
    for (int c = n4 + threadIdx.x; c < 64 * kFusedTrips; c += blockDim.x) xs[c] = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int c = threadIdx.x + STG * blockDim.x; c < n4; c += blockDim.x) xs[c] = xr[c];  // blocks with few waves
#pragma unroll
    for (int i = 0; i < STG; ++i) {
        const int c = threadIdx.x + i * blockDim.x;
        if (c < n4) {
            xs[c] = xv_st[i];
            if (x_bf16)
                reinterpret_cast<uint2*>(x_bf16 + (size_t)t * H)[c] =
                    make_uint2(pack_bf16x2(xv_st[i].x, xv_st[i].y), pack_bf16x2(xv_st[i].z, xv_st[i].w));
        }
    }
    if (x_bf16)
        for (int c = threadIdx.x + STG * blockDim.x; c < n4; c += blockDim.x) {
            const float4 v = xr[c];
            reinterpret_cast<uint2*>(x_bf16 + (size_t)t * H)[c] = make_uint2(pack_bf16x2(v.x, v.y), pack_bf16x2(v.z, v.w));
        }
    __syncthreads();
    auto score_group = [&](int grp) {
        double acc[NE];
#pragma unroll
        for (int i = 0; i < NE; ++i) acc[i] = 0.0;
#pragma unroll
        for (int j = 0; j < kFusedTrips; ++j) {
            const bool live = lane + 64 * j < n4;
            const float4 xv = xs[lane + 64 * j];
#pragma unroll
            for (int i = 0; i < NE; ++i) {
                const uint2 wv = live ? wb[j][i] : make_uint2(0u, 0u);  // zeros on both sides: the sum stays
                acc[i] += (double)__fmul_rn(__uint_as_float(wv.x << 16), xv.x);
                acc[i] += (double)__fmul_rn(__uint_as_float(wv.x & 0xFFFF0000u), xv.y);
                acc[i] += (double)__fmul_rn(__uint_as_float(wv.y << 16), xv.z);
                acc[i] += (double)__fmul_rn(__uint_as_float(wv.y & 0xFFFF0000u), xv.w);
            }
        }
#pragma unroll
        for (int i = 0; i < NE; ++i) {
            const double total = wave_sum(acc[i]);
            const int e = grp * NE + i;
            if (lane == 0 && e < E) sc[e] = (float)total + bf16_bits_to_f32(bias[e]);
        }
    };
    // the usual case, one group per wave, is straight-line code (a loop here makes the compiler hoist
    // every trip's address arithmetic out of it and hold it in registers)
    if (wave < n_groups) score_group(wave);
    if (n_groups > n_waves) {
#pragma nounroll
        for (int grp = wave + n_waves; grp < n_groups; grp += n_waves) {
            load_rows(grp);
            score_group(grp);
        }
    }
    __syncthreads();
    if (wave != 0) return;
    if (scores_out)
        for (int e = lane; e < E; e += 64) scores_out[(size_t)t * E + e] = sc[e];
    float my_v;
    int my_i;
    select_topk(sc, E, K, lane, my_v, my_i);
    write_topk(my_v, my_i, K, lane, do_softmax, topk_v + (size_t)t * K, topk_i + (size_t)t * K);
}

// Bound of a token's approximate scores, from the squared norms of its row and of the longest router row.  Squares of small values are
// lost from the sums, up to 2^-126 each: a sum is taken to be at least 2^-95, which covers those and the bits that the lower pieces of
// such values lack.  Not a number stays one.
MOE_DEVICE float screen_bound(float err_coeff, float x2, float x2_margin, float w2, float amax) {
    if (x2 < 0x1p-95f) x2 = 0x1p-95f;
    if (w2 < 0x1p-95f) w2 = 0x1p-95f;
    return err_coeff * (sqrtf(x2) * x2_margin) * (sqrtf(w2) * 1.001f) + amax * 0x1p-20f;
}

// ---------------------------------------------------------------------------------------------
// Second pass of the two-pass router: one wave per token.
//   1. approximate scores a[e] = float(sum_s partial[s][t][e]) + bias[e] from the screening pass,
//      each within d of the exact score, d = err_coeff * |x_t|_2 * max_e |w_e|_2 (Cauchy-Schwarz
//      on sum|w_k x_k|; err_coeff from the screening pass's error model) plus the final roundings;
//   2. vK = K-th largest a.  An expert with a[e] < vK - 2d has an exact score below those of the K
//      experts with a >= vK, so the exact top K lies inside C = {e : a[e] >= vK - 2d};
//   3. the exact score (fp32 products, fp64 sum: src/run.cpp:341-354, 635-637) of every member
//      of C, each lane summing its own k in ascending order, lanes combined by a butterfly;
//   4. top-k and softmax over those exact scores, as in router_finalize_kernel.
// The result equals router_partial_kernel + router_finalize_kernel up to the order of
// the fp64 additions; |C| is K except for near-ties at the boundary (every exact tie is in C).
// grid = ceil(T/4), block = 256, dynamic LDS = 4 * 3 * E * 4 bytes.
// ---------------------------------------------------------------------------------------------
__global__ __launch_bounds__(256, 4) void router_refine_kernel(const float* __restrict__ partial, int S,
                                                            const float* __restrict__ wn2,
                                                            const float* __restrict__ xn2,
                                                            const float* __restrict__ x,
                                                            const uint16_t* __restrict__ w,
                                                            const uint16_t* __restrict__ bias, float err_coeff,
                                                            float* __restrict__ topk_v, int* __restrict__ topk_i,
                                                            int T, int H, int E, int K, int do_softmax,
                                                            float* __restrict__ approx_out,
                                                            float* __restrict__ delta_out,
                                                            int* __restrict__ n_cand_out) {
    extern __shared__ float sc[];
    __shared__ float w2_of_wave[4];
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int t = min(blockIdx.x * 4 + wave, T - 1);  // a surplus wave repeats the last token
    float* approx = sc + (size_t)wave * 3 * E;
    float* exact = approx + E;
    int* cand = reinterpret_cast<int*>(exact + E);

    // largest squared router-row norm: the same for every token, so the block's threads share it
    float w2max = 0.f;
#pragma nounroll
    for (int e = threadIdx.x; e < E; e += 256) {
        float q = 0.f;
#pragma nounroll
        for (int s0 = 0; s0 < S; s0 += 16) {
            float wq[16];
#pragma unroll
            for (int i = 0; i < 16; ++i) wq[i] = wn2[(size_t)min(s0 + i, S - 1) * E + e];
#pragma unroll
            for (int i = 0; i < 16; ++i) q += s0 + i < S ? wq[i] : 0.f;
        }
        w2max = fmaxf(w2max, q);
    }
    // approximate scores: all loads of up to two experts per lane in flight, summed in segment order
    float amax = 0.f;
#pragma nounroll
    for (int e0 = lane; e0 < E; e0 += 128) {
#pragma nounroll
        for (int s0 = 0; s0 < S; s0 += 16) {
            float part[2][16];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int e = min(e0 + 64 * h, E - 1);
#pragma unroll
                for (int i = 0; i < 16; ++i) part[h][i] = partial[((size_t)min(s0 + i, S - 1) * T + t) * E + e];
            }
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int e = e0 + 64 * h;
                double sum = s0 == 0 ? 0.0 : (double)exact[min(e, E - 1)];  // carries the sum when S > 16
#pragma unroll
                for (int i = 0; i < 16; ++i) sum += s0 + i < S ? (double)part[h][i] : 0.0;
                if (e < E) exact[e] = (float)sum;
            }
        }
    }
    float x2 = 0.f;
#pragma unroll 4
    for (int s = 0; s < S; ++s) x2 += xn2[(size_t)s * T + t];
    w2max = wave_max_nonneg(w2max);
    if (lane == 0) w2_of_wave[wave] = w2max;
    __syncthreads();
    if (blockIdx.x * 4 + wave >= T) return;  // no block-wide barrier below
    w2max = fmaxf(fmaxf(w2_of_wave[0], w2_of_wave[1]), fmaxf(w2_of_wave[2], w2_of_wave[3]));
#pragma nounroll
    for (int e = lane; e < E; e += 64) {
        const float v = exact[e] + bf16_bits_to_f32(bias[e]);
        approx[e] = v;
        exact[e] = -INFINITY;
        amax = fmaxf(amax, fabsf(v));
        if (approx_out) approx_out[(size_t)t * E + e] = v;  // what the screening decides on, for whoever checks the bound
    }
    amax = wave_max_nonneg(amax);
    // upper bound of |approx - exact| for every expert of this token; the 1.001 factors cover the
    // rounding of the two norms themselves, the last term the final roundings of both scores
    const float delta = screen_bound(err_coeff, x2, 1.001f, w2max, amax);
    __builtin_amdgcn_wave_barrier();

    float my_v;
    int my_i;
    select_topk(approx, E, K, lane, my_v, my_i);
    const float thr = lane_value(my_v, K - 1) - 2.f * delta;

    int n_cand = 0;
#pragma nounroll
    for (int e0 = 0; e0 < E; e0 += 64) {
        const int e = e0 + lane;
        // a not-a-number on either side decides nothing: an infinite router weight makes its expert's approximate score one
        // (the two pieces of an activation may differ in sign) where the exact score is an infinity
        const bool in = e < E && !(approx[e] < thr);
        const unsigned long long ballot = __ballot(in);
        if (in) cand[n_cand + __popcll(ballot & ((1ull << lane) - 1ull))] = e;
        n_cand += __popcll(ballot);
    }
    if (lane == 0) {
        if (delta_out) delta_out[t] = delta;
        if (n_cand_out) n_cand_out[t] = n_cand;
    }
    __builtin_amdgcn_wave_barrier();

    // exact scores of the candidates, four at a time
    const float* x_row = x + (size_t)t * H;
#pragma nounroll
    for (int c0 = 0; c0 < n_cand; c0 += 4) {
        int e[4];
        double total[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) e[i] = __builtin_amdgcn_readfirstlane(cand[min(c0 + i, n_cand - 1)]);
        exact_dots<4, 4>(x_row, w, e, H, lane, total);
        if (lane == 0) {
#pragma unroll
            for (int i = 0; i < 4; ++i) exact[e[i]] = (float)total[i] + bf16_bits_to_f32(bias[e[i]]);
        }
    }
    __builtin_amdgcn_wave_barrier();

    select_topk(exact, E, K, lane, my_v, my_i);
    write_topk(my_v, my_i, K, lane, do_softmax, topk_v + (size_t)t * K, topk_i + (size_t)t * K);
}

// ---------------------------------------------------------------------------------------------
// Both passes of the two-pass router in one launch, for up to 128 experts and rows of up to 3072 values: a block of 16
// waves takes TPB tokens whole.  Same steps and the same error model as router_screen_kernel and router_refine_kernel; the
// waves share the k range instead of the tokens while they screen (16 MFMA rows are 16 / TPB copies of each token, the sums of
// the 16 waves meet in LDS), and the tokens' candidates afterwards.
// What bounds it: a chain of latencies in a single round of blocks (256 tokens x 32 experts, in cycles: loads and screening 10400,
// sums 900, candidates 2300, their exact scores 3700, top-k and softmax 1800), and with eight tokens or more to a block the
// fp64 sums (16 cycles per product and wave) and the router rows through one compute unit's L1.  Screen + refine kernels : this
// one inside a block, us: E = 32, 512 tokens 23 : 13, 1000 25 : 17, 4096 43 : 40, 16384 149 : 135; E = 128, 1024 tokens 31 : 25.
// grid = ceil(T / TPB), block = 1024.
// ---------------------------------------------------------------------------------------------
constexpr int kRowsWaves = 16;
constexpr int kRowsPairs = 3;  // pairs of k-steps (64 values) per wave: rows of up to 3072 values
constexpr int kHeldTrips = 64 * kRowsWaves * kRowsPairs / 256;  // float4s of a row per lane

// The lanes of a wave exchange values through its own LDS area: no instruction is needed (a wave's LDS accesses are carried out in
// order), but the compiler must neither move accesses across nor run the two sides under different lane masks.
MOE_DEVICE void wave_lds_order() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}
// the area holds pieces of activations, of router rows and sums in turn
typedef __attribute__((may_alias)) u32x4 lds_u32x4;
typedef __attribute__((may_alias)) f32x4 lds_f32x4;
typedef __attribute__((may_alias)) float lds_f32;

template <int NE, int TPB>
__global__ __launch_bounds__(64 * kRowsWaves) void router_rows_kernel(const float* __restrict__ x, const uint16_t* __restrict__ w,
                                                                      const uint16_t* __restrict__ bias, float err_coeff,
                                                                      uint16_t* __restrict__ x_bf16, float* __restrict__ topk_v,
                                                                      int* __restrict__ topk_i, int T, int H, int E, int K,
                                                                      int do_softmax, float* __restrict__ approx_out,
                                                                      float* __restrict__ delta_out, int* __restrict__ n_cand_out) {
    constexpr int W = kRowsWaves, NP = kRowsPairs;
    constexpr int DUP = 16 / TPB;           // copies of a token among the 16 MFMA rows, and waves per token afterwards
    constexpr int EP = 16 * NE;             // experts, padded
    constexpr int LDP = EP + 4;             // floats from one token's partial row to the next
    constexpr int XI = TPB > 4 ? TPB / 4 : 1;                                 // loads that take a pair of all tokens
    constexpr int kStageBytes = 1024 * XI > 2048 ? 1024 * XI : 2048, kPartBytes = TPB * LDP * 4;
    constexpr int kArea = kStageBytes > kPartBytes ? kStageBytes : kPartBytes;  // LDS of one wave
    __shared__ __attribute__((aligned(16))) uint8_t area[W][(kArea + 15) & ~15];
    __shared__ float wsq[W][EP], xsq[W][16];
    __shared__ float approx[TPB][EP], exact[TPB][EP], w2[EP], x2[16];
    __shared__ int cand[TPB][EP], n_cands[TPB];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane & 15, g = lane >> 4;
    const int t0 = blockIdx.x * TPB;
    const int pairs = H >> 6;
    const int per = ceil_div(pairs, W);
    const int first = wave * per;
    const int count = min(max(pairs - first, 0), per);  // pairs of this wave, <= NP
    uint8_t* const mine = area[wave];
    lds_f32* const part = reinterpret_cast<lds_f32*>(mine);  // [TPB][LDP], once the wave has read all else

    // All loads take whole lines, consecutive lanes consecutive pieces of 16 bytes, and are turned into the MFMA operands'
    // layout in LDS: a load whose lanes follow the operand's layout (16 rows) runs at a lane a cycle, 16 bytes per compute unit
    // where these reach 50 to 60 (E = 128, one pass over the router rows from L2 50 thousand cycles against 14).
    // Buffer loads: the pair is the scalar part of an address, so that a lane keeps one offset per row.  Pairs that do not
    // exist re-read the last one.
    auto k_of = [&](int p) { return 64 * min(first + p, pairs - 1); };
    const __amdgpu_buffer_rsrc_t x_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(x + (size_t)t0 * H), 0, min(TPB, T - t0) * H * 4, 0x00020000);
    const __amdgpu_buffer_rsrc_t w_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(w), 0, E * H * 2, 0x00020000);
    u32x4 xf[NP][XI], wf[NP][2];
    // four tokens x 256 bytes a load
    const int last_row = min(TPB, T - t0) - 1;
#pragma unroll
    for (int p = 0; p < NP; ++p)
#pragma unroll
        for (int i = 0; i < XI; ++i)
            xf[p][i] = __builtin_amdgcn_raw_buffer_load_b128(x_rsrc, min(4 * i + g, last_row) * H * 4 + r * 16, k_of(p) * 4, 0);
    // eight router rows x 128 bytes a load
    auto load_w = [&](int tile, int p) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
            wf[p][i] = __builtin_amdgcn_raw_buffer_load_b128(w_rsrc, min(16 * tile + 8 * i + (lane >> 3), E - 1) * H * 2 + (lane & 7) * 16,
                                                             k_of(p) * 2, 0);
    };
#pragma unroll
    for (int p = 0; p < NP; ++p) load_w(0, p);
    __builtin_amdgcn_sched_barrier(0);
    // The activations in two bf16 pieces.  In k-step h of a pair a lane holds elements 32 h + 8 g .. + 7 of the 64.  LDS: token
    // row i at i * 256, its sixteen pieces of four values permuted, piece c at c ^ i.
    u32x4 hi[NP][2], lo[NP][2];
    {
        const int row = r / DUP;
        f32x4 xn = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int p = 0; p < NP; ++p) {
#pragma unroll
            for (int i = 0; i < XI; ++i) {
                *reinterpret_cast<lds_u32x4*>(mine + (4 * i + g) * 256 + ((r ^ (4 * i + g)) << 4)) = xf[p][i];
                if (x_bf16 != nullptr && p < count && 4 * i + g <= last_row)
                    *reinterpret_cast<u32x2*>(x_bf16 + (size_t)(t0 + 4 * i + g) * H + k_of(p) + 4 * r) =
                        u32x2{pack_bf16x2(__uint_as_float(xf[p][i][0]), __uint_as_float(xf[p][i][1])),
                              pack_bf16x2(__uint_as_float(xf[p][i][2]), __uint_as_float(xf[p][i][3]))};
            }
            wave_lds_order();
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                float v[8];
#pragma unroll
                for (int c = 0; c < 2; ++c) {
                    const f32x4 q = *reinterpret_cast<const lds_f32x4*>(mine + row * 256 + (((8 * h + 2 * g + c) ^ row) << 4));
#pragma unroll
                    for (int j = 0; j < 4; ++j) v[4 * c + j] = q[j];
                }
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const uint32_t h2 = pack_bf16x2(v[2 * i], v[2 * i + 1]);
                    hi[p][h][i] = h2;
                    lo[p][h][i] = pack_bf16x2(v[2 * i] - __uint_as_float(h2 << 16), v[2 * i + 1] - __uint_as_float(h2 & 0xFFFF0000u));
                }
                if (p < count) {  // wave-uniform
                    xn = mfma_16x16x32(hi[p][h], hi[p][h], xn);
                }
            }
            wave_lds_order();
        }
        // element (i, i) of a 16 x 16 product in the accumulator layout: lane (r, g = r / 4), value r % 4
        if (g == r >> 2) xsq[wave][r] = (r & 2) ? ((r & 1) ? xn[3] : xn[2]) : ((r & 1) ? xn[1] : xn[0]);
    }
    f32x4 acc[NE];
    // LDS: router row i of the tile at i * 128, its eight pieces of eight values permuted, piece c at c ^ (i / 2)
#pragma unroll
    for (int n = 0; n < NE; ++n) {
        f32x4 wn = {0.f, 0.f, 0.f, 0.f};
        acc[n] = wn;
#pragma unroll
        for (int p = 0; p < NP; ++p) {
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int row = 8 * i + (lane >> 3);
                *reinterpret_cast<lds_u32x4*>(mine + row * 128 + (((lane & 7) ^ (row >> 1)) << 4)) = wf[p][i];
            }
            wave_lds_order();
            if (n + 1 < NE) load_w(n + 1, p);
            if (p < count) {  // wave-uniform
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const u32x4 b = *reinterpret_cast<const lds_u32x4*>(mine + r * 128 + (((4 * h + g) ^ (r >> 1)) << 4));
                    acc[n] = mfma_16x16x32(hi[p][h], b, acc[n]);
                    wn = mfma_16x16x32(b, b, wn);
                    acc[n] = mfma_16x16x32(lo[p][h], b, acc[n]);
                }
            }
            wave_lds_order();
        }
        if (g == r >> 2) wsq[wave][16 * n + r] = (r & 2) ? ((r & 1) ? wn[3] : wn[2]) : ((r & 1) ? wn[1] : wn[0]);
    }
    // accumulator layout: lane holds MFMA rows 4 g + i (i = 0..3) for expert 16 n + r
#pragma unroll
    for (int n = 0; n < NE; ++n)
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if ((4 * g + i) % DUP == 0) part[(4 * g + i) / DUP * LDP + 16 * n + r] = acc[n][i];
    const int tl = wave / DUP, sub = wave % DUP;  // the wave's token, and its place among the token's waves
    const int t = t0 + tl;
    const float* x_row = x + (size_t)min(t, T - 1) * H;
    // Up to four tokens to a block the wave's row comes while the candidates are found (us, so : with them, E = 32, 300 tokens 11.1 : 10.6,
    // 1000 tokens 17.0 : 15.0; E = 128, 1024 tokens 24.2 : 22.8).  From eight on the waves take several candidates at a time, and a
    // held row costs them registers (2000 tokens 23.2 : 27.7, 4096 tokens 35.7 : 35.4).
    constexpr bool HELD = TPB <= 4;
    float4 x_held[HELD ? kHeldTrips : 1];
    if constexpr (HELD) row_load<kHeldTrips>(x_row, H, lane, x_held);
    __syncthreads();
    for (int i = threadIdx.x; i < TPB * EP; i += 64 * W) {
        const int ti = i / EP, e = i % EP;
        float sum = 0.f;
#pragma unroll
        for (int p = 0; p < W; ++p) sum += reinterpret_cast<const lds_f32*>(area[p])[ti * LDP + e];
        approx[ti][e] = e < E ? sum + bf16_bits_to_f32(bias[e]) : 0.f;
    }
    // from the other end, where the waves have no sum of their own while there are few tokens
    const int back = 64 * W - 1 - (int)threadIdx.x;
    if (back < EP + 16) {
        float q = 0.f;
        const float* from = back < EP ? &wsq[0][back] : &xsq[0][back - EP];
        const int stride = back < EP ? EP : 16;
#pragma unroll
        for (int p = 0; p < W; ++p) q += from[p * stride];
        if (back < EP) w2[back] = q;
        else x2[back - EP] = q;
    }
    __syncthreads();
    if (sub == 0) {  // candidates, as in router_refine_kernel
        const float* my = approx[tl];
        float amax = 0.f, wmax = 0.f;
#pragma unroll
        for (int e = lane; e < EP; e += 64) {
            amax = fmaxf(amax, fabsf(my[e]));
            wmax = fmaxf(wmax, w2[e]);
            if (approx_out && e < E && t < T) approx_out[(size_t)t * E + e] = my[e];
        }
        amax = wave_max_nonneg(amax);
        wmax = wave_max_nonneg(wmax);
        // the activations' norm is that of their upper pieces, each within 2^-8 of its activation
        const float delta = screen_bound(err_coeff, x2[tl * DUP], 1.006f, wmax, amax);
        float my_v;
        int my_i;
        select_topk_of<(EP + 63) / 64>(my, E, K, lane, my_v, my_i);
        const float thr = lane_value(my_v, K - 1) - 2.f * delta;
        int n = 0;
#pragma unroll
        for (int e0 = 0; e0 < EP; e0 += 64) {
            const int e = e0 + lane;
            const bool in = e < E && !(my[e < EP ? e : 0] < thr);  // a not-a-number decides nothing
            const unsigned long long ballot = __ballot(in);
            if (in) cand[tl][n + __popcll(ballot & ((1ull << lane) - 1ull))] = e;
            n += __popcll(ballot);
        }
        if (lane == 0) {
            n_cands[tl] = n;
            if (delta_out && t < T) delta_out[t] = delta;
            if (n_cand_out && t < T) n_cand_out[t] = n;
        }
    }
    __syncthreads();
    const int n_cand = __builtin_amdgcn_readfirstlane(n_cands[tl]);
    // exact scores: the waves of a token take its candidates in turn, C at a time
    constexpr int C = TPB == 16 ? 4 : TPB == 8 ? 2 : 1;
#pragma nounroll
    for (int c0 = C * sub; c0 < n_cand; c0 += C * DUP) {
        int e[C];
        double total[C];
#pragma unroll
        for (int i = 0; i < C; ++i) e[i] = __builtin_amdgcn_readfirstlane(cand[tl][min(c0 + i, n_cand - 1)]);
        if constexpr (HELD) total[0] = exact_dot_held<kHeldTrips>(x_held, w + (size_t)e[0] * H, H, lane);
        else exact_dots<C, C == 4 ? 4 : 12>(x_row, w, e, H, lane, total);
        if (lane == 0) {
#pragma unroll
            for (int i = 0; i < C; ++i)
                if (c0 + i < n_cand) exact[tl][c0 + i] = (float)total[i] + bf16_bits_to_f32(bias[e[i]]);
        }
    }
    __syncthreads();
    if (sub == 0 && t < T) {
        float my_v;
        int my_i;
        // candidates are in ascending order: ties as by expert id
        if (EP <= 64 || n_cand <= 64) select_topk_of<1>(exact[tl], n_cand, K, lane, my_v, my_i);  // wave-uniform
        else select_topk_of<2>(exact[tl], n_cand, K, lane, my_v, my_i);
        write_topk(my_v, cand[tl][my_i], K, lane, do_softmax, topk_v + (size_t)t * K, topk_i + (size_t)t * K);
    }
}

// In-place softmax over the last dimension, one thread per row, the reference's order of
// operations (src/run.cpp:321-339).  Up to eight values are loaded together instead of one after the other (256 rows of four, us,
// 4.6 : 4.5; two rows 2.5 : 2.0).
__global__ void softmax_rows_kernel(float* __restrict__ x, int B, int size) {
    const int b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= B) return;
    float* r = x + (size_t)b * size;
    if (size <= 8) {
        float v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = r[min(i, size - 1)];
        double max_val = v[0];
#pragma unroll
        for (int i = 1; i < 8; ++i)
            if (v[i] > max_val) max_val = v[i];  // the last value again past the end
        double sum = 0.0;
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if (i < size) {
                v[i] = expf((float)((double)v[i] - max_val));
                sum += v[i];
            }
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if (i < size) r[i] = (float)((double)v[i] / sum);
        return;
    }
    double max_val = r[0];
    for (int i = 1; i < size; ++i)
        if (r[i] > max_val) max_val = r[i];
    double sum = 0.0;
    for (int i = 0; i < size; ++i) {
        const float ex = expf((float)((double)r[i] - max_val));
        r[i] = ex;
        sum += ex;
    }
    for (int i = 0; i < size; ++i) r[i] = (float)((double)r[i] / sum);
}

// ---------------------------------------------------------------------------------------------
// Host launchers
// ---------------------------------------------------------------------------------------------
// Experts per wave: the largest group that still leaves about four waves per SIMD once the k range
// is cut into at most 16 segments (a larger group reuses each LDS read of an activation more often).
static int router_expert_group(int T, int E) {
    const long long tiles = ceil_div(T, 64);
    for (int eg = 4; eg > 1; eg >>= 1)
        if (tiles * ceil_div(E, eg) * 16 >= 4096) return eg;
    return 1;
}

int router_segments(int T, int E, int H, bool strict) {
    if (strict) return 1;
    const long long waves_one = (long long)ceil_div(T, 64) * ceil_div(E, router_expert_group(T, E));
    int S = 1;
    while (S < 16 && waves_one * S < 4096 && H / (S * 2) >= 64) S *= 2;
    return S;
}

int launch_router_partial(const float* x, const uint16_t* w, double* partial, uint16_t* x_bf16, int T, int H,
                          int E, int S, hipStream_t stream) {
    int seg_len = ceil_div(ceil_div(H, S), 8) * 8;
    const int eg = router_expert_group(T, E);
    dim3 grid(ceil_div(T, 64), ceil_div(E, 4 * eg), S);
    if (eg == 1 && seg_len <= kSmallSeg) {
        hipLaunchKernelGGL(router_partial_small_kernel, grid, dim3(256), 0, stream, x, w, partial, x_bf16, T, H, E,
                           seg_len);
    } else if (eg == 1) {
        hipLaunchKernelGGL((router_partial_kernel<1, 64>), grid, dim3(256), 0, stream, x, w, partial, x_bf16, T, H, E,
                           seg_len);
    } else if (eg == 2) {
        hipLaunchKernelGGL((router_partial_kernel<2, 64>), grid, dim3(256), 0, stream, x, w, partial, x_bf16, T, H, E,
                           seg_len);
    } else {
        hipLaunchKernelGGL((router_partial_kernel<4, 64>), grid, dim3(256), 0, stream, x, w, partial, x_bf16, T, H, E,
                           seg_len);
    }
    return launch_status();
}

// ---- two-pass router -----------------------------------------------------------------------------
// Worth it once the exact pass is throughput bound (16 cycles per term and wave), or once the fused kernel (a block
// per token) would need a second round of blocks over the 256 compute units (the lines below are its rounds there, not asked
// of the device).  With up to 32 experts a block holds a wave per two of them, several blocks share a compute unit, and
// what counts is scores per batch.  Up to 128 experts and rows of 3072 router_rows says when router_rows_kernel runs instead of
// these or the exact passes.  Whole block of tiny experts, rows of
// 2880, before the top-k became shorter in all of them (4 us), us, fused : screen + refine: E = 64, 256 tokens 48 : 57, 640 84 :
// 71; E = 128, 256 tokens 62 : 62, 257 82 : 63.
bool router_two_pass(int T, int E, int H) {
    if (H % 32 != 0) return false;
    const long long scores = (long long)T * E;
    if (scores >= 65536) return true;
    return E > 48 ? T > 256 : E > 32 ? T > 512 : E > 16 && scores >= 20480;
}

// Partial sums and finalize in two launches instead of the fused kernel: beyond 32 experts its eight waves score a token's
// experts in passes of 32, a memory round trip each, while few tokens leave most compute units idle.  The same block at that time, us,
// fused : two launches: E = 33, 1 token 24 : 24, 32 30 : 31, 128 37 : 38; E = 48, 1 token 29 : 24, 8 29 : 28, 64 32 : 33, 128 38 : 39; E = 64, 1
// token 28 : 24, 64 36 : 34, 128 40 : 38, 200 46 : 49; E = 128, 1 token 39 : 26, 33 tokens 55 : 44, 128 57 : 53; E = 1000, 16 tokens
// 199 : 92.  Up to 32 experts one launch is the faster one (1 token 22 : 24, 8 25 : 27, 256 41 : 45).
bool router_split(int T, int E) { return E > 32 && T <= (E > 48 ? 128 : 16); }

// Of those, a wave per (token, expert) for the scores rather than segments and their sums: a router row comes through the compute unit
// once per token.  Block of tiny experts, partial + finalize : scores + finalize, us: E = 49, rows of 64, 40 tokens 22.8 : 20.9; E = 128, rows
// of 2880, 9 tokens 31.4 : 28.3, 40 tokens 44.8 : 42.3 (48 and 64 tokens of the router alone 13.7 : 13.8 and 14.2 : 17.6); E = 512, rows of 320, 9
// tokens 25.8 : 23.0, 40 tokens 28.0 : 27.1; E = 1000, rows of 2880, 9 tokens 61 : 40, 32 tokens 78 : 75, 40 tokens 85 : 87, rows of 64, 32
// tokens 27.8 : 27.9, 40 tokens 28.2 : 29.5.
bool router_scores(int T, int E) { return T <= 40 && T * E <= 32000; }

static int screen_tiles(int E) { return E <= 16 ? 1 : E <= 32 ? 2 : 4; }  // 16-expert tiles per wave

// Segment length (multiple of 32) and count of the screening pass: enough segments for about 2048
// waves, and short enough for the block's router rows to fit 64 KB of LDS.
static void screen_plan(int T, int E, int H, int* seg_len, int* S) {
    const int ne = screen_tiles(E);
    const long long waves_one = (long long)ceil_div(T, 16) * ceil_div(E, 16 * ne);
    int want = 1;
    while (want < 16 && waves_one * want < 2048 && H / (want * 2) >= 64) want *= 2;
    const int seg_max = (65536 / (2 * 16 * ne) - 8) / 32 * 32;
    const int seg = min(seg_max, ceil_div(ceil_div(H, want), 32) * 32);
    *seg_len = seg;
    *S = ceil_div(H, seg);
}

size_t router_screen_bytes(int T, int E, int H) {
    int seg_len, S;
    screen_plan(T, E, H, &seg_len, &S);
    return ((size_t)S * T * E + (size_t)S * E + (size_t)S * T) * sizeof(float);
}

static bool router_rows_fits(int E, int H) { return E <= 128 && H % 64 == 0 && H <= 64 * kRowsWaves * kRowsPairs; }

// As few tokens to a block as one round of blocks over 256 compute units allows; more than 64 experts leave LDS for eight.
static int router_rows_tokens(int T, int E) {
    return T <= 256 ? 1 : T <= 512 ? 2 : T <= 1024 ? 4 : T <= 2048 || E > 64 ? 8 : 16;
}

// Whether router_rows_kernel runs, instead of the exact passes or, where router_two_pass holds, instead of screen + refine.
// Blocks of tiny experts, rows as said, us.
//   Exact passes : this, rows of 2880: E = 16, 1000 tokens 69 : 61; E = 32, 257 tokens 48 : 42 (64 tokens 8.9 : 9.4 for the router
// alone); E = 48, 17 tokens 31.4 : 30.2; E = 64, 65 tokens 34.4 : 31.9; E = 128, 65 tokens 49 : 43, but 33 tokens 13.3 : 15.5 alone, and
// with rows of 320 65 tokens 25.1 : 25.9, 128 25.1 : 26.0.  Up to eight experts a block of sixteen tokens does little more than load
// them, so its rounds have to be full: E = 8, 3300 tokens 107 : 105, 4200 (half of two rounds) 121 : 131, 7400 177 : 168, rows of 320, 4200
// 61 : 59; E = 6, 4000 tokens 112 : 112, 4500 120 : 133; E = 4 loses everywhere (5000 tokens 121 : 138, rows of 320 56 : 61).
//   Screen + refine : this: E = 16, 4097 tokens 125 : 129, 8192 189 : 181, rows of 320 8194 tokens 72 : 77; E = 64, 4096 tokens 214 : 204 and
// 65535, rows of 64, 381 : 419; E = 128, 2048 tokens 137 : 123, 2049 (a second round) rows of 1024 73 : 77, of 2048 106 : 109, of 2880 137 : 137;
// 4096 tokens, rows of 640 93 : 97, of 1024 101 : 97, of 2880 242 : 214; 30000 tokens, rows of 1024 591 : 636, of 1536 830 : 837.
bool router_rows(int T, int E, int H) {
    if (!router_rows_fits(E, H)) return false;
    const long long blocks = ceil_div(T, router_rows_tokens(T, E));
    const int full = (int)(100 * blocks / (ceil_div(blocks, 256LL) * 256));  // percent of the places in its rounds
    if (router_two_pass(T, E, H))
        return E > 64   ? T <= 2048 || H >= 2560 || (H >= 1024 && T > 3072 && T <= 16384)
               : E > 16 ? T <= 16384 || H >= 640
                        : H >= 1024 && full >= 70;
    return E > 64   ? T > (H < 1024 ? 128 : 64)
           : E > 48 ? T > 64
           : E > 32 ? T > 16
           : E > 16 ? T > 256
                    : (long long)T * E > 12000 && (E > 8 || (E > 4 && full >= (H >= 2048 ? 80 : E > 6 ? 0 : 60)));
}

// moe_router_two_pass_report takes it for all batches that moe_block_forward would not screen in a launch of its own.
bool router_one_launch(int T, int E, int H) { return router_rows(T, E, H) || (router_rows_fits(E, H) && !router_two_pass(T, E, H)); }

static int launch_router_rows(const float* x, const uint16_t* w, const uint16_t* bias, uint16_t* x_bf16, float* topk_v,
                              int* topk_i, int T, int H, int E, int K, int do_softmax, hipStream_t stream, float* approx_out,
                              float* delta_out, int* n_cand_out) {
    const int per_wave = 2 * ceil_div(H / 64, kRowsWaves);
    // per wave and segment as in launch_router_two_pass, and 16 additions of the waves' sums
    const float err_coeff = ((float)(33 + 2 * per_wave + 16) * 0x1p-23f + 0x1p-16f + 8 * 0x1p-24f) * 1.01f;
    const int tpb = router_rows_tokens(T, E);
#define MOE_ROWS(NE_, TPB_)                                                                                             \
    if (tpb == TPB_) {                                                                                                  \
        hipLaunchKernelGGL((router_rows_kernel<NE_, TPB_>), dim3(ceil_div(T, TPB_)), dim3(64 * kRowsWaves), 0, stream, x, w, \
                           bias, err_coeff, x_bf16, topk_v, topk_i, T, H, E, K, do_softmax, approx_out, delta_out, n_cand_out); \
        return launch_status();                                                                                         \
    }
#define MOE_ROWS_NE(NE_) MOE_ROWS(NE_, 1) MOE_ROWS(NE_, 2) MOE_ROWS(NE_, 4) MOE_ROWS(NE_, 8)
    if (E <= 32) {
        MOE_ROWS_NE(2) MOE_ROWS(2, 16)
    } else if (E <= 64) {
        MOE_ROWS_NE(4) MOE_ROWS(4, 16)
    } else {
        MOE_ROWS_NE(8)
    }
#undef MOE_ROWS_NE
#undef MOE_ROWS
    return MOE_ERR_LIMIT;
}

int launch_router_two_pass(const float* x, const uint16_t* w, const uint16_t* bias, void* scratch, uint16_t* x_bf16,
                           float* topk_v, int* topk_i, int T, int H, int E, int K, int do_softmax,
                           hipStream_t stream, hipEvent_t between, float* approx_out, float* delta_out,
                           int* n_cand_out) {
    if (router_one_launch(T, E, H)) {
        int rc = launch_router_rows(x, w, bias, x_bf16, topk_v, topk_i, T, H, E, K, do_softmax, stream, approx_out, delta_out,
                                    n_cand_out);
        if (rc) return rc;
        if (between) MOE_RETURN_IF_HIP(hipEventRecord(between, stream));
        return MOE_OK;
    }
    int seg_len, S;
    screen_plan(T, E, H, &seg_len, &S);
    float* partial = static_cast<float*>(scratch);
    float* wn2 = partial + (size_t)S * T * E;
    float* xn2 = wn2 + (size_t)S * E;
    const int ne = screen_tiles(E);
    dim3 grid(ceil_div(T, 64), ceil_div(E, 16 * ne), S);
    const size_t lds = (size_t)16 * ne * (seg_len + 8) * sizeof(uint16_t);
    // the whole segment in flight where it is short enough for the registers (D * 8 per lane)
    const int steps = seg_len / 32;
    const int depth = steps >= 12 ? 12 : steps >= 6 ? 6 : 4;
#define MOE_SCREEN(NE_, D_)                                                                                          \
    hipLaunchKernelGGL((router_screen_kernel<NE_, D_>), grid, dim3(256), lds, stream, x, w, partial, wn2, xn2, x_bf16, T, H, \
                       E, seg_len)
#define MOE_SCREEN_NE(NE_)          \
    if (depth == 12) {              \
        MOE_SCREEN(NE_, 12);        \
    } else if (depth == 6) {        \
        MOE_SCREEN(NE_, 6);         \
    } else {                        \
        MOE_SCREEN(NE_, 4);         \
    }
    if (ne == 1) {
        MOE_SCREEN_NE(1)
    } else if (ne == 2) {
        MOE_SCREEN_NE(2)
    } else {
        MOE_SCREEN_NE(4)
    }
#undef MOE_SCREEN_NE
#undef MOE_SCREEN
    int rc = launch_status();
    if (rc) return rc;
    if (between) MOE_RETURN_IF_HIP(hipEventRecord(between, stream));
    // error model of the screening pass per unit of |x| |w|: 33 + 2 * k-steps roundings of 2^-23 inside
    // a segment, the 2^-16 the two bf16 pieces leave out, and 8 * 2^-24 for the product roundings of
    // the exact path; 1 % slack
    const float err_coeff = ((float)(33 + 2 * (seg_len / 32)) * 0x1p-23f + 0x1p-16f + 8 * 0x1p-24f) * 1.01f;
    hipLaunchKernelGGL(router_refine_kernel, dim3(ceil_div(T, 4)), dim3(256),
                       (size_t)4 * 3 * E * sizeof(float), stream, partial, S, wn2, xn2, x, w, bias, err_coeff, topk_v,
                       topk_i, T, H, E, K, do_softmax, approx_out, delta_out, n_cand_out);
    return launch_status();
}

int launch_router_finalize(const double* partial, int S, const float* scores_in, const uint16_t* bias,
                           float* scores_out, float* topk_v, int* topk_i, int T, int E, int K, int do_topk,
                           int do_softmax, hipStream_t stream) {
    hipLaunchKernelGGL(router_finalize_kernel, dim3(ceil_div(T, 4)), dim3(256), (size_t)4 * E * sizeof(float),
                       stream, partial, S, scores_in, bias, scores_out, topk_v, topk_i, T, E, K, do_topk,
                       do_softmax);
    return launch_status();
}

// Rows the fused router can take (all of a wave's loads are held in registers at once).
bool router_fused_fits(int H) { return H % 4 == 0 && H <= 256 * kFusedTrips; }

// Up to 32 experts: two per wave, up to 16 waves (the shortest critical path per token); beyond: four
// per wave, 8 waves, as many passes as that takes.
int launch_router_fused(const float* x, const uint16_t* w, const uint16_t* bias, uint16_t* x_bf16, float* scores_out,
                        float* topk_v, int* topk_i, int T, int H, int E, int K, int do_softmax, hipStream_t stream) {
    if (!router_fused_fits(H)) return MOE_ERR_LIMIT;
    const size_t lds = (size_t)(256 * kFusedTrips + E) * sizeof(float);
    if (E <= 32) {
        hipLaunchKernelGGL(router_fused_kernel<2>, dim3(T), dim3(64 * min(16, ceil_div(E, 2))), lds, stream, x, w, bias,
                           x_bf16, scores_out, topk_v, topk_i, H, E, K, do_softmax);
    } else {
        hipLaunchKernelGGL(router_fused_kernel<4>, dim3(T), dim3(64 * min(8, ceil_div(E, 4))), lds, stream, x, w, bias,
                           x_bf16, scores_out, topk_v, topk_i, H, E, K, do_softmax);
    }
    return launch_status();
}

int launch_router_scores(const float* x, const uint16_t* w, const uint16_t* bias, uint16_t* x_bf16, float* scores, int T, int H,
                         int E, hipStream_t stream) {
    hipLaunchKernelGGL(router_scores_kernel, dim3(ceil_div(E, 4), T), dim3(256), 0, stream, x, w, bias, x_bf16, scores, H, E);
    return launch_status();
}

int launch_softmax_rows(float* x, int B, int size, hipStream_t stream) {
    hipLaunchKernelGGL(softmax_rows_kernel, dim3(ceil_div(B, 64)), dim3(64), 0, stream, x, B, size);
    return launch_status();
}

}  // namespace moe
