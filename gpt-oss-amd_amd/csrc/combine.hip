// Weighted top-k combine, residual add and the FFN RMSNorm around the block.
#include <type_traits>

#include "common.h"
#include "kernels.h"

namespace moe {

// K, the experts per token, is a constant of these kernels (combine_of picks the instance): with a runtime K every step was a branch,
// the routing was loaded a value at a time, a scalar round trip each, and a row's loads waited for the branch in front of them.
// Rows of 2880, K = 4, us, so : now: by assignment 256 tokens 5.2 : 5.2, by slot 1000 tokens 12.7 : 10.1, 4096 tokens 48.4 : 35.6 (6.6 TB/s);
// with the norm, 100 tokens 8.7 : 5.1, 1024 tokens 17.6 : 14.9.  Other K, stage of the block, 2048 tokens: K = 1 18.3 : 10.7, K = 2 18.7 : 13.8,
// K = 6 27.7 : 27.3, K = 8 35.0 : 34.6; with the norm, K = 2 25.3 : 23.5, K = 6 41.1 : 38.3, K = 8 58.9 : 48.0.

// The token's K (slot, weight) pairs in ascending expert id (block-uniform: scalar loads and a
// fully unrolled insertion sort on K register entries).
template <int K>
MOE_DEVICE void sorted_slots(const int* __restrict__ slot_of, const int* __restrict__ topk_i,
                             const float* __restrict__ topk_v, int t, int (&sl)[K], float (&wt)[K]) {
    int ex[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
        ex[k] = topk_i[(size_t)t * K + k];
        sl[k] = slot_of[(size_t)t * K + k];
        wt[k] = topk_v[(size_t)t * K + k];
    }
#pragma unroll
    for (int i = 1; i < K; ++i) {
#pragma unroll
        for (int j = i; j > 0; --j) {
            const bool swap = ex[j] < ex[j - 1];
            const int te = ex[j], ts = sl[j];
            const float tw = wt[j];
            ex[j] = swap ? ex[j - 1] : te;
            sl[j] = swap ? sl[j - 1] : ts;
            wt[j] = swap ? wt[j - 1] : tw;
            ex[j - 1] = swap ? te : ex[j - 1];
            sl[j - 1] = swap ? ts : sl[j - 1];
            wt[j - 1] = swap ? tw : wt[j - 1];
        }
    }
}

MOE_DEVICE float4 fma4(const float4& v, float w, const float4& acc) {
    return make_float4(fmaf(v.x, w, acc.x), fmaf(v.y, w, acc.y), fmaf(v.z, w, acc.z), fmaf(v.w, w, acc.w));
}

// NT: the rows by slot are more than the last-level cache holds and not in it any more; they are read past it.  e_agg is written past it
// too: what the cache takes of it is written back during the launch after this one (the next call's router, 16384 tokens 125 us : 132 with the
// loads alone : 121 with both; whole block 2624 : 2604 : 2594, 8192 tokens 1335 : 1324 : 1323; with the norm, stage and router together, 12000
// tokens 324 : 298 : 278).
template <bool NT>
MOE_DEVICE float4 load_value(const float4* p) {
    if constexpr (NT) {
        const u32x4 v = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p));
        return make_float4(__uint_as_float(v[0]), __uint_as_float(v[1]), __uint_as_float(v[2]), __uint_as_float(v[3]));
    } else {
        return *p;
    }
}

template <bool NT>
MOE_DEVICE void store_value(float4* p, const float4& v) {
    if constexpr (NT) {
        const u32x4 bits = {__float_as_uint(v.x), __float_as_uint(v.y), __float_as_uint(v.z), __float_as_uint(v.w)};
        __builtin_nontemporal_store(bits, reinterpret_cast<u32x4*>(p));
    } else {
        *p = v;
    }
}

// NI float4 columns (from c0, `step` apart, those below H4) of the token's combined row: K fused multiply-adds in ascending expert id.
// slot_of == NULL: rows are stored by assignment, the row of (t, k) is t * K + k, known without looking at the routing, so
// their loads go out together with the loads of the routing itself (one memory round trip instead of two).  The order of the
// additions is fixed afterwards: the rank of each k by expert id is block-uniform, and rank r is added in step r.
template <int K, int NI, bool NT>
MOE_DEVICE void combine_columns(const float4* __restrict__ y, const int* __restrict__ slot_of, const int* __restrict__ topk_i,
                                const float* __restrict__ topk_v, int t, int H4, int c0, int step, float4 (&acc)[NI]) {
    float4 v[NI][K];
    float wt[K];
    if (slot_of) {  // uniform
        int sl[K];
        sorted_slots<K>(slot_of, topk_i, topk_v, t, sl, wt);
#pragma unroll
        for (int i = 0; i < NI; ++i) acc[i] = make_float4(0.f, 0.f, 0.f, 0.f);
        // Rows whose loads are in flight together.  Eight rows of a multiple of 4096 meet in the same L2 sets (stage of the block, 1024 tokens of
        // 4096 values, a runtime K : eight rows : two, 26.4 : 30.3 : 28.7; with the norm 34.1 : 35.3 : 33.6; of 2880 values 19.6 : 19.3 : 19.2).
        constexpr int AT_ONCE = K < 8 ? K : 2;
#pragma unroll
        for (int k0 = 0; k0 < K; k0 += AT_ONCE) {
#pragma unroll
            for (int i = 0; i < NI; ++i)
#pragma unroll
                for (int k = k0; k < min(k0 + AT_ONCE, K); ++k)
                    v[i][k] = load_value<NT>(y + (size_t)sl[k] * H4 + min(c0 + i * step, H4 - 1));
#pragma unroll
            for (int i = 0; i < NI; ++i)
#pragma unroll
                for (int k = k0; k < min(k0 + AT_ONCE, K); ++k) acc[i] = fma4(v[i][k], wt[k], acc[i]);
            if (AT_ONCE < K) __builtin_amdgcn_sched_barrier(0);
        }
        return;
    }
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int k = 0; k < K; ++k) v[i][k] = y[((size_t)t * K + k) * H4 + min(c0 + i * step, H4 - 1)];
    int ex[K], rank[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
        ex[k] = topk_i[(size_t)t * K + k];
        wt[k] = topk_v[(size_t)t * K + k];
    }
#pragma unroll
    for (int k = 0; k < K; ++k) {
        rank[k] = 0;
#pragma unroll
        for (int j = 0; j < K; ++j) rank[k] += (ex[j] < ex[k] || (ex[j] == ex[k] && j < k)) ? 1 : 0;
    }
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        acc[i] = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
        for (int r = 0; r < K; ++r) {
            float4 x = v[i][0];
            float w = wt[0];
#pragma unroll
            for (int k = 1; k < K; ++k) {
                const bool at = rank[k] == r;
                x.x = at ? v[i][k].x : x.x;
                x.y = at ? v[i][k].y : x.y;
                x.z = at ? v[i][k].z : x.z;
                x.w = at ? v[i][k].w : x.w;
                w = at ? wt[k] : w;
            }
            acc[i] = fma4(x, w, acc[i]);
        }
    }
}

// Whether the rows by slot are more than the 256 MiB of the last-level cache (NT).  Stage of the block, us, a runtime K : this without NT : with
// it, 8192 tokens: K = 4 of 2880 values 106 : 95 : 74 (6.4 TB/s), K = 6 of 5120 253 : 260 : 188, K = 8 of 8192 492 : 510 : 417; with the norm, K = 4 of 2880
// 166 : 153 : 116; 16384 tokens, K = 4 of 2880, 213 : 209 : 147.  Rows that the cache does hold are read from there: 2048 tokens, K = 7 of 4096 (235 MB)
// without : with 41.4 : 44.5, K = 5 of 5120 (210 MB) 38.3 : 39.2, and just past it K = 7 of 5120 (294 MB) 59.6 : 56.0, K = 8 of 4096 (268 MB) 54.8 : 50.8.
static bool rows_past_cache(const int* slot_of, int T, int K, int H) { return slot_of && (long long)T * K * H * 4 > (256ll << 20); }

// f(integral_constant<int, K>, bool_constant<NT>) for the runtime K of 1 .. 8
template <class Fn>
static int combine_of(int K, bool nt, Fn&& f) {
    auto with = [&](auto k) { return nt ? f(k, std::true_type{}) : f(k, std::false_type{}); };
    switch (K) {
        case 1: return with(std::integral_constant<int, 1>{});
        case 2: return with(std::integral_constant<int, 2>{});
        case 3: return with(std::integral_constant<int, 3>{});
        case 4: return with(std::integral_constant<int, 4>{});
        case 5: return with(std::integral_constant<int, 5>{});
        case 6: return with(std::integral_constant<int, 6>{});
        case 7: return with(std::integral_constant<int, 7>{});
        case 8: return with(std::integral_constant<int, 8>{});
    }
    return MOE_ERR_LIMIT;
}

// e_agg[t,:] = sum over the token's K experts, visited in ASCENDING EXPERT ID, of
// y_by_slot[slot,:] * weight, each step one fused multiply-add — the order and rounding of the
// reference CPU loop (src/run.cpp:645-706).  Replaces the atomicAdd scatter of
// moe_mlp2_scatter_mfma_kernel (src/hip/moe.hip:464-492), whose order is not fixed.
// Optionally also residual_x += e_agg (src/forward.cpp:514).
// grid = (ceil(H/4/256), T), block = 256.
template <int K, bool NT>
__global__ __launch_bounds__(256) void combine_kernel(const float4* __restrict__ y, const int* __restrict__ slot_of,
                                                      const int* __restrict__ topk_i,
                                                      const float* __restrict__ topk_v, float4* __restrict__ e_agg,
                                                      float4* __restrict__ residual_x, int T, int H4) {
    const int t = blockIdx.y;
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= H4) return;
    float4 before, acc[1];
    if (residual_x) before = residual_x[(size_t)t * H4 + c];  // uniform
    combine_columns<K, 1, NT>(y, slot_of, topk_i, topk_v, t, H4, c, 0, acc);
    store_value<NT>(e_agg + (size_t)t * H4 + c, acc[0]);
    if (residual_x)
        residual_x[(size_t)t * H4 + c] =
            make_float4(before.x + acc[0].x, before.y + acc[0].y, before.z + acc[0].z, before.w + acc[0].w);
}

int launch_combine(const float* y_by_slot, const int* slot_of, const int* topk_i, const float* topk_v,
                   float* e_agg, float* residual_x, int T, int K, int H, hipStream_t stream) {
    const int H4 = H / 4;
    return combine_of(K, rows_past_cache(slot_of, T, K, H), [&](auto k, auto nt) {
        hipLaunchKernelGGL((combine_kernel<decltype(k)::value, decltype(nt)::value>), dim3(ceil_div(H4, 256), T), dim3(256), 0, stream,
                           reinterpret_cast<const float4*>(y_by_slot), slot_of, topk_i, topk_v,
                           reinterpret_cast<float4*>(e_agg), reinterpret_cast<float4*>(residual_x), T, H4);
        return launch_status();
    });
}

// a += b * weight; b = 0   (src/hip/vecadd.hip:19-39)
// V: one value, or four where both arrays lie at 16-byte boundaries and the length allows it (1024 x 2880 9.6 : 8.9 us).
template <typename V>
__global__ void vecadd_and_zero_kernel(V* __restrict__ a, V* __restrict__ b, float weight, size_t n) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    V v = a[i];
    v += b[i] * weight;
    a[i] = v;
    b[i] = V{};
}

int launch_vecadd_and_zero(float* a, float* b, float weight, int batch, int size, hipStream_t stream) {
    const size_t n = (size_t)batch * size;
    if (n % 4 == 0 && (((uintptr_t)a | (uintptr_t)b) & 15u) == 0)
        hipLaunchKernelGGL(vecadd_and_zero_kernel<f32x4>, dim3((unsigned)ceil_div(n / 4, (size_t)256)), dim3(256), 0, stream,
                           reinterpret_cast<f32x4*>(a), reinterpret_cast<f32x4*>(b), weight, n / 4);
    else
        hipLaunchKernelGGL(vecadd_and_zero_kernel<float>, dim3((unsigned)ceil_div(n, (size_t)256)), dim3(256), 0, stream, a, b,
                           weight, n);
    return launch_status();
}

// RMSNorm of src/run.cpp:306-319 with the reference CPU's mixed precision: fp32 squares summed in
// fp64, sqrtf and the reciprocal in fp32, the scaling in fp64, one rounding to fp32 at the end.
// A row is owned by one block of 256 threads; thread i holds float4 columns i, i + 256, ... and adds
// their squares in ascending order, the fp64 sum over the block is a fixed tree over each wave and then the waves in order: results
// are run-to-run identical, and identical between the plain kernel and the one fused into the combine.
MOE_DEVICE double sumsq(double ss, const float4& v) {
    ss += (double)__fmul_rn(v.x, v.x);
    ss += (double)__fmul_rn(v.y, v.y);
    ss += (double)__fmul_rn(v.z, v.z);
    ss += (double)__fmul_rn(v.w, v.w);
    return ss;
}

// red: a value per wave of the block of 256
MOE_DEVICE double block_inv_rms(double ss, double* red, int size) {
    const int wave0 = __builtin_amdgcn_readfirstlane(threadIdx.x & ~63u);
    const double sum = 4 * wave0 < size ? wave_sum(ss) : 0.0;  // short rows: waves without a value (8192 x 64 7.6 : 4.5 us)
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = sum;
    __syncthreads();
    double m = ((red[0] + red[1]) + red[2] + red[3]) / size;
    m += (double)1e-5f;
    return (double)(1.0f / sqrtf((float)m));
}

MOE_DEVICE float4 norm_scale(const float4& v, const uint16_t* __restrict__ weight, int c, double inv) {
    const uint2 wb = *reinterpret_cast<const uint2*>(weight + 4 * c);
    float4 o;
    o.x = (float)((double)bf16_bits_to_f32(wb.x & 0xFFFFu) * (inv * (double)v.x));
    o.y = (float)((double)bf16_bits_to_f32(wb.x >> 16) * (inv * (double)v.y));
    o.z = (float)((double)bf16_bits_to_f32(wb.y & 0xFFFFu) * (inv * (double)v.z));
    o.w = (float)((double)bf16_bits_to_f32(wb.y >> 16) * (inv * (double)v.w));
    return o;
}

// grid = rows, block = 256; size % 4 == 0.  NI > 0: rows of up to 1024 NI values, read once into registers; NI = 0: any, read twice.
// 256 x 2880, us, eight barriers and two passes : now 5.0 : 4.9, 2 x 2880 4.3 : 3.3.
template <int NI>
__global__ __launch_bounds__(256) void rmsnorm_kernel(float* __restrict__ o, const float* __restrict__ x,
                                                      const uint16_t* __restrict__ weight, int size) {
    __shared__ double red[4];
    const int H4 = size >> 2;
    const float4* xr = reinterpret_cast<const float4*>(x + (size_t)blockIdx.x * size);
    float4* orow = reinterpret_cast<float4*>(o + (size_t)blockIdx.x * size);
    double ss = 0.0;
    float4 v[NI > 0 ? NI : 1];
    if constexpr (NI > 0) {
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            const int c = threadIdx.x + 256 * i;
            v[i] = c < H4 ? xr[c] : make_float4(0.f, 0.f, 0.f, 0.f);
        }
#pragma unroll
        for (int i = 0; i < NI; ++i) ss = sumsq(ss, v[i]);
    } else {
        for (int c = threadIdx.x; c < H4; c += 256) ss = sumsq(ss, xr[c]);
    }
    const double inv = block_inv_rms(ss, red, size);
    if constexpr (NI > 0) {
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            const int c = threadIdx.x + 256 * i;
            if (c < H4) orow[c] = norm_scale(v[i], weight, c, inv);
        }
    } else {
        for (int c = threadIdx.x; c < H4; c += 256) orow[c] = norm_scale(xr[c], weight, c, inv);
    }
}

// Combine, residual add and the RMSNorm that follows it in the layer loop (the attention norm of the
// next layer, src/forward.cpp:262, or the final norm, :997), in one pass over the token's row:
//   e_agg = combine;  residual_x += e_agg;  norm_out = rmsnorm(residual_x, norm_weight).
// Same arithmetic as combine_kernel followed by rmsnorm_kernel.  A thread keeps its NI float4 columns
// of the updated residual in registers.  grid = T, block = 256, H/4 <= 256 * NI.
template <int NI, int K, bool NT>
__global__ __launch_bounds__(256) void combine_norm_kernel(const float4* __restrict__ y, const int* __restrict__ slot_of,
                                                           const int* __restrict__ topk_i,
                                                           const float* __restrict__ topk_v, float4* __restrict__ e_agg,
                                                           float4* __restrict__ residual_x,
                                                           const uint16_t* __restrict__ norm_weight,
                                                           float4* __restrict__ norm_out, int H4) {
    __shared__ double red[4];
    const int t = blockIdx.x;
    float4 r[NI], acc[NI];
#pragma unroll
    for (int i = 0; i < NI; ++i) r[i] = residual_x[(size_t)t * H4 + min((int)threadIdx.x + 256 * i, H4 - 1)];
    combine_columns<K, NI, NT>(y, slot_of, topk_i, topk_v, t, H4, threadIdx.x, 256, acc);
    double ss = 0.0;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        const int c = threadIdx.x + 256 * i;
        if (c < H4) {
            store_value<NT>(e_agg + (size_t)t * H4 + c, acc[i]);
            r[i].x += acc[i].x;
            r[i].y += acc[i].y;
            r[i].z += acc[i].z;
            r[i].w += acc[i].w;
            residual_x[(size_t)t * H4 + c] = r[i];
            ss = sumsq(ss, r[i]);
        }
    }
    const double inv = block_inv_rms(ss, red, 4 * H4);
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        const int c = threadIdx.x + 256 * i;
        if (c < H4) norm_out[(size_t)t * H4 + c] = norm_scale(r[i], norm_weight, c, inv);
    }
}

bool combine_norm_fits(int H) { return H <= 4 * 1024; }

// Returns MOE_ERR_LIMIT when the row is too long for the fused kernel (the caller then runs the two
// kernels one after the other).
int launch_combine_norm(const float* y_by_slot, const int* slot_of, const int* topk_i, const float* topk_v,
                        float* e_agg, float* residual_x, const uint16_t* norm_weight, float* norm_out, int T, int K,
                        int H, hipStream_t stream) {
    if (!combine_norm_fits(H)) return MOE_ERR_LIMIT;
    const int H4 = H / 4;
    const int ni = ceil_div(H4, 256);
    auto y = reinterpret_cast<const float4*>(y_by_slot);
    auto e = reinterpret_cast<float4*>(e_agg);
    auto r = reinterpret_cast<float4*>(residual_x);
    auto o = reinterpret_cast<float4*>(norm_out);
    return combine_of(K, rows_past_cache(slot_of, T, K, H), [&](auto k, auto nt) {
        constexpr int KC = decltype(k)::value;
        constexpr bool NT = decltype(nt)::value;
        auto launch = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, dim3(T), dim3(256), 0, stream, y, slot_of, topk_i, topk_v, e, r, norm_weight, o, H4);
            return launch_status();
        };
        if (ni <= 1) return launch(combine_norm_kernel<1, KC, NT>);
        if (ni <= 2) return launch(combine_norm_kernel<2, KC, NT>);
        if (ni <= 3) return launch(combine_norm_kernel<3, KC, NT>);
        return launch(combine_norm_kernel<4, KC, NT>);
    });
}

int launch_rmsnorm(float* o, const float* x, const uint16_t* weight, int batch, int size, hipStream_t stream) {
    if (size <= 1024) hipLaunchKernelGGL(rmsnorm_kernel<1>, dim3(batch), dim3(256), 0, stream, o, x, weight, size);
    else if (size <= 3072) hipLaunchKernelGGL(rmsnorm_kernel<3>, dim3(batch), dim3(256), 0, stream, o, x, weight, size);
    else hipLaunchKernelGGL(rmsnorm_kernel<0>, dim3(batch), dim3(256), 0, stream, o, x, weight, size);
    return launch_status();
}

}  // namespace moe
