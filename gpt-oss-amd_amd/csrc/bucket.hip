// Expert token bucketing: histogram, exclusive scan, ordered compaction and the token-block map
// of the expert kernels in one launch.  Replaces count_tokens_per_expert /
// exclusive_scan_expert_offsets / compact_by_expert_kernel (src/hip/scheduler.hip:11-61), whose
// slot claim by atomicAdd leaves the order inside a bucket to chance; here every bucket lists its
// tokens in ascending token id (wave ballot + lane prefix count), so the output is a pure function
// of topk_i.
#include "common.h"
#include "kernels.h"

namespace moe {

// Copies of the histogram in LDS: a wave's atomic adds go to random experts, and adds of several
// lanes to one counter run one after the other; with one copy per lane (mod kHistCopies, the copy
// index being the bank) two lanes meet only when they are 32 apart.
constexpr int kHistCopies = 32;
static int hist_copies(int E) { return E <= 256 ? kHistCopies : E <= 512 ? 16 : 8; }

// V4: four experts per token and ids at 16-byte boundaries, up to kHeldTokens tokens: a thread holds the ids of its tokens in
// registers from one 16-byte load each, for the histogram and for the compaction (the general form reads them twice, word by word, a
// round trip per 8192 ids and per 4096 tokens).  32 experts, us, general : V4: 1000 tokens 9.2 : 8.6, 4096 tokens 12.6 : 9.8, 16384 tokens 35 : 20.
constexpr int kHeldTokens = 16 * 1024;

// grid = E blocks (one expert each), block = 1024 threads, dynamic LDS = (E * copies + E + 32) ints.
// The tile map lists the tiles of token_blocks in the order of TileOrder.  With map.second > 0 the same tiles are listed a second time,
// from index map.second of the three arrays, in bucket order (an expert's tiles together, the shortest one last).
// EVEN is a constant: as a runtime choice it cost the launches without a map 0.35 of 5.8 us.
template <bool V4, int EVEN>
__global__ __launch_bounds__(1024) void bucket_kernel(const int* __restrict__ topk_i,
                                                      const float* __restrict__ topk_v, int T, int K, int E,
                                                      int copies, int* __restrict__ expert_offsets,
                                                      int* __restrict__ tokens_flat,
                                                      float* __restrict__ weights_flat,
                                                      int* __restrict__ slot_of, TileMap map) {
    extern __shared__ int lds[];
    __shared__ int wave_cnt[4 * 16];  // matches per wave of the four compaction steps in flight
    int* hist = lds;                  // [E]
    int* scal = lds + E + 16;         // [0] rows before this expert, [1] tiles before it, [2] tiles in all,
                                      // [3] tiles ahead of this expert's full ones in the map's order, [4] ahead of its last one
    int* hist_c = lds + E + 32;       // [E][copies]
    const int e = blockIdx.x;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int A = T * K;
    constexpr int HELD = V4 ? kHeldTokens / 1024 : 1;
    int4 held[HELD];
    if constexpr (V4) {
#pragma unroll
        for (int u = 0; u < HELD; ++u) {
            const int t = u * 1024 + tid;
            held[u] = make_int4(-1, -1, -1, -1);
            if (u * 1024 < T && t < T) held[u] = reinterpret_cast<const int4*>(topk_i)[t];
        }
    }

    for (int i = tid; i < E * copies; i += blockDim.x) hist_c[i] = 0;
    if (tid < 8) scal[tid] = 0;
    __syncthreads();
    const int my_copy = tid & (copies - 1);
    auto count = [&](int id) {
        if ((unsigned)id < (unsigned)E) atomicAdd(&hist_c[id * copies + my_copy], 1);
    };
    if constexpr (V4) {
#pragma unroll
        for (int u = 0; u < HELD; ++u)
            if (u * 1024 < T) {
                count(held[u].x);
                count(held[u].y);
                count(held[u].z);
                count(held[u].w);
            }
    }
    // eight loads per thread in flight: the pass costs memory round trips, not adds
    for (int a0 = V4 ? A : tid; a0 < A; a0 += 8 * 1024) {
        int id[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) id[u] = a0 + u * 1024 < A ? topk_i[a0 + u * 1024] : -1;
#pragma unroll
        for (int u = 0; u < 8; ++u)
            count(id[u]);
    }
    __syncthreads();
    for (int i = tid; i < E; i += blockDim.x) {
        int c = 0;
        for (int j = 0; j < copies; ++j) c += hist_c[i * copies + ((j + i) & (copies - 1))];  // rotated: no common bank
        hist[i] = c;
    }
    __syncthreads();
    const int my_cnt = hist[e];
    const bool mapped = map.tile_tokens > 0;
    const TokenBlocks mine = mapped ? token_blocks<EVEN>(map.tile_tokens, my_cnt) : TokenBlocks{};
    {
        int rows_before = 0, tiles_before = 0, tiles_all = 0, ahead_of_full = 0, ahead_of_last = 0;
        const TileOrder<EVEN> order{map.tile_tokens, map.by_size};
        for (int i = tid; i < E; i += blockDim.x) {
            const int c = hist[i];
            if (i < e) rows_before += c;
            if (mapped) {
                const TokenBlocks b = token_blocks<EVEN>(map.tile_tokens, c);
                const int tiles = b.full + (b.rem > 0);
                tiles_all += tiles;
                if (i < e) tiles_before += tiles;
                ahead_of_full += order.ahead_of_full(b, i, mine, e);
                ahead_of_last += order.ahead_of_last(b, i, mine, e);
            }
        }
        // wave sums first, one add per wave and quantity (an atomic add of a different value per lane
        // is carried out lane by lane)
        int sums[5] = {rows_before, tiles_before, tiles_all, ahead_of_full, ahead_of_last};
        if (wave * 64 < E) {  // wave-uniform: later waves hold zeros
#pragma unroll
            for (int i = 0; i < 5; ++i) {
                const int total = wave_sum(sums[i]);
                if (lane == 0 && total) atomicAdd(&scal[i], total);
            }
        }
    }
    __syncthreads();
    const int my_off = scal[0];
    if (tid == 0) {
        expert_offsets[e] = my_off;
        if (e == E - 1) expert_offsets[E] = my_off + my_cnt;
    }
    if (mapped) {
        const int nb = mine.rows, my_full = mine.full, my_rem = mine.rem;
        for (int j = tid; j < my_full; j += blockDim.x) {
            map.tile_expert[scal[3] + j] = e;
            map.tile_row0[scal[3] + j] = my_off + j * nb;
            map.tile_rows[scal[3] + j] = nb;
        }
        if (my_rem > 0 && tid == 0) {
            const int at = scal[4];
            map.tile_expert[at] = e;
            map.tile_row0[at] = my_off + my_full * nb;
            map.tile_rows[at] = my_rem;
        }
        if (map.second > 0) {  // the same tiles in bucket order: an expert's tiles together, its partial one last
            const int first = map.second + scal[1];
            for (int j = tid; j < my_full + (my_rem > 0); j += blockDim.x) {
                map.tile_expert[first + j] = e;
                map.tile_row0[first + j] = my_off + j * nb;
                map.tile_rows[first + j] = min(nb, my_cnt - j * nb);
            }
        }
        if (e == E - 1 && tid == 0) *map.n_tiles = scal[2];
    }

    // ordered compaction: tokens visited in ascending id, 1024 tokens per step; the ids of four steps
    // are fetched together (K <= 8 per token)
    int base = my_off;
    auto steps = [&](int t00, auto ids_of) {  // tokens t00 .. t00 + 4095
        int mk4[4];
        float wv4[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            int ids[8];
            ids_of(u, t00 + u * 1024 + tid, ids);
            int mk = -1;
#pragma unroll
            for (int k = 7; k >= 0; --k) mk = ids[k] == e ? k : mk;  // the first k that names this expert
            mk4[u] = mk;
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {  // the matching routing weights, again before anything waits
            const int t = t00 + u * 1024 + tid;
            wv4[u] = mk4[u] >= 0 ? topk_v[(size_t)t * K + mk4[u]] : 0.f;
        }
        // the four steps' wave counts go through LDS together: one exchange (two barriers) per 4096 tokens
        int prefix4[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const unsigned long long ballot = __ballot(mk4[u] >= 0);
            prefix4[u] = __popcll(ballot & ((1ull << lane) - 1ull));
            if (lane == 0) wave_cnt[u * 16 + wave] = __popcll(ballot);
        }
        __syncthreads();
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int t = t00 + u * 1024 + tid;
            int wave_base = 0, total = 0;
#pragma unroll
            for (int w = 0; w < 16; ++w) {
                const int c = wave_cnt[u * 16 + w];
                if (w < wave) wave_base += c;
                total += c;
            }
            if (mk4[u] >= 0) {
                const int dst = base + wave_base + prefix4[u];
                tokens_flat[dst] = t;
                weights_flat[dst] = wv4[u];
                if (slot_of) slot_of[(size_t)t * K + mk4[u]] = dst;
            }
            base += total;
        }
        __syncthreads();
    };
    if constexpr (V4) {
#pragma unroll
        for (int h = 0; h < HELD / 4; ++h)
            if (4096 * h < T)  // block-uniform
                steps(4096 * h, [&](int u, int, int(&ids)[8]) {
                    const int4 v = held[4 * h + u];
                    ids[0] = v.x;
                    ids[1] = v.y;
                    ids[2] = v.z;
                    ids[3] = v.w;
                    ids[4] = ids[5] = ids[6] = ids[7] = -1;
                });
    } else {
        for (int t00 = 0; t00 < T; t00 += 4 * 1024)
            steps(t00, [&](int, int t, int(&ids)[8]) {
#pragma unroll
                for (int k = 0; k < 8; ++k) ids[k] = (t < T && k < K) ? topk_i[(size_t)t * K + k] : -1;
            });
    }
}

int launch_bucket(const int* topk_i, const float* topk_v, int T, int K, int E, int* expert_offsets,
                  int* tokens_flat, float* weights_flat, int* slot_of, TileMap map, hipStream_t stream) {
    const int copies = hist_copies(E);
    const size_t lds = (size_t)(E * copies + E + 32) * sizeof(int);
    auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(E), dim3(1024), lds, stream, topk_i, topk_v, T, K, E, copies, expert_offsets, tokens_flat,
                           weights_flat, slot_of, map);
    };
    const bool v4 = K == 4 && T <= kHeldTokens && ((uintptr_t)topk_i & 15u) == 0;
    if (map.even == kPrefillStep) launch(v4 ? bucket_kernel<true, kPrefillStep> : bucket_kernel<false, kPrefillStep>);
    else if (map.even == kPrefillStepBf16) launch(v4 ? bucket_kernel<true, kPrefillStepBf16> : bucket_kernel<false, kPrefillStepBf16>);
    else launch(v4 ? bucket_kernel<true, 0> : bucket_kernel<false, 0>);
    return launch_status();
}

// Y[row,:] = X[idx[row],:], fp32 rows of H (H % 4 == 0).  src/hip/scheduler.hip:63-85.
__global__ void gather_rows_kernel(const float4* __restrict__ X, const int* __restrict__ idx,
                                   float4* __restrict__ Y, int rows, int H4) {
    const int row = blockIdx.y;
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (row >= rows || c >= H4) return;
    Y[(size_t)row * H4 + c] = X[(size_t)idx[row] * H4 + c];
}

// One grid row per table row: launched in slabs of kMaxGridRows rows (the grid's y limit).
constexpr int kMaxGridRows = 65535;

int launch_gather_rows(const float* X, const int* idx, float* Y, int rows, int H, hipStream_t stream) {
    const int H4 = H / 4;
    for (int r0 = 0; r0 < rows; r0 += kMaxGridRows) {
        const int n = rows - r0 < kMaxGridRows ? rows - r0 : kMaxGridRows;
        hipLaunchKernelGGL(gather_rows_kernel, dim3(ceil_div(H4, 256), n), dim3(256), 0, stream,
                           reinterpret_cast<const float4*>(X), idx + r0, reinterpret_cast<float4*>(Y) + (size_t)r0 * H4, n,
                           H4);
    }
    return launch_status();
}

// X[idx[row],:] = Y[row,:]: the inverse of gather_rows (rows of a compact batch back to the table
// rows they were gathered from; idx must not repeat).
__global__ void scatter_rows_kernel(const float4* __restrict__ Y, const int* __restrict__ idx,
                                    float4* __restrict__ X, int rows, int H4) {
    const int row = blockIdx.y;
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (row >= rows || c >= H4) return;
    X[(size_t)idx[row] * H4 + c] = Y[(size_t)row * H4 + c];
}

int launch_scatter_rows(const float* Y, const int* idx, float* X, int rows, int H, hipStream_t stream) {
    const int H4 = H / 4;
    for (int r0 = 0; r0 < rows; r0 += kMaxGridRows) {
        const int n = rows - r0 < kMaxGridRows ? rows - r0 : kMaxGridRows;
        hipLaunchKernelGGL(scatter_rows_kernel, dim3(ceil_div(H4, 256), n), dim3(256), 0, stream,
                           reinterpret_cast<const float4*>(Y) + (size_t)r0 * H4, idx + r0, reinterpret_cast<float4*>(X), n,
                           H4);
    }
    return launch_status();
}

// (expert, row_offset, row_count) triples of the non-empty experts, ascending expert id
// (entry format of src/hip/scheduler.hip:163-166).  One wave; ballot + prefix count per 64 experts.
__global__ __launch_bounds__(64) void work_queue_kernel(const int* __restrict__ expert_offsets, int E,
                                                        int* __restrict__ work_queue,
                                                        int* __restrict__ work_count) {
    const int lane = threadIdx.x;
    int base = 0;
    for (int e0 = 0; e0 < E; e0 += 64) {
        const int e = e0 + lane;
        int off = 0, ne = 0;
        if (e < E) {
            off = expert_offsets[e];
            ne = expert_offsets[e + 1] - off;
        }
        const unsigned long long ballot = __ballot(ne > 0);
        if (ne > 0) {
            const int dst = base + __popcll(ballot & ((1ull << lane) - 1ull));
            work_queue[3 * dst + 0] = e;
            work_queue[3 * dst + 1] = off;
            work_queue[3 * dst + 2] = ne;
        }
        base += __popcll(ballot);
    }
    if (lane == 0) *work_count = base;
}

int launch_build_work_queue(const int* expert_offsets, int E, int* work_queue, int* work_count,
                            hipStream_t stream) {
    hipLaunchKernelGGL(work_queue_kernel, dim3(1), dim3(64), 0, stream, expert_offsets, E, work_queue, work_count);
    return launch_status();
}

}  // namespace moe
