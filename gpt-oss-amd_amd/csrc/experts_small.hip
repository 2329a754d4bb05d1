// Expert GEMMs of the MoE block for batches that give an expert a handful of rows: every wave streams 16 weight rows of
// one expert over the whole contraction range on its own.  Replaces moe_mlp1_swiglu_mfma_kernel (src/hip/moe.hip:9-235)
// and moe_mlp2_scatter_mfma_kernel (src/hip/moe.hip:261-512) at those sizes.
//
// What bounds it: the weights of the experts that got a row, and below that the launch's chain of latencies (expert ids,
// then weights and activation rows, then the stores).  The producer/consumer kernels cut an expert into blocks of 320 to
// 768 weight rows, one to a compute unit: one token's four experts occupy 32 of 256 compute units, and the 20 experts of
// seven tokens are 320 blocks, i.e. two rounds for the work of 1.25.  Here the bucket's few rows are staged once, whole,
// the stage barriers go, and the work is cut by MFMA tile.  Gate/up + down launch, us: one token, E = 32 MXFP4 25 + 15 -> 10 + 7
// (3.4 TB/s in the larger: ids, rows and weights are a chain of three round trips), bf16 124 + 65 -> 25 + 14; 7 tokens, E = 32
// bf16 138 + 66 -> 105 + 52 (6.2 TB/s); 33 tokens, E = 128 MXFP4 116 + 70 -> 108 + 59 (6.8).  Two tiles a wave, and three
// blocks a compute unit instead of two: no faster.
#include <type_traits>

#include "expert_tiles.h"
#include "topk.h"

namespace moe {

namespace {

constexpr int kSmallWaves = 8;         // at most
constexpr int kSmallMaxAssign = 512;   // one expert id per thread of a full block
constexpr int kSmallRows = 32;         // bucket rows of one pass over the weights (two token tiles)
constexpr int kSmallLds = 64 * 1024;   // of staged activations, so that two blocks fit a compute unit
constexpr int kSmallGroup = 8;         // a phase (what is staged at once) is a multiple of so many stages

// Tile `tile` (16 weight rows, order of tile_row_in_group) against the nrows <= 16 NT bucket rows starting at row0.  The
// activations of `per_phase` stages of 128 contraction elements are staged at a time, rows_img (nrows rounded up to four)
// rows to a stage, 256 bytes each, chunk c of row r at position ws_pos(c) ^ (r % 16).  All waves of the block call this
// with the same bucket; those without a tile (active false) only stage.
// ACT_F32: the rows are fp32 (rows slot_of_row(i) of a.act_f32), rounded to bf16 while they are staged.
template <int FMT, int NT, int EPI, bool ACT_F32, class SlotFn>
MOE_DEVICE void small_tile(const ExpertGemmArgs& a, uint8_t* lds, int e, SlotFn slot_of_row, int nrows, int tile, bool active,
                           int lds_bytes) {
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int waves = blockDim.x >> 6;
    const int q = lane & 15;
    const int g = lane >> 4;
    const int K = a.K;
    const int n_stages = ceil_div(K, kStageElems);
    const int rows_img = (nrows + 3) & ~3;
    const int stage_bytes = rows_img * 256;
    const int per_phase = min(n_stages, lds_bytes / stage_bytes / kSmallGroup * kSmallGroup);
    // token of assignment s = s / assign_div, as a float multiplication (exact for s < 4096, assign_div <= 8)
    const float inv_div = 1.0f / (float)a.assign_div;
    // stages [s0, s0 + per_phase) to LDS: instruction n moves four rows of one stage, whole 256-byte pieces; the waves
    // take them in turn
    auto stage_rows = [&](int s0) {
        const int quads = rows_img >> 2;
        const int n_instr = min(per_phase, n_stages - s0) * quads;
        int st = wave / quads, rq = wave - st * quads;  // wave-uniform
        const int dst_step = waves / quads, dq_step = waves - dst_step * quads;
        auto next = [&]() {
            st += dst_step;
            rq += dq_step;
            if (rq >= quads) {
                rq -= quads;
                ++st;
            }
        };
        // the lane's row, and the contraction element at its position (of the padding if it lies past the row)
        auto slot = [&]() { return slot_of_row(min(rq * 4 + g, nrows - 1)); };
        auto elem = [&]() { return (s0 + st) * kStageElems + 8 * ws_chunk_at<FMT>(q ^ ((rq * 4 + g) & 15)); };
        if constexpr (ACT_F32) {
            constexpr int B = 4;  // loads of a batch are in flight together
            for (int n = wave; n < n_instr; n += B * waves) {
                float4 x[B][2];
                bool live[B];
#pragma unroll
                for (int i = 0; i < B; ++i) {
                    if (n + i * waves < n_instr) {  // wave-uniform
                        const int k = elem();
                        live[i] = k < K;
                        const float4* src = reinterpret_cast<const float4*>(a.act_f32 + (size_t)slot() * K + (live[i] ? k : 0));
                        x[i][0] = src[0];
                        x[i][1] = src[1];
                    }
                    next();
                }
#pragma unroll
                for (int i = 0; i < B; ++i)
                    if (n + i * waves < n_instr) {
                        u32x4 v = {pack_bf16x2(x[i][0].x, x[i][0].y), pack_bf16x2(x[i][0].z, x[i][0].w),
                                   pack_bf16x2(x[i][1].x, x[i][1].y), pack_bf16x2(x[i][1].z, x[i][1].w)};
                        // zeros past the row: the weights count as zero there, and zero times an infinity or a NaN
                        // from elsewhere in the row would reach all of its outputs (bf16 never multiplies them)
                        if (FMT == FMT_MXFP4 && !live[i]) v = u32x4{0u, 0u, 0u, 0u};
                        *reinterpret_cast<u32x4*>(lds + (size_t)(n + i * waves) * 1024 + lane * 16) = v;
                    }
            }
        } else {
            for (int n = wave; n < n_instr; n += waves) {
                const int s = slot();
                const int src = a.gather ? (int)(((float)s + 0.5f) * inv_div) : s;
                const int k = elem();  // a position past the row re-reads its start: its weights count as zero
                dma16(reinterpret_cast<const uint8_t*>(a.act + (size_t)src * K + (k < K ? k : 0)), lds + (size_t)n * 1024);
                next();
            }
        }
    };
    auto restage = [&](int s0) {  // all waves are past the reads of the stages before
        stage_rows(s0);
        wait_vmcnt<0>();
        __syncthreads();
    };
    if (!active) {
        restage(0);
        for (int s0 = per_phase; s0 < n_stages; s0 += per_phase) {
            __syncthreads();
            restage(s0);
        }
        return;
    }
    const int group = tile >> 2;
    const int r0 = tile & 3;
    uint2 bias_raw[1];
    load_bias<1>(a, e, group, r0, bias_raw);
    // the columns past the bucket's end take its last staged row again; they are never stored.  MFMA step j of lane group g
    // reads position 2g + (j & 1) + 8 (j >> 1) of its row in either format's image: the steps differ in address bits 4 and 7
    uint32_t b_lane[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        const int row = min(t * 16 + q, rows_img - 1);
        b_lane[t] = (uint32_t)(row * 256 + ((ws_pos<FMT>(ws_chunk<FMT>(0, g)) ^ (row & 15)) << 4));
    }
    int phase0 = 0;  // first stage that is staged now
    uint32_t b_at[NT];
    auto at_stage = [&](int s) {
        uint32_t off = (uint32_t)(s - phase0) * (uint32_t)stage_bytes;
        asm volatile("" : "+s"(off));  // kept a scalar: otherwise every stage's addresses are held in registers of their own
#pragma unroll
        for (int t = 0; t < NT; ++t) b_at[t] = b_lane[t] + off;
    };
    auto b_frag = [&](int j, int t) {
        return *reinterpret_cast<const u32x4*>(lds + (b_at[t] ^ (uint32_t)((j & 1) * 16 + (j >> 1) * 128)));
    };
    auto next_phase = [&](int s) {  // stage s is the next to be computed
        if (s == phase0 + per_phase) {
            phase0 = s;
            __syncthreads();
            restage(s);
        }
    };
    f32x4 acc[1][NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[0][t] = f32x4{0.f, 0.f, 0.f, 0.f};

    if constexpr (FMT == FMT_BF16) {
        // Weights as in ws_consumer: pairs of MFMA steps, each fetched by two non-temporal loads of whole 128-byte lines
        // whose lane halves trade places at use; a ring of four pairs (two stages).
        constexpr int D = 4;
        const int n_pairs = K / 64;
        const __amdgpu_buffer_rsrc_t w_rsrc = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<uint16_t*>(reinterpret_cast<const uint16_t*>(a.w) + (size_t)e * a.w_expert_stride), 0,
            (int)((uint32_t)a.rows * (uint32_t)K * 2u), 0x00020000);
        const uint32_t a_tile = (uint32_t)(group * 64 + tile_row_in_group(r0, 0)) * (uint32_t)K * 2u;
        const uint32_t a_lane = (uint32_t)(tile_row_in_group(0, q & 7) * K + 8 * (2 * g + (q >> 3))) * 2u;
        const uint32_t second_half = 32u * (uint32_t)K * 2u;  // tile row q + 8 is weight row + 32 (tile_row_in_group)
        u32x4 ar[D][2];
        auto load_a = [&](int slot, int pair) {
            const uint32_t off = a_tile + (uint32_t)(pair < n_pairs ? pair : 0) * 128u;  // past the end: unused
#pragma unroll
            for (int i = 0; i < 2; ++i)
                ar[slot][i] = __builtin_amdgcn_raw_buffer_load_b128(w_rsrc, (int)a_lane, (int)(off + second_half * i), 2 /* nt */);
        };
#pragma unroll
        for (int i = 0; i < D - 1; ++i) load_a(i, i);
        restage(0);
        auto pair_step = [&](int u, int pair) {
            load_a((u + D - 1) % D, pair + D - 1);
            __builtin_amdgcn_sched_barrier(0);  // the loads are issued here, three pairs ahead of their use
            if ((u & 1) == 0) at_stage(pair >> 1);
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                u32x4 av;
#pragma unroll
                for (int d = 0; d < 4; ++d)
                    av[d] = h == 0 ? (uint32_t)__builtin_amdgcn_update_dpp((int)ar[u][0][d], (int)ar[u][1][d], 0x128, 0xF, 0xC, false)
                                   : (uint32_t)__builtin_amdgcn_update_dpp((int)ar[u][1][d], (int)ar[u][0][d], 0x128, 0xF, 0x3, false);
#pragma unroll
                for (int t = 0; t < NT; ++t) acc[0][t] = mfma_16x16x32(av, b_frag(2 * (u & 1) + h, t), acc[0][t]);
            }
        };
        const int full = n_pairs / D;
        for (int i = 0; i < full; ++i) {
            next_phase(2 * i);
#pragma unroll
            for (int u = 0; u < D; ++u) pair_step(u, D * i + u);
        }
        if (D * full < n_pairs) {
            next_phase(2 * full);
            pair_step(0, D * full);
            if (D * full + 1 < n_pairs) pair_step(1, D * full + 1);
            if (D * full + 2 < n_pairs) pair_step(2, D * full + 2);
        }
    } else {
        // Weights as in ws_consumer: one 1 KiB chunk per stage, one scale dword per four stages, reads past the tile only
        // where the scale byte is 0 or nobody looks; a ring of eight stages, scales one group of eight ahead.
        constexpr int D = kSmallGroup;
        const int G = K / 32;
        const uint32_t wtile = (uint32_t)tile * (uint32_t)G * 256u;
        const uint32_t stile = (uint32_t)tile * (uint32_t)ceil_div(ceil_div(G, 4), 4) * 256u;
        const __amdgpu_buffer_rsrc_t w_rsrc = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<uint8_t*>(reinterpret_cast<const uint8_t*>(a.w) + (size_t)e * a.w_expert_stride), 0,
            (int)a.w_expert_stride, 0x00020000);
        const __amdgpu_buffer_rsrc_t s_rsrc = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<uint8_t*>(a.w_scales + (size_t)e * a.s_expert_stride), 0, (int)a.s_expert_stride, 0x00020000);
        u32x4 araw[D];
        uint32_t sw_cur[2], sw_nxt[2];
        auto load_a = [&](int slot, int s) {
            araw[slot] = __builtin_amdgcn_raw_buffer_load_b128(w_rsrc, lane * 16, (int)(wtile + (uint32_t)s * 1024u), 2 /* nt */);
        };
        auto load_scales = [&](uint32_t (&dst)[2], int grp) {
#pragma unroll
            for (int i = 0; i < 2; ++i)
                dst[i] = __builtin_amdgcn_raw_buffer_load_b32(s_rsrc, lane * 4, (int)(stile + (uint32_t)(2 * grp + i) * 256u), 0);
        };
        load_scales(sw_cur, 0);
#pragma unroll
        for (int i = 0; i < D - 1; ++i) load_a(i, i);
        restage(0);
        auto stage = [&](auto i_tag, int s, auto more_tag) {
            constexpr int i = decltype(i_tag)::value;
            if constexpr (decltype(more_tag)::value) load_a((i + D - 1) % D, s + D - 1);
            __builtin_amdgcn_sched_barrier(0);  // the load is issued here, seven stages ahead of its use
            at_stage(s);
            const float sc = mxfp4_scale_to_f32((sw_cur[i >> 2] >> (8 * (i & 3))) & 0xFFu);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                uint32_t d[4];
                mxfp4_dword_to_bf16x8(araw[i][j], sc, d);
                const u32x4 av = {d[0], d[1], d[2], d[3]};
#pragma unroll
                for (int t = 0; t < NT; ++t) acc[0][t] = mfma_16x16x32(av, b_frag(j, t), acc[0][t]);
            }
            // the stage's products are formed here: the compiler otherwise gathers the (dependent) MFMAs of all stages of
            // the group behind their conversions and spills the operands
#pragma unroll
            for (int t = 0; t < NT; ++t) asm volatile("" : "+v"(acc[0][t]));
        };
        const int full = n_stages / D;
        for (int i = 0; i < full; ++i) {
            next_phase(D * i);
            load_scales(sw_nxt, i + 1);
            const int s = D * i;
            stage(std::integral_constant<int, 0>{}, s, std::true_type{});
            stage(std::integral_constant<int, 1>{}, s + 1, std::true_type{});
            stage(std::integral_constant<int, 2>{}, s + 2, std::true_type{});
            stage(std::integral_constant<int, 3>{}, s + 3, std::true_type{});
            stage(std::integral_constant<int, 4>{}, s + 4, std::true_type{});
            stage(std::integral_constant<int, 5>{}, s + 5, std::true_type{});
            stage(std::integral_constant<int, 6>{}, s + 6, std::true_type{});
            stage(std::integral_constant<int, 7>{}, s + 7, std::true_type{});
            sw_cur[0] = sw_nxt[0];
            sw_cur[1] = sw_nxt[1];
        }
        const int s = D * full, tail = n_stages - s;  // all of the tail's weights are in the ring
        if (tail > 0) {
            next_phase(s);
            auto last = [&](auto u) {
                if (tail > decltype(u)::value) stage(u, s + decltype(u)::value, std::false_type{});
            };
            last(std::integral_constant<int, 0>{});
            last(std::integral_constant<int, 1>{});
            last(std::integral_constant<int, 2>{});
            last(std::integral_constant<int, 3>{});
            last(std::integral_constant<int, 4>{});
            last(std::integral_constant<int, 5>{});
            last(std::integral_constant<int, 6>{});
        }
    }
    stream_epilogue<1, NT, EPI>(a, acc, e, slot_of_row, nrows, group, r0, bias_raw);
}

// All rows of a bucket, max_rows (a multiple of four that the LDS holds eight stages of) to a pass over the weights.
template <int FMT, int EPI, bool ACT_F32, class SlotFn>
MOE_DEVICE void small_rows(const ExpertGemmArgs& a, uint8_t* lds, int e, SlotFn slot_of_row, int n_rows, int rb, int max_rows,
                           int lds_bytes) {
    const int tile = rb * (blockDim.x >> 6) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const bool active = tile < a.rows / 16;
    for (int row0 = 0; row0 < n_rows; row0 += max_rows) {
        if (row0 > 0) __syncthreads();  // everyone is done with the staged rows
        const int nrows = min(max_rows, n_rows - row0);
        auto slot = [&](int i) { return slot_of_row(row0 + i); };
        if (nrows > 16) small_tile<FMT, 2, EPI, ACT_F32>(a, lds, e, slot, nrows, tile, active, lds_bytes);
        else small_tile<FMT, 1, EPI, ACT_F32>(a, lds, e, slot, nrows, tile, active, lds_bytes);
    }
}

// Block index -> (i-th expert that has a row, row block).  Experts are counted off in the assignment list itself, so blocks
// of experts without rows (most of them at one token) are neither launched nor scheduled between the others.
// grid = min(E, assignments) x row blocks, block = 64 waves, one tile of 16 weight rows per wave.
// Three blocks to a compute unit (with 84 registers two, 7 tokens, 32 and 128 MXFP4 experts, us, 50.7 and 71.2 instead of 49.4 and 68.8).
template <int FMT, int EPI>
__global__ __launch_bounds__(64 * kSmallWaves, 6) void expert_small_kernel(ExpertGemmArgs a, int max_rows, int lds_bytes) {
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    __shared__ uint32_t present[32];
    __shared__ int counts[8];
    __shared__ int bucket[kSmallMaxAssign];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int waves = blockDim.x >> 6;
    const int ordinal = blockIdx.x / a.row_blocks;
    const int rb = blockIdx.x - ordinal * a.row_blocks;
    if constexpr (EPI == EPI_SWIGLU_BF16) {
        if (a.scores) {  // at most 64 assignments: the list goes through bucket[]
            const int T = a.n_assign / a.assign_div;
            for (int t = wave; t < T; t += waves) {
                float my_v;
                int my_i;
                select_topk(a.scores + (size_t)t * a.n_experts, a.n_experts, a.assign_div, lane, my_v, my_i);
                if (lane < a.assign_div) bucket[t * a.assign_div + lane] = my_i;
                if (blockIdx.x == 0)
                    write_topk(my_v, my_i, a.assign_div, lane, 1, a.topk_v_out + (size_t)t * a.assign_div,
                               a.topk_i_out + (size_t)t * a.assign_div);
            }
            __syncthreads();
        }
    }
    const int* const list = EPI == EPI_SWIGLU_BF16 && a.scores ? bucket : a.topk_i;
    // chunk c of 64 assignments: wave c % waves (a block of four waves takes two chunks each)
    int ids[kSmallMaxAssign / 64 / 4];
#pragma unroll
    for (int p = 0; p < 2; ++p) {
        const int s = (p * waves + wave) * 64 + lane;
        // an id that names no expert is skipped, as by the other kernels: the down GEMM entry takes the list from its caller
        const int id = s < a.n_assign ? list[s] : -1;
        ids[p] = (unsigned)id < (unsigned)a.n_experts ? id : -1;
    }
    if (threadIdx.x < 32) present[threadIdx.x] = 0u;
    __syncthreads();
#pragma unroll
    for (int p = 0; p < 2; ++p)
        if (ids[p] >= 0) atomicOr(&present[ids[p] >> 5], 1u << (ids[p] & 31));
    __syncthreads();
    int e;
    {
        uint32_t word = lane < 32 ? present[lane] : 0u;
        uint32_t incl = __popc(word);
#define MOE_STEP(C, M) incl += dpp_move<C, M>(0u, incl);
        MOE_DPP_STEPS(MOE_STEP)
#undef MOE_STEP
        if (ordinal >= (int)__builtin_amdgcn_readlane(incl, 63)) return;  // block-uniform
        const int w = __popcll(__ballot((int)incl <= ordinal));  // words whose experts all come before
        word = __builtin_amdgcn_readlane(word, w);
        int skip = ordinal - ((int)__builtin_amdgcn_readlane(incl, w) - __popc(word));
        while (skip-- > 0) word &= word - 1u;
        e = 32 * w + __builtin_ctz(word);
    }
    int n_bucket = 0;
    {
        unsigned long long match[2];
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            match[p] = __ballot(ids[p] == e);
            const int c = p * waves + wave;
            if (lane == 0 && c < 8) counts[c] = __popcll(match[p]);
        }
        __syncthreads();
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            int base = 0;
            for (int c = 0; c < 8; ++c) {
                const int n = __builtin_amdgcn_readfirstlane(counts[c]);
                if (c < p * waves + wave) base += n;
                if (p == 0) n_bucket += n;
            }
            if (ids[p] == e) bucket[base + __popcll(match[p] & ((1ull << lane) - 1ull))] = (p * waves + wave) * 64 + lane;
        }
    }
    __syncthreads();
    small_rows<FMT, EPI, false>(a, lds, e, [&](int i) { return bucket[i]; }, n_bucket, rb, max_rows, lds_bytes);
}

// The same for the entries that keep the reference's data flow: queue entries (expert, row_offset, row_count), fp32 rows by
// slot.  grid = entries x row blocks.
template <int FMT, int EPI>
__global__ __launch_bounds__(64 * kSmallWaves, 4) void expert_small_queue_kernel(ExpertGemmArgs a, int max_rows, int lds_bytes) {
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    const int item = blockIdx.x / a.row_blocks;
    const int rb = blockIdx.x - item * a.row_blocks;
    const int* entry = a.work_queue + 3 * (size_t)(a.work_start + item);
    const int off = entry[1];
    small_rows<FMT, EPI, true>(a, lds, entry[0], [&](int i) { return off + i; }, entry[2], rb, max_rows, lds_bytes);
}

// ---- down GEMM of up to 16 assignments: a wave per (assignment, tile of 16 weight rows); the waves of a block share the tile --------
// What bounds it: round trips (ids and rows, then weights, then the stores).  The block that holds all of a token's rows of its
// tile also combines them, which takes the combine's launch away; a wave needs nobody else's row until then.  MXFP4, us, down
// + combine, two launches : one: 1 token 7.7 + 3.8 : 8.3, 2 tokens 9.9 + 3.9 : 10.4.  The gate/up GEMM in this form was no faster (1
// token 12.2 : 11.9), and neither was a whole MXFP4 tile requested at once instead of a ring of eight stages: straight-line code for 24
// stages is fetched anew by every launch.
constexpr int kTinyAssign = 16;

// The wave's activation row, as it is (the 16 columns of the product are this one row), zeros past its end.  Loaded ahead of the
// expert's id, stored to LDS before the weights are requested.
constexpr int kTinyRowLoads = 6;  // loads of 512 values: rows of up to 3072 values, what is longer in a loop
MOE_DEVICE void tiny_row_load(u32x4 (&xr)[kTinyRowLoads], const uint16_t* row, int K) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int i = 0; i < kTinyRowLoads; ++i) {
        const int k = 512 * i + 8 * lane;
        xr[i] = k < K ? *reinterpret_cast<const u32x4*>(row + k) : u32x4{0u, 0u, 0u, 0u};
    }
}
MOE_DEVICE void tiny_row_store(const u32x4 (&xr)[kTinyRowLoads], uint8_t* row_lds, const uint16_t* row, int K) {
    const int lane = threadIdx.x & 63;
    const int padded = ceil_div(K, kStageElems) * kStageElems;
#pragma unroll
    for (int i = 0; i < kTinyRowLoads; ++i)
        if (512 * i + 8 * lane < padded) *reinterpret_cast<u32x4*>(row_lds + 1024 * i + 16 * lane) = xr[i];
    for (int k = 512 * kTinyRowLoads + 8 * lane; k < padded; k += 512)
        *reinterpret_cast<u32x4*>(row_lds + 2 * k) = k < K ? *reinterpret_cast<const u32x4*>(row + k) : u32x4{0u, 0u, 0u, 0u};
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();  // the wave's own LDS accesses are carried out in order
}

template <int FMT>
MOE_DEVICE f32x4 tiny_tile(const ExpertGemmArgs& a, const uint8_t* row_lds, int e, int tile) {
    const int lane = threadIdx.x & 63;
    const int q = lane & 15;
    const int g = lane >> 4;
    const int K = a.K;
    auto b_frag = [&](int s, int j) { return *reinterpret_cast<const u32x4*>(row_lds + s * 256 + ws_chunk<FMT>(j, g) * 16); };
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    if constexpr (FMT == FMT_BF16) {
        constexpr int D = 4;
        const int n_pairs = K / 64;
        const __amdgpu_buffer_rsrc_t w_rsrc = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<uint16_t*>(reinterpret_cast<const uint16_t*>(a.w) + (size_t)e * a.w_expert_stride), 0,
            (int)((uint32_t)a.rows * (uint32_t)K * 2u), 0x00020000);
        const uint32_t a_tile = (uint32_t)((tile >> 2) * 64 + tile_row_in_group(tile & 3, 0)) * (uint32_t)K * 2u;
        const uint32_t a_lane = (uint32_t)(tile_row_in_group(0, q & 7) * K + 8 * (2 * g + (q >> 3))) * 2u;
        const uint32_t second_half = 32u * (uint32_t)K * 2u;
        u32x4 ar[D][2];
        auto load_a = [&](int slot, int pair) {
            const uint32_t off = a_tile + (uint32_t)(pair < n_pairs ? pair : 0) * 128u;  // past the end: unused
#pragma unroll
            for (int i = 0; i < 2; ++i)
                ar[slot][i] = __builtin_amdgcn_raw_buffer_load_b128(w_rsrc, (int)a_lane, (int)(off + second_half * i), 2 /* nt */);
        };
#pragma unroll
        for (int i = 0; i < D - 1; ++i) load_a(i, i);
        for (int p0 = 0; p0 < n_pairs; p0 += D) {
#pragma unroll
            for (int u = 0; u < D; ++u) {
                load_a((u + D - 1) % D, p0 + u + D - 1);
                __builtin_amdgcn_sched_barrier(0);
                if (p0 + u < n_pairs) {  // wave-uniform
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        u32x4 av;
#pragma unroll
                        for (int d = 0; d < 4; ++d)
                            av[d] = h == 0 ? (uint32_t)__builtin_amdgcn_update_dpp((int)ar[u][0][d], (int)ar[u][1][d], 0x128, 0xF, 0xC, false)
                                           : (uint32_t)__builtin_amdgcn_update_dpp((int)ar[u][1][d], (int)ar[u][0][d], 0x128, 0xF, 0x3, false);
                        acc = mfma_16x16x32(av, b_frag((p0 + u) >> 1, 2 * (u & 1) + h), acc);
                    }
                }
            }
        }
    } else {
        const int G = K / 32;
        const int n_stages = ceil_div(K, kStageElems);
        const uint32_t wtile = (uint32_t)tile * (uint32_t)G * 256u;
        const uint32_t stile = (uint32_t)tile * (uint32_t)ceil_div(ceil_div(G, 4), 4) * 256u;
        const __amdgpu_buffer_rsrc_t w_rsrc = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<uint8_t*>(reinterpret_cast<const uint8_t*>(a.w) + (size_t)e * a.w_expert_stride), 0,
            (int)a.w_expert_stride, 0x00020000);
        const __amdgpu_buffer_rsrc_t s_rsrc = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<uint8_t*>(a.w_scales + (size_t)e * a.s_expert_stride), 0, (int)a.s_expert_stride, 0x00020000);
        constexpr int D = kSmallGroup;
        u32x4 araw[D];
        uint32_t sw_cur[2], sw_nxt[2];
        auto load_a = [&](int slot, int s) {
            araw[slot] = __builtin_amdgcn_raw_buffer_load_b128(w_rsrc, lane * 16, (int)(wtile + (uint32_t)s * 1024u), 2 /* nt */);
        };
        auto load_scales = [&](uint32_t (&dst)[2], int grp) {
#pragma unroll
            for (int i = 0; i < 2; ++i)
                dst[i] = __builtin_amdgcn_raw_buffer_load_b32(s_rsrc, lane * 4, (int)(stile + (uint32_t)(2 * grp + i) * 256u), 0);
        };
        load_scales(sw_cur, 0);
#pragma unroll
        for (int i = 0; i < D; ++i) load_a(i, i);
        for (int s0 = 0; s0 < n_stages; s0 += D) {
            load_scales(sw_nxt, s0 / D + 1);
#pragma unroll
            for (int i = 0; i < D; ++i) {
                if (s0 + i < n_stages) {  // wave-uniform
                    const float sc = mxfp4_scale_to_f32((sw_cur[i >> 2] >> (8 * (i & 3))) & 0xFFu);
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        uint32_t d[4];
                        mxfp4_dword_to_bf16x8(araw[i][j], sc, d);
                        acc = mfma_16x16x32(u32x4{d[0], d[1], d[2], d[3]}, b_frag(s0 + i, j), acc);
                    }
                }
                // reads past the tile only where the scale byte is 0 or nobody looks, as in small_tile
                load_a(i, s0 + i + D);
                __builtin_amdgcn_sched_barrier(0);
            }
            sw_cur[0] = sw_nxt[0];
            sw_cur[1] = sw_nxt[1];
        }
    }
    return acc;
}

// grid = tiles, block = 64 x assignments, dynamic LDS = assignments x padded row.
template <int FMT>
__global__ __launch_bounds__(64 * kTinyAssign, 4) void expert_tiny_down_kernel(ExpertGemmArgs a, int row_bytes) {
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    __shared__ float y[kTinyAssign][16];  // by token, then by rank of the expert id among the token's
    __shared__ float weight[kTinyAssign];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // the assignment
    const int g = lane >> 4;
    const int top = a.assign_div;
    const int t = wave / top, k = wave - t * top;
    const int tile = blockIdx.x;
    uint8_t* const row_lds = lds + (size_t)wave * row_bytes;
    const uint16_t* const row = a.act + (size_t)wave * a.K;
    u32x4 xr[kTinyRowLoads];
    tiny_row_load(xr, row, a.K);
    const int id = lane < top ? a.topk_i[t * top + lane] : 0x7FFFFFFF;
    const int e = __builtin_amdgcn_readlane(id, k);
    const int at = t * top + __popcll(__ballot(id < e || (id == e && lane < k)));
    if (lane == 0) weight[at] = a.combine_v[wave];
    tiny_row_store(xr, row_lds, row, a.K);
    uint2 bias_raw[1];
    const int group = tile >> 2, r0 = tile & 3;
    load_bias<1>(a, e, group, r0, bias_raw);
    const f32x4 acc = tiny_tile<FMT>(a, row_lds, e, tile);
    if ((lane & 15) == 0)  // all columns are the same row
        *reinterpret_cast<f32x4*>(&y[at][4 * g]) =
            f32x4{acc[0] + bf16_bits_to_f32(bias_raw[0].x & 0xFFFFu), acc[1] + bf16_bits_to_f32(bias_raw[0].x >> 16),
                  acc[2] + bf16_bits_to_f32(bias_raw[0].y & 0xFFFFu), acc[3] + bf16_bits_to_f32(bias_raw[0].y >> 16)};
    __syncthreads();
    // the weighted sum in ascending expert id, each step one fused multiply-add (combine_kernel)
    const int ct = threadIdx.x >> 4, r = threadIdx.x & 15;
    if (ct < a.n_assign / top) {
        // tile row 4 g + j is weight row g * 16 + r0 * 4 + j of the group (stream_epilogue)
        const size_t out = (size_t)ct * a.rows + group * 64 + (r >> 2) * 16 + r0 * 4 + (r & 3);
        const float before = a.residual_x ? a.residual_x[out] : 0.f;
        float sum = 0.f;
        for (int i = 0; i < top; ++i) sum = fmaf(y[ct * top + i][r], weight[ct * top + i], sum);
        a.e_agg[out] = sum;
        if (a.residual_x) a.residual_x[out] = before + sum;
    }
}

}  // namespace

// Assignments, and buffer descriptors that reach an expert's whole matrix (31-bit byte offsets).
bool expert_small_fits(int n_assign, int rows, int K, int format) {
    size_t bytes = 2ull * (size_t)rows * (size_t)K, scales = 0;
    if (format == FMT_MXFP4) mxfp4_tiled_bytes(rows, K, &bytes, &scales);
    return n_assign <= kSmallMaxAssign && bytes <= 0x7fffffffull;
}

// Every block of the gate/up launch finds the top-k of all tokens itself, a token to a wave: worth the router's second half while that
// is one token each.  Whole block, us, router and small kernels : this, MXFP4, E = 32, 1 token 30 : 24, 4 tokens 50 : 47, 8 tokens 61.5 : 59, 10
// tokens 68 : 69; E = 128, 1 token 34 : 25, 4 tokens 60 : 50, 8 tokens 87 : 80, 10 tokens 100 : 100, 16 tokens 131 : 134.  More experts, K = 8:
// blocks of 1024 x 1024, scores + finalize and small kernels : this, MXFP4, E = 256, 1 token 28 : 18, 8 tokens 50 : 44; E = 1000, 1 token 47 :
// 21, 8 tokens 73 : 52; bf16, E = 1000, 8 tokens 108 : 90.
bool expert_small_takes_scores(int n_tokens, int n_assign) { return n_tokens <= kSmallWaves && n_assign <= 64; }

// bf16 weights of 16 assignments load a compute unit longer than the combine's launch takes (4 tokens, E = 32, two launches : one, us,
// MXFP4 18.7 : 17.3, bf16 49.0 : 49.9; 3 tokens 16.2 : 13.7 and 40.3 : 38.5).
bool expert_small_combines(int n_assign, int K, int format) {
    return n_assign <= (format == FMT_BF16 ? 12 : kTinyAssign) && (long long)n_assign * K <= 64 * 1024 - kTinyAssign * kStageElems;
}

int launch_expert_small(const ExpertGemmArgs& a, int epi, hipStream_t stream) {
    const bool queue = a.work_queue != nullptr;
    if (a.rows % 64 != 0 || a.K % (a.format == FMT_BF16 ? 64 : 32) != 0 || (!queue && !a.topk_i)) return MOE_ERR_SHAPE;
    if (!expert_small_fits(queue ? 0 : a.n_assign, a.rows, a.K, a.format)) return MOE_ERR_LIMIT;
    if (!queue && (a.assign_div <= 0 || a.assign_div > 8 || a.n_experts > 1024)) return MOE_ERR_LIMIT;
    ExpertGemmArgs b = a;
    if (!queue && a.combine_v && epi == EPI_ROWS_F32 && expert_small_combines(a.n_assign, a.K, a.format)) {
        const int row_bytes = ceil_div(a.K, kStageElems) * kStageElems * 2;
        const dim3 grid(a.rows / 16), block(64 * a.n_assign);
        if (a.format == FMT_BF16) hipLaunchKernelGGL(expert_tiny_down_kernel<FMT_BF16>, grid, block, row_bytes * a.n_assign, stream, b, row_bytes);
        else hipLaunchKernelGGL(expert_tiny_down_kernel<FMT_MXFP4>, grid, block, row_bytes * a.n_assign, stream, b, row_bytes);
        return launch_status();
    }
    if (a.combine_v || (a.scores && !expert_small_takes_scores(a.n_assign / a.assign_div, a.n_assign))) return MOE_ERR_LIMIT;
    const int items = queue ? a.work_count : min(a.n_assign, a.n_experts);
    if (items <= 0) return MOE_OK;
    const int tiles = a.rows / 16;
    // half-sized blocks while whole ones would not give every compute unit one
    const int waves = items * ceil_div(tiles, kSmallWaves) < a.n_cus ? kSmallWaves / 2 : kSmallWaves;
    b.row_blocks = ceil_div(tiles, waves);
    // a bucket has at most one row per token; what smaller ones do not stage leaves room for more blocks.  An entry may have
    // more rows than its caller says: passes of full length then (with passes of as many rows as the caller said, 32 entries
    // of 40 rows under a hint of 1 read every weight ten times: bf16 2460 us : 586)
    const int rows = queue ? kSmallRows : ceil_div(a.n_assign, a.assign_div);
    const int max_rows = min(kSmallRows, (max(rows, 1) + 3) & ~3);
    const int n_stages = ceil_div(a.K, kStageElems);
    const int lds_bytes = (int)min((long long)kSmallLds, (long long)ceil_div(n_stages, kSmallGroup) * kSmallGroup * max_rows * 256);
    const dim3 grid((unsigned)items * b.row_blocks), block(64 * waves);
#define MOE_SMALL(KERNEL, FMT, EPI)                                                                           \
    if (a.format == FMT && epi == EPI) {                                                                      \
        hipLaunchKernelGGL((KERNEL<FMT, EPI>), grid, block, lds_bytes, stream, b, max_rows, lds_bytes);       \
        return launch_status();                                                                               \
    }
    if (queue) {
        MOE_SMALL(expert_small_queue_kernel, FMT_BF16, EPI_SWIGLU_F32)
        MOE_SMALL(expert_small_queue_kernel, FMT_BF16, EPI_SCATTER)
        MOE_SMALL(expert_small_queue_kernel, FMT_MXFP4, EPI_SWIGLU_F32)
        MOE_SMALL(expert_small_queue_kernel, FMT_MXFP4, EPI_SCATTER)
    } else {
        MOE_SMALL(expert_small_kernel, FMT_BF16, EPI_SWIGLU_BF16)
        MOE_SMALL(expert_small_kernel, FMT_BF16, EPI_ROWS_F32)
        MOE_SMALL(expert_small_kernel, FMT_MXFP4, EPI_SWIGLU_BF16)
        MOE_SMALL(expert_small_kernel, FMT_MXFP4, EPI_ROWS_F32)
    }
#undef MOE_SMALL
    return MOE_ERR_FORMAT;
}

}  // namespace moe
