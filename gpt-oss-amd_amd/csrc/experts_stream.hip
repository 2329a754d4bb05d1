// Expert GEMMs of the MoE block: y = W x + b per expert over its bucket of token rows, with the
// SwiGLU (gate/up launch) or the per-slot row store (down launch) in the epilogue.
// Replaces moe_mlp1_swiglu_mfma_kernel (src/hip/moe.hip:9-235) and moe_mlp2_scatter_mfma_kernel
// (src/hip/moe.hip:261-512); the arithmetic contract is the CPU path's (src/run.cpp:657-705).
//
// Common to all kernels here: every weight byte is loaded from HBM once per token block, straight
// into the MFMA A-operand registers with 128-bit loads (no LDS for weights: a weight element is
// used by one wave only); the bucket's activation rows are the B operand and are shared by the
// waves of a block through LDS, 128 contraction elements (one stage) at a time, one barrier per
// stage; fp32 accumulation in v_mfma_f32_16x16x32_bf16.  A wave owns R MFMA row tiles (16 R weight
// rows) over the whole contraction length and up to NT*16 tokens.
//
// The contraction index is a dummy index, so lanes are free to pick which k each of their eight
// operand elements stands for as long as A and B agree.  Inside a stage, k-step j (0..3) and lane
// group g = lane/16 take
//   bf16  : elements 64(j/2) + 16g + 8(j%2) .. +8  (a lane's two loads of a pair of steps are adjacent: whole
//           128-byte lines per row)
//   MXFP4 : elements 32g + 8j .. +8  (lane group g owns MX block g of the stage: one 128-bit load + one scale byte
//           per row tile and stage, dequantised in registers to four A operands)
//
// Kernels: expert_stream_direct_kernel and expert_stream_ws_kernel (decode-sized buckets, producer and consumer waves) and
// expert_prefill_kernel (128-token blocks, 64 x 128 tile per wave) are what the fused block uses;
// expert_stream_queue_ws_kernel (the same consumers, producers that round fp32 rows) serves the entries that keep the
// reference's signatures and work queue.
#include <type_traits>

#include "expert_tiles.h"

namespace moe {

namespace {

// ---------------------------------------------------------------------------------------------
// Producer/consumer variant used by the fused block: a block has CONS consumer waves (R = 2 row
// tiles each, 32 CONS weight rows per block) and two producer waves.  Producers move the bucket's
// activation rows global -> LDS with direct-to-LDS 128-bit loads (no registers, a ring of four
// 16 KiB stage slots, three stages ahead of the consumers); consumers only have weight loads in
// their memory queue.  One barrier per stage; every wave of the block executes exactly
// 1 + ceil(K / 128) barriers.
// Positions of the contraction range that do not exist (ragged last stage, padding stages) carry
// a weight operand of exact zeros; the activation operand there is a clamped re-read of real data.
// ---------------------------------------------------------------------------------------------


// act_row(i): row of a.act that holds bucket row i of the token block (i < nrows).
// The stages of the bucket's rows are streamed `passes` times over (once per pass of the consumers
// over their row units), without a break in between.
template <int FMT, int NT, int PROD, class RowFn>
MOE_DEVICE void ws_producer(const ExpertGemmArgs& a, uint8_t* lds, RowFn act_row, int nrows, int p, int passes) {
    constexpr int BP = 4 / PROD;  // four-row blocks of a token tile moved by this wave
    constexpr int Q = BP * NT;    // direct-to-LDS loads per stage issued by this wave
    const int lane = threadIdx.x & 63;
    const int pos = lane & 15;   // chunk position inside the row's LDS image
    const int sub = lane >> 4;   // row inside the instruction's block of four
    const int K = a.K;
    const int n_stages = ceil_div(K, kStageElems);
    // this wave moves row blocks BP*p .. BP*p + BP-1 of every token tile; in the bucket's last token
    // tile only those that hold a row of the bucket (n_last of them), and of those only the lanes whose row
    // exists.  The places of the rows past the bucket's end are cleared once, below, in every ring slot, and no
    // load ever writes them.  The accumulator columns they feed are never stored, so any value would do for
    // the result; zeros are what the matrix pipe spends least on (measured on a synthetic kernel of this shape:
    // a token tile of zeros costs a stage 0.0-0.1 us, a tile of arbitrary values 0.15-0.25 us, at the same
    // instruction count), and a bucket of 33 rows has 15 such columns in its third tile.
    int n_last = 0;
#pragma unroll
    for (int ii = 0; ii < BP; ++ii) n_last += (16 * (NT - 1) + 4 * (BP * p + ii) < nrows) ? 1 : 0;
    const uint8_t* row[NT][BP];
    int chunk[BP];
    bool last_live[BP];  // this lane's row of the last token tile exists
#pragma unroll
    for (int ii = 0; ii < BP; ++ii) {
        const int q = 4 * (BP * p + ii) + sub;
        chunk[ii] = ws_chunk_at<FMT>(pos ^ q);
        last_live[ii] = 16 * (NT - 1) + q < nrows;
        if (!last_live[ii]) {
#pragma unroll
            for (int slot = 0; slot < kWsRing; ++slot)
                *reinterpret_cast<u32x4*>(lds + (size_t)slot * kLdsStageBytes + (NT - 1) * 4096 + (BP * p + ii) * 1024 +
                                          lane * 16) = u32x4{0u, 0u, 0u, 0u};
        }
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const int idx = min(t * 16 + q, nrows - 1);
            row[t][ii] = reinterpret_cast<const uint8_t*>(a.act + (size_t)act_row(idx) * K);
        }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the clearing stores, before this wave's first barrier
    // stage st of the rows into ring slot gs % 4 (gs counts stages over all passes)
    auto issue = [&](int gs, int st) {
        uint8_t* slot = lds + (size_t)(gs & (kWsRing - 1)) * kLdsStageBytes;
#pragma unroll
        for (int ii = 0; ii < BP; ++ii) {
            const int k = st * kStageElems + 8 * chunk[ii];
            const size_t off = (k < K) ? (size_t)k * 2 : 0;  // a position past the row re-reads its start
#pragma unroll
            for (int t = 0; t < NT - 1; ++t) dma16(row[t][ii] + off, slot + t * 4096 + (BP * p + ii) * 1024);
            // the last tile: a block without a row is skipped (wave-uniform, the waits below count on it); in a block
            // with rows the lanes without one sit the instruction out (it is issued, and counted, all the same)
            if (ii < n_last && last_live[ii]) dma16(row[NT - 1][ii] + off, slot + (NT - 1) * 4096 + (BP * p + ii) * 1024);
        }
    };
    // stage s has landed once only the loads of the two stages issued after it are outstanding
    auto wait_two_stages = [&]() {
        static_assert(BP == 2, "three possible load counts per stage");
        if (n_last == 2) wait_vmcnt<2 * Q>();
        else if (n_last == 1) wait_vmcnt<2 * Q - 2>();
        else wait_vmcnt<2 * Q - 4>();
    };
    // Bare s_barrier, not __syncthreads(): the fence of __syncthreads() makes the compiler wait for
    // every outstanding direct-to-LDS load (vmcnt(0)) in front of each barrier, i.e. also for the
    // stages issued just now, and the ring would hide nothing.  The explicit wait above each barrier
    // is the guarantee the consumers need: the stage they read next has been written to LDS.
    int st = 0;  // stage (inside a pass) issued next
    auto next_stage = [&]() { st = (st + 1 == n_stages) ? 0 : st + 1; };
    for (int gs = 0; gs < 3; ++gs) {
        issue(gs, st);
        next_stage();
    }
    wait_two_stages();  // stage 0 has landed
    __builtin_amdgcn_s_barrier();
    const int total = passes * n_stages;
    for (int i = 0; i < total; ++i) {
        issue(i + 3, st);  // past the last stage of the last pass: a re-read nobody consumes
        next_stage();
        wait_two_stages();  // stage i+1 has landed
        __builtin_amdgcn_s_barrier();
    }
    wait_vmcnt<0>();  // nothing may still be writing this block's LDS when the wave ends
}

// The lane id; for the work-queue entries (epilogue EPI) as a value that the compiler takes to be new at every call: what
// follows from it is then worked out per token block, not ahead of the loop over an entry list's whole blocks, where it would
// wait in scratch memory and be fetched in the stage loops (a spill access there waits for every weight load in flight).
template <int EPI>
MOE_DEVICE int ws_lane() {
    int lane = threadIdx.x & 63;
    if constexpr (EPI == EPI_SWIGLU_F32 || EPI == EPI_SCATTER) asm volatile("" : "+v"(lane));
    return lane;
}

// The producer for fp32 activations (the entries that keep the reference's data flow): rows first_row .. first_row + nrows of
// a.act_f32, rounded to bf16 on their way into the same LDS image.  An instruction takes two rows of 512 contiguous bytes; the
// loads of a stage are issued one stage before it is written, i.e. four before it is read.
template <int FMT, int NT, int PROD>
MOE_DEVICE void ws_producer_f32(const ExpertGemmArgs& a, uint8_t* lds, int first_row, int nrows, int p, int passes) {
    static_assert(PROD == 4, "eight rows of a token tile per step of the loops below");
    constexpr int Q = 2 * NT;  // loads per stage of this wave
    const int lane = ws_lane<EPI_SCATTER>();
    const int col = lane & 31;  // float4 of the row's 128 elements
    const int K = a.K;
    const int n_stages = ceil_div(K, kStageElems);
    const uint8_t* const base = reinterpret_cast<const uint8_t*>(a.act_f32 + (size_t)first_row * K);
    const int r0 = 2 * p + (lane >> 5);  // this lane's rows are r0, r0 + 8, ..
    uint32_t src[Q];
#pragma unroll
    for (int i = 0; i < Q; ++i)  // places past the bucket's end hold its last row, never stored
        src[i] = ((uint32_t)min(r0 + 8 * i, nrows - 1) * (uint32_t)K + 4u * (uint32_t)col) * 4u;
    uint8_t* const dst = lds + r0 * 256 + ((ws_pos<FMT>(col >> 1) ^ r0) << 4) + (col & 1) * 8;
    const int swap = (ws_pos<FMT>(col >> 1) ^ r0) & 8 ? -128 : 128;  // row r0 + 8 has bit 3 of the position flipped
    float4 v[Q];
    bool live = true;
    auto load = [&](int st) {
        // a position past the row re-reads its start
        live = st * kStageElems + 4 * col < K;
        const uint32_t off = live ? (uint32_t)st * (kStageElems * 4u) : 0u - 16u * (uint32_t)col;
#pragma unroll
        for (int i = 0; i < Q; ++i) v[i] = *reinterpret_cast<const float4*>(base + (src[i] + off));
    };
    auto store = [&](int gs) {
        uint8_t* at[2];
        at[0] = dst + (size_t)(gs & (kWsRing - 1)) * kLdsStageBytes;
        at[1] = at[0] + 2048 + swap;
        // and is written as zeros where its weights count as zero (MXFP4; bf16 never multiplies it): zero times an
        // infinity or a NaN from elsewhere in the row would reach all of its outputs
        const uint32_t keep = FMT == FMT_BF16 || live ? 0xffffffffu : 0u;
#pragma unroll
        for (int i = 0; i < Q; ++i)
            *reinterpret_cast<u32x2*>(at[i & 1] + (i >> 1) * 4096) =
                u32x2{pack_bf16x2(v[i].x, v[i].y) & keep, pack_bf16x2(v[i].z, v[i].w) & keep};
    };
    int st = 0;  // stage (inside a pass) loaded next
    auto next_stage = [&]() { st = (st + 1 == n_stages) ? 0 : st + 1; };
    load(st);
    next_stage();
    for (int gs = 0; gs < 3; ++gs) {
        store(gs);
        load(st);
        next_stage();
    }
    __syncthreads();  // stages 0 .. 2 are written
    const int total = passes * n_stages;
    for (int i = 0; i < total; ++i) {
        store(i + 3);  // past the last stage of the last pass: a re-read nobody consumes
        load(st);
        next_stage();
        __syncthreads();
    }
}

// slot_of_row(i): output row of bucket row i.  PRE: one more barrier comes first, right after the
// first weight loads have been issued (the kernel that finds the bucket itself completes the bucket
// list behind that barrier; the consumers need the list only in their epilogue, so their weights are
// already on the way while the producers read it).
// tile0: the first of the wave's R row tiles of 16 weight rows (R = 2: a row unit, tile0 even; R = 1: a single
// tile, for blocks whose range of tiles starts or ends inside a unit).
template <int FMT, int NT, int EPI, bool PRE = false, int R = 2, class SlotFn>
MOE_DEVICE void ws_consumer(const ExpertGemmArgs& a, const uint8_t* lds, int e, SlotFn slot_of_row, int nrows, int tile0,
                            bool active) {
    static_assert(R == 1 || R == 2, "one or two row tiles per wave");
    const int lane = ws_lane<EPI>();
    const int g = lane >> 4;
    const int q = lane & 15;
    const int K = a.K;
    const int n_stages = ceil_div(K, kStageElems);
    if (!active) {
        for (int i = 0; i <= n_stages + (PRE ? 1 : 0); ++i) __syncthreads();
        return;
    }
    const int group = tile0 >> 2;
    const int r0 = tile0 & 3;
    uint2 bias_raw[R];  // fetched now, used by the epilogue
    load_bias<R>(a, e, group, r0, bias_raw);
    const uint8_t* const lds_rd = lds + (size_t)q * 256;
    auto b_frag = [&](int s, int j, int t) {
        return *reinterpret_cast<const u32x4*>(lds_rd + (size_t)(s & (kWsRing - 1)) * kLdsStageBytes + t * 4096 +
                                               ((ws_pos<FMT>(ws_chunk<FMT>(j, g)) ^ q) << 4));
    };
    f32x4 acc[R][NT];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[r][t] = f32x4{0.f, 0.f, 0.f, 0.f};

    if constexpr (FMT == FMT_BF16) {
        // The contraction range is walked in pairs of MFMA steps (64 elements = one 128-byte line of a
        // weight row).  A pair of a row tile is fetched by two instructions that each take WHOLE lines:
        // instruction i holds tile rows 8i .. 8i+7, its lane (g, q) the 16-byte chunk 2g + (q >> 3) of tile
        // row 8i + (q & 7).  Every line is then requested by one instruction only, which is what lets the
        // loads be non-temporal (a line shared by two instructions is fetched twice under that hint) and
        // takes the stream from the plain-load rate to the streaming rate of the memory system.  The MFMA
        // operand of step h wants lane (g, q) to hold chunk 2g + h of tile row q: lanes 8..15 of every
        // 16-lane row of instruction 0 and lanes 0..7 of instruction 1 trade places (row_ror:8 under a bank
        // mask, in the stage that consumes the pair).  Ring of four pairs, loads issued three pairs (one
        // and a half stages) ahead of their use; nothing touches a loaded value before that pair.
        constexpr int DP = 4;
        const int n_pairs = K / 64;
        // Buffer loads: the expert's matrix is the buffer, the wave-uniform part of an address (row tile, pair,
        // instruction) is the scalar offset and the lane's part a 32-bit register that never changes, so a load
        // costs no vector arithmetic (and a read past the matrix would return zeros instead of faulting).
        const uint16_t* wbase = reinterpret_cast<const uint16_t*>(a.w) + (size_t)e * a.w_expert_stride;
        const __amdgpu_buffer_rsrc_t w_rsrc = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<uint16_t*>(wbase), 0, (int)((uint32_t)a.rows * (uint32_t)K * 2u), 0x00020000);
        uint32_t a_tile[R];  // wave-uniform byte offset of the row tile's first row
#pragma unroll
        for (int r = 0; r < R; ++r) a_tile[r] = (uint32_t)(group * 64 + tile_row_in_group(r0 + r, 0)) * (uint32_t)K * 2u;
        const uint32_t a_lane = (uint32_t)(tile_row_in_group(0, q & 7) * K + 8 * (2 * g + (q >> 3))) * 2u;
        const uint32_t second_half = 32u * (uint32_t)K * 2u;  // tile row q + 8 is weight row + 32 (tile_row_in_group)
        u32x4 ar[DP][2][R];
        auto load_a = [&](int slot, int pair) {
            const uint32_t off = (uint32_t)(pair < n_pairs ? pair : 0) * 128u;  // a padding pair re-reads pair 0 (unused)
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int r = 0; r < R; ++r)
                    ar[slot][i][r] = __builtin_amdgcn_raw_buffer_load_b128(w_rsrc, (int)a_lane,
                                                                           (int)(a_tile[r] + off + second_half * i), 2 /* nt */);
        };
#pragma unroll
        for (int i = 0; i < DP - 1; ++i) load_a(i, i);
        if constexpr (PRE) __syncthreads();
        __syncthreads();
        // one stage = two pairs; `ss` (stage parity) fixes the ring slots at compile time.  HALF: the ragged
        // last stage of a K that is an odd number of pairs runs its first pair only.
        auto stage = [&](auto ss_tag, auto half_tag, int st) {
            constexpr int ss = decltype(ss_tag)::value;
            constexpr bool HALF = decltype(half_tag)::value;
#pragma unroll
            for (int pp = 0; pp < (HALF ? 1 : 2); ++pp) {
                constexpr int kSlots = DP;
                const int u = 2 * ss + pp;  // ring slot of this pair
                const int pair = 2 * st + pp;
                load_a((u + kSlots - 1) % kSlots, pair + kSlots - 1);
                __builtin_amdgcn_sched_barrier(0);  // the loads are issued here, three pairs ahead of their use
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    u32x4 av[R];
#pragma unroll
                    for (int r = 0; r < R; ++r)
#pragma unroll
                        for (int d = 0; d < 4; ++d)
                            av[r][d] = h == 0 ? (uint32_t)__builtin_amdgcn_update_dpp((int)ar[u][0][r][d], (int)ar[u][1][r][d],
                                                                                      0x128, 0xF, 0xC, false)
                                              : (uint32_t)__builtin_amdgcn_update_dpp((int)ar[u][1][r][d], (int)ar[u][0][r][d],
                                                                                      0x128, 0xF, 0x3, false);
                    if constexpr (NT == 4) {
                        // four token tiles: one activation operand at a time, for both row tiles (the four of them
                        // held at once cost the registers that keep this loop free of spills; a spill access in
                        // here waits for every weight load in flight, since it counts in the same counter)
#pragma unroll
                        for (int t = 0; t < NT; ++t) {
                            const u32x4 b = b_frag(st, 2 * pp + h, t);
#pragma unroll
                            for (int r = 0; r < R; ++r) acc[r][t] = mfma_16x16x32(av[r], b, acc[r][t]);
                        }
                    } else {
                        u32x4 b[NT];
#pragma unroll
                        for (int t = 0; t < NT; ++t) b[t] = b_frag(st, 2 * pp + h, t);
#pragma unroll
                        for (int r = 0; r < R; ++r)
#pragma unroll
                            for (int t = 0; t < NT; ++t) acc[r][t] = mfma_16x16x32(av[r], b[t], acc[r][t]);
                    }
                }
            }
            __syncthreads();
        };
        const int full_stages = n_pairs >> 1;
        const int n_even = full_stages & ~1;
        for (int s0 = 0; s0 < n_even; s0 += 2) {
            stage(std::integral_constant<int, 0>{}, std::false_type{}, s0);
            stage(std::integral_constant<int, 1>{}, std::false_type{}, s0 + 1);
        }
        if (full_stages & 1) {
            stage(std::integral_constant<int, 0>{}, std::false_type{}, n_even);
            if (n_pairs & 1) stage(std::integral_constant<int, 1>{}, std::true_type{}, n_even + 1);
        } else if (n_pairs & 1) {
            stage(std::integral_constant<int, 0>{}, std::true_type{}, n_even);
        }
    } else {
        // Weights: a ring of four stages (one 128-bit load per row tile and stage, issued three
        // stages ahead of its use); scales: one word per row tile covers four stages and is
        // fetched one group of four ahead.  Addresses are a wave-uniform base (scalar registers)
        // plus a per-lane 32-bit offset that never changes, so a stage costs scalar arithmetic
        // only.  Nothing touches a loaded value before the stage that consumes it: an instruction
        // on it at load time would pin the wait for the load to the stage that issued it.
        constexpr int D = 4;
        const int G = K / 32;
        const uint32_t tile_bytes = (uint32_t)G * 256u;
        const uint32_t stile_bytes = (uint32_t)ceil_div(ceil_div(G, 4), 4) * 256u;
        // Buffer loads: the expert's tiled blocks (scales) are the buffer, the wave-uniform part of an address
        // (row tile, stage) is the scalar offset and the lane's part a constant register.  A read past the
        // buffer returns zeros instead of faulting, and a read past the tile inside it returns another tile's
        // bytes: both only ever happen in lanes or stages whose values are dropped (scale 0) or never used,
        // so no address needs a guard.
        const __amdgpu_buffer_rsrc_t w_rsrc = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<uint8_t*>(reinterpret_cast<const uint8_t*>(a.w) + (size_t)e * a.w_expert_stride), 0,
            (int)a.w_expert_stride, 0x00020000);
        const __amdgpu_buffer_rsrc_t s_rsrc = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<uint8_t*>(a.w_scales + (size_t)e * a.s_expert_stride), 0, (int)a.s_expert_stride, 0x00020000);
        uint32_t wtile[R], stile[R];  // wave-uniform byte offsets inside the expert
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const uint32_t tile = (uint32_t)(group * 4 + (r0 + r));
            wtile[r] = tile * tile_bytes;
            stile[r] = tile * stile_bytes;
        }
        const int voff_w = lane * 16;
        const int voff_s = lane * 4;
        u32x4 araw[D][R];
        uint32_t sw_cur[R], sw_nxt[R];
        auto load_a = [&](int slot, int s) {  // s may lie past the last stage: padding that nobody consumes
#pragma unroll
            for (int r = 0; r < R; ++r)
                // non-temporal: a 1 KiB chunk is read once, by this instruction alone, so keeping its
                // lines in L1/L2 only evicts the activation rows (measured: -5 % kernel time; the prefill
                // kernel, where neighbouring token blocks re-read the weights, is slower with it)
                araw[slot][r] = __builtin_amdgcn_raw_buffer_load_b128(w_rsrc, voff_w, (int)(wtile[r] + (uint32_t)s * 1024u),
                                                                      2 /* nt */);
        };
        auto load_scales = [&](uint32_t (&dst)[R], int quad) {
#pragma unroll
            for (int r = 0; r < R; ++r)
                dst[r] = __builtin_amdgcn_raw_buffer_load_b32(s_rsrc, voff_s, (int)(stile[r] + (uint32_t)quad * 256u), 0);
        };
        load_scales(sw_cur, 0);
#pragma unroll
        for (int i = 0; i < D - 1; ++i) load_a(i, i);
        if constexpr (PRE) __syncthreads();
        __syncthreads();
        // stage st, the i-th of its group of four (i fixes ring slot and scale byte at compile time)
        auto stage = [&](auto i_tag, int st) {
            constexpr int i = decltype(i_tag)::value;
            load_a((i + D - 1) % D, st + D - 1);
            __builtin_amdgcn_sched_barrier(0);  // the loads are issued here, three stages ahead of their use
            // In a ragged last stage the lane groups past the last MX block hold another tile's bytes (or zeros);
            // the tiled scale tensor has scale byte 0 in the slots of blocks that do not exist (moe_mxfp4_repack
            // writes it), which converts to a factor of exactly 0: no select needed.
            float sc[R];
#pragma unroll
            for (int r = 0; r < R; ++r) sc[r] = mxfp4_scale_to_f32((sw_cur[r] >> (8 * i)) & 0xFFu);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                u32x4 b[NT];
#pragma unroll
                for (int t = 0; t < NT; ++t) b[t] = b_frag(st, j, t);
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    uint32_t d[4];
                    mxfp4_dword_to_bf16x8(araw[i][r][j], sc[r], d);
                    const u32x4 av = {d[0], d[1], d[2], d[3]};
#pragma unroll
                    for (int t = 0; t < NT; ++t) acc[r][t] = mfma_16x16x32(av, b[t], acc[r][t]);
                }
            }
            __syncthreads();
        };
        const int full_quads = n_stages / 4;
        for (int qd = 0; qd < full_quads; ++qd) {
            load_scales(sw_nxt, qd + 1);
            stage(std::integral_constant<int, 0>{}, 4 * qd + 0);
            stage(std::integral_constant<int, 1>{}, 4 * qd + 1);
            stage(std::integral_constant<int, 2>{}, 4 * qd + 2);
            stage(std::integral_constant<int, 3>{}, 4 * qd + 3);
#pragma unroll
            for (int r = 0; r < R; ++r) sw_cur[r] = sw_nxt[r];
        }
        // the last, partial group of four (wave-uniform conditions; its weights are already in the ring)
        const int tail = n_stages - 4 * full_quads;
        if (tail > 0) stage(std::integral_constant<int, 0>{}, 4 * full_quads + 0);
        if (tail > 1) stage(std::integral_constant<int, 1>{}, 4 * full_quads + 1);
        if (tail > 2) stage(std::integral_constant<int, 2>{}, 4 * full_quads + 2);
    }
    stream_epilogue<R, NT, EPI>(a, acc, e, slot_of_row, nrows, group, r0, bias_raw);
}

// ws_consumer for blocks that cover up to 2 CONS row units.
// The wave takes row units unit0 and, with two passes, unit0 + unit_step (each if < unit_end), one per
// pass over the bucket's activation stages (which the producers stream `passes` <= 2 times); in a pass
// without a unit of its own it only takes part in the barriers.  The weight ring runs on across passes: the loads that the last
// stages of a pass issue are the first stages of the next pass's unit, so only the first pass of a
// block starts from an empty pipeline, and a pass's epilogue runs while those loads are in flight.
// Kept apart from ws_consumer: the second pass's code costs registers even when it does not run, so
// blocks that make one pass use the single-pass function.
template <int FMT, int NT, int EPI, bool PRE = false, class SlotFn>
MOE_DEVICE void ws_consumer_two(const ExpertGemmArgs& a, const uint8_t* lds, int e, SlotFn slot_of_row, int nrows, int unit0,
                            int unit_end, int unit_step, int passes) {
    constexpr int R = 2;
    constexpr bool TWO = true;
    const int lane = ws_lane<EPI>();
    const int g = lane >> 4;
    const int q = lane & 15;
    const int K = a.K;
    const int n_stages = ceil_div(K, kStageElems);
    if (unit0 >= unit_end) {  // no unit at all: barriers only
        for (int i = 0; i < 1 + (PRE ? 1 : 0) + passes * n_stages; ++i) __syncthreads();
        return;
    }
    const uint8_t* const lds_rd = lds + (size_t)q * 256;
    // gs: stage counted over all passes (the producers' ring slot)
    auto b_frag = [&](int gs, int j, int t) {
        return *reinterpret_cast<const u32x4*>(lds_rd + (size_t)(gs & (kWsRing - 1)) * kLdsStageBytes + t * 4096 +
                                               ((ws_pos<FMT>(ws_chunk<FMT>(j, g)) ^ q) << 4));
    };
    f32x4 acc[R][NT];
    uint2 bias_raw[R];

    // MXFP4 only: the bf16 stage loops have no registers to spare for a second pass's addresses at 128 registers a
    // lane (built and measured: 390 spilled registers, gate/up launch 206 against 190 us), so bf16 blocks make one pass.
    static_assert(FMT == FMT_MXFP4, "two-pass blocks exist for MXFP4 weights only");
    {
        // Weights: a ring of four stages (one 128-bit load per row tile and stage, issued three
        // stages ahead of its use); scales: one word per row tile covers four stages and is
        // fetched one group of four ahead.  Addresses are a wave-uniform base (scalar registers)
        // plus a per-lane 32-bit offset that never changes, so a stage costs scalar arithmetic
        // only.  Nothing touches a loaded value before the stage that consumes it: an instruction
        // on it at load time would pin the wait for the load to the stage that issued it.
        // Stage numbers at or past n_pad (the stage count rounded up to whole groups of four) mean the
        // next pass's unit; those in between are never used and re-read stage 0 with scale 0.
        constexpr int D = 4;
        const int G = K / 32;
        const uint32_t tile_bytes = (uint32_t)G * 256u;
        const uint32_t stile_bytes = (uint32_t)ceil_div(ceil_div(G, 4), 4) * 256u;
        // Buffer loads: the expert's tiled blocks (scales) are the buffer, the wave-uniform part of an address
        // (row tile, stage) is the scalar offset and the lane's part a constant register.  A read past the
        // buffer returns zeros instead of faulting, and a read past the tile inside it returns another tile's
        // bytes: both only ever happen in lanes or stages whose values are dropped (scale 0) or never used,
        // so no address needs a guard.
        const __amdgpu_buffer_rsrc_t w_rsrc = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<uint8_t*>(reinterpret_cast<const uint8_t*>(a.w) + (size_t)e * a.w_expert_stride), 0,
            (int)a.w_expert_stride, 0x00020000);
        const __amdgpu_buffer_rsrc_t s_rsrc = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<uint8_t*>(a.w_scales + (size_t)e * a.s_expert_stride), 0, (int)a.s_expert_stride, 0x00020000);
        uint32_t wtile[R], stile[R], wnext[R], snext[R];  // wave-uniform byte offsets inside the expert
        const int voff_w = lane * 16;
        const int voff_s = lane * 4;
        const int n_quads = ceil_div(n_stages, 4);
        const int n_pad = 4 * n_quads;
        u32x4 araw[D][R];
        uint32_t sw_cur[R], sw_nxt[R];
        // stage s of the current pass, or (s >= n_pad) stage s - n_pad of the next pass's unit; a stage number in
        // between is padding that nobody consumes
        auto load_a = [&](int slot, int s) {
            const bool nxt = TWO && s >= n_pad;  // wave-uniform
            const uint32_t so = (uint32_t)(nxt ? s - n_pad : s) * 1024u;
#pragma unroll
            for (int r = 0; r < R; ++r)
                // non-temporal: a 1 KiB chunk is read once, by this instruction alone, so keeping its
                // lines in L1/L2 only evicts the activation rows (measured: -5 % kernel time; the prefill
                // kernel, where neighbouring token blocks re-read the weights, is slower with it)
                araw[slot][r] = __builtin_amdgcn_raw_buffer_load_b128(w_rsrc, voff_w, (int)((nxt ? wnext[r] : wtile[r]) + so),
                                                                      2 /* nt */);
        };
        auto load_scales = [&](uint32_t (&dst)[R], int quad) {  // quad n_quads = the next pass's first
            const bool nxt = TWO && quad >= n_quads;
#pragma unroll
            for (int r = 0; r < R; ++r)
                dst[r] = __builtin_amdgcn_raw_buffer_load_b32(
                    s_rsrc, voff_s, (int)(nxt ? snext[r] : stile[r] + (uint32_t)quad * 256u), 0);
        };
        // one pass; written out once per pass instead of looped (see the bf16 branch)
        auto do_pass = [&](auto first_tag, int unit, bool more, int gs0) {
            constexpr bool first = decltype(first_tag)::value;
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const uint32_t tile = (uint32_t)((unit >> 1) * 4 + ((unit & 1) * R + r));
                const uint32_t tile_n = more ? (uint32_t)(((unit + unit_step) >> 1) * 4 + (((unit + unit_step) & 1) * R + r)) : tile;
                wtile[r] = tile * tile_bytes;
                stile[r] = tile * stile_bytes;
                if constexpr (TWO) {
                    wnext[r] = tile_n * tile_bytes;
                    snext[r] = tile_n * stile_bytes;
                }
            }
            load_bias<R>(a, e, unit >> 1, (unit & 1) * R, bias_raw);  // fetched now, used by the epilogue
#pragma unroll
            for (int r = 0; r < R; ++r)
#pragma unroll
                for (int t = 0; t < NT; ++t) acc[r][t] = f32x4{0.f, 0.f, 0.f, 0.f};
            if constexpr (first) {
                load_scales(sw_cur, 0);
#pragma unroll
                for (int i = 0; i < D - 1; ++i) load_a(i, i);
                if constexpr (PRE) __syncthreads();
                __syncthreads();
            }
            // stage st, the i-th of its group of four (i fixes ring slot and scale byte at compile time)
            // In a ragged last stage the lane groups past the last MX block hold another tile's bytes (or zeros); the
            // tiled scale tensor has scale byte 0 in the slots of blocks that do not exist (moe_mxfp4_repack clears
            // the tensor before it scatters), which converts to a factor of exactly 0, so their products vanish
            // without a select.
            auto stage = [&](auto i_tag, int st) {
                constexpr int i = decltype(i_tag)::value;
                load_a((i + D - 1) % D, st + D - 1);
                __builtin_amdgcn_sched_barrier(0);  // the loads are issued here, three stages ahead of their use
                float sc[R];
#pragma unroll
                for (int r = 0; r < R; ++r) sc[r] = mxfp4_scale_to_f32((sw_cur[r] >> (8 * i)) & 0xFFu);
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    u32x4 b[NT];
#pragma unroll
                    for (int t = 0; t < NT; ++t) b[t] = b_frag(gs0 + st, j, t);
#pragma unroll
                    for (int r = 0; r < R; ++r) {
                        uint32_t d[4];
                        mxfp4_dword_to_bf16x8(araw[i][r][j], sc[r], d);
                        const u32x4 av = {d[0], d[1], d[2], d[3]};
#pragma unroll
                        for (int t = 0; t < NT; ++t) acc[r][t] = mfma_16x16x32(av, b[t], acc[r][t]);
                    }
                }
                __syncthreads();
            };
            const int full_quads = n_stages / 4;
            for (int qd = 0; qd < full_quads; ++qd) {
                load_scales(sw_nxt, qd + 1);
                stage(std::integral_constant<int, 0>{}, 4 * qd + 0);
                stage(std::integral_constant<int, 1>{}, 4 * qd + 1);
                stage(std::integral_constant<int, 2>{}, 4 * qd + 2);
                stage(std::integral_constant<int, 3>{}, 4 * qd + 3);
#pragma unroll
                for (int r = 0; r < R; ++r) sw_cur[r] = sw_nxt[r];
            }
            // the last, partial group of four (wave-uniform conditions; its weights are already in the
            // ring); the stages it lacks still issue their loads, which belong to the next pass
            const int tail = n_stages - 4 * full_quads;
            if constexpr (TWO) {
                if (tail > 0) {
                    load_scales(sw_nxt, n_quads);
                    stage(std::integral_constant<int, 0>{}, 4 * full_quads + 0);
                    if (tail > 1) stage(std::integral_constant<int, 1>{}, 4 * full_quads + 1);
                    else load_a(0, 4 * full_quads + 4);
                    if (tail > 2) stage(std::integral_constant<int, 2>{}, 4 * full_quads + 2);
                    else load_a(1, 4 * full_quads + 5);
                    load_a(2, 4 * full_quads + 6);
#pragma unroll
                    for (int r = 0; r < R; ++r) sw_cur[r] = sw_nxt[r];
                }
            } else {
                if (tail > 0) stage(std::integral_constant<int, 0>{}, 4 * full_quads + 0);
                if (tail > 1) stage(std::integral_constant<int, 1>{}, 4 * full_quads + 1);
                if (tail > 2) stage(std::integral_constant<int, 2>{}, 4 * full_quads + 2);
            }
            stream_epilogue<R, NT, EPI>(a, acc, e, slot_of_row, nrows, unit >> 1, (unit & 1) * R, bias_raw);
        };
        if constexpr (TWO) {
            const int unit1 = unit0 + unit_step;
            do_pass(std::true_type{}, unit0, passes > 1 && unit1 < unit_end, 0);
            if (passes > 1) {
                if (unit1 < unit_end) do_pass(std::false_type{}, unit1, false, n_stages);
                else for (int i = 0; i < n_stages; ++i) __syncthreads();  // wave-uniform: no unit left for this wave
            }
        } else {
            do_pass(std::true_type{}, unit0, false, 0);
        }
    }
}

template <int FMT, int NT, int EPI, bool PRE, bool TWO, class SlotFn>
MOE_DEVICE void ws_consume_units(const ExpertGemmArgs& a, const uint8_t* lds, int e, SlotFn slot_of_row, int nrows,
                                 int unit0, int unit_end, int unit_step, int passes) {
    if constexpr (TWO) ws_consumer_two<FMT, NT, EPI, PRE>(a, lds, e, slot_of_row, nrows, unit0, unit_end, unit_step, passes);
    else ws_consumer<FMT, NT, EPI, PRE>(a, lds, e, slot_of_row, nrows, 2 * unit0, unit0 < unit_end);
}

// The same for a block whose rows are a range of row TILES [t0, t1) that need not start or end on a unit: a
// tile in front of the first whole unit goes to wave 0 and one behind the last whole unit to the wave after the
// last whole unit, each as a single tile; the launch sees to it that CONS waves are enough.
template <int FMT, int NT, int EPI, bool PRE, class SlotFn>
MOE_DEVICE void ws_consume_tiles(const ExpertGemmArgs& a, const uint8_t* lds, int e, SlotFn slot_of_row, int nrows,
                                 int t0, int t1, int wave) {
    const int lead = (t0 & 1) && t0 < t1;  // an empty range has no waves at work
    const int first = (wave == 0 || !lead) ? t0 + 2 * wave : t0 + 2 * wave - 1;  // wave-uniform
    if (lead && wave == 0) {
        ws_consumer<FMT, NT, EPI, PRE, 1>(a, lds, e, slot_of_row, nrows, t0, true);
    } else if (first + 1 == t1) {
        ws_consumer<FMT, NT, EPI, PRE, 1>(a, lds, e, slot_of_row, nrows, first, true);
    } else {
        ws_consumer<FMT, NT, EPI, PRE, 2>(a, lds, e, slot_of_row, nrows, first, first + 1 < t1);
    }
}

// One token block: the producer or consumer role of this wave, for the block's token-tile count.
// u0, u1: the block's row units [u0, u1), walked in passes of CONS units; with TILES its row tiles [u0, u1)
// (one pass, see ws_consume_tiles).
template <int FMT, int EPI, int CONS, int PROD, bool PRE = false, bool TWO = false, bool TILES = false, bool ACT_F32 = false,
          class RowFn, class SlotFn>
MOE_DEVICE void ws_token_block(const ExpertGemmArgs& a, uint8_t* lds, int wave, int u0, int u1, int e, RowFn act_row,
                               SlotFn slot_of_row, int nrows) {
    const int nt = (nrows + 15) >> 4;  // block-uniform
    const int passes = TWO ? min(2, max(1, ceil_div(u1 - u0, CONS))) : 1;
    if (wave >= CONS) {
        const int p = wave - CONS;
        if constexpr (PRE) __syncthreads();  // no direct-to-LDS load is in flight yet
        if constexpr (ACT_F32) {
            const int r0 = act_row(0);
            if (nt == 4) ws_producer_f32<FMT, 4, PROD>(a, lds, r0, nrows, p, passes);
            else if (nt == 3) ws_producer_f32<FMT, 3, PROD>(a, lds, r0, nrows, p, passes);
            else if (nt == 2) ws_producer_f32<FMT, 2, PROD>(a, lds, r0, nrows, p, passes);
            else ws_producer_f32<FMT, 1, PROD>(a, lds, r0, nrows, p, passes);
        } else if (nt == 4) ws_producer<FMT, 4, PROD>(a, lds, act_row, nrows, p, passes);
        else if (nt == 3) ws_producer<FMT, 3, PROD>(a, lds, act_row, nrows, p, passes);
        else if (nt == 2) ws_producer<FMT, 2, PROD>(a, lds, act_row, nrows, p, passes);
        else ws_producer<FMT, 1, PROD>(a, lds, act_row, nrows, p, passes);
    } else if constexpr (TILES) {
        static_assert(!TWO, "a range of tiles is walked in one pass");
        if (nt == 4) ws_consume_tiles<FMT, 4, EPI, PRE>(a, lds, e, slot_of_row, nrows, u0, u1, wave);
        else if (nt == 3) ws_consume_tiles<FMT, 3, EPI, PRE>(a, lds, e, slot_of_row, nrows, u0, u1, wave);
        else if (nt == 2) ws_consume_tiles<FMT, 2, EPI, PRE>(a, lds, e, slot_of_row, nrows, u0, u1, wave);
        else ws_consume_tiles<FMT, 1, EPI, PRE>(a, lds, e, slot_of_row, nrows, u0, u1, wave);
    } else {
        if (nt == 4) ws_consume_units<FMT, 4, EPI, PRE, TWO>(a, lds, e, slot_of_row, nrows, u0 + wave, u1, CONS, passes);
        else if (nt == 3) ws_consume_units<FMT, 3, EPI, PRE, TWO>(a, lds, e, slot_of_row, nrows, u0 + wave, u1, CONS, passes);
        else if (nt == 2) ws_consume_units<FMT, 2, EPI, PRE, TWO>(a, lds, e, slot_of_row, nrows, u0 + wave, u1, CONS, passes);
        else ws_consume_units<FMT, 1, EPI, PRE, TWO>(a, lds, e, slot_of_row, nrows, u0 + wave, u1, CONS, passes);
    }
}

// Linear block index -> (token block or expert, row block).  Workgroups go to the eight XCDs
// round-robin by linear index; with xcd_tiles all row blocks of an item run on one XCD (its
// activations enter one L2 once), otherwise they are spread over all of them.
MOE_DEVICE void ws_block_coords(const ExpertGemmArgs& a, int& item, int& rb) {
    const int n_rb = a.row_blocks;
    item = a.xcd_tiles ? ((blockIdx.x >> 3) / n_rb) * 8 + (blockIdx.x & 7) : blockIdx.x / n_rb;
    rb = a.xcd_tiles ? (blockIdx.x >> 3) % n_rb : blockIdx.x % n_rb;
}

// the row units of the weight matrix are spread evenly over the row blocks (sizes differ by at most one unit):
// block rb takes [u0, u1)
MOE_DEVICE void ws_row_units(const ExpertGemmArgs& a, int rb, int& u0, int& u1) {
    const int units = a.rows / 32;
    // the blocks with one unit more come first in the launch order: when the blocks take more than one round
    // over the compute units, the second-round blocks are handed out in that order to the units as they finish,
    // so a unit whose first block was a long one ends with a short one (measured: bf16 gate/up launch at 256
    // tokens, 512 blocks of 11 or 12 units, -3 %)
    const int q = units / a.row_blocks, rem = units - q * a.row_blocks;
    u0 = rb * q + min(rb, rem);
    u1 = u0 + q + (rb < rem ? 1 : 0);
}

// The same split in row tiles of 16 rows (two per unit), for blocks that make one pass: block sizes then differ
// by half a unit at most.  A block whose range starts or ends inside a unit needs a wave for each of those single
// tiles, so this split is only used while a block stays below 2 CONS tiles; otherwise the unit split, in tiles.
template <int CONS>
MOE_DEVICE void ws_row_tiles(const ExpertGemmArgs& a, int rb, int& t0, int& t1) {
    const int tiles = a.rows / 16;
    const int q = tiles / a.row_blocks, rem = tiles - q * a.row_blocks;
    if (q + (rem ? 1 : 0) <= 2 * CONS - 1) {
        t0 = rb * q + min(rb, rem);
        t1 = t0 + q + (rb < rem ? 1 : 0);
    } else {
        ws_row_units(a, rb, t0, t1);
        t0 *= 2;
        t1 *= 2;
    }
}

// Token blocks from the tile map written by the bucketing kernel.
// grid = row blocks x token blocks (padded to a multiple of 8), block = 64 (CONS + PROD); one block per CU: twelve
// waves leave 168 registers per lane, fourteen leave 128.
template <int FMT, int EPI, int CONS, int PROD>
__global__ __launch_bounds__((CONS + PROD) * 64, (CONS + PROD > 12) ? 4 : 3) void expert_stream_ws_kernel(ExpertGemmArgs a) {
    __shared__ __attribute__((aligned(16))) uint8_t lds[kWsRing * kLdsStageBytes];
    int tile, rb;
    ws_block_coords(a, tile, rb);
    if (tile >= *a.n_tiles) return;  // block-uniform
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int e = a.tile_expert[tile];
    const int row0 = a.tile_row0[tile];
    const int nrows = a.tile_rows[tile];
    int u0, u1;
    ws_row_units(a, rb, u0, u1);
    ws_token_block<FMT, EPI, CONS, PROD>(
        a, lds, wave, u0, u1, e, [&](int i) { return a.gather ? a.tokens_flat[row0 + i] : row0 + i; },
        [&](int i) { return row0 + i; }, nrows);
}

// ---------------------------------------------------------------------------------------------
// The same expert GEMM without a bucketing launch in front of it, for batches of at most
// kDirectMaxAssign assignments (tokens x experts per token).  A block is one (expert, row block)
// pair, known from the block index alone, and finds the expert's bucket itself: every wave compares
// chunks of 64 consecutive assignments of topk_i with the expert id, the per-chunk match counts go
// through LDS, one wave-wide prefix sum gives every chunk its offset, and the matching assignment
// ids (token * experts_per_token + k, ascending: the bucket order of bucket_kernel) land in an LDS
// list.
// Rows are addressed by assignment id: the activation row of assignment s is s / assign_div (gate/up
// launch: the token's row) or s itself (down launch), and the output row is s.
// grid = row blocks x experts (padded to a multiple of 8), block = 64 (CONS + PROD).
// ---------------------------------------------------------------------------------------------
constexpr int kDirectMaxAssign = 4096;  // 64 chunks of 64: one lane per chunk in the prefix sum
constexpr int kDirectMaxRows = 2048;    // longest bucket the LDS list holds

// Item f of the list of the buckets' whole blocks of 64 rows but each one's first, expert by expert: its expert and first
// row; false past the end of the list.  A bucket ends at kDirectMaxRows rows here as in direct_list_bucket: a caller's list may name
// an expert more often, and bucket[] holds no more.
MOE_DEVICE bool direct_whole_block(const int* hist, int n_experts, int f, int& e, int& row0) {
    const int lane = threadIdx.x & 63;
    for (int c = 0; c < n_experts; c += 64) {
        const int n = c + lane < n_experts ? min(hist[c + lane], kDirectMaxRows) : 0;
        const int whole = max(n - 65, 0) >> 6;
        uint32_t incl = (uint32_t)whole;
#define MOE_STEP(C, M) incl += dpp_move<C, M>(0u, incl);
        MOE_DPP_STEPS(MOE_STEP)
#undef MOE_STEP
        const int total = (int)__builtin_amdgcn_readlane(incl, 63);
        if (f < total) {
            const int j = __popcll(__ballot((int)incl <= f));  // experts whose whole blocks all come before
            const int before = (int)__builtin_amdgcn_readlane(incl, j) - __builtin_amdgcn_readlane(whole, j);
            e = c + j;
            row0 = __builtin_amdgcn_readlane(n - 64 * whole, j) + 64 * (f - before);
            return true;
        }
        f -= total;
    }
    return false;
}

// This wave's chunks (p * WAVES + wave) of the assignment list.
template <int WAVES, int P>
MOE_DEVICE void direct_load_ids(const ExpertGemmArgs& a, int wave, int (&ids)[P]) {
#pragma unroll
    for (int p = 0; p < P; ++p) {
        const int s = (p * WAVES + wave) * 64 + (threadIdx.x & 63);
        ids[p] = s < a.n_assign ? a.topk_i[s] : -1;
    }
}

// Lists the expert's bucket (complete behind the next barrier) and returns its rows.
template <int WAVES, int P>
MOE_DEVICE int direct_list_bucket(const ExpertGemmArgs& a, int wave, const int (&ids)[P], int e, int* bucket, int* chunk_cnt) {
    const int lane = threadIdx.x & 63;
    const int n_chunks = (a.n_assign + 63) >> 6;
    unsigned long long match[P];
#pragma unroll
    for (int p = 0; p < P; ++p) {
        const int c = p * WAVES + wave;
        match[p] = __ballot(ids[p] == e);
        if (lane == 0 && c < n_chunks) chunk_cnt[c] = __popcll(match[p]);
    }
    __syncthreads();
    // inclusive prefix sum of the chunk counts over the wave's lanes
    uint32_t incl = lane < n_chunks ? (uint32_t)chunk_cnt[lane] : 0u;
#define MOE_STEP(C, M) incl += dpp_move<C, M>(0u, incl);
    MOE_DPP_STEPS(MOE_STEP)
#undef MOE_STEP
#pragma unroll
    for (int p = 0; p < P; ++p) {
        const int c = p * WAVES + wave;
        if (c < n_chunks) {  // wave-uniform
            const int base = (int)__builtin_amdgcn_readlane(incl, c) - __popcll(match[p]);
            const int dst = base + __popcll(match[p] & ((1ull << lane) - 1ull));
            if (ids[p] == e && dst < kDirectMaxRows) bucket[dst] = c * 64 + lane;
        }
    }
    return min((int)__builtin_amdgcn_readlane(incl, 63), kDirectMaxRows);
}

// TWO: blocks cover up to 2 CONS row units, in two passes over the bucket's activations.
// MXFP4: the first a.main_blocks blocks of the launch take their bucket's remainder (1 .. 64 rows) and its first whole block of 64
// rows.  What a skewed router leaves beyond that is dealt out over the other blocks, which come last and leave at once where
// there is nothing.  With all of a bucket's token blocks run by its expert's own compute units, one after the other, the
// hottest expert set the launch's time.  Whole block, us, so : dealt out, E = 32, router of no preference, 256 tokens 109 : 109, 384
// tokens 147 : 146; Zipf 1.0, 256 tokens 187 : 182, 384 tokens 267 : 198; Zipf 1.5 245 : 174 and 375 : 189; E = 128, Zipf 1.0, 512 tokens
// 548 : 446, 1024 tokens 859 : 540.
// bf16 blocks keep to that: the second way into the stage loops costs the first its registers (256 tokens 280 : 287).  It costs the
// MXFP4 loops over whole blocks a few more spill accesses as well (gate/up 36 : 57 in the kernel, most of them around the stage loops),
// which no launch shows: 8 to 1000 tokens of 8 to 128 experts, blocks of 1024 to 4096, router of no preference, as fast or faster.
template <int FMT, int EPI, int CONS, int PROD, bool TWO>
__global__ __launch_bounds__((CONS + PROD) * 64, (CONS + PROD > 12) ? 4 : 3) void expert_stream_direct_kernel(ExpertGemmArgs a) {
    constexpr int WAVES = CONS + PROD;
    constexpr int P = (64 + WAVES - 1) / WAVES;  // chunks per wave
    constexpr bool DEAL = FMT == FMT_MXFP4;
    __shared__ __attribute__((aligned(16))) uint8_t lds[kWsRing * kLdsStageBytes];
    __shared__ int bucket[kDirectMaxRows];
    __shared__ int chunk_cnt[64];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // bf16 blocks make one pass over their rows and take them as a range of row tiles; MXFP4 blocks make up to two
    // passes of CONS units each, whose time does not depend on how many units a pass holds
    constexpr bool TILES = !TWO && FMT == FMT_BF16;
    // token of assignment s = s / assign_div, as a float multiplication (exact for s < 4096, assign_div <= 8)
    const float inv_div = 1.0f / (float)a.assign_div;
    auto token_of = [&](int s) { return (int)(((float)s + 0.5f) * inv_div); };
    int ids[P];
    if constexpr (DEAL) {
        if ((int)blockIdx.x >= a.main_blocks) {  // block-uniform, as all of the following
            __shared__ int hist[1024];  // rows per expert
            const int slot = ((int)blockIdx.x - a.main_blocks) / a.row_blocks;
            const int rb = (int)blockIdx.x - a.main_blocks - slot * a.row_blocks;
            const int slots = ((int)gridDim.x - a.main_blocks) / a.row_blocks;
            direct_load_ids<WAVES, P>(a, wave, ids);
            for (int i = threadIdx.x; i < a.n_experts; i += 64 * WAVES) hist[i] = 0;
            __syncthreads();
#pragma unroll
            for (int p = 0; p < P; ++p)
                if ((unsigned)ids[p] < (unsigned)a.n_experts) atomicAdd(&hist[ids[p]], 1);
            __syncthreads();
            int f = slot, e, row0;
            if (!direct_whole_block(hist, a.n_experts, f, e, row0)) return;
            int u0, u1;
            ws_row_units(a, rb, u0, u1);
            const int passes = TWO ? min(2, max(1, ceil_div(u1 - u0, CONS))) : 1;
            do {
                direct_load_ids<WAVES, P>(a, wave, ids);
                direct_list_bucket<WAVES, P>(a, wave, ids, e, bucket, chunk_cnt);
                __syncthreads();
                ExpertGemmArgs b = a;
                asm volatile("" : "+s"(b.K));  // new in every round: nothing that depends on it is worked out ahead of the loop
                auto act_row = [&](int i) { return a.gather ? token_of(bucket[row0 + i]) : bucket[row0 + i]; };
                auto slot_of_row = [&](int i) { return bucket[row0 + i]; };
                if (wave >= CONS) ws_producer<FMT, 4, PROD>(b, lds, act_row, 64, wave - CONS, passes);
                else ws_consume_units<FMT, 4, EPI, false, TWO>(b, lds, e, slot_of_row, 64, u0 + wave, u1, CONS, passes);
                __syncthreads();  // everyone is done with the list and the stages
                f += slots;
            } while (direct_whole_block(hist, a.n_experts, f, e, row0));
            return;
        }
    }
    int e, rb;
    ws_block_coords(a, e, rb);
    if (e >= a.n_experts) return;  // block-uniform (grid padding)
    int u0, u1;
    if constexpr (TILES) ws_row_tiles<CONS>(a, rb, u0, u1);
    else ws_row_units(a, rb, u0, u1);
    direct_load_ids<WAVES, P>(a, wave, ids);
    const int n_bucket = direct_list_bucket<WAVES, P>(a, wave, ids, e, bucket, chunk_cnt);
    if (n_bucket == 0) return;
    // The first token block takes the bucket's remainder (1..64 rows, any tile count) in straight-line
    // code; what is left are whole blocks of 64 rows, run by a loop that holds the four-tile variant
    // only (a loop around all tile-count variants costs every variant 30 registers per lane).
    // The barrier that completes the list is the first one of the token block.
    const int first = n_bucket - ((n_bucket - 1) & ~63);
    ws_token_block<FMT, EPI, CONS, PROD, true, TWO, TILES>(
        a, lds, wave, u0, u1, e, [&](int i) { return a.gather ? token_of(bucket[i]) : bucket[i]; },
        [&](int i) { return bucket[i]; }, first);
    const int passes = TWO ? min(2, max(1, ceil_div(u1 - u0, CONS))) : 1;
    const int end = DEAL ? min(n_bucket, first + 64) : n_bucket;
    for (int row0 = first; row0 < end; row0 += 64) {
        auto act_row = [&](int i) { return a.gather ? token_of(bucket[row0 + i]) : bucket[row0 + i]; };
        auto slot_of_row = [&](int i) { return bucket[row0 + i]; };
        if (wave >= CONS) ws_producer<FMT, 4, PROD>(a, lds, act_row, 64, wave - CONS, passes);
        else if constexpr (TILES) ws_consume_tiles<FMT, 4, EPI, false>(a, lds, e, slot_of_row, 64, u0, u1, wave);
        else ws_consume_units<FMT, 4, EPI, false, TWO>(a, lds, e, slot_of_row, 64, u0 + wave, u1, CONS, passes);
    }
}

// ---------------------------------------------------------------------------------------------
// The entries that keep the reference's data flow (work queue of (expert, row_offset, row_count) triples, entry format of
// src/hip/scheduler.hip:163-166; fp32 rows by slot in, fp32 rows or an atomic scatter out) on the same main loop.  Bound by the
// weights like the kernels above.  The queue's token blocks form one list: every entry's remainder (1 .. 64 rows, see
// expert_stream_direct_kernel), every entry's first whole block of 64 rows (where it has one: on the XCD of its remainder,
// where a short remainder leaves compute units early), then all other whole blocks, entry by entry.  Slot i of the launch
// takes list items i, i + slots, .., so an entry of many rows among short ones is dealt out over all compute units and XCDs
// (the row blocks of one slot run on one of them), whatever the caller's row-count hint says.  With a share of the launch to
// each entry the longest one set the launch's time: gate/up + down of 31 entries of 8 rows and one of 4000, bf16, 8057 us : 1010
// now (MXFP4 2816 : 395); one entry of 4000 rows alone, on one XCD then, 4639 : 788; 2048 tokens x 4 of 32 entries, skewed, 4380
// : 1459; evenly spread 1503 : 1412, 256 tokens 279 : 281.
// grid = row blocks x slots (xcd_tiles: slots a multiple of 8), block = 64 (CONS + PROD); slots >= work_count.
// ---------------------------------------------------------------------------------------------

// The next whole block of the slot at list item u or after: its expert and first row; false past the end of the list.
// `items`: the entries, rounded up to whole rounds of XCDs.  Every wave looks for itself, 64 entries at a time: no state lives
// across a block's main loop.
MOE_DEVICE bool queue_next_whole(const ExpertGemmArgs& a, int items, int slots, int& u, int& e, int& row0) {
    const int lane = threadIdx.x & 63;
    const int* queue = a.work_queue + 3 * (size_t)a.work_start;
    int n = lane < a.work_count ? queue[3 * lane + 2] : 0;
    if (u < 2 * items) {
        const int* entry = queue + 3 * (size_t)min(u - items, a.work_count - 1);
        if (u - items < a.work_count && entry[2] > 64) {
            e = entry[0];
            row0 = entry[1] + entry[2] - ((entry[2] - 1) & ~63);
            return true;
        }
        u += slots;  // >= 2 * items
    }
    int f = u - 2 * items;
    for (int c = 0; c < a.work_count; c += 64) {
        if (c > 0) n = c + lane < a.work_count ? queue[3 * (c + lane) + 2] : 0;
        const int whole = max(n - 65, 0) >> 6;  // but the first
        uint32_t incl = (uint32_t)whole;
#define MOE_STEP(C, M) incl += dpp_move<C, M>(0u, incl);
        MOE_DPP_STEPS(MOE_STEP)
#undef MOE_STEP
        const int total = (int)__builtin_amdgcn_readlane(incl, 63);
        if (f < total) {
            const int j = __popcll(__ballot((int)incl <= f));  // entries whose whole blocks all come before
            const int before = (int)__builtin_amdgcn_readlane(incl, j) - __builtin_amdgcn_readlane(whole, j);
            const int rem = __builtin_amdgcn_readlane(n - 64 * whole, j);  // remainder and first whole block
            e = __builtin_amdgcn_readfirstlane(queue[3 * (c + j)]);
            row0 = __builtin_amdgcn_readfirstlane(queue[3 * (c + j) + 1]) + rem + 64 * (f - before);
            return true;
        }
        f -= total;
    }
    return false;
}

template <int FMT, int EPI, int CONS, int PROD, bool TWO>
__global__ __launch_bounds__((CONS + PROD) * 64, (CONS + PROD > 12) ? 4 : 3) void expert_stream_queue_ws_kernel(ExpertGemmArgs a) {
    __shared__ __attribute__((aligned(16))) uint8_t lds[kWsRing * kLdsStageBytes];
    int slot, rb;
    ws_block_coords(a, slot, rb);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    constexpr bool TILES = !TWO && FMT == FMT_BF16;
    int u0, u1;
    if constexpr (TILES) ws_row_tiles<CONS>(a, rb, u0, u1);
    else ws_row_units(a, rb, u0, u1);
    const int passes = TWO ? min(2, max(1, ceil_div(u1 - u0, CONS))) : 1;
    if (slot < a.work_count) {  // block-uniform, as all of the following
        const int* entry = a.work_queue + 3 * (size_t)(a.work_start + slot);
        const int off = entry[1], n = entry[2];
        if (n > 0) {
            auto row = [&](int i) { return off + i; };
            ws_token_block<FMT, EPI, CONS, PROD, false, TWO, TILES, true>(a, lds, wave, u0, u1, entry[0], row, row,
                                                                          n - ((n - 1) & ~63));
        }
    }
    const int slots = gridDim.x / a.row_blocks;
    const int items = a.xcd_tiles && a.work_count >= 32 ? (a.work_count + 7) & ~7 : a.work_count;  // <= slots
    int u = slot < items ? slot + slots : slot, e, row0;
    // The exit in front of the loop is written out: with the search as the loop's condition every block paid for what the
    // compiler computes ahead of the loop and keeps in scratch memory (0.7 MB, 20 us), also without a whole block.
    if (!queue_next_whole(a, items, slots, u, e, row0)) return;
    do {
        ExpertGemmArgs b = a;
        asm volatile("" : "+s"(b.K));  // new in every round: nothing that depends on it is worked out ahead of the loop (ws_lane)
        auto row = [&](int i) { return row0 + i; };
        if (wave >= CONS) ws_producer_f32<FMT, 4, PROD>(b, lds, row0, 64, wave - CONS, passes);
        else if constexpr (TILES) ws_consume_tiles<FMT, 4, EPI, false>(b, lds, e, row, 64, u0, u1, wave);
        else ws_consume_units<FMT, 4, EPI, false, TWO>(b, lds, e, row, 64, u0 + wave, u1, CONS, passes);
        u += slots;
    } while (queue_next_whole(a, items, slots, u, e, row0));
}

// ---------------------------------------------------------------------------------------------
// Prefill-sized buckets: a 64-row x 128-token tile per wave (R = 4 row tiles, up to 8 token tiles),
// so a weight operand — for MXFP4 dequantised once in registers — feeds eight MFMAs, and the LDS
// holds the 128-token activation stage (2 x 32 KiB).  MXFP4 weights: activations are moved
// global -> LDS by direct-to-LDS loads issued one stage ahead by all eight waves (no staging
// registers), weights are fetched one stage ahead into registers.  MXFP4 only: bf16 experts have
// experts_tile.hip.
// grid = (ceil(rows / (64 WAVES)), max_tiles), token blocks of up to 128 rows.
// ---------------------------------------------------------------------------------------------
template <int NT, int EPI, int WAVES>
MOE_DEVICE void prefill_body_mxfp4(const ExpertGemmArgs& a, uint8_t* lds, int e, int row0, int nrows, int unit,
                                   bool active) {
    constexpr int R = 4;
    constexpr int NTMAX = 8;
    constexpr int kStageBytes = kStageSteps * NTMAX * 1024;
    constexpr int kStagers = WAVES / 4;                 // waves that stage the same k-step
    constexpr int TS = (NT + kStagers - 1) / kStagers;  // token tiles staged per wave
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int q = lane & 15;
    const int g = lane >> 4;
    const int K = a.K;
    const int G = K / 32;
    const int n_stages = ceil_div(K, kStageElems);
    const int n_quads = ceil_div(n_stages, 4);
    const int rem_groups = G & 3;

    // activation staging, LDS image as in the producer/consumer kernel (token tile t at t*4096, row
    // q at q*256, 16-byte chunk c at position c ^ q): this wave moves the four-row block wave%4
    // (256 contiguous bytes per row, whole cache lines) of token tiles wave/4, wave/4 + WAVES/4, ...
    const int blk_w = wave & 3;
    const int half_w = wave >> 2;
    const int q_dma = 4 * blk_w + (lane >> 4);     // row of the token tile this lane moves
    const int chunk_dma = ws_chunk_at<FMT_MXFP4>((lane & 15) ^ q_dma);  // chunk of the stage it fetches
    // Rows in units of 64 bytes (32 values): a register each, where a pointer takes two, and they reach 256 GiB.  Whole block, us,
    // pointers : bytes, which reach 4 GiB : so, 32 experts: 1000 tokens 232.2 : 232.3 : 230.9, 16384 tokens 2653.6 : 2654.2 : 2651.7, which two
    // runs of one build differ by as well.
    uint32_t b_row[TS];
#pragma unroll
    for (int i = 0; i < TS; ++i) {
        const int idx = min((half_w + kStagers * i) * 16 + q_dma, nrows - 1);
        const int src = a.gather ? a.tokens_flat[row0 + idx] : idx;  // rows by slot: counted from the block's first
        b_row[i] = (uint32_t)src * ((uint32_t)K / 32u);
    }
    const uint8_t* const b_base = reinterpret_cast<const uint8_t*>(a.act + (a.gather ? 0 : (size_t)row0 * K));
    // Rows of the last token tile past the block's end are cleared once and never loaded: products of zeros take the least power
    // (up to 15 such rows to a bucket; whole block, the last row again : zeros, 1000 tokens 243.8 : 241.4 us, from 4096 tokens on
    // within two runs of one build).
    static_assert(kStagers == 1, "this wave's last tile is the block's");
    const bool last_live = (NT - 1) * 16 + q_dma < nrows;
    if (!last_live) {
#pragma unroll
        for (int slot = 0; slot < 2; ++slot)
            *reinterpret_cast<u32x4*>(lds + (size_t)slot * kStageBytes + (NT - 1) * 4096 + blk_w * 1024 + lane * 16) = u32x4{0u, 0u, 0u, 0u};
    }
    auto issue_b = [&](int s) {
        const int k = s * kStageElems + 8 * chunk_dma;
        const uint8_t* const b_at = b_base + ((k < K) ? (size_t)k * 2 : 0);  // past the row: re-read its start (weights are 0 there)
        uint8_t* dst = lds + (size_t)(s & 1) * kStageBytes + (size_t)half_w * 4096 + blk_w * 1024;
#pragma unroll
        for (int i = 0; i < TS - 1; ++i) dma16(b_at + (size_t)b_row[i] * 64, dst + i * kStagers * 4096);
        if (last_live) dma16(b_at + (size_t)b_row[TS - 1] * 64, dst + (TS - 1) * kStagers * 4096);
    };
    const uint8_t* const lds_rd = lds + (size_t)q * 256;
    auto b_frag = [&](int s, int j, int t) {  // lane group g owns MX block g of a stage: chunk 4g + j
        return *reinterpret_cast<const u32x4*>(lds_rd + (size_t)(s & 1) * kStageBytes + t * 4096 +
                                               ((ws_pos<FMT_MXFP4>(4 * g + j) ^ q) << 4));
    };

    if (!active) {
        issue_b(0);
        wait_vmcnt<0>();
        __syncthreads();
        for (int s = 0; s < n_stages; ++s) {
            issue_b(s + 1);
            wait_vmcnt<0>();
            __syncthreads();
        }
        return;
    }

    const size_t tile_bytes = (size_t)G * 256;
    const size_t stile_bytes = (size_t)ceil_div(ceil_div(G, 4), 4) * 256;
    // wave-uniform bases (scalar registers) + per-lane 32-bit offsets that never change
    const uint8_t* const a_base = reinterpret_cast<const uint8_t*>(a.w) + (size_t)e * a.w_expert_stride +
                                  (size_t)unit * 4 * tile_bytes;
    const uint8_t* const s_base = a.w_scales + (size_t)e * a.s_expert_stride + (size_t)unit * 4 * stile_bytes;
    const uint32_t voff_w = (uint32_t)lane * 16;
    // ragged last stage: a lane group past the last MX block re-reads block 0 and gets scale 0
    const uint32_t voff_w_ragged = (uint32_t)((g < rem_groups ? lane : q) * 16);
    const uint32_t voff_s = (uint32_t)lane * 4;
    f32x4 acc[R][NT];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[r][t] = f32x4{0.f, 0.f, 0.f, 0.f};
    u32x4 araw[2][R];
    uint32_t sw_cur[R], sw_nxt[R];
    // Nothing touches a loaded weight before the stage that consumes it (an instruction on it at
    // load time would make the wave wait for the load right there): a stage or MX block that does
    // not exist re-reads one that does and is multiplied by scale 0.
    auto load_a = [&](int slot, int s) {
        const int su = s < n_stages ? s : 0;
        const bool ragged = rem_groups != 0 && su == n_stages - 1;
        const uint32_t vo = ragged ? voff_w_ragged : voff_w;
#pragma unroll
        for (int r = 0; r < R; ++r)
            araw[slot][r] = *reinterpret_cast<const u32x4*>(a_base + r * tile_bytes + (size_t)su * 1024 + vo);
    };
    auto load_scales = [&](uint32_t (&dst)[R], int quad) {
        const size_t off = (size_t)min(quad, n_quads - 1) * 256;
#pragma unroll
        for (int r = 0; r < R; ++r)
            dst[r] = *reinterpret_cast<const uint32_t*>(s_base + r * stile_bytes + off + voff_s);
    };
    auto do_stage = [&](int slot, int qpos, int s) {
        issue_b(s + 1);
        load_a(slot ^ 1, s + 1);
        __builtin_amdgcn_sched_barrier(0);  // next stage's loads are issued here, before this stage's MFMAs
        const bool live = s < n_stages && !(rem_groups != 0 && s == n_stages - 1 && g >= rem_groups);
        float sc[R];
#pragma unroll
        for (int r = 0; r < R; ++r) sc[r] = live ? mxfp4_scale_to_f32((sw_cur[r] >> (8 * qpos)) & 0xFFu) : 0.0f;
        u32x4 bq[2];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            u32x4 av[R];
#pragma unroll
            for (int r = 0; r < R; ++r) {
                uint32_t d[4];
                mxfp4_dword_to_bf16x8(araw[slot][r][j], sc[r], d);
                av[r] = u32x4{d[0], d[1], d[2], d[3]};
            }
            // activation operands are read from LDS two token tiles ahead of the MFMAs that use
            // them, across the k-steps of the stage
            if (j == 0) {
                bq[0] = b_frag(s, 0, 0);
                bq[1] = b_frag(s, 0, 1);
            }
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                const int slot_b = (j * NT + t) & 1;
                const u32x4 b = bq[slot_b];
                if (t + 2 < NT) bq[slot_b] = b_frag(s, j, t + 2);
                else if (j + 1 < 4) bq[slot_b] = b_frag(s, j + 1, t + 2 - NT);
                __builtin_amdgcn_sched_barrier(0);  // keep the read above ahead of the MFMAs below
#pragma unroll
                for (int i = 0; i < R; ++i) {
                    // there and back over the row tiles: every product has an operand of the one before it.  The launch's clock
                    // hangs on the power that changing operands take: whole block, us, one way : so, 32 experts, 1000 tokens 233.5 : 232.3, 4096
                    // tokens 706 : 704, skewed 712 : 708, 8192 tokens 1359 : 1352, 16384 tokens 2667 : 2654.
                    const int r = (t & 1) ? R - 1 - i : i;
                    acc[r][t] = mfma_16x16x32(av[r], b, acc[r][t]);
                }
            }
        }
        wait_vmcnt<0>();  // next stage's activations (direct-to-LDS) and weights have landed
        __syncthreads();
    };
    // weights, scales and biases first: their addresses need the tile's expert only, while the activation
    // loads wait for the token ids of the tile's rows (one memory round trip more)
    load_scales(sw_cur, 0);
    load_a(0, 0);
    uint2 bias_raw[R];  // fetched with the first stage: its latency stays off the block's tail
    load_bias<R>(a, e, unit, 0, bias_raw);
    __builtin_amdgcn_sched_barrier(0);
    issue_b(0);
    wait_vmcnt<0>();
    __syncthreads();
    for (int qd = 0; qd < n_quads; ++qd) {
        load_scales(sw_nxt, qd + 1);
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (4 * qd + i < n_stages) do_stage(i & 1, i, 4 * qd + i);  // block-uniform: the last group may be partial
#pragma unroll
        for (int r = 0; r < R; ++r) sw_cur[r] = sw_nxt[r];
    }
    stream_epilogue<R, NT, EPI>(a, acc, e, [&](int i) { return row0 + i; }, nrows, unit, 0, bias_raw);
}

// Two blocks of WAVES = 4 waves per CU: their barriers are independent, so one block's stage
// hand-over overlaps the other's MFMAs (one block of eight waves measured slower).
template <int FMT, int EPI, int WAVES>
__global__ __launch_bounds__(WAVES * 64, 2) void expert_prefill_kernel(ExpertGemmArgs a) {
    static_assert(FMT == FMT_MXFP4, "bf16 experts have a kernel of their own (experts_tile.hip)");
    constexpr int NTMAX = 8;
    __shared__ __attribute__((aligned(16))) uint8_t lds[2 * kStageSteps * NTMAX * 1024];
    // Row block fastest: neighbouring blocks share one token block's activations, which measured
    // faster than the order that keeps an expert's token blocks (same weights) together on one XCD.
    // Workgroups go to the eight XCDs round-robin by linear index, and each XCD has its own L2.
    // All row blocks of a token block run on ONE XCD, back to back in that XCD's sequence, so the
    // block's activations are fetched into that L2 once instead of once per XCD (measured: 40 %
    // less traffic into the L2s, -3 % time; sharing the weights between neighbouring token blocks
    // as well cut the traffic further but ran slower).  A launch of few blocks deals each token block's
    // row blocks out in two parts instead: with seven token blocks on one XCD and six on another the
    // launch would end with the one's third round of blocks (see ExpertPlan::few_blocks).
    const int n_rb = a.row_blocks, halves = a.xcd_tiles - 1;  // one or two parts: no division by them (0.4 % of 4096 tokens)
    const int per_part = (n_rb + halves) >> halves;
    const int m = blockIdx.x >> 3, round = m / per_part;
    const int share = round * 8 + (blockIdx.x & 7);  // (tile, part of its row blocks)
    const int tile = share >> halves;
    const int row_block = (share & halves) * per_part + m - round * per_part;
    if (row_block >= n_rb) return;  // block-uniform
    if (tile >= *a.n_tiles) return;  // block-uniform
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int unit = row_block * WAVES + wave;
    const bool active = unit < a.rows / 64;
    const int e = a.tile_expert[tile];
    const int row0 = a.tile_row0[tile];
    const int nrows = a.tile_rows[tile];
    const int nt = (nrows + 15) >> 4;  // block-uniform
    switch (nt) {
        case 8: prefill_body_mxfp4<8, EPI, WAVES>(a, lds, e, row0, nrows, unit, active); break;
        case 7: prefill_body_mxfp4<7, EPI, WAVES>(a, lds, e, row0, nrows, unit, active); break;
        case 6: prefill_body_mxfp4<6, EPI, WAVES>(a, lds, e, row0, nrows, unit, active); break;
        case 5: prefill_body_mxfp4<5, EPI, WAVES>(a, lds, e, row0, nrows, unit, active); break;
        case 4: prefill_body_mxfp4<4, EPI, WAVES>(a, lds, e, row0, nrows, unit, active); break;
        case 3: prefill_body_mxfp4<3, EPI, WAVES>(a, lds, e, row0, nrows, unit, active); break;
        default: prefill_body_mxfp4<2, EPI, WAVES>(a, lds, e, row0, nrows, unit, active); break;
    }
}

template <int FMT, int EPI>
int launch_cfg(const ExpertGemmArgs& a, hipStream_t stream) {
    if (a.work_queue) {
        if (a.work_count <= 0) return MOE_OK;
        if constexpr (EPI == EPI_SWIGLU_F32 || EPI == EPI_SCATTER) {
            ExpertGemmArgs b = a;
            const int cons = a.waves_per_block == 1 ? 12 : 10;
            const int units = a.rows / 32;
            b.row_blocks = max(a.row_blocks, ceil_div(units, (FMT == FMT_MXFP4 ? 2 : 1) * cons));
            // Slots: one per entry, and more where that would leave compute units idle (two blocks to each, while the list may
            // be that long).  If even one slot per token block leaves some idle, the blocks get shorter.
            const long long blocks = (long long)a.work_count * ceil_div(a.max_rows_hint, 64);
            if (blocks * b.row_blocks < a.n_cus) b.row_blocks = min(units, a.n_cus / (int)blocks);
            int slots = max(a.work_count, (int)min(blocks, (long long)ceil_div(2 * a.n_cus, b.row_blocks)));
            // few slots that do not divide by the XCDs are spread over all of them: 12 entries would put twice as many blocks on
            // four XCDs as on the others (12 short entries, MXFP4, gate/up + down 57 us : 37)
            b.xcd_tiles = slots % 8 == 0 || slots > 32;
            if (b.xcd_tiles) slots = ceil_div(slots, 8) * 8;
            const dim3 grid(slots * b.row_blocks), block((cons + 4) * 64);
            const bool two = ceil_div(units, b.row_blocks) > cons;
            if constexpr (FMT == FMT_MXFP4) {
                if (two && cons == 12) hipLaunchKernelGGL((expert_stream_queue_ws_kernel<FMT, EPI, 12, 4, true>), grid, block, 0, stream, b);
                else if (two) hipLaunchKernelGGL((expert_stream_queue_ws_kernel<FMT, EPI, 10, 4, true>), grid, block, 0, stream, b);
                if (two) return launch_status();
            }
            if (cons == 12) hipLaunchKernelGGL((expert_stream_queue_ws_kernel<FMT, EPI, 12, 4, false>), grid, block, 0, stream, b);
            else hipLaunchKernelGGL((expert_stream_queue_ws_kernel<FMT, EPI, 10, 4, false>), grid, block, 0, stream, b);
            return launch_status();
        }
    }
    if constexpr (EPI == EPI_SWIGLU_BF16 || EPI == EPI_ROWS_F32) {
        if (a.topk_i) {  // bucketing inside the expert kernel
            if (a.n_assign > kDirectMaxAssign || a.assign_div <= 0 || a.assign_div > 8 || a.n_experts <= 0 || a.n_experts > 1024) return MOE_ERR_LIMIT;
            ExpertGemmArgs b = a;
            const int cons = a.waves_per_block == 1 ? 12 : 10;
            // a block covers at most `cons` row units per pass; MXFP4 blocks may make two passes (the
            // second pass's code would cost the bf16 stage loops registers they do not have)
            const int units = a.rows / 32;
            b.row_blocks = max(a.row_blocks, ceil_div(units, (FMT == FMT_MXFP4 ? 2 : 1) * cons));
            const bool two = ceil_div(units, b.row_blocks) > cons;
            b.main_blocks = ceil_div(a.n_experts, 8) * 8 * b.row_blocks;
            // and blocks for the token blocks from a bucket's third on: at most so many, one round of them
            const int more = FMT == FMT_MXFP4 ? min((a.n_assign - 1) / 128, ceil_div(a.n_cus, b.row_blocks)) : 0;
            dim3 grid(b.main_blocks + more * b.row_blocks);
            if constexpr (FMT == FMT_MXFP4) {
                if (two && cons == 12) {
                    hipLaunchKernelGGL((expert_stream_direct_kernel<FMT, EPI, 12, 2, true>), grid, dim3(896), 0, stream, b);
                    return launch_status();
                }
                if (two) {
                    hipLaunchKernelGGL((expert_stream_direct_kernel<FMT, EPI, 10, 2, true>), grid, dim3(768), 0, stream, b);
                    return launch_status();
                }
            }
            if (cons == 12) {
                hipLaunchKernelGGL((expert_stream_direct_kernel<FMT, EPI, 12, 2, false>), grid, dim3(896), 0, stream, b);
            } else {
                hipLaunchKernelGGL((expert_stream_direct_kernel<FMT, EPI, 10, 2, false>), grid, dim3(768), 0, stream, b);
            }
        } else if (a.waves_per_block == 16) {
            if constexpr (FMT == FMT_MXFP4) {
                ExpertGemmArgs b = a;
                b.row_blocks = ceil_div(a.rows / 64, 4);
                // every XCD gets whole token blocks, or whole parts of their row blocks
                dim3 grid(ceil_div(a.max_tiles * a.xcd_tiles, 8) * 8 * ceil_div(b.row_blocks, a.xcd_tiles));
                hipLaunchKernelGGL((expert_prefill_kernel<FMT, EPI, 4>), grid, dim3(256), 0, stream, b);
            } else {
                return MOE_ERR_FORMAT;
            }
        } else if (a.waves_per_block == 17) {
            return launch_expert_tile_bf16(a, EPI, stream);
        } else if (a.waves_per_block == 0) {
            ExpertGemmArgs b = a;
            b.row_blocks = max(a.row_blocks, ceil_div(a.rows / 32, 10));
            dim3 grid(ceil_div(a.max_tiles, 8) * 8 * b.row_blocks);
            hipLaunchKernelGGL((expert_stream_ws_kernel<FMT, EPI, 10, 2>), grid, dim3(768), 0, stream, b);
        } else if (a.waves_per_block == 1) {
            ExpertGemmArgs b = a;
            b.row_blocks = max(a.row_blocks, ceil_div(a.rows / 32, 12));
            dim3 grid(ceil_div(a.max_tiles, 8) * 8 * b.row_blocks);
            hipLaunchKernelGGL((expert_stream_ws_kernel<FMT, EPI, 12, 2>), grid, dim3(896), 0, stream, b);
        } else {
            return MOE_ERR_FORMAT;
        }
    } else {
        return MOE_ERR_FORMAT;
    }
    return launch_status();
}

template <int FMT>
int launch_fmt(const ExpertGemmArgs& a, int epi, hipStream_t stream) {
    switch (epi) {
        case EPI_SWIGLU_BF16: return launch_cfg<FMT, EPI_SWIGLU_BF16>(a, stream);
        case EPI_ROWS_F32: return launch_cfg<FMT, EPI_ROWS_F32>(a, stream);
        case EPI_SWIGLU_F32: return launch_cfg<FMT, EPI_SWIGLU_F32>(a, stream);
        case EPI_SCATTER: return launch_cfg<FMT, EPI_SCATTER>(a, stream);
    }
    return MOE_ERR_FORMAT;
}

}  // namespace

int expert_direct_max_assignments() { return kDirectMaxAssign; }

// epi: 0 fused gate/up (bf16 SwiGLU out), 1 fused down (fp32 rows per slot), 2 gate/up with fp32
// in/out, 3 down with fp32 in and atomic scatter.  Token blocks hold at most 64 rows.
int launch_expert_stream(const ExpertGemmArgs& a, int epi, hipStream_t stream) {
    if (a.rows % 64 != 0 || a.K % 32 != 0) return MOE_ERR_SHAPE;
    const bool queue = a.work_queue != nullptr;
    if (queue != (epi == EPI_SWIGLU_F32 || epi == EPI_SCATTER)) return MOE_ERR_FORMAT;
    if (a.waves_per_block == 18) return launch_expert_small(a, epi, stream);
    if (a.format == FMT_BF16) {
        // the streaming consumers address an expert's matrix through a buffer descriptor: 32-bit byte offsets
        if ((unsigned long long)a.rows * (unsigned long long)a.K * 2ull > 0x7fffffffull) return MOE_ERR_LIMIT;
        return launch_fmt<FMT_BF16>(a, epi, stream);
    }
    if (a.format == FMT_MXFP4) {
        if (a.w_expert_stride > 0x7fffffffll || a.s_expert_stride > 0x7fffffffll) return MOE_ERR_LIMIT;
        return launch_fmt<FMT_MXFP4>(a, epi, stream);
    }
    return MOE_ERR_FORMAT;
}

}  // namespace moe
