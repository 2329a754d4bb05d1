// Expert GEMMs of the MoE block for prefill-sized buckets of bf16 experts: 256 tokens x 256 weight rows per block, both
// operands shared through LDS.  Replaces moe_mlp1_swiglu_mfma_kernel (src/hip/moe.hip:9-235) and
// moe_mlp2_scatter_mfma_kernel (src/hip/moe.hip:261-512) at those sizes.
//
// What bounds it: with 128 tokens to a block the launch was bound by the weights on their way to the compute units
// (96 KiB a CU for every 2048 cycles of matrix work; 5.1 GB into the L2s per gate/up launch at 4096 tokens x 32 experts,
// 1077 us).  Here a stage brings 64 KiB for the same work, and an XCD's blocks share it: 1.4 to 2.1 GB, 484 to 525 us,
// i.e. 1.1 PFLOP/s (down launch 564 -> 304 us).  Gate/up launch at that size with the other parts taken out: matrix
// instructions and epilogues 366 us, fragment reads from LDS 284, loads into LDS 247 from L2 and 435 from where the data are.
#include <type_traits>

#include "expert_tiles.h"

namespace moe {

namespace {

constexpr int kTileStageElems = 64;                  // contraction elements of a stage: one 128-byte line of every row
constexpr int kTileRows = 256;                       // weight rows of a block (four row groups of 64)
constexpr int kTileHalf = kTileRows * 128;           // one operand of a stage: 256 rows x 128 bytes
constexpr int kTileLds = 5 * kTileHalf;              // all of a CU's LDS

// LDS image of an operand's stage: row i (16 rows to an MFMA tile) at i * 128, its eight 16-byte chunks permuted: chunk
// c sits at position c ^ tile_swz(i % 16).  A fragment read (ds_read_b128) is served 16 lanes at a time, tile rows
// 0-3 and 12-15 of one lane group together with rows 4-11 of the next, over 64 banks; two rows share the 256 bytes of
// all banks, and the chunks of two neighbouring lane groups are 2 apart, so the positions of the even (and of the odd)
// rows of such a set are eight different ones exactly if {f(0), f(1), f(6), f(7)} and {f(2) ^ 2, .., f(5) ^ 2} are
// disjoint for f(row / 2): f below maps them to {0..3} and {4..7}.
MOE_DEVICE int tile_swz(int q) {
    const int h = q >> 1;
    return ((h ^ (h << 1)) & 4) | ((h >> 1) & 2) | (h & 1);
}

// 64 lanes x 16 bytes from base + the lane's 32-bit offset to 1 KiB of LDS at a wave-uniform address.  In assembly: the
// compiler puts a wait for every direct-to-LDS load it knows of in front of the wave's next LDS read, so loads that
// run a stage ahead must be invisible to it.  They count in vmcnt; the caller waits.  Writes M0, which the compiler
// reserves and does not take in a clobber list: nothing else in a kernel that calls this may use it.
MOE_DEVICE void tile_dma16(const void* base_uniform, uint32_t lane_off, uint32_t lds_addr_uniform) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(lane_off), "s"(base_uniform),
                 "s"(lds_addr_uniform)
                 : "memory");
}

// The same for the lanes of `lanes` only, by all lanes of a wave; it counts in vmcnt even if there are none.
MOE_DEVICE void tile_dma16_lanes(const void* base_uniform, uint32_t lane_off, uint32_t lds_addr_uniform, unsigned long long lanes) {
    asm volatile("s_mov_b32 m0, %2\n\ts_mov_b64 exec, %3\n\tglobal_load_lds_dwordx4 %0, %1\n\ts_mov_b64 exec, -1" ::"v"(lane_off),
                 "s"(base_uniform), "s"(lds_addr_uniform), "s"(lanes)
                 : "memory");
}

// All loads of this wave but the YOUNGER last ones have landed and all its LDS reads are back; then the block's barrier.  One
// statement with a memory clobber, so that no LDS access of the compiler's moves across the barrier.
template <int YOUNGER>
MOE_DEVICE void wait_and_meet() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(YOUNGER) : "memory");
}

// A wave's share of a block: NT token tiles of 16 and one group of 64 weight rows, i.e. a 64 x 16 NT tile of the
// output in 16 NT accumulator registers.  TS token shares x 8 / TS row groups make the block's eight waves: 2 x 4 for
// full row blocks, 4 x 2 and 8 x 1 for a last row block that has two groups or one (rows = 2880 leaves one: its block
// then takes a quarter of the time instead of all of it with three idle wave pairs).
template <int NT, int TS, int EPI>
MOE_DEVICE void tile_body(const ExpertGemmArgs& a, uint8_t* lds, int e, int row0, int nrows, int group0) {
    constexpr int R = 4;
    constexpr int RG = 8 / TS;        // row groups of the block
    constexpr int PT = TS * NT / 4;   // direct-to-LDS loads of a stage per wave: tokens,
    constexpr int PW = RG;            // weight rows
    static_assert(TS * NT <= 16 && PT >= 1, "a block holds at most 256 tokens");
    // LDS: a ring of D stages of weight rows and of DT stages of token rows.  The rate of these loads is the bytes in flight
    // over their latency, so the rings take what the LDS holds; with 256 tokens that is three stages of weights, which come
    // from HBM, and two of token rows, which the XCD's other blocks have mostly brought into its L2.
    constexpr int kTokSlot = TS * NT * 2048;
    constexpr int D = TS * NT <= 4 ? 4 : 3;
    constexpr int DT = TS * NT <= 8 ? D : 2;
    constexpr int kWBase = DT * kTokSlot;
    static_assert(kWBase + D * kTileHalf <= kTileLds, "the slots fit the LDS");
    // Stage s requests the token rows of stage s + DT and then the weight rows of s + D.  At its end stage s + 1 is there
    // once only the loads younger than its own are outstanding:
    constexpr int kYounger = DT == D ? (D - 2) * (PT + PW) : PW;
    static_assert(DT == D || (DT == 2 && D == 3), "the count above");
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int q = lane & 15;
    const int g = lane >> 4;
    const int wg = wave % RG;   // row group of this wave
    const int th = wave / RG;   // token share of this wave
    const int K = a.K;
    const int n_stages = K / kTileStageElems;

    // ---- staging: instruction n moves LDS rows 8n .. 8n + 7, whole 128-byte lines; wave w issues n = w, w + 8, .. ----
    // Places past the token block's end are cleared here and never written: what they hold is never stored, and zeros cost the
    // matrix pipe the least power, which the clock hangs on (1.9 of 2.4 GHz; with all weights zero the whole block takes 807
    // instead of 891 us).  4096 tokens, 32 experts (blocks of 176 rows in 192 places), the last row again : zeros 894 : 877 us.
    uint32_t off_t[PT], off_w[PW];
    unsigned long long live[PT];
    const int sub = lane >> 3;
#pragma unroll
    for (int i = 0; i < PT; ++i) {
        const int row = 8 * (wave + 8 * i) + sub;
        const int idx = min(row, nrows - 1);
        live[i] = __ballot(row < nrows);
        if (row >= nrows) {
#pragma unroll
            for (int slot = 0; slot < DT; ++slot)
                *reinterpret_cast<u32x4*>(lds + slot * kTokSlot + (wave + 8 * i) * 1024 + lane * 16) = u32x4{0u, 0u, 0u, 0u};
        }
        const int src = a.gather ? a.tokens_flat[row0 + idx] : idx;  // rows by slot: counted from the block's first
        off_t[i] = (uint32_t)src * (uint32_t)K * 2u + (uint32_t)(((lane & 7) ^ tile_swz(row & 15)) * 16);
    }
#pragma unroll
    for (int i = 0; i < PW; ++i) {
        const int row = 8 * (wave + 8 * i) + sub;
        const int w_row = min((group0 + (row >> 6)) * 64 + tile_row_in_group((row >> 4) & 3, row & 15), a.rows - 1);
        off_w[i] = (uint32_t)w_row * (uint32_t)K * 2u + (uint32_t)(((lane & 7) ^ tile_swz(row & 15)) * 16);
    }
    const uint8_t* const base_t = reinterpret_cast<const uint8_t*>(a.act + (a.gather ? 0 : (size_t)row0 * K));
    const uint8_t* const base_w =
        reinterpret_cast<const uint8_t*>(reinterpret_cast<const uint16_t*>(a.w) + (size_t)e * a.w_expert_stride);
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane(
        (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)lds + (uint32_t)wave * 1024u);
    // Stages past the last one are requested as stage 0, into slots nobody reads again, so that the counts of younger
    // loads hold to the end.
    auto stage_off = [&](int s) { return (size_t)(s < n_stages ? s : 0) * 128; };
    auto dma_tokens = [&](int i, int s, int slot) {  // the wave's i-th load of the stage
        tile_dma16_lanes(base_t + stage_off(s), off_t[i], lds0 + (uint32_t)(slot * kTokSlot + i * 8192), live[i]);
    };
    auto dma_weights = [&](int i, int s, int slot) {
        tile_dma16(base_w + stage_off(s), off_w[i], lds0 + (uint32_t)(kWBase + slot * kTileHalf + i * 8192));
    };

    // ---- fragments: k-step j (0, 1) of a stage, lane group g take elements 16 g + 8 j .. +8 of the 64 (chunk 2g + j), as
    // the other bf16 kernels do, so all of them add in the same order ----
    const int frag = q * 128 + (((2 * g) ^ tile_swz(q)) << 4);
    const uint8_t* const rd_t = lds + th * (NT * 2048);
    const uint8_t* const rd_w = lds + kWBase + wg * 8192;
    u32x4 aw[2][R], bt[2][NT];
    auto read_frag = [&](int j, int i, int ts, int ws) {  // i < R: weight tile i, else token tile i - R
        const int at = frag ^ (j << 4);
        if (i < R) aw[j][i] = *reinterpret_cast<const u32x4*>(rd_w + ws * kTileHalf + at + i * 2048);
        else bt[j][i - R] = *reinterpret_cast<const u32x4*>(rd_t + ts * kTokSlot + at + (i - R) * 2048);
    };

    f32x4 acc[R][NT];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[r][t] = f32x4{0.f, 0.f, 0.f, 0.f};

    const bool active = group0 + wg < a.rows / 64;
    uint2 bias_raw[R];
    load_bias<R>(a, e, active ? group0 + wg : 0, 0, bias_raw);
#pragma unroll
    for (int d = 0; d < D; ++d) {  // with DT < D the order is w0 t0 w1 t1 w2
#pragma unroll
        for (int i = 0; i < PW; ++i) dma_weights(i, d, d);
        if (d < DT) {
#pragma unroll
            for (int i = 0; i < PT; ++i) dma_tokens(i, d, d);
        }
    }
    wait_and_meet<(D - 1) * PW + (DT - 1) * PT>();
#pragma unroll
    for (int i = 0; i < R + NT; ++i) read_frag(0, i, 0, 0);

    // One k-step: the MFMAs of step j, and between them the reads of the step after it (j ^ 1, from slots ts and ws) and,
    // with REQUEST, the loads of stage s into the slots that it has left.
    constexpr int READS = R + NT;
    constexpr int PER = (READS + NT - 1) / NT;  // reads in front of each token tile's MFMAs
    auto k_step = [&](auto j_tag, auto request_tag, int ts, int ws, int s, int free_ts, int free_ws) {
        constexpr int j = decltype(j_tag)::value;
        constexpr bool REQUEST = decltype(request_tag)::value;
#pragma unroll
        for (int t = 0; t < NT; ++t) {
#pragma unroll
            for (int i = t * PER; i < min((t + 1) * PER, READS); ++i) read_frag(j ^ 1, i, ts, ws);
            if constexpr (REQUEST) {
#pragma unroll
                for (int i = t * (PT + PW) / NT; i < (t + 1) * (PT + PW) / NT; ++i) {
                    if (i < PT) dma_tokens(i, s + DT, free_ts);
                    else dma_weights(i - PT, s + D, free_ws);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < R; ++i) {
                // there and back: each product has an operand of the one before it, which takes less power.  Whole block, us, one way :
                // so, 32 experts: 2400 tokens 597 : 591, 3400 tokens 736 : 727, 4096 tokens 855 : 855, skewed 864 : 861, 8192 tokens 1562 : 1548.
                const int r = (t & 1) ? R - 1 - i : i;
                acc[r][t] = mfma_16x16x32(aw[j][r], bt[j][t], acc[r][t]);
            }
        }
    };
    int ts = 0, ws = 0;
    for (int s = 0; s < n_stages; ++s) {
        k_step(std::integral_constant<int, 0>{}, std::false_type{}, ts, ws, 0, 0, 0);
        // this wave has read all of stage s and its loads of stage s + 1 have landed: after the barrier that holds for
        // every wave, so the slots of stage s may be refilled and stage s + 1 read (past the last stage: nobody uses it)
        wait_and_meet<kYounger>();
        const int next_ts = ts + 1 == DT ? 0 : ts + 1, next_ws = ws + 1 == D ? 0 : ws + 1;
        k_step(std::integral_constant<int, 1>{}, std::true_type{}, next_ts, next_ws, s, ts, ws);
        ts = next_ts;
        ws = next_ws;
    }
    wait_vmcnt<0>();  // nothing may still be writing this block's LDS when the wave ends
    if (!active) return;
    const int first = th * NT * 16;
    stream_epilogue<R, NT, EPI>(a, acc, e, [&](int i) { return row0 + first + i; }, nrows - first, group0 + wg, 0, bias_raw);
}

// Block index -> (token tile, row block).  The tile map is in bucket order; an expert's tiles x row blocks are consecutive
// in the launch's sequence, row block by row block, and 32 consecutive blocks run side by side on one XCD (workgroups go to
// the eight XCDs round-robin by linear index, one per CU): they are n tiles of one expert times 32 / n of its row blocks, so
// a stage of theirs takes n + 32 / n operand slabs from beyond the XCD's L2 instead of 64.
constexpr int kXcdCus = 32;

template <int EPI>
__global__ __launch_bounds__(512, 2) void expert_tile_bf16_kernel(ExpertGemmArgs a) {
    __shared__ __attribute__((aligned(16))) uint8_t lds[kTileLds];
    const int n_rb = a.row_blocks;
    const int m = blockIdx.x >> 3;
    const int seq = (m / kXcdCus) * (8 * kXcdCus) + (blockIdx.x & 7) * kXcdCus + m % kXcdCus;
    const int any = seq / n_rb;  // some tile of the block's expert
    if (any >= *a.n_tiles) return;  // block-uniform
    const int e = a.tile_expert[any];
    const int begin = a.expert_offsets[e];
    const int count = a.expert_offsets[e + 1] - begin;
    const int n_et = (count + 255) >> 8;                                             // the expert's tiles,
    const int first = any - (a.tile_row0[any] - begin) / even_tile_rows(count, 256, kPrefillStepBf16);  // the first of them
    const int local = seq - first * n_rb;
    const int rb = local / n_et;
    const int tile = first + local - rb * n_et;
    const int row0 = a.tile_row0[tile];
    const int nrows = a.tile_rows[tile];
    const int groups = min(4, a.rows / 64 - rb * 4);
    const int nt = (nrows + 15) >> 4;
    if (groups == 1) {
        tile_body<2, 8, EPI>(a, lds, e, row0, nrows, rb * 4);
    } else if (groups == 2) {
        if (nt > 8) tile_body<4, 4, EPI>(a, lds, e, row0, nrows, rb * 4);
        else tile_body<2, 4, EPI>(a, lds, e, row0, nrows, rb * 4);
    } else {
        if (nt > 12) tile_body<8, 2, EPI>(a, lds, e, row0, nrows, rb * 4);
        else if (nt > 8) tile_body<6, 2, EPI>(a, lds, e, row0, nrows, rb * 4);
        else if (nt > 4) tile_body<4, 2, EPI>(a, lds, e, row0, nrows, rb * 4);
        else tile_body<2, 2, EPI>(a, lds, e, row0, nrows, rb * 4);
    }
}

}  // namespace

// The kernel addresses an expert's matrix, gathered activation rows and the rows by slot of one block by 32-bit byte offsets.
bool expert_tile_fits(long long gathered_rows, int rows, int K) {
    return (gathered_rows > 256 ? gathered_rows : 256) * K * 2 <= 0xffffffffll && (long long)rows * K * 2 <= 0xffffffffll;
}

int launch_expert_tile_bf16(const ExpertGemmArgs& a, int epi, hipStream_t stream) {
    if (a.format != FMT_BF16 || a.rows % 64 != 0 || a.K % kTileStageElems != 0) return MOE_ERR_SHAPE;
    ExpertGemmArgs b = a;
    b.row_blocks = ceil_div(a.rows, kTileRows);
    const dim3 grid(ceil_div(a.max_tiles * b.row_blocks, 8 * kXcdCus) * 8 * kXcdCus);
    if (epi == EPI_SWIGLU_BF16) {
        hipLaunchKernelGGL((expert_tile_bf16_kernel<EPI_SWIGLU_BF16>), grid, dim3(512), 0, stream, b);
    } else if (epi == EPI_ROWS_F32) {
        hipLaunchKernelGGL((expert_tile_bf16_kernel<EPI_ROWS_F32>), grid, dim3(512), 0, stream, b);
    } else {
        return MOE_ERR_FORMAT;
    }
    return launch_status();
}

}  // namespace moe
