// MXFP4 (e2m1 codes + e8m0 block scales) support: reference-exact dequantisation, the load-time
// repack into the tiled layout the fused expert kernels stream, its inverse, and a tiled -> bf16
// expansion through the same conversion the fused kernels use.
// Arithmetic contract: tools/model_export/gpt-oss-20b/export_model_bin.py:75-133.
#include "common.h"
#include "kernels.h"

namespace moe {

// ---- canonical layout -> bf16, every scale byte ------------------------------------------------
// Bound by its stores (4 bytes out for every byte in).  Four lanes share an MX block and each takes one dword of codes, so
// a store instruction of the wave writes 1 KiB of consecutive bytes; with a thread to a block it wrote 64 pieces of 16
// bytes, 64 apart.  Measured on the expert tensors of a layer (32 experts, 2.02 GB in all): 641 us before, 338 now (6.0
// TB/s; 352 with four dwords to a lane).  A wave works on kDequantRun consecutive runs of 64 dwords, all loads first.  Scale
// bytes 0 and 255 take the integer routine, the hardware conversion is exact for all others.
constexpr int kDequantRun = 8;

__global__ __launch_bounds__(256) void dequant_mxfp4_kernel(const uint32_t* __restrict__ codes,
                                                            const uint8_t* __restrict__ scales, long long n_dwords,
                                                            u32x4* __restrict__ out) {
    const int lane = threadIdx.x & 63;
    const long long first = ((long long)blockIdx.x * 4 + (threadIdx.x >> 6)) * (64 * kDequantRun) + lane;
    uint32_t w[kDequantRun], s[kDequantRun];
#pragma unroll
    for (int i = 0; i < kDequantRun; ++i) {
        const long long d = first + i * 64;
        const bool in = d < n_dwords;
        w[i] = in ? codes[d] : 0u;
        s[i] = in ? scales[d >> 2] : 1u;
    }
#pragma unroll
    for (int i = 0; i < kDequantRun; ++i) {
        uint32_t o[4];
        if (__ballot(s[i] == 0u || s[i] == 255u) == 0) {
            mxfp4_dword_to_bf16x8(w[i], mxfp4_scale_to_f32(s[i]), o);
        } else {
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                const uint32_t byte = (w[i] >> (8 * b)) & 0xFFu;
                o[b] = mxfp4_code_to_bf16_bits(byte & 0xFu, s[i]) | (mxfp4_code_to_bf16_bits(byte >> 4, s[i]) << 16);
            }
        }
        const long long d = first + i * 64;
        if (d < n_dwords) __builtin_nontemporal_store(u32x4{o[0], o[1], o[2], o[3]}, out + d);
    }
}

int launch_dequant_mxfp4(const uint8_t* blocks, const uint8_t* scales, long long n_blocks, uint16_t* out,
                         hipStream_t stream) {
    const unsigned grid = (unsigned)ceil_div(n_blocks * 4, (long long)(256 * kDequantRun));
    hipLaunchKernelGGL(dequant_mxfp4_kernel, dim3(grid), dim3(256), 0, stream,
                       reinterpret_cast<const uint32_t*>(blocks), scales, n_blocks * 4, reinterpret_cast<u32x4*>(out));
    return launch_status();
}

// ---- tiled layout ------------------------------------------------------------------------------
// Per expert, weight rows are taken in groups of 64; each group is four MFMA row tiles of 16 rows
// (row order inside the group: tile_row_in_group).  A tile stores its K/32 MX blocks chunk by
// chunk, a chunk being four consecutive MX blocks (128 elements) of all 16 rows:
//     blocks : tile t, chunk c, lane l = (blk%4)*16 + q, 16 bytes      -> t*G*256 + c*1024 + l*16
//              (a ragged last chunk holds only its G%4 block columns)
//     scales : tile t, chunk quad c/4, lane l, byte c%4               -> t*SQ*256 + (c/4)*256 + l*4 + c%4
// with G = K/32 and SQ = ceil(ceil(G/4)/4).  One wave-wide 128-bit load fetches one chunk of a tile
// (1 KiB, contiguous); one dword load per lane fetches the scales of four chunks.
void mxfp4_tiled_bytes(int rows, int K, size_t* block_bytes, size_t* scale_bytes) {
    const int G = K / 32;
    const size_t tiles = (size_t)(rows / 64) * 4;
    if (block_bytes) *block_bytes = tiles * (size_t)G * 256;
    if (scale_bytes) *scale_bytes = tiles * (size_t)ceil_div(ceil_div(G, 4), 4) * 256;
}

struct TiledAddr {
    size_t block_off;
    size_t scale_off;
};

MOE_DEVICE TiledAddr tiled_addr(int e, int row, int blk, int G, size_t block_bytes, size_t scale_bytes) {
    const int group = row >> 6;
    const int i = row & 63;
    const int r = (i & 15) >> 2;
    const int q = ((i >> 4) << 2) | (i & 3);
    const size_t tile = (size_t)group * 4 + r;
    const int c = blk >> 2;
    const int lane = ((blk & 3) << 4) | q;
    const int SQ = (((G + 3) >> 2) + 3) >> 2;
    TiledAddr a;
    a.block_off = (size_t)e * block_bytes + tile * (size_t)G * 256 + (size_t)c * 1024 + (size_t)lane * 16;
    a.scale_off = (size_t)e * scale_bytes + tile * (size_t)SQ * 256 + (size_t)(c >> 2) * 256 + (size_t)lane * 4 + (c & 3);
    return a;
}

// Repack and its inverse, bound by memory (every byte in once, out once).  A wave takes a quad of chunks of one row tile:
// lane (b, q) = b * 16 + q moves MX blocks 4c + b, c = 0..3, of tile row q, so an instruction's 64 pieces of 16 bytes are
// 1 KiB of consecutive bytes on the tiled side and 64 bytes of each of 16 rows on the checkpoint side, whose lines the
// wave's next three instructions finish; a lane's four scale bytes are one dword on the tiled side.  With a thread to an
// MX block in the order of the checkpoint side every tiled-side access was 64 separate pieces and every scale a store
// of one byte: 369 us for a layer's expert tensors (32 experts, 0.85 GB in all), 188 now (4.5 TB/s, what a plain copy of
// this size reaches).  Non-temporal hints go where an instruction takes whole lines, i.e. on the tiled side only (on both
// sides 221 us, on none 196).  Scale bytes of MX blocks that do not exist (ragged last quad) are written as 0.
template <bool INVERSE>
__global__ __launch_bounds__(256) void mxfp4_repack_kernel(const uint8_t* __restrict__ src_blocks,
                                                           const uint8_t* __restrict__ src_scales,
                                                           uint8_t* __restrict__ dst_blocks,
                                                           uint8_t* __restrict__ dst_scales, int rows, int G,
                                                           long long n_waves) {
    const int lane = threadIdx.x & 63;
    const long long wave = (long long)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (wave >= n_waves) return;
    const int SQ = (((G + 3) >> 2) + 3) >> 2;
    const long long tile = wave / SQ;  // over all experts
    const int quad = (int)(wave - tile * SQ);
    const int q = lane & 15, b = lane >> 4;
    // rows % 64 == 0: the 64-row groups of all experts follow each other on both sides
    const long long row = (tile >> 2) * 64 + tile_row_in_group((int)(tile & 3), q);
    const size_t flat = (size_t)row * G + 16 * quad + b;            // MX block on the checkpoint side, chunk 0
    const size_t tiled = (size_t)tile * G * 256 + (size_t)quad * 4096 + (size_t)lane * 16;
    const size_t tiled_s = ((size_t)tile * SQ + quad) * 256 + (size_t)lane * 4;
    u32x4 v[4];
    uint32_t s = 0;
    if (INVERSE) s = *reinterpret_cast<const uint32_t*>(src_scales + tiled_s);
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        if (16 * quad + 4 * c + b < G) {
            if (INVERSE) v[c] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(src_blocks + tiled + c * 1024));
            else v[c] = *reinterpret_cast<const u32x4*>(src_blocks + (flat + 4 * c) * 16);
            if (!INVERSE) s |= (uint32_t)src_scales[flat + 4 * c] << (8 * c);
        }
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        if (16 * quad + 4 * c + b < G) {
            if (INVERSE) {
                *reinterpret_cast<u32x4*>(dst_blocks + (flat + 4 * c) * 16) = v[c];
                dst_scales[flat + 4 * c] = (uint8_t)(s >> (8 * c));
            } else {
                __builtin_nontemporal_store(v[c], reinterpret_cast<u32x4*>(dst_blocks + tiled + c * 1024));
            }
        }
    }
    if (!INVERSE) *reinterpret_cast<uint32_t*>(dst_scales + tiled_s) = s;
}

__global__ void fill_zero_kernel(uint32_t* __restrict__ p, size_t n) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0u;
}

int launch_fill_zero(uint32_t* words, size_t n, hipStream_t stream) {
    if (n == 0) return MOE_OK;
    hipLaunchKernelGGL(fill_zero_kernel, dim3((unsigned)ceil_div(n, (size_t)256)), dim3(256), 0, stream, words, n);
    return launch_status();
}

int launch_mxfp4_repack(const uint8_t* blocks, const uint8_t* scales, int E, int rows, int K,
                        uint8_t* tiled_blocks, uint8_t* tiled_scales, bool inverse, hipStream_t stream) {
    const int G = K / 32;
    const long long n_waves = (long long)E * (rows / 16) * ceil_div(ceil_div(G, 4), 4);
    const unsigned grid = (unsigned)ceil_div(n_waves, 4ll);
    if (!inverse) {
        hipLaunchKernelGGL(mxfp4_repack_kernel<false>, dim3(grid), dim3(256), 0, stream, blocks, scales, tiled_blocks,
                           tiled_scales, rows, G, n_waves);
    } else {
        // here `blocks`/`scales` are the canonical destination, tiled_* the source
        hipLaunchKernelGGL(mxfp4_repack_kernel<true>, dim3(grid), dim3(256), 0, stream, tiled_blocks, tiled_scales,
                           const_cast<uint8_t*>(blocks), const_cast<uint8_t*>(scales), rows, G, n_waves);
    }
    return launch_status();
}

// Tiled -> row-major bf16 [E, rows, K] through mxfp4_dword_to_bf16x8, the conversion of the fused
// expert kernels.
__global__ __launch_bounds__(256) void mxfp4_tiled_to_bf16_kernel(const uint8_t* __restrict__ tiled_blocks,
                                                                  const uint8_t* __restrict__ tiled_scales,
                                                                  u32x4* __restrict__ out, int E, int rows, int G,
                                                                  size_t block_bytes, size_t scale_bytes) {
    const long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    const long long total = (long long)E * rows * G;
    if (idx >= total) return;
    const int blk = (int)(idx % G);
    const long long er = idx / G;
    const int row = (int)(er % rows);
    const int e = (int)(er / rows);
    const TiledAddr t = tiled_addr(e, row, blk, G, block_bytes, scale_bytes);
    const u32x4 raw = *reinterpret_cast<const u32x4*>(tiled_blocks + t.block_off);
    const float sc = mxfp4_scale_to_f32(tiled_scales[t.scale_off]);
#pragma unroll
    for (int d = 0; d < 4; ++d) {
        uint32_t o[4];
        mxfp4_dword_to_bf16x8(raw[d], sc, o);
        out[idx * 4 + d] = u32x4{o[0], o[1], o[2], o[3]};
    }
}

int launch_mxfp4_tiled_to_bf16(const uint8_t* tiled_blocks, const uint8_t* tiled_scales, int E, int rows, int K,
                               uint16_t* out, hipStream_t stream) {
    const int G = K / 32;
    size_t bb, sb;
    mxfp4_tiled_bytes(rows, K, &bb, &sb);
    const long long total = (long long)E * rows * G;
    hipLaunchKernelGGL(mxfp4_tiled_to_bf16_kernel, dim3((unsigned)ceil_div(total, (long long)256)), dim3(256), 0,
                       stream, tiled_blocks, tiled_scales, reinterpret_cast<u32x4*>(out), E, rows, G, bb, sb);
    return launch_status();
}

}  // namespace moe
