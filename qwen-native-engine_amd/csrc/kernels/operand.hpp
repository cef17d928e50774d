// The x operand of the batched GEMM (k_gemm) in memory, and the device helpers that write and read
// it: the kernels that produce a GEMM's input (the embedding, the split reduce, the GDN step, the
// attention combine) stage it directly in this form.
//
// x is staged in chunks of 64 columns for tiles of 64 rows: per chunk the f16 halves hi = f16(x),
// lo = f16(x - hi) in v_mfma_f32_32x32x16_f16 A-operand order, then each row's sum of hi + lo and
// sum of x^2 over the chunk.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "common.hpp"

namespace qne {

constexpr int kBM = 64;            // rows of x per GEMM (sequences)
constexpr int kChunk = 64;         // columns per staged chunk
constexpr int kFragBytes = 8192;   // one half (hi or lo) of a chunk: 4 k-steps x 2 row tiles x 64 lanes x 16 B
constexpr int kXsumOff = 2 * kFragBytes;           // per-row sums of hi + lo over the chunk
constexpr int kSsOff = kXsumOff + kBM * 4;           // per-row sums of x^2 (raw x) over the chunk
constexpr int kChunkBytes = kSsOff + kBM * 4;        // a staged chunk in memory

// Operand layout of v_mfma_f32_32x32x16_f16 (lane l): A[l % 32][8 (l / 32) + i], B[8 (l / 32) + i][l % 32],
// D register j = [8 (j / 4) + 4 (l / 32) + j % 4][l % 32]. The 16 k-slots of k-step s of a chunk are
// chunk columns 32 (l / 32) + 8 s + i, the same for A and B, so a lane's q4 bytes of a chunk (16) are
// contiguous. In a staged chunk, fragment (s, row tile mt) of a half is 64 lanes x 16 bytes.
__device__ __forceinline__ int frag_offset(int s, int mt, int lane) { return ((s * 2 + mt) * 64 + lane) * 16; }

// Writes one value of the x operand of a GEMM: row r, column c, value v (times gain g). The 64
// lanes of the calling wave hold the 64 columns of one chunk of row r (all lanes call it), so the
// chunk's sums of hi + lo and of v^2 are wave sums. lo is what hi leaves of the unrounded product
// v g (one fma), and a pair's squares are added with one rounding. q4order: the column order of the q4 GEMM's B
// operand within each 8 columns, [0, 4, 1, 5, 2, 6, 3, 7] (nibbles8); else natural. Rows come in
// tiles of 64: tile r / 64 of the operand starts tile_bytes (the K / 64 chunks of one tile) after
// the previous one.
__device__ __forceinline__ void emit_x(uint8_t* __restrict__ frag, size_t tile_bytes, int r, int c, float v, float g,
                                       int q4order, int lane) {
#pragma clang fp contract(off)  // the sums' rounding is the same wherever an operand is staged
    const float xg = v * g;
    const float hi = (float)(_Float16)xg;
    const float lo = (float)(_Float16)fmaf(v, g, -hi);
    const int chunk = c / kChunk, kk = c % kChunk, hf = kk / 32, st = (kk % 32) / 8, i = kk % 8;
    const int slot = q4order ? 2 * (i % 4) + i / 4 : i;
    const int rr = r & (kBM - 1);
    uint8_t* tile = frag + (size_t)(r / kBM) * tile_bytes + (size_t)chunk * kChunkBytes;
    uint8_t* dst = tile + frag_offset(st, rr >> 5, 32 * hf + (rr & 31)) + 2 * slot;
    *(uint16_t*)dst = __builtin_bit_cast(uint16_t, (_Float16)hi);
    *(uint16_t*)(dst + kFragBytes) = __builtin_bit_cast(uint16_t, (_Float16)lo);
    const float sq = v * v;
    const float xs = wave_sum_dpp(hi + lo), ss = wave_sum_dpp_pairs(fmaf(v, v, QNE_DPP(sq, kDppXor1)));
    if (lane == 0) {
        float* sums = (float*)tile;
        sums[kXsumOff / 4 + rr] = xs;
        sums[kSsOff / 4 + rr] = ss;
    }
}

// The same for a wave that holds 32 rows of one chunk: lane 32 hf + row has the chunk's columns
// 32 hf + 8 s + i (s, i: v[8 s + i], times g[8 s + i]) of row r = 32 k + row, so each half's eight
// stores are whole contiguous KiB (emit_x: 2 bytes a lane). The sums are added in emit_x's order
// (a balanced tree over the columns), so the operand's bits are the same. Rows >= m are not written.
__device__ __forceinline__ void emit_x_rows(uint8_t* __restrict__ frag, size_t tile_bytes, int r, int m, int chunk,
                                            const float (&v)[32], const float (&g)[32], int q4order, int lane) {
#pragma clang fp contract(off)
    uint8_t* tile = frag + (size_t)(r / kBM) * tile_bytes + (size_t)chunk * kChunkBytes;
    const int rr = r & (kBM - 1);
    float xs[4], ss[4];
#pragma unroll
    for (int s = 0; s < 4; s++) {
        uint16_t hi[8], lo[8];
        float xt[8], st[4];
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const float xg = v[8 * s + i] * g[8 * s + i];
            const _Float16 h = (_Float16)xg, l = (_Float16)fmaf(v[8 * s + i], g[8 * s + i], -(float)h);
            hi[i] = __builtin_bit_cast(uint16_t, h);
            lo[i] = __builtin_bit_cast(uint16_t, l);
            xt[i] = (float)h + (float)l;
        }
        // emit_x's lane 0 sees the first four columns from their even lanes and the next four, mirrored, from
        // their odd ones: that lane's square is the unrounded one
#pragma unroll
        for (int p = 0; p < 4; p++) {
            const int own = 2 * p + p / 2, other = own ^ 1;
            st[p] = fmaf(v[8 * s + own], v[8 * s + own], v[8 * s + other] * v[8 * s + other]);
        }
        xs[s] = ((xt[0] + xt[1]) + (xt[2] + xt[3])) + ((xt[4] + xt[5]) + (xt[6] + xt[7]));
        ss[s] = (st[0] + st[1]) + (st[2] + st[3]);
        uint32_t hw[4], lw[4];
#pragma unroll
        for (int p = 0; p < 4; p++) {  // word p: slots 2 p, 2 p + 1 (q4 order: columns p, p + 4)
            const int a = 2 * p, b = 2 * p + 1;
            hw[p] = q4order ? hi[p] | (uint32_t)hi[p + 4] << 16 : hi[a] | (uint32_t)hi[b] << 16;
            lw[p] = q4order ? lo[p] | (uint32_t)lo[p + 4] << 16 : lo[a] | (uint32_t)lo[b] << 16;
        }
        if (r < m) {
            uint8_t* dst = tile + frag_offset(s, rr >> 5, lane);
            *(uint4*)dst = make_uint4(hw[0], hw[1], hw[2], hw[3]);
            *(uint4*)(dst + kFragBytes) = make_uint4(lw[0], lw[1], lw[2], lw[3]);
        }
    }
    float xt = (xs[0] + xs[1]) + (xs[2] + xs[3]), st = (ss[0] + ss[1]) + (ss[2] + ss[3]);
    xt += lane_xor32(xt, lane);
    st += lane_xor32(st, lane);
    if (r < m && lane < 32) {
        float* sums = (float*)tile;
        sums[kXsumOff / 4 + rr] = xt;
        sums[kSsOff / 4 + rr] = st;
    }
}

// 1 / rms of row r from the staged chunk sums of x^2 (the RMSNorm of the GEMM's input, applied to
// its output: y = (1 / rms) W (x * gain)). Called by every one of the NT threads of the workgroup
// (a multiple of 256: with K <= 16384 the wave sums and their order are those of a 256-thread
// workgroup, the waves past the fourth adding zeros).
template <int NT>
__device__ __forceinline__ float row_inv_rms(const uint8_t* __restrict__ frag, int nchunks, int K, float eps, int r,
                                             float* red) {
    const uint8_t* tile = frag + (size_t)(r / kBM) * nchunks * kChunkBytes;
    float ss = 0.0f;
    for (int c = threadIdx.x; c < nchunks; c += NT) ss += ((const float*)(tile + (size_t)c * kChunkBytes))[kSsOff / 4 + (r & (kBM - 1))];
    ss = block_sum<NT>(ss, red);
    return 1.0f / sqrtf(ss / (float)K + eps);
}

// Up to 8 split partials of one output value in flight at once, summed in split order (the order
// of k_gemm_reduce: terms past the splits are +0 and leave the sum unchanged).
constexpr int kFoldSplits = 8;
struct Split8 {
    float v[kFoldSplits];
    __device__ __forceinline__ void load(const float* p, int splits, size_t stride) {
#pragma unroll
        for (int s = 0; s < kFoldSplits; s++) v[s] = s < splits ? p[s * stride] : 0.0f;
    }
    __device__ __forceinline__ float sum(const float* p, int splits, size_t stride) const {
        float g = v[0];
#pragma unroll
        for (int s = 1; s < kFoldSplits; s++) g += v[s];
        for (int s = kFoldSplits; s < splits; s++) g += p[s * stride];
        return g;
    }
};

}  // namespace qne
