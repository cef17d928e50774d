// The q4 GEMM of a pass over a prompt: many rows of x, y = x W^T.
//
// The batched step's GEMM (batch.hip) keeps one 64-row tile of x and streams W past it; over many
// rows that form read every x fragment from LDS once per 32 columns and every scale and row sum once
// per chunk, and left the matrix units idle for 70 % of the time. Here:
//  - a wave computes 64 rows x 64 columns, so 18 KiB of LDS reads feed 32 MFMAs (17 KiB fed 16), and
//    a weight is dequantised once per 64 rows;
//  - the weights enter the matrix units as q - r, r the integer in 0..15 nearest the group's zero point z,
//    and what is left of the zero points, sum over the chunks of s (r - z) sum x, is the accumulators'
//    first value: one small product on the bf16 matrix units (f32 operands as three bf16 terms, six
//    products, to 2^-24), before the first chunk. A chunk then costs one fma per output value instead of
//    two, and no row sums from LDS. With r the products and the first value have the size of the sums
//    themselves, wherever the zero points lie. Error against 64 bits (2-norm, 1024 x 2048 x 1024, the
//    64-row form / this one): zeros 7.5, codes 0..15 2.0e-7 / 1.0e-7, zeros 0, codes 0..1 1.2e-7 / 1.0e-7,
//    zeros 15, codes 14..15 2.1e-6 / 1.0e-7 (r = 8 for every group: 1.0e-7, 1.2e-6, 1.1e-6). A chain of 32
//    chunks (K = 2048 in one split) adds a little: 1.3e-7, and 1.8e-7 for zeros far outside 0..15;
//  - the epilogue stages the next GEMM's operand 16 bytes a lane.
// A workgroup is 8 waves over 256 columns. 128 rows (KG = 1): 2 x 4 waves, every wave takes every
// chunk. 64 rows (KG = 2): 4 waves across, and the two halves of the workgroup take the even and the
// odd chunks; their sums meet in LDS at the end. The second form gives matrices with few columns twice
// the workgroups at the same LDS traffic per MFMA. Which form a column runs in depends on the matrix
// and GemmArgs::row_tiles, never on the rows of the call beside them, so where a caller fixes row_tiles a
// row's sums are added in the same order in every call.
// Measured (2048 rows, K = 2048; before: the 64-row form of batch.hip at two workgroups per CU): N =
// 12288 with its epilogue 257 -> 198 us (206 GFLOP of MFMA, 1.0 PFLOP/s; a loop of these MFMAs alone, on
// such data, reaches 1.85: the card's power limit), N = 8224 186 -> 161 us, N = 2048 60 -> 43 us, N = 2048
// over the 2B model's K (2048, 4096, 6144) 105 -> 76 us. What is left: a workgroup's start and end are
// ~10 us with its CU's matrix units idle, and a chunk takes 1.7 us for 1.1 of MFMA. Without the DMAs, the
// LDS reads and the vector work together the loop is 11 % faster. Measured and not kept: two 4-wave
// workgroups of 64 x 256 on a CU (N = 12288: 305 us), the halves of a workgroup one phase apart (+5 %),
// raised wave priority around the MFMAs (+3 %), the DMAs early or late in a chunk (+1 %), no scheduling
// fences, contiguous columns per XCD (no change).
#include <algorithm>
#include <type_traits>

#include "../error.hpp"
#include "common.hpp"
#include "launch.hpp"
#include "lds_dma.hpp"
#include "operand.hpp"
#include "q4_mfma.hpp"

namespace qne {

namespace {

using namespace lds_dma;

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));

// v as three bf16 terms (round to nearest: 27 bits in all, so the sum is v).
struct Bf3 {
    bf16x8_t t[3];
    __device__ __forceinline__ void set(int i, float v) {
        const __bf16 a = (__bf16)v;
        const float r = v - (float)a;
        const __bf16 b = (__bf16)r;
        t[0][i] = a;
        t[1][i] = b;
        t[2][i] = (__bf16)(r - (float)b);
    }
};

// s (r - z): what the products of q - r leave of a group's zero point (r as zero_int has it: both round
// halves to even). The empty asm keeps the compiler from a branch around it where only some lanes want it.
__device__ __forceinline__ float zero_rest(uint32_t szw) {
    const float z = hi_h(szw);
    float v = lo_h(szw) * (__builtin_amdgcn_fmed3f(rintf(z), 0.0f, 15.0f) - z);
    asm volatile("" : "+v"(v));
    return v;
}

constexpr int kWideCols = 256;  // W rows (output columns) of a workgroup
constexpr int kWideWaves = 8;
constexpr int kWideRing = 3;    // slots: one computed, two in flight

}  // namespace

// LDS of a workgroup: the ring of slots (x of two (row tile | chunk) halves, 8 W tiles of 32 rows, their
// scale / zero words), reused for the output tile; and the rows' 1 / rms.
template <int KG>
struct WideLds {
    static constexpr int kRows = 128 / KG;
    static constexpr int kSquares = 4;                // classes of 64 chunks
    static constexpr int kX = 2 * 2 * kFragBytes;
    static constexpr int kW = KG * 8 * 1024;
    static constexpr int kSz = KG * 8 * 128;
    static constexpr int kSlot = kX + kW + kSz;
    static constexpr int kOutStride = kWideCols + 4;  // staged output rows, padded against bank conflicts
    static constexpr int kRing = kWideRing * kSlot > kRows * kOutStride * 4 ? kWideRing * kSlot : kRows * kOutStride * 4;
    __attribute__((aligned(16))) uint8_t ring[kRing];
    float sinv[kRows];
    float parts[kSquares][512];                       // partial sums of the rows' x^2
};

// Column tile bx, row tile bz (of 128 / KG rows), split by: chunks [by cps, (by + 1) cps).
template <int KG>
__device__ __forceinline__ void wide_tile(const GemmArgs& a, WideLds<KG>& lds, const int bx, const int by, const int bz) {
    typedef WideLds<KG> L;
    constexpr int kRows = L::kRows, kX = L::kX, kW = L::kW, kSlot = L::kSlot, kOutStride = L::kOutStride;
    constexpr int kPer = 4 + KG + 1;                // DMAs of a wave per ring slot
    uint8_t* const ring = lds.ring;
    float* const sinv = lds.sinv;
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int hf = lane >> 5, l32 = lane & 31;
    const int half = w >> 2, nw = w & 3;            // half: row tile (KG 1) or chunk parity (KG 2)
    const int nchunks = a.K / kChunk, cpg = a.group / kChunk, ngroups = nchunks / cpg;
    const int c0 = by * a.cps, c1 = min(nchunks, c0 + a.cps);
    const int iters = (c1 - c0 + KG - 1) / KG;
    const int row0 = bz * kRows;
    const int last_tile = a.mpad / kBM - 1;
    const size_t tile_bytes = (size_t)nchunks * kChunkBytes;
    // this wave's half of x: rows 64 half.. of the workgroup (a tile past the rows: the last one, not
    // stored), or all its rows for every second chunk
    const uint8_t* xtile = a.frag + (size_t)min(KG == 1 ? bz * 2 + half : bz, last_tile) * tile_bytes;
    const int cfirst = c0 + (KG == 2 ? half : 0);   // this wave's first chunk
    // first W row (= output column) of tile t; a SwiGLU's even tiles are gate rows, the odd ones the
    // matching up rows, so a wave holds both factors of its 32 columns
    auto wrow0 = [&](int t) -> int {
        if (a.fuse == 1) return (t & 1 ? a.n_out : 0) + (bx * 4 + (t >> 1)) * 32;
        return (bx * 8 + t) * 32;
    };

    // sources of this wave's DMAs: 4 KiB of its half's x, W tile w, its words
    constexpr int kPieces = 2 * KG;                 // 16-byte pieces of a W row per slot
    const int tile0 = min(wrow0(w), a.N - 1);       // past N: row N - 1, not stored
    const uint8_t* wbase = (const uint8_t*)a.W + (size_t)tile0 * (a.K / 2);
    const uint8_t* szbase = (const uint8_t*)a.SZT + (size_t)(tile0 >> 5) * ngroups * 128;
    uint32_t woff[KG];
    int wchunk[KG];                                 // the piece's chunk within the slot
#pragma unroll
    for (int u = 0; u < KG; u++) {
        const int row = (64 / kPieces) * u + lane / kPieces;
        int piece = lane % kPieces;
        if (KG == 2) piece ^= (row >> 2) & 3;       // rows 4 apart on different banks
        wchunk[u] = piece >> 1;
        woff[u] = (uint32_t)(min(wrow0(w) + row, a.N - 1) - tile0) * (a.K / 2) + 16 * (piece & 1);
    }
    auto group = [&](int c) -> int { return cpg == 1 ? c : (int)((unsigned)c / (unsigned)cpg); };
    // DMA u (of kPer) of slot j: the words, x, W
    const uint32_t ring_lds = lds_address(ring);
    auto issue = [&](int j, int slot, int u) {
        const uint32_t base = ring_lds + slot * kSlot;
        const int c = c0 + KG * j;
        if (u == 0) {
            if (lane < 8 * KG) {
                if (KG == 1) dma16_at(szbase + (size_t)group(c) * 128, 16 * lane, base + kX + kW + 128 * w);
                else dma16_at(szbase, (uint32_t)group(min(c + (lane >> 3), c1 - 1)) * 128 + 16 * (lane & 7), base + kX + kW + KG * 128 * w);
            }
        } else if (u < 5) {
            const int o = 4096 * nw + 1024 * (u - 1);
            dma16_at(xtile + (size_t)min(c + (KG == 2 ? half : 0), c1 - 1) * kChunkBytes + o, 16 * lane, base + 2 * kFragBytes * half + o);
        } else {
            if (KG == 1) dma16_at(wbase + (size_t)c * 32, woff[0], base + kX + 1024 * w);
            else dma16_at(wbase, woff[u - 5] + min(c + wchunk[u - 5], c1 - 1) * 32, base + kX + KG * 1024 * w + 1024 * (u - 5));
        }
    };
    // acc's first value: sum over this wave's chunks of s (r - z) sum x. The chunks are the contraction,
    // 16 at a time; a batch's loads are in flight together, the first batch's (and the first sums of
    // x^2) ahead of the first chunks' DMAs.
    const int nmine = (c1 - cfirst + KG - 1) / KG;
    const float* xsum = (const float*)(xtile + kXsumOff) + l32;
    const uint32_t* szt[2];
#pragma unroll
    for (int t = 0; t < 2; t++) szt[t] = a.SZT + (size_t)(min(wrow0(2 * nw + t), a.N - 1) >> 5) * ngroups * 32 + l32;
    float xv[2][8];
    uint32_t sz[2][8];
    auto load_sums = [&](int b) {
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const int c = cfirst + KG * max(0, min(b + 8 * hf + i, nmine - 1)), g = group(min(c, c1 - 1));
#pragma unroll
            for (int t = 0; t < 2; t++) {
                xv[t][i] = xsum[(size_t)min(c, c1 - 1) * (kChunkBytes / 4) + 32 * t];
                sz[t][i] = szt[t][(size_t)g * 32];
            }
        }
    };
    load_sums(0);
    // A row's sum of x^2 in the order of row_inv_rms, whose thread c of 256 takes chunks c, c + 256, .. and
    // whose four waves of 64 threads are a butterfly each: here class q of 64 threads is thread t of the
    // row's 4 KG with the chunks 64 q + t + 4 KG k, and the trees below are the butterfly.
    const bool norm = a.norm && (a.direct || a.fuse);
    constexpr int TR = 4 * KG, KR = 64 / TR;
    const int rr = threadIdx.x % kRows, tr = threadIdx.x / kRows;
    const float* ssp = (const float*)(a.frag + (size_t)min((row0 + rr) / kBM, last_tile) * tile_bytes + kSsOff) + (rr & (kBM - 1));
    const int classes = min(L::kSquares, (nchunks + 63) / 64);
    float sq[KR];
    auto load_squares = [&](int first) {  // the chunks first.. of a class of 64 threads
#pragma unroll
        for (int k = 0; k < KR; k++) {
            const int c = first + tr + TR * k;
            const float v = ssp[(size_t)min(c, nchunks - 1) * (kChunkBytes / 4)];
            sq[k] = c < nchunks ? v : 0.0f;
        }
    };
    if (norm) load_squares(0);
    for (int j = 0; j < min(kWideRing - 1, iters); j++)
#pragma unroll
        for (int u = 0; u < kPer; u++) issue(j, j, u);
    if (norm) {
        for (int q = 0; q < classes; q++) {
            if (q > 0) load_squares(64 * q);
            for (int c0n = 64 * q + 256; c0n < nchunks; c0n += 256)
#pragma unroll
                for (int k = 0; k < KR; k++) {
                    const int c = c0n + tr + TR * k;
                    const float v = ssp[(size_t)min(c, nchunks - 1) * (kChunkBytes / 4)];
                    sq[k] += c < nchunks ? v : 0.0f;
                }
#pragma unroll
            for (int d = KR / 2; d >= 1; d >>= 1)
#pragma unroll
                for (int k = 0; k < d; k++) sq[k] += sq[k + d];
            lds.parts[q][tr * kRows + rr] = sq[0];
        }
    }
    float16_t acc[2][2] = {};
    for (int b = 0; b < nmine; b += 16) {
        Bf3 xa[2], wb[2];
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const bool live = b + 8 * hf + i < nmine;
#pragma unroll
            for (int t = 0; t < 2; t++) {
                const float rest = zero_rest(sz[t][i]);
                xa[t].set(i, live ? xv[t][i] : 0.0f);
                wb[t].set(i, live ? rest : 0.0f);
            }
        }
        if (b + 16 < nmine) load_sums(b + 16);
#pragma unroll
        for (int p = 2; p >= 0; p--)
#pragma unroll
            for (int q = 0; q <= p; q++)
#pragma unroll
                for (int cf = 0; cf < 2; cf++)
#pragma unroll
                    for (int rt = 0; rt < 2; rt++)
                        acc[cf][rt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xa[rt].t[q], wb[cf].t[p - q], acc[cf][rt], 0, 0, 0);
    }

    // A chunk runs as two phases, one per 32-row tile, of four k-steps: the first dequantises the
    // weights and keeps them for the second, which reads the next chunk's words and rounds its zero
    // points (at the start of their own chunk they delay its first product: N = 12288 201 -> 205 us). The scaled sums of a phase are added during the next
    // one, and the DMAs of a later slot go out between the steps, so the matrix unit has work
    // throughout a phase. The empty asm statements pin each step's vector work to its step: left
    // alone, the compiler gathers it at the end of the chunk and copies grp to keep it alive.
    int slot = 0, next_slot = kWideRing - 1;
    float16_t grp[2][2] = {};       // [column tile][row tile]
    float sc[2] = {};
    uint32_t szw[2];                // this wave's words of the chunk that comes next
    ZeroInt zi[2];
    auto read_words = [&](int at) {
        const uint8_t* wsz = ring + at * kSlot + kX + kW + 2 * nw * KG * 128 + (KG == 2 ? 128 * half : 0) + 4 * l32;
#pragma unroll
        for (int cf = 0; cf < 2; cf++) szw[cf] = *(const uint32_t*)(wsz + cf * KG * 128);
    };
    const int piece = KG == 1 ? hf : (2 * half + hf) ^ ((l32 >> 2) & 3);
    auto chunk = [&](int j, auto sends) {
        const uint8_t* xs = ring + slot * kSlot + 2 * kFragBytes * half;
        const uint8_t* ws = ring + slot * kSlot + kX + 2 * nw * KG * 1024;
        uint4 wq[2];
        half8_t b[2][4];
#pragma unroll
        for (int cf = 0; cf < 2; cf++) wq[cf] = *(const uint4*)(ws + cf * KG * 1024 + (l32 * kPieces + piece) * 16);
        half8_t ah = *(const half8_t*)(xs + frag_offset(0, 0, lane)), al = *(const half8_t*)(xs + kFragBytes + frag_offset(0, 0, lane));
#pragma unroll
        for (int p = 0; p < 8; p++) {
            const int rt = p >> 2, s = p & 3, np = p + 1;
            half8_t nh = ah, nl = al;
            if (np < 8) {
                nh = *(const half8_t*)(xs + frag_offset(np & 3, np >> 2, lane));
                nl = *(const half8_t*)(xs + kFragBytes + frag_offset(np & 3, np >> 2, lane));
            }
            if (rt == 0) {
#pragma unroll
                for (int cf = 0; cf < 2; cf++) b[cf][s] = nibbles8(s == 0 ? wq[cf].x : s == 1 ? wq[cf].y : s == 2 ? wq[cf].z : wq[cf].w, zi[cf]);
            }
            const float16_t zero = {};
#pragma unroll
            for (int cf = 0; cf < 2; cf++) grp[cf][rt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah, b[cf][s], s == 0 ? zero : grp[cf][rt], 0, 0, 0);
#pragma unroll
            for (int cf = 0; cf < 2; cf++) grp[cf][rt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(al, b[cf][s], grp[cf][rt], 0, 0, 0);
            if (p == 4) {
#pragma unroll
                for (int cf = 0; cf < 2; cf++) sc[cf] = lo_h(szw[cf]);
                read_words(slot + 1 == kWideRing ? 0 : slot + 1);
            }
            if (p == 7) {
#pragma unroll
                for (int cf = 0; cf < 2; cf++) zi[cf] = zero_int(szw[cf]);
            }
#pragma unroll
            for (int cf = 0; cf < 2; cf++)
#pragma unroll
                for (int e = 4 * s; e < 4 * s + 4; e++) {
                    float v = fmaf(sc[cf], grp[cf][1 - rt][e], acc[cf][1 - rt][e]);
                    asm volatile("" : "+v"(v));
                    acc[cf][1 - rt][e] = v;
                }
            if (sends && p < kPer) issue(j + kWideRing - 1, next_slot, p);
            __builtin_amdgcn_sched_barrier(0);
            ah = nh;
            al = nl;
        }
        slot = slot + 1 == kWideRing ? 0 : slot + 1;
        next_slot = next_slot + 1 == kWideRing ? 0 : next_slot + 1;
    };
    // A wave whose columns all lie past N only sends. At the barrier every part of slot j and the words
    // of slot j + 1 (its first DMA) have landed, and every wave is done with slot j - 1.
    const bool dead = wrow0(2 * nw) >= a.N;
    wait_vm<kPer - 1>();
    __syncthreads();
    read_words(0);
#pragma unroll
    for (int cf = 0; cf < 2; cf++) zi[cf] = zero_int(szw[cf]);
    for (int j = 0; j < iters - (kWideRing - 1); j++) {
        wait_vm<kPer - 1>();
        __syncthreads();
        if (dead) {
#pragma unroll
            for (int u = 0; u < kPer; u++) issue(j + kWideRing - 1, next_slot, u);
            next_slot = next_slot + 1 == kWideRing ? 0 : next_slot + 1;
        } else {
            chunk(j, std::true_type());
        }
    }
    if (iters > 1) {
        wait_vm<kPer - 1>();
        __syncthreads();
        if (!dead) chunk(iters - 2, std::false_type());
    }
    wait_vm<0>();
    __syncthreads();
    if (!dead && (KG == 1 || cfirst + KG * (iters - 1) < c1)) chunk(iters - 1, std::false_type());  // the odd half may have no last chunk
    if (threadIdx.x < kRows) {
        float inv = 1.0f;
        if (norm) {
            float sum = 0.0f;
            for (int q = 0; q < classes; q++) {
                float t[TR];
#pragma unroll
                for (int k = 0; k < TR; k++) t[k] = lds.parts[q][k * kRows + threadIdx.x];
#pragma unroll
                for (int d = TR / 2; d >= 1; d >>= 1)
#pragma unroll
                    for (int k = 0; k < d; k++) t[k] += t[k + d];
                sum += t[0];
            }
            inv = 1.0f / sqrtf(sum / (float)a.K + a.eps);
        }
        sinv[threadIdx.x] = inv;
    }
#pragma unroll
    for (int cf = 0; cf < 2; cf++)
#pragma unroll
        for (int e = 0; e < 16; e++) acc[cf][1][e] = fmaf(sc[cf], grp[cf][1][e], acc[cf][1][e]);
    __syncthreads();  // ring no longer read

    // KG = 2: the halves' sums, even + odd chunks; each half then owns one 32-row tile
    constexpr int RT = KG == 1 ? 2 : 1;
    if (KG == 2) {
        float* x = (float*)ring;  // [half's gift][nw][cf][e][lane]
#pragma unroll
        for (int cf = 0; cf < 2; cf++)
#pragma unroll
            for (int e = 0; e < 16; e++) x[(((half * 4 + nw) * 2 + cf) * 16 + e) * 64 + lane] = half ? acc[cf][0][e] : acc[cf][1][e];
        __syncthreads();
#pragma unroll
        for (int cf = 0; cf < 2; cf++)
#pragma unroll
            for (int e = 0; e < 16; e++) {
                const float o = x[((((1 - half) * 4 + nw) * 2 + cf) * 16 + e) * 64 + lane];
                acc[cf][0][e] = half ? o + acc[cf][1][e] : acc[cf][0][e] + o;
            }
        __syncthreads();
    }
    const int rb = KG == 1 ? 64 * half : 32 * half;  // this wave's first row of the workgroup
    if (!a.direct && !a.fuse) {  // split partials
#pragma unroll
        for (int cf = 0; cf < 2; cf++) {
            const int n = wrow0(2 * nw + cf) + l32;
            if (n >= a.N) continue;
#pragma unroll
            for (int rt = 0; rt < RT; rt++)
#pragma unroll
                for (int e = 0; e < 16; e++) {
                    const int r = row0 + rb + 32 * rt + 8 * (e / 4) + 4 * hf + (e % 4);
                    if (r < a.mpad) store_through(a.part + ((size_t)by * a.mpad + r) * a.N + n, acc[cf][rt][e]);
                }
        }
        return;
    }
    // the epilogue in registers; with frag_out the values also go to LDS, [row][column]
    float* so = (float*)ring;
    if (a.fuse == 1) {
        const int col = 32 * nw + l32, n = bx * 128 + col;
#pragma unroll
        for (int rt = 0; rt < RT; rt++)
#pragma unroll
            for (int e = 0; e < 16; e++) {
                const int r = rb + 32 * rt + 8 * (e / 4) + 4 * hf + (e % 4);
                const float v = silu(acc[0][rt][e] * sinv[r]) * (acc[1][rt][e] * sinv[r]);
                if (a.y && row0 + r < a.m) store_through(a.y + (size_t)(row0 + r) * a.y_stride + n, v);
                if (a.frag_out) so[r * kOutStride + col] = v;
            }
    } else {
#pragma unroll
        for (int cf = 0; cf < 2; cf++) {
            const int n = wrow0(2 * nw + cf) + l32;
            // the residual's loads all in flight before the first is used
            float hv[RT][16];
#pragma unroll
            for (int rt = 0; rt < RT; rt++)
#pragma unroll
                for (int e = 0; e < 16; e++) {
                    const int r = row0 + rb + 32 * rt + 8 * (e / 4) + 4 * hf + (e % 4);
                    hv[rt][e] = a.epi == EPI_ACCUMULATE && n < a.N && r < a.m ? a.y[(size_t)r * a.y_stride + n] : 0.0f;
                }
#pragma unroll
            for (int rt = 0; rt < RT; rt++)
#pragma unroll
                for (int e = 0; e < 16; e++) {
                    const int r = rb + 32 * rt + 8 * (e / 4) + 4 * hf + (e % 4);
                    const float g = acc[cf][rt][e] * sinv[r];
                    const float v = a.epi == EPI_ACCUMULATE ? hv[rt][e] + g : g;
                    if (a.y && n < a.N && row0 + r < a.m) store_through(a.y + (size_t)(row0 + r) * a.y_stride + n, v);
                    if (a.frag_out) so[r * kOutStride + (2 * nw + cf) * 32 + l32] = v;
                }
        }
    }
    if (!a.frag_out) return;
    __syncthreads();
    // the next GEMM's operand: a wave takes 32 rows x 64 columns at a time
    const int cols = a.fuse == 1 ? kWideCols / 2 : kWideCols, nck = cols / kChunk;
    const size_t out_tile = (size_t)(a.n_out / kChunk) * kChunkBytes;
    for (int it = w; it < kRows / 32 * nck; it += kWideWaves) {
        const int ch = it % nck, r = (it / nck) * 32 + l32, col = bx * cols + ch * kChunk;
        if (col >= a.n_out) continue;  // a whole chunk past the outputs
        float v[32], g[32];
#pragma unroll
        for (int q = 0; q < 8; q++) {
            const float4 t = *(const float4*)(so + r * kOutStride + ch * kChunk + 32 * hf + 4 * q);
            const float4 u = a.gain_out ? *(const float4*)(a.gain_out + col + 32 * hf + 4 * q) : make_float4(1.0f, 1.0f, 1.0f, 1.0f);
            v[4 * q] = t.x, v[4 * q + 1] = t.y, v[4 * q + 2] = t.z, v[4 * q + 3] = t.w;
            g[4 * q] = u.x, g[4 * q + 1] = u.y, g[4 * q + 2] = u.z, g[4 * q + 3] = u.w;
        }
        emit_x_rows(a.frag_out, out_tile, row0 + r, a.m, col / kChunk, v, g, a.order_out, lane);
    }
}

// Column tiles [0, a.wide_cols) as workgroups of 128 rows, the others as 64 rows with the chunks in two
// halves. One dimension, so that the second form's workgroups (half the time each) start as the first
// form's leave CUs free. Neighbouring workgroups take neighbouring column tiles of the same rows.
__global__ __launch_bounds__(64 * kWideWaves) void k_gemm_wide(const GemmArgs a) {
    __shared__ union {
        WideLds<1> one;
        WideLds<2> two;
    } lds;
    const int id = blockIdx.x, n1 = a.wide_cols, first = n1 * ((a.mpad + 127) / 128);
    if (id < first) {
        wide_tile<1>(a, lds.one, id % n1, 0, id / n1);
    } else {
        const int n2 = (a.N + kWideCols - 1) / kWideCols - n1, i = id - first;
        wide_tile<2>(a, lds.two, n1 + i % n2, i / n2 % a.splits, i / n2 / a.splits);
    }
}

// The same sums for a call of few rows, where the workgroups above would leave most CUs idle (64 rows,
// N = 2048: 8 of them, 43 us). A workgroup takes 32 rows x 32 CT columns, and its 8 waves take 8
// chunks at once: the products of a chunk do not depend on the other chunks', only the fma that scales
// them into the accumulator does. So each wave forms its chunk's products, from x and W straight out of
// L2 (nothing is shared between the waves), and leaves them in LDS, where wave w adds the 8 chunks'
// products of its 2 CT of the tile's accumulator registers in chunk order: the sums are bit for bit
// those of wide_tile. Every workgroup streams its rows of x whole, which bounds it (64 bytes a clock and
// CU; 264 KB at K = 2048). Writes split partials; the reduce applies the epilogue.
// Grid (ceil(N / (32 CT)), splits, ceil(m / 32)).
template <int CT>
__global__ __launch_bounds__(64 * kWideWaves) void k_gemm_short(const GemmArgs a) {
    constexpr int OWN = 2 * CT;                     // accumulator registers of a wave
    __shared__ float prod[kWideWaves][16 * CT][64];
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int hf = lane >> 5, l32 = lane & 31;
    const int nchunks = a.K / kChunk, cpg = a.group / kChunk, ngroups = nchunks / cpg;
    const int c0 = blockIdx.y * a.cps, c1 = min(nchunks, c0 + a.cps), nch = c1 - c0;
    const int row0 = blockIdx.z * 32, col0 = blockIdx.x * 32 * CT;
    const bool two = col0 / kWideCols >= a.wide_cols;  // even and odd chunks apart (the 64-row form)
    const uint8_t* xtile = a.frag + (size_t)(row0 / kBM) * nchunks * kChunkBytes;
    const int rt = (row0 / 32) & 1;                 // which half of the 64-row tile
    const uint32_t* szt[CT];
    const uint8_t* wrow[CT];
#pragma unroll
    for (int t = 0; t < CT; t++) {
        const int r = min(col0 + 32 * t, a.N - 1);
        szt[t] = a.SZT + (size_t)(r >> 5) * ngroups * 32 + l32;
        wrow[t] = (const uint8_t*)a.W + (size_t)min(col0 + 32 * t + l32, a.N - 1) * (a.K / 2) + 16 * hf;
    }
    const uint64_t inv_cpg = (uint64_t)(0xFFFFFFFFu / (unsigned)cpg) + 1;  // ceil(2^32 / cpg): c / cpg with no branch
    auto group = [&](int c) -> int { return (int)(((uint64_t)(unsigned)c * inv_cpg) >> 32); };
    const int own_t = w * OWN / 16, own_e = w * OWN % 16;  // this wave's column tile and registers

    struct Operands {
        half8_t h[4], l[4];
        uint4 w[CT];
        uint32_t wz[CT], sz[kWideWaves];
    } ops[2];  // of two rounds: one computed, the next one's loads in flight
    auto load = [&](Operands& o, int r) {  // round r: this wave's chunk, and the scales of its registers in all of them
        const int c = c0 + min(8 * r + w, nch - 1);
        const uint8_t* xs = xtile + (size_t)c * kChunkBytes;
#pragma unroll
        for (int s = 0; s < 4; s++) {
            o.h[s] = *(const half8_t*)(xs + frag_offset(s, rt, lane));
            o.l[s] = *(const half8_t*)(xs + kFragBytes + frag_offset(s, rt, lane));
        }
#pragma unroll
        for (int t = 0; t < CT; t++) {
            o.w[t] = *(const uint4*)(wrow[t] + (size_t)c * 32);
            o.wz[t] = szt[t][(size_t)group(c) * 32];
        }
        const uint32_t* sp = CT == 1 || own_t == 0 ? szt[0] : szt[CT - 1];
#pragma unroll
        for (int k = 0; k < kWideWaves; k++) o.sz[k] = sp[(size_t)group(c0 + min(8 * r + k, nch - 1)) * 32];
    };
    load(ops[0], 0);

    // the accumulators' first values, as in wide_tile: wave (parity, column tile)
    if (w < (two ? 2 : 1) * CT) {
        const int t = w % CT, step = two ? 2 : 1, cfirst = c0 + w / CT, nmine = (c1 - cfirst + step - 1) / step;
        const float* xsum = (const float*)(xtile + kXsumOff) + 32 * rt + l32;
        float16_t z = {};
        for (int b = 0; b < nmine; b += 16) {
            Bf3 xa, wb;
            float xv[8];
            uint32_t sv[8];
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const int c = cfirst + step * min(b + 8 * hf + i, nmine - 1);
                xv[i] = xsum[(size_t)c * (kChunkBytes / 4)];
                sv[i] = (CT == 1 || t == 0 ? szt[0] : szt[CT - 1])[(size_t)group(c) * 32];
            }
#pragma unroll
            for (int i = 0; i < 8; i++) asm volatile("" : "+v"(xv[i]), "+v"(sv[i]));  // keeps the loads together
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const bool live = b + 8 * hf + i < nmine;
                const float rest = zero_rest(sv[i]);
                xa.set(i, live ? xv[i] : 0.0f);
                wb.set(i, live ? rest : 0.0f);
            }
#pragma unroll
            for (int p = 2; p >= 0; p--)
#pragma unroll
                for (int q = 0; q <= p; q++) z = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xa.t[q], wb.t[p - q], z, 0, 0, 0);
        }
#pragma unroll
        for (int e = 0; e < 16; e++) prod[w / CT][16 * t + e][lane] = z[e];
    }
    __syncthreads();
    float acc[2][OWN];
#pragma unroll
    for (int i = 0; i < OWN; i++) {
        acc[0][i] = prod[0][w * OWN + i][lane];
        acc[1][i] = two ? prod[1][w * OWN + i][lane] : 0.0f;
    }
    const int rounds = (nch + kWideWaves - 1) / kWideWaves;
    auto round = [&](const Operands& cur, int r) {
        float16_t grp[CT] = {};
        ZeroInt zi[CT];
#pragma unroll
        for (int t = 0; t < CT; t++) zi[t] = zero_int(cur.wz[t]);
#pragma unroll
        for (int s = 0; s < 4; s++) {
            half8_t b[CT];
#pragma unroll
            for (int t = 0; t < CT; t++) b[t] = nibbles8(s == 0 ? cur.w[t].x : s == 1 ? cur.w[t].y : s == 2 ? cur.w[t].z : cur.w[t].w, zi[t]);
#pragma unroll
            for (int t = 0; t < CT; t++) grp[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(cur.h[s], b[t], grp[t], 0, 0, 0);
#pragma unroll
            for (int t = 0; t < CT; t++) grp[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(cur.l[s], b[t], grp[t], 0, 0, 0);
        }
        __syncthreads();  // the previous round's products are used
#pragma unroll
        for (int t = 0; t < CT; t++)
#pragma unroll
            for (int e = 0; e < 16; e++) prod[w][16 * t + e][lane] = grp[t][e];
        __syncthreads();
        float p[kWideWaves][OWN];
#pragma unroll
        for (int k = 0; k < kWideWaves; k++)
#pragma unroll
            for (int i = 0; i < OWN; i++) p[k][i] = prod[k][w * OWN + i][lane];
        const int live = nch - kWideWaves * r;  // chunks past the split leave the sums as they are
#pragma unroll
        for (int k = 0; k < kWideWaves; k++) {
            const float sc = lo_h(cur.sz[k]);
#pragma unroll
            for (int i = 0; i < OWN; i++) {
                float& d = two ? acc[k & 1][i] : acc[0][i];
                const float v = fmaf(sc, p[k][i], d);
                d = k < live ? v : d;
            }
        }
    };
    for (int r = 0; r < rounds; r += 2) {
        load(ops[1], r + 1);
        round(ops[0], r);
        if (r + 1 >= rounds) break;
        load(ops[0], r + 2);
        round(ops[1], r + 1);
    }
    const int n = col0 + 32 * own_t + l32;
    if (n >= a.N) return;
#pragma unroll
    for (int i = 0; i < OWN; i++) {
        const int e = own_e + i, r = row0 + 8 * (e / 4) + 4 * hf + (e % 4);
        store_through(a.part + ((size_t)blockIdx.y * a.mpad + r) * a.N + n, two ? acc[0][i] + acc[1][i] : acc[0][i]);
    }
}

// How many column tiles run as 128-row workgroups: all, none, or as many as fill whole rounds of the
// 256 CUs, whichever takes the fewest rounds in all (a 64-row workgroup counts as 0.6 of one: 42
// against 70 us at K = 2048). Split K and a caller's pass of one row tile take the second form.
int gemm_wide_cols(int N, int row_tiles, int splits) {
    const int cols = (N + kWideCols - 1) / kWideCols, mt = (row_tiles + 1) / 2;
    if (splits > 1) return 0;
    auto rounds = [](int wgs) { return (wgs + 255) / 256; };
    int best = 0;
    float cost = 0.0f;
    for (int n : {cols, cols * mt / 256 * 256 / mt, 0}) {
        const float c = (float)rounds(n * mt) + 0.6f * (float)rounds((cols - n) * row_tiles);
        if (n == cols || c < cost) best = n, cost = c;
    }
    return best;
}

// Where the short form (with its reduce) beats wide_tile, both measured on the 2B model's matrices, mean
// over the layers, us, short / wide: N = 2048, 64 rows 24 / 59, 256 rows (256 workgroups) 33 / 59, 512
// rows (512) 53 / 60; N = 8224, 64 rows 32 / 57, 128 rows (516) 49 / 57, 256 rows (1032) 81 / 58; N =
// 12288, 128 rows (768) 51 / 57, 256 rows (1536) 93 / 60.
bool gemm_is_short(const GemmArgs& a) {
    const int wgs = (a.N + 63) / 64 * ((a.m + 31) / 32) * a.splits;
    return wgs <= (a.m <= 128 ? 768 : 512);
}

// Calls of 257 to 2048 rows, N 64..12288, K 512..6144. A CU pays ~10 us for a pass's form before its matrix
// units are busy, so it takes 5 of the 64-row form's 256 x 64 x 64 tile chunks a CU to be worth that (N x K
// x rows, us, 64-row form / pass: 1847 x 640 x 502, 640 tile chunks, 25 / 29; 1557 x 1216 x 361, 798, 26 / 29;
// 977 x 2816 x 445, 1232, 34 / 29; 442 x 5824 x 1489, 4368, 60 / 43), unless the pass saves the partials
// too, one split with its own epilogue (3233 x 640 x 600, 1300, 39 / 24). Of 500 drawn calls (log-uniform)
// 2 are over 1 % slower than the 64-row form with its staging in two launches (2 and 5 %); with passes
// throughout a third were, by up to 1.4x.
bool gemm_wide_pays(const GemmArgs& a) {
    const int64_t tiles = (int64_t)((a.N + kWideCols - 1) / kWideCols) * a.row_tiles;
    if (tiles * (a.K / kChunk) > 1344) return true;
    const bool own = a.epi != EPI_SWIGLU || (a.n_out % (kWideCols / 2) == 0 && a.K <= 64 * kChunk);
    return a.splits == 1 && own && !gemm_is_short(a);
}

void launch_gemm_wide(GemmArgs a, hipStream_t st) {
    const int cols = (a.N + kWideCols - 1) / kWideCols;
    a.wide_cols = gemm_wide_cols(a.N, a.row_tiles, a.splits);
    if (!a.fuse && !a.direct && gemm_is_short(a)) {
        const int tiles = (a.m + 31) / 32;
        if ((a.N + 63) / 64 * tiles * a.splits < 256)
            hipLaunchKernelGGL(k_gemm_short<1>, dim3((a.N + 31) / 32, a.splits, tiles), dim3(64 * kWideWaves), 0, st, a);
        else
            hipLaunchKernelGGL(k_gemm_short<2>, dim3((a.N + 63) / 64, a.splits, tiles), dim3(64 * kWideWaves), 0, st, a);
        return;
    }
    const int wgs = a.wide_cols * ((a.mpad + 127) / 128) + (cols - a.wide_cols) * a.splits * (a.mpad / kBM);
    hipLaunchKernelGGL(k_gemm_wide, dim3(wgs), dim3(64 * kWideWaves), 0, st, a);
}

}  // namespace qne
