// append_int8.h -- the quantising append into an int8 paged cache, shared by pa_kv_append, the
// last-token append of pa_paged_decode_append and pa_write_block_f32.
//
// Policy (the reference's QuantizeSymmetric / Dequantize, Quantization/Operations/
// QuantizationOperations.cs:188-200, applied per (block, KV head) with a running absmax): a
// segment is a maximal run of consecutive tokens of the call whose slots are valid and lie in one
// block. Segments are applied in call order. Writing row 0 starts the block afresh (scale =
// segment absmax / 127); otherwise a segment whose absmax exceeds the block's grows the scale and
// requantises every row it does not overwrite; the segment's rows are then quantised with the
// block's (possibly grown) scale.
//
// Runs: a block whose tokens of the call are one run of consecutive slots takes append_int8_run.
// Ownership, otherwise: the workgroup of the first token of the call that lands in a block owns that
// block and applies every segment of it, in call order, one wave per (KV head, K|V)
// (append_int8_segments). A block's tokens may therefore arrive in any order, split by invalid slots
// or by other blocks' tokens, without two workgroups touching one block.
#pragma once

#include "pa_internal.h"

namespace pa {

__device__ __forceinline__ float load_act(const void* p, bool bf16, int64_t i) {
    return bf16 ? bf16_to_f32(static_cast<const uint16_t*>(p)[i]) : static_cast<const float*>(p)[i];
}

// One segment [s, e) of block blk for KV head h, K (is_v false) or V, applied by one wave (64
// lanes; lane l owns dims l, l + 64, ..). slot_at(t) is token t's slot; src holds the tokens'
// values in the activation dtype, token t's (head h, dim d) at t * tok_stride + h * D + d. The
// tile of (blk, h) is K [16][D] or V [D][16] in `cache`. (amax, cur_scale) carry the block's
// statistics from one segment of this (block, head) to the next: have_stats false loads them.
template <int D, typename SlotAt>
__device__ __forceinline__ void append_int8_apply(const void* src, bool in_bf16, int64_t tok_stride, SlotAt slot_at,
                                                  int32_t s, int32_t e, int64_t blk, int8_t* cache, float* scale,
                                                  float* absmax, int h, int32_t num_kv_heads, bool is_v, float& amax,
                                                  float& cur_scale, bool& have_stats) {
#pragma clang fp contract(off)
    static_assert(D % 64 == 0, "int8 caches take head_dim 64, 128 or 256");
    constexpr int kPer = D / 64;  // elements per lane
    const int lane = threadIdx.x & 63;
    // Rows the segment writes (lane j looks at tokens s + j, s + j + 64, ..) and its absmax.
    uint32_t written = 0;
    for (int t = s + lane; t < e; t += 64) written |= 1u << static_cast<int>(slot_at(t) % kBlockSize);
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) written |= static_cast<uint32_t>(__shfl_xor(static_cast<int>(written), o, 64));
    const bool fresh = (written & 1u) != 0;
    const int64_t sidx = blk * num_kv_heads + h;
    int8_t* block_codes = cache + ((blk * num_kv_heads + h) * kBlockSize) * D;
    // Element (row off, dim d) of the tile: K is [16][D], V is [D][16].
    auto at = [&](int off, int d) -> int8_t* {
        return is_v ? block_codes + d * kBlockSize + off : block_codes + off * D + d;
    };
    // One round trip for everything the segment reads: the block's statistics, its codes (needed
    // only if the scale grows, so fetched unless the segment starts the block) as 16-byte chunks
    // of the tile (chunk c of lane: c = lane + 64 i, K row c / (D/16) or V dim c), and, for a
    // one-token segment, the token's values (kept for its quantisation).
    const float amax_mem = have_stats ? 0.0f : absmax[sidx];
    const float scale_mem = have_stats ? 0.0f : scale[sidx];
    constexpr int kChunks = kBlockSize * D / 16 / 64;  // 16-byte chunks of the tile per lane
    uint4 old_chunk[kChunks];
    if (!fresh) {
#pragma unroll
        for (int i = 0; i < kChunks; i++) old_chunk[i] = reinterpret_cast<const uint4*>(block_codes)[lane + 64 * i];
    }
    const bool one = e - s == 1;
    float x1[kPer];
    float seg_amax = 0.0f;
    for (int t = s; t < e; t++) {
        const int64_t base = static_cast<int64_t>(t) * tok_stride + static_cast<int64_t>(h) * D;
#pragma unroll
        for (int k = 0; k < kPer; k++) {
            const float x = load_act(src, in_bf16, base + lane + 64 * k);
            if (t == s) x1[k] = x;
            const float a = fabsf(x);
            seg_amax = a > seg_amax ? a : seg_amax;  // NaN never wins, as `if (a > m) m = a`
        }
    }
    seg_amax = wave_max(seg_amax);

    if (fresh) {
        // Writing row 0 starts the block: earlier contents and statistics are discarded.
        amax = seg_amax;
        cur_scale = seg_amax / 127.0f;
        if (lane == 0) {
            absmax[sidx] = amax;
            scale[sidx] = cur_scale;
        }
    } else {
        if (!have_stats) {
            amax = amax_mem;
            cur_scale = scale_mem;
        }
        if (seg_amax > amax) {
            const float old_scale = cur_scale;
            cur_scale = seg_amax / 127.0f;
            amax = seg_amax;
            // Requantise every row this segment does not overwrite:
            // QuantizeSymmetric(Dequantize(q, old_scale), new_scale). The rows it writes keep
            // their old codes here; its own stores below replace them, after these have landed.
#pragma unroll
            for (int i = 0; i < kChunks; i++) {
                const int c = lane + 64 * i;
                uint32_t w[4] = {old_chunk[i].x, old_chunk[i].y, old_chunk[i].z, old_chunk[i].w};
#pragma unroll
                for (int b = 0; b < 16; b++) {
                    const int row = is_v ? b : c / (D / 16);
                    if (written & (1u << row)) continue;
                    const uint32_t sh = 8 * (b & 3);
                    const int32_t q = static_cast<int32_t>(w[b >> 2] << (24 - sh)) >> 24;
                    const float deq = static_cast<float>(q) * old_scale;
                    const uint32_t nq = static_cast<uint32_t>(static_cast<uint8_t>(quantize_symmetric(deq, cur_scale)));
                    w[b >> 2] = (w[b >> 2] & ~(0xffu << sh)) | (nq << sh);
                }
                reinterpret_cast<uint4*>(block_codes)[c] = make_uint4(w[0], w[1], w[2], w[3]);
            }
            __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): the tile's stores precede the new rows'

            if (lane == 0) {
                absmax[sidx] = amax;
                scale[sidx] = cur_scale;
            }
        }
    }
    have_stats = true;
    for (int t = s; t < e; t++) {
        const int off = static_cast<int>(slot_at(t) % kBlockSize);
        const int64_t base = static_cast<int64_t>(t) * tok_stride + static_cast<int64_t>(h) * D;
#pragma unroll
        for (int k = 0; k < kPer; k++) {
            const float x = one ? x1[k] : load_act(src, in_bf16, base + lane + 64 * k);
            *at(off, lane + 64 * k) = quantize_symmetric(x, cur_scale);
        }
    }
}

// One token appended alone into its block (the block receives no other token of the call), by one
// wave for (KV head h, K or V): the same bytes and statistics as append_int8_apply with a one-token
// segment, in fewer memory round trips. x holds the token's values (lane l: dims l, l + 64, ..),
// loaded by the caller before the slot was known. The block's statistics and its codes come in one
// round trip; the token's codes are merged into the tile's 16-byte chunks (V: byte off of the chunk
// of each dim, the lane's own dims; K: row off's chunks, staged through `stage`, D bytes of LDS), so
// the tile goes back in one set of whole-chunk stores with no store-then-wait ordering between the
// requantised rows and the token's row.
template <int D>
__device__ __forceinline__ void append_int8_one_token(const float (&x)[D / 64], int64_t slot, int8_t* cache,
                                                      float* scale, float* absmax, int h, int32_t num_kv_heads,
                                                      bool is_v, int8_t* stage) {
#pragma clang fp contract(off)
    constexpr int kPer = D / 64;
    constexpr int kChunks = kBlockSize * D / 16 / 64;  // 16-byte chunks of the tile per lane (= kPer)
    const int lane = threadIdx.x & 63;
    const int64_t blk = slot / kBlockSize;
    const int off = static_cast<int>(slot % kBlockSize);
    const int64_t sidx = blk * num_kv_heads + h;
    int8_t* block_codes = cache + ((blk * num_kv_heads + h) * kBlockSize) * D;
    uint4* chunks = reinterpret_cast<uint4*>(block_codes);
    const float amax_mem = absmax[sidx];
    const float scale_mem = scale[sidx];
    uint4 ch[kChunks];
#pragma unroll
    for (int i = 0; i < kChunks; i++) ch[i] = chunks[lane + 64 * i];
    float seg_amax = 0.0f;
#pragma unroll
    for (int k = 0; k < kPer; k++) {
        const float a = fabsf(x[k]);
        seg_amax = a > seg_amax ? a : seg_amax;  // NaN never wins, as `if (a > m) m = a`
    }
    seg_amax = wave_max(seg_amax);
    const bool fresh = off == 0;  // writing row 0 starts the block afresh
    float cur_scale;
    bool grow = false, new_stats = false;
    float old_scale = 0.0f, amax = 0.0f;
    if (fresh) {
        amax = seg_amax;
        cur_scale = seg_amax / 127.0f;
        new_stats = true;
    } else {
        amax = amax_mem;
        cur_scale = scale_mem;
        if (seg_amax > amax) {
            old_scale = cur_scale;
            cur_scale = seg_amax / 127.0f;
            amax = seg_amax;
            grow = true;
            new_stats = true;
        }
    }
    // the token's codes: lane l, dims l + 64 k
    uint32_t code[kPer];
#pragma unroll
    for (int k = 0; k < kPer; k++) code[k] = static_cast<uint32_t>(static_cast<uint8_t>(quantize_symmetric(x[k], cur_scale)));
    if (!is_v) {  // K row off: D consecutive bytes, chunks off * D / 16 .. (+ D / 16), via LDS
#pragma unroll
        for (int k = 0; k < kPer; k++) stage[lane + 64 * k] = static_cast<int8_t>(code[k]);
        __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
        __builtin_amdgcn_wave_barrier();
    }
#pragma unroll
    for (int i = 0; i < kChunks; i++) {
        const int c = lane + 64 * i;  // K: row c / (D / 16), dims 16 (c % (D / 16)) ..; V: dim c, tokens 0 .. 15
        uint32_t w[4] = {ch[i].x, ch[i].y, ch[i].z, ch[i].w};
        if (grow) {
            // QuantizeSymmetric(Dequantize(q, old_scale), new_scale) on every row but `off`
#pragma unroll
            for (int b = 0; b < 16; b++) {
                const int row = is_v ? b : c / (D / 16);
                if (row == off) continue;
                const uint32_t sh = 8 * (b & 3);
                const int32_t q = static_cast<int32_t>(w[b >> 2] << (24 - sh)) >> 24;
                const float deq = static_cast<float>(q) * old_scale;
                const uint32_t nq = static_cast<uint32_t>(static_cast<uint8_t>(quantize_symmetric(deq, cur_scale)));
                w[b >> 2] = (w[b >> 2] & ~(0xffu << sh)) | (nq << sh);
            }
        }
        if (is_v) {  // byte off of dim c's chunk: this lane's own code of dim c = lane + 64 i
            const uint32_t sh = 8 * (off & 3);
            w[off >> 2] = (w[off >> 2] & ~(0xffu << sh)) | (code[i] << sh);
        } else if (c / (D / 16) == off) {  // a chunk of row off: 16 codes from the stage
            const uint4 n = *reinterpret_cast<const uint4*>(stage + 16 * (c % (D / 16)));
            w[0] = n.x;
            w[1] = n.y;
            w[2] = n.z;
            w[3] = n.w;
        }
        chunks[c] = make_uint4(w[0], w[1], w[2], w[3]);
    }
    if (new_stats && lane == 0) {
        absmax[sidx] = amax;
        scale[sidx] = cur_scale;
    }
}

// A run of m <= 16 consecutive slots (rows r0 .. r0 + m - 1 of block blk, tokens s .. s + m - 1) that are the
// call's only tokens of their block, appended by one wave for (KV head h, K or V): the bytes and
// statistics of append_int8_apply with that segment. All of the run's values are loaded at once and
// held in registers between the maximum and the quantisation (token by token, as append_int8_apply
// takes a segment of any length, a prompt's block waits for 32 round trips), lane = (row of a pass, 8
// dims). K codes go out as 8-byte pieces of their rows; V codes are turned into [dim][row] through
// `stage` (16 D bytes of LDS), 4 dims x D / 16 rows a lane, and merged with the rows that are kept. K
// and V share the code: run once per wave, it is bound by its own fetch when unrolled for both
// (17 us where this form takes 14). Sources are 16-byte aligned.
template <int D, bool IN_BF16>
__device__ __forceinline__ void append_int8_run(const void* src, int64_t tok_stride, int32_t s, int m, int r0,
                                                int64_t blk, int8_t* cache, float* scale, float* absmax, int h,
                                                int32_t num_kv_heads, bool is_v, int8_t* stage) {
#pragma clang fp contract(off)
    constexpr int kRows = 512 / D;             // rows of one pass, D / 8 lanes each
    constexpr int kPasses = kBlockSize / kRows;
    constexpr int kVRows = D / 16;             // V: rows of a lane (4 dims each), 256 / D lanes per 4 dims
    const int lane = threadIdx.x & 63;
    const int64_t sidx = blk * num_kv_heads + h;
    int8_t* tile = cache + sidx * kBlockSize * D;
    const bool fresh = r0 == 0;
    const int c = lane % (D / 8);                 // the lane's 8 dims of a row
    const int g = lane % (D / 4), vr = lane / (D / 4) * kVRows;  // V: its 4 dims and first row
    // One round trip: the statistics, the tile's codes where they may be needed (requantised when the
    // scale grows; V keeps the rows that are not written), the run's values. Old codes of K: 8 bytes of
    // each pass; of V: kVRows bytes of each of the 4 dims.
    const float amax_mem = fresh ? 0.0f : absmax[sidx];
    const float scale_mem = fresh ? 0.0f : scale[sidx];
    constexpr int kOld = kPasses * 2;  // words: the same number for V
    static_assert(kOld == kVRows, "4 dims of kVRows / 4 words");
    uint32_t old[kOld];
#pragma unroll
    for (int i = 0; i < kOld; i++) old[i] = 0;
    if (!is_v && !fresh) {
#pragma unroll
        for (int p = 0; p < kPasses; p++) {
            const uint2 w = *reinterpret_cast<const uint2*>(tile + (p * kRows + lane / (D / 8)) * D + 8 * c);
            old[2 * p] = w.x;
            old[2 * p + 1] = w.y;
        }
    } else if (is_v && (!fresh || m < kBlockSize)) {
#pragma unroll
        for (int e = 0; e < 4; e++)
#pragma unroll
            for (int k = 0; k < kVRows / 4; k++)
                old[e * (kVRows / 4) + k] = *reinterpret_cast<const uint32_t*>(tile + (4 * g + e) * kBlockSize + vr + 4 * k);
    }
    float x[kPasses * 8];
    {
        const int64_t base = static_cast<int64_t>(s) * tok_stride + static_cast<int64_t>(h) * D + 8 * c;
        constexpr int kWords = IN_BF16 ? 1 : 2;
        uint4 raw[kPasses][kWords];
#pragma unroll
        for (int p = 0; p < kPasses; p++) {
            // rows outside the run read one of its rows: no new maximum, and their codes are not used
            const int j = min(max(p * kRows + lane / (D / 8) - r0, 0), m - 1);
            const char* at = static_cast<const char*>(src) + (base + j * tok_stride) * (IN_BF16 ? 2 : 4);
#pragma unroll
            for (int w = 0; w < kWords; w++) raw[p][w] = reinterpret_cast<const uint4*>(at)[w];
        }
#pragma unroll
        for (int p = 0; p < kPasses; p++) {
            const uint32_t w0[4] = {raw[p][0].x, raw[p][0].y, raw[p][0].z, raw[p][0].w};
            const uint4 hi = raw[p][kWords - 1];
            const uint32_t w1[4] = {hi.x, hi.y, hi.z, hi.w};
#pragma unroll
            for (int e = 0; e < 8; e++) {
                if constexpr (IN_BF16) x[8 * p + e] = (e & 1) ? bf16_hi(w0[e >> 1]) : bf16_lo(w0[e >> 1]);
                else x[8 * p + e] = __uint_as_float(e < 4 ? w0[e] : w1[e - 4]);
            }
        }
    }
    float seg_amax = 0.0f;
#pragma unroll
    for (int i = 0; i < kPasses * 8; i++) {
        const float a = fabsf(x[i]);
        seg_amax = a > seg_amax ? a : seg_amax;  // NaN never wins, as `if (a > m) m = a`
    }
    seg_amax = wave_max_dpp(seg_amax);
    const bool grow = !fresh && seg_amax > amax_mem;
    const float cur_scale = fresh || grow ? seg_amax / 127.0f : scale_mem;
    if (grow) {
        // QuantizeSymmetric(Dequantize(q, old scale), new scale) of every old code
#pragma unroll
        for (int i = 0; i < kOld; i++) {
            uint32_t w = old[i], o = 0;
#pragma unroll 1
            for (int b = 0; b < 4; b++) {
                const float deq = static_cast<float>(static_cast<int8_t>(w & 0xffu)) * scale_mem;
                o = (o >> 8) | (static_cast<uint32_t>(static_cast<uint8_t>(quantize_symmetric(deq, cur_scale))) << 24);
                w >>= 8;
            }
            old[i] = o;
        }
    }
#pragma unroll
    for (int p = 0; p < kPasses; p++) {
        if ((p + 1) * kRows <= r0 && (is_v || !grow)) continue;  // a pass without a row of the run
        if (p * kRows >= r0 + m && (is_v || !grow)) continue;
        const int r = p * kRows + lane / (D / 8);
        uint32_t o[2] = {0, 0};
#pragma unroll
        for (int e = 0; e < 8; e++)
            o[e >> 2] |= static_cast<uint32_t>(static_cast<uint8_t>(quantize_symmetric(x[8 * p + e], cur_scale))) << (8 * (e & 3));
        const bool in = r >= r0 && r < r0 + m;
        if (is_v) *reinterpret_cast<uint2*>(stage + r * D + 8 * c) = make_uint2(o[0], o[1]);
        else if (in || grow)
            *reinterpret_cast<uint2*>(tile + r * D + 8 * c) = in ? make_uint2(o[0], o[1]) : make_uint2(old[2 * p], old[2 * p + 1]);
    }
    if (is_v) {
        __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): the wave's codes are in LDS
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int k = 0; k < kVRows / 4; k++) {
            // rows vr + 4 k .. + 3 of dims 4 g .. + 3: a 4 x 4 byte transpose
            uint32_t w[4];
#pragma unroll
            for (int i = 0; i < 4; i++) w[i] = *reinterpret_cast<const uint32_t*>(stage + (vr + 4 * k + i) * D + 4 * g);
            const uint32_t a = __builtin_amdgcn_perm(w[1], w[0], 0x05010400u), b = __builtin_amdgcn_perm(w[3], w[2], 0x05010400u);
            const uint32_t e = __builtin_amdgcn_perm(w[1], w[0], 0x07030602u), f = __builtin_amdgcn_perm(w[3], w[2], 0x07030602u);
            const uint32_t t[4] = {__builtin_amdgcn_perm(b, a, 0x05040100u), __builtin_amdgcn_perm(b, a, 0x07060302u),
                                   __builtin_amdgcn_perm(f, e, 0x05040100u), __builtin_amdgcn_perm(f, e, 0x07060302u)};
            uint32_t keep = 0;  // bytes of rows outside the run
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int r = vr + 4 * k + i;
                keep |= r >= r0 && r < r0 + m ? 0u : 0xffu << (8 * i);
            }
#pragma unroll
            for (int d = 0; d < 4; d++) {
                uint32_t& o = old[d * (kVRows / 4) + k];
                o = (o & keep) | (t[d] & ~keep);
            }
        }
#pragma unroll
        for (int d = 0; d < 4; d++) {
            int8_t* at = tile + (4 * g + d) * kBlockSize + vr;
            const uint32_t* o = old + d * (kVRows / 4);
            if constexpr (kVRows == 4) *reinterpret_cast<uint32_t*>(at) = o[0];
            else if constexpr (kVRows == 8) *reinterpret_cast<uint2*>(at) = make_uint2(o[0], o[1]);
            else *reinterpret_cast<uint4*>(at) = make_uint4(o[0], o[1], o[2], o[3]);
        }
        __builtin_amdgcn_wave_barrier();  // the stage is written again by the wave's next run
    }
    if ((fresh || grow) && lane == 0) {
        absmax[sidx] = seg_amax;
        scale[sidx] = cur_scale;
    }
}

// Segments [starts[k], ends[k]), k < nseg (LDS), of block blk for (KV head h, K|V) by one wave: the bytes and
// statistics of append_int8_apply called with each in turn. The tile's codes stay in registers from the
// first segment to the last (lane l: the 16 rows of dims l, l + 64, ..), the absmax of up to 64 tokens is taken
// before any is quantised, and their values are loaded kAhead tokens at a time. lut: 64 words of LDS. (Segment by segment each
// waits for its values and its tile, and after a grown scale for the tile's stores: a block whose 16 tokens
// come one by one, between other blocks' tokens, 55 us.)
template <int D, typename SlotAt>
__device__ __forceinline__ void append_int8_segments(const void* src, bool in_bf16, int64_t tok_stride,
                                                     SlotAt slot_at, const int* starts, const int* ends, int nseg,
                                                     int64_t blk, int8_t* cache, float* scale, float* absmax, int h,
                                                     int32_t num_kv_heads, bool is_v, uint32_t* lut) {
#pragma clang fp contract(off)
    constexpr int kPer = D / 64, kAhead = 8;
    const int lane = threadIdx.x & 63;
    const int64_t sidx = blk * num_kv_heads + h;
    int8_t* tile = cache + sidx * kBlockSize * D;
    float amax = absmax[sidx], cur_scale = scale[sidx];
    bool new_stats = false;
    uint32_t dirty = 0;      // rows whose codes changed
    uint32_t w[kPer][4];     // codes: byte r % 4 of word r / 4 is row r
#pragma unroll
    for (int k = 0; k < kPer; k++) {
        const int d = lane + 64 * k;
        if (is_v) {
            const uint4 x = *reinterpret_cast<const uint4*>(tile + d * kBlockSize);
            w[k][0] = x.x;
            w[k][1] = x.y;
            w[k][2] = x.z;
            w[k][3] = x.w;
        } else {
            uint32_t b[kBlockSize];
#pragma unroll
            for (int r = 0; r < kBlockSize; r++) b[r] = static_cast<uint8_t>(tile[r * D + d]);
#pragma unroll
            for (int q = 0; q < 4; q++) w[k][q] = b[4 * q] | b[4 * q + 1] << 8 | b[4 * q + 2] << 16 | b[4 * q + 3] << 24;
        }
    }
    auto load_token = [&](int t, float (&v)[kPer]) {
        const int64_t base = static_cast<int64_t>(t) * tok_stride + static_cast<int64_t>(h) * D;
#pragma unroll
        for (int e = 0; e < kPer; e++) v[e] = load_act(src, in_bf16, base + lane + 64 * e);
    };
    auto token_max = [&](const float (&v)[kPer]) {
        float m = 0.0f;
#pragma unroll
        for (int e = 0; e < kPer; e++) {
            const float a = fabsf(v[e]);
            m = a > m ? a : m;  // NaN never wins, as `if (a > m) m = a`
        }
        return m;
    };
    auto begin_segment = [&](bool fresh, float seg_amax) {
        if (!fresh && !(seg_amax > amax)) return;
        const float old_scale = cur_scale;
        amax = seg_amax;
        cur_scale = seg_amax / 127.0f;
        new_stats = true;
        if (fresh) return;
        // QuantizeSymmetric(Dequantize(q, old scale), new scale) of every code, each of the 256 taken once (the
        // lane's four; code by code a grown tile of head_dim 128 costs about 2 us); the segment's own rows are
        // overwritten by its tokens.
        dirty = (1u << kBlockSize) - 1;
        uint32_t mine = 0;
#pragma unroll
        for (int b = 0; b < 4; b++) {
            const float deq = static_cast<float>(static_cast<int8_t>(4 * lane + b)) * old_scale;
            mine |= static_cast<uint32_t>(static_cast<uint8_t>(quantize_symmetric(deq, cur_scale))) << (8 * b);
        }
        lut[lane] = mine;
        __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
        __builtin_amdgcn_wave_barrier();
        const uint8_t* const to = reinterpret_cast<const uint8_t*>(lut);
#pragma unroll
        for (int e = 0; e < kPer; e++)
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const uint32_t in = w[e][q];
                w[e][q] = to[in & 0xffu] | to[in >> 8 & 0xffu] << 8 | to[in >> 16 & 0xffu] << 16 |
                          static_cast<uint32_t>(to[in >> 24]) << 24;
            }
        __builtin_amdgcn_wave_barrier();  // the table is written again when the scale grows again
    };
    auto put = [&](int r, const float (&v)[kPer]) {
        const uint32_t sh = 8 * (r & 3), keep = ~(0xffu << sh);
        dirty |= 1u << r;
#pragma unroll
        for (int e = 0; e < kPer; e++) {
            const uint32_t code = static_cast<uint32_t>(static_cast<uint8_t>(quantize_symmetric(v[e], cur_scale))) << sh;
#pragma unroll
            for (int q = 0; q < 4; q++) w[e][q] = (r >> 2) == q ? (w[e][q] & keep) | code : w[e][q];
        }
    };
#pragma unroll 1
    for (int k = 0; k < nseg;) {
        // The next whole segments, up to 64 tokens: token of lane i, its row; the tokens that start a segment.
        int tok = 0, cnt = 0;
        uint64_t firsts = 0;
        for (; k < nseg; k++) {
            const int s = __builtin_amdgcn_readfirstlane(starts[k]);
            const int len = __builtin_amdgcn_readfirstlane(ends[k]) - s;
            if (cnt + len > 64) break;
            if (lane >= cnt && lane < cnt + len) tok = s + lane - cnt;
            firsts |= 1ull << cnt;
            cnt += len;
        }
        if (cnt == 0) {  // a segment of more than 64 tokens: slots written several times; one after another
            const int s = __builtin_amdgcn_readfirstlane(starts[k]), e = __builtin_amdgcn_readfirstlane(ends[k]);
            bool fresh = false;
            float m = 0.0f, v[kPer];
            for (int t = s; t < e; t++) {
                fresh = fresh || slot_at(t) % kBlockSize == 0;
                load_token(t, v);
                m = fmaxf(m, token_max(v));
            }
            begin_segment(fresh, wave_max_dpp(m));
            for (int t = s; t < e; t++) {
                load_token(t, v);
                put(__builtin_amdgcn_readfirstlane(static_cast<int>(slot_at(t) % kBlockSize)), v);
            }
            k++;
            continue;
        }
        const int row = lane < cnt ? static_cast<int>(slot_at(tok) % kBlockSize) : 0;
        float x[kAhead][kPer];
        auto load = [&](int i0) {
#pragma unroll
            for (int j = 0; j < kAhead; j++)
                load_token(__builtin_amdgcn_readlane(tok, min(i0 + j, cnt - 1)), x[j]);
        };
        float tok_amax = 0.0f;  // lane i: token i's
#pragma unroll 1
        for (int i0 = 0; i0 < cnt; i0 += kAhead) {
            load(i0);
#pragma unroll
            for (int j = 0; j < kAhead; j++) {
                const float m = wave_max_dpp(token_max(x[j]));
                tok_amax = lane == i0 + j ? m : tok_amax;
            }
        }
#pragma unroll 1
        for (int i0 = 0; i0 < cnt; i0 += kAhead) {
            if (cnt > kAhead) load(i0);  // else still in x
#pragma unroll 1
            for (int j = 0; j < kAhead && i0 + j < cnt; j++) {
                const int i = i0 + j;
                float v[kPer];
#pragma unroll
                for (int e = 0; e < kPer; e++) {
                    v[e] = x[0][e];
#pragma unroll
                    for (int q = 1; q < kAhead; q++) v[e] = j == q ? x[q][e] : v[e];
                }
                if (firsts >> i & 1) {
                    const uint64_t later = firsts >> i >> 1;
                    const int end = later != 0 ? i + 1 + __builtin_ctzll(later) : cnt;
                    bool fresh = false;
                    float seg_amax = 0.0f;
                    for (int t = i; t < end; t++) {
                        fresh = fresh || __builtin_amdgcn_readlane(row, t) == 0;
                        seg_amax = fmaxf(seg_amax, __int_as_float(__builtin_amdgcn_readlane(__float_as_int(tok_amax), t)));
                    }
                    begin_segment(fresh, seg_amax);
                }
                put(__builtin_amdgcn_readlane(row, i), v);
            }
        }
    }
#pragma unroll
    for (int k = 0; k < kPer; k++) {
        const int d = lane + 64 * k;
        if (is_v) {
            if (dirty != 0) *reinterpret_cast<uint4*>(tile + d * kBlockSize) = make_uint4(w[k][0], w[k][1], w[k][2], w[k][3]);
        } else {
#pragma unroll
            for (int r = 0; r < kBlockSize; r++)
                if (dirty >> r & 1) tile[r * D + d] = static_cast<int8_t>(w[k][r >> 2] >> (8 * (r & 3)));
        }
    }
    if (new_stats && lane == 0) {
        absmax[sidx] = amax;
        scale[sidx] = cur_scale;
    }
}

// Segments collected per pass of the owner's scan (a block has at most 16 rows, so more than one
// pass only happens when slots repeat).
constexpr int kAppendSegList = 64;
// Threads of an int8 append workgroup: one wave per (KV head, K|V) up to 16 waves.
constexpr int kAppendMaxThreads = 1024;
inline int append_int8_threads(int32_t num_kv_heads) {
    const int64_t waves = 2 * static_cast<int64_t>(num_kv_heads);
    return static_cast<int>(64 * (waves < kAppendMaxThreads / 64 ? waves : kAppendMaxThreads / 64));
}

// Tokens per thread of the scans over the call's slots.
constexpr int kAppendCoarse = 8;

// The workgroup of token i (blockDim.x a multiple of 64, at most kAppendMaxThreads; `parts`
// workgroups of one token share its (KV head, K|V) pairs, this one being `part`): if token i
// is the first token of the call that lands in its block, or (OWNER) the caller has chosen it among
// them, applies every segment of that block, in call order; otherwise returns. The owner reads the call's slot list once,
// kAppendCoarse slots per thread at a time: a call of n tokens costs each touched block one pass over n
// slots (a few memory round trips for calls of up to ~16k tokens; split much larger calls).
template <int D, bool OWNER = false, typename SlotAt>
__device__ __forceinline__ void append_int8_block(const void* k_src, const void* v_src, bool in_bf16,
                                                  int64_t tok_stride, SlotAt slot_at, int32_t i, int32_t n_tok,
                                                  int8_t* k_cache, int8_t* v_cache, float* k_scale, float* v_scale,
                                                  float* k_absmax, float* v_absmax, int32_t num_kv_heads,
                                                  int64_t capacity, int32_t part = 0, int32_t parts = 1) {
    __shared__ int s_start[kAppendSegList], s_end[kAppendSegList];
    __shared__ int s_wcnt[kAppendMaxThreads / 64];
    __shared__ uint32_t s_lut[kAppendMaxThreads / 64][64];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nthreads = blockDim.x, nwaves = nthreads >> 6;
    auto valid = [&](int64_t sl) { return sl >= 0 && sl < capacity; };
    // Token i's slot and its predecessor's, loaded together.
    const int64_t slot_i = slot_at(i);
    const int64_t slot_p = !OWNER && i > 0 ? slot_at(i - 1) : -1;
    if (!valid(slot_i)) return;
    const int64_t blk = __builtin_amdgcn_readfirstlane(static_cast<int>(slot_i / kBlockSize));
    if (valid(slot_p) && slot_p / kBlockSize == blk) return;  // not the first token of its segment
    auto in_blk = [&](int t) {
        if (t < 0 || t >= n_tok) return false;
        const int64_t sl = slot_at(t);
        return valid(sl) && sl / kBlockSize == blk;
    };
    const int coarse = kAppendCoarse * nthreads;
    if constexpr (!OWNER) {
        // An earlier token of the call in the block: its workgroup owns the block.
        for (int c0 = 0; c0 < i; c0 += coarse) {
            bool f = false;
#pragma unroll
            for (int k = 0; k < kAppendCoarse; k++) {
                const int t = c0 + k * nthreads + tid;
                f |= t < i && in_blk(t);
            }
            if (__syncthreads_or(f)) return;
        }
    }

    // Passes: from seg_from on, segment starts and ends are compacted, in order, into s_start /
    // s_end until kAppendSegList segments are complete or the call ends; then they are applied.
    int seg_from = OWNER ? 0 : i;
    while (seg_from < n_tok) {
        int nseg = 0, nstart = 0;
        int resume = n_tok;  // where the next pass starts if this one fills the list
        for (int c0 = seg_from; c0 < n_tok; c0 += coarse) {
            // kAppendCoarse consecutive tokens a thread: bit j of `in`, token t0 - 1 + j lands in the block
            const int t0 = c0 + kAppendCoarse * tid;
            uint32_t in = 0;
#pragma unroll
            for (int j = 0; j < kAppendCoarse + 2; j++) in |= static_cast<uint32_t>(in_blk(t0 - 1 + j)) << j;
            constexpr uint32_t kOwn = ((1u << kAppendCoarse) - 1) << 1;
            const uint32_t starts = in & ~(in << 1) & kOwn, ends = in & ~(in >> 1) & kOwn;
            // places in the lists: starts in the low half, ends in the high one
            const int mine = __popc(starts) | __popc(ends) << 16;
            int incl = mine;
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) {
                const int v = __shfl_up(incl, o, 64);
                if (lane >= o) incl += v;
            }
            __syncthreads();  // s_wcnt is no longer read
            if (lane == 63) s_wcnt[wave] = incl;
            __syncthreads();
            int before = incl - mine, total = 0;
            for (int v = 0; v < nwaves; v++) {
                if (v < wave) before += s_wcnt[v];
                total += s_wcnt[v];
            }
            int rs = nstart + (before & 0xffff), re = nseg + (before >> 16);
            for (uint32_t left = starts; left != 0; left &= left - 1, rs++)
                if (rs < kAppendSegList) s_start[rs] = t0 - 1 + __builtin_ctz(left);
            for (uint32_t left = ends; left != 0; left &= left - 1, re++)
                if (re < kAppendSegList) s_end[re] = t0 + __builtin_ctz(left);
            nstart += total & 0xffff;
            nseg += total >> 16;
            if (nseg >= kAppendSegList) break;
        }
        __syncthreads();  // the lists are complete
        if (nseg >= kAppendSegList) {
            nseg = kAppendSegList;
            resume = s_end[kAppendSegList - 1];
        }
        // Apply the complete segments, in order, one wave per (KV head, K|V).
        for (int p = part * nwaves + wave; p < 2 * num_kv_heads; p += parts * nwaves) {
            const int h = p >> 1;
            const bool is_v = (p & 1) != 0;
            append_int8_segments<D>(is_v ? v_src : k_src, in_bf16, tok_stride, slot_at, s_start, s_end, nseg, blk,
                                    is_v ? v_cache : k_cache, is_v ? v_scale : k_scale, is_v ? v_absmax : k_absmax, h,
                                    num_kv_heads, is_v, s_lut[wave]);
        }
        if (resume >= n_tok) break;
        __syncthreads();  // this pass's statistics and codes are visible to the next pass's waves
        seg_from = resume;
    }
}

}  // namespace pa
