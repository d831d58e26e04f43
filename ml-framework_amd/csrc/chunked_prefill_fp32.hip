// chunked_prefill_fp32.hip -- chunked prefill over an fp32 paged cache, fp32 throughout.
//
// The same operation as the bf16 / int8 chunked prefill (queries at positions prefix_lens[s] + i
// over keys [0, prefix_lens[s] + chunk_len) of the block table, the reference's
// StandardPagedAttentionKernel, Kernels/StandardPagedAttentionKernel.cs:21-84, with the mask of
// :57-66 / :219-255), for caches that hold fp32: K tile [16][D], V tile [D][16] per
// (block, KV head). It serves callers that hand over fp32 activations and expect fp32 results,
// such as the dense ComputePagedAttention(query, cachedKeys, cachedValues, phase) of the
// reference's IPagedAttentionKernel (Kernels/IPagedAttentionKernel.cs:13-28) with more than one
// query: one launch in which a key block is read once per 16 or 32 queries instead of once per query.
//
// Work decomposition: a unit is one 16-query tile of one query head. A wave computes NU = 2 units of
// one (sequence, KV head) on the same K/V operands, one from either end of the tile order, so that
// under the causal mask every pair has about the same work; or one unit (head_dim 256, calls of at most
// one unit per CU, and chunks of few tiles). KS waves share their keys: wave i of them takes blocks i, i + KS,
// .., and at the end the waves leave their (max, sum, O) in LDS and add them up, each a part of the
// output dims. A workgroup has 4 waves, and two of them fit a CU (one for head_dim 256), or the 8 of KS = 8.
// KS is the number for which generations of workgroups times a wave's blocks are least.
//
// A wave's blocks come one at a time into an LDS slot of its own (LDS-direct loads of whole lines;
// operands loaded straight into registers held the kernel at 42 us where this one takes 31): the
// next block's K goes out when the QK products have read the slot's K, its V after the PV products.
// No wave waits for another in the stream. Per block, on v_mfma_f32_16x16x4_f32 (fp32 operands,
// fp32 accumulation):
//   S^T[16 keys][16 queries] = K . Q^T, MFMA 4 t + e taking head dims 16 t + 4 (lane / 16) + e, so a
//     lane's K operands of four MFMAs are one 16-byte LDS read;
//   online softmax per query in fp32 (log2 domain: the scale times log2(e) folded into Q), the
//     maximum raised only past a margin of 2^8;
//   O^T[D][16 queries] += V^T . P^T, where MFMA s of an output tile takes keys 4 (lane / 16) + s:
//     the lane's own four S^T values are its P operands, its V operand is one 16-byte read of
//     the [D][16] V tile, and all of the lane's accumulators belong to its own query, so the
//     rescale by the running maximum needs no exchange between lanes.
// What bounds it: the fp32 MFMAs, D / 2 of 32 clocks per block and unit. 2 x 512 queries on 350
// tokens, 8 heads of 128: 98 -> 31 us (82 TFLOP/s; a large fp32 GEMM reaches 140); 8 such: 164 -> 92 us
// (110); 30 queries on 5000: 547 -> 85 us.
#include <string>
#include <type_traits>

#include "decode_common.h"

namespace pa {
namespace {

constexpr int kF32Margin = 8;  // log2 units

struct PrefillF32Args {
    float* out;
    const void* q;
    const float* k_cache;
    const float* v_cache;
    const int32_t* q_start_loc;
    const int32_t* prefix_lens;
    const int32_t* block_tables;
    int32_t num_kv_heads;
    int32_t group;
    int32_t max_blocks_per_seq;
    int32_t num_blocks;
    int32_t mask_mode;  // 0 causal, 1 causal only when the prefix is non-empty, 2 no mask
    float scale;
    int32_t wg_per_group;  // workgroups per (sequence, KV head)
    int32_t num_groups;    // num_seqs * num_kv_heads
    int32_t q_bf16;
};

// LDS layout of a block: the K tile's 16-byte chunk (row r, column c) at chunk r RC + (c ^ swz(r)), then
// the V tile's (dim d, tokens 4 q .. + 3) at 4 d + (q ^ h((d / 4) % 4)), h = 0 2 3 1. An operand read
// takes column 4 t + lane / 16 of row lane % 16 (K) or dim 16 t + lane % 16 (V); with these XORs the 16
// lanes that gfx950 serves in one clock (quads {0, 3, 5, 6} and {1, 2, 4, 7} of each half-wave) fall
// on 16 different 16-byte positions of a 256-byte line.
template <int D> struct F32Tile {
    static constexpr int RC = D / 4;       // chunks per K row
    static constexpr int CHUNKS = 16 * RC;  // of a tile
    static constexpr int SEG = CHUNKS / 64;  // KiB, loads of one tile
    __device__ static constexpr int swz(int r) { return RC >= 16 ? r : r >> 1; }
    __device__ static constexpr int kpos(int r, int c) { return r * RC + (c ^ swz(r)); }
    __device__ static constexpr int h(int x) { return ((x << 1) ^ ((x >> 1) * 7)) & 3; }
    __device__ static constexpr int vpos(int d, int q) { return CHUNKS + 4 * d + (q ^ h((d >> 2) & 3)); }
};

// LDS-direct loads of NS KiB into LDS from m0 on, 16 bytes a lane: segment j at immediate offset 1024 j,
// which advances both the memory and the LDS address; off[j] is the lane's offset within segment j.
template <int NS>
__device__ __forceinline__ void lds_load_segments(u32x4_t r, const uint32_t* off, uint32_t m0) {
    uint32_t saved;
    if constexpr (NS == 2) {
        asm volatile(
            "s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\t"
            "buffer_load_dwordx4 %3, %1, 0 offen lds\n\t"
            "buffer_load_dwordx4 %4, %1, 0 offen offset:1024 lds\n\t"
            "s_mov_b32 m0, %0"
            : "=&s"(saved)
            : "s"(r), "s"(m0), "v"(off[0]), "v"(off[1])
            : "memory");
    } else if constexpr (NS == 4) {
        asm volatile(
            "s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\t"
            "buffer_load_dwordx4 %3, %1, 0 offen lds\n\t"
            "buffer_load_dwordx4 %4, %1, 0 offen offset:1024 lds\n\t"
            "buffer_load_dwordx4 %5, %1, 0 offen offset:2048 lds\n\t"
            "buffer_load_dwordx4 %6, %1, 0 offen offset:3072 lds\n\t"
            "s_mov_b32 m0, %0"
            : "=&s"(saved)
            : "s"(r), "s"(m0), "v"(off[0]), "v"(off[1]), "v"(off[2]), "v"(off[3])
            : "memory");
    } else {
        static_assert(NS % 4 == 0, "2 KiB or multiples of 4");
#pragma unroll
        for (int i = 0; i < NS / 4; i++) {
            const uint32_t o[4] = {off[4 * i] + 4096 * i, off[4 * i + 1] + 4096 * i, off[4 * i + 2] + 4096 * i,
                                   off[4 * i + 3] + 4096 * i};
            lds_load_segments<4>(r, o, m0 + 4096 * i);
        }
    }
}

// Waves of a workgroup: 4, or the 8 that share a unit's keys; and workgroups a CU's LDS holds (head_dim 256: one).
__host__ __device__ constexpr int f32_waves(int ks) { return ks > 4 ? 8 : 4; }
__host__ __device__ constexpr int f32_per_cu(int d, int ks) { return d > 128 || ks > 4 ? 1 : 2; }

template <int D, int KS, int NU>
__global__ __launch_bounds__((64 * f32_waves(KS)), (f32_waves(KS) / 4 * f32_per_cu(D, KS))) void chunked_prefill_fp32_kernel(const PrefillF32Args a) {
    using TL = F32Tile<D>;
    constexpr int NT = D / 16;  // 16-dim slabs of K and output tiles
    constexpr int WAVES = f32_waves(KS);
    constexpr int SEG = TL::SEG;
    // The waves' slots, reused for their states.
    __shared__ uint4 s_tile[WAVES * 2 * TL::CHUNKS];
    __shared__ float2 s_ml[KS > 1 ? WAVES * NU * 64 : 1];
    static_assert(NU * NT * 64 <= 2 * TL::CHUNKS, "a state fits a slot");
    int gi, qg;
    if (!place_workgroup(a.num_groups, a.wg_per_group, gi, qg)) return;
    const int seq = gi / a.num_kv_heads, kvh = gi - seq * a.num_kv_heads;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int uw = wave / KS, ks = wave % KS;  // set of units of the workgroup, share of its keys
    const int G = a.group, Hq = a.num_kv_heads * G;
    const int n = lane & 15, q4 = lane >> 4;

    const int q0 = a.q_start_loc[seq];
    const int Lc = a.q_start_loc[seq + 1] - q0;
    const int P = max(a.prefix_lens[seq], 0);
    const int T = min(P + Lc, a.max_blocks_per_seq * 16);
    const bool causal = a.mask_mode == 0 || (a.mask_mode == 1 && P > 0);
    // Units of the set: u0 from the end of the list, with the most keys, and u1 from its start. Unit k:
    // head hq of the 16 queries from i0; query i0 + n is this lane's (rows past the chunk are computed on
    // its last query and not stored). nblk: its key blocks, 0 for a unit that does not exist.
    const int units = (Lc + 15) / 16 * G;
    const int set = qg * (WAVES / KS) + uw;
    int hq[NU], i0[NU], nblk[NU];
#pragma unroll
    for (int k = 0; k < NU; k++) {
        const int u = k == 0 ? units - 1 - set : set;
        const bool live = NU == 1 ? set < units : 2 * set + k < units;
        const int qt = live ? u / G : 0;
        hq[k] = kvh * G + (live ? u - qt * G : 0);
        i0[k] = 16 * qt;
        const int kend = causal ? min(T, P + min(i0[k] + 16, Lc)) : T;
        nblk[k] = live ? (kend + 15) / 16 : 0;
    }
    const int nkb = nblk[0];
    if (KS == WAVES && nkb == 0) return;  // no unit in the workgroup

    // Q operands: dims 16 t + 4 (lane / 16) .. + 3 of the lane's query, times scale * log2(e).
    const float c2 = a.scale * 1.4426950408889634f;
    f32x4_t qv[NU][NT];
#pragma unroll
    for (int k = 0; k < NU; k++) {
        const int64_t row = (static_cast<int64_t>(q0) + max(min(i0[k] + n, Lc - 1), 0)) * Hq + hq[k];
        const int64_t base = row * D + 4 * q4;
#pragma unroll
        for (int t = 0; t < NT; t++) {
            if (nblk[k] == 0) {
                qv[k][t] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
            } else if (a.q_bf16) {
                const uint2 w = *reinterpret_cast<const uint2*>(static_cast<const uint16_t*>(a.q) + base + 16 * t);
                qv[k][t] = f32x4_t{bf16_lo(w.x), bf16_hi(w.x), bf16_lo(w.y), bf16_hi(w.y)} * c2;
            } else {
                qv[k][t] = *reinterpret_cast<const f32x4_t*>(static_cast<const float*>(a.q) + base + 16 * t) * c2;
            }
        }
    }

    const int32_t* table = a.block_tables + static_cast<int64_t>(seq) * a.max_blocks_per_seq;
    f32x4_t acc[NU][NT];
    // A wave may meet no key of an early query: its maximum then stays the lowest finite value, against
    // which masked scores (-inf) give P = 0, and which the sum of the waves weighs with 0.
    float m_run[NU], l_run[NU];
#pragma unroll
    for (int k = 0; k < NU; k++) {
        m_run[k] = -__FLT_MAX__;
        l_run[k] = 0.0f;
#pragma unroll
        for (int t = 0; t < NT; t++) acc[k][t] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    }

    // Lane l's memory chunk for position 64 j + l of the K tile: row r = (64 j + l) / RC, column
    // ((64 j + l) % RC) ^ swz(r); of the V tile: 64 j plus the same for every segment.
    const uint4* const slot = s_tile + wave * 2 * TL::CHUNKS;
    const uint32_t slot_lds = lds_address(s_tile) + 16 * 2 * TL::CHUNKS * wave;
    const uint32_t voff = 16 * ((lane & ~3) | ((lane & 3) ^ TL::h(lane >> 4)));
    uint32_t koffs[SEG], voffs[SEG];
#pragma unroll
    for (int j = 0; j < SEG; j++) {
        koffs[j] = 16 * TL::kpos((64 * j + lane) / TL::RC, lane % TL::RC) - 1024 * j;
        voffs[j] = voff;
    }
    // Ids of this wave's blocks ks + KS j, j = 64 w .. 64 w + 63, in lane j % 64.
    int ids = -1;
    auto bid_at = [&](int j) {  // j wave-uniform, ascending
        if ((j & 63) == 0) {
            const int b = ks + KS * (j + lane);
            ids = b < nkb ? table[b] : -1;
            __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): the stream counts its own loads only
        }
        const int id = __builtin_amdgcn_readlane(ids, j & 63);
        return id < a.num_blocks ? id : -1;
    };
    // The K / V tile of block bid; an invalid id, or none (past the list), reads as zeros through a
    // zero-sized descriptor.
    auto issue = [&](const float* cache, const uint32_t (&off)[SEG], int bid, uint32_t lds) {
        const int64_t tile = (static_cast<int64_t>(bid >= 0 ? bid : 0) * a.num_kv_heads + kvh) * (16 * D);
        lds_load_segments<SEG>(buffer_rsrc_words(cache + tile, bid >= 0 ? 16 * D * 4 : 0), off, lds);
    };

    const int nb = nkb > ks ? (nkb - ks + KS - 1) / KS : 0;  // this wave's blocks
    int bid = nb > 0 ? bid_at(0) : -1;
    if (nb > 0) {
        issue(a.k_cache, koffs, bid, slot_lds);
        issue(a.v_cache, voffs, bid, slot_lds + 16 * TL::CHUNKS);
    }
    // One block for the first nu units.
    auto block = [&](auto nu, int j) {
        constexpr int N = decltype(nu)::value;
        const int b = ks + KS * j;
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(SEG) : "memory");  // this block's K is in the slot
        f32x4_t s[N];
#pragma unroll
        for (int k = 0; k < N; k++) s[k] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int t = 0; t < NT; t++) {
            const f32x4_t kx = __builtin_bit_cast(f32x4_t, slot[TL::kpos(n, 4 * t + q4)]);
#pragma unroll
            for (int e = 0; e < 4; e++)
#pragma unroll
                for (int k = 0; k < N; k++) s[k] = __builtin_amdgcn_mfma_f32_16x16x4f32(kx[e], qv[k][t][e], s[k], 0, 0, 0);
        }
        bid = bid_at(j + 1);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        issue(a.k_cache, koffs, bid, slot_lds);
        float p[N][4];
#pragma unroll
        for (int k = 0; k < N; k++) {
            // lane holds keys 16 b + 4 q4 + i of its query; all of the unit's see the first of them
            if (16 * b + 16 > (causal ? min(T, P + i0[k] + 1) : T)) {
                const int qlim = (causal ? min(T, P + i0[k] + n + 1) : T) - (16 * b + 4 * q4);
#pragma unroll
                for (int i = 0; i < 4; i++) s[k][i] = i < qlim ? s[k][i] : -INFINITY;
            }
            const float ml = fmaxf(fmaxf(s[k][0], s[k][1]), fmaxf(s[k][2], s[k][3]));
            if (__any(ml > m_run[k] + kF32Margin)) {
                const float mb = rows_max(ml);
                const float m_new = mb > m_run[k] + kF32Margin ? mb : m_run[k];
                const float alpha = __builtin_amdgcn_exp2f(m_run[k] - m_new);
                m_run[k] = m_new;
                l_run[k] *= alpha;
#pragma unroll
                for (int t = 0; t < NT; t++) acc[k][t] *= alpha;
            }
#pragma unroll
            for (int i = 0; i < 4; i++) p[k][i] = __builtin_amdgcn_exp2f(s[k][i] - m_run[k]);
            l_run[k] += (p[k][0] + p[k][1]) + (p[k][2] + p[k][3]);
        }
        // O^T += V^T . P^T: MFMA (t, i) takes keys 4 q4 + i of the block
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(SEG) : "memory");  // its V too
#pragma unroll
        for (int t = 0; t < NT; t++) {
            const f32x4_t vx = __builtin_bit_cast(f32x4_t, slot[TL::vpos(16 * t + n, q4)]);
#pragma unroll
            for (int i = 0; i < 4; i++)
#pragma unroll
                for (int k = 0; k < N; k++)
                    acc[k][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(vx[i], p[k][i], acc[k][t], 0, 0, 0);
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        issue(a.v_cache, voffs, bid, slot_lds + 16 * TL::CHUNKS);
    };
    for (int j = 0; j < nb; j++) {
        if (NU == 2 && ks + KS * j < nblk[NU - 1]) block(std::integral_constant<int, NU>{}, j);
        else block(std::integral_constant<int, 1>{}, j);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no LDS-direct write may outlive the stream

    auto out_row = [&](int k) {
        return a.out + ((static_cast<int64_t>(q0) + i0[k] + n) * Hq + hq[k]) * D + 4 * q4;
    };
    auto stored = [&](int k) { return nblk[k] > 0 && i0[k] + n < Lc; };
    if constexpr (KS > 1) {
        // Every wave leaves its state in its own slot; piece i (unit i / NT, dims 16 (i % NT) .. + 15) of a set is
        // added up and stored by wave i % KS of it.
#pragma unroll
        for (int k = 0; k < NU; k++) {
            if (nkb == 1) break;
            s_ml[(wave * NU + k) * 64 + lane] = make_float2(m_run[k], l_run[k]);
#pragma unroll
            for (int t = 0; t < NT; t++)
                s_tile[wave * 2 * TL::CHUNKS + (k * NT + t) * 64 + lane] = __builtin_bit_cast(uint4, acc[k][t]);
        }
        __syncthreads();
        if (nkb != 1) {
            const int w0 = uw * KS;
#pragma unroll
            for (int k = 0; k < NU; k++) {
                if (nblk[k] == 0) continue;
                float2 ml[KS];
                float mt = -__FLT_MAX__;
#pragma unroll
                for (int i = 0; i < KS; i++) {
                    ml[i] = s_ml[((w0 + i) * NU + k) * 64 + lane];
                    mt = fmaxf(mt, ml[i].x);
                }
                float l = 0.0f, f[KS];
#pragma unroll
                for (int i = 0; i < KS; i++) {
                    f[i] = __builtin_amdgcn_exp2f(ml[i].x - mt);
                    l += ml[i].y * f[i];
                }
                const float inv = 1.0f / rows_sum(l);  // lanes n, n + 16, .. held partial sums of query n
#pragma unroll
                for (int t = 0; t < NT; t++) {
                    if ((k * NT + t) % KS != ks) continue;
                    f32x4_t o = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                    for (int i = 0; i < KS; i++)
                        o += __builtin_bit_cast(f32x4_t, s_tile[(w0 + i) * 2 * TL::CHUNKS + (k * NT + t) * 64 + lane]) * f[i];
                    if (stored(k)) *reinterpret_cast<f32x4_t*>(out_row(k) + 16 * t) = o * inv;
                }
            }
            return;
        }
        if (ks > 0) return;  // one block of keys: wave 0 of the set has it all
    }
#pragma unroll
    for (int k = 0; k < NU; k++) {
        const float inv = 1.0f / rows_sum(l_run[k]);
        if (!stored(k)) continue;
#pragma unroll
        for (int t = 0; t < NT; t++) *reinterpret_cast<f32x4_t*>(out_row(k) + 16 * t) = acc[k][t] * inv;
    }
}

template <int D>
void launch_ks(const PrefillF32Args& a, int nu, int ks, dim3 grid, hipStream_t s) {
    const int threads = 64 * f32_waves(ks);
    if constexpr (D > 128) {
        switch (ks) {
            case 1: chunked_prefill_fp32_kernel<D, 1, 1><<<grid, threads, 0, s>>>(a); break;
            case 2: chunked_prefill_fp32_kernel<D, 2, 1><<<grid, threads, 0, s>>>(a); break;
            default: chunked_prefill_fp32_kernel<D, 4, 1><<<grid, threads, 0, s>>>(a); break;
        }
    } else if (nu == 1) {
        switch (ks) {
            case 1: chunked_prefill_fp32_kernel<D, 1, 1><<<grid, threads, 0, s>>>(a); break;
            case 2: chunked_prefill_fp32_kernel<D, 2, 1><<<grid, threads, 0, s>>>(a); break;
            case 4: chunked_prefill_fp32_kernel<D, 4, 1><<<grid, threads, 0, s>>>(a); break;
            default: chunked_prefill_fp32_kernel<D, 8, 1><<<grid, threads, 0, s>>>(a); break;
        }
    } else {
        switch (ks) {
            case 1: chunked_prefill_fp32_kernel<D, 1, 2><<<grid, threads, 0, s>>>(a); break;
            case 2: chunked_prefill_fp32_kernel<D, 2, 2><<<grid, threads, 0, s>>>(a); break;
            case 4: chunked_prefill_fp32_kernel<D, 4, 2><<<grid, threads, 0, s>>>(a); break;
            default: chunked_prefill_fp32_kernel<D, 8, 2><<<grid, threads, 0, s>>>(a); break;
        }
    }
}

}  // namespace

pa_status launch_chunked_prefill_fp32(hipStream_t s, const pa_config* cfg, float* out, const void* q,
                                      const int32_t* q_start_loc, const int32_t* prefix_lens, const float* k_cache,
                                      const float* v_cache, const int32_t* block_tables, int32_t num_seqs,
                                      int32_t max_blocks_per_seq, int32_t max_chunk_len, int32_t mask_mode) {
    PrefillF32Args a{};
    a.out = out;
    a.q = q;
    a.k_cache = k_cache;
    a.v_cache = v_cache;
    a.q_start_loc = q_start_loc;
    a.prefix_lens = prefix_lens;
    a.block_tables = block_tables;
    a.num_kv_heads = cfg->num_kv_heads;
    a.group = cfg->num_q_heads / cfg->num_kv_heads;
    a.max_blocks_per_seq = max_blocks_per_seq;
    a.num_blocks = cfg->num_blocks;
    a.mask_mode = mask_mode;
    a.scale = resolve_scale(cfg);
    a.q_bf16 = cfg->q_dtype == PA_DTYPE_BF16;
    const int64_t ng = static_cast<int64_t>(num_seqs) * cfg->num_kv_heads;
    const int64_t units = static_cast<int64_t>(a.group) * ((static_cast<int64_t>(max_chunk_len) + 15) / 16);
    // One unit a wave while every unit can have a CU, and for chunks of few tiles (40 x 33 tokens, 16 / 4 heads of 128:
    // 13.5 us against 17.2; 16 x 100: 20.4 against 22.3); two beyond (16 x 128: 23.7 against 26.0; 8 x 512: 88 against
    // 102; 2 x 512 on 350: 52.6 against 54.7).
    const int64_t tiles = units / a.group;
    const int nu = cfg->head_dim > 128 || ng * units <= device_cus() || tiles < 8 ? 1 : 2;
    const int64_t sets = (units + nu - 1) / nu;  // per (sequence, KV head)
    // Waves on a set's keys: the number with the least generations of workgroups times (a constant part, the
    // launch, first loads and the exchange, about two and a half blocks, and a wave's blocks; the table's width bounds them).
    auto groups = [&](int n) { return (sets + f32_waves(n) / n - 1) / (f32_waves(n) / n); };
    int ks = 1;
    int64_t least = 0;
    for (int n = 1; n <= (cfg->head_dim > 128 ? 4 : 8); n *= 2) {
        const int64_t hold = static_cast<int64_t>(f32_per_cu(cfg->head_dim, n)) * device_cus();
        const int64_t cost = (ng * groups(n) + hold - 1) / hold * (5 + 2 * ((max_blocks_per_seq + n - 1) / n));
        if (n == 1 || cost <= least) {
            ks = n;
            least = cost;
        }
    }
    const int64_t wpg = groups(ks);
    const int64_t nwg = placed_grid(ng, wpg);
    if (nwg > 0x7fffffff) return set_error(PA_ERROR_UNSUPPORTED, "pa_chunked_prefill: grid too large");
    a.wg_per_group = static_cast<int32_t>(wpg);
    a.num_groups = static_cast<int32_t>(ng);
    const dim3 grid(static_cast<uint32_t>(nwg));
    switch (cfg->head_dim) {
        case 32: launch_ks<32>(a, nu, ks, grid, s); break;
        case 64: launch_ks<64>(a, nu, ks, grid, s); break;
        case 128: launch_ks<128>(a, nu, ks, grid, s); break;
        default: launch_ks<256>(a, nu, ks, grid, s); break;
    }
    PA_HIP_CHECK(hipGetLastError());
    return clear_error();
}

}  // namespace pa
