// decode_fp32.h -- the fp32-cache paged-decode kernels: VALU for groups of 1 and 2 query heads, matrix for 4 and 8.
#pragma once

#include "decode_common.h"

namespace pa {

// ================================================================================================
// fp32 caches, groups of 1 or 2 query heads: VALU kernel. (On the matrix kernel below, 16 sequences of
// 64 to 2048 tokens, 8 KV heads of 128: 38.2 against 32.8 us with one head a group, 38.4 against 34.1 with two.)
// ================================================================================================
template <int D, int G, int PART>
__global__ __launch_bounds__(256) void paged_decode_fp32_kernel(const DecodeArgs a) {
    constexpr int CH = D / 4;      // 16-byte chunks per K row
    constexpr int TPI = 64 / CH;   // K rows per wave load instruction
    constexpr int LPB = 16 / TPI;  // K load instructions per block per lane
    constexpr int RPL = D / 16;    // V dim rows per lane per block (lane = (dim row, 4-token chunk))
    constexpr int NBW = PART / 64; // blocks per wave
    constexpr int TPT = PART / 256;
    constexpr int TILE = 16 * D;
    static_assert(CH >= 8 && CH <= 64, "fp32 kernel covers head_dim 32..256");

    __shared__ float s_logits[G][PART];
    __shared__ float s_red[4][G];
    __shared__ float s_o[4][G][D];

    const int part = blockIdx.x, kvh = blockIdx.y, seq = blockIdx.z;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int Hkv = a.num_kv_heads, Hq = Hkv * G;

    const int T = clamp_len(a, a.context_lens[seq]);
    const int tok0 = part * PART;
    if (T <= 0) {
        if (part == 0)
            for (int idx = tid; idx < G * D; idx += 256)
                a.out[(static_cast<int64_t>(seq) * Hq + kvh * G) * D + idx] = 0.0f;
        return;
    }
    if (tok0 >= T) return;
    const int ntok = min(PART, T - tok0);
    const int nparts = (T + PART - 1) / PART;
    const int ti = lane / CH, ch = lane % CH;

    float qf[G][4];
    {
        const int64_t qb = (static_cast<int64_t>(seq) * Hq + kvh * G) * D + ch * 4;
#pragma unroll
        for (int g = 0; g < G; g++)
#pragma unroll
            for (int e = 0; e < 4; e++)
                qf[g][e] = a.q_bf16 ? pa::bf16_to_f32(static_cast<const uint16_t*>(a.q)[qb + g * D + e])
                                    : static_cast<const float*>(a.q)[qb + g * D + e];
    }

    const int32_t* table = a.block_tables + static_cast<int64_t>(seq) * a.max_blocks_per_seq;
    const int lb0 = tok0 / 16;
    int bid[NBW];
#pragma unroll
    for (int i = 0; i < NBW; i++) {
        const int lb = lb0 + i * 4 + wave;
        int id = -1;
        if ((lb - lb0) * 16 < ntok) {
            id = table[lb];
            if (id >= a.num_blocks) id = -1;
        }
        bid[i] = __builtin_amdgcn_readfirstlane(id);
    }
    const float* kc = static_cast<const float*>(a.k_cache);
    const float* vc = static_cast<const float*>(a.v_cache);
    auto kload = [&](int b, int j) -> uint4 {
        if (b < 0) return make_uint4(0, 0, 0, 0);
        return *reinterpret_cast<const uint4*>(kc + (static_cast<int64_t>(b) * Hkv + kvh) * TILE +
                                               (j * TPI + ti) * D + ch * 4);
    };

    // ---- scores ----
#pragma unroll
    for (int i = 0; i < NBW; i++) {
        uint4 kr[LPB];
#pragma unroll
        for (int j = 0; j < LPB; j++) kr[j] = kload(bid[i], j);
#pragma unroll
        for (int j = 0; j < LPB; j++) {
            const float kf[4] = {__uint_as_float(kr[j].x), __uint_as_float(kr[j].y), __uint_as_float(kr[j].z),
                                 __uint_as_float(kr[j].w)};
            float dot[G];
#pragma unroll
            for (int g = 0; g < G; g++) {
                float acc = 0.0f;
#pragma unroll
                for (int e = 0; e < 4; e++) acc += qf[g][e] * kf[e];
                dot[g] = pa::group_sum<CH>(acc);
            }
            const int lt = (i * 4 + wave) * 16 + j * TPI + ti;
            if (ch == 0)
#pragma unroll
                for (int g = 0; g < G; g++) s_logits[g][lt] = lt < ntok ? dot[g] * a.scale : -INFINITY;
        }
    }
    __syncthreads();

    // ---- partition softmax ----
    float m[G], l[G];
#pragma unroll
    for (int g = 0; g < G; g++) {
        float mx = -INFINITY;
#pragma unroll
        for (int k = 0; k < TPT; k++) mx = fmaxf(mx, s_logits[g][tid + 256 * k]);
        mx = pa::wave_max(mx);
        if (lane == 0) s_red[wave][g] = mx;
    }
    __syncthreads();
#pragma unroll
    for (int g = 0; g < G; g++) m[g] = fmaxf(fmaxf(s_red[0][g], s_red[1][g]), fmaxf(s_red[2][g], s_red[3][g]));
    __syncthreads();
#pragma unroll
    for (int g = 0; g < G; g++) {
        float sum = 0.0f;
#pragma unroll
        for (int k = 0; k < TPT; k++) {
            const float p = __expf(s_logits[g][tid + 256 * k] - m[g]);
            s_logits[g][tid + 256 * k] = p;
            sum += p;
        }
        sum = pa::wave_sum(sum);
        if (lane == 0) s_red[wave][g] = sum;
    }
    __syncthreads();
#pragma unroll
    for (int g = 0; g < G; g++) l[g] = (s_red[0][g] + s_red[1][g]) + (s_red[2][g] + s_red[3][g]);

    // ---- o = sum_t p_t v_t; V tile is [D][16]: lane = (dim row vd + 16 r, tokens 4vc..4vc+3) ----
    const int vc4 = lane & 3, vd = lane >> 2;
    float acc[G][RPL];
#pragma unroll
    for (int g = 0; g < G; g++)
#pragma unroll
        for (int r = 0; r < RPL; r++) acc[g][r] = 0.0f;
#pragma unroll
    for (int i = 0; i < NBW; i++) {
        if (bid[i] < 0) continue;  // zero values contribute nothing
        const float* vt = vc + (static_cast<int64_t>(bid[i]) * Hkv + kvh) * TILE + vd * 16 + 4 * vc4;
        uint4 vr[RPL];
#pragma unroll
        for (int r = 0; r < RPL; r++) vr[r] = *reinterpret_cast<const uint4*>(vt + r * 256);
        const int lt = (i * 4 + wave) * 16 + 4 * vc4;
        float4 p[G];
#pragma unroll
        for (int g = 0; g < G; g++) p[g] = *reinterpret_cast<const float4*>(&s_logits[g][lt]);
#pragma unroll
        for (int r = 0; r < RPL; r++) {
            const float v0 = __uint_as_float(vr[r].x), v1 = __uint_as_float(vr[r].y);
            const float v2 = __uint_as_float(vr[r].z), v3 = __uint_as_float(vr[r].w);
#pragma unroll
            for (int g = 0; g < G; g++) acc[g][r] += p[g].x * v0 + p[g].y * v1 + p[g].z * v2 + p[g].w * v3;
        }
    }
#pragma unroll
    for (int g = 0; g < G; g++)
#pragma unroll
        for (int r = 0; r < RPL; r++) acc[g][r] = pa::group_sum<4>(acc[g][r]);
    if (vc4 == 0)
#pragma unroll
        for (int g = 0; g < G; g++)
#pragma unroll
            for (int r = 0; r < RPL; r++) s_o[wave][g][vd + 16 * r] = acc[g][r];
    __syncthreads();

    for (int idx = tid; idx < G * D; idx += 256) {
        const int g = idx / D, d = idx - g * D;
        const float o = (s_o[0][g][d] + s_o[1][g][d]) + (s_o[2][g][d] + s_o[3][g][d]);
        emit(a, seq, kvh * G + g, part, nparts, D, d, o, m[g], l[g]);
    }
}

// ================================================================================================
// fp32 caches, groups of 4 or 8 query heads. One workgroup per (partition of PART tokens, KV head,
// sequence); wave w takes the partition's blocks w, w + 4, .. with a running (max, sum, O) of its own, and
// the four states are combined at the end.
//
// Both products run on v_mfma_f32_4x4x1 (16 independent 4x4 products a wave, fp32 throughout): the four
// query heads of a group that a KV head serves fill its columns, where the 16 x 16 forms would waste
// three quarters or more. Lane l = 16 q4 + 4 ds + c, block of the product (q4, ds):
//   S:  rows = tokens 4 q4 .. 4 q4 + 3 (A: lane c holds its row's dims), columns = heads, dims 16 u + 4 ds + e
//       one step per (u, e); the sum over ds ends with two DPP row rotations. Result: lane c = head c,
//       register i = token 4 q4 + i: the A operand (row = head c, step i = token) of
//   O:  rows = heads, column c of block (q4, ds) = dim 16 t + 4 ds + c, summed over the block's four tokens;
//       the sum over q4 is taken once at the end.
// So neither scores nor probabilities leave registers, and every load is 16 bytes a lane.
//
// What bounds it: the VALU kernel spends its time in per-head dot products, each summed over the lanes of a
// row, in code that grows with heads and head_dim. Here a block takes head_dim / 2 matrix steps for four
// heads, and a wave's next K and V load into the registers just consumed (the first follow one round trip:
// length, Q and block ids are loaded together). Fused append steps of 1 sequence of 200 tokens / 16 of 64 to
// 2048 / 8 of 5000, us, VALU -> now: 16 / 4 heads of 64, 11.7 / 19.5 / 23.9 -> 10.3 / 15.8 / 23.6; 32 / 8 of
// 128, 18.7 / 40.4 / 77.6 -> 13.7 / 39.6 / 72.9; 32 / 4 of 128, 26.5 / 39.4 / 72.4 -> 16.7 / 28.8 / 51.3;
// 16 / 2 of 256, 46 / 56 / 114 -> 31 / 38 / 72 (3.7 TB/s).
//
// Rounding: the scores' chains run over head_dim / 16 dims, then a tree of 16; the four tokens of a lane are
// summed before they join O. Error against float64 1.3e-7 to 2.1e-7 of the output's norm, the VALU kernel's
// 1.3e-7 to 2.0e-7 (single chains: up to 2.3e-7).
// ================================================================================================

// Sum over q4 of x[k], in the lanes of q4 = k.
__device__ __forceinline__ float rows_sum_scatter(const f32x4_t x) {
    const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(x[0]), __float_as_uint(x[2]), false, false);
    const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(x[1]), __float_as_uint(x[3]), false, false);
    const float sa = __uint_as_float(a[0]) + __uint_as_float(a[1]), sb = __uint_as_float(b[0]) + __uint_as_float(b[1]);
    const auto t = __builtin_amdgcn_permlane16_swap(__float_as_uint(sa), __float_as_uint(sb), false, false);
    return __uint_as_float(t[0]) + __uint_as_float(t[1]);
}

// Sum over ds (the quads of a row of 16 lanes), the same bits in each: rotations by 8, then by 4 lanes.
__device__ __forceinline__ float sum_ds(float x) {
    x += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0x128, 0xF, 0xF, false));
    return x + __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0x124, 0xF, 0xF, false));
}
// The values of a quad's four lanes.
__device__ __forceinline__ f32x4_t quad_values(float x) {
    const int b = __float_as_int(x);
    return f32x4_t{__int_as_float(__builtin_amdgcn_mov_dpp(b, 0x00, 0xF, 0xF, false)),
                   __int_as_float(__builtin_amdgcn_mov_dpp(b, 0x55, 0xF, 0xF, false)),
                   __int_as_float(__builtin_amdgcn_mov_dpp(b, 0xAA, 0xF, 0xF, false)),
                   __int_as_float(__builtin_amdgcn_mov_dpp(b, 0xFF, 0xF, 0xF, false))};
}

// Waves per SIMD whose registers the kernel is compiled for: what fits without spilling (head_dim 256 at two
// waves, 8 / 2 heads, 16 sequences of 64 to 2048: 52 us against 25 at one).
__host__ __device__ constexpr int fp32_mfma_waves(int D, int G) {
    return D == 256 ? 1 : D == 128 ? (G == 8 ? 2 : 3) : (G == 8 ? 3 : 5);
}

template <int D, int G, int PART>
__global__ __launch_bounds__(256, fp32_mfma_waves(D, G)) void paged_decode_fp32_mfma_kernel(const DecodeArgs a) {
    constexpr int NU = D / 16;     // 16-byte loads per lane of a K tile, and of a V tile
    constexpr int HG = (G + 3) / 4;  // groups of four heads
    constexpr int NBW = PART / 64; // blocks per wave
    constexpr int TILE = 16 * D;
    static_assert(D >= 32 && D <= 256, "fp32 kernel covers head_dim 32..256");
    static_assert(NBW < 64, "a lane per block id");

    __shared__ __align__(16) float s_q[HG * 4][D + 16];  // rows 64 bytes apart in the banks
    __shared__ float s_m[4][HG * 4], s_l[4][HG * 4];
    __shared__ float s_o[4][HG * 4][D];

    const int part = blockIdx.x, kvh = blockIdx.y, seq = blockIdx.z;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int Hkv = a.num_kv_heads, Hq = Hkv * G;
    const int tok0 = part * PART;
    const int c = lane & 3, ds = (lane >> 2) & 3, q4 = lane >> 4, n = lane & 15;

    // Ids of the wave's blocks (lane i: block i), loaded without waiting for the length.
    const int lb = tok0 / 16 + lane * 4 + wave;
    int ids = -1;
    if (lane < NBW && lb < a.max_blocks_per_seq) ids = a.block_tables[static_cast<int64_t>(seq) * a.max_blocks_per_seq + lb];
    // Q, by all threads (zeros past the group): in registers it would cost occupancy
    float qv[(HG * 4 * D + 255) / 256];
#pragma unroll
    for (int k = 0; k < (HG * 4 * D + 255) / 256; k++) {
        const int idx = min(tid + 256 * k, G * D - 1);
        const int64_t at = (static_cast<int64_t>(seq) * Hq + kvh * G) * D + idx;
        qv[k] = a.q_bf16 ? pa::bf16_to_f32(static_cast<const uint16_t*>(a.q)[at]) : static_cast<const float*>(a.q)[at];
    }
    const int T = clamp_len(a, a.context_lens[seq]);
    if (T <= 0) {
        if (part == 0)
            for (int idx = tid; idx < G * D; idx += 256)
                a.out[(static_cast<int64_t>(seq) * Hq + kvh * G) * D + idx] = 0.0f;
        return;
    }
    if (tok0 >= T) return;
    const int ntok = min(PART, T - tok0);
    const int nparts = (T + PART - 1) / PART;
    const int nbw = ((ntok + 15) / 16 - wave + 3) / 4;  // the wave's blocks

    // Loads of block i through a descriptor of its tile, which is empty (zeros, no traffic) for a
    // block past the wave's last or an id outside the cache.
    const char* const kc = static_cast<const char*>(a.k_cache);
    const char* const vc = static_cast<const char*>(a.v_cache);
    auto tile_rsrc = [&](const char* base, int i) {
        const int id = __builtin_amdgcn_readlane(ids, i);
        const bool ok = i < nbw && id >= 0 && id < a.num_blocks;
        const int64_t off = ok ? (static_cast<int64_t>(id) * Hkv + kvh) * (TILE * 4) : 0;
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(base) + off, 0, ok ? TILE * 4 : 0, kBufferFlags);
    };
    f32x4_t kr[NU], vr[NU];
    auto load_k = [&](int i) {
        const __amdgpu_buffer_rsrc_t rk = tile_rsrc(kc, i);
#pragma unroll
        for (int u = 0; u < NU; u++) kr[u] = buffer_load<f32x4_t>(rk, (4 * q4 + c) * (D * 4) + 16 * ds + 64 * u);
    };
    auto load_v = [&](int i) {
        const __amdgpu_buffer_rsrc_t rv = tile_rsrc(vc, i);
#pragma unroll
        for (int u = 0; u < NU; u++) vr[u] = buffer_load<f32x4_t>(rv, 64 * n + 16 * q4 + 1024 * u);
    };

    load_k(0);
    load_v(0);
#pragma unroll
    for (int k = 0; k < (HG * 4 * D + 255) / 256; k++) {
        const int idx = tid + 256 * k;
        if (idx < HG * 4 * D) s_q[idx / D][idx % D] = idx < G * D ? qv[k] : 0.0f;
    }
    __syncthreads();
    float m[HG], l[HG];  // head 4 h + c: running max; this q4's share of the sum
    f32x4_t acc[HG][NU];  // heads 4 h + i of dim 16 u + n: this q4's share
#pragma unroll
    for (int h = 0; h < HG; h++) {
        m[h] = -INFINITY;
        l[h] = 0.0f;
#pragma unroll
        for (int u = 0; u < NU; u++) acc[h][u] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    }
#pragma unroll 1
    for (int r = 0; r < nbw; r++) {
        int qo = 4 * ds;
        asm volatile("" : "+v"(qo));  // Q is read from LDS each time, not kept in registers
        f32x4_t s[HG];
#pragma unroll
        for (int h = 0; h < HG; h++) {
            f32x4_t part[4];  // by e: short chains, and a tree over them and ds
#pragma unroll
            for (int e = 0; e < 4; e++) part[e] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int u = 0; u < NU; u++) {
                const f32x4_t qf = *reinterpret_cast<const f32x4_t*>(&s_q[4 * h + c][16 * u + qo]);
#pragma unroll
                for (int e = 0; e < 4; e++) part[e] = __builtin_amdgcn_mfma_f32_4x4x1f32(kr[u][e], qf[e], part[e], 0, 0, 0);
            }
            s[h] = (part[0] + part[1]) + (part[2] + part[3]);
        }
        __builtin_amdgcn_sched_barrier(0);  // into the registers just consumed
        load_k(r + 1);                      // past the last block: an empty descriptor
        const int t0 = (r * 4 + wave) * 16 + 4 * q4;
        f32x4_t fr[HG];
#pragma unroll
        for (int h = 0; h < HG; h++) {
            float mx = m[h];
#pragma unroll
            for (int k = 0; k < 4; k++) {
                s[h][k] = t0 + k < ntok ? sum_ds(s[h][k]) * a.scale : -INFINITY;
                mx = fmaxf(mx, s[h][k]);
            }
            mx = rows_max(mx);
            const float ref = mx == -INFINITY ? 0.0f : mx;  // every score so far -inf: weights of 0, not NaN
            const float f = __expf(m[h] - ref);
            m[h] = mx;
            l[h] *= f;
#pragma unroll
            for (int k = 0; k < 4; k++) {
                s[h][k] = __expf(s[h][k] - ref);
                l[h] += s[h][k];
            }
            fr[h] = quad_values(f);
        }
        // O = O * rescale + (the block's four tokens, summed first)
#pragma unroll
        for (int h = 0; h < HG; h++)
#pragma unroll
            for (int u = 0; u < NU; u++) {
                f32x4_t o = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int k = 0; k < 4; k++) o = __builtin_amdgcn_mfma_f32_4x4x1f32(s[h][k], vr[u][k], o, 0, 0, 0);
#pragma unroll
                for (int i = 0; i < 4; i++) acc[h][u][i] = __builtin_fmaf(acc[h][u][i], fr[h][i], o[i]);
                if constexpr (D >= 128) {
                    if (u % 4 == 3) __builtin_amdgcn_sched_barrier(0);  // few partial sums at a time
                }
            }
        __builtin_amdgcn_sched_barrier(0);
        load_v(r + 1);
    }
    // ---- the waves' states combined (a wave without blocks: max -inf, sum and O 0) ----
#pragma unroll
    for (int h = 0; h < HG; h++) {
        const float lw = rows_sum(l[h]);
        if (lane < 4) {
            s_m[wave][4 * h + c] = m[h];
            s_l[wave][4 * h + c] = lw;
        }
#pragma unroll
        for (int u = 0; u < NU; u++) s_o[wave][4 * h + q4][16 * u + n] = rows_sum_scatter(acc[h][u]);
    }
    __syncthreads();
    for (int idx = tid; idx < G * D; idx += 256) {
        const int g = idx / D, d = idx - g * D;
        const float M = fmaxf(fmaxf(s_m[0][g], s_m[1][g]), fmaxf(s_m[2][g], s_m[3][g]));
        float o = 0.0f, lt = 0.0f;
#pragma unroll
        for (int w = 0; w < 4; w++) {
            const float f = __expf(s_m[w][g] - M);
            o += s_o[w][g][d] * f;
            lt += s_l[w][g] * f;
        }
        emit(a, seq, kvh * G + g, part, nparts, D, d, o, M, lt);
    }
}

// ================================================================================================

}  // namespace pa
