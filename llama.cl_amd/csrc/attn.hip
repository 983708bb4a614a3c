// Rotary embedding, KV-cache update and attention over the cache
// (attention_rope2 / attention_rope, /root/reference/ops/op_attn.hpp:721-1029 and :518-718).
//
// One query token: attn_decode_kernel (everything in one launch) and the merge of 3.  More:
//   1. attn_prep_kernel   rotate q and k in place (rope_embed, ops/op_attn.hpp:44-94), write the
//                         rotated k and the v rows into the cache at slots[p] (:764-773), and
//                         from 32 tokens on record which cache rows were written by which token of this call
//                         (attn_few_kernel does the first two itself where that saves time).  From 32 tokens on, all dimensions
//                         rotating, attn_prep_rows_kernel: the same without q, which attn_prefill_kernel rotates.
//   2. below 32 tokens    attn_split_kernel or attn_few_kernel: a workgroup takes a chunk of cache rows and leaves
//                         per query the chunk's score maximum, its sum of exponentials and its weighted V sum.
//      from 32 on         attn_prefill_kernel: 128 queries to a workgroup, the cache rows in one piece or in several.
//   3. merge_records      (attn_merge_rows_kernel or attn_merge_kernel) merges the chunks of a query with the usual max/sum rescaling and
//                         overwrites q with the result (:1018-1025).
// The cache element type is fp32 (reference layout) or fp16 (all arithmetic still fp32).
//
// In-chunk causal mask (:1007-1011): for query token pq, cache row slots[p'] is excluded for
// every p' in (pq, qL).  Excluded rows get weight exactly 0, as the reference's exp() returns 0
// for lowest()-max.
#include <float.h>
#include <limits.h>

#include "common.h"
#include "gemv_device.h"

namespace llmops {

typedef float v16f __attribute__((ext_vector_type(16)));

// ---- rope ------------------------------------------------------------------------------------
// theta = inv_freq[i] * (float)pos, cosf/sinf in fp32 (CosSin_cache::update, ops/op_attn.hpp:25-32)
__device__ __forceinline__ void rotate_pair(float& x0, float& x1, float c, float s) {
    const float y0 = c * x0 - s * x1;
    const float y1 = s * x0 + c * x1;
    x0 = y0;
    x1 = y1;
}
__device__ __forceinline__ void rotate4(float4& a, float4& b, float4 c, float4 s) {
    rotate_pair(a.x, b.x, c.x, s.x);
    rotate_pair(a.y, b.y, c.y, s.y);
    rotate_pair(a.z, b.z, c.z, s.z);
    rotate_pair(a.w, b.w, c.w, s.w);
}
__device__ __forceinline__ void rope_pair(float& x0, float& x1, float inv_freq, int pos) {
    const float xita = inv_freq * (float)pos;
    rotate_pair(x0, x1, cosf(xita), sinf(xita));
}

// x [B,H,L,S] in place; one thread per rotated pair
__global__ void rope_kernel(float* __restrict__ x, int64_t BH, int64_t L, int64_t S, const float* __restrict__ inv_freq,
                            int64_t half, int position_id) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= BH * L * half) return;
    const int64_t p = i % half, l = (i / half) % L, bh = i / (half * L);
    float* px = x + (bh * L + l) * S;
    float x0 = px[p], x1 = px[p + half];
    rope_pair(x0, x1, inv_freq[p], (int)l + position_id);
    px[p] = x0;
    px[p + half] = x1;
}

template <typename T>
__device__ __forceinline__ void store_cache(T* dst, float v);
template <>
__device__ __forceinline__ void store_cache<float>(float* dst, float v) {
    *dst = v;
}
template <>
__device__ __forceinline__ void store_cache<__half>(__half* dst, float v) {
    *dst = __float2half_rn(v);
}

// A workgroup's 64 entries of row_token (64 rows from 64 blockIdx.x on) and the two token ranges that go with them
__device__ __forceinline__ void fill_row_tokens(int32_t* token, int64_t qL, const int32_t* __restrict__ slots, int32_t* __restrict__ row_token,
                                                int2* __restrict__ tile_tokens, int64_t kvLen) {
    const int64_t row0 = (int64_t)blockIdx.x * 64;
    if (threadIdx.x < 64) token[threadIdx.x] = -1;
    __syncthreads();
    for (int64_t l = threadIdx.x; l < qL; l += blockDim.x) {
        const int64_t at = (int64_t)slots[l] - row0;
        if (at >= 0 && at < 64) atomicMax(&token[at], (int32_t)l);
    }
    __syncthreads();
    if (threadIdx.x >= 64) return;
    const int32_t mine = row0 + threadIdx.x < kvLen ? token[threadIdx.x] : INT_MAX;
    row_token[row0 + threadIdx.x] = mine;
    int lo = mine, hi = mine;
#pragma unroll
    for (int off = 1; off < 32; off <<= 1) lo = min(lo, __shfl_xor(lo, off, 64)), hi = max(hi, __shfl_xor(hi, off, 64));
    if ((threadIdx.x & 31) == 0) tile_tokens[row0 / 32 + threadIdx.x / 32] = make_int2(lo, hi);
}

// q,k,v [B,qL,H,S].  One workgroup of a wave per (b, l, h); thread i handles element i (and i+half).  TABLES: before those, `tables`
// workgroups each write 64 entries of row_token: the (last) token of this call that a cache row belongs to, -1, or from kvLen on
// INT_MAX, and the smallest and largest token of each 32 rows.  (us for the
// whole call, 32 heads, with a launch that filled the table with -1 and a scattered store per token / so: 64 tokens 17.9 / 17.2,
// 300 behind 300 50.0 / 48.3, 1024 tokens 84.6 / 82.1, 2048 tokens 175 / 172.)
template <typename T, bool TABLES>
__global__ void attn_prep_kernel(float* __restrict__ q, float* __restrict__ k, const float* __restrict__ v, int64_t qL,
                                 int64_t H, int64_t S, const float* __restrict__ inv_freq, int64_t half,
                                 T* __restrict__ kc, T* __restrict__ vc, int64_t maxlen, const int32_t* __restrict__ slots,
                                 int position_id, int32_t* __restrict__ row_token, int2* __restrict__ tile_tokens, int64_t kvLen, unsigned tables) {
    if (TABLES && blockIdx.x < tables) {
        __shared__ int32_t token[64];
        fill_row_tokens(token, qL, slots, row_token, tile_tokens, kvLen);
        return;
    }
    const int64_t item = TABLES ? blockIdx.x - tables : blockIdx.x;
    const int64_t h = item % H, l = (item / H) % qL, b = item / (H * qL);
    const int64_t base = ((b * qL + l) * H + h) * S;
    const int slot = slots[l];
    // slots live in device memory and cannot be validated on the host: a slot outside the cache is
    // dropped (q and k are still rotated) rather than written through
    const bool slot_ok = slot >= 0 && slot < maxlen;
    T* kdst = kc + ((b * H + h) * maxlen + (slot_ok ? slot : 0)) * S;
    T* vdst = vc + ((b * H + h) * maxlen + (slot_ok ? slot : 0)) * S;
    for (int64_t i = threadIdx.x; i < S; i += blockDim.x) {
        if (i < half) {
            float q0 = q[base + i], q1 = q[base + i + half];
            float k0 = k[base + i], k1 = k[base + i + half];
            const float f = inv_freq[i];
            rope_pair(q0, q1, f, (int)l + position_id);
            rope_pair(k0, k1, f, (int)l + position_id);
            q[base + i] = q0;
            q[base + i + half] = q1;
            k[base + i] = k0;
            k[base + i + half] = k1;
            if (slot_ok) {
                store_cache(kdst + i, k0);
                store_cache(kdst + i + half, k1);
            }
        } else if (i >= 2 * half && slot_ok) {
            store_cache(kdst + i, k[base + i]);
        }
        if (slot_ok) store_cache(vdst + i, v[base + i]);
    }
}

__device__ __forceinline__ float4 load4(const float* p) { return *reinterpret_cast<const float4*>(p); }
__device__ __forceinline__ float4 load4(const __half* p) {
    const uint2 u = *reinterpret_cast<const uint2*>(p);
    const __half2 a = *reinterpret_cast<const __half2*>(&u.x), b = *reinterpret_cast<const __half2*>(&u.y);
    const float2 fa = __half22float2(a), fb = __half22float2(b);
    return make_float4(fa.x, fa.y, fb.x, fb.y);
}

// a value as the cache holds it
template <typename T>
__device__ __forceinline__ float cache_round(float v);
template <>
__device__ __forceinline__ float cache_round<float>(float v) {
    return v;
}
template <>
__device__ __forceinline__ float cache_round<__half>(float v) {
    return __half2float(__float2half_rn(v));
}
template <typename T>
__device__ __forceinline__ void store4(T* dst, float4 v);
template <>
__device__ __forceinline__ void store4<float>(float* dst, float4 v) {
    *reinterpret_cast<float4*>(dst) = v;
}
template <>
__device__ __forceinline__ void store4<__half>(__half* dst, float4 v) {
    const __half2 a = __floats2half2_rn(v.x, v.y), b = __floats2half2_rn(v.z, v.w);
    uint2 u;
    u.x = *reinterpret_cast<const uint32_t*>(&a);
    u.y = *reinterpret_cast<const uint32_t*>(&b);
    *reinterpret_cast<uint2*>(dst) = u;
}

// The same ahead of attn_prefill_kernel where all 128 dimensions rotate (half 64): q stays as it is and is rotated by that kernel's
// workgroups on its way to their LDS; they take the cosines and sines from `turns` ([qL][cos 64, sin 64]).  Bound by memory, and q is 2/7 of
// what the kernel above moves.  A wave computes its token's 64 angles once, a lane each, for eight heads, 16 bytes to a lane.
// (The case of a whole call as a program makes it, q and k put back before it, us, both launches by the kernel above / so, the same bits: 32
// heads, 2048 tokens 185 / 174, 384 tokens halves 35.1 / 31.4, 128 behind 2000 37.9 / 35.5, 32 tokens 13.9 / 13.8; batches of 2 x 1000 137 / 124,
// 4 x 40 behind 100 halves 21.7 / 19.6, 8 x 200 behind 50 99 / 88.)
template <typename T>
__global__ __launch_bounds__(256) void attn_prep_rows_kernel(float* __restrict__ k, const float* __restrict__ v, int qL, int H, const float* __restrict__ inv_freq,
                                                             T* __restrict__ kc, T* __restrict__ vc, int64_t maxlen, const int32_t* __restrict__ slots,
                                                             int position_id, int32_t* __restrict__ row_token, int2* __restrict__ tile_tokens, int64_t kvLen,
                                                             unsigned tables, unsigned head_groups, float* __restrict__ turns) {
    constexpr int S = 128, kHeads = 32;
    __shared__ __align__(16) float turn[4][S];
    if (blockIdx.x < tables) {
        fill_row_tokens(reinterpret_cast<int32_t*>(turn), qL, slots, row_token, tile_tokens, kvLen);
        return;
    }
    const unsigned item = blockIdx.x - tables, bl = item / head_groups, group = item - bl * head_groups, b = bl / (unsigned)qL, l = bl - b * (unsigned)qL;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, c4 = 4 * (threadIdx.x & 15);
    const int slot = slots[l];
    const bool slot_ok = slot >= 0 && slot < maxlen;  // (as above)
    float4 kl[2], kh[2], vl[2], vh[2];
    const size_t base = ((size_t)bl * H) * S + c4;
    int head[2];
#pragma unroll
    for (int u = 0; u < 2; u++) {
        head[u] = (int)(group * kHeads) + 16 * u + (threadIdx.x >> 4);
        const size_t at = base + (size_t)min(head[u], H - 1) * S;  // (heads past the last re-read that one and store nothing)
        kl[u] = load4(k + at), kh[u] = load4(k + at + S / 2);
        vl[u] = load4(v + at), vh[u] = load4(v + at + S / 2);
    }
    const float xita = inv_freq[lane] * (float)((int)l + position_id);
    const float cs = cosf(xita), sn = sinf(xita);
    turn[wave][lane] = cs, turn[wave][S / 2 + lane] = sn;
    if (b == 0 && group == 0 && wave == 0) turns[(size_t)l * S + lane] = cs, turns[(size_t)l * S + S / 2 + lane] = sn;
    __syncthreads();
    const float4 c = load4(&turn[wave][c4]), s = load4(&turn[wave][S / 2 + c4]);
#pragma unroll
    for (int u = 0; u < 2; u++) {
        if (head[u] >= H) continue;
        const size_t at = base + (size_t)head[u] * S;
        rotate4(kl[u], kh[u], c, s);
        store4(k + at, kl[u]), store4(k + at + S / 2, kh[u]);
        if (slot_ok) {
            const size_t row = (((size_t)b * H + head[u]) * maxlen + slot) * S + c4;
            store4(kc + row, kl[u]), store4(kc + row + S / 2, kh[u]);
            store4(vc + row, vl[u]), store4(vc + row + S / 2, vh[u]);
        }
    }
}

// ---- split-KV attention of few query tokens over a short cache ----
// Per-chunk record in the workspace: [max, sum, out[S]]
// Workgroup = 4 waves; wave w owns rows w*PW .. w*PW+PW-1 of the chunk (C = 4*PW rows);
// lane = 32*hf + e: row parity hf, elements 4e..4e+3 (S == 128).
template <typename T, int PW>
__global__ __launch_bounds__(256) void attn_split_kernel(const float* __restrict__ q, const T* __restrict__ kc,
                                                          const T* __restrict__ vc, int64_t qL, int64_t H, int64_t maxlen,
                                                          int64_t kvLen, const int32_t* __restrict__ slots,
                                                          float* __restrict__ part, int nchunks) {
    constexpr int S = 128, C = 4 * PW, NL = PW / 2;
    __shared__ float sc[C];
    __shared__ float osh[4][2][S];
    __shared__ float stat[2];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int hf = lane >> 5, e = lane & 31;
    const int chunk = blockIdx.x % nchunks;
    const int64_t bhq = blockIdx.x / nchunks;  // ((b*H)+h)*qL + pq
    const int64_t pq = bhq % qL, h = (bhq / qL) % H, b = bhq / (qL * H);
    const int64_t p0 = (int64_t)chunk * C;
    const T* kbase = kc + (b * H + h) * maxlen * S;
    const T* vbase = vc + (b * H + h) * maxlen * S;

    // issue every K and V load of this wave before anything is consumed
    float4 kv[NL], vv[NL];
#pragma unroll
    for (int i = 0; i < NL; i++) {
        const int64_t p = p0 + wave * PW + i * 2 + hf;
        const int64_t pc = p < kvLen ? p : kvLen - 1;
        kv[i] = load4(kbase + pc * S + e * 4);
        vv[i] = load4(vbase + pc * S + e * 4);
    }
    const float4 qv = load4(q + ((b * qL + pq) * H + h) * S + e * 4);
    const int my_slot = slots[lane < qL ? lane : 0];  // (fewer than 32 tokens: a lane per slot)
    const float d_scale = 1.0f / sqrtf((float)S);

#pragma unroll
    for (int i = 0; i < NL; i++) {
        float s = qv.x * kv[i].x;
        s = fmaf(qv.y, kv[i].y, s);
        s = fmaf(qv.z, kv[i].z, s);
        s = fmaf(qv.w, kv[i].w, s);
#pragma unroll
        for (int o = 16; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
        const int r = wave * PW + i * 2 + hf;
        const int64_t p = p0 + r;
        if (e == 0) sc[r] = p < kvLen ? s * d_scale : -FLT_MAX;
    }
    __syncthreads();
    if (wave == 0) {
        float v = lane < C ? sc[lane] : -FLT_MAX;
        // rows that a later token of this call has written (slots from registers: with a scalar load for each, in every
        // wave, 31 tokens behind 97 of 8 heads took 15.6 us instead of 12.6)
        for (int l = (int)pq + 1; l < (int)qL; l++)
            if ((int64_t)__builtin_amdgcn_readlane(my_slot, l) == p0 + lane) v = -FLT_MAX;
        const float mx = wave_max(v);
        // a row counts only if it is live; a chunk with no live row reports sum 0
        float ex = (lane < C && v != -FLT_MAX) ? expf(v - mx) : 0.0f;
        if (lane < C) sc[lane] = ex;
        const float sum = wave_sum(ex);
        if (lane == 0) {
            stat[0] = mx;
            stat[1] = sum;
        }
    }
    __syncthreads();
    float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int i = 0; i < NL; i++) {
        const float w = sc[wave * PW + i * 2 + hf];
        o.x = fmaf(w, vv[i].x, o.x);
        o.y = fmaf(w, vv[i].y, o.y);
        o.z = fmaf(w, vv[i].z, o.z);
        o.w = fmaf(w, vv[i].w, o.w);
    }
    *reinterpret_cast<float4*>(&osh[wave][hf][e * 4]) = o;
    __syncthreads();
    float* rec = part + ((int64_t)bhq * nchunks + chunk) * (S + 2);
    if (threadIdx.x < S) {
        float a = 0.0f;
#pragma unroll
        for (int w = 0; w < 4; w++) a += osh[w][0][threadIdx.x] + osh[w][1][threadIdx.x];
        rec[2 + threadIdx.x] = a;
    }
    if (threadIdx.x == 0) {
        rec[0] = stat[0];
        rec[1] = stat[1];
    }
}

// ---- split-KV attention of few query tokens (fewer than 32, or one that the decode kernel does not take) ----
// Bound by reading the cache once: all query tokens of a head share every K and V row, through the matrix cores.  A
// workgroup takes 128 cache rows of a head, each of its four waves 32 of them, every load asked for before the first use;
// the waves' results meet in LDS and leave one record per query, [max, sum, out[S]], for attn_merge_kernel.  (One
// workgroup per query and chunk, on the vector ALU, read and multiplied the rows once per token: 16 tokens behind 1500,
// 32 heads, the whole call 68 us against 25; 31 behind 3500 239 against 44.)
//
// Arithmetic: fp32 operands are cut into three bf16 pieces, exactly (8 bits each, rounded to nearest; the exponent range
// is fp32's own); a product a*b is a1b1 + a1b2 + a2b1 + a2b2 + a1b3 + a3b1, each exact in the fp32 accumulators; what is
// dropped is below 2^-25 of the product.  Halves of an fp16 cache are two pieces.
//   S^T = K * Q^T: A = the lane's cache row (lane % 32), dims 16i + 8*hf .. +7; B = the lane's query (lane % 32), same dims.
//                  The result puts query lane % 32 into the lane, cache rows 8j + 4*hf + v.
//   O^T = V^T * P^T: A = V[those rows][column 4 * (lane % 32) + c], one 16-byte load per row; B = the probabilities as
//                  they sit in registers.  Result register 4j + v of product c: column 4 * (8j + 4*hf + v) + c.
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
union V8bfBits {
    v8bf h;
    uint32_t u[4];
};
struct Bf3 {
    V8bfBits p[3];
};
typedef __bf16 v2bf __attribute__((ext_vector_type(2)));
typedef float v2f_a __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t pack_bf(float a, float b) {  // rounded to nearest even (v_cvt_pk_bf16_f32)
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v2f_a{a, b}, v2bf));
}
// elements 2e, 2e+1 of the pieces
template <int PIECES>
__device__ __forceinline__ void split_bf(Bf3& d, int e, float a, float b) {
#pragma unroll
    for (int k = 0; k < PIECES; k++) {
        const uint32_t u = pack_bf(a, b);
        d.p[k].u[e] = u;
        a -= __uint_as_float(u << 16), b -= __uint_as_float(u & 0xFFFF0000u);
    }
}

// What does not go through the pieces: infinities (and what rounds to one, or whose products of pieces overflow where
// the sum would not) and values whose later pieces are subnormal, which the matrix cores take as zero.  A wave that meets
// such rows or queries forms its sums in fp32, as the per-query kernel does.  Scores: the former leave a score that is
// not finite; of the latter less than 2^-126 of the other factor is lost, which an exponent does not notice while |q| and
// |k| stay below 2^90.  Outputs: the lane's values are all below 2^56 and, unless all are zero, one of them reaches 2^-90.
constexpr float kFewMax = 0x1p56f, kFewMin = 0x1p-90f;
__device__ __forceinline__ float max_abs(float m, float4 v) {
    return fmaxf(fmaxf(fmaxf(fmaxf(m, fabsf(v.x)), fabsf(v.y)), fabsf(v.z)), fabsf(v.w));  // (in this order: two v_max3_f32)
}
// the wave's 32 x qL scores before scaling, into the layout of the MFMA's result; k_at(d), q_at(l, d): four dims from
// d + 8 * hf on of the lane's row and of query l; buf: 32 * 32 floats of the wave's own
template <typename K, typename Q>
__device__ __forceinline__ void few_scores_fp32(K k_at, Q q_at, int qL, float* buf, int c32, int hf, v16f& pr) {
    for (int l = 0; l < qL; l++) {
        float s = 0.0f;
#pragma unroll 1
        for (int i = 0; i < 8; i++) {
#pragma unroll
            for (int e = 0; e < 8; e += 4) {
                const float4 a = k_at(16 * i + e), w = q_at(l, 16 * i + e);
                s = fmaf(a.x, w.x, s), s = fmaf(a.y, w.y, s), s = fmaf(a.z, w.z, s), s = fmaf(a.w, w.w, s);
            }
        }
        s += __shfl_xor(s, 32, 64);
        if (hf == 0) buf[l * 32 + c32] = s;
    }
    __builtin_amdgcn_wave_barrier();
    const float* mine = buf + min(c32, qL - 1) * 32 + 4 * hf;
#pragma unroll
    for (int jj = 0; jj < 4; jj++) {
        const float4 x = *reinterpret_cast<const float4*>(mine + 8 * jj);
        pr[4 * jj] = x.x, pr[4 * jj + 1] = x.y, pr[4 * jj + 2] = x.z, pr[4 * jj + 3] = x.w;
    }
}
// the wave's 64 output elements of the lane's query; v_at(row, col): four columns of a row of the wave's 32; dst: the lane's
// place in the first of the 16 result registers
template <typename V>
__device__ __forceinline__ void few_outputs_fp32(V v_at, int hf, const v16f& pr, float* dst) {
    float w[2][16];  // [half that holds the row][register]
#pragma unroll
    for (int r = 0; r < 16; r++) {
        const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(pr[r]), __float_as_uint(pr[r]), false, false);
        w[0][r] = __uint_as_float(sw[0]), w[1][r] = __uint_as_float(sw[1]);
    }
#pragma unroll 1
    for (int r = 0; r < 16; r++) {
        const int col = 4 * (8 * (r >> 2) + 4 * hf + (r & 3));
        float4 a = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
        for (int row = 0; row < 32; row++) {
            const float4 v = v_at(row, col);
            const float p = w[(row >> 2) & 1][4 * (row >> 3) + (row & 3)];
            a.x = fmaf(p, v.x, a.x), a.y = fmaf(p, v.y, a.y), a.z = fmaf(p, v.z, a.z), a.w = fmaf(p, v.w, a.w);
        }
        *reinterpret_cast<float4*>(dst + r * 256) = a;
    }
}

// ROPE: rotation and cache update happen here too (a launch and its gap less).
// Every workgroup rotates the queries on their way to LDS, a thread per token and pair of dims.  The rows that this call
// writes are nobody's cache rows: they are masked, and their stale contents kept out of the products, wherever they lie in the
// cache; one more workgroup per head (the last chunk: FRESH) takes the call's own k and v in their place, rotates k, and
// writes k and the cache -- memory that no other workgroup uses.  Rotary pairs are 64 dims apart (other widths and the
// unrotated build: attn_prep_kernel before).
struct FewSmem {
    int tok[4][32];
    float wm[4][64], wl[4][64];
    float os[4][16][64][4];  // [wave][4j + v][lane][c]
    // Until the outputs, 22 rows of 132 floats lie behind the first 4 KB of an os[w] (which are the fp32 path's): the rotated
    // queries in os[3] and os[2], the FRESH workgroup's rotated k in os[1] and os[0].  (132: 16-byte reads of 32 rows at once
    // fall on different banks)
    __device__ __forceinline__ float* row(int l, int first) { return (l < 22 ? &os[first][4][0][0] + l * 132 : &os[first - 1][4][0][0] + (l - 22) * 132); }
};
template <typename T, bool ROPE, bool FRESH>
__device__ __forceinline__ void attn_few_body(FewSmem& sm, const float* __restrict__ q, T* __restrict__ kc, T* __restrict__ vc, int qL, int64_t H, int64_t maxlen,
                                              int kvLen, const int32_t* __restrict__ slots, float* __restrict__ part, int nchunks,
                                              float* __restrict__ k, const float* __restrict__ v, const float* __restrict__ inv_freq,
                                              int position_id) {
    constexpr int S = 128, P = sizeof(T) == 4 ? 3 : 2, IT = 8;  // (qL < 32: at most 8 tokens per wave)
    auto& tok = sm.tok;
    auto &wm = sm.wm, &wl = sm.wl;
    auto& os = sm.os;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int hf = lane >> 5, c32 = lane & 31;
    const int chunk = blockIdx.x % nchunks;
    const int64_t bh = blockIdx.x / nchunks, b = bh / H, h = bh % H;
    const int p0 = chunk * 128 + wave * 32;  // this wave's first cache row (FRESH: wave 0's row is token c32)
    T* kbase = kc + bh * maxlen * S;
    T* vbase = vc + bh * maxlen * S;
    const int64_t tokens = b * qL * H * S + h * S, stride = H * S;  // where the head's q, k, v rows start, and their distance
    const T* krow = kbase + (int64_t)min(p0 + c32, kvLen - 1) * S + 8 * hf;
    // row r of the wave's 32, four columns
    const auto v_at = [&](int row, int col) {
        if (!FRESH) return load4(vbase + (int64_t)min(p0 + row, kvLen - 1) * S + col);
        const float4 x = load4(v + tokens + min(row, qL - 1) * stride + col);
        return make_float4(cache_round<T>(x.x), cache_round<T>(x.y), cache_round<T>(x.z), cache_round<T>(x.w));
    };
    // (loads return in order: what masks and rotation need first)
    const int my_slot = ROPE ? slots[min(lane, qL - 1)] : 0;  // (fewer than 32 tokens: a lane per slot)
    float freq = 0.0f, qa[IT], qb[IT];
    float4 qr[16];  // (unrotated build: the lane's query straight from memory)
    if (ROPE) {
        freq = inv_freq[lane];
#pragma unroll
        for (int it = 0; it < IT; it++) {
            const float* at = q + tokens + min(wave + 4 * it, qL - 1) * stride + lane;
            qa[it] = at[0], qb[it] = at[64];
        }
    } else {
        const float* at = q + tokens + min(c32, qL - 1) * stride + 8 * hf;
#pragma unroll
        for (int i = 0; i < 8; i++) qr[2 * i] = load4(at + 16 * i), qr[2 * i + 1] = load4(at + 16 * i + 4);
    }
    float4 kr[16], vr[16];
    if (!FRESH) {
#pragma unroll
        for (int i = 0; i < 8; i++) kr[2 * i] = load4(krow + 16 * i), kr[2 * i + 1] = load4(krow + 16 * i + 4);
    }
#pragma unroll
    for (int r = 0; r < 16; r++) vr[r] = v_at(8 * (r >> 2) + 4 * hf + (r & 3), 4 * c32);
    __builtin_amdgcn_sched_barrier(0);
    if (!FRESH) {
        // which token of this call wrote the lane's cache row (-1: none); rows past the end belong to nobody, and with ROPE
        // neither do those of this call
        const int row = p0 + c32;
        int t = -1;
        for (int l = 0; l < qL; l++) t = (ROPE ? __builtin_amdgcn_readlane(my_slot, l) : slots[l]) == row ? l : t;
        tok[wave][c32] = row < kvLen && (!ROPE || t == -1) ? t : INT_MAX;
    }
    if (ROPE) {
#pragma unroll 1
        for (int l = wave; l < qL; l += 4) {  // (a loop of its own: one copy of the long code behind cosf and sinf)
            const float xita = freq * (float)(l + position_id);
            float* to = sm.row(l, 3);
            sincosf(xita, &to[lane + 64], &to[lane]);
        }
    }
#pragma unroll
    for (int it = 0; it < IT; it++) {
        const int l = wave + 4 * it;  // (uniform)
        if (!ROPE || l >= qL) break;
        float* to = sm.row(l, 3);
        const float c = to[lane], s = to[lane + 64];
        to[lane] = c * qa[it] - s * qb[it];
        to[lane + 64] = s * qa[it] + c * qb[it];
        if (FRESH) {
            const int slot = __builtin_amdgcn_readlane(my_slot, l);
            // (of several tokens with one slot the last one's row stays)
            const bool last = !__any(lane > l && lane < qL && my_slot == slot), stored = last && slot >= 0 && slot < maxlen;
            float* at = k + tokens + l * stride + lane;
            const float* vat = v + tokens + l * stride + lane;
            const float k0 = at[0], k1 = at[64], r0 = c * k0 - s * k1, r1 = s * k0 + c * k1;
            at[0] = r0, at[64] = r1;
            if (stored) {
                T *kdst = kbase + (int64_t)slot * S + lane, *vdst = vbase + (int64_t)slot * S + lane;
                store_cache(kdst, r0), store_cache(kdst + 64, r1);
                store_cache(vdst, vat[0]), store_cache(vdst + 64, vat[64]);
            }
            float* kto = sm.row(l, 1);
            kto[lane] = cache_round<T>(r0), kto[lane + 64] = cache_round<T>(r1);
            if (lane == 0) tok[0][l] = last && slot >= 0 && slot < kvLen ? l : INT_MAX;
        }
    }
    if (FRESH) {
        if (wave > 0 || lane >= qL) {
            if (lane < 32) tok[wave][lane] = INT_MAX;
        }
    }
    if (ROPE) __syncthreads();
    // no product with what a row holds that nobody sees: a weight of 0 does not take away an infinity
    const auto unseen = [&](int row) { return ROPE && tok[wave][row] == INT_MAX; };
    if (FRESH) {
        const float* mine = sm.row(min(c32, qL - 1), 1) + 8 * hf;
#pragma unroll
        for (int i = 0; i < 8; i++) kr[2 * i] = load4(mine + 16 * i), kr[2 * i + 1] = load4(mine + 16 * i + 4);
    }
    if (ROPE && (FRESH || __any(unseen(c32)))) {
        const bool none = unseen(c32);
#pragma unroll
        for (int i = 0; i < 16; i++) kr[i] = make_float4(none ? 0.f : kr[i].x, none ? 0.f : kr[i].y, none ? 0.f : kr[i].z, none ? 0.f : kr[i].w);
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const bool off = unseen(8 * (r >> 2) + 4 * hf + (r & 3));
            vr[r] = make_float4(off ? 0.f : vr[r].x, off ? 0.f : vr[r].y, off ? 0.f : vr[r].z, off ? 0.f : vr[r].w);
        }
    }
    const float* qrow = sm.row(min(c32, qL - 1), 3) + 8 * hf;
    // (two accumulators for the leading products and one for the small ones: fewer roundings at full size)
    v16f s0[2], s1;
#pragma unroll
    for (int r = 0; r < 16; r++) s0[0][r] = s0[1][r] = s1[r] = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; i++) {
        Bf3 a, w;
        split_bf<P>(a, 0, kr[2 * i].x, kr[2 * i].y), split_bf<P>(a, 1, kr[2 * i].z, kr[2 * i].w);
        split_bf<P>(a, 2, kr[2 * i + 1].x, kr[2 * i + 1].y), split_bf<P>(a, 3, kr[2 * i + 1].z, kr[2 * i + 1].w);
        const float4 q0 = ROPE ? load4(qrow + 16 * i) : qr[2 * i], q1 = ROPE ? load4(qrow + 16 * i + 4) : qr[2 * i + 1];
        split_bf<3>(w, 0, q0.x, q0.y), split_bf<3>(w, 1, q0.z, q0.w);
        split_bf<3>(w, 2, q1.x, q1.y), split_bf<3>(w, 3, q1.z, q1.w);
        s0[i & 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.p[0].h, w.p[0].h, s0[i & 1], 0, 0, 0);
        if (P == 3) s1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.p[2].h, w.p[0].h, s1, 0, 0, 0);
        s1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.p[0].h, w.p[2].h, s1, 0, 0, 0);
        s1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.p[1].h, w.p[1].h, s1, 0, 0, 0);
        s1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.p[1].h, w.p[0].h, s1, 0, 0, 0);
        s1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.p[0].h, w.p[1].h, s1, 0, 0, 0);
    }
    const float d_scale = 1.0f / sqrtf((float)S);
    const int pq = c32 < qL ? c32 : INT_MIN;
    __builtin_amdgcn_wave_barrier();
    v16f pr = (s0[0] + s0[1]) + s1;
    float z = 0.0f;  // NaN if a score is not finite
#pragma unroll
    for (int r = 0; r < 16; r++) z = fmaf(pr[r], 0.0f, z);
    if (__builtin_expect(__any(z != 0.0f), 0))
        few_scores_fp32(
            [&](int d) {
                if (unseen(c32)) return make_float4(0.f, 0.f, 0.f, 0.f);
                return FRESH ? load4(sm.row(min(c32, qL - 1), 1) + 8 * hf + d) : load4(krow + d);
            },
            [&](int l, int d) { return load4((ROPE ? sm.row(l, 3) : q + tokens + l * stride) + 8 * hf + d); }, qL, &os[wave][0][0][0], c32, hf, pr);
    float mx = -FLT_MAX;
#pragma unroll
    for (int jj = 0; jj < 4; jj++) {
        const int4 t4 = *reinterpret_cast<const int4*>(&tok[wave][8 * jj + 4 * hf]);
        const int tt[4] = {t4.x, t4.y, t4.z, t4.w};
#pragma unroll
        for (int v = 0; v < 4; v++) {
            pr[4 * jj + v] = tt[v] <= pq ? pr[4 * jj + v] * d_scale : -FLT_MAX;
            mx = fmaxf(mx, pr[4 * jj + v]);
        }
    }
    {  // the other half of the lane pair holds the other 16 rows
        const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(mx), __float_as_uint(mx), false, false);
        mx = fmaxf(__uint_as_float(sw[0]), __uint_as_float(sw[1]));
    }
    // the workgroup's maximum of every query, before the exponentials: all four waves use the same one
    wm[wave][lane] = mx;
    __syncthreads();
    mx = fmaxf(fmaxf(wm[0][lane], wm[1][lane]), fmaxf(wm[2][lane], wm[3][lane]));
    const float m0 = mx == -FLT_MAX ? 0.0f : mx;  // (a query that sees no row of the workgroup: all weights 0, sum 0)
    float sum = 0.0f;
#pragma unroll
    for (int r = 0; r < 16; r++) {
        pr[r] = expf(pr[r] - m0);
        sum += pr[r];
    }
    wl[wave][lane] = sum;
    float big[2] = {0.0f, 0.0f};
#pragma unroll
    for (int r = 0; r < 16; r++) big[r & 1] = max_abs(big[r & 1], vr[r]);
    big[0] = fmaxf(big[0], big[1]);
    if (__builtin_expect(__any(big[0] > kFewMax || (big[0] < kFewMin && big[0] > 0.0f)), 0)) {
        few_outputs_fp32([&](int row, int col) { return unseen(row) ? make_float4(0.f, 0.f, 0.f, 0.f) : v_at(row, col); }, hf, pr,
                         &os[wave][0][lane][0]);
    } else {
        v16f o[4];
#pragma unroll
        for (int c = 0; c < 4; c++)
#pragma unroll
            for (int r = 0; r < 16; r++) o[c][r] = 0.0f;
        Bf3 w[2];
#pragma unroll
        for (int e = 0; e < 8; e++) split_bf<3>(w[e >> 2], e & 3, pr[2 * e], pr[2 * e + 1]);
#pragma unroll
        for (int c = 0; c < 4; c++) {
            Bf3 a[2];
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const float4 v0 = vr[2 * e], v1 = vr[2 * e + 1];
                const float x0 = c == 0 ? v0.x : c == 1 ? v0.y : c == 2 ? v0.z : v0.w, x1 = c == 0 ? v1.x : c == 1 ? v1.y : c == 2 ? v1.z : v1.w;
                split_bf<P>(a[e >> 2], e & 3, x0, x1);
            }
#pragma unroll
            for (int bb = 0; bb < 2; bb++) {  // the small products first, while the sum is small
                if (P == 3) o[c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[bb].p[2].h, w[bb].p[0].h, o[c], 0, 0, 0);
                o[c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[bb].p[0].h, w[bb].p[2].h, o[c], 0, 0, 0);
                o[c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[bb].p[1].h, w[bb].p[1].h, o[c], 0, 0, 0);
            }
#pragma unroll
            for (int bb = 0; bb < 2; bb++) {
                o[c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[bb].p[1].h, w[bb].p[0].h, o[c], 0, 0, 0);
                o[c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[bb].p[0].h, w[bb].p[1].h, o[c], 0, 0, 0);
            }
#pragma unroll
            for (int bb = 0; bb < 2; bb++) o[c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[bb].p[0].h, w[bb].p[0].h, o[c], 0, 0, 0);
        }
#pragma unroll
        for (int r = 0; r < 16; r++) *reinterpret_cast<float4*>(&os[wave][r][lane][0]) = make_float4(o[0][r], o[1][r], o[2][r], o[3][r]);
    }
    __syncthreads();
    // wave w finishes the result registers 4w .. 4w+3: columns 4 * (8w + 4*hf + v) + c of the lane's query
    if (c32 >= qL) return;
    float* rec = part + ((bh * qL + c32) * nchunks + chunk) * (S + 2);
#pragma unroll
    for (int v = 0; v < 4; v++) {
        float4 a = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
        for (int w = 0; w < 4; w++) {
            const float4 x = *reinterpret_cast<const float4*>(&os[w][4 * wave + v][lane][0]);
            a.x += x.x, a.y += x.y, a.z += x.z, a.w += x.w;
        }
        float2* dst = reinterpret_cast<float2*>(rec + 2 + 4 * (8 * wave + 4 * hf + v));
        dst[0] = make_float2(a.x, a.y);
        dst[1] = make_float2(a.z, a.w);
    }
    if (wave == 0 && hf == 0) {
        float l = 0.0f;
#pragma unroll
        for (int w = 0; w < 4; w++) l += wl[w][lane] + wl[w][lane + 32];
        *reinterpret_cast<float2*>(rec) = make_float2(mx, l);
    }
}
template <typename T, bool ROPE>
__global__ __launch_bounds__(256, 2) void attn_few_kernel(const float* __restrict__ q, T* __restrict__ kc, T* __restrict__ vc, int qL, int64_t H, int64_t maxlen,
                                                           int kvLen, const int32_t* __restrict__ slots, float* __restrict__ part,
                                                           int nchunks, float* __restrict__ k, const float* __restrict__ v,
                                                           const float* __restrict__ inv_freq, int position_id) {
    __shared__ __align__(16) FewSmem sm;
    if (ROPE && blockIdx.x % nchunks == nchunks - 1)
        attn_few_body<T, ROPE, true>(sm, q, kc, vc, qL, H, maxlen, kvLen, slots, part, nchunks, k, v, inv_freq, position_id);
    else
        attn_few_body<T, ROPE, false>(sm, q, kc, vc, qL, H, maxlen, kvLen, slots, part, nchunks, k, v, inv_freq, position_id);
}

// Merge of the chunk records of one query: out = sum_c exp(m_c - M) o_c / sum_c exp(m_c - M) s_c.
// LOAD fetches one float of a record.
template <typename LOAD>
__device__ __forceinline__ float merge_chunks(const float* rec, int nchunks, int tid, LOAD load) {
    constexpr int S = 128, CB = 32;
    float M = -FLT_MAX, den = 0.0f, num = 0.0f;
    // every thread reads the (few) chunk statistics itself, so all loads of a batch of chunks are
    // independent and in flight together; batches are folded in with the running-max rescaling
    for (int c0 = 0; c0 < nchunks; c0 += CB) {
        float m[CB], sm[CB], o[CB];
#pragma unroll
        for (int u = 0; u < CB; u++) {
            const bool ok = c0 + u < nchunks;
            const float* r = rec + (int64_t)(ok ? c0 + u : c0) * (S + 2);
            m[u] = ok ? load(r) : -FLT_MAX;
            sm[u] = ok ? load(r + 1) : 0.0f;
            o[u] = ok ? load(r + 2 + tid) : 0.0f;
        }
        float Mb = M;
#pragma unroll
        for (int u = 0; u < CB; u++) Mb = fmaxf(Mb, m[u]);
        const float rescale = (den == 0.0f) ? 0.0f : expf(M - Mb);
        den *= rescale;
        num *= rescale;
#pragma unroll
        for (int u = 0; u < CB; u++) {
            const float sc = (sm[u] == 0.0f) ? 0.0f : expf(m[u] - Mb);
            den = fmaf(sc, sm[u], den);
            num = fmaf(sc, o[u], num);
        }
        M = Mb;
    }
    return num * (1.0f / den);
}

// `nchunks` records per query are laid out; with pos_dev (decode graphs) only the first
// ceil(min(pos_dev[0] + 1, maxlen) / chunk_rows) of them were written by this call.
__global__ __launch_bounds__(128) void attn_merge_kernel(float* __restrict__ q, const float* __restrict__ part, int64_t qL,
                                                          int64_t H, int nchunks, int chunk_rows = 1,
                                                          const int32_t* __restrict__ pos_dev = nullptr, int64_t maxlen = 0) {
    constexpr int S = 128;
    __shared__ float wsh[2][64];
    const int64_t bhq = blockIdx.x;
    const int64_t pq = bhq % qL, h = (bhq / qL) % H, b = bhq / (qL * H);
    const float* rec = part + (int64_t)bhq * nchunks * (S + 2);
    if (pos_dev != nullptr) nchunks = (int)((min((int64_t)pos_dev[0] + 1, maxlen) + chunk_rows - 1) / chunk_rows);
    float r;
    if (nchunks <= 64) {
        // The chunk weights exp(m_c - M) / sum are the same for all 128 output elements: each wave computes
        // them once, one chunk per lane (one expf per lane instead of one per chunk and thread), and every
        // thread then only accumulates its element over the chunks.  Loads in order of use (statistics, then
        // the partial outputs, the first 32 in flight together with the statistics), addresses clamped instead of branched around.
        const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
        const float* rc = rec + (int64_t)min(lane, nchunks - 1) * (S + 2);
        const float m = rc[0], sm0 = rc[1];
        // (the first 32 partial outputs do not depend on the weights: asked for before the weights are computed)
        float o0[32];
#pragma unroll
        for (int u = 0; u < 32; u++) o0[u] = rec[(int64_t)min(u, nchunks - 1) * (S + 2) + 2 + threadIdx.x];
        __builtin_amdgcn_sched_barrier(0);
        float acc = 0.0f;
        const float mm = lane < nchunks ? m : -FLT_MAX;
        const float sm = lane < nchunks ? sm0 : 0.0f;
        const float M = wave_max(mm);
        const float w = (sm == 0.0f) ? 0.0f : expf(mm - M);
        const float den = wave_sum(w * sm);
        wsh[wave][lane] = w * (1.0f / den);
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int u = 0; u < 32; u++) acc = fmaf(u < nchunks ? wsh[wave][u] : 0.0f, o0[u], acc);
        for (int c0 = 32; c0 < nchunks; c0 += 16) {
            float o[16];
#pragma unroll
            for (int u = 0; u < 16; u++) o[u] = rec[(int64_t)min(c0 + u, nchunks - 1) * (S + 2) + 2 + threadIdx.x];
#pragma unroll
            for (int u = 0; u < 16; u++) acc = fmaf(c0 + u < nchunks ? wsh[wave][c0 + u] : 0.0f, o[u], acc);
        }
        r = acc;
    } else {
        r = merge_chunks(rec, nchunks, threadIdx.x, [](const float* p) { return *p; });
    }
    q[((b * qL + pq) * H + h) * S + threadIdx.x] = r;
}

// The same, bit for bit, for up to N records of a query whose number is known: half a wave to a query, 16 bytes to a lane, all records of
// eight queries asked for at once.  Bound by one round trip to memory with few queries, by the records with many.  (512 tokens behind 1500,
// 32 heads, two records each: 20 us by attn_merge_kernel's workgroup per query, 7; fewer tokens: at merge_records.)
template <int N>
__global__ __launch_bounds__(256) void attn_merge_rows_kernel(float* __restrict__ q, const float* __restrict__ part, int qL, int H,
                                                               unsigned queries, int nchunks) {
#pragma clang fp contract(off)  // (the products of den are rounded as those of attn_merge_kernel are)
    constexpr int S = 128;
    const unsigned bhq = blockIdx.x * 8 + (threadIdx.x >> 5);
    const int at = 4 * (threadIdx.x & 31);
    if (bhq >= queries) return;
    const float* rec = part + (size_t)bhq * nchunks * (S + 2);
    float2 st[N], lo[N], hi[N];
#pragma unroll
    for (int c = 0; c < N; c++) {
        const float* rc = rec + min(c, nchunks - 1) * (S + 2);
        st[c] = *reinterpret_cast<const float2*>(rc);
        lo[c] = *reinterpret_cast<const float2*>(rc + 2 + at);
        hi[c] = *reinterpret_cast<const float2*>(rc + 4 + at);
    }
    float M = -FLT_MAX, den[N], w[N];
#pragma unroll
    for (int c = 0; c < N; c++) M = fmaxf(M, st[c].x);  // (records past the last are copies of it)
#pragma unroll
    for (int c = 0; c < N; c++) {
        w[c] = c >= nchunks || st[c].y == 0.0f ? 0.0f : expf(st[c].x - M);
        den[c] = w[c] * st[c].y;
    }
#pragma unroll
    for (int o = N / 2; o > 0; o >>= 1)  // (the order of wave_sum: the bits of attn_merge_kernel)
#pragma unroll
        for (int c = 0; c < o; c++) den[c] += den[c + o];
    const float inv = 1.0f / den[0];
    float4 acc = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll
    for (int c = 0; c < N; c++) {
        const float wc = w[c] * inv;
        acc.x = fmaf(wc, lo[c].x, acc.x), acc.y = fmaf(wc, lo[c].y, acc.y);
        acc.z = fmaf(wc, hi[c].x, acc.z), acc.w = fmaf(wc, hi[c].y, acc.w);
    }
    const unsigned pq = bhq % (unsigned)qL, bh = bhq / (unsigned)qL, h = bh % (unsigned)H, b = bh / (unsigned)H;
    *reinterpret_cast<float4*>(q + (((size_t)b * qL + pq) * H + h) * S + at) = acc;
}

// ---- decode attention (one query token) ------------------------------------------------------
// attention_rope2 for qL == 1: every workgroup rotates q itself (cos/sin of the position computed once
// per workgroup, one angle per lane), the workgroup whose chunk holds the new token's cache row rotates
// k, writes the rotated k back in place and k, v into the cache, and attends to the new row from
// registers.  The chunk records (max, sum, weighted V sum) are merged by attn_merge_kernel, a second
// launch.  (Merging inside this kernel, by whichever workgroup of a head takes the last arrival ticket, was
// measured slower at every size: the record stores must be acknowledged before the ticket is taken and the
// last workgroup then fetches the records, three round trips to memory against one launch -- kv 256: 9.2
// against 8.2 us, kv 2048: 25.4 against 19.0 us.  One workgroup of 16 wavefronts per head, which needs no
// merge, is bound by what one compute unit can fetch: kv 256 9.1 against 8.2 us, kv 512 with an fp16 cache 20.4
// against 9.4 us.)  A head with a single chunk (nchunks == 1) is finished here and written straight into q.
//
// A lane always fetches 16 bytes of a cache row: 4 floats or 8 halves.  A 128-element row is therefore
// LPR = 32 (fp32) or 16 (fp16) lanes wide and one wave-wide load covers RPW = 2 or 4 rows; a wave owns PW
// rows of the chunk, NL = PW / RPW loads per lane for K and as many for V.
//
// The position may come from device memory (pos_dev != nullptr): a HIP graph of a decode step captures the
// launch once, for the largest kv length (the grid and the record layout are sized by `nchunks`), and every
// replay reads the current position; workgroups whose chunk lies beyond the current kv length leave at once.
// rotate the lane's 4 elements (index e4 = first element) of a 128-wide head vector at `base`;
// cs = cos table [half], sn = sin table [half] of the current position (LDS)
__device__ __forceinline__ float4 rope4(const float* base, int e4, const float* cs, const float* sn, int half) {
    const float4 own = *reinterpret_cast<const float4*>(base + e4);
    if (e4 >= 2 * half) return own;
    const bool low = e4 < half;
    const float4 other = *reinterpret_cast<const float4*>(base + (low ? e4 + half : e4 - half));
    const int f0 = low ? e4 : e4 - half;
    float o[4] = {own.x, own.y, own.z, own.w}, p[4] = {other.x, other.y, other.z, other.w}, r[4];
#pragma unroll
    for (int c = 0; c < 4; c++) {
        // pair (x0 = element i, x1 = element i+half): y0 = c*x0 - s*x1, y1 = s*x0 + c*x1
        r[c] = low ? cs[f0 + c] * o[c] - sn[f0 + c] * p[c] : sn[f0 + c] * p[c] + cs[f0 + c] * o[c];
    }
    return make_float4(r[0], r[1], r[2], r[3]);
}

// the same on values already in registers: `own` = the lane's 4 elements at e4, `other` = their partners
__device__ __forceinline__ float4 rope4_regs(float4 own, float4 other, int e4, const float* cs, const float* sn, int half) {
    if (e4 >= 2 * half) return own;
    const bool low = e4 < half;
    const int f0 = low ? e4 : e4 - half;
    float o[4] = {own.x, own.y, own.z, own.w}, p[4] = {other.x, other.y, other.z, other.w}, r[4];
#pragma unroll
    for (int c = 0; c < 4; c++) r[c] = low ? cs[f0 + c] * o[c] - sn[f0 + c] * p[c] : sn[f0 + c] * p[c] + cs[f0 + c] * o[c];
    return make_float4(r[0], r[1], r[2], r[3]);
}
__device__ __forceinline__ int rope_partner(int e4, int half) {
    return e4 >= 2 * half ? e4 : (e4 < half ? e4 + half : e4 - half);
}

// 16 bytes of a cache row as they come from memory, and their widening to floats
template <typename T>
struct RowPiece;
template <>
struct RowPiece<float> {
    static constexpr int EPL = 4;  // elements per lane
    static __device__ __forceinline__ void widen(const uint4& r, float out[4]) {
        out[0] = __uint_as_float(r.x), out[1] = __uint_as_float(r.y), out[2] = __uint_as_float(r.z), out[3] = __uint_as_float(r.w);
    }
    // the 16 bytes as the cache stores them
    static __device__ __forceinline__ uint4 pack(const float4* v) {
        return make_uint4(__float_as_uint(v[0].x), __float_as_uint(v[0].y), __float_as_uint(v[0].z), __float_as_uint(v[0].w));
    }
};
template <>
struct RowPiece<__half> {
    static constexpr int EPL = 8;
    static __device__ __forceinline__ float lo(uint32_t w) { return __half2float(__ushort_as_half((unsigned short)(w & 0xFFFFu))); }
    static __device__ __forceinline__ float hi(uint32_t w) { return __half2float(__ushort_as_half((unsigned short)(w >> 16))); }
    static __device__ __forceinline__ void widen(const uint4& r, float out[8]) {
        out[0] = lo(r.x), out[1] = hi(r.x), out[2] = lo(r.y), out[3] = hi(r.y);
        out[4] = lo(r.z), out[5] = hi(r.z), out[6] = lo(r.w), out[7] = hi(r.w);
    }
    static __device__ __forceinline__ uint32_t pack2(float a, float b) {
        return (uint32_t)__half_as_ushort(__float2half_rn(a)) | ((uint32_t)__half_as_ushort(__float2half_rn(b)) << 16);
    }
    static __device__ __forceinline__ uint4 pack(const float4* v) {
        return make_uint4(pack2(v[0].x, v[0].y), pack2(v[0].z, v[0].w), pack2(v[1].x, v[1].y), pack2(v[1].z, v[1].w));
    }
};
// cache rows are read exactly once per call: non-temporal, so that they do not displace the records and the
// activations that are reused out of the caches
__device__ __forceinline__ uint4 load_row16(const void* p) {
    typedef unsigned int u32x4_a __attribute__((ext_vector_type(4)));
    const u32x4_a v = __builtin_nontemporal_load(reinterpret_cast<const u32x4_a*>(p));
    return make_uint4(v.x, v.y, v.z, v.w);
}

//
// RECS: the chunk records are not merged here at all but handed to the FC that consumes the attention output
// (the o projection merges them as it loads its input, llmops_fc_Q4A_decode_attn): workgroups of NWV = 16
// wavefronts take 256 or 512 cache rows each, so that a head has at most kAttnRecChunks records, laid out as
// stats [B*H][kAttnRecChunks][2] (max, sum) and outs [B*H][kAttnRecChunks][128]; a chunk beyond the current kv
// length leaves an empty record (sum 0, zeros).  q is then left as it came in.
constexpr int kAttnRecChunks = 8;

template <typename T, int PW, int NWV = 4, bool RECS = false>
__global__ __launch_bounds__(NWV * 64) void attn_decode_kernel(const int32_t* __restrict__ pos_dev, int position_id, int nchunks,
                                                           int maxlen, T* kc, T* vc, const int32_t* __restrict__ slots,
                                                           float* q, float* k, const float* __restrict__ v,
                                                           const float* __restrict__ inv_freq, int half, float* part,
                                                           float* rec_stats = nullptr, float* rec_outs = nullptr) {
    // (argument order: the first 14 dwords arrive in scalar registers with the wave (kernel-argument preload);
    // they are what the position, the slot and the cache rows' addresses need)
    constexpr int S = 128, C = NWV * PW;
    constexpr int EPL = RowPiece<T>::EPL, LPR = S / EPL, RPW = 64 / LPR, NL = PW / RPW;
    static_assert(NL >= 1 && NL <= LPR, "rows per lane");
    __shared__ float sc[C];
    __shared__ float osh[NWV][RPW][S];
    __shared__ float stat[2];
    __shared__ float cs_sh[64], sn_sh[64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int rsel = lane / LPR, e = lane % LPR;  // which of the RPW rows of a wave-wide load, which 16 bytes of it
    // grid = (chunks, heads): no division, and 32-bit row arithmetic throughout -- every instruction in front of
    // the first cache row is paid once per wave before the memory system has anything to do
    const int chunk = blockIdx.x;
    const uint32_t bh = blockIdx.y;
    // One round trip for everything that did not come with the wave: the slot, the position (read through a
    // pointer that is always valid, so that there is no branch around the load) and the remaining arguments,
    // which the compiler would otherwise fetch one by one where the code first uses them.
    const int slot = slots[0];
    const int pos_loaded = (pos_dev != nullptr ? pos_dev : slots)[0];
    asm volatile("" ::"s"(slot), "s"(pos_loaded), "s"(k), "s"(v), "s"(inv_freq), "s"(half), "s"(rec_stats), "s"(rec_outs), "s"(part));
    if (pos_dev != nullptr) position_id = pos_loaded;
    const int kvLen = position_id < maxlen ? position_id + 1 : maxlen;
    const int nact = (int)((unsigned)(kvLen + C - 1) / C);  // chunks that hold rows at this position (none if kvLen <= 0)
    if (chunk >= nact || kvLen <= 0) {
        if (RECS) {  // an empty record: weight 0 whatever the others hold
            if (threadIdx.x < S) rec_outs[((size_t)bh * kAttnRecChunks + chunk) * S + threadIdx.x] = 0.0f;
            if (threadIdx.x == 0) {
                rec_stats[((size_t)bh * kAttnRecChunks + chunk) * 2] = -FLT_MAX;
                rec_stats[((size_t)bh * kAttnRecChunks + chunk) * 2 + 1] = 0.0f;
            }
        }
        return;
    }
    const int p0 = chunk * C;
    // a head's plane of the cache is below 4 GiB (checked by the launcher): uniform 64-bit base, 32-bit lane offsets
    T* kbase = kc + (size_t)bh * ((uint32_t)maxlen * (uint32_t)S);
    T* vbase = vc + (size_t)bh * ((uint32_t)maxlen * (uint32_t)S);
    const float* qrow = q + (size_t)bh * S;
    float* krow = k + (size_t)bh * S;
    const float* vrow = v + (size_t)bh * S;

    // Loads return in issue order and a wave can only wait for "all but the youngest n".  So the small
    // loads whose data the rotation needs go first, then the K rows, then the V rows: the cos/sin table,
    // the rotation of q (and k) and the scores are then computed while the rows behind them are still in
    // flight, instead of after the last V row has landed.
    const bool slot_ok = slot >= 0 && slot < maxlen;
    // the workgroup that owns the new token's row (or the last chunk, if the row lies beyond kvLen)
    const int owner = (slot_ok && slot / C < nact) ? slot / C : nact - 1;
    const int e0 = e * EPL;  // the lane's first element of the row
    const float freq = inv_freq[min((int)threadIdx.x, half - 1)];
    float4 q_own[EPL / 4], q_oth[EPL / 4];
#pragma unroll
    for (int u = 0; u < EPL / 4; u++) {
        q_own[u] = *reinterpret_cast<const float4*>(qrow + (uint32_t)(e0 + 4 * u));
        q_oth[u] = *reinterpret_cast<const float4*>(qrow + (uint32_t)rope_partner(e0 + 4 * u, half));
    }
    // The new token's k and v rows: only the owner uses them, but every workgroup asks for them (48-96 bytes per
    // lane out of L2): a branch around these loads would leave the registers with two definitions, and the copies
    // that merge them wait for the loads -- one memory round trip in front of the owner's first cache row.
    float4 kn[EPL / 4], k_oth[EPL / 4], vn[EPL / 4];
#pragma unroll
    for (int u = 0; u < EPL / 4; u++) {
        kn[u] = *reinterpret_cast<const float4*>(krow + (uint32_t)(e0 + 4 * u));
        k_oth[u] = *reinterpret_cast<const float4*>(krow + (uint32_t)rope_partner(e0 + 4 * u, half));
        vn[u] = *reinterpret_cast<const float4*>(vrow + (uint32_t)(e0 + 4 * u));
    }
    __builtin_amdgcn_sched_barrier(0);
    uint4 kraw[NL], vraw[NL];
#pragma unroll
    for (int i = 0; i < NL; i++) {
        const int pc = min(p0 + wave * PW + i * RPW + rsel, kvLen - 1);
        kraw[i] = load_row16(kbase + (uint32_t)(pc * S + e0));
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < NL; i++) {
        const int pc = min(p0 + wave * PW + i * RPW + rsel, kvLen - 1);
        vraw[i] = load_row16(vbase + (uint32_t)(pc * S + e0));
    }
    __builtin_amdgcn_sched_barrier(0);
    if (threadIdx.x < half) {
        const float xita = freq * (float)position_id;
        cs_sh[threadIdx.x] = cosf(xita);
        sn_sh[threadIdx.x] = sinf(xita);
    }
    __syncthreads();
    float qv[EPL];
#pragma unroll
    for (int u = 0; u < EPL / 4; u++) {
        const float4 r = rope4_regs(q_own[u], q_oth[u], e0 + 4 * u, cs_sh, sn_sh, half);
        qv[4 * u] = r.x, qv[4 * u + 1] = r.y, qv[4 * u + 2] = r.z, qv[4 * u + 3] = r.w;
    }
    // the new token's row as the cache holds it (rounded to T): it is attended to from registers
    uint4 knraw = make_uint4(0, 0, 0, 0), vnraw = knraw;
    if (chunk == owner) {
        // The new v row is only needed here, and its conversion to the cache's type must stay here: the compiler
        // otherwise moves it up into the block that loads the row, in front of the cache rows' loads, and the
        // owner workgroup then waits for one round trip before it asks for its first cache row.  Tying the values
        // to something read after the barrier keeps the conversion below it.
        const float after_barrier = cs_sh[0];
#pragma unroll
        for (int u = 0; u < EPL / 4; u++)
            asm volatile("" : "+v"(vn[u].x), "+v"(vn[u].y), "+v"(vn[u].z), "+v"(vn[u].w) : "v"(after_barrier));
#pragma unroll
        for (int u = 0; u < EPL / 4; u++) kn[u] = rope4_regs(kn[u], k_oth[u], e0 + 4 * u, cs_sh, sn_sh, half);
        knraw = RowPiece<T>::pack(kn);
        vnraw = RowPiece<T>::pack(vn);
        __syncthreads();  // every wave has read the raw k before it is overwritten
        if (wave == 0 && rsel == 0) {
#pragma unroll
            for (int u = 0; u < EPL / 4; u++) *reinterpret_cast<float4*>(krow + (uint32_t)(e0 + 4 * u)) = kn[u];
            if (slot_ok) {
                *reinterpret_cast<uint4*>(kbase + (uint32_t)(slot * S + e0)) = knraw;
                *reinterpret_cast<uint4*>(vbase + (uint32_t)(slot * S + e0)) = vnraw;
            }
        }
#pragma unroll
        for (int i = 0; i < NL; i++)
            if (p0 + wave * PW + i * RPW + rsel == slot) kraw[i] = knraw;
    }
    const float d_scale = 1.0f / sqrtf((float)S);
    // NL partial dot products per lane, each to be summed over the LPR lanes of a row.  Summing them one
    // by one takes log2(LPR) lane exchanges each; instead the lanes split the rows between them while they
    // add: at every exchange a lane keeps one half of its rows and hands the other half to its partner,
    // so NL rows cost NL/2 + NL/4 + .. + 1 exchanges plus one per remaining lane bit.
    float sp[NL];
#pragma unroll
    for (int i = 0; i < NL; i++) {
        float kf[EPL];
        RowPiece<T>::widen(kraw[i], kf);
        float s = 0.0f;
#pragma unroll
        for (int c = 0; c < EPL; c++) s = fmaf(qv[c], kf[c], s);
        sp[i] = s;
    }
    int row_of_lane = 0;  // which of the NL rows this lane ends up holding
    {
        int n = NL, off = LPR / 2;
#pragma unroll
        for (; n > 1; n >>= 1, off >>= 1) {
            const bool up = (e & off) != 0;
#pragma unroll
            for (int j = 0; j < NL / 2; j++) {
                if (j < n / 2) {
                    const float keep = up ? sp[j + n / 2] : sp[j];
                    const float send = up ? sp[j] : sp[j + n / 2];
                    sp[j] = keep + __shfl_xor(send, off, 64);
                }
            }
            row_of_lane = row_of_lane * 2 + (up ? 1 : 0);
        }
#pragma unroll
        for (; off > 0; off >>= 1) sp[0] += __shfl_xor(sp[0], off, 64);
    }
    {
        // lanes whose remaining (low) bits are zero write the row they hold
        constexpr int kLowMask = LPR / NL - 1;
        const int r = wave * PW + row_of_lane * RPW + rsel;
        if ((e & kLowMask) == 0) sc[r] = (p0 + r < kvLen) ? sp[0] * d_scale : -FLT_MAX;
    }
    __syncthreads();
    if (wave == 0) {
        float mx = -FLT_MAX;
#pragma unroll
        for (int u = 0; u < (C + 63) / 64; u++) mx = fmaxf(mx, lane + 64 * u < C ? sc[lane + 64 * u] : -FLT_MAX);
        mx = wave_max(mx);
        float sum = 0.0f;
#pragma unroll
        for (int u = 0; u < (C + 63) / 64; u++) {
            const int r = lane + 64 * u;
            if (r < C) {
                const float x = sc[r];
                const float ex = (x != -FLT_MAX) ? expf(x - mx) : 0.0f;
                sc[r] = ex;
                sum += ex;
            }
        }
        sum = wave_sum(sum);
        if (lane == 0) {
            stat[0] = mx;
            stat[1] = sum;
        }
    }
    __syncthreads();
    if (chunk == owner) {
#pragma unroll
        for (int i = 0; i < NL; i++)
            if (p0 + wave * PW + i * RPW + rsel == slot) vraw[i] = vnraw;
    }
    float o[EPL];
#pragma unroll
    for (int c = 0; c < EPL; c++) o[c] = 0.0f;
#pragma unroll
    for (int i = 0; i < NL; i++) {
        float vf[EPL];
        RowPiece<T>::widen(vraw[i], vf);
        const float w = sc[wave * PW + i * RPW + rsel];
#pragma unroll
        for (int c = 0; c < EPL; c++) o[c] = fmaf(w, vf[c], o[c]);
    }
#pragma unroll
    for (int u = 0; u < EPL / 4; u++)
        *reinterpret_cast<float4*>(&osh[wave][rsel][e0 + 4 * u]) = make_float4(o[4 * u], o[4 * u + 1], o[4 * u + 2], o[4 * u + 3]);
    __syncthreads();
    float* rec = part + ((size_t)bh * nchunks + chunk) * (S + 2);
    float mine = 0.0f;  // this thread's element of the chunk's weighted V sum (threads 0..127)
    if (threadIdx.x < S) {
#pragma unroll
        for (int w = 0; w < NWV; w++)
#pragma unroll
            for (int r = 0; r < RPW; r++) mine += osh[w][r][threadIdx.x];
    }
    if (RECS) {
        if (threadIdx.x < S) rec_outs[((size_t)bh * kAttnRecChunks + chunk) * S + threadIdx.x] = mine;
        if (threadIdx.x == 0) {
            rec_stats[((size_t)bh * kAttnRecChunks + chunk) * 2] = stat[0];
            rec_stats[((size_t)bh * kAttnRecChunks + chunk) * 2 + 1] = stat[1];
        }
        return;
    }
    if (nchunks == 1) {  // the workgroup saw every row of the head
        if (threadIdx.x < S) q[(size_t)bh * S + threadIdx.x] = mine * (1.0f / stat[1]);
        return;
    }
    if (threadIdx.x < S) rec[2 + threadIdx.x] = mine;
    if (threadIdx.x == 0) {
        rec[0] = stat[0];
        rec[1] = stat[1];
    }
}

// ---- prefill: tiled attention on the fp16 matrix cores, fp32 values carried as two halves -------
// Many query tokens share the K and V rows they look at, so the split kernel above (one workgroup
// per query and chunk) re-reads the cache qL times.  Here a workgroup owns 128 queries of one head
// and walks the cache in tiles of 32 rows that are staged once in LDS.  It has two sets of 4 waves
// (32 queries per wave, ONE QUERY PER LANE PAIR): both sets hold the same queries, set 0 takes the even
// tiles and set 1 the odd ones, each with its own online softmax, and the two results are merged through
// LDS at the end.  (A tile's chain -- stage, products, softmax, products -- is a sequence of latencies
// that one wave per SIMD cannot hide, and under the causal mask the last query tile of a head has 16
// times the tiles of the first; two sets halve the longest chain.)  Query tiles are dealt out from the
// last to the first, one workgroup per compute unit at a time.
//
// Arithmetic.  On this part v_mfma_f32_32x32x2_f32 runs at the vector ALU's rate and keeps the vector ALU
// busy while it runs (a wave's -- or its SIMD neighbour's -- vector instructions simply add to its time:
// measured), so an fp32-MFMA kernel pays for the softmax, the staging and the products one after the
// other.  The fp16 MFMAs are 16 times faster and leave the vector ALU free.  Every fp32 operand x is
// therefore split into two halves, hi = fp16(x) (rounded toward zero) and lo = fp16(x - hi), whose sum
// carries 22 bits of x, and a product a*b is computed as hi_a*hi_b + hi_a*lo_b + lo_a*hi_b: three
// v_mfma_f32_32x32x16_f16 with fp32 accumulation (each half-by-half product is exact in fp32; the dropped
// lo*lo term is 2^-22 of the product).  Results agree with fp32 arithmetic to about 1e-6 of the largest
// output, like two fp32 evaluations in different summation orders.  Values beyond the fp16 range
// (|x| >= 65504) are not representable this way; activations and cache rows of a transformer are far below.
// An fp16 cache has no low halves: two MFMAs per product.
//
//   S^T = K_tile * Q^T     8 steps of 16 head dims.  A = K[kv = lane%32][16i + 8*hf .. +7]: 16 bytes of the
//                          row's hi plane (and of its lo plane) in LDS.  B = the lane's own query row, same
//                          dims, split once into 64 registers.  The result puts query lane%32 into the
//                          lane, 16 cache rows 8j + 4*hf + v each.  hi*hi goes to one accumulator, the cross
//                          terms to another.
//   mask, online softmax   per lane, fp32, plus one exchange with lane^32 (the other 16 rows of the tile)
//   O^T += V_tile^T * P^T  2 steps of 16 cache rows x 4 blocks of 32 output columns.  B = the lane's 8
//                          probabilities 8b .. 8b+7 exactly as they sit in registers (rows 8j + 4*hf + v,
//                          j = 2b, 2b+1), split into halves.  A = V[those 8 rows][column 32c + lane%32]:
//                          the tile is staged transposed, with the rows of a column permuted so that these
//                          8 halves are 16 contiguous bytes.
//
// Everything a lane holds (running max, sum, 4 x 16 output values) belongs to its own query, so
// the rescaling needs no cross-lane traffic, and no probability ever goes through LDS.  Tiles that
// no query of a wave may see (in-chunk causal mask, ops/op_attn.hpp:1007-1011) are skipped.  K rows
// take 272 bytes per plane and V columns 80, so that the 16 lanes one phase of a 16-byte read serves
// touch 16 different 16-byte slots of the 256-byte bank line (17 and 5 are odd).
//
// Bound: the products are 3072 cycles of a pass (two tiles) on each SIMD, a pass takes 5400; the vector instructions of its two waves
// (330 each, most of them the halves of K, V and P and the exponentials) do not overlap them all.  Beside the passes a workgroup spent 23000
// cycles (10 us) on fetching its queries and on the merge, both by lanes that each followed a row of their own, 16 KB apart; through LDS, rows
// of 512 bytes on either side, these are 14000, most of it the memory's latency and the masked tiles.  One set now stages its next tile before
// its products and the other behind them, so that one's vector work meets the other's products (5500 / 5300 cycles a pass).  (whole call, us,
// before / with all of these, 32 heads: 128 tokens 23.0 / 19.8, 512 48.6 / 41.3, 2048 174 / 159, halves 143 / 127; 512 behind 1500 105 / 79 with
// the merge by rows.)
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef _Float16 v2h __attribute__((ext_vector_type(2)));

// (a, b) -> packed halves hi and lo with a = hi.x + lo.x, b = hi.y + lo.y to 22 bits
__device__ __forceinline__ void split2(float a, float b, uint32_t& hi, uint32_t& lo) {
    const v2h h = __builtin_bit_cast(v2h, __builtin_amdgcn_cvt_pkrtz(a, b));
    hi = __builtin_bit_cast(uint32_t, h);
    float la, lb;  // a - h.x, b - h.y: one instruction each (the compiler converts, then subtracts)
    asm("v_fma_mix_f32 %0, -%1, 1.0, %2 op_sel_hi:[1,0,0]" : "=v"(la) : "v"(hi), "v"(a));
    asm("v_fma_mix_f32 %0, -%1, 1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(lb) : "v"(hi), "v"(b));
    lo = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(la, lb));
}
__device__ __forceinline__ uint32_t pack_hi(float a, float b) {
    return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(a, b));
}
union V8hBits {
    v8h h;
    uint32_t u[4];
    uint4 q;
};

// 4 and 2 elements of a cache row, asked for through a descriptor
template <typename T>
__device__ __forceinline__ float4 buffer_load4(buffer_rsrc rs, uint32_t at) {
    if constexpr (sizeof(T) == 4) {
        return __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(rs, at, 0, 0));
    } else {
        const uint2 u = __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(rs, at, 0, 0));
        const float2 a = __half22float2(__builtin_bit_cast(__half2, u.x)), b = __half22float2(__builtin_bit_cast(__half2, u.y));
        return make_float4(a.x, a.y, b.x, b.y);
    }
}
template <typename T>
__device__ __forceinline__ float2 buffer_load2(buffer_rsrc rs, uint32_t at) {
    if constexpr (sizeof(T) == 4) return __builtin_bit_cast(float2, __builtin_amdgcn_raw_buffer_load_b64(rs, at, 0, 0));
    else return __half22float2(__builtin_bit_cast(__half2, (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rs, at, 0, 0)));
}

// One tile in LDS (fp16 planes, the tile's tokens); each wave set has two of them; the merge at the end reuses the memory
template <bool LO>
struct PrefillSmem {
    static constexpr int S = 128, BK = 32, KSB = 272, VSB = 80;
    uint8_t k_hi[BK * KSB];
    uint8_t k_lo[LO ? BK * KSB : 16];
    uint8_t v_hi[S * VSB];
    uint8_t v_lo[LO ? S * VSB : 16];
    int tok[BK];
};
constexpr int kPrefillRow = 528;                      // bytes of a row of 128 floats in LDS: 33 16-byte slots
constexpr size_t kPrefillRowsBytes = 128 * kPrefillRow;
// The queries on their way to the registers: beside fp32 rows half of them in each set's second tile buffer (filled behind the first
// pass's barrier), beside halves behind the buffers.  The merge at the end: both sets' outputs, then (max, sum) of each and the weights.
constexpr size_t kPrefillMergeBytes = 2 * kPrefillRowsBytes + 3 * 128 * sizeof(float2);
template <bool LO>
constexpr size_t prefill_smem_bytes() {
    const size_t walk = 4 * sizeof(PrefillSmem<LO>) + (LO ? 0 : kPrefillRowsBytes);
    return walk > kPrefillMergeBytes ? walk : kPrefillMergeBytes;
}
static_assert(sizeof(PrefillSmem<true>) >= kPrefillRowsBytes / 2 && prefill_smem_bytes<true>() <= 160 * 1024 && prefill_smem_bytes<false>() <= 160 * 1024, "");

template <typename T>
__global__ __launch_bounds__(512) void attn_prefill_kernel(float* q, const T* __restrict__ kc, const T* __restrict__ vc,
                                                          int64_t qL, int64_t H, int64_t maxlen, int64_t kvLen,
                                                          const int32_t* __restrict__ row_token, const int2* __restrict__ tile_tokens, int qtiles, int kv_span,
                                                          float* __restrict__ part, int nsplit, const float* __restrict__ turns) {
    constexpr bool LO = sizeof(T) == 4;  // an fp16 cache holds no low halves
    constexpr int S = 128, BQ = 128, BK = 32, KSB = 272, VSB = 80;
    extern __shared__ __align__(16) uint8_t smem_raw[];
    const int lane = threadIdx.x & 63, wave8 = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int set = wave8 >> 2, wave = wave8 & 3;  // (wave: within the set)
    // two tile buffers per set, used alternately: while a tile is multiplied the next one is written
    PrefillSmem<LO>* const sm2 = reinterpret_cast<PrefillSmem<LO>*>(smem_raw) + 2 * set;
    const int hf = lane >> 5, c32 = lane & 31;
    // late query tiles see the most cache rows: they are dealt out first so that they do not form the tail
    // (gridDim.y = nsplit workgroups share a query tile, each with kv_span cache rows; one: kv_span covers them all)
    const unsigned bhs = gridDim.x / (unsigned)qtiles, turn = __builtin_amdgcn_readfirstlane(blockIdx.x / bhs);
    const int qt = qtiles - 1 - (int)turn;
    const int64_t bh = blockIdx.x - turn * bhs, b = bh / H, h = bh % H;
    const int kv_begin = (int)blockIdx.y * kv_span;
    // (32-bit arithmetic from here on: the launcher keeps qL and kvLen below 2^31 and a head's cache plane below 4 GiB)
    const int qLi = (int)qL, kvLeni = (int)kvLen;
    const int q_lo_wave = qt * BQ + wave * 32;
    const int pq = q_lo_wave + c32;  // this lane's query token
    const bool valid = pq < qLi;
    const int q_hi_wave = min(q_lo_wave + 31, qLi - 1);
    float* const q0 = q + ((b * qL + qt * BQ) * H + h) * S;  // the first query's row, H * S floats to the next
    const int q_rows = min(BQ, qLi - qt * BQ);
    const T* kbase = kc + bh * maxlen * S;
    const T* vbase = vc + bh * maxlen * S;

    const float d_scale = 1.0f / sqrtf((float)S);
    float m_run = -FLT_MAX, l_run = 0.0f;
    v16f o[4];
#pragma unroll
    for (int c = 0; c < 4; c++)
#pragma unroll
        for (int r = 0; r < 16; r++) o[c][r] = 0.0f;

    // Staging.  K: a wave moves two whole rows at a time, 16 bytes (8 of halves) to a lane.  V is written transposed,
    // cache row r of the tile at position 16*(r/16) + 8*((r/4)%2) + 4*((r%16)/8) + r%4 of its column: a thread
    // moves the 8 rows that share an aligned run of 8 positions (rows 16b + 4h + w and 16b + 8 + 4h + w, w = 0..3;
    // (b, h) = the thread's wave) of two neighbouring columns, so that a column's share is one 16-byte store.
    // (Four rows of four columns per thread meant 8-byte stores 320 bytes apart: eight lanes on every bank.)
    // The next tile's global loads are issued before the current tile is computed on and land in registers
    // meanwhile.
    const int krow = 2 * wave + hf, kseg = c32;  // rows krow + 8u
    const int vb = wave >> 1, vh = wave & 1, vcp = lane;  // rows 16*vb + 8*(e/4) + 4*vh + e%4, columns 2*vcp, 2*vcp+1
    float4 kst[4];
    float2 vst[8];
    int tst = INT_MAX;
    const uint32_t kv_row = S * sizeof(T), k_at = (uint32_t)krow * kv_row + (uint32_t)kseg * 4 * sizeof(T),
                   v_at = (uint32_t)(16 * vb + 4 * vh) * kv_row + (uint32_t)vcp * 2 * sizeof(T);
    // (rows from kvLen on read as zero: the loads go through a descriptor that ends there)
#define LLMOPS_STAGE_LOAD(KV0)                                                                          \
    do {                                                                                                \
        const uint32_t bytes_ = (uint32_t)__builtin_amdgcn_readfirstlane(max(0, min(BK, kvLeni - (KV0)))) * kv_row; \
        const buffer_rsrc rk_ = make_rsrc(kbase + (int64_t)(KV0) * S, bytes_), rv_ = make_rsrc(vbase + (int64_t)(KV0) * S, bytes_); \
        _Pragma("unroll") for (int u = 0; u < 4; u++) kst[u] = buffer_load4<T>(rk_, k_at + 8 * u * kv_row); \
        _Pragma("unroll") for (int e = 0; e < 8; e++) vst[e] = buffer_load2<T>(rv_, v_at + (8 * (e >> 2) + (e & 3)) * kv_row); \
        if (wave == 0) tst = row_token[(KV0) + c32]; /* (the table ends on a multiple of 64 rows) */    \
    } while (0)
    // Writing a staged tile: halves of K row-major, halves of V transposed, the tile's tokens and their range.
#define LLMOPS_STAGE_STORE(SM)                                                                                  \
    do {                                                                                                        \
        _Pragma("unroll") for (int u = 0; u < 4; u++) {                                                         \
            uint2 hi_, lo_;                                                                                     \
            split2(kst[u].x, kst[u].y, hi_.x, lo_.x);                                                           \
            split2(kst[u].z, kst[u].w, hi_.y, lo_.y);                                                           \
            const int at_ = (krow + 8 * u) * KSB + kseg * 8;                                                    \
            *reinterpret_cast<uint2*>(&(SM).k_hi[at_]) = hi_;                                                   \
            if (LO) *reinterpret_cast<uint2*>(&(SM).k_lo[at_]) = lo_;                                           \
        }                                                                                                       \
        {                                                                                                       \
            uint32_t h_[2][4], l_[2][4]; /* [column][pair of rows] */                                           \
            _Pragma("unroll") for (int e2 = 0; e2 < 4; e2++) {                                                  \
                split2(vst[2 * e2].x, vst[2 * e2 + 1].x, h_[0][e2], l_[0][e2]);                                 \
                split2(vst[2 * e2].y, vst[2 * e2 + 1].y, h_[1][e2], l_[1][e2]);                                 \
            }                                                                                                   \
            _Pragma("unroll") for (int j = 0; j < 2; j++) {                                                     \
                const int at_ = (2 * vcp + j) * VSB + (16 * vb + 8 * vh) * 2;                                   \
                *reinterpret_cast<uint4*>(&(SM).v_hi[at_]) = make_uint4(h_[j][0], h_[j][1], h_[j][2], h_[j][3]); \
                if (LO) *reinterpret_cast<uint4*>(&(SM).v_lo[at_]) = make_uint4(l_[j][0], l_[j][1], l_[j][2], l_[j][3]); \
            }                                                                                                   \
        }                                                                                                       \
        if (wave == 0 && lane < BK) (SM).tok[lane] = tst;                                                       \
    } while (0)
    // Set 0 walks the tiles 0, 2, 4, ..., set 1 the tiles 1, 3, 5, ...: both make the same number of passes.  One
    // barrier per pass: behind it the pass's buffer is complete and nobody reads the other buffer any more, which
    // the pass then fills -- set 0 after its own products, set 1 before them -- from the registers that the loads of the pass before filled.
    LLMOPS_STAGE_LOAD(kv_begin + set * BK);
    // The queries, a row by sixteen lanes that hold the two halves of its rotary pairs, through LDS into the lane's share of its own
    // row as halves (step i covers dims 16i + 8*hf .. +7).  (Each lane fetching from its own row, 64 rows apart in one load: 4 us.)
    uint8_t* const q_lds = LO ? smem_raw + sizeof(PrefillSmem<LO>) : smem_raw + 4 * sizeof(PrefillSmem<LO>);
    constexpr int kQHalf = LO ? 2 * (int)sizeof(PrefillSmem<LO>) : 64 * kPrefillRow;  // rows 64 .. from here on
    {
        const int qrow = threadIdx.x >> 4, qcol = 4 * (threadIdx.x & 15);  // rows qrow + 32u, columns qcol .. and 64 + qcol ..
        float4 t[8];
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const float* at = q0 + min(qrow + 32 * u, q_rows - 1) * (H * S) + qcol;
            t[2 * u] = load4(at), t[2 * u + 1] = load4(at + 64);
        }
        if (turns != nullptr) {  // (q as the caller left it: see attn_prep_rows_kernel)
            const float* const turns0 = turns + (int64_t)qt * (BQ * S) + qcol;
            float4 c[4], s[4];
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const float* at = turns0 + min(qrow + 32 * u, q_rows - 1) * S;
                c[u] = load4(at), s[u] = load4(at + 64);
            }
#pragma unroll
            for (int u = 0; u < 4; u++) rotate4(t[2 * u], t[2 * u + 1], c[u], s[u]);
        }
#pragma unroll
        for (int u = 0; u < 4; u++) {
            uint8_t* at = q_lds + (u >> 1) * kQHalf + (qrow + 32 * (u & 1)) * kPrefillRow + 4 * qcol;
            *reinterpret_cast<float4*>(at) = t[2 * u];
            *reinterpret_cast<float4*>(at + 256) = t[2 * u + 1];
        }
    }
    // The last cache tile that any query of the workgroup may see bounds the walk (rows of later tokens and rows
    // beyond it are masked anyway; without the bound an early query tile would stage, barrier by barrier, all the
    // tiles that only later tiles need).
    int kv_end = kv_begin;
    {
        const int q_hi_wg = min((qt + 1) * BQ, qLi) - 1, first = kv_begin / BK, last = (min(kvLeni, kv_begin + kv_span) + BK - 1) / BK;
        for (int t0 = (last - first - 1) / 64 * 64 + first; t0 >= first; t0 -= 64) {
            const unsigned long long seen = __ballot(t0 + lane < last && tile_tokens[min(t0 + lane, last - 1)].x <= q_hi_wg);
            if (seen != 0) {
                kv_end = (t0 + 64 - __builtin_clzll(seen)) * BK;
                break;
            }
        }
    }
    const int2* const ranges = tile_tokens + kv_begin / BK + set;
    int2 range = ranges[0], range_next = range;  // smallest and largest token of the set's tile
    LLMOPS_STAGE_STORE(sm2[0]);
    __syncthreads();
    V8hBits qh[8], ql[8];
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const float4* at = reinterpret_cast<const float4*>(q_lds + (wave >> 1) * kQHalf + (32 * (wave & 1) + c32) * kPrefillRow + 64 * i + 32 * hf);
        const float4 t0 = at[0], t1 = at[1];
        split2(t0.x, t0.y, qh[i].u[0], ql[i].u[0]);
        split2(t0.z, t0.w, qh[i].u[1], ql[i].u[1]);
        split2(t1.x, t1.y, qh[i].u[2], ql[i].u[2]);
        split2(t1.z, t1.w, qh[i].u[3], ql[i].u[3]);
    }
    if (kv_begin + 2 * BK < kv_end) {
        LLMOPS_STAGE_LOAD(kv_begin + set * BK + 2 * BK);
        range_next = ranges[2];
    }
    for (int kv_pair = kv_begin, pass = 0; kv_pair < kv_end; kv_pair += 2 * BK, pass++) {
        PrefillSmem<LO>& sm = sm2[pass & 1];
        const uint8_t* kp_hi = &sm.k_hi[c32 * KSB + 16 * hf];  // + 32 i
        const uint8_t* kp_lo = &sm.k_lo[LO ? c32 * KSB + 16 * hf : 0];
        const uint8_t* vp_hi = &sm.v_hi[c32 * VSB + 16 * hf];  // + 32 c * VSB + 32 b
        const uint8_t* vp_lo = &sm.v_lo[LO ? c32 * VSB + 16 * hf : 0];
        const int* tok = sm.tok;
        __syncthreads();
        // skip the tile if even the wave's last query may not see any of its rows; a tile that every query of the
        // wave sees whole (the usual case away from the diagonal) needs no masks
        const int tmin = range.x, tmax = range.y;
        if (set == 1 && kv_pair + 2 * BK < kv_end) {
            LLMOPS_STAGE_STORE(sm2[(pass + 1) & 1]);
            range = range_next;
            if (kv_pair + 4 * BK < kv_end) {
                LLMOPS_STAGE_LOAD(kv_pair + set * BK + 4 * BK);
                range_next = ranges[(kv_pair - kv_begin) / BK + 4];
            }
        }
        if (q_lo_wave < qLi && tmin <= q_hi_wave) {
        const bool all_visible = tmax <= q_lo_wave && q_lo_wave + 31 < qLi;

        v16f s0, s1;
#pragma unroll
        for (int r = 0; r < 16; r++) s0[r] = 0.0f, s1[r] = 0.0f;
        {
            // operand reads run two steps ahead of the MFMAs that use them
            v8h ah[3], al[3];
            ah[0] = *reinterpret_cast<const v8h*>(kp_hi);
            ah[1] = *reinterpret_cast<const v8h*>(kp_hi + 32);
            if (LO) {
                al[0] = *reinterpret_cast<const v8h*>(kp_lo);
                al[1] = *reinterpret_cast<const v8h*>(kp_lo + 32);
            }
#pragma unroll
            for (int i = 0; i < 8; i++) {
                if (i + 2 < 8) {
                    ah[(i + 2) % 3] = *reinterpret_cast<const v8h*>(kp_hi + 32 * (i + 2));
                    if (LO) al[(i + 2) % 3] = *reinterpret_cast<const v8h*>(kp_lo + 32 * (i + 2));
                }
                __builtin_amdgcn_sched_barrier(0);
                s0 = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah[i % 3], qh[i].h, s0, 0, 0, 0);
                s1 = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah[i % 3], ql[i].h, s1, 0, 0, 0);
                if (LO) s1 = __builtin_amdgcn_mfma_f32_32x32x16_f16(al[i % 3], qh[i].h, s1, 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        v16f sacc = s0 + s1;

        // scale, mask (rows written by later tokens of this call, rows beyond kvLen), running max
        float mx = -FLT_MAX;
        if (all_visible) {  // (the same for the whole wave)
#pragma unroll
            for (int r = 0; r < 16; r++) {
                sacc[r] *= d_scale;
                mx = fmaxf(mx, sacc[r]);
            }
        } else {
            const int pq32 = valid ? pq : INT_MIN;
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int4 t4 = *reinterpret_cast<const int4*>(&tok[8 * j + 4 * hf]);
                const int tt[4] = {t4.x, t4.y, t4.z, t4.w};
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    const float sv = (tt[v] <= pq32) ? sacc[4 * j + v] * d_scale : -FLT_MAX;
                    sacc[4 * j + v] = sv;
                    mx = fmaxf(mx, sv);
                }
            }
        }
        {  // the other half of the lane pair (lane ^ 32) holds the other 16 rows of the query's tile
            const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(mx), __float_as_uint(mx), false, false);
            mx = fmaxf(__uint_as_float(sw[0]), __uint_as_float(sw[1]));
        }
        const float m_new = fmaxf(m_run, mx);
        const float alpha = expf(m_run - m_new);  // 0 on the first visible tile, 1 while nothing is visible
        float psum = 0.0f;
        if (all_visible) {
#pragma unroll
        for (int r = 0; r < 16; r++) {
            // e^x as 2^(x * log2 e) on the exponential unit: x <= 0, and wherever the result matters (|x| < 20)
            // the product's rounding moves it by less than 1e-6 of itself
            const float pv = __builtin_amdgcn_exp2f((sacc[r] - m_new) * 1.44269504088896341f);
            sacc[r] = pv;
            psum += pv;
        }
        } else {
#pragma unroll
        for (int r = 0; r < 16; r++) {
            // e^x as 2^(x * log2 e) on the exponential unit: x <= 0, and wherever the result matters (|x| < 20)
            // the product's rounding moves it by less than 1e-6 of itself
            const float pv = (sacc[r] == -FLT_MAX) ? 0.0f : __builtin_amdgcn_exp2f((sacc[r] - m_new) * 1.44269504088896341f);
            sacc[r] = pv;
            psum += pv;
        }
        }
        {
            const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(psum), __float_as_uint(psum), false, false);
            psum = __uint_as_float(sw[0]) + __uint_as_float(sw[1]);
        }
        l_run = l_run * alpha + psum;
        if (__any(m_new != m_run)) {  // (alpha is exactly 1 for a query whose maximum did not move)
#pragma unroll
            for (int c = 0; c < 4; c++)
#pragma unroll
                for (int r = 0; r < 16; r++) o[c][r] *= alpha;
        }
        m_run = m_new;

        // O^T += V^T P^T: step b takes the lane's probabilities 8b .. 8b+7 (cache rows 8j + 4*hf + v, j = 2b, 2b+1)
#pragma unroll
        for (int bb = 0; bb < 2; bb++) {
            V8hBits ph, pl;
#pragma unroll
            for (int e = 0; e < 4; e++) split2(sacc[8 * bb + 2 * e], sacc[8 * bb + 2 * e + 1], ph.u[e], pl.u[e]);
            v8h ah[4], al[4];
#pragma unroll
            for (int c = 0; c < 4; c++) {
                ah[c] = *reinterpret_cast<const v8h*>(vp_hi + 32 * c * VSB + 32 * bb);
                if (LO) al[c] = *reinterpret_cast<const v8h*>(vp_lo + 32 * c * VSB + 32 * bb);
            }
#pragma unroll
            for (int c = 0; c < 4; c++) o[c] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah[c], ph.h, o[c], 0, 0, 0);
#pragma unroll
            for (int c = 0; c < 4; c++) o[c] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah[c], pl.h, o[c], 0, 0, 0);
            if (LO) {
#pragma unroll
                for (int c = 0; c < 4; c++) o[c] = __builtin_amdgcn_mfma_f32_32x32x16_f16(al[c], ph.h, o[c], 0, 0, 0);
            }
        }
        }  // (tile visible to the wave)
        if (set == 0 && kv_pair + 2 * BK < kv_end) {
            LLMOPS_STAGE_STORE(sm2[(pass + 1) & 1]);
            range = range_next;
            if (kv_pair + 4 * BK < kv_end) {
                LLMOPS_STAGE_LOAD(kv_pair + set * BK + 4 * BK);
                range_next = ranges[(kv_pair - kv_begin) / BK + 4];
            }
        }
    }

#undef LLMOPS_STAGE_STORE
#undef LLMOPS_STAGE_LOAD
    // Merge of the two sets, through LDS: every lane leaves what it holds of its query's output, then half a wave takes a row of
    // both sets, so that the rows leave as whole lines.  (From the lanes that hold them, 32 rows apart in one store: 4.4 us.)
    __syncthreads();  // every wave is done with its tile
    // (the lane's number anew: no register held it through the walk)
    const int ln = (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)), lq = ln & 31, lh = ln >> 5;
    uint8_t* const o_lds = smem_raw;
    float2* const stats = reinterpret_cast<float2*>(smem_raw + 2 * kPrefillRowsBytes);  // [set][query] (max, sum), then [query] weights
    {
        uint8_t* const at = o_lds + set * kPrefillRowsBytes + (wave * 32 + lq) * kPrefillRow + 16 * lh;
        // (the lane holds columns 32c + 8j + 4*hf + v of its query's output row)
#pragma unroll
        for (int c = 0; c < 4; c++)
#pragma unroll
            for (int j = 0; j < 4; j++)
                *reinterpret_cast<float4*>(at + 128 * c + 32 * j) = make_float4(o[c][4 * j], o[c][4 * j + 1], o[c][4 * j + 2], o[c][4 * j + 3]);
        if (lh == 0) stats[set * 128 + wave * 32 + lq] = make_float2(m_run, l_run);
    }
    __syncthreads();
    if (wave8 < 2) {
        const int at = wave8 * 64 + ln;
        const float2 s0 = stats[at], s1 = stats[128 + at];
        const float mm = fmaxf(s0.x, s1.x);
        const float a0 = expf(s0.x - mm), a1 = expf(s1.x - mm);  // (a set that saw no row has sum 0 and outputs 0)
        stats[256 + at] = make_float2(a0, a1);
        const float l = s0.y * a0 + s1.y * a1;
        stats[at] = make_float2(mm, nsplit > 1 ? l : 1.0f / l);
    }
    __syncthreads();
    float4 z[8];
    float2 st[8];
#pragma unroll
    for (int u = 0; u < 8; u++) {
        const int row = 2 * wave8 + lh + 16 * u;
        const float2 a = stats[256 + row];
        const float4 x = *reinterpret_cast<const float4*>(o_lds + row * kPrefillRow + 16 * lq);
        const float4 y = *reinterpret_cast<const float4*>(o_lds + kPrefillRowsBytes + row * kPrefillRow + 16 * lq);
        st[u] = stats[row];
        z[u] = make_float4(x.x * a.x + y.x * a.y, x.y * a.x + y.y * a.y, x.z * a.x + y.z * a.y, x.w * a.x + y.w * a.y);
    }
    if (nsplit > 1) {  // records [max, sum, out[S]] for attn_merge_kernel
        float* const rec = part + ((bh * qL + qt * BQ) * nsplit + blockIdx.y) * (S + 2);
#pragma unroll
        for (int u = 0; u < 8; u++) {
            const int row = 2 * wave8 + lh + 16 * u;
            if (row >= q_rows) break;
            float* const at = rec + (int64_t)row * nsplit * (S + 2);
            if (lq == 0) *reinterpret_cast<float2*>(at) = st[u];
            float2* dst = reinterpret_cast<float2*>(at + 2 + 4 * lq);
            dst[0] = make_float2(z[u].x, z[u].y);
            dst[1] = make_float2(z[u].z, z[u].w);
        }
        return;
    }
#pragma unroll
    for (int u = 0; u < 8; u++) {
        const int row = 2 * wave8 + lh + 16 * u;
        if (row >= q_rows) break;
        *reinterpret_cast<float4*>(q0 + row * (H * S) + 4 * lq) = make_float4(z[u].x * st[u].y, z[u].y * st[u].y, z[u].z * st[u].y, z[u].w * st[u].y);
    }
}

// ---- softmax op (ops/op_misc.hpp:183-194): one workgroup per row ------------------------------
__global__ __launch_bounds__(256) void softmax_kernel(float* __restrict__ x, int64_t K) {
    __shared__ float red[4];
    float* row = x + (int64_t)blockIdx.x * K;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    float mx = -FLT_MAX;
    for (int64_t i = threadIdx.x; i < K; i += 256) mx = fmaxf(mx, row[i]);
    mx = wave_max(mx);
    if (lane == 0) red[wave] = mx;
    __syncthreads();
    mx = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    __syncthreads();
    float sum = 0.0f;
    for (int64_t i = threadIdx.x; i < K; i += 256) {
        const float ex = expf(row[i] - mx);
        row[i] = ex;
        sum += ex;
    }
    sum = wave_sum(sum);
    if (lane == 0) red[wave] = sum;
    __syncthreads();
    const float scale = 1.0f / (((red[0] + red[1]) + red[2]) + red[3]);
    for (int64_t i = threadIdx.x; i < K; i += 256) row[i] *= scale;
}

static inline size_t align_up(size_t v, size_t a) { return (v + a - 1) / a * a; }

static int g_prefill_min_tokens = 32;  // query tokens per call from which the tiled MFMA kernel is used

static int pick_pw(int64_t bhq, int64_t kvLen) {
    // smallest chunk count that still gives ~1024 workgroups; chunk = 4*PW rows
    for (int pw : {16, 8, 4}) {
        const int64_t chunks = (kvLen + 4 * pw - 1) / (4 * pw);
        if (bhq * chunks >= 1024 || pw == 4) return pw;
    }
    return 4;
}

// Calls that the decode kernel does not take: which kernel, and how many cache rows a workgroup of it has.
struct TokensPlan {
    int kernel;  // 1 attn_split_kernel (a workgroup per query and chunk), 2 attn_few_kernel (all tokens of a head), 3 attn_prefill_kernel
    int pw;      // split kernel: cache rows per wavefront
    int rows;    // cache rows per workgroup
    int pieces;  // workgroups that share a query's cache rows
};
static TokensPlan plan_tokens(int64_t bh, int64_t qL, int64_t kvLen, bool half_cache, int64_t max_records) {
    const int64_t bhq = bh * qL;
    TokensPlan p{};
    if (qL >= g_prefill_min_tokens) {
        // A workgroup takes a compute unit: with fewer query tiles than those, ns workgroups share a tile's cache rows, at
        // least 128 each.  A row costs a tile 0.0365 us (halves 0.0305: two products instead of three); the launch that merges the
        // records costs 2.6 us and 0.15 us per 1000 records, beside either cache.  Against every number of pieces at 710 sizes of each
        // cache (8 to 256 heads in all, 32 to 2048 tokens behind 0 to 3500): 0.03 % slower than the best on average and 3 % at worst, beside
        // halves 0.13 % and 8 %.  (us with the copy that puts q and k back, one piece / several, 32 heads: 32 tokens behind 100 19.3 / 19.6, behind
        // 500 34.7 / 21.4; 128 behind 200 30.7 / 27.2, behind 2500 114 / 41; 256 behind none 30.45 / 30.5, behind 300 42.7 / 33.2; 512 behind none
        // 43.4 / 40.8, behind 1500 98 / 75; 8 heads, 2048 tokens 100 / 70.  Halves: 64 behind 100 19.1 / 19.9, 200 behind 300 34.7 / 28.6; 256 behind
        // none 26.9 / 28.6, behind 300 37.9 / 31.4; 512 behind 300 50.8 / 45.3; 16 heads, 512 behind 100 39.7 / 32.1.)
        p.kernel = 3;
        const double row = half_cache ? 0.0305 : 0.0365, record = 0.15e-3;
        int64_t ns = 256 / (bh * ((qL + 127) / 128));
        if (ns > (kvLen + 127) / 128) ns = (kvLen + 127) / 128;
        if (ns < 2 || bhq * ns > max_records || row * (double)(kvLen - kvLen / ns) < 2.6 + record * (double)(bhq * ns)) ns = 1;
        p.rows = (int)(((kvLen + ns - 1) / ns + 63) / 64 * 64);
        p.pieces = (int)((kvLen + p.rows - 1) / p.rows);
        return p;
    }
    // One workgroup per query and chunk while there is little to read and multiply again for every token: a wave of
    // attn_few_kernel runs some 2500 instructions however few of its 32 columns and 128 rows are in use.  Estimates in us, up
    // to what both have in common; per query: rounds of the 1024 workgroups with chunks of 64 rows that the chip holds, rows
    // multiplied, rows read, queries, chunks beyond the merge's 64 lanes; together: workgroups, up to one and up to two on
    // a compute unit and more.  Measured with both kernels at 2620 sizes (1 to 31 tokens, 4 to 4096 heads in all, 1 to 8192
    // cache rows of both types, in memory and not in a cache): the choice is 0.08 % slower than the better one on average,
    // 13 % at worst.  (us, per query / together, fp32: 32 heads, 2 tokens behind 1000 17.4 / 18.3, behind 4000 35.9 / 36.8;
    // 4 behind 500 15.0 / 17.2, behind 1000 21.0 / 18.6; 8 behind 120 11.7 / 16.0, behind 250 15.0 / 16.5; 31 behind 33
    // 15.3 / 18.2, behind 97 19.9 / 18.9; 512 heads, 4 tokens, 32 rows 23.7 / 22.1; 4096 heads, 1 token, 48 rows 53 / 87,
    // fp16 37 / 73; 4 heads, 1 token, 8192 rows 41 / 20.)
    p.pw = pick_pw(bhq, kvLen);
    const int64_t chunk = 4 * p.pw, chunks = (kvLen + chunk - 1) / chunk, few_chunks = (kvLen + 127) / 128, wgs = bh * few_chunks;
    struct Cost {
        double round, query_row, row, query, chunk, few, few_two, few_wg, few_wg_more;
    };
    const Cost c = half_cache ? Cost{0.273, 16.6e-6, 14.1e-6, 0.844e-3, 0.0568, 2.01, 1.9, 0.0, 7.56e-3}
                              : Cost{0.5, 7.84e-6, 38.8e-6, 1.225e-3, 0.0347, 2.025, 2.0, 1.71e-3, 5.09e-3};
    const double per_query = c.round * (double)(chunk == 64 ? (bhq * chunks + 1023) / 1024 : 0) + c.query_row * (double)(bhq * kvLen) +
                             c.row * (double)(bh * kvLen) + c.query * (double)bhq + c.chunk * (double)(chunks > 64 ? chunks - 64 : 0);
    const double together = c.few + (wgs > 256 ? c.few_two : 0.0) + c.few_wg * (double)wgs + c.few_wg_more * (double)(wgs > 512 ? wgs - 512 : 0);
    p.kernel = per_query < together ? 1 : 2;
    p.rows = p.kernel == 1 ? (int)chunk : 128;
    p.pieces = (int)(p.kernel == 1 ? chunks : few_chunks);
    return p;
}

// cache rows per chunk when the chunk records go to the consumer FC (at most kAttnRecChunks chunks per head): 0 = the
// cache is too long for that
static int records_chunk_rows(int64_t maxlen, bool half_cache) {
    if (maxlen <= kAttnRecChunks * 256) return 256;
    if (half_cache && maxlen <= kAttnRecChunks * 512) return 512;
    return 0;
}

// Decode (one query token): cache rows per wavefront (a chunk is 4 times that).  g_decode_pw forces it (tests,
// measurements); 0 = choose.
static int g_decode_pw = 0;
struct DecodePlan {
    int pw;
};
static DecodePlan plan_decode(int64_t bh, int64_t kv, bool half_cache, int64_t max_records) {
    // fp32 rows are 32 lanes wide (2 rows per wave-wide load), fp16 rows 16 lanes (4 rows): 2..8 loads per lane
    const int lo = half_cache ? 8 : 4, hi = half_cache ? 32 : 16;
    auto chunks = [&](int pw) { return (kv + 4 * pw - 1) / (4 * pw); };
    // Chunks of 4 wavefronts, merged by a second launch: the largest chunk that still gives 256
    // workgroups, and 512 for the two larger chunk sizes (measured, us, fp32: kv 256 -- 16/32/64-row chunks 8.6 / 8.2 /
    // 9.3; kv 512 -- 11.1 / 10.1 / 10.3; kv 1024 -- 15.1 / 13.3 / 13.1; kv 2048 -- 30.7 / 19.7 / 19.0)
    DecodePlan p{lo};
    for (int pw = hi; pw >= lo; pw >>= 1)
        if (bh * chunks(pw) >= (pw > 2 * lo ? 512 : 256)) {
            p.pw = pw;
            break;
        }
    if (g_decode_pw >= lo && g_decode_pw <= hi && (g_decode_pw & (g_decode_pw - 1)) == 0) p.pw = g_decode_pw;
    while (p.pw < hi && bh * chunks(p.pw) > max_records) p.pw <<= 1;  // the records must fit the workspace
    return p;
}

}  // namespace llmops

using namespace llmops;

extern "C" int llmops_rope_embed(float* x, int64_t B, int64_t H, int64_t L, int64_t S, const float* inv_freq,
                                 int64_t half, int position_id, llmops_stream_t stream) {
    LLMOPS_REQUIRE(x != nullptr && inv_freq != nullptr);
    LLMOPS_REQUIRE(B > 0 && H > 0 && L > 0 && S > 0 && half > 0 && 2 * half <= S);
    const int64_t total = B * H * L * half;
    rope_kernel<<<(unsigned)((total + 255) / 256), 256, 0, as_stream(stream)>>>(x, B * H, L, S, inv_freq, half, position_id);
    LLMOPS_LAUNCH_CHECK();
    return LLMOPS_OK;
}

extern "C" size_t llmops_attention_workspace_bytes(int64_t B, int64_t qL, int64_t H, int64_t S, int64_t maxlen) {
    if (B <= 0 || qL <= 0 || H <= 0 || S <= 0 || maxlen <= 0) return 0;
    // the planners use 64-row chunks (128 with an fp16 cache) unless that gives fewer than 1024 workgroups, and the
    // finer chunkings they then fall back to stay below 2048 workgroups; a plan that does not fit is coarsened
    const int64_t bhq = B * H * qL;
    int64_t records = bhq * ((maxlen + 63) / 64);
    if (records < 2048) records = 2048;
    return LLMOPS_ATTN_COUNTER_BYTES + align_up((size_t)maxlen * sizeof(int32_t), 256) +
           (size_t)records * (S + 2) * sizeof(float);
}

// Merging the records where their number is known here: up to eight by half waves whatever the queries; up to sixteen from 512 queries on
// (attn_merge_kernel asks for 32 records however few there are, but has a workgroup to every query: with 64 queries of 16 records, 2 tokens
// behind 1000, it is 0.3 us the faster one).  us for the whole call in a graph, 32 heads, by attn_merge_kernel / so: 3 tokens 11.5 / 10.4, 31 behind 97
// 20.8 / 19.1, 16 behind 1500 24.9 / 24.9, batches 8 x 31 behind 100 halves 39.8 / 32.8, 8 x 31 behind 400 55.9 / 49.8, 4 x 16 behind 60 20.4 / 17.6,
// 4 x 20 behind 900 45.0 / 43.4; one token behind 100 9.5 / 8.9, of eight sequences behind 100 halves 11.9 / 10.7, behind 500 halves 18.9 / 18.0.
static void merge_records(float* q, const float* part, int64_t bhq, int64_t qL, int64_t H, int records, hipStream_t st) {
    const unsigned groups = (unsigned)((bhq + 7) / 8);
    if (records <= 2) attn_merge_rows_kernel<2><<<groups, 256, 0, st>>>(q, part, (int)qL, (int)H, (unsigned)bhq, records);
    else if (records <= 4) attn_merge_rows_kernel<4><<<groups, 256, 0, st>>>(q, part, (int)qL, (int)H, (unsigned)bhq, records);
    else if (records <= 8) attn_merge_rows_kernel<8><<<groups, 256, 0, st>>>(q, part, (int)qL, (int)H, (unsigned)bhq, records);
    else if (records <= 16 && bhq >= 512) attn_merge_rows_kernel<16><<<groups, 256, 0, st>>>(q, part, (int)qL, (int)H, (unsigned)bhq, records);
    else attn_merge_kernel<<<(unsigned)bhq, 128, 0, st>>>(q, part, qL, H, records);
}

template <typename T>
static int attention_impl(float* q, float* k, const float* v, int64_t B, int64_t qL, int64_t H, int64_t S,
                          const float* inv_freq, int64_t half, T* cache, int64_t maxlen, const int32_t* slots,
                          int position_id, const int32_t* pos_dev, int layer_id, void* workspace, size_t workspace_bytes,
                          hipStream_t st, float* rec_stats = nullptr, float* rec_outs = nullptr) {
    constexpr bool kHalfCache = sizeof(T) == 2;
    T* kc = cache + (int64_t)(2 * layer_id + 0) * B * H * maxlen * S;
    T* vc = cache + (int64_t)(2 * layer_id + 1) * B * H * maxlen * S;
    uint8_t* wsb = reinterpret_cast<uint8_t*>(workspace);
    int32_t* row_token = reinterpret_cast<int32_t*>(wsb + LLMOPS_ATTN_COUNTER_BYTES);
    const size_t part_off = LLMOPS_ATTN_COUNTER_BYTES + align_up((size_t)maxlen * 4, 256);
    float* part = reinterpret_cast<float*>(wsb + part_off);
    const int64_t max_records = (int64_t)((workspace_bytes - part_off) / ((S + 2) * sizeof(float)));
    int64_t kvLen = (int64_t)position_id + qL;
    if (kvLen > maxlen) kvLen = maxlen;
    const int64_t bhq = B * H * qL;
    if (rec_stats != nullptr) {
        // decode with the merge left to the consumer: 16 wavefronts x 16 rows per chunk, or x 32 with an fp16 cache
        // longer than 2048 rows
        const int64_t kv_plan = pos_dev ? maxlen : kvLen;
        const int rows = records_chunk_rows(maxlen, kHalfCache);
        if (qL != 1 || (half % 4) != 0 || rows == 0) return fail(LLMOPS_EINVAL, "chunk records need one query token, half %% 4 == 0 and a cache of at most %d rows", kAttnRecChunks * (kHalfCache ? 512 : 256));
        const int nchunks = (int)((kv_plan + rows - 1) / rows);
        if (bhq > 65535 || maxlen * S * (int64_t)sizeof(T) >= ((int64_t)1 << 32))
            return fail(LLMOPS_EINVAL, "decode attention: at most 65535 heads in all and a cache plane per head below 4 GiB");
        const dim3 grid((unsigned)nchunks, (unsigned)bhq);
        if (rows == 256)
            attn_decode_kernel<T, 16, 16, true><<<grid, 1024, 0, st>>>(pos_dev, position_id, nchunks, (int)maxlen, kc, vc, slots, q, k, v,
                                                                       inv_freq, (int)half, nullptr, rec_stats, rec_outs);
        else if constexpr (kHalfCache)
            attn_decode_kernel<T, 32, 16, true><<<grid, 1024, 0, st>>>(pos_dev, position_id, nchunks, (int)maxlen, kc, vc, slots, q, k, v,
                                                                       inv_freq, (int)half, nullptr, rec_stats, rec_outs);
        LLMOPS_LAUNCH_CHECK();
        return LLMOPS_OK;
    }
    // (the decode kernels index heads with the grid's y dimension: more than 65535 heads in all take the general
    // path below, which the position in device memory cannot)
    if (qL == 1 && (half % 4) == 0 && (bhq <= 65535 || pos_dev != nullptr)) {
        // decode: rope, cache update and split-KV attention in one launch, then the merge of the chunk records
        // (none when a head has a single chunk).  With the position in device memory the launch is sized for a
        // full cache.
        const int64_t kv_plan = pos_dev ? maxlen : kvLen;
        const DecodePlan p = plan_decode(bhq, kv_plan, kHalfCache, max_records);
        const int nchunks = (int)((kv_plan + 4 * p.pw - 1) / (4 * p.pw));
        if ((int64_t)bhq * nchunks > max_records)
            return fail(LLMOPS_EWORKSPACE, "attention workspace too small for %lld chunk records", (long long)bhq * nchunks);
        if (bhq > 65535 || maxlen * S * (int64_t)sizeof(T) >= ((int64_t)1 << 32))
            return fail(LLMOPS_EINVAL, "decode attention: at most 65535 heads in all and a cache plane per head below 4 GiB");
        const dim3 grid((unsigned)nchunks, (unsigned)bhq);
#define LLMOPS_DECODE(PWV)                                                                                         \
    attn_decode_kernel<T, PWV><<<grid, 256, 0, st>>>(pos_dev, position_id, nchunks, (int)maxlen, kc, vc, slots, q, k, v, inv_freq, \
                                                     (int)half, part)
        switch (p.pw) {
            case 4: if constexpr (!kHalfCache) LLMOPS_DECODE(4); break;
            case 8: LLMOPS_DECODE(8); break;
            case 16: LLMOPS_DECODE(16); break;
            case 32: if constexpr (kHalfCache) LLMOPS_DECODE(32); break;
        }
#undef LLMOPS_DECODE
        LLMOPS_LAUNCH_CHECK();
        if (nchunks > 1) {
            if (pos_dev != nullptr) attn_merge_kernel<<<(unsigned)bhq, 128, 0, st>>>(q, part, qL, H, nchunks, 4 * p.pw, pos_dev, maxlen);
            else merge_records(q, part, bhq, qL, H, nchunks, st);
            LLMOPS_LAUNCH_CHECK();
        }
        return LLMOPS_OK;
    }
    if (pos_dev != nullptr) return fail(LLMOPS_EINVAL, "a position in device memory needs one query token and half %% 4 == 0");
    const TokensPlan plan = plan_tokens(B * H, qL, kvLen, kHalfCache, max_records);
    const int nchunks = plan.pieces;
    // the tiled kernel finds the token of a cache row in row_token; the others compare the slots themselves
    const bool tiled = plan.kernel == 3;
    // (beside it the token ranges of the tiles, ahead of the records, of which there are at least a row's more than any plan takes)
    const unsigned tables = tiled ? (unsigned)((kvLen + 63) / 64) : 0;
    int2* const tile_tokens = reinterpret_cast<int2*>(part);
    const size_t tile_bytes = align_up((size_t)tables * 2 * sizeof(int2), 256), turn_bytes = (size_t)qL * S * sizeof(float);
    part += tile_bytes / sizeof(float);
    // q is rotated by the tiled kernel where all dimensions rotate and the angles' table fits ahead of the records (a record's place per
    // query and head is free: it does in any workspace of the size asked for)
    float* const turns = part;
    const bool late_q = tiled && half == 64 && B * qL * ((H + 31) / 32) < ((int64_t)1 << 30) && H < ((int64_t)1 << 31) &&
                        tile_bytes + turn_bytes + (nchunks > 1 ? (size_t)bhq * nchunks * (S + 2) * sizeof(float) : 0) <= workspace_bytes - part_off;
    if (late_q) part += turn_bytes / sizeof(float);
    if (!tiled && (int64_t)bhq * nchunks > max_records)
        return fail(LLMOPS_EWORKSPACE, "attention workspace too small for %lld chunk records", (long long)bhq * nchunks);
    // All tokens of a head together: rotation and cache update ride in the same launch where the rotary pairs suit it, the
    // workspace has a record more per query, and the workgroup more per head makes no compute unit take one more: then the
    // launch saved is worth more than what every workgroup does for it, 1.2 us (us, separate / together, 32 heads: 8 tokens
    // behind 500 18.4 / 16.3, 31 behind 97 20.5 / 18.4, 16 behind 1500 26.4 / 24.5, halves 23.1 / 21.6; 4 behind 1000 20.2 / 21.1, 31
    // behind 3500 48.3 / 48.7; 128 heads, 16 behind 500 34.3 / 35.7).
    const int64_t wgs = B * H * nchunks, wgs_rope = wgs + B * H;
    if (plan.kernel == 2 && half == 64 && (int64_t)bhq * (nchunks + 1) <= max_records && wgs_rope <= 512 && (wgs > 256) == (wgs_rope > 256)) {
        attn_few_kernel<T, true><<<(unsigned)wgs_rope, 256, 0, st>>>(q, kc, vc, (int)qL, H, maxlen, (int)kvLen, slots, part,
                                                                                   nchunks + 1, k, v, inv_freq, position_id);
        LLMOPS_LAUNCH_CHECK();
        merge_records(q, part, bhq, qL, H, nchunks + 1, st);
        LLMOPS_LAUNCH_CHECK();
        return LLMOPS_OK;
    }
    if (late_q) {
        const unsigned head_groups = (unsigned)((H + 31) / 32);
        attn_prep_rows_kernel<T><<<(unsigned)(B * qL) * head_groups + tables, 256, 0, st>>>(k, v, (int)qL, (int)H, inv_freq, kc, vc, maxlen, slots, position_id,
                                                                                            row_token, tile_tokens, kvLen, tables, head_groups, turns);
    } else if (tiled) {
        attn_prep_kernel<T, true><<<(unsigned)(B * qL * H) + tables, 64, 0, st>>>(q, k, v, qL, H, S, inv_freq, half, kc, vc, maxlen, slots,
                                                                                 position_id, row_token, tile_tokens, kvLen, tables);
    } else {
        attn_prep_kernel<T, false><<<(unsigned)(B * qL * H), 64, 0, st>>>(q, k, v, qL, H, S, inv_freq, half, kc, vc, maxlen, slots,
                                                                         position_id, nullptr, nullptr, 0, 0);
    }
    LLMOPS_LAUNCH_CHECK();
    if (tiled) {
        // enough query tokens to share K/V tiles: the MFMA kernel reads the cache once per 128 queries
        if (maxlen * S * (int64_t)sizeof(T) >= ((int64_t)1 << 32))
            return fail(LLMOPS_EINVAL, "attention over 32 or more query tokens: a head's cache plane must be below 4 GiB");
        const int qtiles = (int)((qL + 127) / 128);
        constexpr size_t smem = prefill_smem_bytes<!kHalfCache>();
        static bool configured = false;  // opt in to more than 64 KiB of dynamic LDS once per kernel
        if (!configured) {
            LLMOPS_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(&attn_prefill_kernel<T>),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem));
            configured = true;
        }
        attn_prefill_kernel<T><<<dim3((unsigned)(B * H * qtiles), (unsigned)nchunks), 512, smem, st>>>(q, kc, vc, qL, H, maxlen, kvLen, row_token, tile_tokens,
                                                                                                       qtiles, plan.rows, part, nchunks, late_q ? turns : nullptr);
        LLMOPS_LAUNCH_CHECK();
        if (nchunks > 1) {
            merge_records(q, part, bhq, qL, H, nchunks, st);
            LLMOPS_LAUNCH_CHECK();
        }
        return LLMOPS_OK;
    }
    if (plan.kernel == 2)
        attn_few_kernel<T, false><<<(unsigned)(B * H * nchunks), 256, 0, st>>>(q, kc, vc, (int)qL, H, maxlen, (int)kvLen, slots, part,
                                                                               nchunks, nullptr, nullptr, nullptr, 0);
    else if (plan.pw == 16)
        attn_split_kernel<T, 16><<<(unsigned)(bhq * nchunks), 256, 0, st>>>(q, kc, vc, qL, H, maxlen, kvLen, slots, part, nchunks);
    else if (plan.pw == 8)
        attn_split_kernel<T, 8><<<(unsigned)(bhq * nchunks), 256, 0, st>>>(q, kc, vc, qL, H, maxlen, kvLen, slots, part, nchunks);
    else
        attn_split_kernel<T, 4><<<(unsigned)(bhq * nchunks), 256, 0, st>>>(q, kc, vc, qL, H, maxlen, kvLen, slots, part, nchunks);
    LLMOPS_LAUNCH_CHECK();
    merge_records(q, part, bhq, qL, H, nchunks, st);
    LLMOPS_LAUNCH_CHECK();
    return LLMOPS_OK;
}

static int attention_entry(float* q, float* k, const float* v, int64_t B, int64_t qL, int64_t H, int64_t S,
                           const float* inv_freq, int64_t half, void* kv_cache, int cache_dtype, int64_t planes,
                           int64_t maxlen, const int32_t* slots, int position_id, const int32_t* pos_dev, int layer_id,
                           void* workspace, size_t workspace_bytes, llmops_stream_t stream, float* rec_stats = nullptr,
                           float* rec_outs = nullptr) {
    LLMOPS_REQUIRE(q != nullptr && k != nullptr && v != nullptr && inv_freq != nullptr && kv_cache != nullptr);
    LLMOPS_REQUIRE(slots != nullptr && workspace != nullptr);
    LLMOPS_REQUIRE(B > 0 && qL > 0 && H > 0 && maxlen > 0);
    LLMOPS_REQUIRE(S == 128);  // head size of every supported model shape (the reference needs S % 16 == 0)
    LLMOPS_REQUIRE(half > 0 && 2 * half <= S);
    LLMOPS_REQUIRE(layer_id >= 0 && 2 * (int64_t)layer_id + 1 < planes);
    LLMOPS_REQUIRE(position_id >= 0);
    LLMOPS_REQUIRE(cache_dtype == LLMOPS_CACHE_F32 || cache_dtype == LLMOPS_CACHE_F16);
    LLMOPS_REQUIRE(aligned(q, 16) && aligned(k, 16) && aligned(v, 16) && aligned(kv_cache, 16) && aligned(workspace, 256));
    LLMOPS_REQUIRE(B * H * qL * ((maxlen + 63) / 64) < ((int64_t)1 << 31));
    const size_t need = llmops_attention_workspace_bytes(B, qL, H, S, maxlen);
    if (workspace_bytes < need)
        return fail(LLMOPS_EWORKSPACE, "attention_rope needs %zu workspace bytes, got %zu", need, workspace_bytes);
    hipStream_t st = as_stream(stream);
    if (cache_dtype == LLMOPS_CACHE_F32)
        return attention_impl<float>(q, k, v, B, qL, H, S, inv_freq, half, reinterpret_cast<float*>(kv_cache), maxlen, slots,
                                     position_id, pos_dev, layer_id, workspace, workspace_bytes, st, rec_stats, rec_outs);
    return attention_impl<__half>(q, k, v, B, qL, H, S, inv_freq, half, reinterpret_cast<__half*>(kv_cache), maxlen, slots,
                                  position_id, pos_dev, layer_id, workspace, workspace_bytes, st, rec_stats, rec_outs);
}

extern "C" int llmops_attention_rope(float* q, float* k, const float* v, int64_t B, int64_t qL, int64_t H, int64_t S,
                                     const float* inv_freq, int64_t half, void* kv_cache, int cache_dtype,
                                     int64_t planes, int64_t maxlen, const int32_t* slots, int position_id,
                                     int layer_id, void* workspace, size_t workspace_bytes, llmops_stream_t stream) {
    return attention_entry(q, k, v, B, qL, H, S, inv_freq, half, kv_cache, cache_dtype, planes, maxlen, slots, position_id,
                           nullptr, layer_id, workspace, workspace_bytes, stream);
}

extern "C" int llmops_attention_rope_decode(float* q, float* k, const float* v, int64_t B, int64_t H, int64_t S,
                                            const float* inv_freq, int64_t half, void* kv_cache, int cache_dtype,
                                            int64_t planes, int64_t maxlen, const int32_t* slot,
                                            const int32_t* position_id, int layer_id, void* workspace,
                                            size_t workspace_bytes, llmops_stream_t stream) {
    LLMOPS_REQUIRE(position_id != nullptr && (half % 4) == 0);
    return attention_entry(q, k, v, B, 1, H, S, inv_freq, half, kv_cache, cache_dtype, planes, maxlen, slot, 0, position_id,
                           layer_id, workspace, workspace_bytes, stream);
}

extern "C" int64_t llmops_attention_records_chunks(int64_t maxlen, int cache_dtype) {
    return records_chunk_rows(maxlen, cache_dtype == LLMOPS_CACHE_F16) ? kAttnRecChunks : 0;
}

extern "C" int64_t llmops_attention_records_chunk_rows(int64_t maxlen, int cache_dtype) {
    return records_chunk_rows(maxlen, cache_dtype == LLMOPS_CACHE_F16);
}

extern "C" int llmops_attention_rope_decode_records(float* q, float* k, const float* v, int64_t B, int64_t H, int64_t S,
                                                    const float* inv_freq, int64_t half, void* kv_cache, int cache_dtype,
                                                    int64_t planes, int64_t maxlen, const int32_t* slot, int position_id,
                                                    const int32_t* position_id_dev, int layer_id, float* rec_stats,
                                                    float* rec_outs, void* workspace, size_t workspace_bytes,
                                                    llmops_stream_t stream) {
    LLMOPS_REQUIRE(rec_stats != nullptr && rec_outs != nullptr && aligned(rec_stats, 16) && aligned(rec_outs, 16));
    return attention_entry(q, k, v, B, 1, H, S, inv_freq, half, kv_cache, cache_dtype, planes, maxlen, slot, position_id,
                           position_id_dev, layer_id, workspace, workspace_bytes, stream, rec_stats, rec_outs);
}

extern "C" int llmops_test_attn_plan(int64_t B, int64_t qL, int64_t H, int64_t maxlen, int position_id, int cache_dtype, int* kernel,
                                     int* rows, int* pieces) {
    LLMOPS_TEST_HOOK();
    LLMOPS_REQUIRE(B > 0 && qL > 0 && H > 0 && maxlen > 0 && position_id >= 0 && kernel != nullptr && rows != nullptr && pieces != nullptr);
    const size_t head = LLMOPS_ATTN_COUNTER_BYTES + align_up((size_t)maxlen * 4, 256);
    const int64_t max_records = (int64_t)((llmops_attention_workspace_bytes(B, qL, H, 128, maxlen) - head) / (130 * sizeof(float)));
    const int64_t kv = position_id + qL < maxlen ? position_id + qL : maxlen;
    const TokensPlan p = plan_tokens(B * H, qL, kv, cache_dtype == LLMOPS_CACHE_F16, max_records);
    *kernel = p.kernel, *rows = p.rows, *pieces = p.pieces;
    return LLMOPS_OK;
}

extern "C" void llmops_test_attn_set_decode_plan(int rows_per_wave) {
    if (llmops::test_hooks_enabled("llmops_test_attn_set_decode_plan")) llmops::g_decode_pw = rows_per_wave;
}

extern "C" int llmops_softmax(float* x, int64_t rows, int64_t K, llmops_stream_t stream) {
    LLMOPS_REQUIRE(x != nullptr && rows > 0 && K > 0 && rows < ((int64_t)1 << 31));
    softmax_kernel<<<(unsigned)rows, 256, 0, as_stream(stream)>>>(x, K);
    LLMOPS_LAUNCH_CHECK();
    return LLMOPS_OK;
}
