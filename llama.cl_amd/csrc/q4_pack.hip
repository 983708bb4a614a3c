// Q4_1 weight packing and unpacking on the device.
//
// A packed dword holds the 8 consecutive k-values 8r..8r+7 of one column (low nibbles = k 8r..8r+3,
// high nibbles = k 8r+4..8r+7); one thread forms it.  The G/8 threads of a column sit in adjacent
// lanes, so the per-column min/max is a short exchange between lanes of a row of 16.
//
// Arithmetic follows offline_FC_quant_Q4A (/root/reference/ops/op_fc.hpp:151-219) operation for
// operation so the packed bytes are identical: d=(max-min)/15, id=1/d (IEEE division), code =
// clamp(roundf((w-m)*id),0,15) with the *unrounded* fp32 d and m, and d, m stored as RNE fp16.
#include "common.h"

namespace llmops {

// the value of lane (own ^ O); all lanes are active and O stays inside a row of 16 lanes
template <int O>
__device__ __forceinline__ float lane_xor(float v) {
    const int b = __float_as_int(v);
    if constexpr (O == 1) return __int_as_float(__builtin_amdgcn_mov_dpp(b, 0xB1, 0xF, 0xF, true));  // quad_perm [1,0,3,2]
    if constexpr (O == 2) return __int_as_float(__builtin_amdgcn_mov_dpp(b, 0x4E, 0xF, 0xF, true));  // quad_perm [2,3,0,1]
    if constexpr (O == 4)  // row_half_mirror (^7), then quad_perm [3,2,1,0] (^3)
        return __int_as_float(__builtin_amdgcn_mov_dpp(__builtin_amdgcn_mov_dpp(b, 0x141, 0xF, 0xF, true), 0x1B, 0xF, 0xF, true));
    if constexpr (O == 8) return __int_as_float(__builtin_amdgcn_mov_dpp(b, 0x128, 0xF, 0xF, true));  // row_ror:8
}

// min/max with the reference's "first occurrence wins" behaviour on equal values
// (get_min_max, ops/op_fc.hpp:112-122, compares strictly), which decides the sign of a zero.
template <int O, int R>
__device__ __forceinline__ void column_min_max(float& vmin, float& vmax) {
    if constexpr (O < R) {
        const float omin = lane_xor<O>(vmin), omax = lane_xor<O>(vmax);
        const bool partner_first = (threadIdx.x & O) != 0;  // partner holds lower k
        if (omin < vmin || (omin == vmin && partner_first)) vmin = omin;
        if (omax > vmax || (omax == vmax && partner_first)) vmax = omax;
        column_min_max<2 * O, R>(vmin, vmax);
    }
}

typedef float float4_4 __attribute__((ext_vector_type(4), aligned(4)));  // 16 bytes from any 4

// Bound by reading the fp32 matrix (the vector ALU issues 73 % of the time beside it).  A workgroup takes 128 k-values of 32 columns (one block of group 128, four of group
// 32); a thread loads 8 values of each of two columns, 16 bytes a load, before it uses any (128 KB in flight per compute
// unit), and the packed dwords go through LDS so that a wave writes 256 consecutive bytes instead of 16 bytes in each of
// 16 rows.  11008 x 4096, before (4-byte loads, one block of 512 threads per column set) / now: group 128 99 / 36.4 us
// (5.6 TB/s), group 32 117 / 36.5 us; in a graph 1000 x 4096 12.0 / 5.8 us, 512 x 512, too little to fill the chip, 4.3 / 3.2
// and 3.4 / 3.0 us.  Rows may start on any 4 bytes: the loads do not ask for more (2048 x 4098 21.7 / 9.4 us; four bytes a
// load 20.4).  A thread that K cuts loads the last value again instead of branching around each (513 x 513 4.4 / 3.4 and, group
// 32, 3.5 / 3.1 us; with the branches 4.7 and 4.4).
template <int G>
__global__ __launch_bounds__(256) void quant_w_kernel(const float* __restrict__ wei, int64_t N, int64_t K, int64_t ld,
                                                      uint8_t* __restrict__ out, int64_t Kg) {
    constexpr int R = G / 8;         // packed rows (and lanes of a column) per block
    constexpr int kSub = 128 / G;    // blocks per workgroup
    constexpr int kPitch = 33;       // dwords; lanes of a column write consecutive rows: an odd pitch spreads the banks
    __shared__ uint32_t tile[kSub * (R + 1) * kPitch];
    const int r16 = threadIdx.x & 15, c0 = threadIdx.x >> 4;
    const int nb = blockIdx.y;
    const int64_t kb0 = (int64_t)blockIdx.x * kSub;
    const int64_t k0 = kb0 * G + r16 * 8;
    const int sub = r16 / R, r = r16 % R;
    const int cnt = (int)(K - k0 >= 8 ? 8 : K > k0 ? K - k0 : 0);

    float v[2][8];
    if (cnt == 8) {
#pragma unroll
        for (int c = 0; c < 2; c++) {
            const int64_t n = (int64_t)nb * kGroupN + c0 + 16 * c;
            const float4_4* src = reinterpret_cast<const float4_4*>(wei + (n < N ? n : N - 1) * ld + k0);
            const float4_4 lo = src[0], hi = src[1];
#pragma unroll
            for (int j = 0; j < 4; j++) v[c][j] = lo[j], v[c][4 + j] = hi[j];
        }
    } else {
#pragma unroll
        for (int c = 0; c < 2; c++) {
            const int64_t n = (int64_t)nb * kGroupN + c0 + 16 * c;
            const float* src = wei + (n < N ? n : N - 1) * ld;
            // (values past K repeat the last one: no effect on strict comparisons; their codes are cleared below)
#pragma unroll
            for (int j = 0; j < 8; j++) v[c][j] = src[k0 + j < K ? k0 + j : K - 1];
        }
    }
#pragma unroll
    for (int c = 0; c < 2; c++) {
        const int ni = c0 + 16 * c;
        const bool row_ok = (int64_t)nb * kGroupN + ni < N;
        float vmin = v[c][0], vmax = v[c][0];
#pragma unroll
        for (int j = 1; j < 8; j++) {
            if (vmax < v[c][j]) vmax = v[c][j];
            if (vmin > v[c][j]) vmin = v[c][j];
        }
        if (cnt == 0) vmin = __builtin_inff(), vmax = -__builtin_inff();
        column_min_max<1, R>(vmin, vmax);
        const float d = (vmax - vmin) / 15.0f, m = vmin;
        const float id = (d != 0.0f) ? (1.0f / d) : 0.0f;
        uint32_t packed = 0;
#pragma unroll
        for (int j = 0; j < 8; j++) {
            // roundf (half away from zero) of t in [0, 15]: the integer part of t + (the float below 0.5), the sum rounded
            // to nearest even, for every such t.  0 and 15 are whole, so clamping may come first; a NaN becomes 0
            float t = (v[c][j] - m) * id;
            t = fminf(15.0f, fmaxf(t, 0.0f));
            const uint32_t q = (uint32_t)__fadd_rn(t, 0x1.fffffep-2f);
            packed |= q << ((j & 3) * 8 + (j >> 2) * 4);
        }
        if (cnt < 8) {
            uint32_t keep = 0;
#pragma unroll
            for (int j = 0; j < 8; j++)
                if (j < cnt) keep |= 0xFu << ((j & 3) * 8 + (j >> 2) * 4);
            packed &= keep;
        }
        uint32_t* blk = tile + sub * (R + 1) * kPitch;
        blk[r * kPitch + ni] = row_ok ? packed : 0u;
        if (r == 0) {
            uint16_t* wd = reinterpret_cast<uint16_t*>(blk + R * kPitch);
            wd[ni] = row_ok ? f32_to_f16_bits(d) : (uint16_t)0;
            wd[32 + ni] = row_ok ? f32_to_f16_bits(m) : (uint16_t)0;
        }
    }
    __syncthreads();
    const int subs = (int)(Kg - kb0 < kSub ? Kg - kb0 : kSub);  // the last workgroup of group 32 may have fewer blocks
    uint32_t* dst = reinterpret_cast<uint32_t*>(out + ((int64_t)nb * Kg + kb0) * block_bytes(G));
    for (int i = threadIdx.x; i < subs * (R + 1) * 32; i += 256) dst[i] = tile[(i >> 5) * kPitch + (i & 31)];
}

// out[n, k] = fp32(d)*q + fp32(m) (q4_1_block::get, ops/op_fc.hpp:49-61).  d has 11 significant
// bits and q 4, so the product is exact and contraction cannot change the result.
// Bound by writing the fp32 matrix.  A workgroup takes 128 k-values of 32 columns, as above: the blocks come through LDS
// with consecutive reads, and 32 lanes write 512 consecutive bytes of a row, 16 bytes a lane.
// 11008 x 4096, before / now: group 128 46.1 / 40.7 us (5.0 TB/s), group 32 42.7 / 41.1 us; 1000 x 4096 6.3 / 5.1, 5.7 / 5.1 us;
// 512 x 512, all latency, 2.5 / 2.6 us.
template <int G>
__global__ __launch_bounds__(256) void dequant_w_kernel(const uint8_t* __restrict__ weiq, int64_t Kg, float* __restrict__ out) {
    constexpr int R = G / 8, kSub = 128 / G, kPitch = 33;  // (33: the rows of a column fall into different banks)
    __shared__ uint32_t tile[kSub * (R + 1) * kPitch];
    const int nb = blockIdx.y;
    const int64_t kb0 = (int64_t)blockIdx.x * kSub;
    const int subs = (int)(Kg - kb0 < kSub ? Kg - kb0 : kSub);
    const uint32_t* src = reinterpret_cast<const uint32_t*>(weiq + ((int64_t)nb * Kg + kb0) * block_bytes(G));
    for (int i = threadIdx.x; i < subs * (R + 1) * 32; i += 256) tile[(i >> 5) * kPitch + (i & 31)] = src[i];
    __syncthreads();
    const int k4 = threadIdx.x & 31, sub = k4 / (G / 4), r = (k4 % (G / 4)) >> 1, hi = (k4 & 1) * 4;
    if (sub >= subs) return;
    const uint32_t* blk = tile + sub * (R + 1) * kPitch;
    const uint16_t* wd = reinterpret_cast<const uint16_t*>(blk + R * kPitch);
    float* dst = out + (int64_t)nb * kGroupN * (Kg * G) + kb0 * G + k4 * 4;
#pragma unroll
    for (int c = 0; c < 4; c++) {
        const int ni = (threadIdx.x >> 5) + 8 * c;
        const uint32_t w = blk[r * kPitch + ni] >> hi;
        const float d = f16_bits_to_f32(wd[ni]), m = f16_bits_to_f32(wd[32 + ni]);
        float o[4];
#pragma unroll
        for (int j = 0; j < 4; j++) o[j] = d * (float)((w >> (8 * j)) & 0xFu) + m;
        *reinterpret_cast<float4*>(dst + ni * (Kg * G)) = make_float4(o[0], o[1], o[2], o[3]);
    }
}

}  // namespace llmops

using namespace llmops;

extern "C" int64_t llmops_q4a_block_bytes(int group_k) { return valid_group(group_k) ? block_bytes(group_k) : 0; }

extern "C" int llmops_offline_FC_quant_Q4A(const float* wei, int64_t N, int64_t K, int64_t ld, int group_k,
                                           int8_t* weiq, llmops_stream_t stream) {
    LLMOPS_REQUIRE(valid_group(group_k));
    LLMOPS_REQUIRE(wei != nullptr && weiq != nullptr);
    LLMOPS_REQUIRE(N > 0 && K > 0 && ld >= K);
    LLMOPS_REQUIRE(aligned(weiq, 4));
    const int64_t Ng = (N + kGroupN - 1) / kGroupN, Kg = (K + group_k - 1) / group_k;
    LLMOPS_REQUIRE(Ng <= 65535 && Kg <= 0x7fffffff);
    uint8_t* out = reinterpret_cast<uint8_t*>(weiq);
    if (group_k == 32)
        quant_w_kernel<32><<<dim3((unsigned)((Kg + 3) / 4), (unsigned)Ng), 256, 0, as_stream(stream)>>>(wei, N, K, ld, out, Kg);
    else
        quant_w_kernel<128><<<dim3((unsigned)Kg, (unsigned)Ng), 256, 0, as_stream(stream)>>>(wei, N, K, ld, out, Kg);
    LLMOPS_LAUNCH_CHECK();
    return LLMOPS_OK;
}

extern "C" int llmops_offline_FC_dequant_Q4A(const int8_t* weiq, int64_t Ng, int64_t Kg, int group_k, float* out,
                                             llmops_stream_t stream) {
    LLMOPS_REQUIRE(valid_group(group_k));
    LLMOPS_REQUIRE(weiq != nullptr && out != nullptr);
    LLMOPS_REQUIRE(Ng > 0 && Kg > 0 && Ng <= 65535);
    LLMOPS_REQUIRE(aligned(weiq, 4) && aligned(out, 16));
    const uint8_t* in = reinterpret_cast<const uint8_t*>(weiq);
    if (group_k == 32)
        dequant_w_kernel<32><<<dim3((unsigned)((Kg + 3) / 4), (unsigned)Ng), 256, 0, as_stream(stream)>>>(in, Kg, out);
    else
        dequant_w_kernel<128><<<dim3((unsigned)Kg, (unsigned)Ng), 256, 0, as_stream(stream)>>>(in, Kg, out);
    LLMOPS_LAUNCH_CHECK();
    return LLMOPS_OK;
}
