// Q4_1 x Q8 fully-connected product for more than 8 activation rows, group 32: int8 MFMA (fc_Q4A,
// /root/reference/ops/op_fc.hpp:381-412).
//
// What bounds it: with a group of 32 every v_mfma_i32_32x32x32_i8 (32 cycles) is a whole k-group of its tile, and its 16
// results per lane are folded into the fp32 accumulators with 32 vector instructions.  Products and vector instructions of a
// SIMD's waves hardly overlap (registers only: 8 such MFMAs take 256 cycles, 64 fold instructions 296 in one wave and 296 in
// two waves together, both 360 in one wave, 680 in two, 1000 in three): a step of 32 x 64 is 96 cycles of products, the min
// term's included, and about 98 vector instructions of 2 cycles.  So everything else is kept off the vector ALU and out of
// its way, and three workgroups share a compute unit (a stage of four k-groups: one alone 0.95 us, two 1.24, three 1.46):
//   * 168 registers: the operands of one k-group are in registers, those of the next on their way from LDS, and not those of a
//     whole stage (216, two workgroups: 512 x 11008 x 4096, whose 688 tiles are then more than a round, 105.5 us against 87.2,
//     128 x 11008 x 4096 40.9 / 35.0, 2048 x 4096^2 133 / 127).
//   * tile 32 rows x 256 columns, four waves side by side (each 32 x 64 = two strips): a strip's weights are unpacked by
//     one wave only, and the rows' codes and scales are read from LDS by all four.  (Sixty-four rows x 128 columns, two
//     waves either way, measured with two workgroups to a compute unit: 0 to 3 % slower at almost every size; 128 x 128 with
//     64 x 64 per wave: 7 %.)
//   * a stage is four k-groups.  Codes, packed blocks, scales and sums are all copied to LDS asynchronously
//     (global_load_lds) one stage ahead: no registers, no LDS store instructions, 16 bytes per lane where the layout has
//     them.  (Weights taken straight from memory into operand registers, one dword per lane and load, cost more than
//     all of the arithmetic: 1.6 times the time of the call.)
//   * the fold of one step runs while the next step's MFMA does: two accumulators, the order pinned.
//   * f += d * dx * sum in two instructions: the sums start at the bit pattern of 1.5 * 2^23 (gemm_device.h), so the
//     register read as a float X is bias + sum and fma(X, d, -bias * d) = sum * d, exact before its one rounding
//     (|sum| <= 32 * 15 * 127 < 2^22; bias * d has 2 + 11 significant bits).
//   * the min term, sum over k-groups of m[column] * gsum[row], is a product with K = number of k-groups, on the matrix
//     cores instead of a third vector instruction per element: gsum = three and m = two bf16 pieces, exactly and at any
//     scale, and the six products of two k-groups fill one v_mfma_f32_32x32x16_bf16 per strip.  It runs between the folds
//     of its two groups: the weights' codes are positive, so what a fold adds is several times what the min term
//     leaves of it, and the fewer groups a sum holds uncorrected the less it loses to rounding.  rms error of the outputs,
//     64 x 1024, against 64 bits, in 1e-7 of their rms, two instructions per element and group as before / fp16 halves of
//     gsum every eight groups / now: K = 512 1.16 / 2.91 / 1.16, 1024 1.36 / 3.04 / 1.30, 4096 2.22 / 3.54 / 1.58, 11008
//     2.18 / 3.52 / 1.79.  (Four groups at a time, a bf16 and a half-length bf16 product: 1.20 / 1.25 / 1.51 / 1.72, and
//     0 to 2 % faster.)
#include <type_traits>

#include "gemm_device.h"
#include "gemv_device.h"

namespace llmops {

constexpr int kG32Blk = 640;       // bytes of a packed block: 512 of nibbles, 32 fp16 scales, 32 fp16 mins
constexpr int kG32Rows = 32;       // rows and strips of a tile
constexpr int kG32Strips = 8;
constexpr int kG32Gps = 4;         // k-groups per stage

typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
union Bf16x8 {
    v8bf h;
    uint32_t u[4];
};
// the first 8 significant bits of a float (what its upper half is as a bf16), and the upper halves of two floats
__device__ __forceinline__ float bf_piece(float v) { return __uint_as_float(__float_as_uint(v) & 0xFFFF0000u); }
__device__ __forceinline__ uint32_t bf_pair(float lo, float hi) {
    return __builtin_amdgcn_perm(__float_as_uint(hi), __float_as_uint(lo), 0x07060302u);
}

// PARTIALS: test build that stores the int32 sums of every (row, column, k-group) into out_i ([rows][Ng*32][Kg])
// WIDE: lane offsets of 64 bits, for a K whose eight strips are 4 GiB and more (K above 26.8 million)
template <bool PARTIALS, bool WIDE>
__global__ __launch_bounds__(256, 3) void fc_gemm_g32_kernel(const uint8_t* __restrict__ weiq, const int8_t* __restrict__ xq,
                                                              const float* __restrict__ xd, const float* __restrict__ gs,
                                                              const float2* __restrict__ xsT, float* __restrict__ out,
                                                              int32_t* __restrict__ out_i, int Ng, int Kg, int64_t ldo, int64_t N,
                                                              int rows, int st_per_split, int64_t split_stride,
                                                              const float* __restrict__ residual) {
    constexpr int BM = kG32Rows, STRIPS = kG32Strips, GPS = kG32Gps, BLK = kG32Blk;
    using offset_t = typename std::conditional<WIDE, uint64_t, uint32_t>::type;
    __shared__ __align__(16) uint8_t sa[2][BM * 128];           // codes, 128 bytes per row
    __shared__ __align__(16) uint8_t sbn[2][STRIPS * 2048];     // nibbles, 16 k8-rows of 128 bytes per strip
    __shared__ __align__(16) float sx[2][GPS * BM];             // activation scales [k-group][row]
    __shared__ __align__(16) uint16_t sdm[2][GPS * STRIPS * 64];  // [k-group][strip][32 scales, 32 mins]
    __shared__ __align__(16) float sg[2][GPS * BM];             // activation sums [k-group][row]

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int h = lane >> 5, j = lane & 31;
    // tile numbering: one contiguous run of tiles per XCD (workgroups go to the XCDs round robin), bands of 8 row blocks,
    // rows fastest, so that what is resident on one XCD shares its L2
    const int nbx = (Ng + STRIPS - 1) / STRIPS, nby = (rows + BM - 1) / BM;
    int bx, by;
    {
        const int total = nbx * nby, per_xcd = (total + 7) / 8;
        const int i = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
        if ((int)(blockIdx.x >> 3) >= per_xcd || i >= total) return;  // uniform for the workgroup
        constexpr int kBand = 8;
        const int band = i / (kBand * nbx), in_band = i % (kBand * nbx);
        const int first = band * kBand, rows_in_band = min(kBand, nby - first);
        by = first + in_band % rows_in_band;
        bx = in_band / rows_in_band;
    }
    const int tstrip = bx * STRIPS, strip0 = tstrip + 2 * wave;  // the tile's and this wave's first strip (may lie beyond Ng)
    const int row0 = by * BM;
    const int nst = (Kg + GPS - 1) / GPS;
    const int st0 = blockIdx.z * st_per_split, st1 = min(nst, st0 + st_per_split);
    const int kg1 = min(Kg, st1 * GPS);
    const offset_t Kp = (offset_t)Kg * 32;

    // ---- what this wave copies per stage.  Sources past the end (rows, strips, the last stage's k-groups) re-read the
    // last one that exists. ----
    // codes: rows 8*wave .. +7.  16-byte chunk c of row r lies at position c ^ key(r), key(r) = (r + ((r >> 3) & 1)) & 7: the
    // 16 rows that one phase of a ds_read_b128 touches fall on 16 different bank groups
    const uint8_t* abase = reinterpret_cast<const uint8_t*>(xq) + (int64_t)row0 * (int64_t)Kp;
    const offset_t arow = (offset_t)(min(rows - 1, row0 + wave * 8 + (lane >> 3)) - row0) * Kp;
    const uint32_t achunk = (uint32_t)(((lane & 7) ^ (((lane >> 3) + (wave & 1)) & 7)) * 16);
    const uint32_t lds_a = lds_off(&sa[0][0]), lds_b = lds_off(&sbn[0][0]), lds_x = lds_off(&sx[0][0]), lds_d = lds_off(&sdm[0][0]),
                   lds_g = lds_off(&sg[0][0]);
    // nibbles: two strips, 8 k8-rows to a copy, the two low bits of the row number exchanged: the rows 4s+2h+p that the lane
    // halves h = 0, 1 read together lie side by side
    const offset_t sb = (offset_t)Kg * BLK;  // bytes of a strip
    const uint8_t* bbase = weiq + (int64_t)tstrip * (int64_t)sb;
    offset_t boff[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int slot = (i & 1) * 8 + (lane >> 3), r = (slot & 12) | ((slot & 1) << 1) | ((slot >> 1) & 1);
        boff[i] = (offset_t)(min(Ng - 1, strip0 + (i >> 1)) - tstrip) * sb + (uint32_t)((r & 3) * kRowBytes + (lane & 7) * 16);
    }
    // scales and mins: k-group `wave` of the stage, 128 bytes per block, eight strips
    const offset_t doff = (offset_t)(min(Ng - 1, tstrip + (lane >> 3)) - tstrip) * sb + (uint32_t)(512 + (lane & 7) * 16);
    // activation scales (waves 0, 1) and sums (waves 2, 3): two k-groups of 32 rows to a copy
    const int xrow = min(rows - 1, row0 + j);
    auto copy_stage = [&](int st, int buf) {
        const int kg0 = st * GPS;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int kg = min(Kg - 1, kg0 + (i & 1) * 2 + h);
            copy16_to_lds(bbase, boff[i] + (offset_t)kg * BLK, uniform_u32(lds_b + buf * (STRIPS * 2048) + (wave * 4 + i) * 1024));
        }
        copy16_to_lds(abase, arow + min((offset_t)st * 128u + achunk, Kp - 16u), uniform_u32(lds_a + buf * (BM * 128) + wave * 1024));
        if (PARTIALS) return;
        {
            const int c = wave & 1, kg = min(Kg - 1, kg0 + 2 * c + h);
            const bool sums = wave >= 2;  // uniform
            const uint32_t dst = uniform_u32((sums ? lds_g : lds_x) + (buf * GPS * BM + c * 64) * 4);
            if (xsT) {
                const int kgb = min(Kg - 1, kg0 + 2 * c);
                copy4_to_lds(uniform_ptr(reinterpret_cast<const float*>(xsT + (int64_t)kgb * rows) + (sums ? 1 : 0)),
                             (offset_t)((kg - kgb) * rows + xrow) * 8u, dst);
            } else {
                copy4_to_lds(uniform_ptr((sums ? gs : xd) + (int64_t)row0 * Kg), ((offset_t)(xrow - row0) * Kg + kg) * 4u, dst);
            }
        }
        copy16_to_lds(bbase + (int64_t)min(Kg - 1, kg0 + wave) * BLK, doff, uniform_u32(lds_d + (buf * GPS + wave) * (STRIPS * 128)));
    };

    if (st0 < st1) copy_stage(st0, 0);
    v16f f[2];
    v16i bias;
#pragma unroll
    for (int i = 0; i < 16; i++) f[0][i] = f[1][i] = 0.0f, bias[i] = PARTIALS ? 0 : kFoldBiasBits;
    asm volatile("" : "+v"(bias));
    constexpr int kVmcnt0 = 0x0F70;  // vmcnt(0), the other counters left alone
    __builtin_amdgcn_s_waitcnt(kVmcnt0);
    __syncthreads();

    const int akey = (j + ((j >> 3) & 1)) & 7;

    for (int st = st0; st < st1; st++) {
        const int buf = (st - st0) & 1;
        const bool more = st + 1 < st1;
        const int nk = min(GPS, kg1 - st * GPS);
        v4i af[2];
        uint32_t raw[2][2];
        uint16_t dbits[2];
        float4 xf[4];
        auto load_ops = [&](int kk) {
            af[kk & 1] = *reinterpret_cast<const v4i*>(&sa[buf][j * 128 + (((2 * kk + h) ^ akey) * 16)]);
#pragma unroll
            for (int s = 0; s < 2; s++) {
                const uint8_t* bs = &sbn[buf][(2 * wave + s) * 2048 + h * 128 + j * 4 + kk * 512];
                raw[s][0] = *reinterpret_cast<const uint32_t*>(bs), raw[s][1] = *reinterpret_cast<const uint32_t*>(bs + 256);
                dbits[s] = sdm[buf][kk * (STRIPS * 64) + (2 * wave + s) * 64 + j];
            }
        };
        // lane half h holds the tile rows 8b + 4h + v (result register 4b + v)
        auto load_x = [&](int kk, int b) {
            if (!PARTIALS) xf[b] = *reinterpret_cast<const float4*>(&sx[buf][kk * BM + 8 * b + 4 * h]);
        };
        load_ops(0);
#pragma unroll
        for (int b = 0; b < 4; b++) load_x(0, b);
        __builtin_amdgcn_sched_barrier(0);
        if (more) copy_stage(st + 1, buf ^ 1);
        __builtin_amdgcn_sched_barrier(0);

        v4i bu[2];
        float d[2][2];  // scales [k-group, odd or even][strip]
        auto unpack = [&](int kk) {
#pragma unroll
            for (int s = 0; s < 2; s++) {
                bu[s] = v4i{(int)lo4(raw[s][0]), (int)hi4(raw[s][0]), (int)lo4(raw[s][1]), (int)hi4(raw[s][1])};
                d[kk & 1][s] = f16_bits_to_f32(dbits[s]);
                // converted once, not inside every fma of the fold (v_fma_mix runs at half the rate of v_fma)
                asm volatile("" : "+v"(d[kk & 1][s]));
            }
        };
        // Min term operands: lane half h has the k-groups 2p + h of the stage.  The row's sum g = g1 + g2 + g3 and the
        // column's min m = m1 + m2 in bf16 pieces (g3 and m2 have at most 8 bits left, so their low halves are zero; the low
        // half of m meets that of g3).
        Bf16x8 ga, ma[2];
        float gsum;
        uint16_t mbits[2];
        auto load_min = [&](int p) {
            gsum = sg[buf][(2 * p + h) * BM + j];
#pragma unroll
            for (int s = 0; s < 2; s++) mbits[s] = sdm[buf][(2 * p + h) * (STRIPS * 64) + (2 * wave + s) * 64 + 32 + j];
        };
        auto min_ops = [&](int p) {
            const float g1 = 2 * p + h < nk ? gsum : 0.0f;  // (k-groups past the end add nothing)
            const float g2 = g1 - bf_piece(g1), g3 = g2 - bf_piece(g2);
            ga.u[0] = ga.u[2] = bf_pair(g1, g2), ga.u[1] = ga.u[3] = __float_as_uint(g3);
#pragma unroll
            for (int s = 0; s < 2; s++) {
                const float m = f16_bits_to_f32(mbits[s]), m2 = m - bf_piece(m);
                ma[s].u[0] = bf_pair(m, m), ma[s].u[1] = __float_as_uint(m);
                ma[s].u[2] = bf_pair(m2, m2), ma[s].u[3] = __float_as_uint(m2);
            }
        };
        v16i acc[2];  // steps (k-group i >> 1, strip i & 1) alternate between the two
        auto mma = [&](int i) { acc[i & 1] = __builtin_amdgcn_mfma_i32_32x32x32_i8(af[(i >> 1) & 1], bu[i & 1], bias, 0, 0, 0); };
        auto fold = [&](int i) {
            const int s = i & 1, kk = i >> 1;
            if (PARTIALS) {
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    const int row = row0 + 8 * (r >> 2) + 4 * h + (r & 3), kg = st * GPS + kk;
                    if (strip0 + s < Ng && row < rows && kg < Kg)
                        out_i[((int64_t)row * ((int64_t)Ng * kGroupN) + (strip0 + s) * kGroupN + j) * Kg + kg] = acc[s][r];
                }
                return;
            }
            const float dd = d[kk & 1][s], nbd = -kFoldBias * dd;
#pragma unroll
            for (int b = 0; b < 4; b++) {
                const float xv[4] = {xf[b].x, xf[b].y, xf[b].z, xf[b].w};
                float t[4];
#pragma unroll
                for (int v = 0; v < 4; v++) t[v] = fmaf(__int_as_float(acc[s][4 * b + v]), dd, nbd);
#pragma unroll
                for (int v = 0; v < 4; v++) f[s][4 * b + v] = fmaf(t[v], xv[v], f[s][4 * b + v]);
                if (s == 1 && kk + 1 < GPS) {
                    asm volatile("" : "+v"(f[s]));
                    load_x(kk + 1, b);
                }
            }
            // (the strip's next fold is two steps away: nothing waits for the product)
            if ((kk & 1) == 0) f[s] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ga.h, ma[s].h, f[s], 0, 0, 0);
        };
        unpack(0);
        mma(0);
#pragma unroll
        for (int kk = 0; kk < GPS; kk++) {
            if (kk >= nk) break;  // (uniform: the last stage may have fewer k-groups)
            __builtin_amdgcn_sched_barrier(0);
            mma(2 * kk + 1);
            if (kk + 1 < GPS) load_ops(kk + 1);
            if (!PARTIALS && (kk & 1) == 0) load_min(kk >> 1);
            __builtin_amdgcn_sched_barrier(0);
            if (!PARTIALS && (kk & 1) == 0) min_ops(kk >> 1);
            fold(2 * kk);
            __builtin_amdgcn_sched_barrier(0);
            if (kk + 1 < GPS) {
                unpack(kk + 1);
                mma(2 * kk + 2);
            }
            __builtin_amdgcn_sched_barrier(0);
            fold(2 * kk + 1);
        }
        __builtin_amdgcn_s_waitcnt(kVmcnt0);  // this wave's copies for the next stage have landed
        __syncthreads();
    }

    if (PARTIALS) return;
#pragma unroll
    for (int s = 0; s < 2; s++) {
        const int64_t n = (int64_t)(strip0 + s) * kGroupN + j;
        if (strip0 + s >= Ng || n >= N) continue;
        float* o = out + (int64_t)blockIdx.z * split_stride + n;
        // residual != nullptr only without split-K: then o is the result itself, row stride ldo
        const float* res = residual ? residual + n : nullptr;
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const int row = row0 + 8 * (r >> 2) + 4 * h + (r & 3);
            if (row < rows) o[(int64_t)row * ldo] = res ? f[s][r] + res[(int64_t)row * ldo] : f[s][r];
        }
    }
}

// Split-K factor.  Estimated time in us: a workgroup's run of stages and 3.6 more for what it does around them, 0.95 us each, times
// how many workgroups a compute unit has to run (three fit; two together take 1.19, three 1.45 times what one does alone); the
// second launch that adds the partial sums 1.8 us, 0.77 more per four splits (its loads in flight) and their traffic.  Against up to
// thirteen factors from 1 to 24 at up to 30 row counts from 9 to 2048 of eighteen shapes from 1024 x 512 to 22016 x 4096: 0.7 % slower than the
// best on average, 8 % at worst (65 x 22016 x 4096, 2 splits where 5 are best).  (With nothing for the ends of a run and 0.44 us for the
// second launch 2.0 % and 22 %: us, 9 x 12288 x 4096 22.4 in 16 splits / 19.4 in 8, 32 x 22016 x 4096 31.5 / 30.2 in 4, 300 x 8192 x 2048
// 36.7 in 2 / 34.7 in one, 1024 x 2048^2 33.5 in 2 / 29.7 in one.)
// Partial sums never take a workspace that fits the built-in scratch of llmops_fc_Q4A_noalloc beyond it.
int plan_gemm_g32(int64_t rows, int64_t Ng, int64_t Kg, int force_split, int* st_per_split) {
    const int64_t nst = (Kg + kG32Gps - 1) / kG32Gps;
    const int64_t tiles = ((Ng + kG32Strips - 1) / kG32Strips) * ((rows + kG32Rows - 1) / kG32Rows);
    // codes, scales, sums and pairs of a k-group: 48 bytes; the alignment of the five areas and the pairs' slack
    const int64_t room = (int64_t)LLMOPS_FC_NOALLOC_SCRATCH_BYTES - LLMOPS_FC_COUNTER_BYTES - rows * Kg * 48 - 2048;
    int64_t best_s = 1, best_per = nst;
    double best = 0.0;
    for (int64_t s = 1; s <= 24 && s <= nst; s++) {
        if (force_split > 0 && s != (force_split < nst ? (force_split < 24 ? force_split : 24) : nst)) continue;
        const int64_t per = (nst + s - 1) / s, S = (nst + per - 1) / per;
        if (S > 1 && room >= 0 && S * rows * Ng * kGroupN * 4 > room && force_split <= 0) continue;
        const int64_t full = tiles * S / 768, rest = tiles * S % 768;
        double t = 0.95 * ((double)per + 3.6) * ((double)full * 1.45 + (rest == 0 ? 0.0 : rest <= 256 ? 1.0 : rest <= 512 ? 1.19 : 1.45));
        if (S > 1) t += 1.8 + 0.77 * (double)((S + 3) / 4) + 1.05e-6 * (double)S * (double)rows * (double)(Ng * kGroupN);
        if (best == 0.0 || t < best) best = t, best_s = S, best_per = per;
    }
    *st_per_split = (int)best_per;
    return (int)best_s;
}

// 32-bit lane offsets reach into a tile's strips (5120 bytes per k-group) and, of fewer bytes, its rows' codes and scales
static bool g32_wide(int64_t Kg) { return Kg * kG32Blk * kG32Strips >= ((int64_t)1 << 32); }

int launch_gemm_g32(const uint8_t* w, const int8_t* xq, const float* xd, const float* gs, const float2* xsT, float* out, int64_t Ng,
                    int64_t Kg, int64_t ldo, int64_t N, int64_t rows, int st_per_split, int S, int64_t split_stride,
                    const float* residual, hipStream_t st) {
    if (rows >= ((int64_t)1 << 28)) return fail(LLMOPS_EINVAL, "fc_Q4A group 32: rows must be below 2^28");  // (pairs of two k-groups)
    const int64_t tiles = ((Ng + kG32Strips - 1) / kG32Strips) * ((rows + kG32Rows - 1) / kG32Rows);
    const dim3 grid((unsigned)(8 * ((tiles + 7) / 8)), 1, (unsigned)S);  // one run of tiles per XCD
    if (g32_wide(Kg))
        fc_gemm_g32_kernel<false, true><<<grid, 256, 0, st>>>(w, xq, xd, gs, xsT, out, nullptr, (int)Ng, (int)Kg, ldo, N, (int)rows,
                                                              st_per_split, split_stride, residual);
    else
        fc_gemm_g32_kernel<false, false><<<grid, 256, 0, st>>>(w, xq, xd, gs, xsT, out, nullptr, (int)Ng, (int)Kg, ldo, N, (int)rows,
                                                               st_per_split, split_stride, residual);
    LLMOPS_LAUNCH_CHECK();
    return LLMOPS_OK;
}

int launch_gemm_g32_partials(const uint8_t* w, const int8_t* xq, int32_t* acc, int64_t rows, int64_t Ng, int64_t Kg, hipStream_t st) {
    if (rows >= ((int64_t)1 << 28)) return fail(LLMOPS_EINVAL, "fc_Q4A group 32: rows must be below 2^28");
    const int64_t tiles = ((Ng + kG32Strips - 1) / kG32Strips) * ((rows + kG32Rows - 1) / kG32Rows);
    const unsigned grid = (unsigned)(8 * ((tiles + 7) / 8));
    const int nst = (int)((Kg + kG32Gps - 1) / kG32Gps);
    if (g32_wide(Kg))
        fc_gemm_g32_kernel<true, true><<<grid, 256, 0, st>>>(w, xq, nullptr, nullptr, nullptr, nullptr, acc, (int)Ng, (int)Kg, 0, 0, (int)rows,
                                                             nst, 0, nullptr);
    else
        fc_gemm_g32_kernel<true, false><<<grid, 256, 0, st>>>(w, xq, nullptr, nullptr, nullptr, nullptr, acc, (int)Ng, (int)Kg, 0, 0, (int)rows,
                                                              nst, 0, nullptr);
    LLMOPS_LAUNCH_CHECK();
    return LLMOPS_OK;
}

}  // namespace llmops
