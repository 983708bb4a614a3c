// Q4_1 x Q8 fully-connected product for 3 to some hundreds of activation rows (group 128): weight streaming like
// the one-row kernel, inner product on the int8 matrix cores (fc_Q4A, /root/reference/ops/op_fc.hpp:381-412).
//
// The work is cut like the decode kernel's: one workgroup per strip of 32 output columns (or two strips) and block of 16 to 64
// rows, its 4 or 8 waves split K into contiguous runs of k-groups, and the waves' fp32 results meet in LDS.  Nothing is staged
// through LDS on the way in, and nobody waits for anybody until the end: a lane fetches exactly the dwords that make up its B
// operands of v_mfma_i32_16x16x64_i8 (dword (k8-row r, column n) of a block holds k = 8r..8r+7 of that column; lane (g, j) of
// the MFMA needs k = 16g..16g+15 of one column), those of columns 2j and 2j + 1 together in one 8-byte load per k8-row --
// column tile tau of a strip is its columns 2j + tau, whose scales and mins are the two halves of one dword --, unpacks them
// with two ANDs and a shift, and takes its A operand (16 int8 codes of one activation row) straight from the quantized
// activations in L2.  Per k-group and output element the fold is three instructions: f = fma(fma(X, d, -B*d), dx, f), the int32
// sums starting at the bit pattern of B = 1.5 * 2^23 (gemm_device.h), and f = fma(m, gsum, f).
//
// What bounds it: the weight stream with few rows; from about 32 rows the loads of the A operands, which every strip's workgroup
// fetches again.  Hence
//   * the quantization launch leaves the codes in the order of these loads: for every 16 rows, k-group and half of it, the 64
//     lanes' 16 bytes one after the other (tile_code_offset in common.h).  In row-major order such a load touches 16 half
//     lines and takes about three times as long (64 x 11008 x 4096 26.6 -> 18.4 us, 128 x 4096^2 16.4 -> 12.4).
//   * registers are asked to be filled again as soon as their last reader has issued: weights behind their unpacking, a row
//     tile's codes behind its products.  A whole k-group's work is then between a load and its use at the price of one set of
//     registers (64 x 11008 x 4096 18.4 -> 15.1).
//   * weights are ordinary loads: non-temporal ones are 0 to 1 % faster where they come from memory, 10 to 20 % slower where the
//     256 MB cache in front of it has them or other row blocks read them too (16 x 11008 x 4096, three weights in turn, 13.3 / 11.0).
//   * two strips to a workgroup halve the codes' traffic where that leaves enough workgroups.
// Measured, us for the whole call in a graph, weights from memory, kernels before (one for up to 16 or 32 rows, the tiled one from
// there on) / now: 16 x 4096^2 7.5 / 7.2, 16 x 11008 x 4096 12.0 / 10.9, 16 x 22016 x 4096 16.1 / 14.8, 32 x 11008 x 4096 18.2 / 12.7, 64 x
// 4096^2 14.1 / 9.0, 64 x 11008 x 4096 21.4 / 16.1, 64 x 512 x 4096 10.7 / 6.5, 128 x 4096 x 11008 25.1 / 22.6, 128 x 11008 x 4096
// 27.9 / 23.2, 256 x 4096^2 20.9 / 16.3.  rms error of the outputs against 64 bits, 1e-7 of theirs: 16 rows 2.5 / 2.4, 64 to 256
// rows 2.4-2.6 / 2.1-2.3.
#include "common.h"
#include "gemm_device.h"
#include "gemv_device.h"

namespace llmops {

typedef int v4i_r __attribute__((ext_vector_type(4)));
typedef float v4f_r __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2_r __attribute__((ext_vector_type(2)));

bool streams(int64_t rows, int64_t Ng, int64_t Kg, int group_k);  // fc.hip

static int g_rows_split = 1;  // 0: never cut K in two for tensors with few strips
constexpr int kRowsBlk = 2176;

// RT: row tiles of 16 to a workgroup; SW: strips to it; NW: waves, each with a run of its k-groups; D: 1, registers filled again as
// soon as they are free, or as many k-groups as are asked for together.  tiled: the codes lie as
// tile_code_offset says (else row by row).  All loads go through buffer descriptors (scalar base + scalar offset + 32-bit lane
// offset); what lies past a wave's last k-group is asked for through descriptors of size 0, which return 0 without touching
// memory, so that every k-group issues the same loads and waits for exactly its own.
// (argument order: what the first loads need comes in the first 14 dwords, which arrive in scalar registers with the wave)
// DUMP: test build that stores the int32 sums of every (row, column, k-group) into `dump`
// ([rows][Ng*32][Kg]) instead of the outputs (llmops_fc_Q4A_partials with use_mfma = 3).
template <int RT, int SW, int NW, int D, bool DUMP = false>
__global__ __launch_bounds__(NW * 64, (RT * SW > 4 ? 2 : RT * SW > 2 ? 3 : 4)) void fc_stream_kernel(
    const uint8_t* __restrict__ weiq, const int8_t* __restrict__ xq, const float2* __restrict__ xsT, unsigned long long* slots, int Kg,
    int rows, int row_blocks, int strips, int tiled, int part_strips, int64_t N, float* __restrict__ y, const float* __restrict__ residual,
    int32_t* dump = nullptr) {
    constexpr int BM = 16 * RT, C = 2 * SW;
    constexpr int PT = 2 / SW, PH = (RT + PT - 1) / PT, LD = 32 * SW + 8;  // row tiles to a pass of the final sums, passes, row stride
    __shared__ __align__(16) float red[DUMP ? 1 : NW][16 * PT][LD];
    __shared__ __align__(16) float2 xsl[NW][64];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // uniform: block offsets stay scalar
    const int g = lane >> 4, jj = lane & 15;
    // slots != nullptr: two workgroups with half of K each; the halves meet through one 64-bit exchange per output (below).
    // Workgroups go to the XCDs round robin: the row blocks and halves of a strip follow one another on one XCD, whose L2 then
    // has its weights.
    const int per = slots ? 2 : 1;
    const int in = blockIdx.x % (8 * row_blocks * per), nb0 = (blockIdx.x / (8 * row_blocks * per) * 8 + (in & 7)) * SW;
    const int rb = (in >> 3) % row_blocks, split = (in >> 3) / row_blocks;
    if (nb0 >= strips) return;  // uniform for the workgroup
    const int row0 = rb * BM;
    const uint32_t Kp = (uint32_t)Kg * 128u;
    const int k_lo = slots ? (split * Kg) / 2 : 0, k_n = slots ? ((split + 1) * Kg) / 2 - k_lo : Kg;
    const int t0 = k_lo + (wave * k_n) / NW, t1 = k_lo + ((wave + 1) * k_n) / NW;  // this wave's k-groups

    v4f_r f[RT][C];
#pragma unroll
    for (int t = 0; t < RT; t++)
#pragma unroll
        for (int c = 0; c < C; c++) f[t][c] = v4f_r{0.f, 0.f, 0.f, 0.f};
    constexpr int kInit = DUMP ? 0 : kFoldBiasBits;
    v4i_r bias = {kInit, kInit, kInit, kInit};
    asm volatile("" : "+v"(bias));

    const uint32_t w_bytes = (uint32_t)Kg * (uint32_t)kRowsBlk, xq_bytes = (uint32_t)rows * Kp, xs_bytes = DUMP ? 0u : (uint32_t)Kg * (uint32_t)rows * 8u;
    const uint32_t lane_w = (uint32_t)(2 * g * kRowBytes + jj * 8), lane_s = (uint32_t)(jj * 4);
    uint32_t lane_a[RT], step_a[RT];
#pragma unroll
    for (int t = 0; t < RT; t++) {
        const int first = min(row0 + 16 * t, (rows - 1) & ~15), n = min(16, rows - first);  // (a tile past the last re-reads that one)
        lane_a[t] = tiled ? (uint32_t)first * Kp + (uint32_t)((g * n + min(jj, n - 1)) * 16) : (uint32_t)(first + min(jj, n - 1)) * Kp + 16u * g;
        step_a[t] = tiled ? (uint32_t)n * 64u : 64u;
    }
    const uint32_t lane_x = (uint32_t)min(rows - 1, row0 + min(lane, BM - 1)) * 8u;

    u32x2_r w[D][SW][2][2];     // [strip][64-k half][k8-row of the pair], the lane's column in either tile
    uint32_t dw[D][SW], mw[D][SW];  // the dwords that hold the fp16 scales / mins of the lane's two columns
    u32x2_r xs[D];               // (dx, gsum) of row `lane` of the block
    v4i_r a[D][RT][2];           // activation codes: row tile, 64-k half
    const uint8_t* strip = weiq + (int64_t)nb0 * w_bytes;
    auto load_w = [&](int kb, int i) {
        const bool wanted = kb < t1;
        const uint32_t sw = (uint32_t)kb * (uint32_t)kRowsBlk;
#pragma unroll
        for (int s = 0; s < SW; s++) {
            const buffer_rsrc rw = make_rsrc(strip + (int64_t)(s < strips - nb0 ? s : 0) * w_bytes, wanted ? w_bytes : 0u);
#pragma unroll
            for (int h = 0; h < 2; h++)
#pragma unroll
                for (int p = 0; p < 2; p++) w[i][s][h][p] = __builtin_amdgcn_raw_buffer_load_b64(rw, lane_w, sw + (uint32_t)((8 * h + p) * kRowBytes), 0);
            dw[i][s] = __builtin_amdgcn_raw_buffer_load_b32(rw, lane_s, sw + 2048u, 0);
            mw[i][s] = __builtin_amdgcn_raw_buffer_load_b32(rw, lane_s, sw + 2048u + 64u, 0);
        }
        xs[i] = __builtin_amdgcn_raw_buffer_load_b64(make_rsrc(xsT, wanted ? xs_bytes : 0u), lane_x, (uint32_t)kb * (uint32_t)rows * 8u, 0);
    };
    auto load_a = [&](int kb, int t, int i) {
        const buffer_rsrc rq = make_rsrc(xq, kb < t1 ? xq_bytes : 0u);
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(rq, lane_a[t], ((uint32_t)kb * 2u + h) * step_a[t], 0);
            a[i][t][h] = v4i_r{(int)v.x, (int)v.y, (int)v.z, (int)v.w};
        }
    };
    if constexpr (D == 1) {
        load_w(t0, 0);
#pragma unroll
        for (int t = 0; t < RT; t++) load_a(t0, t, 0);
    }
    auto compute = [&](int kb, int i) {
        // a lane holds results of 4 rows: their pairs go round through LDS (a wave's accesses to it stay in order)
        *reinterpret_cast<u32x2_r*>(&xsl[wave][lane]) = xs[i];
        asm volatile("" : : : "memory");
        v4i_r b[2][C];
        float d[C], m[C], nbd[C];
#pragma unroll
        for (int c = 0; c < C; c++) {
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const uint32_t pa = w[i][c >> 1][h][0][c & 1], pb = w[i][c >> 1][h][1][c & 1];
                b[h][c] = v4i_r{(int)lo4(pa), (int)hi4(pa), (int)lo4(pb), (int)hi4(pb)};
            }
            d[c] = f16_bits_to_f32((uint16_t)(dw[i][c >> 1] >> (16 * (c & 1)))), m[c] = f16_bits_to_f32((uint16_t)(mw[i][c >> 1] >> (16 * (c & 1))));
            asm volatile("" : "+v"(d[c]), "+v"(m[c]));
            nbd[c] = -kFoldBias * d[c];
        }
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (D == 1) load_w(kb + 1, 0);
        __builtin_amdgcn_sched_barrier(0);
        v4i_r acc[2][C];
        auto fold = [&](int t) {
            if constexpr (DUMP) {
#pragma unroll
                for (int c = 0; c < C; c++)
#pragma unroll
                    for (int v = 0; v < 4; v++) {
                        const int row_ = row0 + 16 * t + 4 * g + v, nb = nb0 + (c >> 1);
                        if (row_ < rows && nb < strips && kb < t1) dump[((int64_t)row_ * ((int64_t)strips * kGroupN) + nb * kGroupN + 2 * jj + (c & 1)) * Kg + kb] = acc[t & 1][c][v];
                    }
                return;
            }
            const float4 x01 = *reinterpret_cast<const float4*>(&xsl[wave][16 * t + 4 * g]), x23 = *reinterpret_cast<const float4*>(&xsl[wave][16 * t + 4 * g + 2]);
            const float dx[4] = {x01.x, x01.z, x23.x, x23.z}, gs[4] = {x01.y, x01.w, x23.y, x23.w};
#pragma unroll
            for (int c = 0; c < C; c++) {
                float u[4];
#pragma unroll
                for (int v = 0; v < 4; v++) u[v] = fmaf(__int_as_float(acc[t & 1][c][v]), d[c], nbd[c]);
#pragma unroll
                for (int v = 0; v < 4; v++) f[t][c][v] = fmaf(u[v], dx[v], f[t][c][v]);
#pragma unroll
                for (int v = 0; v < 4; v++) f[t][c][v] = fmaf(m[c], gs[v], f[t][c][v]);
            }
        };
#pragma unroll
        for (int t = 0; t < RT; t++) {
#pragma unroll
            for (int h = 0; h < 2; h++)
#pragma unroll
                for (int c = 0; c < C; c++) acc[t & 1][c] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[i][t][h], b[h][c], h == 0 ? bias : acc[t & 1][c], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (D == 1) load_a(kb + 1, t, 0);
            __builtin_amdgcn_sched_barrier(0);
            if (t > 0) fold(t - 1);
            __builtin_amdgcn_sched_barrier(0);
        }
        fold(RT - 1);
        asm volatile("" : : : "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    for (int kb = t0; kb < t1; kb += D) {
        if constexpr (D > 1) {
#pragma unroll
            for (int i = 0; i < D; i++) {
                load_w(kb + i, i);
#pragma unroll
                for (int t = 0; t < RT; t++) load_a(kb + i, t, i);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int i = 0; i < D; i++) compute(kb + i, i);  // (what was not wanted holds zeros and adds nothing)
    }
    if constexpr (DUMP) return;

    // the waves' sums meet in LDS, 1024 outputs at a time; one thread finishes each output
#pragma unroll
    for (int ph = 0; ph < PH; ph++) {
        if (ph > 0) __syncthreads();
#pragma unroll
        for (int i = 0; i < PT && ph * PT + i < RT; i++)
#pragma unroll
            for (int v = 0; v < 4; v++)
#pragma unroll
                for (int s = 0; s < SW; s++)
                    *reinterpret_cast<float2*>(&red[wave][16 * i + 4 * g + v][32 * s + 2 * jj]) = make_float2(f[ph * PT + i][2 * s][v], f[ph * PT + i][2 * s + 1][v]);
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 1024 / (NW * 64); i++) {
            const int idx = threadIdx.x + NW * 64 * i, row = idx / (32 * SW), col = idx % (32 * SW), nb = nb0 + (col >> 5);
            const int br = 16 * PT * ph + row, r = row0 + br, part = nb / part_strips;
            const int64_t n = (int64_t)(nb - part * part_strips) * kGroupN + (col & 31);
            if (br < BM && r < rows && nb < strips && n < N) {
                float v = 0.0f;
#pragma unroll
                for (int k = 0; k < NW; k++) v += red[k][row][col];
                if (slots != nullptr) {
                    // A slot is empty (0) or holds (1 << 32 | value bits).  Whoever finds the other half's value
                    // adds the two (a + b: the same bits whichever came first), stores the output and empties the
                    // slot for the next launch; whoever finds it empty has parked its own value and is done.
                    unsigned long long* slot = slots + ((int64_t)r * strips + nb) * kGroupN + (col & 31);
                    const unsigned long long parked = (1ull << 32) | (unsigned long long)__float_as_uint(v);
                    const unsigned long long old = __hip_atomic_exchange(slot, parked, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    if ((old >> 32) == 0ull) continue;
                    v += __uint_as_float((unsigned)(old & 0xFFFFFFFFull));
                    __hip_atomic_store(slot, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
                y[((int64_t)part * rows + r) * N + n] = residual ? v + residual[(int64_t)r * N + n] : v;
            }
        }
    }
}

// Which build: the least estimated time (us) of 1 .. 4 row tiles x one or two strips x 4 or 8 waves, K whole or in halves.  A
// round of workgroups takes 0.57 us and, per k-group of a wave, 0.10 + 0.038 RT * SW of latency and what the waves of its SIMD
// take together, 0.114 SW + 0.073 RT each; 0.35 RT * SW per workgroup of the compute unit at the end; halves 0.6 us and 4.9 us
// per million outputs; a workgroup that follows another alone on its compute unit 1.4 us; the weights 0.10 us per MB.  Fitted
// to all of these at 3 .. 512 rows of 13 shapes from 1024 x 512 to 22016 x 4096 and 11008 x 11008, weights from memory: the choices are
// 0.8 % slower than the best measured on average, 14 % at worst (256 x 4096 x 512, two strips where one is better, 9.3 against 8.2; above 4
// k-groups 8 %, 16 x 4096^2 in halves 7.3 against 6.7).
struct StreamPlan {
    int RT, SW, NW;
    bool split;
    double us;
};
static StreamPlan g_stream_forced{0, 0, 0, false, 0.0};  // RT > 0: that build (tests)
bool stream_forced() { return g_stream_forced.RT > 0; }
static StreamPlan plan_stream(int64_t rows, int64_t Ng, int64_t Kg, size_t slot_bytes) {
    // workgroups of 4 and of 8 waves that a compute unit holds, by the registers and LDS of [RT - 1][SW - 1]
    static const int kPlace[4][2][2] = {{{7, 3}, {4, 2}}, {{5, 2}, {3, 1}}, {{4, 2}, {2, 1}}, {{3, 1}, {2, 1}}};
    StreamPlan best{0, 0, 0, false, 0.0};
    if (stream_forced()) {
        best = g_stream_forced;
        best.split = best.split && Kg >= 2 && (size_t)rows * Ng * kGroupN * 8 <= slot_bytes;
        return best;
    }
    const bool may_split = g_rows_split && Kg >= 2 && (size_t)rows * Ng * kGroupN * 8 <= slot_bytes;
    // (a call plans more than once, and programs repeat their sizes: the last plan of the thread; 0.3 us each)
    static thread_local struct {
        int64_t rows = 0, Ng = 0, Kg = 0;
        bool may_split = false;
        StreamPlan plan{};
    } last;
    if (last.rows == rows && last.Ng == Ng && last.Kg == Kg && last.may_split == may_split) return last.plan;
    const unsigned strips = (unsigned)Ng, groups = (unsigned)Kg, n_rows = (unsigned)rows;  // (Ng <= kTicketBytes / 4, rows <= 2^25 here)
    const double stored = 0.103e-6 * (double)(Ng * Kg * kRowsBlk), exchange = 0.615 + 4.9e-6 * (double)(rows * Ng * kGroupN);
    for (int RT = 1; RT <= 4 && 16u * (RT - 1) < n_rows; RT++) {
        const unsigned blocks = (n_rows + 16 * RT - 1) / (16 * RT);
        for (int SW = 1; SW <= 2; SW++) {
            // (as many for every XCD: the strips go round them)
            const unsigned units = ((strips + SW - 1) / SW + 7) / 8 * 8 * blocks;
            const double step = 0.103 + 0.038 * RT * SW, wave = 0.25 * (0.114 * SW + 0.0733 * RT), write = 0.347 * RT * SW;
            for (int NW = 4; NW <= 8; NW += 4) {
                const unsigned place = kPlace[RT - 1][SW - 1][NW / 8];
                for (int split = 0; split <= (may_split ? 1 : 0); split++) {
                    const unsigned wgs = units << split, run = (((groups + split) >> split) + NW - 1) / NW;
                    const auto round = [&](unsigned n) { return 0.565 + run * (step + (double)(n * NW) * wave) + write * (double)n; };
                    const unsigned full = wgs / (256 * place), rest = wgs - full * 256 * place;
                    double us = (full ? (double)full * round(place) : 0.0) + (rest ? round((rest + 255) / 256) : 0.0) + stored;
                    if (split) us += exchange;
                    if (place == 1 && full > 0) us += 1.41 * (double)(rest ? full : full - 1);
                    if (best.RT == 0 || us < best.us) best = StreamPlan{RT, SW, NW, split != 0, us};
                }
            }
        }
    }
    last.rows = rows, last.Ng = Ng, last.Kg = Kg, last.may_split = may_split, last.plan = best;
    return best;
}

// what 32-bit offsets reach: codes, pairs, a strip
bool stream_fits(int64_t rows, int64_t Kg) {
    return rows * Kg * 128 < ((int64_t)1 << 32) && Kg * kRowsBlk < ((int64_t)1 << 32);
}

// estimated time of the kernel, without the quantization
double stream_estimate(int64_t rows, int64_t Ng, int64_t Kg, size_t slot_bytes) { return plan_stream(rows, Ng, Kg, slot_bytes).us; }

template <bool DUMP>
static int launch_stream(const StreamPlan& p, const uint8_t* w, const int8_t* xq, const float2* xsT, unsigned long long* slots, int64_t rows,
                         int64_t Ng, int64_t Kg, bool tiled, int64_t parts, int64_t N, float* y, const float* residual, int32_t* dump,
                         hipStream_t st) {
    const int64_t blocks = (rows + 16 * p.RT - 1) / (16 * p.RT), units = (Ng + p.SW - 1) / p.SW;
    const unsigned grid = (unsigned)((units + 7) / 8 * 8 * blocks * (p.split ? 2 : 1));
    unsigned long long* sl = p.split ? slots : nullptr;
    const bool pairs = ((Kg + p.split) / (p.split + 1) + p.NW - 1) / p.NW > 1;
#define LLMOPS_STREAM(RT, SW, NW, D)                                                                                                   \
    fc_stream_kernel<RT, SW, NW, D, DUMP><<<grid, NW * 64, 0, st>>>(w, xq, xsT, sl, (int)Kg, (int)rows, (int)blocks, (int)Ng, (int)tiled, \
                                                                    (int)(Ng / parts), N, y, residual, dump)
#define LLMOPS_STREAM_NW(RT, SW, D)                      \
    do {                                                 \
        if (p.NW == 4) LLMOPS_STREAM(RT, SW, 4, D);      \
        else LLMOPS_STREAM(RT, SW, 8, D);                \
    } while (0)
    // one row tile and strip: a wave's work on a k-group covers nothing of the memory's latency, two are asked for at a time (one by one
    // / two / four, us, weights from memory: 9 x 4096^2 7.24 / 7.05 / 7.46, 16 x 22016 x 4096 16.0 / 14.8 / 14.2, 16 x 4096 x 11008
    // 10.9 / 10.6, 64 x 512 x 4096 6.8 / 6.5 / 7.1; two row tiles at 64 x 4096^2 9.0 / 9.2, at 64 x 4096 x 11008 16.1 / 17.3)
    if (p.RT == 1 && p.SW == 1 && pairs) LLMOPS_STREAM_NW(1, 1, 2);
    else if (p.RT == 1 && p.SW == 1) LLMOPS_STREAM_NW(1, 1, 1);
    else if (p.RT == 1) LLMOPS_STREAM_NW(1, 2, 1);
    else if (p.RT == 2 && p.SW == 1) LLMOPS_STREAM_NW(2, 1, 1);
    else if (p.RT == 2) LLMOPS_STREAM_NW(2, 2, 1);
    else if (p.RT == 3 && p.SW == 1) LLMOPS_STREAM_NW(3, 1, 1);
    else if (p.RT == 3) LLMOPS_STREAM_NW(3, 2, 1);
    else if (p.SW == 1) LLMOPS_STREAM_NW(4, 1, 1);
    else LLMOPS_STREAM_NW(4, 2, 1);
#undef LLMOPS_STREAM_NW
#undef LLMOPS_STREAM
    LLMOPS_LAUNCH_CHECK();
    return LLMOPS_OK;
}

// group 128, activations already quantized (codes [rows, Kg*128], tiled: in the order of the loads; pairs [Kg][rows])
// parts > 1 (no residual): y is [parts][rows][N], part i the columns of strips i * Ng / parts ..
// `slots`: the zeroed exchange area of the FC workspace, `slot_bytes` of it
int launch_fc_rows(const uint8_t* w, const int8_t* xq, bool tiled, const float2* xsT, float* y, int64_t rows, int64_t Ng, int64_t Kg,
                   int64_t N, const float* residual, int64_t parts, unsigned long long* slots, size_t slot_bytes, hipStream_t st) {
    if (!stream_fits(rows, Kg)) return fail(LLMOPS_EINVAL, "the streaming MFMA kernel takes at most 4 GiB of codes and per strip");
    return launch_stream<false>(plan_stream(rows, Ng, Kg, slot_bytes), w, xq, xsT, slots, rows, Ng, Kg, tiled, parts, N, y, residual, nullptr, st);
}

// The same loop in its dump build, launched with the workgroup shape and K split that launch_fc_rows picks for
// these sizes, codes row by row.  The (scale, sum) pairs are not needed for the integer sums: their descriptor has size 0.
int launch_fc_rows_partials(const uint8_t* w, const int8_t* xq, int32_t* acc, int64_t rows, int64_t Ng, int64_t Kg,
                            hipStream_t st) {
    if (!stream_fits(rows, Kg)) return fail(LLMOPS_EINVAL, "the streaming MFMA kernel takes at most 4 GiB of codes and per strip");
    // (slots are only tested against nullptr in the dump build, never dereferenced)
    return launch_stream<true>(plan_stream(rows, Ng, Kg, LLMOPS_FC_COUNTER_BYTES - kTicketBytes), w, xq, nullptr, reinterpret_cast<unsigned long long*>(acc),
                               rows, Ng, Kg, false, 1, 0, nullptr, nullptr, acc, st);
}

}  // namespace llmops

extern "C" void llmops_test_fc_stream_set(int row_tiles, int strips, int waves, int halves) {
    if (!llmops::test_hooks_enabled(__func__)) return;
    const bool known = row_tiles >= 1 && row_tiles <= 4 && (strips == 1 || strips == 2) && (waves == 4 || waves == 8);
    llmops::g_stream_forced = known ? llmops::StreamPlan{row_tiles, strips, waves, halves != 0, 0.0} : llmops::StreamPlan{0, 0, 0, false, 0.0};
}
extern "C" int llmops_test_fc_stream_plan(int64_t rows, int64_t Ng, int64_t Kg, int* row_tiles, int* strips, int* waves, int* halves) {
    LLMOPS_TEST_HOOK();
    if (rows < 1 || Ng < 1 || Kg < 1 || !row_tiles || !strips || !waves || !halves) return LLMOPS_EINVAL;
    *row_tiles = 0;
    if (!llmops::streams(rows, Ng, Kg, 128)) return LLMOPS_OK;
    const llmops::StreamPlan p = llmops::plan_stream(rows, Ng, Kg, LLMOPS_FC_COUNTER_BYTES - llmops::kTicketBytes);
    *row_tiles = p.RT, *strips = p.SW, *waves = p.NW, *halves = p.split;
    return LLMOPS_OK;
}
extern "C" void llmops_test_fc_rows_set_split(int on) {
    if (llmops::test_hooks_enabled(__func__)) llmops::g_rows_split = on != 0;
}
