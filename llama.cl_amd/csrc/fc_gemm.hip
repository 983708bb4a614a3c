// Q4_1 x Q8 fully-connected product for many activation rows (prefill), group 128: int8 MFMA, and the planning and
// launching of the product for both group sizes (group 32: fc_gemm_g32.hip).
//
// Operand layout of v_mfma_i32_16x16x64_i8: lane = 16*g + jj; the A lane holds row jj, the B lane holds column jj, both
// for the same set of k-values chosen by g.  A packed block has 8 k-values of a column in a dword, k8-row after k8-row; lane
// (g, jj) takes the k8-rows 2g and 2g + 1 of columns 2*jj and 2*jj + 1 (one 8-byte read per k8-row), column 2*jj + c is its
// operand for MFMA number c.  Unpacking is two ANDs and a shift per dword; nothing is shuffled between lanes.
// One MFMA covers 8 k8-rows; two of them make one k-group.  Result register v of MFMA c: row 4*g + v, column 2*jj + c.
// After every k-group the int32 tile is folded into fp32 accumulators:
//   f += (d[n]*dx[row]) * float(acc) ; f += m[n]*gsum[row]        (fc_Q4A,
//   /root/reference/ops/op_fc.hpp:381-412; min term is m * raw group sum).
// The first term is computed as fma(fma(X, d, -B*d), dx, f): the
// int32 sums start at the bit pattern of the float B = 1.5 * 2^23, so the sum's register, read as a
// float X, IS B + sum (|sum| <= 128*15*127 < 2^22), and X*d - B*d = sum*d is exact before the fma's
// one rounding because B*d (2 significant bits times the 11 of an fp16) is itself a float.  Two
// vector instructions per output element and k-group instead of three (convert, multiply, fma).
#include "gemm_device.h"
#include "gemv_device.h"

namespace llmops {

// two adjacent results, columns n0 and n0 + 1 of n, (+ residual) to a row of stride ld
__device__ __forceinline__ void store_pair(float* dst, const float* res, float a, float b, int64_t n0, int64_t n, int64_t ld) {
    if (n0 + 1 < n && (ld & 3) == 0) {
        if (res) {
            const float2 r = *reinterpret_cast<const float2*>(res);
            a += r.x, b += r.y;
        }
        *reinterpret_cast<float2*>(dst) = make_float2(a, b);
    } else {
        if (n0 < n) dst[0] = res ? a + res[0] : a;
        if (n0 + 1 < n) dst[1] = res ? b + res[1] : b;
    }
}

// ---- split-K without a second launch -------------------------------------------------------------------
// Every split stores its tile of partial sums with device-scope (write-through) stores, waits for them and
// takes a ticket on the tile's counter; the split that draws the last ticket adds all splits' tiles in
// index order (so the sum does not depend on who arrives when), adds the residual and writes the result.
// Nobody waits for anybody.  Called by every thread of the workgroup, with LDS no longer in use once all have arrived.
// row0 / tile_rows: first row and row count of the tile; a thread holds rows 16t + 4g + v of it, columns
// 32*strip + 2*jj + c in f[t][c][v]; n0: where the first of them goes in a row of y_final.
// Where the sums of a tile lie: a row block's rows * Np floats strip by strip, a strip's rows in pairs, a pair as
// [jj][row of the pair][c]: 16 bytes per lane, 256 of them consecutive (and the last of an odd number of rows by itself, 8 bytes
// per lane).  Accesses of rows beyond `rows` fall outside the buffer descriptor (loads return 0, stores are dropped), as do
// those of strips beyond Ng.
// The last arrival works two row tiles at a time with all of its loads (up to SU splits x 8 rows) in flight
// together: the reduction then costs about T / 2 round trips to memory whatever the split count.  A split past
// the last is asked for through an empty descriptor: it returns 0 without touching memory.
template <int T, int SU>
__device__ __forceinline__ void splitk_finish(const v4f (&f)[T][2], float* __restrict__ out, int64_t split_stride, int64_t Np,
                                              int row0, int tile_rows, int strip, int Ng, int jj, int g, int rows,
                                              float* __restrict__ y_final, int64_t Ny, int64_t n0, const float* __restrict__ residual,
                                              unsigned* counter, int tid, unsigned* ticket_sh) {
    constexpr int kAgent = 16;  // sc1: coherent at device scope, as a relaxed atomic store / load would be
    const int S = (int)gridDim.z;
    const bool strip_ok = strip < Ng, odd = (tile_rows & 1) != 0;
    const uint32_t strip_bytes = strip_ok ? (uint32_t)tile_rows * (kGroupN * 4u) : 0u;
    float* base = out + (int64_t)row0 * Np + (int64_t)strip * kGroupN * tile_rows;
    // rows r = 16t + 4g + 2e and r + 1, or (last) r alone
    const auto place = [&](int t, int e) {
        const int r = t * 16 + 4 * g + 2 * e;
        return r + 1 < tile_rows ? (uint32_t)(r * (kGroupN * 4) + jj * 16) : 0xFFFFFF00u;
    };
    const auto place_last = [&](int t, int e) {
        const int r = t * 16 + 4 * g + 2 * e;
        return r + 1 == tile_rows ? (uint32_t)(r * (kGroupN * 4) + jj * 8) : 0xFFFFFF00u;
    };
    {
        const buffer_rsrc rs = make_rsrc(base + (int64_t)blockIdx.z * split_stride, strip_bytes);
#pragma unroll
        for (int t = 0; t < T; t++)
#pragma unroll
            for (int e = 0; e < 2; e++) {
                const u32x4 val = {__float_as_uint(f[t][0][2 * e]), __float_as_uint(f[t][1][2 * e]), __float_as_uint(f[t][0][2 * e + 1]),
                                   __float_as_uint(f[t][1][2 * e + 1])};
                __builtin_amdgcn_raw_buffer_store_b128(val, rs, place(t, e), 0, kAgent);
                if (odd) __builtin_amdgcn_raw_buffer_store_b64(v2u{val[0], val[1]}, rs, place_last(t, e), 0, kAgent);
            }
    }
    __builtin_amdgcn_s_waitcnt(0);  // this wave's stores have been acknowledged
    __syncthreads();
    if (tid == 0) *ticket_sh = __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    if (*ticket_sh != (unsigned)(S - 1)) return;
    if (tid == 0) __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // next launch
    if (!strip_ok) return;
#pragma unroll
    for (int t = 0; t < T; t += 2) {
        float a[4][4];
#pragma unroll
        for (int p = 0; p < 4; p++)
#pragma unroll
            for (int v = 0; v < 4; v++) a[p][v] = 0.0f;
        for (int s0 = 0; s0 < S; s0 += SU) {
            u32x4 pv[SU][4];
#pragma unroll
            for (int u = 0; u < SU; u++) {
                const buffer_rsrc rs = make_rsrc(base + (int64_t)min(s0 + u, S - 1) * split_stride, s0 + u < S ? strip_bytes : 0u);
#pragma unroll
                for (int p = 0; p < 4; p++) pv[u][p] = __builtin_amdgcn_raw_buffer_load_b128(rs, place(t + (p >> 1), p & 1), 0, kAgent);
            }
#pragma unroll
            for (int u = 0; u < SU; u++)
#pragma unroll
                for (int p = 0; p < 4; p++)
#pragma unroll
                    for (int v = 0; v < 4; v++) a[p][v] += __uint_as_float(pv[u][p][v]);
        }
        if (odd && t * 16 + 32 >= tile_rows && t * 16 < tile_rows) {
            for (int sp = 0; sp < S; sp++) {
                const buffer_rsrc rs = make_rsrc(base + (int64_t)sp * split_stride, strip_bytes);
#pragma unroll
                for (int p = 0; p < 4; p++) {
                    const v2u last = __builtin_amdgcn_raw_buffer_load_b64(rs, place_last(t + (p >> 1), p & 1), 0, kAgent);
                    a[p][0] += __uint_as_float(last[0]), a[p][1] += __uint_as_float(last[1]);
                }
            }
        }
#pragma unroll
        for (int p = 0; p < 4; p++)
#pragma unroll
            for (int i = 0; i < 2; i++) {
                const int row = row0 + (t + (p >> 1)) * 16 + 4 * g + 2 * (p & 1) + i;
                if (row < rows)
                    store_pair(y_final + (int64_t)row * Ny + n0, residual ? residual + (int64_t)row * Ny + n0 : nullptr, a[p][2 * i], a[p][2 * i + 1], n0, Ny, Ny);
            }
    }
}

// ---- the tiled kernel -------------------------------------------------------------------------------
// What bounds it: everything at once.  Per k-group and 128 x 128 tile a wave has 32 int8 MFMAs (512 cycles), 128 fold
// instructions and about 40 others (600 cycles and more of vector issue, which the int8 MFMA shares only in part: 395 cycles
// for two waves' 4 x 32x32x32 and 32 fold instructions each, against 263 and 193 alone), 26 KB of LDS reads and 6.4 KB
// of copies.  With parts left out (2048 x 11008 x 4096, 163 us at that point): no copies 141, no code reads 151, no fold 133,
// no MFMA 133, neither 114, copies alone 107.  So each is kept small, and two to four workgroups share a compute unit so that
// one's waits are another's work:
//   * tile 32*RT rows x 128 columns, four waves side by side, a strip each: a strip's weights are unpacked by one wave only
//     (2 x 2 waves of 64 x 64 unpack twice as much: 32-row tiles 2 to 7 % slower, 128 rows even), codes are read by all four.
//     (The weights as the A operand, a row and eight adjacent columns in a lane: 2 % faster with 128 rows, but eight scales to
//     convert instead of two, 2 to 6 % slower with 32 and 64.)
//   * codes, nibbles, scales, sums and mins are copied to LDS asynchronously (global_load_lds), asked for two k-groups before
//     they are multiplied and waited for one k-group later, where everyone passes the same barrier: what is on its way has the
//     time of one k-group.  No registers, no LDS store instructions.  (Through registers: 5 to 13 % slower, 512 x 22016 x
//     4096 103 us against 90.)  Codes, scales and nibbles have three slots; sums and mins six, since the min term is formed
//     for four k-groups together.
//   * the first operands of a k-group are read from LDS while the last row tiles of the one before are multiplied, and the
//     fold of one pair of row tiles runs beside the products of the next: the order is pinned.
// A 256 x 128 tile with two wave groups (one workgroup per compute unit, 20 % less to copy) takes 165 to 170 us at
// 2048 x 11008 x 4096 where 128 rows take 156: nothing covers its barriers, its first fetch and its stores.
// Measured, us for the whole call in a graph, kernels before (weights and codes through registers below 512 rows, two wave
// groups in alternating phases from there on) and now: 128 x 4096 x 11008 27.5 / 23.4, 300 x 4090 x 11008 46 / 39, 512 x 4096^2
// 33.8 / 27.7, 512 x 22016 x 4096 102.5 / 90, 512 x 4096 x 11008 57 / 53, 2048 x 11008 x 4096 164 / 157, 2048 x 4096 x 11008 153 / 151.
constexpr int kBlk128 = 2176;
constexpr int kStages = 3;    // LDS slots of a k-group: one is multiplied, one has landed (its first operands are read), one is on its way
constexpr int kMinRing = 6;   // LDS slots of sums and mins: the last four k-groups and the two ahead
template <int RT>
struct GemmTile {
    static constexpr int BM = RT * 32;
    static constexpr int T = BM / 16;  // row tiles of a wave: all of them
    struct Stage {
        uint8_t a[BM * 128];     // codes
        uint8_t b[4 * 2048];     // nibbles of the four strips
        uint16_t d[4 * 32];      // their scales
        float dx[BM];            // the rows' scales
    };
    Stage st[kStages];
    float gs[kMinRing][BM];      // the rows' sums
    uint16_t m[kMinRing][4 * 32];  // the strips' mins
};

template <int RT, bool PARTIALS>
__global__ __launch_bounds__(256, (RT == 4 ? 2 : (RT == 2 ? 3 : 4))) void fc_gemm_tile_kernel(
    const uint8_t* __restrict__ weiq, const int8_t* __restrict__ xq, const float* __restrict__ xd, const float* __restrict__ gs,
    const float2* __restrict__ xsT, float* __restrict__ out, int32_t* __restrict__ out_i, int Ng, int Kg, int64_t ldo, int64_t N,
    int rows, int kb_per_split, int64_t split_stride, const float* __restrict__ residual, float* __restrict__ y_final, int64_t Ny,
    int part_strips, unsigned* __restrict__ counters) {
    using Tile = GemmTile<RT>;
    constexpr int BM = Tile::BM, T = Tile::T;
    extern __shared__ __align__(16) uint8_t smem_raw[];
    Tile& sm = *reinterpret_cast<Tile*>(smem_raw);

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = lane >> 4, jj = lane & 15;
    // Which tile: workgroups go to the 8 XCDs round robin, each XCD has its own L2, and an XCD runs
    // about 32 CUs x (workgroups per CU) workgroups at a time.  The tiles are therefore numbered so that
    // each XCD gets one contiguous run of them and a run walks the tile grid in bands of 8 row blocks,
    // rows fastest: the workgroups resident on one XCD then cover about 8 row blocks x 8..16 column
    // blocks and every activation and weight tile is fetched into that L2 once instead of once per
    // workgroup.  (With column blocks fastest across the whole chip the weights, re-read by every row
    // block, came from beyond the L2 each time.)
    const int nbx = (Ng + 3) / 4, nby = (rows + BM - 1) / BM;
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
    const int strip0 = bx * 4;
    const int row0 = by * BM;
    const int kb0 = blockIdx.z * kb_per_split, kb1 = min(Kg, kb0 + kb_per_split);
    const int64_t Kp = (int64_t)Kg * 128;

    // ---- what this wave copies per k-group (rows and strips past the end re-read the last one that exists) ----
    // codes: BM / 4 rows, 8 rows of 128 bytes to a copy.  16-byte chunk c of row r lies at position c ^ key(r), key(r) =
    // (r >> 1) & 7.  A ds_read_b128 serves lanes 0-3, 12-15 and 20-27 together, then 4-11, 16-19 and 28-31, and so on: rows and
    // chunks of such sixteen fall on 16 different bank groups.  (With a key that spreads 16 consecutive lanes only,
    // (r + (r >> 3)) & 7, every one of these reads took twice its time: a third of all LDS cycles, 2048 x 4096 x 11008 153.7 us against 151.)
    constexpr int AC = RT;
    const uint8_t* abase = reinterpret_cast<const uint8_t*>(xq) + (int64_t)row0 * Kp;
    uint32_t aoff[AC];
#pragma unroll
    for (int i = 0; i < AC; i++) {
        const int r = (wave * AC + i) * 8 + (lane >> 3), key = (r >> 1) & 7;
        aoff[i] = (uint32_t)(min(rows - 1, row0 + r) - row0) * (uint32_t)Kp + (uint32_t)(((lane & 7) ^ key) * 16);
    }
    // nibbles: 8 k8-rows of 128 bytes to a copy, row 2g + p of the eight at place 4p + g: the rows that the lane groups
    // g = 0..3 read together lie side by side
    constexpr int BC = 2;
    const uint8_t* tbase = weiq + (int64_t)strip0 * Kg * kBlk128;
    const auto strip_off = [&](int s) { return (uint32_t)(min(Ng - 1, strip0 + s) - strip0) * (uint32_t)Kg * (uint32_t)kBlk128; };
    uint32_t boff[BC];
#pragma unroll
    for (int i = 0; i < BC; i++) {
        const int c = wave * BC + i, place = lane >> 3;
        boff[i] = strip_off(c >> 1) + (uint32_t)((c & 1) * 1024 + (2 * (place & 3) + (place >> 2)) * 128 + (lane & 7) * 16);
    }
    // the rows' scales and sums, 64 rows to a copy, then the strips' scales and mins: copies 0 .. 2*XC+1, one or two per wave
    constexpr int XC = BM > 64 ? BM / 64 : 1;
    const uint8_t* sbase[2] = {nullptr, nullptr};
    uint32_t soff[2] = {0, 0}, sdst[2] = {0, 0}, sring[2] = {0, 0};
    int64_t sstep[2] = {0, 0};
    bool slive[2];
    const uint32_t lds0 = lds_off(smem_raw);
#pragma unroll
    for (int u = 0; u < 2; u++) {
        const int s = wave + u * 4;
        slive[u] = s < 2 * XC + 2;
        if (s < 2 * XC) {
            const bool sums = s >= XC;
            const int part = sums ? s - XC : s, row = min(rows - 1, row0 + part * 64 + min(lane, BM - 1));
            if (PARTIALS) slive[u] = false;
            if (xsT != nullptr) {
                sbase[u] = reinterpret_cast<const uint8_t*>(xsT) + (sums ? 4 : 0);
                soff[u] = (uint32_t)row * 8u, sstep[u] = (int64_t)rows * 8;
            } else {
                sbase[u] = reinterpret_cast<const uint8_t*>((sums ? gs : xd) + (int64_t)row0 * Kg);
                soff[u] = (uint32_t)(row - row0) * (uint32_t)Kg * 4u, sstep[u] = 4;
            }
            sring[u] = sums ? BM * 4 : 0;
            sdst[u] = (sums ? lds_off(&sm.gs[0][0]) : lds_off(&sm.st[0].dx[0])) + part * 256;
        } else {
            const bool mins = s == 2 * XC + 1;
            sbase[u] = tbase + 2048 + (mins ? 64 : 0);
            soff[u] = strip_off(lane >> 4) + (uint32_t)(lane & 15) * 4u, sstep[u] = kBlk128;
            sring[u] = mins ? 256 : 0;
            sdst[u] = mins ? lds_off(&sm.m[0][0]) : lds_off(&sm.st[0].d[0]);
        }
    }
    auto copy_stage = [&](int kb, int slot, int ring) {
        const uint32_t base = uniform_u32(lds0 + slot * (int)sizeof(typename Tile::Stage));
        const uint8_t* as = abase + (int64_t)kb * 128;
#pragma unroll
        for (int i = 0; i < AC; i++) copy16_to_lds(as, aoff[i], base + (wave * AC + i) * 1024);
        const uint8_t* bs = tbase + (int64_t)kb * kBlk128;
#pragma unroll
        for (int i = 0; i < BC; i++) copy16_to_lds(bs, boff[i], base + BM * 128 + (wave * BC + i) * 1024);
#pragma unroll
        for (int u = 0; u < 2; u++)
            if (slive[u]) {  // (uniform)
                const uint32_t dst = uniform_u32(sdst[u] + (sring[u] != 0 ? ring * sring[u] : slot * (uint32_t)sizeof(typename Tile::Stage)));
                const void* from = uniform_ptr(sbase[u] + (int64_t)kb * sstep[u]);
                if (RT > 1) copy4_to_lds(from, soff[u], dst);
                else if (lane < 32 || wave >= 2) copy4_to_lds(from, soff[u], dst);  // (32 rows; the strips' copies are whole)
            }
    };

    v4f f[T][2];
#pragma unroll
    for (int t = 0; t < T; t++)
#pragma unroll
        for (int c = 0; c < 2; c++) f[t][c] = v4f{0.f, 0.f, 0.f, 0.f};
    // the sums start at the bit pattern of 1.5 * 2^23, so that the fold needs no convert instruction
    constexpr int kInit = PARTIALS ? 0 : kFoldBiasBits;
    v4i bias = {kInit, kInit, kInit, kInit};
    asm volatile("" : "+v"(bias));  // (in registers once, not set up for every product)

#pragma unroll
    for (int i = 0; i < kStages - 1; i++)
        if (kb0 + i < kb1) copy_stage(kb0 + i, i, i);

    const int akey = jj >> 1;
    const int a_rd[2] = {jj * 128 + ((g ^ akey) * 16), jj * 128 + (((4 + g) ^ akey) * 16)};
    const int b_rd = wave * 2048 + g * 128 + jj * 8;
    // what the next k-group starts with is read while the last row tiles of this one are multiplied
    v4i a[2][2][2];  // [pair of row tiles, odd or even][tile][k half]
    uint2 wraw[2][2];
    uint32_t dh;
    constexpr int P = T / 2;
    auto load_a = [&](const typename Tile::Stage& st, int p) {
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int h = 0; h < 2; h++) a[p & 1][i][h] = *reinterpret_cast<const v4i*>(&st.a[a_rd[h] + (2 * p + i) * 2048]);
    };
    auto load_first = [&](const typename Tile::Stage& st) {
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int h = 0; h < 2; h++) a[P & 1][i][h] = *reinterpret_cast<const v4i*>(&st.a[a_rd[h] + i * 2048]);
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
            for (int p = 0; p < 2; p++) wraw[h][p] = *reinterpret_cast<const uint2*>(&st.b[b_rd + h * 1024 + p * 512]);
        dh = *reinterpret_cast<const uint32_t*>(&st.d[wave * 32 + jj * 2]);
    };
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" : : : "memory");
    load_first(sm.st[0]);
    int slot = 0, ring = 0, since = 0;  // since: k-groups whose min term is not in yet
    for (int kb = kb0; kb < kb1; kb++) {
        // this wave's copies for k-group kb + 1 have landed, then everyone's; the slot of kb - 1 is free
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" : : : "memory");
        if (kb + 2 < kb1) copy_stage(kb + 2, slot == 0 ? 2 : slot - 1, ring >= kMinRing - 2 ? ring + 2 - kMinRing : ring + 2);
        const typename Tile::Stage& st = sm.st[slot];
        slot = slot == kStages - 1 ? 0 : slot + 1;

        v4i b[2][2];
#pragma unroll
        for (int h = 0; h < 2; h++) {
            b[h][0] = v4i{(int)lo4(wraw[h][0].x), (int)hi4(wraw[h][0].x), (int)lo4(wraw[h][1].x), (int)hi4(wraw[h][1].x)};
            b[h][1] = v4i{(int)lo4(wraw[h][0].y), (int)hi4(wraw[h][0].y), (int)lo4(wraw[h][1].y), (int)hi4(wraw[h][1].y)};
        }
        if (P & 1) {
#pragma unroll
            for (int i = 0; i < 2; i++)
#pragma unroll
                for (int h = 0; h < 2; h++) a[0][i][h] = a[1][i][h];
        }
        float d[2] = {f16_bits_to_f32((uint16_t)(dh & 0xFFFFu)), f16_bits_to_f32((uint16_t)(dh >> 16))}, nbd[2];
#pragma unroll
        for (int c = 0; c < 2; c++) {
            asm volatile("" : "+v"(d[c]));  // (converted once: v_fma_mix runs at half the rate of v_fma)
            nbd[c] = -kFoldBias * d[c];
        }

        v4i acc[2][2][2];  // [pair][tile][c]
        float4 x[2][2];
        auto mma = [&](int p) {
#pragma unroll
            for (int h = 0; h < 2; h++)
#pragma unroll
                for (int i = 0; i < 2; i++)
#pragma unroll
                    for (int c = 0; c < 2; c++)
                        acc[p & 1][i][c] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[p & 1][i][h], b[h][c], h == 0 ? bias : acc[p & 1][i][c], 0, 0, 0);
        };
        auto fold = [&](int p) {
#pragma unroll
            for (int i = 0; i < 2; i++) {
                const int t = 2 * p + i;
                if (PARTIALS) {
                    const int strip = strip0 + wave;
#pragma unroll
                    for (int v = 0; v < 4; v++) {
                        const int row = row0 + t * 16 + g * 4 + v;
                        if (strip >= Ng || row >= rows) continue;
#pragma unroll
                        for (int c = 0; c < 2; c++)
                            out_i[((int64_t)row * ((int64_t)Ng * kGroupN) + strip * kGroupN + 2 * jj + c) * Kg + kb] = acc[p & 1][i][c][v];
                    }
                    continue;
                }
                const float dxv[4] = {x[p & 1][i].x, x[p & 1][i].y, x[p & 1][i].z, x[p & 1][i].w};
#pragma unroll
                for (int v = 0; v < 4; v++)
#pragma unroll
                    for (int c = 0; c < 2; c++)
                        f[t][c][v] = fmaf(fmaf(__int_as_float(acc[p & 1][i][c][v]), d[c], nbd[c]), dxv[v], f[t][c][v]);
                // (register arithmetic, which the compiler would gather behind the last product)
                asm volatile("" : "+v"(f[t][0]), "+v"(f[t][1]));
            }
        };
#pragma unroll
        for (int p = 0; p < P; p++) {
            if (p + 1 < P) load_a(st, p + 1);
            if (!PARTIALS) {
                // dx of the 4 rows this lane holds results for: rows 16t + 4g + v
#pragma unroll
                for (int i = 0; i < 2; i++) x[p & 1][i] = *reinterpret_cast<const float4*>(&st.dx[(2 * p + i) * 16 + g * 4]);
            }
            mma(p);
            __builtin_amdgcn_sched_barrier(0);
            if (p == P - 1) load_first(sm.st[slot]);  // (past the last k-group: what the slot still holds, unused)
            if (p > 0) {
                fold(p - 1);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        fold(P - 1);
        if (!PARTIALS && (since == 3 || kb + 1 == kb1)) {
            // Min term sum_kb m[n,kb]*gsum[row,kb]: a rank-Kg product, done four k-groups at a time straight into the fp32
            // accumulators by v_mfma_f32_16x16x4_f32; lane (jj, g) has gsum of row jj and m of its columns for the group with
            // index g of the four.  (On the bf16 matrix cores, both factors in exact pieces, it is no faster -- 2048 x 11008 x 4096
            // 158.7 to 159.9 us against 160.1 to 162.9, 2048 x 4096 x 11008 151.5 against 151 -- and its sums lose more: rms error
            // against 64 bits 1.85e-7 of the outputs at K = 4096 where this has 1.62e-7.)
            int mine = ring - since + g;
            mine += mine < 0 ? kMinRing : 0;
            const bool live = g <= since;
            const uint32_t mh = *reinterpret_cast<const uint32_t*>(&sm.m[live ? mine : 0][wave * 32 + jj * 2]);
            const float* gsr = &sm.gs[live ? mine : 0][jj];
            float gv[T];
#pragma unroll
            for (int t = 0; t < T; t++) gv[t] = gsr[t * 16];
            __builtin_amdgcn_sched_barrier(0);
            float mv[2];
#pragma unroll
            for (int c = 0; c < 2; c++) mv[c] = live ? f16_bits_to_f32((uint16_t)(c == 0 ? mh & 0xFFFFu : mh >> 16)) : 0.0f;
#pragma unroll
            for (int t = 0; t < T; t++) {
                gv[t] = live ? gv[t] : 0.0f;
#pragma unroll
                for (int c = 0; c < 2; c++) f[t][c] = __builtin_amdgcn_mfma_f32_16x16x4f32(gv[t], mv[c], f[t][c], 0, 0, 0);
            }
        }
        since = since == 3 ? 0 : since + 1;
        ring = ring == kMinRing - 1 ? 0 : ring + 1;
    }

    if (PARTIALS) return;
    const int strip = strip0 + wave;
    // results in parts: part_strips strips to a dense matrix of its own (of partial sums only the finished ones are)
    const int part = strip / part_strips;
    const int64_t n0 = (int64_t)(strip - part * part_strips) * kGroupN + 2 * jj;
    if (counters != nullptr) {
        splitk_finish<T, (RT == 4 ? 12 : (RT == 2 ? 6 : 4))>(f, out, split_stride, ldo, row0, min(BM, rows - row0), strip, Ng, jj, g,
                                                            rows, y_final + (int64_t)part * rows * Ny, Ny, n0, residual, &counters[by * nbx + bx], tid,
                                                            reinterpret_cast<unsigned*>(smem_raw));
        return;
    }
    if (strip >= Ng) return;
    float* o = out + (int64_t)blockIdx.z * split_stride + (int64_t)part * rows * ldo;
#pragma unroll
    for (int t = 0; t < T; t++)
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const int row = row0 + t * 16 + g * 4 + v;
            if (row >= rows) continue;
            // residual != nullptr only without split-K: then o is the result itself, row stride ldo
            store_pair(o + (int64_t)row * ldo + n0, residual ? residual + (int64_t)row * ldo + n0 : nullptr, f[t][0][v], f[t][1][v], n0, N, ldo);
        }
}

// y[p][row][n] = sum over splits (index order) of part[s][row][p * N + n] (+ residual[row][n]); four columns per
// thread (the partial sums' row stride ldp is a multiple of 32 floats, so their 16-byte loads are aligned)
__global__ void gemm_reduce_kernel(const float* __restrict__ part, float* __restrict__ y, int64_t rows, int64_t N,
                                   int64_t ldp, int64_t split_stride, int S, const float* __restrict__ residual) {
    const int64_t nq = (N + 3) / 4;
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= rows * nq) return;
    const int64_t r = i / nq, n = (i % nq) * 4, p = blockIdx.y;
    float4 a = make_float4(0.f, 0.f, 0.f, 0.f);
    part += p * N;
    float* dst = y + (p * rows + r) * N + n;
    const float* res = residual ? residual + r * N + n : nullptr;
    const bool whole = n + 3 < N && (N & 3) == 0;
    float4 r4 = make_float4(0.f, 0.f, 0.f, 0.f);
    if (whole && res) r4 = *reinterpret_cast<const float4*>(res);
    // four splits' loads in flight at a time (a split past the last re-reads the last and is not added)
    for (int s0 = 0; s0 < S; s0 += 4) {
        float4 v[4];
#pragma unroll
        for (int u = 0; u < 4; u++)
            v[u] = *reinterpret_cast<const float4*>(part + (int64_t)min(s0 + u, S - 1) * split_stride + r * ldp + n);
#pragma unroll
        for (int u = 0; u < 4; u++)
            if (s0 + u < S) a.x += v[u].x, a.y += v[u].y, a.z += v[u].z, a.w += v[u].w;
    }
    if (whole) {
        if (res) a.x += r4.x, a.y += r4.y, a.z += r4.z, a.w += r4.w;
        *reinterpret_cast<float4*>(dst) = a;
    } else {
        const float av[4] = {a.x, a.y, a.z, a.w};
        for (int c = 0; c < 4; c++)
            if (n + c < N) dst[c] = res ? av[c] + res[c] : av[c];
    }
}

int plan_gemm_g32(int64_t rows, int64_t Ng, int64_t Kg, int force_split, int* st_per_split);
int launch_gemm_g32(const uint8_t* w, const int8_t* xq, const float* xd, const float* gs, const float2* xsT, float* out, int64_t Ng,
                    int64_t Kg, int64_t ldo, int64_t N, int64_t rows, int st_per_split, int S, int64_t split_stride,
                    const float* residual, hipStream_t st);
int launch_gemm_g32_partials(const uint8_t* w, const int8_t* xq, int32_t* acc, int64_t rows, int64_t Ng, int64_t Kg, hipStream_t st);

struct GemmPlan {
    int RT, S, kb_per_split;  // rows of a tile / 32; group 32: RT = 1 (32-row tiles), kb_per_split in stages of four k-groups
    bool lds;
};

static int g_gemm_rt = 0;  // 0 = choose per shape; 1, 2, 4 = that tile; -1 = also what the weight-streaming kernel would take
static int g_gemm_fused_reduce = 1;  // split-K partial sums added by the product kernel itself (0: by a second launch)
static int g_gemm_force_split = 0;   // > 0: the split-K factor to use whatever the estimate says (tests)
bool gemm_rows_kernel_enabled() { return g_gemm_rt >= 0; }
bool gemm_tile_forced() { return g_gemm_rt != 0 || g_gemm_force_split > 0; }

// Row tile and split-K factor of the tiled kernel: the least estimated time (us) of 128, 64 or 32 rows x 1 .. 12 splits.  A
// k-group of a resident round takes 1.2 / 0.95 / 0.81 us (two, three, four workgroups per compute unit), a workgroup
// counts as its run plus 0.3 k-groups, and a round that is not full takes 1 / 0.54 / 0.85 of that plus the rest in
// proportion; the last split of a tile to arrive adds the sums (1.7 us, 0.32 more per split and 32 rows, 0.42 us per million of them).
// Fitted to every tile x {1 .. 8, 10, 11} splits at 17 row counts from 24 to 2048 of 4096^2, 11008 | 22016 x 4096, 4096 x 11008 and
// 1500 x 2048: the choices are 1.4 % slower than the best measured one on average and 8 % at worst (11008 x 4096 at 64 rows: 5 splits,
// 4 would be better), against 5 % and 65 % (1500 x 2048 at 384 rows) of the rule that counted whole rounds.
// room: what partial sums may take (bytes).
template <typename I>
static double plan_gemm_tile_in(I rows, I Ng, I Kg, int64_t room, GemmPlan& p) {
    static const int kRT[3] = {4, 2, 1}, kSlots[3] = {512, 768, 1024};
    static const double kGroupUs[3] = {1.2, 0.947, 0.811}, kPartRound[3] = {1.0, 0.541, 0.852};
    double best = 0.0;
    const double part_us = 0.42e-6 * (double)rows * (double)(Ng * kGroupN);
    for (int i = 0; i < 3; i++) {
        if (g_gemm_rt > 0 && kRT[i] != g_gemm_rt) continue;
        const I bm = 32 * kRT[i], tiles = ((Ng + 3) / 4) * ((rows + bm - 1) / bm), slots = kSlots[i];
        I last = 0;
        for (I s = 1; s <= 12; s++) {
            const I want = g_gemm_force_split > 0 ? (I)g_gemm_force_split : s;
            const I per = want >= Kg ? 1 : (Kg + want - 1) / want;
            if (per == last) continue;
            last = per;
            const I S = (Kg + per - 1) / per;
            if (S > 1 && g_gemm_force_split <= 0 && (int64_t)S * (int64_t)rows * (int64_t)Ng * kGroupN * 4 > room) continue;
            const I full = tiles * S / slots, rest = tiles * S - full * slots;
            const double rounds = (double)full + (rest == 0 ? 0.0 : kPartRound[i] + (1.0 - kPartRound[i]) * (double)rest / kSlots[i]);
            double t = kGroupUs[i] * ((double)per + 0.289) * rounds;
            if (S > 1) t += 1.726 + 0.319 * (double)(S * kRT[i]) + (double)S * part_us;
            if (best == 0.0 || t < best) {
                best = t;
                p.RT = kRT[i], p.S = (int)S, p.kb_per_split = (int)per;
            }
        }
    }
    return best;
}

static double plan_gemm_tile(int64_t rows, int64_t Ng, int64_t Kg, int64_t room, GemmPlan& p) {
    // (a call plans up to three times, and programs repeat their sizes: the last plan of the thread; 0.2 us each)
    static thread_local struct {
        int64_t rows = 0, Ng = 0, Kg = 0, room = 0;
        int rt = 0, split = 0;
        GemmPlan plan{};
        double us = 0.0;
    } last;
    if (last.rows != rows || last.Ng != Ng || last.Kg != Kg || last.room != room || last.rt != g_gemm_rt || last.split != g_gemm_force_split) {
        last.us = rows * Ng < ((int64_t)1 << 31) && Kg < ((int64_t)1 << 24)
                      ? plan_gemm_tile_in<unsigned>((unsigned)rows, (unsigned)Ng, (unsigned)Kg, room, last.plan)
                      : plan_gemm_tile_in<int64_t>(rows, Ng, Kg, room, last.plan);
        last.rows = rows, last.Ng = Ng, last.Kg = Kg, last.room = room, last.rt = g_gemm_rt, last.split = g_gemm_force_split;
    }
    p.RT = last.plan.RT, p.S = last.plan.S, p.kb_per_split = last.plan.kb_per_split;
    return last.us;
}

// estimated time of the tiled kernel (group 128), us
double gemm_tile_estimate(int64_t rows, int64_t Ng, int64_t Kg) {
    GemmPlan p;
    return plan_gemm_tile(rows, Ng, Kg, INT64_MAX, p);
}

static GemmPlan plan_gemm(int64_t rows, int64_t Ng, int64_t Kg, int G, int64_t room) {
    GemmPlan p;
    p.lds = (G == 128);
    if (p.lds) {
        plan_gemm_tile(rows, Ng, Kg, room, p);
    } else {
        p.RT = 1;
        p.S = plan_gemm_g32(rows, Ng, Kg, g_gemm_force_split, &p.kb_per_split);
    }
    return p;
}

size_t gemm_workspace_bytes(int64_t rows, int64_t Ng, int64_t Kg, int G, int64_t room) {
    const GemmPlan p = plan_gemm(rows, Ng, Kg, G, room);
    return p.S > 1 ? (size_t)p.S * rows * Ng * kGroupN * sizeof(float) : 0;
}

// the kernel's launch needs more than 64 KiB of dynamic LDS: opted in to once per build of it
template <int RT, bool PARTIALS>
static int configure_gemm_tile() {
    static bool configured = false;
    if (!configured) {
        LLMOPS_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(&fc_gemm_tile_kernel<RT, PARTIALS>),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)sizeof(GemmTile<RT>)));
        configured = true;
    }
    return LLMOPS_OK;
}

template <int RT>
static int launch_gemm_tile(const uint8_t* w, const int8_t* xq, const float* xd, const float* gs, const float2* xsT,
                            float* out, int64_t Ng, int64_t Kg, int64_t ldo, int64_t N, int64_t rows, const GemmPlan& p,
                            int64_t split_stride, const float* residual, float* y_final, int64_t Ny, int64_t part_strips,
                            unsigned* counters, hipStream_t st) {
    const int bad = configure_gemm_tile<RT, false>();
    if (bad) return bad;
    // (the copies take 32-bit offsets into the scale pairs of a k-group and into a tile's rows and strips)
    if (rows * Kg * 8 >= ((int64_t)1 << 32) || Kg * 128 * 128 >= ((int64_t)1 << 32))
        return fail(LLMOPS_EINVAL, "fc_Q4A: rows * Kg must be below 2^29 for the tiled kernel");
    const int64_t tiles = ((Ng + 3) / 4) * ((rows + RT * 32 - 1) / (RT * 32));
    dim3 grid((unsigned)(8 * ((tiles + 7) / 8)), 1, (unsigned)p.S);  // one run of tiles per XCD
    fc_gemm_tile_kernel<RT, false><<<grid, 256, sizeof(GemmTile<RT>), st>>>(
        w, xq, xd, gs, xsT, out, nullptr, (int)Ng, (int)Kg, ldo, N, (int)rows, p.kb_per_split, split_stride, residual, y_final, Ny,
        (int)part_strips, counters);
    return LLMOPS_OK;
}

// y = product (+ residual, fp32 [rows, N], may be y itself); room: as gemm_workspace_bytes was asked with; parts > 1 (group 128,
// no residual): y is [parts][rows][N], part i the columns of strips i * Ng / parts ..
int launch_gemm(const uint8_t* w, const int8_t* xq, const float* xd, const float* gs, const float2* xsT, float* y,
                float* part, unsigned* counters, int64_t rows, int64_t Ng, int64_t Kg, int G, int64_t N, const float* residual,
                int64_t room, int64_t parts, hipStream_t st) {
    const GemmPlan p = plan_gemm(rows, Ng, Kg, G, room);
    // With up to 12 splits the tiled kernel adds the partial sums itself (the last split of a tile to arrive
    // does), given one zeroed arrival counter per tile; otherwise a second launch adds them (8-11 us whatever the shape).
    const int64_t tiles = ((Ng + 3) / 4) * ((rows + p.RT * 32 - 1) / (p.RT * 32));
    const bool fused_reduce = g_gemm_fused_reduce && p.S > 1 && p.lds && counters != nullptr && p.S <= 12 * g_gemm_fused_reduce &&
                              tiles <= kTicketBytes / 4;
    // the residual is added where the result is written: in the kernel's stores without split-K, in
    // the reduction of the partial sums with it
    const float* kres = (p.S > 1 && !fused_reduce) ? nullptr : residual;
    unsigned* kcnt = fused_reduce ? counters : nullptr;
    const int64_t Np = Ng * kGroupN;
    float* out = p.S > 1 ? part : y;
    const int64_t ldo = p.S > 1 ? Np : N;
    const int64_t Nw = p.S > 1 ? Np : N;
    const int64_t part_strips = p.S > 1 && !fused_reduce ? Ng : Ng / parts;
    const int64_t ss = rows * Np;
    if (p.lds) {
        int rc;
        if (p.RT == 4) rc = launch_gemm_tile<4>(w, xq, xd, gs, xsT, out, Ng, Kg, ldo, Nw, rows, p, ss, kres, y, N, part_strips, kcnt, st);
        else if (p.RT == 2) rc = launch_gemm_tile<2>(w, xq, xd, gs, xsT, out, Ng, Kg, ldo, Nw, rows, p, ss, kres, y, N, part_strips, kcnt, st);
        else rc = launch_gemm_tile<1>(w, xq, xd, gs, xsT, out, Ng, Kg, ldo, Nw, rows, p, ss, kres, y, N, part_strips, kcnt, st);
        if (rc) return rc;
    } else {
        const int rc = launch_gemm_g32(w, xq, xd, gs, xsT, out, Ng, Kg, ldo, Nw, rows, p.kb_per_split, p.S, ss, kres, st);
        if (rc) return rc;
    }
    LLMOPS_LAUNCH_CHECK();
    if (p.S > 1 && !fused_reduce) {
        const int64_t total = rows * ((N + 3) / 4);
        gemm_reduce_kernel<<<dim3((unsigned)((total + 255) / 256), (unsigned)parts), 256, 0, st>>>(part, y, rows, N, Np, ss, p.S, residual);
        LLMOPS_LAUNCH_CHECK();
    }
    return LLMOPS_OK;
}

// the production loop, writing its int32 tiles instead of folding them
template <int RT>
static int launch_gemm_tile_partials(const uint8_t* w, const int8_t* xq, int32_t* acc, int64_t rows, int64_t Ng, int64_t Kg, hipStream_t st) {
    if (Kg * 128 * (RT * 32) >= ((int64_t)1 << 32))  // (32-bit offsets into a tile's rows)
        return fail(LLMOPS_EINVAL, "fc_Q4A_partials: K must be below 2^32 / %d for tiles of that many rows", RT * 32);
    const int bad = configure_gemm_tile<RT, true>();
    if (bad) return bad;
    const int64_t tiles = ((Ng + 3) / 4) * ((rows + RT * 32 - 1) / (RT * 32));
    fc_gemm_tile_kernel<RT, true><<<(unsigned)(8 * ((tiles + 7) / 8)), 256, sizeof(GemmTile<RT>), st>>>(
        w, xq, nullptr, nullptr, nullptr, nullptr, acc, (int)Ng, (int)Kg, 0, 0, (int)rows, (int)Kg, 0, nullptr, nullptr, 0, (int)Ng, nullptr);
    LLMOPS_LAUNCH_CHECK();
    return LLMOPS_OK;
}

int launch_gemm_partials(const uint8_t* w, const int8_t* xq, int32_t* acc, int64_t rows, int64_t Ng, int64_t Kg, int G,
                         bool rows128, hipStream_t st) {
    if (G != 128) return launch_gemm_g32_partials(w, xq, acc, rows, Ng, Kg, st);
    return rows128 ? launch_gemm_tile_partials<4>(w, xq, acc, rows, Ng, Kg, st) : launch_gemm_tile_partials<2>(w, xq, acc, rows, Ng, Kg, st);
}

}  // namespace llmops

extern "C" void llmops_test_gemm_set_tuning(int row_tile_factor) {
    const bool known = row_tile_factor == -1 || row_tile_factor == 1 || row_tile_factor == 2 || row_tile_factor == 4;
    if (llmops::test_hooks_enabled(__func__)) llmops::g_gemm_rt = known ? row_tile_factor : 0;
}
extern "C" void llmops_test_gemm_set_split(int splits) {
    if (llmops::test_hooks_enabled(__func__)) llmops::g_gemm_force_split = splits < 0 ? 0 : splits;
}
extern "C" int llmops_test_gemm_plan(int64_t rows, int64_t Ng, int64_t Kg, int group_k, int* row_tile_factor, int* splits) {
    LLMOPS_TEST_HOOK();
    if (rows < 1 || Ng < 1 || Kg < 1 || (group_k != 32 && group_k != 128) || !row_tile_factor || !splits) return LLMOPS_EINVAL;
    const llmops::GemmPlan p = llmops::plan_gemm(rows, Ng, Kg, group_k, INT64_MAX);
    *row_tile_factor = p.RT;
    *splits = p.S;
    return LLMOPS_OK;
}
extern "C" void llmops_test_gemm_set_reduce(int in_kernel) {
    if (llmops::test_hooks_enabled(__func__)) llmops::g_gemm_fused_reduce = in_kernel < 0 ? 0 : in_kernel;
}
