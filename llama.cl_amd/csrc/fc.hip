// C ABI of the Q4_1 x Q8 fully-connected op: argument checks, workspace layout and dispatch
// between the dot4 streaming kernel (few rows) and the int8 MFMA kernel (many rows).
#include "common.h"

#include <mutex>

namespace llmops {

constexpr int kMaxGemvRows = 8;

int launch_quant_x(const float* x, int64_t rows, int64_t K, int group_k, int8_t* xq, float* xd, float* gsum, float2* xsT,
                   bool exact_sum, bool* tile, hipStream_t stream);
int launch_quant_x_fused(const float* x, int64_t rows, int64_t K, int group_k, const float* norm_w, float eps, bool glu_in,
                         int8_t* xq, float2* xsT, bool tiled, hipStream_t stream);
int launch_strip_sumsq(const float* y, int64_t rows, int64_t N, float* out, hipStream_t st);
size_t gemv_workspace_bytes(int64_t rows, int64_t Ng, int64_t Kg, int G);
int launch_gemv(const uint8_t* w, const int8_t* xq, const float* xd, const float* gs, float* y, float* part,
                unsigned* counters, int64_t rows, int64_t Ng, int64_t Kg, int G, int64_t N, hipStream_t st);
int launch_gemv_fused(const uint8_t* w, const float* x, float* y, float* part, unsigned* counters, int64_t rows, int64_t Ng,
                      int64_t Kg, int G, int64_t N, const float* residual, const float* norm_w, float eps, int glu,
                      const float* sumsq_in, int sumsq_parts, float* sumsq_out, hipStream_t st, const DumpBufs* dump = nullptr,
                      const float* rec_stats = nullptr, const float* rec_outs = nullptr, int rec_chunks = 0);
int launch_add(float* a, const float* b, int64_t total, hipStream_t st);
int launch_gemv_partials(const uint8_t* w, const int8_t* xq, int32_t* acc, int64_t rows, int64_t Ng, int64_t Kg, int G,
                         hipStream_t st);
size_t gemm_workspace_bytes(int64_t rows, int64_t Ng, int64_t Kg, int G, int64_t room);
int launch_gemm(const uint8_t* w, const int8_t* xq, const float* xd, const float* gs, const float2* xsT, float* y,
                float* part, unsigned* counters, int64_t rows, int64_t Ng, int64_t Kg, int G, int64_t N, const float* residual,
                int64_t room, int64_t parts, hipStream_t st);
int launch_gemm_partials(const uint8_t* w, const int8_t* xq, int32_t* acc, int64_t rows, int64_t Ng, int64_t Kg, int G,
                         bool rows128, hipStream_t st);
int launch_fc_rows(const uint8_t* w, const int8_t* xq, bool tiled, const float2* xsT, float* y, int64_t rows, int64_t Ng, int64_t Kg,
                   int64_t N, const float* residual, int64_t parts, unsigned long long* slots, size_t slot_bytes, hipStream_t st);
int launch_fc_rows_partials(const uint8_t* w, const int8_t* xq, int32_t* acc, int64_t rows, int64_t Ng, int64_t Kg,
                            hipStream_t st);
bool stream_fits(int64_t rows, int64_t Kg);
bool stream_forced();
bool streams(int64_t rows, int64_t Ng, int64_t Kg, int group_k);  // below
double stream_estimate(int64_t rows, int64_t Ng, int64_t Kg, size_t slot_bytes);
bool gemm_rows_kernel_enabled();
bool gemm_tile_forced();
double gemm_tile_estimate(int64_t rows, int64_t Ng, int64_t Kg);

static inline size_t align_up(size_t v, size_t a) { return (v + a - 1) / a * a; }

struct FcWorkspace {
    size_t off_xq, off_xd, off_gs, off_xst, off_part, total;
    int64_t room;  // what partial sums may take
};

// limit: bytes that the workspace has, where that is fixed (the tiled product then splits K no further than they allow; what
// fits without the limit is split as without it)
static FcWorkspace fc_layout(int64_t rows, int64_t Ng, int64_t Kg, int G, size_t limit = 0) {
    FcWorkspace w;
    size_t o = LLMOPS_FC_COUNTER_BYTES;
    w.off_xq = o;
    o = align_up(o + (size_t)rows * Kg * G, 256);
    w.off_xd = o;
    o = align_up(o + (size_t)rows * Kg * sizeof(float), 256);
    w.off_gs = o;
    o = align_up(o + (size_t)rows * Kg * sizeof(float), 256);
    w.off_xst = o;
    // (+256: no kernel reads behind the last pair; the sizes that callers have asked for count it)
    o = align_up(o + (size_t)rows * Kg * 2 * sizeof(float) + 256, 256);
    w.off_part = o;
    w.room = limit == 0 ? INT64_MAX : (int64_t)limit - (int64_t)o;  // (multiples of 256 both)
    o = align_up(o + (rows <= kMaxGemvRows ? gemv_workspace_bytes(rows, Ng, Kg, G) : gemm_workspace_bytes(rows, Ng, Kg, G, w.room)), 256);
    w.total = o;
    return w;
}

}  // namespace llmops

using namespace llmops;

extern "C" size_t llmops_fc_Q4A_workspace_bytes(int64_t rows, int64_t K, int64_t Ng, int64_t Kg, int group_k) {
    (void)K;
    if (!valid_group(group_k) || rows <= 0 || Ng <= 0 || Kg <= 0) return 0;
    return fc_layout(rows, Ng, Kg, group_k).total;
}

// from how many rows the weight-streaming MFMA kernel takes over from the streaming kernel that quantizes
// on the fly, where tests say it: tensors of up to 256 strips / of more; 0: rows_from() below, and in
// decode_quantizes_first 4 / 3
static int g_rows_from_small = 0, g_rows_from_large = 0;

// .. in fc_Q4A.  The first kernel's work per weight byte grows with the row count (every row is quantized and dotted separately); the
// second's time hardly depends on it up to 16 rows, but it has a launch more, and a program that issues call by call needs 6.5 to 8.4 us for two
// launches, 4.0 to 5.2 for one: below that only a captured graph would have what the second saves.  us in a graph, weights from memory, first / second:
//   4096x4096 (128 strips): 2 rows 5.8 / 6.8, 3 7.4 / 6.9 (call by call 6.9 / 8.6), 4 8.0 / 7.0, 8 9.7 / 7.0
//   6000x4096 (188), 8192x4096 (256): 3 rows 7.5 / 7.7 and 8.2 / 8.2, 4 8.5 / 7.8 and 9.1 / 8.2
//   11008x4096, 12288x4096: 2 rows 9.1 / 11.4 and 9.3 / 11.5, 3 13.1 / 10.5 and 13.7 / 11.4
//   4096x11008:             2 rows 8.7 / 10.8, 3 10.7 / 10.9 (from a cache 12.2 / 10.9), 4 12.4 / 10.4, 8 19.6 / 10.6; 2500x11008: 3 14.9 / 9.7
//   1500x2048, 2048x2048:   4 rows 5.7 / 5.5, 8 8.3 / 5.5
//   1024x512 .. 4096x1024:  4 rows 4.2 / 5.0, 8 6.3 / 5.3 (call by call 6.3 / 8.6)
//   1 to 64 strips, within 15 % whatever their number: x 2048 4 rows 5.6 / 5.5, 8 8.5 / 5.7 (call by call 8.3 / 6.5 to 8.4); x 4096 3 rows 6.9 / 6.0,
//   6 8.6 / 6.6, 8 9.3 / 6.7 (9.0 / 6.4 to 8.4); x 8192 4 rows 8.4 / 7.9, 8 11.2 / 8.1; x 11008 4 rows with 8 strips 8.6 / 9.1, with 16 9.2 / 9.2,
//   with 47 14.4 / 9.6; 5 with 8 strips 10.0 / 9.1
static int rows_from(int64_t Ng, int64_t Kg) {
    const int forced = Ng > 256 ? g_rows_from_large : g_rows_from_small;
    if (forced > 0) return forced;
    if (Kg < 12) return kMaxGemvRows + 1;
    if (Ng < 64) return Kg < 24 ? kMaxGemvRows + 1 : Kg < 64 ? 6 : Ng < 16 ? 5 : 4;
    if (Ng > 256 || Kg >= 64) return 3;
    return Kg < 24 ? 5 : 4;
}

// argument checks of fc_Q4A that do not involve the workspace
static int fc_check_args(const float* x, int64_t rows, int64_t K, const int8_t* weiq, int64_t Ng, int64_t Kg, int group_k,
                         int64_t N, const float* y) {
    LLMOPS_REQUIRE(valid_group(group_k));
    LLMOPS_REQUIRE(x != nullptr && weiq != nullptr && y != nullptr);
    LLMOPS_REQUIRE(rows > 0 && K > 0 && Ng > 0 && Kg > 0);
    LLMOPS_REQUIRE(K > (Kg - 1) * group_k && K <= Kg * group_k);  // a short last k-group is zero padded (ops/op_fc.hpp:259-261)
    LLMOPS_REQUIRE(N > (Ng - 1) * kGroupN && N <= Ng * kGroupN);
    LLMOPS_REQUIRE(Ng <= kTicketBytes / 4);
    LLMOPS_REQUIRE(Ng * 64 < ((int64_t)1 << 31));
    LLMOPS_REQUIRE(aligned(weiq, 16) && aligned(x, K != Kg * group_k ? 4 : 8));
    return LLMOPS_OK;
}

// Whether the product of quantized activations (group 128) is the weight-streaming kernel's or the tiled one's.  Up to 16
// rows are bound by the weight stream (tiled / streaming, us: 9 x 1024 x 512 7.6 / 5.0, 16 x 512 x 4096 9.6 / 6.5).  Above, the
// streaming kernel fetches every row's codes for each strip again, the tiled one shares them between four strips but needs splits
// of K and barriers: whichever is estimated to take less, with 7 us on the tiled side, which its estimate leaves out (first fetch, finish,
// quantization); 4.75 up to 11 k-groups, where the quantization costs less and most of this kernel's time is its results; 2 from 513 rows on,
// where both estimates are less even.  Beyond 1024 rows what there is to gain is a few percent.  Of 687 sizes (17 .. 1024 rows of fifteen shapes
// from 1024 x 512 to 22016 x 4096 and 11008 x 11008, both kernels in turn, weights from memory) none that is streamed would be more than 1.7 % faster in
// tiles (768 x 600 x 11008 29.8 / 30.3); 37 that are tiled would be 2 % and more faster streamed, most of them within 8 % (us, tiled / streaming:
// 192 x 12288 x 4096 35.0 / 29.9, 96 x 22016 x 4096 34.8 / 30.5, 192 x 11008 x 4096 31.1 / 29.0, 576 x 4096^2 33.5 / 31.1, 832 x 2000 x 8192 44.0 / 40.4).
// Some times: 64 x 4096^2 13.8 / 8.5, 128 x 4096 x 11008 25.4 / 22.6, 256 x 4096^2 20.2 / 16.0, 512 x 2048^2 16.0 / 12.5, 384 x 4096 x 512 10.4 / 10.0,
// 448 10.5 / 11.2, 256 x 22016 x 4096 48.1 / 57.5, 128 x 11008 x 11008 40.6 / 46.2, 1024 x 1500 x 3072 25.4 / 22.4.  Neither is ahead from one row count on:
// tiles, splits and row blocks come in steps, 4096 x 11008 at 256 rows 35.9 / 31.2, 272 40.1 / 43.4, 304 40.7 / 41.5, 336 43.2 / 42.6, 384 45.8 / 45.2, 512
// 54.0 / 52.2, 544 64.9 / 66.4.
bool llmops::streams(int64_t rows, int64_t Ng, int64_t Kg, int group_k) {
    if (group_k != 128 || rows > 1024 || !gemm_rows_kernel_enabled() || !stream_fits(rows, Kg)) return false;
    if (rows <= 16) return true;
    if (gemm_tile_forced()) return false;
    if (stream_forced()) return true;
    const double ahead = rows > 512 ? 2.0 : Kg < 12 ? 4.75 : 7.0;
    return stream_estimate(rows, Ng, Kg, LLMOPS_FC_COUNTER_BYTES - kTicketBytes) <= gemm_tile_estimate(rows, Ng, Kg) + ahead;
}
// An input that does not start on 16 bytes takes the general quantization, whose codes lie row by row: more than 32 such rows are the tiled
// kernel's (tiled / streaming, us: 32 x 11008 x 4096 15.4 / 12.7, 64 x 11008 x 4096 17.8 / 18.5, 128 x 11008 x 4096 22.8 / 26.9, 500 x 4096 x 11008
// 55.1 / 69.9; 64 x 2048^2 10.5 / 6.8 goes with them).
static bool streams_input(const float* x, int64_t rows, int64_t Ng, int64_t Kg, int group_k) {
    return (rows <= 32 || aligned(x, 16) || stream_forced()) && streams(rows, Ng, Kg, group_k);
}

// the product for activations that a quantization launch has left in the workspace (more rows than the streaming
// kernel that quantizes on the fly takes); streamed: what streams() says; tiled: the codes are in the order of tile_code_offset
static int fc_product_many_rows(const uint8_t* w, uint8_t* ws, const FcWorkspace& lay, bool streamed, bool tiled, int64_t rows, int64_t Ng, int64_t Kg,
                                int group_k, int64_t N, const float* residual, float* y, int64_t parts, hipStream_t st) {
    const int8_t* xq = reinterpret_cast<const int8_t*>(ws + lay.off_xq);
    const float* xd = reinterpret_cast<const float*>(ws + lay.off_xd);
    const float* gs = reinterpret_cast<const float*>(ws + lay.off_gs);
    const float2* xst = reinterpret_cast<const float2*>(ws + lay.off_xst);
    if (streamed)
        return launch_fc_rows(w, xq, tiled, xst, y, rows, Ng, Kg, N, residual, parts, reinterpret_cast<unsigned long long*>(ws + kTicketBytes),
                              LLMOPS_FC_COUNTER_BYTES - kTicketBytes, st);
    return launch_gemm(w, xq, xd, gs, xst, y, reinterpret_cast<float*>(ws + lay.off_part), reinterpret_cast<unsigned*>(ws), rows, Ng,
                       Kg, group_k, N, residual, lay.room, parts, st);
}

static int fc_impl(const float* x, int64_t rows, int64_t K, const int8_t* weiq, int64_t Ng, int64_t Kg, int group_k,
                   int64_t N, const float* residual, float* y, void* workspace, size_t workspace_bytes,
                   llmops_stream_t stream, size_t limit = 0) {
    const int bad = fc_check_args(x, rows, K, weiq, Ng, Kg, group_k, N, y);
    if (bad) return bad;
    LLMOPS_REQUIRE(workspace != nullptr && aligned(workspace, 256));
    const bool k_tail = K != Kg * group_k;
    const FcWorkspace lay = fc_layout(rows, Ng, Kg, group_k, limit);
    if (workspace_bytes < lay.total)
        return fail(LLMOPS_EWORKSPACE, "fc_Q4A needs %zu workspace bytes, got %zu", lay.total, workspace_bytes);
    uint8_t* ws = reinterpret_cast<uint8_t*>(workspace);
    unsigned* counters = reinterpret_cast<unsigned*>(ws);
    int8_t* xq = reinterpret_cast<int8_t*>(ws + lay.off_xq);
    float* xd = reinterpret_cast<float*>(ws + lay.off_xd);
    float* gs = reinterpret_cast<float*>(ws + lay.off_gs);
    float* part = reinterpret_cast<float*>(ws + lay.off_part);
    hipStream_t st = as_stream(stream);
    const uint8_t* w = reinterpret_cast<const uint8_t*>(weiq);
    if (k_tail) {
        // K is not a whole number of k-groups (no shape the reference is used with): the general quantization kernel
        // pads the last group's codes with zeros, as FC_dynamic_quantize_x does, and the product runs on the codes
        float2* xst_t = reinterpret_cast<float2*>(ws + lay.off_xst);
        int rc_t = launch_quant_x(x, rows, K, group_k, xq, xd, gs, xst_t, false, nullptr, st);
        if (rc_t) return rc_t;
        if (rows > kMaxGemvRows) return launch_gemm(w, xq, xd, gs, xst_t, y, part, counters, rows, Ng, Kg, group_k, N, residual, lay.room, 1, st);
        if (residual == y) return fail(LLMOPS_EINVAL, "fc_Q4A with a short last k-group and up to 8 rows: residual must not be y");
        rc_t = launch_gemv(w, xq, xd, gs, y, part, counters, rows, Ng, Kg, group_k, N, st);
        if (rc_t == 0 && residual != nullptr) rc_t = launch_add(y, residual, rows * N, st);
        return rc_t;
    }
    const bool streamed = streams_input(x, rows, Ng, Kg, group_k);
    if (rows <= kMaxGemvRows && !(streamed && rows >= rows_from(Ng, Kg)))  // (one launch)
        return launch_gemv_fused(w, x, y, part, counters, rows, Ng, Kg, group_k, N, residual, nullptr, 0.0f, 0, nullptr, 0,
                                 nullptr, st);
    float2* xst = reinterpret_cast<float2*>(ws + lay.off_xst);
    bool tiled = streamed;
    int rc = launch_quant_x(x, rows, K, group_k, xq, xd, gs, xst, false, &tiled, st);
    if (rc) return rc;
    return fc_product_many_rows(w, ws, lay, streamed, tiled, rows, Ng, Kg, group_k, N, residual, y, 1, st);
}

extern "C" int llmops_fc_Q4A(const float* x, int64_t rows, int64_t K, const int8_t* weiq, int64_t Ng, int64_t Kg,
                             int group_k, int64_t N, float* y, void* workspace, size_t workspace_bytes,
                             llmops_stream_t stream) {
    return fc_impl(x, rows, K, weiq, Ng, Kg, group_k, N, nullptr, y, workspace, workspace_bytes, stream);
}

extern "C" int llmops_fc_Q4A_residual(const float* x, int64_t rows, int64_t K, const int8_t* weiq, int64_t Ng,
                                      int64_t Kg, int group_k, int64_t N, const float* residual, float* y,
                                      void* workspace, size_t workspace_bytes, llmops_stream_t stream) {
    LLMOPS_REQUIRE(residual != nullptr);
    return fc_impl(x, rows, K, weiq, Ng, Kg, group_k, N, residual, y, workspace, workspace_bytes, stream);
}

// Up to 8 rows: whether the producer, the product and the sums of squares are launches of their own (quantization, the
// weight-streaming MFMA product, launch_strip_sumsq) instead of one launch of the streaming kernel.  That one forms a
// producer in every strip's workgroup again for every row, and quantizes and multiplies row by row: a row costs it 0.5 us
// (64 strips x 4 k-groups) to 3 us (688 x 32) and more with a producer, hardly anything the other way, where the second
// launch costs 1.5 to 3 us and the sums 1.9.  In a graph, weights not from a cache, us, streaming / separate launches, at
// rows either side of where the line lies (strips x k-groups):
//   residual:             64x4 4 rows 4.5 / 5.1, 5 5.5 / 5.2; 64x16 4 5.8 / 6.3, 5 7.3 / 6.4; 128x32 3
//                         7.4 / 7.3; 128x86 3 10.4 / 11.4, 4 11.5 / 10.8; 256x32 3 8.0 / 9.0, 4 8.8 / 8.5; 384x32 2 9.3 / 12.3, 3 13.3 / 12.3;
//                         688x32 3 20.1 / 16.4
//   .. and sums:          64x4 8 rows 6.9 / 7.2; 64x16 6 8.0 / 8.5, 8 9.2 / 8.4; 128x32 5 9.3 / 9.4, 6
//                         9.7 / 9.4; 128x86 4 12.3 / 12.7, 5 15.9 / 12.9; 256x32 4 9.2 / 10.5, 5 11.4 / 10.6; 384x32 2 9.6 / 13.2, 3 14.1 / 13.5
//   rmsnorm:              64x4 2 rows 5.9 / 5.2, 3 8.1 / 5.3; 128x32 2 8.3 / 7.7, 3 12.1 / 7.8; 128x86 2 11.0 / 12.8, 3
//                         15.2 / 13.0; 384x32 2 15.7 / 11.7; 688x32 2 23.3 / 15.8
//   .. and sums:          64x16 2 rows 7.0 / 8.6, 3 9.9 / 8.6; 128x32 2 8.6 / 9.9, 3 12.2 / 9.8; 384x32 2 16.5 / 13.7
//   .. sums handed in:    64x4 4 rows 5.2 / 5.3, 5 6.6 / 5.5; 64x16 4 7.0 / 6.5, 5 9.4 / 6.7; 128x32 2 6.6 / 7.7, 3 9.3 / 7.8;
//                         128x86 3 11.9 / 13.1, 4 13.3 / 13.0; 256x32 2 7.0 / 8.9, 3 9.8 / 8.9; 384x32 2 10.7 / 11.7, 3 17.1 / 11.7; 688x32 2 14.7 / 15.8
//   silu * up, residual:  64x4 4 rows 5.1 / 5.2, 5 6.2 / 5.2; 64x16 4 6.8 / 6.4; 128x32 2
//                         6.5 / 7.2, 3 8.6 / 7.3; 128x86 2 9.4 / 10.7, 3 12.0 / 10.8; 384x32 2 10.5 / 11.3; 688x32 2 14.6 / 15.3
//   .. and sums:          64x4 7 rows 7.6 / 7.2, 8 8.1 / 7.1; 64x16 5 9.1 / 8.5; 128x32 3 9.1 / 9.4, 4 10.2 / 9.2; 128x86 3
//                         12.6 / 12.8; 256x32 3 9.5 / 10.5, 4 10.8 / 10.5; 384x32 2 11.2 / 13.3, 3 17.0 / 13.5
// Fewer than 64 strips are one launch, as the header promises, also where the other way would be the faster one (16x4: residual 8 rows 6.5 / 5.2;
// 16x32: residual 5 rows 8.3 / 6.8, .. and sums 7 9.4 / 8.6; 8x32: rmsnorm 3 rows 11.4 / 6.8; 48x86: silu * up 5 rows 20.0 / 9.8).
static bool decode_quantizes_first(int64_t rows, int64_t K, int64_t Ng, int64_t Kg, int group_k, bool norm, bool sums_in, int glu, bool sums_out) {
    if (Ng < 64 || rows > kMaxGemvRows || !streams(rows, Ng, Kg, group_k) || glu == 1 || (norm && K > 16384)) return false;
    const bool large = Ng > 256;
    const int64_t blocks = Ng * Kg;
    int from = large ? (g_rows_from_large > 0 ? g_rows_from_large : 3) : g_rows_from_small > 0 ? g_rows_from_small : 4;
    if (norm && !sums_in) return rows >= from - 1;
    const bool producer = norm || glu == 2;
    if (large) return rows >= from - (producer && !sums_out && (glu == 2 || blocks >= 16384) ? 1 : 0);
    if (blocks < 2048) from += 1;
    else if (producer) from -= 1;
    if (sums_out) from += blocks < 512 ? (producer ? 3 : 4) : (producer || blocks >= 8192 ? 1 : 2);
    return rows >= from;
}

static int fc_decode_impl(const float* x, int64_t rows, int64_t K, const int8_t* weiq, int64_t Ng, int64_t Kg, int group_k,
                          int64_t N_out, const float* norm_w, float eps, const float* residual, int glu,
                          const float* sumsq_in, int64_t sumsq_parts, float* sumsq_out, float* y, int64_t out_parts,
                          void* workspace, size_t workspace_bytes, llmops_stream_t stream) {
    LLMOPS_REQUIRE(valid_group(group_k));
    LLMOPS_REQUIRE(x != nullptr && weiq != nullptr && y != nullptr && workspace != nullptr);
    LLMOPS_REQUIRE(rows > 0);
    LLMOPS_REQUIRE(K > 0 && Ng > 0 && Kg > 0 && K == Kg * group_k);
    LLMOPS_REQUIRE(Ng <= kTicketBytes / 4 && Ng * 64 < ((int64_t)1 << 31));
    LLMOPS_REQUIRE(aligned(weiq, 16) && aligned(workspace, 256) && aligned(x, 8));
    LLMOPS_REQUIRE(glu >= 0 && glu <= 2);
    if (glu == 1) {
        LLMOPS_REQUIRE((Ng % 2) == 0 && residual == nullptr);
        LLMOPS_REQUIRE(N_out > (Ng / 2 - 1) * kGroupN && N_out <= Ng / 2 * kGroupN);
    } else {
        LLMOPS_REQUIRE(N_out > (Ng - 1) * kGroupN && N_out <= Ng * kGroupN);
    }
    if (norm_w != nullptr) LLMOPS_REQUIRE((K % 4) == 0 && aligned(x, 16) && aligned(norm_w, 8));
    if (sumsq_in != nullptr) LLMOPS_REQUIRE(norm_w != nullptr && sumsq_parts > 0 && sumsq_parts <= 65536);
    if (sumsq_out != nullptr) LLMOPS_REQUIRE(glu != 1);
    if (glu == 2) LLMOPS_REQUIRE(norm_w == nullptr && sumsq_in == nullptr);
    LLMOPS_REQUIRE(out_parts >= 1);
    if (out_parts > 1)
        LLMOPS_REQUIRE(glu != 1 && residual == nullptr && sumsq_out == nullptr && (Ng % out_parts) == 0 &&
                       N_out == Ng * kGroupN);
    const FcWorkspace lay = fc_layout(rows, Ng, Kg, group_k);
    // (with groups of 32 parts are products of their own with fewer strips each, and fewer strips are split over K more often:
    // a part can need more room for partial sums than the whole; the offsets in front of them are the same.  One size is
    // asked for with either group, as the header says, although with groups of 128 the whole's is used)
    size_t need = lay.total;
    if (out_parts > 1) {
        const size_t part_need = fc_layout(rows, Ng / out_parts, Kg, group_k).total;
        need = part_need > need ? part_need : need;
    }
    if (workspace_bytes < need)
        return fail(LLMOPS_EWORKSPACE, "fc_Q4A needs %zu workspace bytes, got %zu", need, workspace_bytes);
    uint8_t* ws = reinterpret_cast<uint8_t*>(workspace);
    const bool sums_in = sumsq_in != nullptr && sumsq_parts <= 256;  // (what the streaming kernel reads)
    const bool quantize_first = decode_quantizes_first(rows, K, Ng, Kg, group_k, norm_w != nullptr, sums_in, glu, sumsq_out != nullptr) &&
                                ((norm_w == nullptr && glu != 2) || aligned(x, 16)) && (norm_w == nullptr || aligned(norm_w, 16));
    if (rows > kMaxGemvRows || quantize_first) {
        // More rows than the streaming kernel takes or is good at: the producer is folded into the quantization launch instead
        // (its fp32 result never goes through memory), the residual into the product's stores, and the sums of
        // squares take a launch of their own.  The statistic of the rmsnorm is computed from the row (sumsq_in is
        // not needed: the launch has the whole row in registers).
        if (glu == 1) return fail(LLMOPS_EINVAL, "fc_Q4A_decode with more than 8 rows: gate and up stacked (glu 2), not interleaved");
        hipStream_t st = as_stream(stream);
        int8_t* xq = reinterpret_cast<int8_t*>(ws + lay.off_xq);
        float* xd = reinterpret_cast<float*>(ws + lay.off_xd);
        float* gs = reinterpret_cast<float*>(ws + lay.off_gs);
        float2* xst = reinterpret_cast<float2*>(ws + lay.off_xst);
        const bool streamed = streams_input(x, rows, Ng, Kg, group_k);
        bool tiled = streamed;
        int rc = (norm_w != nullptr || glu == 2)
                     ? launch_quant_x_fused(x, rows, K, group_k, norm_w, eps, glu == 2, xq, xst, tiled, st)
                     : launch_quant_x(x, rows, K, group_k, xq, xd, gs, xst, false, &tiled, st);
        if (rc) return rc;
        if (out_parts > 1) {
            // y is [out_parts][rows][N_out / out_parts]: q, k and v of a fused q|k|v tensor come out as three dense matrices
            // instead of one to be cut up.  Group 128: one product whose stores know the parts (a third of the strips
            // fills the chip less well; us with rmsnorm, 3 x 4096 x 4096, a product each / in one: 12 rows 19.1 / 14.4, 64 rows
            // 37.8 / 19.5, 300 rows 59.4 / 41.1, 512 rows 82.2 / 52.7, 1024 rows 113.5 / 97.8 in one); group 32: a
            // product per slice of strips on the same quantized rows.
            const int64_t ngp = Ng / out_parts, np = N_out / out_parts;
            if (group_k == 128)
                return fc_product_many_rows(reinterpret_cast<const uint8_t*>(weiq), ws, lay, streamed, tiled, rows, Ng, Kg, group_k, np, nullptr, y, out_parts, st);
            for (int64_t p = 0; p < out_parts && rc == 0; p++)
                rc = fc_product_many_rows(reinterpret_cast<const uint8_t*>(weiq) + p * ngp * Kg * block_bytes(group_k), ws, lay, false, false,
                                          rows, ngp, Kg, group_k, np, nullptr, y + p * rows * np, 1, st);
            return rc;
        }
        rc = fc_product_many_rows(reinterpret_cast<const uint8_t*>(weiq), ws, lay, streamed, tiled, rows, Ng, Kg, group_k, N_out, residual, y, 1, st);
        if (rc == 0 && sumsq_out != nullptr) rc = launch_strip_sumsq(y, rows, N_out, sumsq_out, st);
        return rc;
    }
    LLMOPS_REQUIRE(out_parts == 1);  // (up to 8 rows: a slice of a row is as good as a row of its own)
    return launch_gemv_fused(reinterpret_cast<const uint8_t*>(weiq), x, y, reinterpret_cast<float*>(ws + lay.off_part),
                             reinterpret_cast<unsigned*>(ws), rows, Ng, Kg, group_k, N_out, residual, norm_w, eps, glu,
                             sumsq_in, (int)sumsq_parts, sumsq_out, as_stream(stream));
}

extern "C" int llmops_fc_Q4A_decode(const float* x, int64_t rows, int64_t K, const int8_t* weiq, int64_t Ng, int64_t Kg,
                                    int group_k, int64_t N_out, const float* norm_w, float eps, const float* residual,
                                    int glu, const float* sumsq_in, int64_t sumsq_parts, float* sumsq_out, float* y,
                                    void* workspace, size_t workspace_bytes, llmops_stream_t stream) {
    return fc_decode_impl(x, rows, K, weiq, Ng, Kg, group_k, N_out, norm_w, eps, residual, glu, sumsq_in, sumsq_parts, sumsq_out, y,
                          1, workspace, workspace_bytes, stream);
}

extern "C" int llmops_fc_Q4A_decode_wants_sumsq(int64_t rows, int64_t K, int64_t Ng, int64_t Kg, int group_k, int glu) {
    return rows <= kMaxGemvRows && !decode_quantizes_first(rows, K, Ng, Kg, group_k, true, false, glu, false);
}

extern "C" int llmops_test_fc_decode_route(int64_t rows, int64_t K, int64_t Ng, int64_t Kg, int group_k, int norm, int sumsq_in, int glu,
                                           int sumsq_out, int* quantize_first) {
    LLMOPS_TEST_HOOK();
    LLMOPS_REQUIRE(valid_group(group_k) && rows > 0 && K > 0 && Ng > 0 && Kg > 0 && quantize_first != nullptr);
    *quantize_first = rows > kMaxGemvRows || decode_quantizes_first(rows, K, Ng, Kg, group_k, norm != 0, sumsq_in != 0, glu, sumsq_out != 0);
    return LLMOPS_OK;
}

extern "C" int llmops_fc_Q4A_decode_parts(const float* x, int64_t rows, int64_t K, const int8_t* weiq, int64_t Ng, int64_t Kg,
                                          int group_k, int64_t N_out, const float* norm_w, float eps, int glu, int64_t out_parts,
                                          float* y, void* workspace, size_t workspace_bytes, llmops_stream_t stream) {
    LLMOPS_REQUIRE(rows > kMaxGemvRows);
    return fc_decode_impl(x, rows, K, weiq, Ng, Kg, group_k, N_out, norm_w, eps, nullptr, glu, nullptr, 0, nullptr, y, out_parts,
                          workspace, workspace_bytes, stream);
}

static int fc_decode_attn(const float* rec_stats, const float* rec_outs, int64_t chunks, int64_t H, const int8_t* weiq,
                          int64_t Ng, int64_t Kg, int64_t N_out, const float* residual, float* sumsq_out, float* y,
                          void* workspace, size_t workspace_bytes, llmops_stream_t stream, const DumpBufs* dump) {
    LLMOPS_REQUIRE(rec_stats != nullptr && rec_outs != nullptr && weiq != nullptr && y != nullptr && workspace != nullptr);
    LLMOPS_REQUIRE(chunks > 0 && chunks <= 8 && H > 0 && Ng > 0 && Kg > 0 && Kg == H);  // K = H * 128, group 128
    LLMOPS_REQUIRE(N_out > (Ng - 1) * kGroupN && N_out <= Ng * kGroupN);
    LLMOPS_REQUIRE(Ng <= kTicketBytes / 4 && Ng * 64 < ((int64_t)1 << 31));
    LLMOPS_REQUIRE(aligned(weiq, 16) && aligned(workspace, 256) && aligned(rec_stats, 16) && aligned(rec_outs, 16));
    const FcWorkspace lay = fc_layout(1, Ng, Kg, 128);
    if (workspace_bytes < lay.total)
        return fail(LLMOPS_EWORKSPACE, "fc_Q4A needs %zu workspace bytes, got %zu", lay.total, workspace_bytes);
    uint8_t* ws = reinterpret_cast<uint8_t*>(workspace);
    return launch_gemv_fused(reinterpret_cast<const uint8_t*>(weiq), rec_outs, y, reinterpret_cast<float*>(ws + lay.off_part),
                             reinterpret_cast<unsigned*>(ws), 1, Ng, Kg, 128, N_out, residual, nullptr, 0.0f, 0, nullptr, 0,
                             sumsq_out, as_stream(stream), dump, rec_stats, rec_outs, (int)chunks);
}

extern "C" int llmops_fc_Q4A_decode_attn(const float* rec_stats, const float* rec_outs, int64_t chunks, int64_t H,
                                         const int8_t* weiq, int64_t Ng, int64_t Kg, int64_t N_out, const float* residual,
                                         float* sumsq_out, float* y, void* workspace, size_t workspace_bytes,
                                         llmops_stream_t stream) {
    return fc_decode_attn(rec_stats, rec_outs, chunks, H, weiq, Ng, Kg, N_out, residual, sumsq_out, y, workspace, workspace_bytes,
                          stream, nullptr);
}

// the same kernel in its dump build (what it merged and quantized, and its int32 sums)
extern "C" int llmops_test_fc_decode_attn_dump(const float* rec_stats, const float* rec_outs, int64_t chunks, int64_t H,
                                               const int8_t* weiq, int64_t Ng, int64_t Kg, int64_t N_out, float* y, int8_t* xq,
                                               float* xd, float* gsum, int32_t* acc, void* workspace, size_t workspace_bytes,
                                               llmops_stream_t stream) {
    LLMOPS_TEST_HOOK();
    LLMOPS_REQUIRE(xq != nullptr && xd != nullptr && gsum != nullptr && acc != nullptr && aligned(xq, 4));
    const DumpBufs dump{xq, xd, gsum, acc};
    return fc_decode_attn(rec_stats, rec_outs, chunks, H, weiq, Ng, Kg, N_out, nullptr, nullptr, y, workspace, workspace_bytes,
                          stream, &dump);
}

extern "C" int llmops_fc_Q4A_prequantized(const int8_t* xq, const float* xd, const float* gsum, int64_t rows,
                                          const int8_t* weiq, int64_t Ng, int64_t Kg, int group_k, int64_t N, float* y,
                                          void* workspace, size_t workspace_bytes, llmops_stream_t stream) {
    LLMOPS_REQUIRE(valid_group(group_k));
    LLMOPS_REQUIRE(xq != nullptr && xd != nullptr && gsum != nullptr && weiq != nullptr && y != nullptr);
    LLMOPS_REQUIRE(workspace != nullptr);
    LLMOPS_REQUIRE(rows > 0 && Ng > 0 && Kg > 0);
    LLMOPS_REQUIRE(N > (Ng - 1) * kGroupN && N <= Ng * kGroupN);
    LLMOPS_REQUIRE(Ng <= kTicketBytes / 4);
    LLMOPS_REQUIRE(aligned(weiq, 16) && aligned(xq, 16) && aligned(workspace, 256));
    const FcWorkspace lay = fc_layout(rows, Ng, Kg, group_k);
    if (workspace_bytes < lay.total)
        return fail(LLMOPS_EWORKSPACE, "fc_Q4A needs %zu workspace bytes, got %zu", lay.total, workspace_bytes);
    uint8_t* ws = reinterpret_cast<uint8_t*>(workspace);
    float* part = reinterpret_cast<float*>(ws + lay.off_part);
    const uint8_t* w = reinterpret_cast<const uint8_t*>(weiq);
    hipStream_t st = as_stream(stream);
    if (rows <= kMaxGemvRows)
        return launch_gemv(w, xq, xd, gsum, y, part, reinterpret_cast<unsigned*>(ws), rows, Ng, Kg, group_k, N, st);
    return launch_gemm(w, xq, xd, gsum, nullptr, y, part, reinterpret_cast<unsigned*>(ws), rows, Ng, Kg, group_k, N, nullptr, lay.room, 1, st);
}

extern "C" int llmops_fc_Q4A_partials(const int8_t* xq, int64_t rows, const int8_t* weiq, int64_t Ng, int64_t Kg,
                                      int group_k, int32_t* acc, int use_mfma, llmops_stream_t stream) {
    LLMOPS_REQUIRE(valid_group(group_k));
    LLMOPS_REQUIRE(xq != nullptr && weiq != nullptr && acc != nullptr);
    LLMOPS_REQUIRE(rows > 0 && Ng > 0 && Kg > 0);
    LLMOPS_REQUIRE(aligned(weiq, 16) && aligned(xq, 16));
    LLMOPS_REQUIRE(Ng * Kg < ((int64_t)1 << 31));
    const uint8_t* w = reinterpret_cast<const uint8_t*>(weiq);
    LLMOPS_REQUIRE(use_mfma >= 0 && use_mfma <= 3 && (use_mfma < 2 || group_k == 128));
    if (use_mfma == 3) {
        LLMOPS_REQUIRE(rows <= 1024);  // (what streams() sends there)
        return launch_fc_rows_partials(w, xq, acc, rows, Ng, Kg, as_stream(stream));
    }
    if (use_mfma) return launch_gemm_partials(w, xq, acc, rows, Ng, Kg, group_k, use_mfma == 2, as_stream(stream));
    return launch_gemv_partials(w, xq, acc, rows, Ng, Kg, group_k, as_stream(stream));
}

extern "C" void llmops_test_fc_set_row_routing(int rows_from_small, int rows_from_large) {
    if (!test_hooks_enabled(__func__)) return;
    g_rows_from_small = rows_from_small >= 2 ? rows_from_small : 0;
    g_rows_from_large = rows_from_large >= 2 ? rows_from_large : 0;
}

// ---- fc_Q4A for callers that cannot allocate ---------------------------------------------------
// The workspace of llmops_fc_Q4A (arrival counters and exchange slots, activation codes and scales,
// split-K partial sums) lives in a fixed array in the library's device image instead of coming from
// the caller.  Each device holds its own copy of the array at its own address; the address is looked
// up once per device and only that pointer is ever handed to kernels (the array's name is a host-side
// handle, not a device address).
namespace llmops {

static __device__ __align__(256) unsigned char scratch[LLMOPS_FC_NOALLOC_SCRATCH_BYTES];

constexpr int kMaxDevices = 64;
static void* g_scratch_ptr[kMaxDevices];
static std::mutex g_scratch_mutex;

// device pointer of this device's copy of `scratch`, resolved on first use with that device current
static int scratch_of_current_device(void** out) {
    int dev = -1;
    LLMOPS_HIP_CHECK(hipGetDevice(&dev));
    if (dev < 0 || dev >= kMaxDevices) return fail(LLMOPS_EINVAL, "device ordinal %d out of range", dev);
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (g_scratch_ptr[dev] == nullptr) {
        void* ptr = nullptr;
        LLMOPS_HIP_CHECK(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
        if (ptr == nullptr) return fail(LLMOPS_EHIP, "hipGetSymbolAddress returned no address for the scratch array");
        g_scratch_ptr[dev] = ptr;
    }
    *out = g_scratch_ptr[dev];
    return LLMOPS_OK;
}

// zero fill with plain vector stores (a kernel rather than a memset node: callers may be capturing a graph)
__global__ __launch_bounds__(256) void zero16_kernel(uint4* p, int64_t n16) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n16) p[i] = make_uint4(0, 0, 0, 0);
}

}  // namespace llmops

extern "C" size_t llmops_fc_Q4A_noalloc_scratch_bytes(void) { return LLMOPS_FC_NOALLOC_SCRATCH_BYTES; }

extern "C" int llmops_fc_workspace_reset(void* workspace, size_t workspace_bytes, llmops_stream_t stream) {
    LLMOPS_REQUIRE(workspace != nullptr && aligned(workspace, 256) && workspace_bytes >= 16);
    const size_t head = workspace_bytes < (size_t)LLMOPS_FC_COUNTER_BYTES ? workspace_bytes : (size_t)LLMOPS_FC_COUNTER_BYTES;
    const int64_t n16 = (int64_t)(head / 16);
    zero16_kernel<<<(unsigned)((n16 + 255) / 256), 256, 0, as_stream(stream)>>>(reinterpret_cast<uint4*>(workspace), n16);
    LLMOPS_LAUNCH_CHECK();
    return LLMOPS_OK;
}

extern "C" int llmops_fc_Q4A_noalloc(const float* x, int64_t rows, int64_t K, const int8_t* weiq, int64_t Ng, int64_t Kg,
                                     int group_k, int64_t N, float* y, llmops_stream_t stream) {
    // everything fc_impl will check is checked here first: a refused call must not enqueue the zero fill either
    const int bad = fc_check_args(x, rows, K, weiq, Ng, Kg, group_k, N, y);
    if (bad) return bad;
    const size_t need = fc_layout(rows, Ng, Kg, group_k, LLMOPS_FC_NOALLOC_SCRATCH_BYTES).total;
    if (need > (size_t)LLMOPS_FC_NOALLOC_SCRATCH_BYTES)
        return fail(LLMOPS_EWORKSPACE,
                    "llmops_fc_Q4A_noalloc: rows=%lld, strips=%lld, k-groups=%lld need %zu scratch bytes, the built-in "
                    "scratch holds %zu; use llmops_fc_Q4A with a caller-provided workspace",
                    (long long)rows, (long long)Ng, (long long)Kg, need, (size_t)LLMOPS_FC_NOALLOC_SCRATCH_BYTES);
    void* ws = nullptr;
    const int rc = scratch_of_current_device(&ws);
    if (rc) return rc;
    // The array keeps whatever the last call on this device left in it.  Counters and exchange slots must
    // start at zero; the kernels leave them so, but a launch that failed half-way would not.
    const int64_t n16 = LLMOPS_FC_COUNTER_BYTES / 16;
    zero16_kernel<<<(unsigned)((n16 + 255) / 256), 256, 0, as_stream(stream)>>>(reinterpret_cast<uint4*>(ws), n16);
    LLMOPS_LAUNCH_CHECK();
    return fc_impl(x, rows, K, weiq, Ng, Kg, group_k, N, nullptr, y, ws, LLMOPS_FC_NOALLOC_SCRATCH_BYTES, stream, LLMOPS_FC_NOALLOC_SCRATCH_BYTES);
}

// The production decode kernel in its dump build: y as llmops_fc_Q4A computes it for rows <= 8 with the kernel
// that quantizes on the fly, plus what that kernel quantized and its int32 sums.
extern "C" int llmops_test_fc_decode_dump(const float* x, int64_t rows, int64_t K, const int8_t* weiq, int64_t Ng, int64_t Kg,
                                          int group_k, int64_t N, float* y, int8_t* xq, float* xd, float* gsum, int32_t* acc,
                                          void* workspace, size_t workspace_bytes, llmops_stream_t stream) {
    LLMOPS_TEST_HOOK();
    LLMOPS_REQUIRE(valid_group(group_k));
    LLMOPS_REQUIRE(x != nullptr && weiq != nullptr && y != nullptr && workspace != nullptr);
    LLMOPS_REQUIRE(xq != nullptr && xd != nullptr && gsum != nullptr && acc != nullptr);
    LLMOPS_REQUIRE(rows > 0 && rows <= kMaxGemvRows && K > 0 && Ng > 0 && Kg > 0 && K == Kg * group_k);
    LLMOPS_REQUIRE(N > (Ng - 1) * kGroupN && N <= Ng * kGroupN);
    LLMOPS_REQUIRE(Ng <= kTicketBytes / 4 && Ng * Kg * kGroupN * rows < ((int64_t)1 << 31));
    LLMOPS_REQUIRE(aligned(weiq, 16) && aligned(workspace, 256) && aligned(x, 8) && aligned(xq, 4));
    const FcWorkspace lay = fc_layout(rows, Ng, Kg, group_k);
    if (workspace_bytes < lay.total)
        return fail(LLMOPS_EWORKSPACE, "fc_Q4A needs %zu workspace bytes, got %zu", lay.total, workspace_bytes);
    uint8_t* ws = reinterpret_cast<uint8_t*>(workspace);
    const DumpBufs dump{xq, xd, gsum, acc};
    return launch_gemv_fused(reinterpret_cast<const uint8_t*>(weiq), x, y, reinterpret_cast<float*>(ws + lay.off_part),
                             reinterpret_cast<unsigned*>(ws), rows, Ng, Kg, group_k, N, nullptr, nullptr, 0.0f, 0, nullptr, 0,
                             nullptr, as_stream(stream), &dump);
}
