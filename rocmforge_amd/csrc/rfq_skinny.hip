// Launchers of the matrix-core kernels for few rows of activations (rfq_skinny.hpp).  Compiled RFQ_SKINNY_PARTS times
// (-DRFQ_SKINNY_PART=0..3, the formats of skinny_part_of each), so that the formats build side by side; part 0 also holds
// the entry points.
#include <mutex>

#include "rfq_skinny.hpp"

#ifndef RFQ_SKINNY_PART
#error "compile with -DRFQ_SKINNY_PART=0 .. 3 (see the Makefile)"
#endif

namespace rfq {

constexpr int skinny_part_of(int fmt)
{
    switch (fmt) {
    case RFQ_Q4_0: case RFQ_Q4_K: return 0;
    case RFQ_Q8_0: case RFQ_GGUF_Q8_0: return 1;
    case RFQ_Q6_K: case RFQ_GGUF_Q6_K: case RFQ_MXFP4: return 2;
    case RFQ_GGUF_Q4_0: case RFQ_GGUF_Q4_K: case RFQ_MXFP6_E2M3: return 3;
    default: return -1;
    }
}

namespace {

using namespace skinny;

// Wavefronts of a workgroup: they take the 128-element units of k in turn, so no more than there are units.
int waves_for(int k, int most)
{
    const int units = (k / 32 + 3) / 4;
    return units < most ? units : most;
}

constexpr int GEMV_WAVES = 8;

template <int FMT, int TJ, int MV, bool NORM, bool READY>
int gemv_cfg(const SkinnyGemv &c, hipStream_t s)
{
    const int waves = waves_for(c.k, GEMV_WAVES);
    constexpr int D = 2;                                          // units of W in flight per wavefront
    static_assert(gemv_lds<TJ, MV>(GEMV_WAVES) <= 64 * 1024, "LDS a launch gets without asking");
    const size_t lds = (size_t)gemv_lds<TJ, MV>(waves);
    const int rows = c.w2 != nullptr ? 8 * TJ : 16 * TJ;
    note_kernel(c.w2 != nullptr ? READY ? "gemv_skinny_kernel<%s,%d,%d,%d,pair,ready>" : "gemv_skinny_kernel<%s,%d,%d,%d,pair>"
                                : READY ? "gemv_skinny_kernel<%s,%d,%d,%d,ready>" : "gemv_skinny_kernel<%s,%d,%d,%d>", FMT, TJ, MV, NORM);
    hipLaunchKernelGGL((gemv_skinny_kernel<FMT, TJ, MV, D, GEMV_WAVES, NORM, READY>), dim3((c.n + rows - 1) / rows), dim3(64 * waves), lds, s, c.w, c.x,
                       c.y, c.m, c.n, c.k, c.w2, c.norm_w, c.eps, c.keep_infinities, c.ready);
    RFQ_LAUNCH_CHECK("gemv_skinny_kernel");
    return RFQ_OK;
}

// Row tiles per workgroup: one up to 20 rows per CU, where a second tile would leave CUs without a workgroup, then two, four
// from 52 on: every workgroup converts all of x (Q4_0, 8 vectors, k = 4096: n = 4096 8.8 / 10.7 / 14.5 us with 1 / 2 / 4,
// n = 8192 12.7 / 11.5 / 14.9, n = 14336 23.4 / 18.8 / 18.4; MXFP4 n = 14336 22.8 / 22.1 / 18.8).  Two matrices take an even
// number.  Up to four vectors stay at two: converting half as much x matters less than a second workgroup per CU (14336 x 4096,
// 4 vectors: MXFP4 18.4 / 17.2 us with 4 / 2, Q6_K 23.5 / 22.3, GGUF_Q4_K 16.5 / 15.9), but for pairs of MXFP matrices
// (gate and up of 5120 -> 13824, 2 vectors, with the down projection: MXFP4 69.8 / 72.5).
template <int FMT, int MV, bool NORM>
int gemv_rows(const SkinnyGemv &c, hipStream_t s)
{
    // (prepared x: nothing to share between row tiles, so as many workgroups as the pair or the single matrix allows)
    if constexpr (prepared_format(FMT)) {
        if (c.ready != nullptr && c.w2 != nullptr) return gemv_cfg<FMT, 2, MV, NORM, true>(c, s);
        if constexpr (!NORM)
            if (c.ready != nullptr) return gemv_cfg<FMT, 1, MV, NORM, true>(c, s);
    }
    constexpr bool MX = FMT == RFQ_MXFP4 || FMT == RFQ_MXFP6_E2M3;
    const int cus = device_cu_count();
    const long rows = c.w2 != nullptr ? 2L * c.n : c.n;
    if constexpr (MV == 8 || MX)
        if (rows >= 52L * cus && (MV == 8 || c.w2 != nullptr)) return gemv_cfg<FMT, 4, MV, NORM, false>(c, s);
    if (rows > 20L * cus || c.w2 != nullptr) return gemv_cfg<FMT, 2, MV, NORM, false>(c, s);
    return gemv_cfg<FMT, 1, MV, NORM, false>(c, s);
}

template <int FMT> int gemv_fmt(const SkinnyGemv &c, hipStream_t s)
{
    if (c.norm_w != nullptr) return c.m <= 4 ? gemv_rows<FMT, 4, true>(c, s) : gemv_rows<FMT, 8, true>(c, s);
    return c.m <= 4 ? gemv_rows<FMT, 4, false>(c, s) : gemv_rows<FMT, 8, false>(c, s);
}

// How a workgroup fetches and orders its activations (see gemm_skinny_kernel).
struct Form { bool full, pair, deep, turn; };
// Pairs of groups, two ahead where one row tile leaves registers for it.
[[maybe_unused]] constexpr Form usual(int fmt, int mt, int tj, bool arr) { return {false, in_pairs(fmt, mt, arr, false), mt <= 2 && tj == 1, false}; }
[[maybe_unused]] constexpr Form deep(Form f) { f.deep = true; return f; }
[[maybe_unused]] constexpr Form single(Form f) { f.pair = f.deep = false; return f; }
[[maybe_unused]] constexpr Form turned(Form f) { f.turn = true; return f; }
// (one form took 152 registers instead of 118 with the codes turned: GGUF_Q4_0 200 x 1280 -> 5120 15.4 -> 17.5 us)
[[maybe_unused]] constexpr Form full(int fmt, int mt, bool arr)
{
    const bool pair = in_pairs(fmt, mt, arr, true);
    return {true, pair, false, !arr && !pair && fmt == RFQ_GGUF_Q4_0};
}

template <int FMT, int MT, int TJ, bool ARR, int D, int WAVES, bool FULL, bool PAIR, bool DEEP, bool TURN>
int gemm_launch(const uint8_t *w, const uint8_t *a, void *y, int f16_out, int m, int n, int k, int rows, int slices, hipStream_t s)
{
    constexpr bool STAGED = A16<W<FMT>::ORDER, W<FMT>::PAIRS, ARR>::STAGED;
    constexpr int MOST_LDS = gemm_lds<MT, TJ, STAGED, PAIR>(WAVES);
    static_assert(MOST_LDS <= 160 * 1024, "LDS");
    const int waves = waves_for(k, WAVES);
    const size_t lds = (size_t)gemm_lds<MT, TJ, STAGED, PAIR>(waves);
    if constexpr (MOST_LDS > 64 * 1024) {
        static std::once_flag once;
        static hipError_t err = hipSuccess;
        std::call_once(once, [] {
            err = hipFuncSetAttribute(reinterpret_cast<const void *>(&gemm_skinny_kernel<FMT, MT, TJ, ARR, D, WAVES, FULL, PAIR, DEEP, TURN>),
                                      hipFuncAttributeMaxDynamicSharedMemorySize, MOST_LDS);
        });
        if (err != hipSuccess) return hip_fail(err, "hipFuncSetAttribute(gemm_skinny_kernel)");
    }
    constexpr const char *name = ARR ? FULL ? "gemm_skinny_kernel<%s,%d,%d,%d,arranged,full>" : TURN ? "gemm_skinny_kernel<%s,%d,%d,%d,arranged,turned>" : "gemm_skinny_kernel<%s,%d,%d,%d,arranged>"
        : FULL ? PAIR ? "gemm_skinny_kernel<%s,%d,%d,%d,pairs,full>" : TURN ? "gemm_skinny_kernel<%s,%d,%d,%d,full,turned>" : "gemm_skinny_kernel<%s,%d,%d,%d,full>"
        : PAIR ? DEEP ? "gemm_skinny_kernel<%s,%d,%d,%d,pairs,deep>" : "gemm_skinny_kernel<%s,%d,%d,%d,pairs>" : "gemm_skinny_kernel<%s,%d,%d,%d>";
    note_kernel(name, FMT, MT, TJ, slices);
    hipLaunchKernelGGL((gemm_skinny_kernel<FMT, MT, TJ, ARR, D, WAVES, FULL, PAIR, DEEP, TURN>), dim3((n + 16 * TJ - 1) / (16 * TJ), slices),
                       dim3(64 * waves), lds, s, w, a, y, f16_out, m, n, k, rows);
    RFQ_LAUNCH_CHECK("gemm_skinny_kernel");
    return RFQ_OK;
}

// Two row tiles of W beside two to four operands of rows take 121 .. 172 registers, one workgroup per CU, and with a few spilled 128:
// two per CU, which pays as soon as there are more workgroups than CUs (48 x 4096 -> 14336: GGUF_Q4_K 25.1 / 21.4 us, Q8_0 23.6 /
// 22.3, GGUF_Q6_K 28.2 / 25.1; 282 workgroups, 37 x 2048 -> 9000: GGUF_Q4_K 14.4 / 12.0; with 160 workgroups, 64 x 1280 -> 5120: Q8_0 6.8 / 7.4, GGUF_Q4_0 6.7 / 8.0).
// Not GGUF_Q8_0 with four operands, which spills most (60 x 1024 -> 14336 16.0 against 13.9 without, 60 x 4096 -> 8320 34.6 / 30.8).
template <int FMT, int MT, int TJ, bool ARR, int D, int WAVES>
int gemm_cfg(const uint8_t *w, const uint8_t *a, void *y, int f16_out, int m, int n, int k, int rows, int slices, hipStream_t s)
{
    constexpr Form USUAL = usual(FMT, MT, TJ, ARR);
#define RFQ_GEMM_FORM(F)                                                                                     \
    do {                                                                                                     \
        constexpr Form form = F;                                                                             \
        return gemm_launch<FMT, MT, TJ, ARR, D, WAVES, form.full, form.pair, form.deep, form.turn>(w, a, y, f16_out, m, n, k, rows, slices, s); \
    } while (0)
    const bool more = (long)((n + 16 * TJ - 1) / (16 * TJ)) * slices > device_cu_count();
    if constexpr (ARR) {
        // Arranged: codes turned once for all operands, but activations where that cost registers or came too late behind the load of W
        // (17 x 1024 -> 14336 Q8_0 11.6 -> 10.5 us; 17 x 11264 -> 1536 15.7 -> 14.4; with short rows the codes, 9 x 1024 -> 768 3.58 / 3.42).
        if constexpr (FMT == RFQ_Q8_0 && TJ == 2 && MT == 2) RFQ_GEMM_FORM(turned(USUAL));
        if constexpr ((FMT == RFQ_Q8_0 || FMT == RFQ_GGUF_Q8_0) && TJ == 1 && MT == 1)
            if (k > 2048) RFQ_GEMM_FORM(turned(USUAL));
        if constexpr (FMT == RFQ_Q8_0 && TJ == 1 && MT == 2)
            if (k > 4096) RFQ_GEMM_FORM(turned(USUAL));
        // (two registers over the 128 for two workgroups per CU: 17 x 1024 -> 14336 8.7 -> 7.2 us; with 192 workgroups 7.35 / 7.7)
        if constexpr (FMT == RFQ_GGUF_Q4_K && TJ == 2 && MT == 2)
            if (more) RFQ_GEMM_FORM(full(FMT, MT, ARR));
        RFQ_GEMM_FORM(USUAL);
    } else {
        // (one unit of k to a wavefront: single groups, whose second fetch does not wait for a whole pair; 60 x 1024 -> 14336 Q8_0 13.6 /
        // 12.8 us, 90 rows GGUF_Q8_0 17.9 / 17.2, 33 x 1024 -> 4096 4.8 / 4.6, 75 x 2048 -> 1792 6.45 / 6.1, 75 x 3072 -> 1536 7.9 / 7.45)
        if constexpr (TJ == 2 && ((FMT == RFQ_Q8_0 && MT == 4) || (FMT == RFQ_GGUF_Q8_0 && MT == 6)))
            if (more && k <= 1024) RFQ_GEMM_FORM(single(USUAL));
        if constexpr (FMT == RFQ_GGUF_Q8_0 && TJ == 1 && MT == 3) {
            if (k < 4096) RFQ_GEMM_FORM(single(USUAL));
            // (its ten registers a unit leave one unit of W in flight: activations further ahead, 33 x 4096 -> 4096 11.9 -> 10.6 us)
            RFQ_GEMM_FORM(deep(USUAL));
        }
        if constexpr (TJ == 2 && MT >= 2 && MT <= 4 && !(FMT == RFQ_GGUF_Q8_0 && MT == 4))
            if (more) RFQ_GEMM_FORM(full(FMT, MT, ARR));
        // One workgroup per CU has registers for two pairs ahead: long rows of the 4- and 6-bit layouts with nothing else to wait behind
        // (9 x 8192 -> 5120 Q4_K 20.5 -> 18.4 us, Q6_K 20.2 -> 18.9, GGUF_Q4_K 15.7 -> 14.4, Q4_0 16.5 -> 15.6; Q4_K short ones too, 6.8 -> 6.2
        // with k = 1280, where Q4_0 and GGUF_Q4_K lose 2 %; the 8-bit layouts lose 1 to 7 %).
        if constexpr (TJ == 2 && MT <= 2 && (FMT == RFQ_Q4_K || FMT == RFQ_Q6_K || FMT == RFQ_Q4_0 || FMT == RFQ_GGUF_Q4_K))
            if (!more && (FMT == RFQ_Q4_K || k >= 4096)) RFQ_GEMM_FORM(deep(USUAL));
        // (single groups stay ahead in two places: long rows of the 4-bit GGUF layouts, 20 x 14336 -> 4096 GGUF_Q4_K 20.6 / 21.7 us, and six
        // operands of the Q6_K layouts in several rounds, 160 x 3072 -> 6144 GGUF_Q6_K 33.0 / 34.3)
        if constexpr (TJ == 1 && MT == 2 && (FMT == RFQ_GGUF_Q4_0 || FMT == RFQ_GGUF_Q4_K))
            if (k > 8192) RFQ_GEMM_FORM(single(USUAL));
        if constexpr (TJ == 2 && (MT == 5 || MT == 6) && (FMT == RFQ_Q6_K || FMT == RFQ_GGUF_Q6_K))
            if (more) RFQ_GEMM_FORM(single(USUAL));
        RFQ_GEMM_FORM(USUAL);
    }
#undef RFQ_GEMM_FORM
}

// 16-row operands per workgroup at most: six with one row tile (eight leave its registers one wavefront per SIMD: Q8_0
// 4096 -> 1024, 100 rows, 28 us with eight, 160 rows 15 with twice five); eight with two (8192 rows of 4096, 100 rows: Q8_0
// 28.8 us, 40 with two slices of four), but four for the scale-only 4-bit layouts, whose forms of eight spilled (Q4_0, 208
// rows, 1792 -> 5713: 79.7 us with eight, 45 with four).
constexpr int most_tiles(int fmt, bool two) { return !two ? 6 : fmt == RFQ_Q4_0 || fmt == RFQ_GGUF_Q4_0 ? 4 : 8; }

// The rows of a in slices of at most 16 * most_tiles, as even as 16 rows allow.  Where W gives fewer workgroups than the part
// has CUs there are more slices, so that every CU gets one: a workgroup's time grows with its operands of 16 rows, and W that
// small stays in the caches (4096 -> 1024, Q8_0: 48 rows 9.8 -> 6.2 us, 160 rows 15.2 -> 9.8; 1280 -> 1280 GGUF_Q4_K 100 rows
// 8.9 -> 5.2).
struct Slices { int count, tiles; };
Slices slices_of(int fmt, int m, int n, bool two)
{
    const int tiles = (m + 15) / 16, most = most_tiles(fmt, two), groups = two ? (n + 31) / 32 : (n + 15) / 16;
    int count = (tiles + most - 1) / most;
    const int room = device_cu_count() / groups;
    if (room > count) count = room < tiles ? room : tiles;
    const int per = (tiles + count - 1) / count;
    return {(tiles + per - 1) / per, per};
}

// Two row tiles per workgroup from about one workgroup per CU on: a workgroup reads all activations of its slice whether
// it multiplies 16 rows of W or 32 (Q8_0, k = 4096, 48 rows: n = 8192 23.5 -> 18.7 us, n = 14336 43.2 -> 32.7; with fewer
// workgroups than CUs one tile is ahead, n = 4096 11.4 against 13.7 us).
bool two_tiles(int fmt, int m, int n)
{
    return (n + 15) / 16 * slices_of(fmt, m, n, false).count > device_cu_count() + device_cu_count() / 8;
}

template <int FMT, int TJ, bool ARR>
int gemm_mt(const uint8_t *w, const uint8_t *a, void *y, int f16_out, int m, int n, int k, hipStream_t s)
{
    constexpr int MOST = most_tiles(FMT, TJ == 2);
    const Slices sl = slices_of(FMT, m, n, TJ == 2);
    const int rows = 16 * sl.tiles, slices = sl.count;
    // units of W in flight per wavefront: two, one where the registers of a unit leave no room for two
    constexpr int D = TJ * W<FMT>::NR > 9 ? 1 : 2;
    switch (sl.tiles) {
    case 1: return gemm_cfg<FMT, 1, TJ, ARR, 2, 8>(w, a, y, f16_out, m, n, k, rows, slices, s);
    case 2: return gemm_cfg<FMT, 2, TJ, ARR, 2, 8>(w, a, y, f16_out, m, n, k, rows, slices, s);
    case 3: return gemm_cfg<FMT, 3, TJ, ARR, D, 8>(w, a, y, f16_out, m, n, k, rows, slices, s);
    case 4: return gemm_cfg<FMT, 4, TJ, ARR, D, 8>(w, a, y, f16_out, m, n, k, rows, slices, s);
    default:
        // (five beside two row tiles: 160 x 4096 -> 4096 Q8_0 18.9 us as six, 17.7 as five, Q/K/V of 160 tokens GGUF_Q4_K 36.1 / 35.3; but
        // GGUF_Q6_K in several rounds 17.9 / 18.6, 130 x 1280 -> 5120, and arranged 10.7 / 11.05, 75 x 1280 -> 5120, 41.0 / 42.0 with k = 8192)
        if constexpr (MOST >= 6 && TJ == 2) {
            const bool rounds = (long)((n + 31) / 32) * slices > device_cu_count();
            if (sl.tiles == 5 && !(FMT == RFQ_GGUF_Q6_K && (ARR || rounds))) return gemm_cfg<FMT, 5, TJ, ARR, D, 8>(w, a, y, f16_out, m, n, k, rows, slices, s);
        }
        if constexpr (MOST >= 6)
            if (sl.tiles <= 6) return gemm_cfg<FMT, 6, TJ, ARR, D, 8>(w, a, y, f16_out, m, n, k, rows, slices, s);
        if constexpr (MOST >= 8)
            if (sl.tiles <= 8) return gemm_cfg<FMT, 8, TJ, ARR, D, 8>(w, a, y, f16_out, m, n, k, rows, slices, s);
        return fail(RFQ_E_UNSUPPORTED, "rfq_gemm_f16: slices of %d rows", rows);
    }
}

template <int FMT>
int gemm_fmt(const uint8_t *w, const uint8_t *a, bool arranged, void *y, int f16_out, int m, int n, int k, hipStream_t s)
{
    if (two_tiles(FMT, m, n)) return arranged ? gemm_mt<FMT, 2, true>(w, a, y, f16_out, m, n, k, s) : gemm_mt<FMT, 2, false>(w, a, y, f16_out, m, n, k, s);
    return arranged ? gemm_mt<FMT, 1, true>(w, a, y, f16_out, m, n, k, s) : gemm_mt<FMT, 1, false>(w, a, y, f16_out, m, n, k, s);
}

} // namespace

#define RFQ_SKINNY_CAT2(a, b) a##b
#define RFQ_SKINNY_CAT(a, b) RFQ_SKINNY_CAT2(a, b)
#define RFQ_SKINNY_CASES(CALL)                                                                     \
    return [&](auto part) -> int {                                                                  \
        constexpr int P = decltype(part)::value;                                                    \
        switch (fmt) {                                                                              \
        case RFQ_Q4_0: if constexpr (skinny_part_of(RFQ_Q4_0) == P) return CALL(RFQ_Q4_0); break;   \
        case RFQ_Q8_0: if constexpr (skinny_part_of(RFQ_Q8_0) == P) return CALL(RFQ_Q8_0); break;   \
        case RFQ_Q4_K: if constexpr (skinny_part_of(RFQ_Q4_K) == P) return CALL(RFQ_Q4_K); break;   \
        case RFQ_Q6_K: if constexpr (skinny_part_of(RFQ_Q6_K) == P) return CALL(RFQ_Q6_K); break;   \
        case RFQ_GGUF_Q4_0: if constexpr (skinny_part_of(RFQ_GGUF_Q4_0) == P) return CALL(RFQ_GGUF_Q4_0); break; \
        case RFQ_GGUF_Q8_0: if constexpr (skinny_part_of(RFQ_GGUF_Q8_0) == P) return CALL(RFQ_GGUF_Q8_0); break; \
        case RFQ_GGUF_Q4_K: if constexpr (skinny_part_of(RFQ_GGUF_Q4_K) == P) return CALL(RFQ_GGUF_Q4_K); break; \
        case RFQ_GGUF_Q6_K: if constexpr (skinny_part_of(RFQ_GGUF_Q6_K) == P) return CALL(RFQ_GGUF_Q6_K); break; \
        default: break;                                                                             \
        }                                                                                           \
        return fail(RFQ_E_UNSUPPORTED, "no few-row kernel for format %d in this part of the build", fmt); \
    }(std::integral_constant<int, RFQ_SKINNY_PART>{})

int RFQ_SKINNY_CAT(launch_skinny_gemv_part, RFQ_SKINNY_PART)(int fmt, const SkinnyGemv &c, hipStream_t s)
{
#define RFQ_SKINNY_GEMV(F) gemv_fmt<F>(c, s)
    if constexpr (skinny_part_of(RFQ_MXFP4) == RFQ_SKINNY_PART)
        if (fmt == RFQ_MXFP4) return RFQ_SKINNY_GEMV(RFQ_MXFP4);
    if constexpr (skinny_part_of(RFQ_MXFP6_E2M3) == RFQ_SKINNY_PART)
        if (fmt == RFQ_MXFP6_E2M3) return RFQ_SKINNY_GEMV(RFQ_MXFP6_E2M3);
    RFQ_SKINNY_CASES(RFQ_SKINNY_GEMV);
}

int RFQ_SKINNY_CAT(launch_skinny_gemm_part, RFQ_SKINNY_PART)(int fmt, const uint8_t *w, const uint8_t *a, bool arranged, void *y, int f16_out,
                                                             int m, int n, int k, hipStream_t s)
{
#define RFQ_SKINNY_GEMM(F) gemm_fmt<F>(w, a, arranged, y, f16_out, m, n, k, s)
    RFQ_SKINNY_CASES(RFQ_SKINNY_GEMM);
}

#if RFQ_SKINNY_PART == 0

// Whether the few-row kernel is the faster one for a prompt, from estimates of both in microseconds.  The few-row kernel's
// time grows with the 16-row operands a workgroup multiplies per 1024 k (all of them in every workgroup) and, beyond one
// workgroup per CU, with the number of workgroups; the tiled kernel's is nearly flat up to 256 rows: a workgroup's own pass
// over k, in `parts` parts, plus the f32 parts written and read again.  With parts == 1 the answer depends on the shape alone, so
// that arranged and plain activations take the same kernel and give the same bits.
// Q4_K and the Q6_K layouts: the estimates lean to the tiled kernel; of the shapes measured with both (n 768..14336, k
// 1024..14336, 9..255 rows, plain and arranged) three that go to the few-row kernel are slower there by more than 4 % (7 % at most).
// Q4_0, Q8_0, their GGUF layouts and GGUF_Q4_K: the other kernel is the one on integer codes, and the line is drawn by precision.  That
// kernel adds a row in float32 in longer runs: error against 64 bits up to 4.1e-7, 1.5 times the few-row kernel's (0.93..2.9, at
// most 1.6e-7 there), GGUF_Q4_K up to 8.4e-7, 2.7 times (1.4..4.3, at most 2.1e-7).  So a call of few rows goes to it only where it is
// far ahead.  (codes / few-row: Q8_0 9 x 4096 -> 4096 18.7 / 8.0 us, 112 x 4096 -> 4096 23.2 / 16.7, 56 x 4096 -> 14336 29.8 / 33.5, 80 x
// 14336 -> 4096 37.2 / 48.3, 64 x 14336 -> 4096 30.4 / 38.3, 255 x 4096 -> 14336 57.8 / 102.7.  Of 5250 calls measured with both, 4646 go to
// the few-row kernel, 209 of them more than 10 % slower than the other would be, at most 1.67 times; 604 stay, and 40 of those would
// gain more than 10 % by going.)
bool prefer_skinny_gemm(int fmt, int m, int n, int k, int parts)
{
    const double cus = device_cu_count(), ku = k / 1024.0;
    const bool two = two_tiles(fmt, m, n);
    const Slices sl = slices_of(fmt, m, n, two);
    const int row_tiles = (n + 15) / 16 * sl.count;
    const double rounds = two ? 1.45 * (row_tiles / 2 > cus ? row_tiles / 2 / cus : 1.0) : 1.0;
    const double few = 3.0 + ku * rounds * (0.5 + 0.7 * (sl.tiles <= 4 ? sl.tiles : sl.tiles <= 6 ? 6 : 8));
    const double per_ku = fmt == RFQ_Q4_K ? 10.0 : fmt == RFQ_GGUF_Q4_K ? 13.0 : fmt == RFQ_GGUF_Q6_K ? 29.0 : 21.5;
    const int groups = ((m + 255) / 256) * ((n + 127) / 128) * parts;
    double tiled = 8.0 + per_ku * ku / parts * (groups > cus ? groups / cus : 1.0);
    if (parts > 1) tiled += 4.0 + 8.0 * parts * m * (double)n / 5e6;
    return few < tiled;
}

int launch_prepare_x(int fmt, const SkinnyGemv &c, uint8_t *out, hipStream_t s)
{
    const dim3 grid((c.k + 127) / 128), block(c.m <= 4 ? 64 : 128);
#define RFQ_PREPARE(F)                                                                                                                      \
    hipLaunchKernelGGL((prepare_x_kernel<W<F>::ORDER, W<F>::PAIRS>), grid, block, 0, s, c.x, c.norm_w, c.m, c.k, out, c.keep_infinities); \
    break
    switch (fmt) {
    case RFQ_Q4_0: RFQ_PREPARE(RFQ_Q4_0);
    case RFQ_MXFP6_E2M3: RFQ_PREPARE(RFQ_MXFP6_E2M3);
    case RFQ_GGUF_Q4_0: RFQ_PREPARE(RFQ_GGUF_Q4_0);
    case RFQ_GGUF_Q4_K: RFQ_PREPARE(RFQ_GGUF_Q4_K);
    case RFQ_MXFP4: RFQ_PREPARE(RFQ_MXFP4);
    default: return fail(RFQ_E_UNSUPPORTED, "no few-row kernel on prepared x for format %d", fmt);
    }
#undef RFQ_PREPARE
    RFQ_LAUNCH_CHECK("prepare_x_kernel");
    return RFQ_OK;
}

int launch_skinny_gemv(int fmt, const SkinnyGemv &c, hipStream_t s)
{
    switch (skinny_part_of(fmt)) {
    case 0: return launch_skinny_gemv_part0(fmt, c, s);
    case 1: return launch_skinny_gemv_part1(fmt, c, s);
    case 2: return launch_skinny_gemv_part2(fmt, c, s);
    case 3: return launch_skinny_gemv_part3(fmt, c, s);
    default: return fail(RFQ_E_UNSUPPORTED, "no few-row kernel for format %d", fmt);
    }
}

int launch_skinny_gemm(int fmt, const uint8_t *w, const uint8_t *a, bool arranged, void *y, bool f16_out, int m, int n, int k, hipStream_t s)
{
    switch (skinny_part_of(fmt)) {
    case 0: return launch_skinny_gemm_part0(fmt, w, a, arranged, y, f16_out, m, n, k, s);
    case 1: return launch_skinny_gemm_part1(fmt, w, a, arranged, y, f16_out, m, n, k, s);
    case 2: return launch_skinny_gemm_part2(fmt, w, a, arranged, y, f16_out, m, n, k, s);
    case 3: return launch_skinny_gemm_part3(fmt, w, a, arranged, y, f16_out, m, n, k, s);
    default: return fail(RFQ_E_UNSUPPORTED, "no few-row kernel for format %d", fmt);
    }
}

#endif

} // namespace rfq
