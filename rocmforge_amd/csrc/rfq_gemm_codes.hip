// Launcher of the prefill GEMM on integer codes (rfq_gemm_codes.hpp).
#include <mutex>

#include "rfq_gemm_codes.hpp"

namespace rfq {

// 64, 128, 192 or 256 rows: what makes the launch shortest.  One workgroup fits a CU (LDS); a stage of 128 k takes it
// about 0.5 us + 0.48 per 64 rows (Q8_0 512 x 4096 -> 14336: 1.0, 1.5, 1.8, 2.4 us; whole calls 137, 105, 121, 82-87 us; 700 x
// 3840 -> 3712 67, 50, 60, 70; 333 x 13824 -> 5120 119, 109, 83, 96).  GGUF_Q4_K takes 256 rows through the kernel laid out by hand,
// whose stage is 2.1 us: against it (1333 shapes of 256..2048 rows, plain and arranged) this kernel takes 0.84..1.0 of the time, up to
// 1.05 in single rounds of 1024 k, where its estimate is 0.80 of 2.42 us a round, and 1.0..1.16 where it is 0.90 to 0.96.
int codes_rows(int fmt, int m, int n, int kparts)
{
    const int cus = device_cu_count();
    int best = 256;
    double least = 0.0;
    for (int ti = 4; ti >= 1; ti--) {
        const long groups = (long)((m + 64 * ti - 1) / (64 * ti)) * ((n + codes::BN - 1) / codes::BN) * kparts;
        const double t = (double)((groups + cus - 1) / cus) * (ti == 4 && fmt == RFQ_GGUF_Q4_K ? 2.1 : 0.5 + 0.48 * ti);
        if (ti == 4 || t < least) { best = 64 * ti; least = t; }
    }
    return best;
}

namespace {

using namespace codes;

// Four wavefronts along m, two along n: 64 columns of W to a wavefront, the A operands of a row tile fetched twice (eight
// along m, A fetched once and twice the fragments from LDS: level, GGUF_Q4_K 88 -> 97 us).
template <int FMT, int WM, int TI>
int launch_form(const uint8_t *w, const uint8_t *at, const uint8_t *s2, void *out, bool f16_out, int m, int n, int k, int kparts, hipStream_t s)
{
    static std::once_flag once;
    static hipError_t err = hipSuccess;
    std::call_once(once, [] {
        err = hipFuncSetAttribute(reinterpret_cast<const void *>(&gemm_codes_kernel<FMT, WM, TI>), hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes<FMT>());
    });
    if (err != hipSuccess) return hip_fail(err, "hipFuncSetAttribute(gemm_codes_kernel)");
    constexpr int BM = 16 * WM * TI;
    const int tiles = ((m + BM - 1) / BM) * ((n + BN - 1) / BN);
    hipLaunchKernelGGL((gemm_codes_kernel<FMT, WM, TI>), dim3(tiles * kparts), dim3(512), lds_bytes<FMT>(), s, w, reinterpret_cast<const v4u *>(at), s2, out,
                       (int)f16_out, m, n, k, kparts);
    RFQ_LAUNCH_CHECK("gemm_codes_kernel");
    return RFQ_OK;
}

template <int FMT>
int launch_fmt(const uint8_t *w, const uint8_t *at, const uint8_t *s2, void *out, bool f16_out, int m, int n, int k, int kparts, hipStream_t s)
{
    switch (codes_rows(FMT, m, n, kparts)) {
    case 64: return launch_form<FMT, 4, 1>(w, at, s2, out, f16_out, m, n, k, kparts, s);
    case 128: return launch_form<FMT, 4, 2>(w, at, s2, out, f16_out, m, n, k, kparts, s);
    case 192: return launch_form<FMT, 4, 3>(w, at, s2, out, f16_out, m, n, k, kparts, s);
    default:
        if constexpr (FMT != RFQ_GGUF_Q4_K) return launch_form<FMT, 4, 4>(w, at, s2, out, f16_out, m, n, k, kparts, s);
        return fail(RFQ_E_UNSUPPORTED, "no code-operand form of 256 rows for GGUF_Q4_K");   // (gemm_kq_kernel takes them)
    }
}

} // namespace

int launch_gemm_codes(int fmt, const uint8_t *w, const uint8_t *at, const uint8_t *s2, void *out, bool f16_out, int m, int n, int k, int kparts, hipStream_t s)
{
    switch (fmt) {
    case RFQ_Q4_0: return launch_fmt<RFQ_Q4_0>(w, at, s2, out, f16_out, m, n, k, kparts, s);
    case RFQ_Q8_0: return launch_fmt<RFQ_Q8_0>(w, at, s2, out, f16_out, m, n, k, kparts, s);
    case RFQ_GGUF_Q4_0: return launch_fmt<RFQ_GGUF_Q4_0>(w, at, s2, out, f16_out, m, n, k, kparts, s);
    case RFQ_GGUF_Q8_0: return launch_fmt<RFQ_GGUF_Q8_0>(w, at, s2, out, f16_out, m, n, k, kparts, s);
    case RFQ_GGUF_Q4_K: return launch_fmt<RFQ_GGUF_Q4_K>(w, at, s2, out, f16_out, m, n, k, kparts, s);
    default: return fail(RFQ_E_UNSUPPORTED, "no code-operand kernel for format %d", fmt);
    }
}

} // namespace rfq
