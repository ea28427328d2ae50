// Prefill GEMM on integer codes:  out[m, n] = A[m, k] (fp16, arranged) . dequant(W)[n, k]^T  for the formats whose scale
// belongs to 32 elements (Q4_0, Q8_0, GGUF_Q4_0, GGUF_Q8_0), and for GGUF_Q4_K where tiles of fewer than 256 rows save time (codes_rows).
//
// What bounds these calls is the matrix pipe and, behind it, the vector instructions: they do not run beside each other
// freely (a v_mfma_f32_16x16x32_f16 followed by no / one / two / three / four v_fma_f32 takes 9.0 / 9.3 / 10.2 / 11.4 / 13.1
// ns with two wavefronts per SIMD and random operands).  Two fp16 operands per weight (hi + lo) need two matrix
// instructions, 18 ns, before their decoding.  Hence:
//   * The operand of the matrix instruction is the CODE of a weight, exact in fp16; one instruction covers one 32-element
//     group of 16 weight rows, and the group's scale multiplies its sum in float32: acc += scale * sum.  Weights are never
//     rounded and a scale may have any float32 value.  Error against 64 bits 1.0e-6 (hi + lo) -> 2.1e-7 at k = 4096.
//   * GGUF_Q4_K: the operand is sc * q, an integer up to 945; acc runs in units of the running super-block's d and is
//     multiplied by d_prev / d_next between super-blocks; the mins are one more matrix instruction per super-block
//     over the group sums of the activations.
//   * The scale of a lane's weight row is one register where W is the second operand, so W is.
//   * A workgroup is eight wavefronts (two per SIMD) over 64, 128, 192 or 256 rows of A x 128 rows of W: 4 x 2 wavefronts of
//     16 .. 64 x 64.  Rows that do not fill a tile are paid for as matrix instructions, hence four sizes.
//   * A stage is 128 k: thread t fetches group t % 4 of weight row t / 4 (neighbouring lanes on neighbouring bytes), two
//     stages ahead, decodes it beside the matrix instructions into one of three LDS buffers (operand order: reads
//     are linear, the planes of the four groups skewed by 16 banks for the writes) and a stage ends in one barrier; the
//     next stage's first fragments are read before it.  Activations go from the arranged buffer into the operand registers a
//     stage ahead and never pass through LDS.
// Measured (calls on plain activations, with their arrangement and, where split along k, the sum of the parts):
//   512 x 4096 -> 14336   Q8_0 121 -> 82-87 us, GGUF_Q4_0 120 -> 84       333 x 13824 -> 5120  Q8_0 140 -> 83 us
//   300 x 4096 -> 4096    Q8_0 43.6 -> 31.8                               128 x 4096 -> 14336  Q8_0 67.5 -> 36.6
//   256 x 11008 -> 1792   Q8_0 238 -> 80, GGUF_Q4_K 143 -> 90             300 x 1280 -> 5120   Q8_0 35.9 -> 17.2
// Of the 82 us at 512 x 4096 -> 14336 (75 for this kernel: wavefronts issue vector instructions for 67 % of its cycles and wait
// for 26 %), loading A accounts for 5, decoding for 7, fetching W for 1.5; without any of them 70.
#pragma once
#include <type_traits>
#include <utility>

#include "rfq_code_operands.hpp"

namespace rfq {
namespace codes {

typedef uint32_t v4u_a4 __attribute__((ext_vector_type(4), aligned(4)));
template <int N> struct IC { static constexpr int value = N; };
// f(IC<0>{}) ... f(IC<N - 1>{}): a loop that is unrolled whatever its size
template <typename F, int... X> __device__ __forceinline__ void each(F &&f, std::integer_sequence<int, X...>) { (f(IC<X>{}), ...); }
template <int N, typename F> __device__ __forceinline__ void each(F &&f) { each(f, std::make_integer_sequence<int, N>{}); }

// Group<FMT>: the bytes of one 32-element group of a weight row.  octet<o>(): elements 8 o .. 8 o + 7 as fp16 codes in the
// order of arranged activations, (0,4)(1,5)(2,6)(3,7).
template <int FMT> struct Group;

template <> struct Group<RFQ_Q4_0> {
    uint32_t d[5];
    __device__ __forceinline__ void load(const uint8_t *p)
    {
        d[0] = ld<uint32_t>(p);
        const v4u_a4 v = *reinterpret_cast<const v4u_a4 *>(p + 4);
#pragma unroll
        for (int i = 0; i < 4; i++) d[1 + i] = v[i];
    }
    template <int O> __device__ __forceinline__ v4u octet() const
    {
        const uint32_t q = d[1 + O];
        return v4u{nib2h<0>(q, -8.f), nib2h<4>(q, -8.f), nib2h<8>(q, -8.f), nib2h<12>(q, -8.f)};
    }
    __device__ __forceinline__ float scale() const { return __uint_as_float(d[0]); }
};

// GGUF blocks start on multiples of 2: the aligned dwords that hold the block, o (0 or 2) bytes before it.
template <> struct Group<RFQ_GGUF_Q4_0> {
    uint32_t d[5], o;
    __device__ __forceinline__ void load(const uint8_t *p)
    {
        o = (uint32_t)(reinterpret_cast<uintptr_t>(p) & 2u);
        const uint8_t *a = p - o;
        const v4u_a4 v = *reinterpret_cast<const v4u_a4 *>(a);
#pragma unroll
        for (int i = 0; i < 4; i++) d[i] = v[i];
        d[4] = ld<uint32_t>(a + 16);
    }
    // octets 0 and 1: the low nibbles of bytes 0..7 and 8..15, octets 2 and 3 the high ones
    template <int O> __device__ __forceinline__ v4u octet() const
    {
        const uint32_t sel = 0x05040302u + o * 0x01010101u;
        constexpr int B = 2 * (O & 1);
        const uint32_t a = __builtin_amdgcn_perm(d[B + 1], d[B], sel), b = __builtin_amdgcn_perm(d[B + 2], d[B + 1], sel);
        const uint32_t z01 = __builtin_amdgcn_perm(b, a, 0x05040100u), z23 = __builtin_amdgcn_perm(b, a, 0x07060302u);
        constexpr int S = O < 2 ? 0 : 4;
        return v4u{nib2h<S>(z01, -8.f), nib2h<S + 8>(z01, -8.f), nib2h<S>(z23, -8.f), nib2h<S + 8>(z23, -8.f)};
    }
    __device__ __forceinline__ float scale() const { return f16_bits_to_f32((uint16_t)(d[0] >> (8u * o))); }
};

template <int FMT> struct Group8 {                               // Q8_0 (f32 scale, byte - 128), GGUF_Q8_0 (f16 scale, int8)
    uint32_t d[9], o;
    __device__ __forceinline__ void load(const uint8_t *p)
    {
        o = FMT == RFQ_Q8_0 ? 0u : (uint32_t)(reinterpret_cast<uintptr_t>(p) & 2u);
        const uint8_t *a = p - o;
        const v4u_a4 u = *reinterpret_cast<const v4u_a4 *>(a), v = *reinterpret_cast<const v4u_a4 *>(a + 16);
#pragma unroll
        for (int i = 0; i < 4; i++) { d[i] = u[i]; d[4 + i] = v[i]; }
        d[8] = ld<uint32_t>(a + 32);
    }
    template <int O> __device__ __forceinline__ v4u octet() const
    {
        uint32_t a, b;
        if constexpr (FMT == RFQ_Q8_0) {
            a = d[1 + 2 * O];
            b = d[2 + 2 * O];
        } else {
            const uint32_t sel = 0x05040302u + o * 0x01010101u;
            a = __builtin_amdgcn_perm(d[2 * O + 1], d[2 * O], sel) ^ 0x80808080u;
            b = __builtin_amdgcn_perm(d[2 * O + 2], d[2 * O + 1], sel) ^ 0x80808080u;
        }
        uint32_t p[4];
        bytes2h(__builtin_amdgcn_perm(b, a, 0x05010400u), -128.f, p[0], p[1]);
        bytes2h(__builtin_amdgcn_perm(b, a, 0x07030602u), -128.f, p[2], p[3]);
        return v4u{p[0], p[1], p[2], p[3]};
    }
    __device__ __forceinline__ float scale() const
    {
        return FMT == RFQ_Q8_0 ? __uint_as_float(d[0]) : f16_bits_to_f32((uint16_t)(d[0] >> (8u * o)));
    }
};
template <> struct Group<RFQ_Q8_0> : Group8<RFQ_Q8_0> {};
template <> struct Group<RFQ_GGUF_Q8_0> : Group8<RFQ_GGUF_Q8_0> {};

// GGUF_Q4_K: the operand is sc * q, an integer up to 945.  A stage is half a super-block; the header (d, dmin, 6-bit scales
// and mins) is fetched once per super-block and serves both halves.
template <> struct Group<RFQ_GGUF_Q4_K> {
    uint32_t d[8];
    __device__ __forceinline__ void load(const uint8_t *p)       // the 32 bytes whose low or high nibbles are the group
    {
        const v4u_a4 u = *reinterpret_cast<const v4u_a4 *>(p), v = *reinterpret_cast<const v4u_a4 *>(p + 16);
#pragma unroll
        for (int i = 0; i < 4; i++) { d[i] = u[i]; d[4 + i] = v[i]; }
    }
    static __device__ __forceinline__ uint32_t scaled(uint32_t d, v2h sc, v2h off)   // nibbles at bits 0 and 16
    {
        uint32_t mask = 0x000F000Fu, magic = 0x64006400u;
        asm("" : "+s"(mask));
        asm("" : "+v"(magic));
        const uint32_t bits = (d & mask) | magic;
        v2h h;
        __builtin_memcpy(&h, &bits, 4);
        h = __builtin_elementwise_fma(h, sc, off);               // (1024 + q) * sc - 1024 sc: exact, one rounding of a small integer
        uint32_t o;
        __builtin_memcpy(&o, &h, 4);
        return o;
    }
    template <int O> __device__ __forceinline__ v4u octet(uint32_t shift, v2h sc, v2h off) const
    {
        const uint32_t a = d[2 * O] >> shift, b = d[2 * O + 1] >> shift;
        const uint32_t z01 = __builtin_amdgcn_perm(b, a, 0x05040100u), z23 = __builtin_amdgcn_perm(b, a, 0x07060302u);
        return v4u{scaled(z01, sc, off), scaled(z01 >> 8, sc, off), scaled(z23, sc, off), scaled(z23 >> 8, sc, off)};
    }
};

// LDS write completes, then everyone meets; global loads stay in flight.
__device__ __forceinline__ void lds_barrier()
{
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xC07F); // lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

constexpr int BN = 128;                                           // weight rows of a workgroup
constexpr int PLANE = BN * 64 + 64;                               // one group of them in LDS (the planes of a row's four groups bank-skewed)
constexpr int BUF = 4 * PLANE + 4 * BN * 4;                       // one stage (128 k): codes, scales
// GGUF_Q4_K, per super-block: the mins of a row's eight groups as fp16 pairs, then per row the ratio, the min's factor, the unit
constexpr int SB_AREA = BN * 32 + 3 * BN * 4;
template <int FMT> constexpr int lds_bytes() { return 3 * BUF + (FMT == RFQ_GGUF_Q4_K ? 2 * SB_AREA : 0); }

// Eight wavefronts, WM x WN; each multiplies TI x TJ tiles of 16 x 16.  kparts > 1 (few output tiles, long k): kparts workgroups
// per tile, each contracts [k0, k0 + K) of the rows and writes its f32 partial tile to outp[part][M][N].
template <int FMT, int WM, int TI>
__global__ void __launch_bounds__(512)
gemm_codes_kernel(const uint8_t *__restrict__ w, const v4u *__restrict__ at, const uint8_t *__restrict__ s2, void *__restrict__ outp, int f16_out, int M, int N, int Kfull, int kparts)
{
    constexpr int WN = 8 / WM, TJ = BN / 16 / WN, T = TI * TJ, BM = 16 * WM * TI;
    // INT: acc runs in units of the running super-block's d
    constexpr bool INT = FMT == RFQ_GGUF_Q4_K;
    constexpr int LAG = T >= 8 && !INT ? 3 : 2;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    const int tid = threadIdx.x, lane = tid & 63, i = lane & 15, q = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wm = wave % WM, wn = wave / WM;
    const int K = Kfull / kparts;
    const int tiles_m = (M + BM - 1) / BM;
    // (workgroups go round-robin to the 8 XCDs: each gets a contiguous run of tiles, so that the m tiles of a W tile meet in one L2)
    const int nwg = gridDim.x;
    const int slot = nwg % 8 == 0 ? (int)(blockIdx.x % 8) * (nwg / 8) + (int)(blockIdx.x / 8) : (int)blockIdx.x;
    const int tiles_all = nwg / kparts, part = slot / tiles_all, tile = slot % tiles_all;
    const int k0 = part * K, m0 = tile % tiles_m * BM, n0 = tile / tiles_m * BN;
    const int groups = K >> 5, nst = (groups + 3) >> 2;           // stages of 128 k
    const int kst = (K + 63) >> 6, kst_full = (Kfull + 63) >> 6;

    // weights: thread t takes group t % 4 of row t / 4 of a stage
    const int wr = tid >> 2, wg = tid & 3;
    const uint8_t *wrow = w + (size_t)(n0 + wr < N ? n0 + wr : N - 1) * ((size_t)(Kfull / Fmt<FMT>::BE) * Fmt<FMT>::BB) +
                          (size_t)(k0 / Fmt<FMT>::BE) * Fmt<FMT>::BB;
    Group<FMT> raw[2];
    auto load_w = [&](Group<FMT> &dst, int st) __attribute__((always_inline)) {
        int g = 4 * st + wg;
        g = g < groups ? g : groups - 1;
        if constexpr (INT) dst.load(wrow + (uint32_t)(g >> 3) * 144u + 16u + (uint32_t)((g >> 1) & 3) * 32u);
        else dst.load(wrow + (uint32_t)g * (uint32_t)Fmt<FMT>::BB);
    };
    // INT: the header of the super-block being decoded; unit: the unit of its predecessor, then its own
    uint32_t hdr[4] = {0, 0, 0, 0};
    float unit = 1.0f;
    v2h i_sc = {0, 0}, i_off = {0, 0};
    auto load_hdr = [&](int sb) __attribute__((always_inline)) {
        const int last = K / 256 - 1;
        const v4u_a4 v = *reinterpret_cast<const v4u_a4 *>(wrow + (uint32_t)(sb < last ? sb : last) * 144u);
#pragma unroll
        for (int e = 0; e < 4; e++) hdr[e] = v[e];
    };
    uint8_t *const sb_area = lds + 3 * BUF;
    // the scale (as an operand) and the min of this thread's group of half h of super-block sb; with half 0 what the
    // accumulators need to enter the super-block.  d = 0: no weights, the unit stays.
    auto open_hdr = [&](auto hc, int sb) __attribute__((always_inline)) {
        constexpr int H = decltype(hc)::value;
        uint32_t scb, mnb;
        if constexpr (H == 0) {
            scb = hdr[1] & 0x3F3F3F3Fu;
            mnb = hdr[2] & 0x3F3F3F3Fu;
        } else {
            scb = (hdr[3] & 0x0F0F0F0Fu) | ((hdr[1] >> 2) & 0x30303030u);
            mnb = ((hdr[3] >> 4) & 0x0F0F0F0Fu) | ((hdr[2] >> 2) & 0x30303030u);
        }
        const float d = f16_bits_to_f32((uint16_t)hdr[0]);
        const uint32_t s6 = d == 0.0f ? 0u : (scb >> (8 * wg)) & 255u, m6 = (mnb >> (8 * wg)) & 255u;
        const _Float16 sh = (_Float16)(unsigned short)s6, mh = (_Float16)(unsigned short)m6;
        i_sc = v2h{sh, sh};
        i_off = i_sc * v2h{(_Float16)-1024.0f, (_Float16)-1024.0f};
        uint8_t *const area = sb_area + (sb & 1) * SB_AREA;
        *reinterpret_cast<v2h *>(area + wr * 32 + (4 * H + wg) * 4) = v2h{mh, mh};
        if constexpr (H == 0) {
            const float now = d == 0.0f ? unit : d, f = wg == 0 ? unit / now : wg == 1 ? -f16_bits_to_f32((uint16_t)(hdr[0] >> 16)) / now : now;
            unit = now;
            if (wg < 3) *reinterpret_cast<float *>(area + BN * 32 + wg * (BN * 4) + wr * 4) = f;
        }
    };
    // activations: arranged units of 32 rows x 64 k, octet c of half h of row r at ((c * 2 + h) * 32 + r) * 16
    __amdgpu_buffer_rsrc_t a_tile[TI];
#pragma unroll
    for (int t = 0; t < TI; t++) {
        const int last = 2 * ((M + 31) / 32) - 1, mt = m0 / 16 + wm * TI + t, mc = mt < last ? mt : last;
        const int skip = (mc & 1) * 256;
        a_tile[t] = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<uint8_t *>(reinterpret_cast<const uint8_t *>(at)) + ((size_t)(mc >> 1) * kst_full + k0 / 64) * 4096 + skip, 0, kst * 4096 - skip, 0x00020000);
    }
    const uint32_t a_lane = (uint32_t)(q * 1024 + i * 16);
    v4u a[4][TI];
    uint32_t a_off[2];                                            // of the next stage's two units of 64 k (the second may lie past the row: zeros)
    auto a_stage = [&](int st) __attribute__((always_inline)) {
        a_off[0] = a_lane;
        a_off[1] = 2 * st + 1 < kst ? a_lane : 0x80000000u;
    };
    auto load_a = [&](int st, int g, int t) __attribute__((always_inline)) {
        a[g][t] = __builtin_amdgcn_raw_buffer_load_b128(a_tile[t], a_off[g >> 1], st * 8192 + (g >> 1) * 4096 + (g & 1) * 512, 0);
    };
    uint8_t *const w_to = lds + wg * PLANE + (wr >> 4) * 1024 + (wr & 15) * 16;
    uint8_t *const s_to = lds + 4 * PLANE + (wg * BN + wr) * 4;
    const uint8_t *const w_from = lds + wn * (TJ * 1024) + lane * 16;
    const uint8_t *const s_from = lds + 4 * PLANE + (wn * (TJ * 16) + i) * 4;
    auto put_octet = [&](auto oc, const Group<FMT> &src, int buf) __attribute__((always_inline)) {
        constexpr int O = decltype(oc)::value;
        if constexpr (INT) *reinterpret_cast<v4u *>(w_to + buf + O * 256) = src.template octet<O>((wg & 1) * 4, i_sc, i_off);
        else *reinterpret_cast<v4u *>(w_to + buf + O * 256) = src.template octet<O>();
    };
    auto put_scale = [&](const Group<FMT> &src, int st, int buf) __attribute__((always_inline)) {
        if constexpr (!INT) *reinterpret_cast<float *>(s_to + buf) = 4 * st + wg < groups ? src.scale() : 0.0f;
    };
    v4u wf[2][TJ];
    float sc[2][TJ];
    auto get_w = [&](int set, int g, int j, int buf) __attribute__((always_inline)) {
        wf[set][j] = *reinterpret_cast<const v4u *>(w_from + buf + g * PLANE + j * 1024);
        if constexpr (!INT) sc[set][j] = *reinterpret_cast<const float *>(s_from + buf + (g * BN + j * 16) * 4);
    };
    // INT: a super-block's group sums of the activations as fp16 (hi, lo) pairs (group 2 q and 2 q + 1 of row i), its mins, and
    // what its rows' accumulators are multiplied by next
    v2u sums[TI], mins[TJ];
    float ratio[TJ];
    __amdgpu_buffer_rsrc_t s_tile[TI];
    if constexpr (INT) {
#pragma unroll
        for (int t = 0; t < TI; t++) {
            const int last = 2 * ((M + 31) / 32) - 1, mt = m0 / 16 + wm * TI + t, mc = mt < last ? mt : last;
            s_tile[t] = __builtin_amdgcn_make_buffer_rsrc(
                const_cast<uint8_t *>(s2) + ((size_t)(mc >> 1) * (Kfull / 256) + k0 / 256) * 1024 + (mc & 1) * 256, 0, K / 256 * 1024 - (mc & 1) * 256, 0x00020000);
        }
    }
    const uint32_t s_lane = (uint32_t)((q >> 1) * 512 + i * 16 + (q & 1) * 8);
    auto load_sums = [&](int sb, int t) __attribute__((always_inline)) {
        sums[t] = __builtin_amdgcn_raw_buffer_load_b64(s_tile[t], s_lane, (sb < K / 256 ? sb : K / 256 - 1) * 1024, 0);
    };
    auto row_value = [&](int which, int sb, int j) __attribute__((always_inline)) -> float {
        return *reinterpret_cast<const float *>(sb_area + (sb & 1) * SB_AREA + BN * 32 + which * (BN * 4) + (wn * (TJ * 16) + j * 16 + i) * 4);
    };
    v4f acc[TI][TJ], p[4];
#pragma unroll
    for (int x = 0; x < TI; x++)
#pragma unroll
        for (int j = 0; j < TJ; j++) acc[x][j] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int x = 0; x < 4; x++) p[x] = v4f{0.f, 0.f, 0.f, 0.f};

    // the sums of slot x (of 4 T) join the accumulators
    auto settle = [&](auto xc) __attribute__((always_inline)) {
        constexpr int x = decltype(xc)::value, g = x / T, t = x % T / TJ, j = x % TJ;
#pragma unroll
        for (int r = 0; r < 4; r++) acc[t][j][r] = __builtin_fmaf(INT ? ratio[j] : sc[g & 1][j], p[x & 3][r], acc[t][j][r]);
    };
    auto rescale = [&](auto xc) __attribute__((always_inline)) {
        constexpr int x = decltype(xc)::value, t = x / TJ, j = x % TJ;
#pragma unroll
        for (int r = 0; r < 4; r++) acc[t][j][r] *= ratio[j];
    };
    int cur = 0, nxt = BUF, far = 2 * BUF;                        // LDS buffers of this stage, the next, the one after
    auto stage = [&](auto par, int st) __attribute__((always_inline)) {
        Group<FMT> &src = raw[decltype(par)::value];
        a_stage(st + 1 < nst ? st + 1 : nst - 1);
        const int st_a = st + 1 < nst ? st + 1 : nst - 1;
        each<4 * T>([&](auto xc) __attribute__((always_inline)) {
            constexpr int x = decltype(xc)::value, g = x / T, y = x % T, t = y / TJ, j = y % TJ;
            v8h ah, wh;
            __builtin_memcpy(&ah, &a[g][t], 16);
            __builtin_memcpy(&wh, &wf[g & 1][j], 16);
            if constexpr (INT) {
                acc[t][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah, wh, acc[t][j], 0, 0, 0);
                constexpr int PAR = decltype(par)::value;
                // into the next super-block's unit: a tile two slots before its first matrix instruction there
                if constexpr (PAR == 1 && x == 4 * T - LAG) {
                    each<TJ>([&](auto f) __attribute__((always_inline)) { ratio[decltype(f)::value] = row_value(0, (st >> 1) + 1, decltype(f)::value); });
                }
                if constexpr (PAR == 0 && x < T - 2) rescale(IC<x + 2>{});
                if constexpr (PAR == 1 && x == 4 * T - 1) { rescale(IC<0>{}); rescale(IC<1>{}); }
                // the min term, in the second group of the super-block's second half
                if constexpr (PAR == 1 && x == T - 1) {
                    each<TJ>([&](auto f) __attribute__((always_inline)) {
                        constexpr int F = decltype(f)::value;
                        mins[F] = *reinterpret_cast<const v2u *>(sb_area + ((st >> 1) & 1) * SB_AREA + (wn * (TJ * 16) + F * 16 + i) * 32 + q * 8);
                        ratio[F] = row_value(1, st >> 1, F);
                    });
                }
                if constexpr (PAR == 1 && g == 1) {
                    v4h sa, mb;
                    __builtin_memcpy(&sa, &sums[t], 8);
                    __builtin_memcpy(&mb, &mins[j], 8);
                    p[x & 3] = __builtin_amdgcn_mfma_f32_16x16x16f16(sa, mb, v4f{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
                }
                if constexpr (PAR == 1 && x >= T + LAG && x < 2 * T + LAG) settle(IC<x - LAG>{});
                if constexpr (PAR == 1 && x >= 2 * T + LAG && x < 2 * T + LAG + TI) load_sums((st >> 1) + 1, x - 2 * T - LAG);
            } else {
                p[x & 3] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah, wh, v4f{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
                settle(IC<(x + 4 * T - LAG) % (4 * T)>{});
            }
            if constexpr (j == TJ - 1) load_a(st_a, g, t);
            // the next group's fragments, once the last sums of the group before are settled
            each<TJ>([&](auto fc) __attribute__((always_inline)) {
                constexpr int f = decltype(fc)::value;
                if constexpr (y == LAG - 1 + f * (T - LAG + 1) / TJ) get_w((g + 1) & 1, (g + 1) & 3, f, g < 3 ? cur : nxt);
            });
            if constexpr (INT && x == 0) open_hdr(par, (st >> 1) + 1);
            if constexpr (INT && x == 1 && decltype(par)::value == 1) load_hdr((st >> 1) + 2);
            if constexpr (y == T / 2) put_octet(IC<g>{}, src, far);
            if constexpr (g == 0 && y == T / 2 + 1) put_scale(src, st + 2, far);
            if constexpr (g == 3 && y == T / 2 + 1) load_w(src, st + 4);
            __builtin_amdgcn_sched_barrier(0);
        });
        lds_barrier();
        const int was = cur;
        cur = nxt; nxt = far; far = was;
    };

    if constexpr (INT) load_hdr(0);
    load_w(raw[0], 0);
    a_stage(0);
#pragma unroll
    for (int g = 0; g < 4; g++)
#pragma unroll
        for (int t = 0; t < TI; t++) load_a(0, g, t);
    load_w(raw[1], 1);
    if constexpr (INT) {
#pragma unroll
        for (int t = 0; t < TI; t++) load_sums(0, t);
    }
    each<2>([&](auto sc_) __attribute__((always_inline)) {
        constexpr int s = decltype(sc_)::value, buf = s * BUF;
        if constexpr (INT) open_hdr(sc_, 0);
        put_octet(IC<0>{}, raw[s], buf);
        put_octet(IC<1>{}, raw[s], buf);
        put_octet(IC<2>{}, raw[s], buf);
        put_octet(IC<3>{}, raw[s], buf);
        put_scale(raw[s], s, buf);
        load_w(raw[s], s + 2);
    });
    if constexpr (INT) load_hdr(1);
    lds_barrier();
#pragma unroll
    for (int j = 0; j < TJ; j++) {
        get_w(0, 0, j, 0);
        wf[1][j] = v4u{0, 0, 0, 0};
        sc[1][j] = 0.0f;
        ratio[j] = 1.0f;                                          // (nothing accumulated yet)
    }
    int st = 0;
    for (; st + 1 < nst; st += 2) {
        stage(IC<0>{}, st);
        stage(IC<1>{}, st + 1);
    }
    if constexpr (!INT)
        if (st < nst) stage(IC<0>{}, st);
    if constexpr (INT) {
#pragma unroll
        for (int j = 0; j < TJ; j++) {
            const float u = row_value(2, K / 256 - 1, j);
#pragma unroll
            for (int t = 0; t < TI; t++)
#pragma unroll
                for (int r = 0; r < 4; r++) acc[t][j][r] *= u;
        }
    } else each<LAG>([&](auto xc) __attribute__((always_inline)) { settle(IC<4 * T - LAG + decltype(xc)::value>{}); });

    // register r of tile (t, j): row 4 q + r of A, row i of W
    const int mrow = m0 + wm * (16 * TI) + 4 * q, ncol = n0 + wn * (16 * TJ) + i;
    float *const of = reinterpret_cast<float *>(outp) + (size_t)part * M * N;
#pragma unroll
    for (int t = 0; t < TI; t++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int m = mrow + 16 * t + r;
            if (m >= M) continue;
#pragma unroll
            for (int j = 0; j < TJ; j++) {
                const int n = ncol + 16 * j;
                if (n >= N) continue;
                if (f16_out) reinterpret_cast<_Float16 *>(outp)[(size_t)m * N + n] = (_Float16)acc[t][j][r];
                else of[(size_t)m * N + n] = acc[t][j][r];
            }
        }
}

} // namespace codes
} // namespace rfq
