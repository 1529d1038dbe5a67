// Polar quantizer (quantize-on-append and prompt quantization): the HIP
// counterpart of quantize_and_pack_nbit (models/modeling_llama_polar.py:135-157).
//
// One 256-thread workgroup per (batch, KV head, 128-token group).  Thread
// (tl = tid/16, pq = tid%16) owns dimension pairs 4pq..4pq+3 of tokens
// tl, tl+16, ..., tl+112: each load is 8 bytes of x (dims [4pq,4pq+4)) and 8
// bytes of y (dims [64+4pq, ...)), so a wavefront reads four whole 256-byte key
// rows at a time, and each store is the 4 code bytes of one token, so a
// wavefront writes 256 contiguous bytes.  The key tile is read from HBM once:
// angles and radii stay in registers (packed as two 16-bit words) between the
// min/max pass and the code pass.
//
// Arithmetic follows eager torch on half tensors op by op: every reference op
// is evaluated in fp32 and rounded to the key dtype before the next.
//
// What bounds it: the vector unit, about 50 instructions a pair of which two at a quarter of the rate (96 of the 98 us that 131072
// tokens of 8 heads take with the device library's arctangent as the exact routine, 106 with SLEEF's, whose double-float sequence a
// wavefront runs once or twice; their bytes need 68).  It was 65 instructions and 119 us with the angle from the smaller over the
// larger operand (a comparison, two selections and a second turn more), each code converted and bounded by itself, and scales by IEEE
// divisions; keys requested two rows at a time and words read from LDS for each pass cost 8 us of it.
// Gathering a workgroup's entries for the exact routines so that one wavefront does them all: 128 instead of 131 us at best, short
// calls slower; not kept.
#include "pq_device.h"
#include "pq_internal.h"
#include "pq_math.h"

namespace pq {

typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef __bf16 bfloat2v __attribute__((ext_vector_type(2)));
typedef float float2v __attribute__((ext_vector_type(2)));
typedef unsigned short ushort2v __attribute__((ext_vector_type(2)));

template <typename T>
__device__ __forceinline__ float rnd(float f) { return lo2f<T>(f2lo<T>(f)); }

// ---- angle and radius of one pair, rounded to the key dtype -------------------
// Eager torch gives round_dtype(atan2f_sleef(y, x)) and round_dtype(sqrt_rn(x*x + y*y)).
// The exact routines cost ~100 instructions per pair, so a cheap estimate is tried
// first: an arctangent of the half angle (reciprocal, polynomial of degree 7 or 6 in
// its square; half stays within 5 ulp of the exact routine, bfloat16 within 12) and the hardware square
// root (1 ulp).  Rounding the estimate to the key dtype gives the same word as
// rounding the exact value unless the estimate lies within its error bound of a
// rounding boundary of the dtype (a midpoint between two neighbouring dtype
// values, i.e. low fp32 mantissa bits == 100..0).  Only those lanes, plus the
// special operands (zeros, infinities, NaNs, results below the dtype's normal
// range), take the exact path.  That the two paths agree on EVERY pair of half /
// bfloat16 operands is checked exhaustively on the device by pq_selftest_quantizer_math.
template <typename T> struct IsHalf { static constexpr bool value = false; };
template <> struct IsHalf<F16> { static constexpr bool value = true; };
template <typename T> struct DT;
template <> struct DT<F16> { static constexpr uint32_t kMid = 0x1000u; static constexpr int kHighBits = 19; static constexpr float kMinNormal = 6.103515625e-05f; };
template <> struct DT<BF16> { static constexpr uint32_t kMid = 0x8000u; static constexpr int kHighBits = 16; static constexpr float kMinNormal = 1.17549435e-38f; };

// An estimate further than its largest error from a midpoint rounds like the exact value.
constexpr uint32_t kSqrtGuardUlps = 1;   // v_sqrt_f32

// Which arctangent the angle must reproduce.  Eager torch evaluates atan2 on half tensors in fp32 and
// rounds once: on the CPU with SLEEF's Sleef_atan2f_u10 (restated in pq_math.h), on the GPU with the
// device math library's atan2f, which is what `atan2f` in device code here resolves to as well.  The
// two differ in the last fp32 bits on about a third of all operands, and after rounding to half on a
// few dozen per million.  LIBM = true selects the device library's routine as the exact one (the
// exhaustive self-test checks each guard band against its routine).  The bands are the estimate's largest
// distance from the routine over every pair of operands.
template <typename T, bool LIBM> struct Atan { static constexpr uint32_t kGuardUlps = (IsHalf<T>::value ? 5 : 12) + (LIBM ? 1 : 0); };
template <bool LIBM>
__device__ __forceinline__ float atan2_exact(float y, float x) {
    if constexpr (LIBM) return atan2f(y, x);
    else return math::atan2f_sleef_u10(y, x);
}

template <typename T>
__device__ __forceinline__ bool near_rounding_boundary(float a, uint32_t guard) {
    // |low mantissa bits - midpoint pattern| <= guard: the sum's low bits at the top of the word, one shifted addition and one comparison
    const uint32_t low = (__float_as_uint(a) + (guard - DT<T>::kMid)) << DT<T>::kHighBits;
    return low < (2u * guard + 1u) << DT<T>::kHighBits;
}

// the angle's magnitude, r being the pair's radius: twice the arctangent of |y| / (r + |x|), which is the half angle's tangent and never
// above 1, so that no larger of the two operands has to be found and only the side of x to be put right.  Polynomials in the tangent's
// square with the least largest relative error: 1.1e-7 for half, 7.3e-7 for bfloat16.  A coefficient more or less moves it by a factor
// of 6.6; a wider guard band sends more entries to the exact routines.
template <typename T>
__device__ __forceinline__ float atan2_fast_abs(float y, float x, float r) {
    const float t = fabsf(y) * __builtin_amdgcn_rcpf(fabsf(x) + r);
    const float s = t * t;
    float u;
    if constexpr (IsHalf<T>::value) {
        u = 2.0f * -0.00482253451f;
        u = __builtin_fmaf(u, s, 2.0f * 0.0247340649f);
        u = __builtin_fmaf(u, s, 2.0f * -0.0602031313f);
        u = __builtin_fmaf(u, s, 2.0f * 0.0996847302f);
        u = __builtin_fmaf(u, s, 2.0f * -0.140413284f);
        u = __builtin_fmaf(u, s, 2.0f * 0.199742138f);
        u = __builtin_fmaf(u, s, 2.0f * -0.333323926f);
    } else {
        u = 2.0f * 0.00810636859f;
        u = __builtin_fmaf(u, s, 2.0f * -0.0377967246f);
        u = __builtin_fmaf(u, s, 2.0f * 0.0848410428f);
        u = __builtin_fmaf(u, s, 2.0f * -0.135445759f);
        u = __builtin_fmaf(u, s, 2.0f * 0.198978737f);
        u = __builtin_fmaf(u, s, 2.0f * -0.333284914f);
    }
    const float a = t * __builtin_fmaf(u, s, 2.0f);
    return x < 0.0f ? 3.14159274101257324219f - a : a;
}

// Cheap estimates of the angle's magnitude (its sign is y's) and of the radius, NOT yet rounded; returns true when
// the exact routines must be used instead (see above), or when *ss_out says so (squares_out_of_range).
template <typename T, bool LIBM = false>
__device__ __forceinline__ bool angle_radius_fast(float x, float y, float* a_out, float* r_out, float* ss_out) {
    const float ss = __builtin_fmaf(x, x, y * y);          // x*x, y*y are exact for half/bf16 operands
    const float r = __builtin_amdgcn_sqrtf(ss);
    const float a = atan2_fast_abs<T>(y, x, r);
    // (bfloat16 only) magnitudes at which the reciprocal or the hardware square root leave their accurate range; half's
    // finite squares all lie inside (2^-80, 2^80).  Zeros need no test of their own: y == 0 gives exactly 0 or pi (0 then fails
    // the kMinNormal test below); x == 0 gives pi/2 to a few ulps (the polynomials at 1: two below it for half, nine above for bfloat16),
    // and pi/2 is 37 ulps from a midpoint of half and 28709 from one of bfloat16, so that it rounds like the exact angle;
    // x == y == 0 gives a NaN angle with radius 0, which fails the kMinNormal test as well.
    // (bitwise | on purpose: one straight-line predicate instead of a chain of exec-mask branches)
    int special = 0;
    if constexpr (!IsHalf<T>::value) special |= static_cast<int>(!(ss > 0x1p-80f));
    *a_out = a;
    *r_out = r;
    *ss_out = ss;
    return (special | static_cast<int>(fminf(a, r) < DT<T>::kMinNormal) |
            static_cast<int>(near_rounding_boundary<T>(a, Atan<T, LIBM>::kGuardUlps)) |
            static_cast<int>(near_rounding_boundary<T>(r, kSqrtGuardUlps))) != 0;
}
// Infinities, NaNs and large bfloat16 magnitudes, of one pair's squares or, as patterns order like the numbers and NaNs lie above
// them all, of the largest pattern of many.
__device__ __forceinline__ bool squares_out_of_range(uint32_t ss_bits) { return ss_bits >= 0x67800000u; }      // 2^80

// Correctly rounded fp32 square root.  NOT __fsqrt_rn: HIP defines that as the native (1 ulp)
// instruction unless OCML_BASIC_ROUNDED_OPERATIONS is set; sqrtf() is expanded by the compiler to
// the correctly rounded sequence (the default of -fhip-fp32-correctly-rounded-divide-sqrt), and the
// device self-test checks every result against its two neighbours' midpoints in double precision.
__device__ __forceinline__ float sqrt_rn(float s) { return __builtin_sqrtf(s); }

// -> (angle in [-pi, pi], radius), both rounded to the key dtype
template <typename T, bool LIBM = false>
__device__ __forceinline__ void angle_radius(float x, float y, float* phi, float* rad) {
    float a, r, ss;
    const bool risky = angle_radius_fast<T, LIBM>(x, y, &a, &r, &ss);
    a = __builtin_copysignf(a, y);
    if (__builtin_expect(risky || squares_out_of_range(__float_as_uint(ss)), 0)) {
        a = atan2_exact<LIBM>(y, x);
        r = sqrt_rn(__builtin_fmaf(x, x, y * y));
    }
    *phi = rnd<T>(a);
    *rad = rnd<T>(r);
}

template <typename T, bool LIBM = false>
__device__ __forceinline__ void angle_radius_exact(float x, float y, float* phi, float* rad) {
    *phi = rnd<T>(atan2_exact<LIBM>(y, x));
    *rad = rnd<T>(sqrt_rn(__builtin_fmaf(x, x, y * y)));
}

// floor(dtype((v - mn) / scale)) clamped to [0, top] (:148, :153).  `topf` is the clamp bound as a
// float, or 0 for a degenerate pair (scale == 0 or NaN: x/0 and 0/0 are undefined in the reference
// and defined as code 0 here).  v_med3_f32 returns the minimum of its operands when one is NaN, so
// a NaN quotient also comes out as 0 without a separate test.
template <typename T>
__device__ __forceinline__ uint32_t code_of(float v, float mn, float scale, float topf) {
    const float d = rnd<T>(v - mn);
    const float qf = floorf(rnd<T>(d / scale));
    return static_cast<uint32_t>(__builtin_amdgcn_fmed3f(qf, 0.0f, topf));
}
// The same of the rounded distance d >= 0 for scales that fast_div_ok accepts and top <= 127, without a division.
//
// Rounding to the dtype carries a quotient to the integer k or over it exactly if half a unit in the last place of its own binade
// does (an integer up to 128 is even in both dtypes: a tie goes to it).  So only the side of B = k - half a unit on which d / scale
// lies has to be right.  d is a number of 11 bits (bfloat16: 8) and B * scale one of 23 (17), so a quotient below B is below it by
// 2^-23 (2^-17) of it at least.  Half: the inverse in two parts; the product's one rounding then neither reaches B from there nor
// leaves it.  Bfloat16: an inverse too large by 2^-22 to 2^-20 is enough.  Every pair of operands is checked on the device.
template <typename T>
__device__ __forceinline__ Inverse inverse_of(float scale) {
    if constexpr (IsHalf<T>::value) return two_part_inverse(scale);
    const float inv = __builtin_amdgcn_rcpf(scale);                  // within 1 ulp
    return {__builtin_fmaf(inv, 0x1p-21f, inv), 0.0f};
}
// The codes of four pairs: angles in bits tbits - 1 .. 0 of each byte, radii above them.  `add` takes a pair's distances.
// Half: both quotients are rounded by one conversion, the dtype's own (a multiply-add, half a unit and a conversion to a whole number
// for each: 3 instructions a pair more).  A NaN converts to 0.
struct CodeTops { uint32_t both; int tbits; };
template <typename T> struct CodeWord {
    uint32_t c[4];                                                                          // angle code | radius code << 16
    template <int I> __device__ __forceinline__ void add(float da, Inverse ia, float dr, Inverse ir, const CodeTops& top) {
        const ushort2v k = __builtin_convertvector(__builtin_convertvector((float2v{quotient(da, ia), quotient(dr, ir)}), half2v), ushort2v);
        c[I] = __builtin_bit_cast(uint32_t, __builtin_elementwise_min(k, __builtin_bit_cast(ushort2v, top.both)));
    }
    __device__ __forceinline__ uint32_t word(const CodeTops& top) const {
        const uint32_t c01 = __builtin_amdgcn_perm(c[1], c[0], 0x06020400u), c23 = __builtin_amdgcn_perm(c[3], c[2], 0x06020400u);
        return (__builtin_amdgcn_perm(c23, c01, 0x07060302u) << top.tbits) | __builtin_amdgcn_perm(c23, c01, 0x05040100u);
    }
    static __device__ __forceinline__ CodeTops tops(int tbits, int rbits) { return {((1u << tbits) - 1u) | (((1u << rbits) - 1u) << 16), tbits}; }
};
// Bfloat16: adding kMid to the fp32 pattern adds the half unit; the sum is then scaled to 2^8 and converted to a byte, which saturates,
// so that the code is its upper bits and needs no bound.  The conversion rounds to nearest: half is taken off first, without error (below
// 2^8 the difference has the sum's unit), and a tie at a multiple of the code's step goes to it, being even.  A NaN converts to 0.
struct CodeScales { float t, r; int tshift, rshift; uint32_t tmask, rmask; };
template <> struct CodeWord<BF16> {
    uint32_t t, r;                                                                          // bytes: code and fraction
    template <int I> __device__ __forceinline__ void add(float da, Inverse ia, float dr, Inverse ir, const CodeScales& top) {
        auto up = [](float q, float scale) { return __builtin_fmaf(__uint_as_float(__float_as_uint(q) + DT<BF16>::kMid), scale, -0.5f); };
        t = __builtin_amdgcn_cvt_pk_u8_f32(up(da * ia.hi, top.t), I, I == 0 ? 0u : t);
        r = __builtin_amdgcn_cvt_pk_u8_f32(up(dr * ir.hi, top.r), I, I == 0 ? 0u : r);
    }
    __device__ __forceinline__ uint32_t word(const CodeScales& top) const { return ((t >> top.tshift) & top.tmask) | ((r >> top.rshift) & top.rmask); }
    static __device__ __forceinline__ CodeScales tops(int tbits, int rbits) {
        return {static_cast<float>(256 >> tbits), static_cast<float>(256 >> rbits), 8 - tbits, 8 - rbits - tbits,
                0x01010101u * ((1u << tbits) - 1u), 0x01010101u * (((1u << rbits) - 1u) << tbits)};
    }
};
// One code by itself, at most `top`: half a unit added to the fp32 pattern and a conversion to a whole number (a word's four would cost
// two quotients a code where fixed angle bins have one: 65536 tokens of 8 heads, float16 66.8 for 57.9 us).
template <typename T>
__device__ __forceinline__ uint32_t code_of_fast(float d, Inverse inv, uint32_t top) {
    const float q = IsHalf<T>::value ? quotient(d, inv) : d * inv.hi;
    const uint32_t k = static_cast<uint32_t>(__uint_as_float(__float_as_uint(q) + DT<T>::kMid));
    return k < top ? k : top;
}
// the word's code of the same
template <typename T>
__device__ __forceinline__ uint32_t code_of_word(float d, Inverse inv, int bits) {
    const auto top = CodeWord<T>::tops(bits, 0);
    CodeWord<T> w{};
    w.template add<0>(d, inv, 0.0f, inv, top);
    return w.word(top) & 0xffu;
}
// (angle - its minimum | radius - its minimum << 16), each rounded to the dtype.  Half: one packed subtraction (a sum or difference of
// two halves that is rounded to fp32 first is the same half).
template <typename T> __device__ __forceinline__ void pair_distance(uint32_t v, uint32_t mn, float* da, float* dr);
template <> __device__ __forceinline__ void pair_distance<F16>(uint32_t v, uint32_t mn, float* da, float* dr) {
    const half2v d = __builtin_bit_cast(half2v, v) - __builtin_bit_cast(half2v, mn);
    *da = static_cast<float>(d.x);
    *dr = static_cast<float>(d.y);
}
template <> __device__ __forceinline__ void pair_distance<BF16>(uint32_t v, uint32_t mn, float* da, float* dr) {
    const float2v d = {__uint_as_float(v << 16) - __uint_as_float(mn << 16), __uint_as_float(v & 0xffff0000u) - __uint_as_float(mn & 0xffff0000u)};
    const uint32_t w = __builtin_bit_cast(uint32_t, __builtin_convertvector(d, bfloat2v));
    *da = __uint_as_float(w << 16);
    *dr = __uint_as_float(w & 0xffff0000u);
}
__device__ __forceinline__ float clamp_bound(float scale, int top) { return scale > 0.0f ? static_cast<float>(top) : 0.0f; }

constexpr int kQThreads = 256;
constexpr int kTokPerThread = kGroup / 16;   // 8
constexpr int kEntries = kTokPerThread * 4;  // (token, pair) entries per thread

// Packed min / max of two (angle word | radius word << 16) registers.  Both values are
// non-negative (the angle after the 2*pi wrap, the radius always) and their sign bits are
// cleared, so bfloat16 words order like unsigned integers; half words use v_pk_max/min_f16.
template <typename T> __device__ __forceinline__ uint32_t pk_max(uint32_t a, uint32_t b);
template <typename T> __device__ __forceinline__ uint32_t pk_min(uint32_t a, uint32_t b);
template <> __device__ __forceinline__ uint32_t pk_max<F16>(uint32_t a, uint32_t b) {
    uint32_t r;                                 // (the builtin first passes what comes from memory through a maximum of its own)
    asm("v_pk_max_f16 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
template <> __device__ __forceinline__ uint32_t pk_min<F16>(uint32_t a, uint32_t b) {
    uint32_t r;
    asm("v_pk_min_f16 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
template <> __device__ __forceinline__ uint32_t pk_max<BF16>(uint32_t a, uint32_t b) {
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(ushort2v, a), __builtin_bit_cast(ushort2v, b)));
}
template <> __device__ __forceinline__ uint32_t pk_min<BF16>(uint32_t a, uint32_t b) {
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_min(__builtin_bit_cast(ushort2v, a), __builtin_bit_cast(ushort2v, b)));
}
template <typename T> struct PkInit;   // identity elements of pk_max / pk_min
template <> struct PkInit<F16> { static constexpr uint32_t kMax = 0x00000000u, kMin = 0x7c007c00u; };   // 0 / +inf
template <> struct PkInit<BF16> { static constexpr uint32_t kMax = 0x00000000u, kMin = 0xffffffffu; };

// How the angle is binned.  Reference mode: 2^tbits bins over the group's own [min, max] of the
// angle wrapped to [0, 2*pi) (:144-148).  Uniform mode: fixed bins over [-pi, pi), i.e. the same
// formula with the constants tmn = -pi and tscale = 2*pi / 2^tbits (both rounded to the key dtype);
// the angle code is then known in the first pass and is what the angle word carries.
struct AngleMode {
    float two_pi;      // reference mode: the constant added to negative angles
    float tmn, tscale; // uniform mode
    uint32_t ttop;
    float minus_one;
};

// (angle word | radius word << 16) of one pair: wrap applied, sign bits cleared.  ESTIMATE: of angle_radius_fast's values where it
// does not ask for the exact routines; no zero is among them, so neither is a sign that the wrap leaves.
// (its magnitude; the angle is negative where y's sign bit is set)
template <typename T, bool UNIFORM, bool ESTIMATE>
__device__ __forceinline__ uint32_t pack_angle_radius(float a, float r, float y, const AngleMode& am) {
    uint32_t w;
    const bool below = static_cast<int>(__float_as_uint(y)) < 0;
    if constexpr (UNIFORM) {
        const uint32_t aw = code_of_fast<T>(rnd<T>(rnd<T>(__builtin_copysignf(a, y)) - am.tmn), inverse_of<T>(am.tscale), am.ttop);
        w = aw | (static_cast<uint32_t>(f2lo<T>(r)) << 16);
    } else if constexpr (IsHalf<T>::value) {
        // (times minus one: a subtraction with its operand's conversion built in; angle and radius are rounded by one conversion)
        const _Float16 phi = static_cast<_Float16>(a);
        const float turned = __builtin_fmaf(static_cast<float>(phi), am.minus_one, am.two_pi);       // :144
        w = __builtin_bit_cast(uint32_t, __builtin_convertvector((float2v{below && (ESTIMATE || phi > static_cast<_Float16>(0.0f)) ? turned : a, r}), half2v));
    } else {
        const float phi = rnd<T>(a);
        w = __builtin_bit_cast(uint32_t, __builtin_convertvector((float2v{below && (ESTIMATE || phi > 0.0f) ? am.two_pi - phi : phi, r}), bfloat2v));       // :144
    }
    return ESTIMATE ? w : w & 0x7fff7fffu;
}

template <typename T, bool UNIFORM, bool PK6, bool LIBM>
__global__ __launch_bounds__(kQThreads) void quantize_kernel(
    const uint16_t* __restrict__ k, int64_t sb, int64_t sh, int64_t st, int Nk, int rbits, int tbits, AngleMode am,
    uint8_t* __restrict__ codes, uint16_t* __restrict__ rscale, uint16_t* __restrict__ rmn,
    uint16_t* __restrict__ tscale, uint16_t* __restrict__ tmn, int cap, int off) {
    // angle/radius words of the tile, entry-major so that a wavefront's accesses are contiguous
    __shared__ uint32_t pr[kEntries][kQThreads];
    __shared__ uint32_t red[2][4][kPairs];      // max / min, wavefront, pair
    __shared__ uint32_t fin[2][kPairs];

    const int tid = threadIdx.x;
    const int pq4 = tid & 15, tl = tid >> 4;
    const int grp = blockIdx.x, bh = blockIdx.y;
    const int b = bh / Nk, h = bh - b * Nk;
    const uint16_t* kb = k + b * sb + h * sh + static_cast<int64_t>(grp) * kGroup * st;

    // ---- pass 1: cheap estimates for every entry; remember which entries need the exact routines
    // (all of a thread's keys are requested at once: two rows at a time, as the compiler has it, do not cover the way to memory)
    uint32_t risky_mask = 0, ss_most = 0;
    uint2 xr[kTokPerThread], yr[kTokPerThread];
#pragma unroll
    for (int it = 0; it < kTokPerThread; it++) {
        const uint16_t* row = kb + (it * 16 + tl) * st;
        xr[it] = *reinterpret_cast<const uint2*>(row + 4 * pq4);
        yr[it] = *reinterpret_cast<const uint2*>(row + kPairs + 4 * pq4);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int it = 0; it < kTokPerThread; it++) {
        const uint2 xw = xr[it], yw = yr[it];
        const uint16_t xs[4] = {static_cast<uint16_t>(xw.x), static_cast<uint16_t>(xw.x >> 16),
                                static_cast<uint16_t>(xw.y), static_cast<uint16_t>(xw.y >> 16)};
        const uint16_t ys[4] = {static_cast<uint16_t>(yw.x), static_cast<uint16_t>(yw.x >> 16),
                                static_cast<uint16_t>(yw.y), static_cast<uint16_t>(yw.y >> 16)};
#pragma unroll
        for (int i = 0; i < 4; i++) {
            float a, r, ss;
            const float y = lo2f<T>(ys[i]);
            const bool risky = angle_radius_fast<T, LIBM>(lo2f<T>(xs[i]), y, &a, &r, &ss);   // :143, :150
            risky_mask = risky_mask + risky_mask + (risky ? 1u : 0u);                         // (entry e in bit 31 - e)
            ss_most = ss_most > __float_as_uint(ss) ? ss_most : __float_as_uint(ss);
            pr[it * 4 + i][tid] = pack_angle_radius<T, UNIFORM, true>(a, r, y, am);
        }
    }
    if (squares_out_of_range(ss_most)) risky_mask = 0xffffffffu;
    // ---- fix-up: each lane redoes ITS risky entries with the exact routines (a lane has ~0.1 of
    // them, so the wavefront makes one or two trips instead of branching at all 32 entries)
    while (risky_mask) {
        const int e = __builtin_clz(risky_mask);
        risky_mask &= ~(0x80000000u >> e);
        const uint16_t* row = kb + ((e >> 2) * 16 + tl) * st;
        const float x = lo2f<T>(row[4 * pq4 + (e & 3)]), y = lo2f<T>(row[kPairs + 4 * pq4 + (e & 3)]);
        float a, r;
        angle_radius_exact<T, LIBM>(x, y, &a, &r);
        pr[e][tid] = pack_angle_radius<T, UNIFORM, false>(fabsf(a), r, a, am);
    }
    // ---- per-pair max / min of angle and radius over the 128 tokens (packed: both at once)
    // (each word is read back once and stays in a register for the codes)
    uint32_t vmax[4], vmin[4], word[kEntries];
#pragma unroll
    for (int i = 0; i < 4; i++) { vmax[i] = PkInit<T>::kMax; vmin[i] = PkInit<T>::kMin; }
#pragma unroll
    for (int e = 0; e < kEntries; e++) word[e] = pr[e][tid];
#pragma unroll
    for (int e = 0; e < kEntries; e++) {
        vmax[e & 3] = pk_max<T>(vmax[e & 3], word[e]);
        vmin[e & 3] = pk_min<T>(vmin[e & 3], word[e]);
    }
    // the 16 token lanes of a pair: 4 inside the wavefront (lane bits 4,5), 4 wavefronts
#pragma unroll
    for (int i = 0; i < 4; i++) {
#pragma unroll
        for (int o = 16; o <= 32; o <<= 1) {
            vmax[i] = pk_max<T>(vmax[i], static_cast<uint32_t>(__shfl_xor(static_cast<int>(vmax[i]), o)));
            vmin[i] = pk_min<T>(vmin[i], static_cast<uint32_t>(__shfl_xor(static_cast<int>(vmin[i]), o)));
        }
    }
    if ((tid & 48) == 0) {
#pragma unroll
        for (int i = 0; i < 4; i++) { red[0][tid >> 6][4 * pq4 + i] = vmax[i]; red[1][tid >> 6][4 * pq4 + i] = vmin[i]; }
    }
    __syncthreads();
    if (tid < 2 * kPairs) {
        const int s = tid >> 6, p = tid & 63;
        uint32_t v = red[s][0][p];
#pragma unroll
        for (int j = 1; j < 4; j++) v = s ? pk_min<T>(v, red[s][j][p]) : pk_max<T>(v, red[s][j][p]);
        fin[s][p] = v;
    }
    __syncthreads();

    // (a product with the inverse of a power of two is the quotient's one rounding)
    const float inv_t = 1.0f / static_cast<float>(1 << tbits), inv_r = 1.0f / static_cast<float>(1 << rbits);
    float ts[4], tm[4], rs[4], rm[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const uint32_t wmax = fin[0][4 * pq4 + i], wmin = fin[1][4 * pq4 + i];
        tm[i] = lo2f<T>(static_cast<uint16_t>(wmin & 0xffffu));
        rm[i] = lo2f<T>(static_cast<uint16_t>(wmin >> 16));
        ts[i] = rnd<T>(rnd<T>(lo2f<T>(static_cast<uint16_t>(wmax & 0xffffu)) - tm[i]) * inv_t);   // :147
        if constexpr (UNIFORM) { tm[i] = am.tmn; ts[i] = am.tscale; }
        rs[i] = rnd<T>(rnd<T>(lo2f<T>(static_cast<uint16_t>(wmax >> 16)) - rm[i]) * inv_r);       // :152
    }
    const size_t plane = static_cast<size_t>(bh) * cap + off + grp;
    if (tl == 0) {
        auto pack4 = [](const float (&v)[4]) {
            return make_uint2(static_cast<uint32_t>(f2lo<T>(v[0])) | (static_cast<uint32_t>(f2lo<T>(v[1])) << 16),
                              static_cast<uint32_t>(f2lo<T>(v[2])) | (static_cast<uint32_t>(f2lo<T>(v[3])) << 16));
        };
        const size_t mi = plane * kPairs + 4 * pq4;
        *reinterpret_cast<uint2*>(tscale + mi) = pack4(ts);
        *reinterpret_cast<uint2*>(tmn + mi) = pack4(tm);
        *reinterpret_cast<uint2*>(rscale + mi) = pack4(rs);
        *reinterpret_cast<uint2*>(rmn + mi) = pack4(rm);
    }
    // ---- pass 2: codes
    float ttop[4], rtop[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        ttop[i] = clamp_bound(ts[i], (1 << tbits) - 1);
        rtop[i] = clamp_bound(rs[i], (1 << rbits) - 1);
    }
    uint8_t* cb = codes + plane * (kGroup * (PK6 ? kPackedRowBytes : kPairs));
    // scales of 0 (degenerate pairs), infinities and the far ends of the bfloat16 range take the division
    bool fast = true;
    Inverse tinv[4], rinv[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        fast = fast && fast_div_ok(ts[i]) && fast_div_ok(rs[i]);
        tinv[i] = inverse_of<T>(ts[i]);
        rinv[i] = inverse_of<T>(rs[i]);
    }
    auto store_codes = [&](int it, uint32_t w) {
        if constexpr (PK6) {
            // 4 codes -> 24 bits; the 4 lanes that share 12 bytes of the row assemble its 3 words:
            // lane 4k+0 writes x0 | x1 << 24, lane 4k+1 x1 >> 8 | x2 << 16, lane 4k+2 x2 >> 16 | x3 << 8
            const uint32_t x = (w & 0x3Fu) | ((w >> 2) & 0xFC0u) | ((w >> 4) & 0x3F000u) | ((w >> 6) & 0xFC0000u);
            const uint32_t nx = static_cast<uint32_t>(__shfl_down(static_cast<int>(x), 1));
            const int k = pq4 & 3;
            const uint32_t word = (x >> (8 * k)) | (nx << (24 - 8 * k));
            if (k < 3)
                *reinterpret_cast<uint32_t*>(cb + (it * 16 + tl) * kPackedRowBytes + 12 * (pq4 >> 2) + 4 * k) = word;
        } else {
            *reinterpret_cast<uint32_t*>(cb + (it * 16 + tl) * kPairs + 4 * pq4) = w;
        }
    };
    // PK6 exchanges words between lanes, so the whole wavefront takes one side together
    if (__builtin_expect(PK6 ? __all(fast) : fast, 1)) {
        uint32_t least[4];
#pragma unroll
        for (int i = 0; i < 4; i++) least[i] = fin[1][4 * pq4 + i];
        const auto top = CodeWord<T>::tops(tbits, rbits);
        const uint32_t rlast = (1u << rbits) - 1u;
#pragma unroll
        for (int it = 0; it < kTokPerThread; it++) {
            uint32_t w = 0;
            if constexpr (UNIFORM) {                                        // (the angles are codes already)
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const uint32_t v = word[it * 4 + i];
                    float da, dr;
                    pair_distance<T>(v, least[i], &da, &dr);
                    w |= ((code_of_fast<T>(dr, rinv[i], rlast) << tbits) + (v & 0xffffu)) << (8 * i);
                }
            } else {
                CodeWord<T> cw;
                static_for<4>([&](auto II) {
                    constexpr int i = decltype(II)::value;
                    float da, dr;
                    pair_distance<T>(word[it * 4 + i], least[i], &da, &dr);
                    cw.template add<i>(da, tinv[i], dr, rinv[i], top);      // :148, :153
                });
                w = cw.word(top);                                           // :155 (each below 256)
            }
            store_codes(it, w);
        }
    } else {
#pragma unroll
        for (int it = 0; it < kTokPerThread; it++) {
            uint32_t w = 0;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const uint32_t v = word[it * 4 + i];
                const float phi = lo2f<T>(static_cast<uint16_t>(v & 0xffffu));
                const float r = lo2f<T>(static_cast<uint16_t>(v >> 16));
                const uint32_t th = UNIFORM ? (v & 0xffffu) : code_of<T>(phi, tm[i], ts[i], ttop[i]);    // :148
                const uint32_t rh = code_of<T>(r, rm[i], rs[i], rtop[i]);      // :153
                w |= (((rh << tbits) + th) & 0xffu) << (8 * i);             // :155
            }
            store_codes(it, w);
        }
    }
}

#ifdef PQ_PROBE_DIRECT_BINS
#include "pq_quantize_probe.h"
#endif

// Exhaustive check of angle_radius against angle_radius_exact: block == bit pattern of y,
// thread t covers x patterns t, t+256, ...; NaN operands are skipped.
template <typename T, bool LIBM>
__global__ __launch_bounds__(256) void selftest_kernel(unsigned long long* mismatches, unsigned long long* slow_lanes) {
    const uint16_t yb = static_cast<uint16_t>(blockIdx.x);
    const float y = lo2f<T>(yb);
    unsigned int bad = 0, slow = 0;
    for (uint32_t xb = threadIdx.x; xb < 65536u; xb += 256u) {
        const float x = lo2f<T>(static_cast<uint16_t>(xb));
        if (x != x || y != y) continue;
        float p0, r0, p1, r1;
        angle_radius<T, LIBM>(x, y, &p0, &r0);
        angle_radius_exact<T, LIBM>(x, y, &p1, &r1);
        bad += (f2lo<T>(p0) != f2lo<T>(p1)) || (f2lo<T>(r0) != f2lo<T>(r1));
        // the exact radius: s lies between the squares of the midpoints to the two neighbours of sqrt_rn(s)
        const float s = __builtin_fmaf(x, x, y * y);
        if (!LIBM && s > 0.0f && s < INFINITY) {
            const float rr = sqrt_rn(s);
            const double lo = 0.5 * (static_cast<double>(rr) + static_cast<double>(__uint_as_float(__float_as_uint(rr) - 1u)));
            const double hi = 0.5 * (static_cast<double>(rr) + static_cast<double>(__uint_as_float(__float_as_uint(rr) + 1u)));
            bad += !(lo * lo <= static_cast<double>(s) && static_cast<double>(s) <= hi * hi);
        }
        const float r = __builtin_amdgcn_sqrtf(__builtin_fmaf(x, x, y * y)), a = atan2_fast_abs<T>(y, x, r);
        slow += near_rounding_boundary<T>(a, Atan<T, LIBM>::kGuardUlps) || near_rounding_boundary<T>(r, kSqrtGuardUlps);
    }
    if (bad) atomicAdd(mismatches, static_cast<unsigned long long>(bad));
    if (slow) atomicAdd(slow_lanes, static_cast<unsigned long long>(slow));
}

// Exhaustive check of the two-part quotient and of the codes taken from it: block == bit pattern of the dividend d, thread t covers the
// divisor patterns t, t+256, ...  Pairs the quantizers can meet: divisor accepted by fast_div_ok,
// 0 <= d <= 1024 * sc (d is a distance from the group minimum and sc the group's range over at
// most 2^8 bins).  Quotients below 1/4 may differ in denormal digits; floor() and rint() of both
// are 0 there, which is all the quantizers take from them.
template <typename T>
__global__ __launch_bounds__(256) void selftest_div_kernel(unsigned long long* mismatches) {
    const float d = lo2f<T>(static_cast<uint16_t>(blockIdx.x));
    unsigned int bad = 0;
    if (d >= 0.0f && d < INFINITY) {
        for (uint32_t sb = threadIdx.x; sb < 65536u; sb += 256u) {
            const float sc = lo2f<T>(static_cast<uint16_t>(sb));
            if (!fast_div_ok(sc) || !(d <= 1024.0f * sc)) continue;
            const float exact = rnd<T>(d / sc);
            const float fast = rnd<T>(quotient(d, two_part_inverse(sc)));
            bad += (exact != fast) && !(exact < 0.25f && fast < 0.25f);
            for (int bits : {7, 4, 3}) {
                const uint32_t top = (1u << bits) - 1u, code = static_cast<uint32_t>(__builtin_amdgcn_fmed3f(floorf(exact), 0.0f, static_cast<float>(top)));
                bad += code_of_word<T>(d, inverse_of<T>(sc), bits) != code || code_of_fast<T>(d, inverse_of<T>(sc), top) != code;
            }
        }
    }
    if (bad) atomicAdd(mismatches, static_cast<unsigned long long>(bad));
}

int launch_selftest(int dtype, unsigned long long* counters, hipStream_t st) {
    // counters: [0] mismatches, [1] exact-path pairs (SLEEF arctangent); [2] division mismatches;
    // [3] mismatches, [4] exact-path pairs with the device library's arctangent as the exact routine
    if (dtype == 0) {
        hipLaunchKernelGGL((selftest_kernel<F16, false>), dim3(65536), dim3(256), 0, st, counters, counters + 1);
        hipLaunchKernelGGL(selftest_div_kernel<F16>, dim3(65536), dim3(256), 0, st, counters + 2);
        hipLaunchKernelGGL((selftest_kernel<F16, true>), dim3(65536), dim3(256), 0, st, counters + 3, counters + 4);
    } else {
        hipLaunchKernelGGL((selftest_kernel<BF16, false>), dim3(65536), dim3(256), 0, st, counters, counters + 1);
        hipLaunchKernelGGL(selftest_div_kernel<BF16>, dim3(65536), dim3(256), 0, st, counters + 2);
        hipLaunchKernelGGL((selftest_kernel<BF16, true>), dim3(65536), dim3(256), 0, st, counters + 3, counters + 4);
    }
    return static_cast<int>(hipGetLastError());
}

int launch_quantize(const void* k, const int64_t* strides, int dtype, int B, int Nk, int Nb, int rbits, int tbits,
                    unsigned flags, uint8_t* codes, void* rscale, void* rmn, void* tscale, void* tmn,
                    int cap, int off, hipStream_t st) {
    dim3 grid(Nb, B * Nk), block(kQThreads);
    const float two_pi_f = 6.28318548202514648438f;   // (float)(2*pi)
    // eager torch-CPU casts the python scalar 2*pi to the tensor dtype first: 6.28125 in both dtypes
    AngleMode am;
    const bool uniform = (flags & 2u) != 0;
    am.two_pi = (flags & 1u) ? two_pi_f : 6.28125f;
    am.ttop = (1u << tbits) - 1u;
    am.minus_one = -1.0f;
    const bool bf = dtype != 0;
    auto round_dt = [bf](float f) {
        return bf ? math::bf16_bits_to_float(math::float_to_bf16_bits(f)) : math::half_bits_to_float(math::float_to_half_bits(f));
    };
    am.tmn = round_dt(-3.14159274101257324219f);
    am.tscale = round_dt(round_dt(two_pi_f) / static_cast<float>(1 << tbits));
    const bool packed6 = (flags & 4u) != 0;
    const bool libm = (flags & 8u) != 0;
#define PQ_LAUNCH_QPL(T, U, P, L)                                                                                    \
    hipLaunchKernelGGL((quantize_kernel<T, U, P, L>), grid, block, 0, st, (const uint16_t*)k, strides[0], strides[1], \
                       strides[2], Nk, rbits, tbits, am, codes, (uint16_t*)rscale, (uint16_t*)rmn,                  \
                       (uint16_t*)tscale, (uint16_t*)tmn, cap, off)
#define PQ_LAUNCH_QP(T, U, P)                                                                                        \
    do {                                                                                                             \
        if (libm) PQ_LAUNCH_QPL(T, U, P, true);                                                                      \
        else PQ_LAUNCH_QPL(T, U, P, false);                                                                          \
    } while (0)
#define PQ_LAUNCH_Q(T, U)                                                                                            \
    do {                                                                                                             \
        if (packed6) PQ_LAUNCH_QP(T, U, true);                                                                       \
        else PQ_LAUNCH_QP(T, U, false);                                                                              \
    } while (0)
#ifdef PQ_PROBE_DIRECT_BINS
    // the probe build: every launch in the reference's angle mode with byte-per-code rows runs the probe kernel
    if (!uniform && !packed6) {
        if (dtype == 0)
            hipLaunchKernelGGL(quantize_direct_bins_probe_kernel<F16>, grid, block, 0, st, (const uint16_t*)k, strides[0], strides[1],
                               strides[2], Nk, rbits, tbits, am.two_pi, codes, (uint16_t*)rscale, (uint16_t*)rmn, (uint16_t*)tscale, (uint16_t*)tmn, cap, off);
        else
            hipLaunchKernelGGL(quantize_direct_bins_probe_kernel<BF16>, grid, block, 0, st, (const uint16_t*)k, strides[0], strides[1],
                               strides[2], Nk, rbits, tbits, am.two_pi, codes, (uint16_t*)rscale, (uint16_t*)rmn, (uint16_t*)tscale, (uint16_t*)tmn, cap, off);
        return static_cast<int>(hipGetLastError());
    }
#endif
    if (dtype == 0) { if (uniform) PQ_LAUNCH_Q(F16, true); else PQ_LAUNCH_Q(F16, false); }
    else            { if (uniform) PQ_LAUNCH_Q(BF16, true); else PQ_LAUNCH_Q(BF16, false); }
#undef PQ_LAUNCH_Q
#undef PQ_LAUNCH_QP
#undef PQ_LAUNCH_QPL
    return static_cast<int>(hipGetLastError());
}

}  // namespace pq
