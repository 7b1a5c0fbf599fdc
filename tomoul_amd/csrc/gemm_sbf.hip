// gemm_sbf.hip -- GEMM on the bf16 matrix cores, fp32 values split into bf16
// terms: f32, F16 and Q8_K weights (both operands exactly), and the largest int8 /
// int4 ones (A in two terms, as in gemm_qbf.hip).
//
//   C[M,N] = act(alpha * A[M,K] . B[K,N] + beta * C + bias[N] + R)
//
// The reference's products are fp32 (src/core/ops.zig:277-414; f16 and Q8_K
// weights widened to f32, src/core/quantization.zig:559-614, :1921-1962).  An
// fp32 value's 24 bits are three bf16 terms, x = h + m + l, each the nearest
// bf16 of what the ones before leave (|m| <= 2^-8 |x|, |l| <= 2^-17 |x|, the
// sum exact), so
//   a . b = hh + hm + mh + mm + hl + lh  (+ ml + lm + ll, at most 2^-24 |a b|)
// with every kept product exact.  Six v_mfma_f32_16x16x32_bf16 (five for f16
// weights, whose 11 bits are two bf16 terms, h + m, exactly) do the work of eight
// v_mfma_f32_16x16x4_f32 at 16 times their rate: 2.5 PFLOP/s / 6 = 417 against 157
// TFLOP/s.  The dropped terms (for f16 weights lm alone, 2^-25) are at most one fp32
// rounding of the product, and the hh products have an accumulator of their own, which a 32-deep slice rounds
// once where the fp32 matrix cores round theirs eight times: the 2-norm error
// against 64 bits is 0.9e-7 - 4.5e-7 over the shapes at pick_sbf, theirs 3.7e-7 -
// 9.9e-7.
// Int8 and int4 weights are exact in bf16 and A takes two terms, |x - hi - lo| <=
// 2^-17 |x|: two products, the arithmetic of gemm_qbf.hip.  Outside that kernel's
// layouts, where the fp32 matrix cores' general kernel ran, A takes three terms and
// the products are three: fp32 precision as before.
//
// Bound: issue beside the matrix cores -- two (256x128) to three and a half (128x64) other
// vector instructions an MFMA, most of them the split's -- then fill and epilogue, at the clock the power limit
// leaves (1.94 GHz with 240 CUs busy, 2.3 with 48).  The counters have the matrix cores
// busy 69 % of a launch's CU cycles at 1500x5120x1280 (240 tiles of 256x128: 92 us, 214
// TFLOP/s, 162 us before on the fp32 matrix cores), 63 % on 256x96 tiles at
// 1500x3840x1280 (75 us) and 54 % on 128x64 tiles at 1500x1280x5120 (115 us).  Int8,
// 1500x5120x1280: 46 us, 427 TFLOP/s of algorithmic work; its two products take a third of
// the matrix-core time, and LDS and the loads' issue are as large.
//
// Values the split does not carry.  Infinities, NaNs (their residual is NaN) and
// |x| above the largest bf16 make the sum infinite or NaN.  Of a nonzero |x| < 2^-102
// up to 2^-124 may be lost (its terms reach bf16's denormals; values
// below 2^-134 have none at all), so a sum of K products is off by up to K 2^-124 times
// the largest of the other operand, and by K 2^-122 where products of terms
// themselves fall below 2^-126.  An output smaller than 2^24 times what it may be off by
// -- zero included -- is recomputed from the operands (sbf_repair), as is one that
// is not finite.  The split notes the largest magnitudes that pass through it (one
// v_max3 a pair of values, 11 instructions before), so outputs of 2^-70 and more need no
// second look unless an operand is past 2^28 / K, nor do those of a row of zeros.
#include "tml_internal.hpp"

#include <algorithm>
#include <cmath>
#include <type_traits>

namespace tml {
namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef uint32_t uintx4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

constexpr int kSbfXcd = 8;  // XCDs of an MI355X: workgroups are dealt to them round robin

struct SbfArgs {
    int M, N, K;
    const float *A;         // [M,K], 4-byte aligned
    const uint8_t *B;       // [K,N]: f32, binary16, int8, or int4 two a byte (even n in the low nibble)
    const float *scales;    // Q8_K block scales (32 elements each, N % 32 == 0)
    int ldb;                // bytes per B row
    const float *colscale;  // [N] per-column factor on A.B, or nullptr
    const float *bias;      // [N] or nullptr
    const float *res;       // [M,N] residual after the bias, or nullptr (may equal C)
    float *C;
    float alpha, beta;
    int act;
    long long tail0;
    unsigned a_bytes, s_bytes;  // M * K * 4, scale bytes
    int tiles_m, tiles_n;
    int nsplit, spl;        // K splits, k a split (a multiple of the slice)
    float *ws;              // nsplit > 1: [nsplit][M][N] raw partials
    int vec_epi;            // N % 4 == 0 and C, bias, residual, column scales 16-byte aligned
};

__device__ __forceinline__ __amdgpu_buffer_rsrc_t sbf_rsrc(const void *base, unsigned nbytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), (short)0, (int)nbytes, 0x00020000);
}

// Two floats to two bf16 (round to nearest even), a in the low half.
__device__ __forceinline__ uint32_t sbf_pk(float a, float b) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((floatx2){a, b}, bf16x2));
}
// NP bf16 terms of a pair of values.
template <int NP>
__device__ __forceinline__ void sbf_split(float a, float b, uint32_t (&t)[NP]) {
#pragma unroll
    for (int p = 0; p < NP; ++p) {
        t[p] = sbf_pk(a, b);
        if (p + 1 < NP) {
            a -= __uint_as_float(t[p] << 16);
            b -= __uint_as_float(t[p] & 0xFFFF0000u);
        }
    }
}

// Physical slot of logical slot s (8 k) in LDS row r of SL slots: four
// slots (64-byte rows) swap by (r / 2) mod 4, eight (128-byte rows) by r mod 8,
// so that the operand reads (16 rows, one slot each four lanes apart) and the
// staging writes (64 rows, one slot) run at the LDS's full rate: measured 8.3 and
// 13.9 cycles a 16-byte wave access, (r / 4) mod 4 9.3 and 16.3.
template <int SL>
__device__ __forceinline__ int sbf_slot(int r, int s) {
    if constexpr (SL == 4) return r * 4 + (s ^ ((r >> 1) & 3));
    else return r * 8 + (s ^ (r & 7));
}

// bf16 terms of A and B, and the pairs of them multiplied.
// Int8 / int4 at the fp32 products' precision (kSbfExact added to the format): three
// terms of A, three products.
constexpr int kSbfExact = 64;
template <int FMT>
constexpr int kSbfStored = FMT & ~kSbfExact;  // B's format in memory
template <int FMT>
constexpr unsigned kSbfBytes = FMT == TML_FMT_F32 ? 4u : FMT == TML_FMT_F16 ? 2u : 1u;  // an element's (int4: half)
template <int FMT>
constexpr bool kSbfInt = FMT == TML_FMT_Q8_0 || FMT == TML_FMT_Q4_0;
template <int FMT>
constexpr int kSbfPlanesA = kSbfInt<FMT> ? 2 : 3;
template <int FMT>
constexpr int kSbfPlanesB = kSbfInt<FMT> || FMT >= kSbfExact ? 1 : FMT == TML_FMT_F16 ? 2 : 3;
template <int FMT>
constexpr int kSbfProducts = kSbfInt<FMT> ? 2 : FMT >= kSbfExact ? 3 : FMT == TML_FMT_F16 ? 5 : 6;
// The int4 value of column n in the byte that holds it.
__device__ __forceinline__ float sbf_int4(uint32_t byte, int n) {
    return (float)((int32_t)(byte << ((n & 1) ? 24 : 28)) >> 28);
}

// One element of B as the f32 the reference multiplies by.
template <int FMT>
__device__ __forceinline__ float sbf_b(const SbfArgs &a, int k, int n) {
    if constexpr (FMT == TML_FMT_F32) return ((const float *)a.B)[(size_t)k * a.N + n];
    else if constexpr (FMT == TML_FMT_F16) return tml_half_bits(((const uint16_t *)a.B)[(size_t)k * a.N + n]);
    else if constexpr (kSbfStored<FMT> == TML_FMT_Q8_0) return (float)((const int8_t *)a.B)[(size_t)k * a.N + n];
    else if constexpr (kSbfStored<FMT> == TML_FMT_Q4_0) return sbf_int4(a.B[(size_t)k * a.ldb + n / 2], n);
    else return (float)((const int8_t *)a.B)[(size_t)k * a.N + n] * a.scales[((size_t)k * a.N + n) >> 5];
}

__device__ __forceinline__ bool sbf_not_finite(float v) { return (__float_as_uint(v) & 0x7F800000u) == 0x7F800000u; }
// The magnitude B cannot exceed; 0 where the split has to note it.
template <int FMT>
constexpr float kSbfTopB = FMT == TML_FMT_F16 ? 65504.0f : kSbfPlanesB<FMT> == 3 ? 0.0f : 128.0f;
// Below this an output may be off by more than 2^-24 of itself, where no operand of its
// tile exceeds top and kk products are summed (top of the file).
__device__ __forceinline__ float sbf_doubt(float kk, float top) { return kk * 0x1p-98f + kk * 0x1p-99f * top; }

// Recomputes the outputs of a 32 x 16 block that are not finite, on the fp32 matrix
// cores and straight from global memory: one wave, rows row0.. of A and columns col0..
// of B (`rows` and `cols` of them in the matrix), v the block in the staged tile.  A
// lane's 16-byte load of A holds k = 4 g .. 4 g + 3 of a 16-deep step, and
// matrix instruction e multiplies element e of every lane.  Bound: the fp32 matrix
// cores and the loads' issue where a whole tile is recomputed, the loads' latency where
// a row or column is.  1500x5120x1280 (92 us on ordinary values, 160 - 190 on the fp32-MFMA
// kernels): every output NaN 419 us, one row 152, one column 150; with one
// thread an output, all of K in a row, 10.3 ms, 396 us and 8.8 ms.
// U: steps in flight.
template <int FMT, int CS, int U>
__device__ __forceinline__ void sbf_recompute(const SbfArgs &a, float *v, int row0, int col0, int rows, int cols,
                                              int kbase, int kend) {
    const int lane = threadIdx.x & 63, c = lane & 15, g = lane >> 4;
    int bad = 0;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const int r = 16 * (e / 4) + 4 * g + e % 4;
        bad |= r < rows && c < cols && sbf_not_finite(v[r * CS + c]);
    }
    if (!__any(bad)) return;
    const __amdgpu_buffer_rsrc_t rsa = sbf_rsrc(a.A, a.a_bytes), rsb = sbf_rsrc(a.B, (unsigned)kend * (unsigned)a.ldb);
    const __amdgpu_buffer_rsrc_t rss = sbf_rsrc(FMT == TML_FMT_Q8_K ? (const void *)a.scales : a.B, a.s_bytes);
    const unsigned col = (unsigned)(col0 + c);
    const unsigned b_col = kSbfStored<FMT> == TML_FMT_Q4_0 ? col / 2u : col * kSbfBytes<FMT>;
    floatx4 acc[2] = {{0.0f, 0.0f, 0.0f, 0.0f}, {0.0f, 0.0f, 0.0f, 0.0f}};
#pragma unroll 1
    for (int kb = kbase; kb < kend; kb += 16 * U) {
        const int k0 = kb + 4 * g;
        uintx4 x[U][2];
        float y[U][4];
#pragma unroll
        for (int u = 0; u < U; ++u) {
#pragma unroll
            for (int t = 0; t < 2; ++t)
                x[u][t] = __builtin_amdgcn_raw_buffer_load_b128(
                    rsa, ((unsigned)(row0 + 16 * t + c) * (unsigned)a.K + (unsigned)(k0 + 16 * u)) * 4u, 0, 0);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const unsigned k = (unsigned)(k0 + 16 * u + e), off = k * (unsigned)a.ldb + b_col;  // (past kend: zero)
                if constexpr (FMT == TML_FMT_F32) y[u][e] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rsb, off, 0, 0));
                else if constexpr (FMT == TML_FMT_F16) y[u][e] = tml_half_bits(__builtin_amdgcn_raw_buffer_load_b16(rsb, off, 0, 0));
                else if constexpr (kSbfStored<FMT> == TML_FMT_Q4_0) y[u][e] = sbf_int4(__builtin_amdgcn_raw_buffer_load_b8(rsb, off, 0, 0), (int)col);
                else y[u][e] = (float)(int8_t)__builtin_amdgcn_raw_buffer_load_b8(rsb, off, 0, 0);
                if constexpr (FMT == TML_FMT_Q8_K)
                    y[u][e] *= __uint_as_float(
                        __builtin_amdgcn_raw_buffer_load_b32(rss, k * ((unsigned)a.N / 8u) + col / 32u * 4u, 0, 0));
            }
        }
        __builtin_amdgcn_sched_barrier(0);  // (all U steps' loads first: the scheduler would spread them, a wait each)
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    const bool in = k0 + 16 * u + e < kend;  // (A reads on past kend)
                    acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(in ? __uint_as_float(x[u][t][e]) : 0.0f,
                                                                  in ? y[u][e] : 0.0f, acc[t], 0, 0, 0);
                }
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const int r = 16 * (e / 4) + 4 * g + e % 4;
        float *const to = &v[r * CS + c];
        if (r < rows && c < cols && sbf_not_finite(*to)) *to = acc[e / 4][e % 4];
    }
}

// The smallest nonzero and the largest magnitude of what it has seen, as bits.
struct SbfRange {
    uint32_t lo = ~0u, hi = 0u;  // lo: 2 * bits - 1, so that zeros come last
    __device__ __forceinline__ void see(float v) {
        const uint32_t u = __float_as_uint(v);
        lo = min(lo, (u << 1) - 1u);
        hi = max(hi, u & 0x7FFFFFFFu);
    }
    __device__ __forceinline__ void see(SbfRange r) {
        lo = min(lo, r.lo);
        hi = max(hi, r.hi);
    }
    // infinity where all were zero
    __device__ __forceinline__ float least() const {
        return lo == ~0u ? __builtin_huge_valf() : __uint_as_float((lo + 1u) >> 1);
    }
    __device__ __forceinline__ float most() const { return __uint_as_float(hi); }
};

// Puts right the outputs in ct, the tile's sums over k in [kbase, kend), that the split
// does not carry (top of the file).  Small ones are first weighed by what their own
// row of A and column of B hold: a sum of zeros, or of values that cancel, is as good as
// any, and rows of zeros are told apart before any column is read.  512x4096x1024 f32
// with one column of zeros: 50 us, 29 without (cold instructions, then the loads'
// latency).  top: the largest magnitude this lane has split.  ex: LDS, kSbfRepairFloats.
template <int BM, int BN, int NW>
constexpr int kSbfRepairFloats = 2 * (BM + 64 * NW);
template <int FMT, int BM, int BN, int NW>
__device__ __forceinline__ void sbf_repair(const SbfArgs &a, float *ct, float *ex, float top, int m0, int n0, int kbase,
                                           int kend) {
    constexpr int NT = 64 * NW, CS = BN + 4, G = NT / BN;
    constexpr int U = NW == 8 && FMT != TML_FMT_Q8_K ? 8 : 4;  // (no more registers than the K loop's)
    int tid = threadIdx.x;
    __asm__ volatile("" : "+v"(tid));  // (nothing of this is computed before the K loop and held through it)
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int rows = min(BM, a.M - m0), cols = min(BN, a.N - n0);
    const float kk = (float)(kend - kbase);
    SbfRange *const rrow = (SbfRange *)ex, *const rcol = rrow + BM;
    if constexpr (kSbfTopB<FMT> == 0.0f) {
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) top = fmaxf(top, __shfl_xor(top, o));
        if (lane == 0) ex[wave] = top;
        __syncthreads();
        for (int w = 0; w < NW; ++w) top = fmaxf(top, ex[w]);
    }
    const float doubt = sbf_doubt(kk, top);
    int small = 0;
#pragma unroll 4
    for (int e = tid; e < BM * BN; e += NT)
        small |= e / BN < rows && e % BN < cols && fabsf(ct[e / BN * CS + e % BN]) < doubt;
    if (__syncthreads_or(small)) {
        // eight rows at a time, a 128-byte piece of each an instruction
        const __amdgpu_buffer_rsrc_t rsa = sbf_rsrc(a.A, a.a_bytes);
        const int q = lane % 8;
#pragma unroll 1
        for (int r = 8 * wave + lane / 8; r < BM; r += 8 * NW) {
            int any = 0;
            for (int n = q; n < cols; n += 8) any |= r < rows && fabsf(ct[r * CS + n]) < doubt;
            if (!__any(any)) continue;
            SbfRange x;
#pragma unroll 1
            for (int kb = kbase; kb < kend; kb += 32 * 8) {
                uintx4 w[8];
#pragma unroll
                for (int u = 0; u < 8; ++u)
                    w[u] = __builtin_amdgcn_raw_buffer_load_b128(
                        rsa, ((unsigned)(m0 + r) * (unsigned)a.K + (unsigned)(kb + 32 * u + 4 * q)) * 4u, 0, 0);
#pragma unroll
                for (int u = 0; u < 8; ++u)
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        x.see(kb + 32 * u + 4 * q + e < kend ? __uint_as_float(w[u][e]) : 0.0f);
            }
#pragma unroll
            for (int o = 4; o > 0; o >>= 1) {
                SbfRange y;
                y.lo = (uint32_t)__shfl_xor((int)x.lo, o);
                y.hi = (uint32_t)__shfl_xor((int)x.hi, o);
                x.see(y);
            }
            if (q == 0) rrow[r] = x;
        }
        __syncthreads();
        small = 0;
        for (int e = tid; e < BM * BN; e += NT)
            small |= e / BN < rows && e % BN < cols && fabsf(ct[e / BN * CS + e % BN]) < doubt && rrow[e / BN].lo != ~0u;
        if (__syncthreads_or(small)) {
            const int n = tid % BN, grp = tid / BN;
            if (grp < G) {
                SbfRange x;
                if (n < cols) {
#pragma unroll 16
                    for (int k = kbase + grp; k < kend; k += G) x.see(sbf_b<FMT>(a, k, n0 + n));
                }
                rcol[tid] = x;
            }
            __syncthreads();
            if (tid < BN) {
                for (int z = 1; z < G; ++z) rcol[tid].see(rcol[tid + z * BN]);
            }
            __syncthreads();
            for (int e = tid; e < BM * BN; e += NT) {
                const int r = e / BN, c = e % BN;
                float *const v = &ct[r * CS + c];
                if (r >= rows || c >= cols || !(fabsf(*v) < doubt)) continue;
                const SbfRange x = rrow[r], y = rcol[c];
                if (x.lo == ~0u || y.lo == ~0u) continue;  // a sum of zeros
                // (the last bits' product is 2^-46 of the values')
                float off = x.least() * y.least() < 0x1p-80f ? kk * 0x1p-98f : 0.0f;
                if (x.least() < 0x1p-102f) off += kk * 0x1p-100f * y.most();
                if (y.least() < 0x1p-102f) off += kk * 0x1p-100f * x.most();
                if (fabsf(*v) < off) *v = __builtin_nanf("");
            }
            __syncthreads();
        }
    }
#pragma unroll 1
    for (int rb = 0; rb < BM / 32; ++rb)  // (blocks of a row, or of a column, on different waves)
#pragma unroll 1
        for (int cb = 0; cb < BN / 16; ++cb)
            if ((rb + cb) % NW == wave)
                sbf_recompute<FMT, CS, U>(a, ct + 32 * rb * CS + 16 * cb, m0 + 32 * rb, n0 + 16 * cb, rows - 32 * rb,
                                       cols - 16 * cb, kbase, kend);
    __syncthreads();
}

// A workgroup of NW = 4 or 8 waves owns a BM x BN tile of C, each wave a WM x
// WN sub-tile (or, with KW = 2 wave groups, half the k of one), and walks K in
// BK-deep slices.  A wave loads the A it multiplies straight into registers, in
// the MFMA's own layout, and splits it there (int8 / int4, whose products are a
// third: in whole 128-byte rows, turned through LDS rows of the wave's own -- a load
// in the MFMA's layout takes 16 bytes of a row a lane, neighbouring lanes different
// rows, and 30-40 cycles to issue; 1500x3840x1280 54.6 -> 45.3 us, while the
// three-term formats, whose LDS is as busy as their matrix cores, lose up to 18 %); B is loaded once per workgroup,
// split, and passed through three LDS stages as rows of 16-byte slots (8 k), one
// barrier a slice: a slice is written two steps before it is multiplied, so its
// first operands are read before the barrier that starts its step.  (With A in LDS too, its writes -- 64 bytes a clock -- and
// reads took the LDS as long as the products take the matrix cores.)  Slices are
// loaded D ahead, and the splitting of the next slice is dealt out between the
// groups of matrix instructions of this one: VALU work in the wave that waits on
// the matrix core is nearly free, the same work in another wave is not (measured:
// 16 MFMAs and 32 subtractions a wave, two waves a SIMD, 690 cycles interleaved,
// 615 without the subtractions; half the waves on each, the sum of the two).
//
// k order: slot g of a 32-k half holds k = 4 g .. 4 g + 3 and 16 + 4 g .. 16 + 4
// g + 3, so that each of a lane's two 16-byte A loads covers 64 contiguous bytes
// of a row over its four lanes.
template <int FMT, int BM, int BN, int WM, int WN, int BK, int KW, int NW, int D>
__global__ __launch_bounds__(64 * NW) void gemm_sbf_kernel(SbfArgs a) {
    static_assert(KW == 1 ? BK == 32 : KW == 2 && BK == 64, "each wave group multiplies one 32-k half of a slice");
    static_assert(NW == 4 || NW == 8, "one or two waves a SIMD");
    constexpr int NA = kSbfPlanesA<FMT>, NB = kSbfPlanesB<FMT>, NP = kSbfProducts<FMT>;
    constexpr bool AL = kSbfInt<FMT>;  // A through the waves' own LDS rows (below)
    constexpr bool COR = NP > 2;  // the small products have accumulators of their own
    constexpr int SL = BK / 8;    // 16-byte slots (8 k) of an LDS row
    constexpr int NT = 64 * NW;
    constexpr int NWS = NW / KW;  // waves per group, one per sub-tile
    constexpr int TM = WM / 16, TN = WN / 16, WAVES_N = BN / WN;
    static_assert((BM / WM) * (BN / WN) == NWS, "one wave of a group per WM x WN sub-tile");
    // B's staging tasks: one (column, 8-k slot) each, PB a thread.
    constexpr int TB = BN * SL, PB = (TB + NT - 1) / NT;
    constexpr int RW = FMT == TML_FMT_Q8_K ? 16 : 8;  // registers of a task (Q8_K: 8 values, 8 scales)

    constexpr int kStage = BN * SL * NB;  // 16-byte slots of a stage
    constexpr int CS = BN + 4;            // floats of a staged C row (rows 4 apart: 16 banks on)
    constexpr int kARows = 3 * kStage;    // AL: the waves' own A rows, WM x 8 slots each
    constexpr int kLoop = kARows + (AL ? NW * WM * 8 : 0);
    constexpr int kTile = (BM * CS + kSbfRepairFloats<BM, BN, NW> + NW + (KW == 2 ? NWS * (WM / 16) : 0)) / 4;  // the epilogue's
    constexpr int kLds = kLoop > kTile ? kLoop : kTile;
    __shared__ uintx4 lds[kLds];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kg = KW == 2 ? wave / NWS : 0;
    const int sw = wave % NWS;
    const int wm0 = (sw / WAVES_N) * WM, wn0 = (sw % WAVES_N) * WN;
    const int c = lane & 15, g = lane >> 4;

    // Workgroup -> tile: consecutive ids within each XCD (own L2), in groups
    // of eight tile rows so that neighbours share A rows and B columns.
    // K splits split by split: an XCD's workgroups share one k range.
    int tile_m, tile_n, split;
    {
        const int nblk = gridDim.x, b = blockIdx.x;
        const int per = nblk / kSbfXcd, rem = nblk % kSbfXcd;
        const int xcd = b % kSbfXcd, idx = b / kSbfXcd;
        int lin = (xcd < rem) ? xcd * (per + 1) + idx : rem * (per + 1) + (xcd - rem) * per + idx;
        split = lin / (a.tiles_m * a.tiles_n);
        lin -= split * (a.tiles_m * a.tiles_n);
        constexpr int GM = 8;
        const int group = GM * a.tiles_n;
        const int first_m = (lin / group) * GM;
        const int gsize = min(a.tiles_m - first_m, GM);
        tile_m = first_m + (lin % group) % gsize;
        tile_n = (lin % group) / gsize;
    }
    const int m0 = tile_m * BM, n0 = tile_n * BN;
    const int kbase = split * a.spl, kend = min(a.K, kbase + a.spl);  // this split's k

    // ---- loads.  A lane's offsets are fixed; the slice moves the buffer's base
    // and byte count (scalar work only).  Rows of A past M and k-rows of B past
    // kend lie past the byte count and read zeros, as does a slice of A past kend.  A's k past
    // kend in the last slice reads on, against B's zero rows; B columns past N read the next k-row and feed dropped
    // outputs.  (A value there that is not finite makes its sum a NaN, which the
    // epilogue recomputes.)
    auto col_bytes = [](unsigned n) constexpr { return kSbfStored<FMT> == TML_FMT_Q4_0 ? n / 2u : n * kSbfBytes<FMT>; };
    const unsigned b_bytes = (unsigned)kend * (unsigned)a.ldb;
    // A: AL loads 8 rows of 128 bytes an instruction (lane / 8, lane % 8), else 16
    // rows' 16-byte pieces in the MFMA's layout (c, g)
    const unsigned a_off = AL ? ((unsigned)(lane / 8) * (unsigned)a.K + 4u * (unsigned)(lane % 8)) * 4u
                              : ((unsigned)c * (unsigned)a.K + 4u * (unsigned)g) * 4u;
    unsigned b_off[PB], s_off[PB];
    int slot_b[PB];
#pragma unroll
    for (int t = 0; t < PB; ++t) {
        const int j = tid + t * NT, n = j % BN, sl = j / BN;
        const unsigned k = (unsigned)(32 * (sl / 4) + 4 * (sl % 4));
        b_off[t] = k * (unsigned)a.ldb + col_bytes((unsigned)n);
        s_off[t] = k * ((unsigned)a.N / 8u) + (unsigned)n / 32u * 4u;
        slot_b[t] = sbf_slot<SL>(n, sl % SL);
    }
    auto moved = [](const void *base, unsigned nbytes, unsigned adv) __attribute__((always_inline)) {
        adv = min(adv, nbytes);
        return sbf_rsrc((const char *)base + adv, nbytes - adv);
    };
    // the buffers at a slice's first k
    auto at_a = [&](int k0) __attribute__((always_inline)) {
        const int k = kbase + k0 + 32 * kg;
        return moved(a.A, a.a_bytes, k < kend ? ((unsigned)(m0 + wm0) * (unsigned)a.K + (unsigned)k) * 4u : a.a_bytes);
    };
    auto at_b = [&](int k0) __attribute__((always_inline)) {
        return moved(a.B, b_bytes, (unsigned)(kbase + k0) * (unsigned)a.ldb + col_bytes((unsigned)n0));
    };
    auto at_s = [&](int k0) __attribute__((always_inline)) {  // scale of (k, n): scales[k * N / 32 + n / 32]
        return FMT == TML_FMT_Q8_K ? moved(a.scales, a.s_bytes, (unsigned)(kbase + k0) * ((unsigned)a.N / 8u) + (unsigned)n0 / 8u)
                                   : sbf_rsrc(a.B, 0u);
    };
    uint32_t ra[D][TM][8], rb[D][PB][RW];
    // half h of A tile i's eight k, and k-row kk of B task t
    // (off: the lane's offset, from fresh() -- a sum the compiler cannot keep in a
    // register per row over the whole loop, where there is none to spare)
    auto fresh = [](unsigned off) __attribute__((always_inline)) {
        __asm__ volatile("" : "+v"(off));
        return off;
    };
    auto load_a = [&](__amdgpu_buffer_rsrc_t rs, unsigned off, int i, int h, int d) __attribute__((always_inline)) {
        const uintx4 v = __builtin_amdgcn_raw_buffer_load_b128(
            rs, AL ? off + (unsigned)(16 * i + 8 * h) * (unsigned)a.K * 4u
                   : off + (unsigned)(16 * i) * (unsigned)a.K * 4u + 64u * h, 0, 0);
#pragma unroll
        for (int e = 0; e < 4; ++e) ra[d][i][4 * h + e] = v[e];
    };
    auto load_b = [&](__amdgpu_buffer_rsrc_t rs, __amdgpu_buffer_rsrc_t rsc, unsigned off0, int t, int kk, int d)
                      __attribute__((always_inline)) {
        const unsigned row = (unsigned)((kk < 4 ? 0 : 12) + kk);
        const unsigned off = off0 + row * (unsigned)a.ldb;
        if constexpr (FMT == TML_FMT_F32) rb[d][t][kk] = __builtin_amdgcn_raw_buffer_load_b32(rs, off, 0, 0);
        else if constexpr (FMT == TML_FMT_F16) rb[d][t][kk] = __builtin_amdgcn_raw_buffer_load_b16(rs, off, 0, 0);
        else rb[d][t][kk] = __builtin_amdgcn_raw_buffer_load_b8(rs, off, 0, 0);
        if constexpr (FMT == TML_FMT_Q8_K) {
            rb[d][t][8 + kk] = __builtin_amdgcn_raw_buffer_load_b32(rsc, s_off[t] + row * ((unsigned)a.N / 8u), 0, 0);
        }
    };

    // AL: rows 16 i + 8 h .. + 7 through the wave's own LDS rows (no workgroup barrier: one
    // wave's LDS accesses run in order, and turn() keeps the compiler's order of the
    // lanes' writes and reads), 16-byte chunk q of row r in slot q ^ (r % 8).
    auto turn = []() __attribute__((always_inline)) {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    uintx4 *const aw = lds + kARows + wave * (WM * 8);
    const int slot_aw = lane / 8 * 8 + (lane % 8 ^ lane / 8), slot_ar = c * 8 + (g ^ (c & 7));
    uint32_t rr[TM][8];
    auto write_a = [&](int i, int h, int d) __attribute__((always_inline)) {
        aw[slot_aw + (16 * i + 8 * h) * 8] = (uintx4){ra[d][i][4 * h], ra[d][i][4 * h + 1], ra[d][i][4 * h + 2],
                                                      ra[d][i][4 * h + 3]};
    };
    auto read_a = [&](int i) __attribute__((always_inline)) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const uintx4 v = aw[(slot_ar ^ (4 * h)) + 16 * i * 8];
#pragma unroll
            for (int e = 0; e < 4; ++e) rr[i][4 * h + e] = v[e];
        }
    };

    // ---- splitting, a pair of k at a time: A's pair e to word e of the next
    // slice's operands, B's to word e of the slots write_b stores.
    constexpr bool TOP = kSbfTopB<FMT> == 0.0f;
    // the largest magnitudes split: of B, and of A's row 16 i + c (with B bounded by its
    // format, to tell rows of zeros; two terms of A do without)
    float top_b = kSbfTopB<FMT>, top_a[TM];
#pragma unroll
    for (int i = 0; i < TM; ++i) top_a[i] = 0.0f;
    auto note = [&](float &t, float x, float y) __attribute__((always_inline)) {
        t = fmaxf(fmaxf(t, fabsf(x)), fabsf(y));
    };
    uintx4 av[2][NA][TM], bp[PB][NB];
    float bx[PB][4][2];  // B's values, for note()
    auto split_a = [&](int i, int e, int d, int nxt) __attribute__((always_inline)) {
        uint32_t t[NA];
        const float x = __uint_as_float(AL ? rr[i][2 * e] : ra[d][i][2 * e]);
        const float y = __uint_as_float(AL ? rr[i][2 * e + 1] : ra[d][i][2 * e + 1]);
        if constexpr (COR) note(top_a[i], x, y);
        sbf_split<NA>(x, y, t);
#pragma unroll
        for (int p = 0; p < NA; ++p) av[nxt][p][i][e] = t[p];
    };
    auto split_b = [&](int t, int e, int d) __attribute__((always_inline)) {
#pragma clang fp contract(off)  // (the dequantized value is the rounded product, in every tile)
        float *const x = bx[t][e];
#pragma unroll
        for (int z = 0; z < 2; ++z) {
            const uint32_t w = rb[d][t][2 * e + z];
            if constexpr (FMT == TML_FMT_F32) x[z] = __uint_as_float(w);
            else if constexpr (FMT == TML_FMT_F16) x[z] = tml_half_bits(w);
            else if constexpr (kSbfStored<FMT> == TML_FMT_Q8_0) x[z] = (float)(int8_t)w;
            else if constexpr (kSbfStored<FMT> == TML_FMT_Q4_0) x[z] = sbf_int4(w, tid + t * NT);
            else x[z] = (float)(int8_t)w * __uint_as_float(rb[d][t][8 + 2 * e + z]);
        }
        uint32_t v[NB];
        sbf_split<NB>(x[0], x[1], v);
#pragma unroll
        for (int p = 0; p < NB; ++p) bp[t][p][e] = v[p];
    };
    auto write_b = [&](int t, int p, int stage) __attribute__((always_inline)) {
        if (TB % NT == 0 || tid + t * NT < TB) {
            lds[stage + slot_b[t] + p * BN * SL] = bp[t][p];
            if (TOP && p == 0) {  // (here, so that threads without a task split nothing: noted in split_b, 9-16 registers more)
#pragma unroll
                for (int e = 0; e < 4; ++e) note(top_b, bx[t][e][0], bx[t][e][1]);
            }
        }
    };

    // acc holds the hh products, cor the five (four) smaller ones: a slice
    // rounds the large sum once, and the small terms keep their own.  (Two terms
    // of A against int8 or int4 weights share one: the split itself, 2^-17 of a
    // product, is their error.)
    floatx4 acc[TM][TN], cor[COR ? TM : 1][COR ? TN : 1];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            acc[i][j] = (floatx4){0.0f, 0.0f, 0.0f, 0.0f};
            if constexpr (COR) cor[i][j] = acc[i][j];
        }

    // One slice: A's operands av[cur] and the LDS stage at sr are multiplied,
    // while B's register set db becomes the stage at sw (two slices on) and A's
    // set da becomes av[nxt] (the next slice).  Lane (c, g) reads slot g (of its
    // group's half) of B columns wn0 + 16 j + c.  JB columns at a time, plane pair
    // by plane pair: a group of TM * JB MFMAs is independent, and a share of the
    // staging follows each group.  A B plane's registers take the next columns --
    // after the last, the first of the next slice at sn -- as soon as the last
    // product that needs it has run.
    constexpr int JB = TM >= 4 ? 1 : TM >= 2 || TN < 4 ? 2 : 4, kGroups = TN / JB * NP;
    static_assert(TN % JB == 0, "whole groups of columns");
    // (one plane only: the next columns' registers apart, read a whole group of
    // columns ahead; group n of the unrolled slices uses bv[n % 2])
    constexpr int BUF = NB == 1 ? 2 : 1;
    uintx4 bv[BUF][NB][JB];
    const int slot_r = sbf_slot<SL>(wn0 + c, 4 * kg + g);
    auto read_b = [&](int buf, int p, int j0, int stage) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < JB; ++j) bv[buf][p][j] = lds[stage + slot_r + p * BN * SL + 16 * SL * (j0 + j)];
    };
    // When the staging runs: splitting step v (B's tasks, then A's tiles, four
    // pairs each) after group v kGroups / kSplits; a task's or tile's reloads from
    // the group after its last pair on, two k-rows or one half a group, and B's
    // plane writes every few groups: bunched, the writes hold up the operand reads
    // behind them and the loads' issue holds up the wave.
    constexpr int kSplits = 4 * (PB + TM);
    auto split_at = [](int v) constexpr { return v * kGroups / kSplits; };
    auto load_at = [](int task, int i) constexpr {
        const int g0 = (4 * task + 3) * kGroups / kSplits + i;
        return g0 < kGroups ? g0 : kGroups - 1;
    };
    // (AL: A's rows are read back one group before their first split and written
    // one before that; their registers are reloaded at once)
    auto read_a_at = [](int i) constexpr {
        const int g0 = 4 * (PB + i) * kGroups / kSplits - 1;
        return g0 > 0 ? g0 : 0;
    };
    auto write_a_at = [](int i) constexpr {
        const int g0 = 4 * (PB + i) * kGroups / kSplits - 2;
        return g0 > 0 ? g0 : 0;
    };
    auto write_at = [](int t, int p) constexpr {
        const int g0 = (4 * t + 3) * kGroups / kSplits;
        return g0 + (kGroups - 1 - g0) * p / NB;
    };
    auto slice = [&](int cur, int nxt, int sr, int sn, int sw_, int db, int kb, int da,
                     int ka) __attribute__((always_inline)) {
        const __amdgpu_buffer_rsrc_t rsa = at_a(ka), rsb = at_b(kb), rss = at_s(kb);
        const unsigned a_fresh = fresh(a_off);
        unsigned b_fresh[PB];
#pragma unroll
        for (int w = 0; w < PB; ++w) b_fresh[w] = fresh(b_off[w]);
#pragma unroll
        for (int j0 = 0; j0 < TN; j0 += JB) {
            constexpr int QA[6] = {0, 1, 2, 0, 1, 0}, QB[6] = {0, 0, 0, 1, 1, 2};
            const int buf = BUF == 2 ? (TN / JB * cur + j0 / JB) & 1 : 0;
#pragma unroll
            for (int t = 0; t < NP; ++t) {
#pragma unroll
                for (int j = 0; j < JB; ++j)
#pragma unroll
                    for (int i = 0; i < TM; ++i) {
                        floatx4 &to = t == 0 || !COR ? acc[i][j0 + j] : cor[COR ? i : 0][COR ? j0 + j : 0];
                        to = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, av[cur][QA[t]][i]),
                                                                     __builtin_bit_cast(bf16x8, bv[buf][QB[t]][j]), to, 0,
                                                                     0, 0);
                    }
                if (BUF == 2 ? t == 0 : t + 1 == NP || QB[t + 1] != QB[t]) {
                    if (j0 + JB < TN) read_b(BUF == 2 ? buf ^ 1 : 0, QB[t], j0 + JB, sr);
                    else read_b(BUF == 2 ? buf ^ 1 : 0, QB[t], 0, sn);
                }
                const int gi = j0 / JB * NP + t;
                if constexpr (AL) {
#pragma unroll
                    for (int i = 0; i < TM; ++i)
                        if (write_a_at(i) == gi) {
                            turn();
#pragma unroll
                            for (int h = 0; h < 2; ++h) {
                                write_a(i, h, da);
                                load_a(rsa, a_fresh, i, h, da);
                            }
                        }
#pragma unroll
                    for (int i = 0; i < TM; ++i)
                        if (read_a_at(i) == gi) {
                            turn();
                            read_a(i);
                        }
                }
#pragma unroll
                for (int v = 0; v < kSplits; ++v)
                    if (split_at(v) == gi) {
                        if (v < 4 * PB) split_b(v / 4, v % 4, db);
                        else split_a(v / 4 - PB, v % 4, da, nxt);
                    }
#pragma unroll
                for (int w = 0; w < PB; ++w) {
#pragma unroll
                    for (int kk = 0; kk < 8; ++kk)
                        if (load_at(w, kk / 2) == gi) load_b(rsb, rss, b_fresh[w], w, kk, db);
#pragma unroll
                    for (int p = 0; p < NB; ++p)
                        if (write_at(w, p) == gi) write_b(w, p, sw_);
                }
#pragma unroll
                for (int i = 0; i < TM; ++i)
#pragma unroll
                    for (int h = 0; h < 2; ++h)
                        if (!AL && load_at(PB + i, h) == gi) load_a(rsa, a_fresh, i, h, da);
#pragma unroll
                for (int i = 0; i < TM * JB; ++i) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x002, 3, 0);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    };

    // Register sets d hold the slices kt with kt % D == d.  In step kt, A's set
    // (kt + 1) % D becomes av and takes slice kt + 1 + D, B's set (kt + 2) % D
    // becomes the stage (kt + 2) % 3 and takes slice kt + 2 + D.  The step count
    // is rounded up to whole rounds of U = lcm(2, D) steps (steps past K multiply
    // zeros), so a step's register sets are fixed in the code.
    constexpr int U = D % 2 == 0 ? D : 2 * D;
    const int nk = ((kend - kbase + BK - 1) / BK + U - 1) / U * U;
    auto barrier = [&]() __attribute__((always_inline)) {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    };
    auto load_set = [&](bool is_a, int d, int k0) __attribute__((always_inline)) {
        const __amdgpu_buffer_rsrc_t rsa = at_a(k0), rsb = at_b(k0), rss = at_s(k0);
#pragma unroll
        for (int t = 0; t < PB && !is_a; ++t)
#pragma unroll
            for (int kk = 0; kk < 8; ++kk) load_b(rsb, rss, b_off[t], t, kk, d);
#pragma unroll
        for (int i = 0; i < TM && is_a; ++i)
#pragma unroll
            for (int h = 0; h < 2; ++h) load_a(rsa, a_off, i, h, d);
    };
    auto stage_b = [&](int d, int stage) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < PB; ++t) {
#pragma unroll
            for (int e = 0; e < 4; ++e) split_b(t, e, d);
#pragma unroll
            for (int p = 0; p < NB; ++p) write_b(t, p, stage);
        }
    };
#pragma unroll
    for (int d = 0; d < D; ++d) {
        load_set(false, d, d * BK);
        load_set(true, d, d * BK);
    }
    stage_b(0, 0);
    load_set(false, 0, D * BK);
    if constexpr (AL) {
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            write_a(i, 0, 0);
            write_a(i, 1, 0);
            turn();
            read_a(i);
        }
    }
#pragma unroll
    for (int i = 0; i < 4 * TM; ++i) split_a(i / 4, i % 4, 0, 0);
    load_set(true, 0, D * BK);
    stage_b(1 % D, kStage);
    load_set(false, 1 % D, (1 + D) * BK);
    barrier();
#pragma unroll
    for (int p = 0; p < NB; ++p) read_b(0, p, 0, 0);
    int s0 = 0, s1 = kStage, s2 = 2 * kStage;  // the stages of slices kt, kt + 1, kt + 2
    for (int kt0 = 0; kt0 < nk; kt0 += U) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int kt = kt0 + u;
            slice(u & 1, (u + 1) & 1, s0, s1, s2, (u + 2) % D, (kt + 2 + D) * BK, (u + 1) % D, (kt + 1 + D) * BK);
            barrier();
            const int s = s0;
            s0 = s1;
            s1 = s2;
            s2 = s;
        }
    }
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
            if constexpr (COR) acc[i][j] += cor[i][j];

    // ---- epilogue.  The tile's sums go through LDS (free: the loop's last
    // barrier follows every wave's last read) and are written as whole 16-byte
    // pieces of C rows, consecutive lanes a row's consecutive pieces.  Lane
    // (c, g) holds rows 4 g + e, column c of each MFMA tile; with two wave
    // groups, group 1 adds its half of the k first.  The code is kept short --
    // one loop per activation, the recomputation rolled and apart -- because a
    // launch runs it once, from a cold instruction cache: unrolled with every
    // activation in every element it cost 36 k cycles a tile (16 of the 102 us of
    // 1500x5120x1280).
    float *const ct = (float *)lds;
    // not finite, or below `least` (no less than sbf_doubt, top permitting).  Rows past M,
    // whose sums are zeros, are not looked at; columns past N hold other columns' products
    const float kk = (float)(kend - kbase), least = fmaxf(0x1p-70f, sbf_doubt(kk, kSbfTopB<FMT>));
    const uint32_t least2 = __float_as_uint(least) << 1;  // (the sign shifted out)
    uint32_t *const flags = (uint32_t *)(ct + BM * CS + kSbfRepairFloats<BM, BN, NW>);
    // rows of zeros (their lanes c, c + 16, c + 32, c + 48 met nothing else), a bit each
    uint32_t zeros[TM];
#pragma unroll
    for (int i = 0; i < TM; ++i) {
        const uint64_t z = COR ? __builtin_amdgcn_ballot_w64(top_a[i] == 0.0f) : 0;
        zeros[i] = (uint32_t)(z & z >> 16 & z >> 32 & z >> 48) & 0xFFFFu;
    }
    uint32_t worst = 0;
    auto put = [&](bool add) __attribute__((always_inline)) {
        const int rows = a.M - m0 - wm0 - 4 * g;
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                uint32_t w = 0, any = 0;
#pragma unroll
                for (int j = 0; j < TN; ++j) {
                    float *const to = &ct[(wm0 + 16 * i + 4 * g + e) * CS + wn0 + 16 * j + c];
                    const float v = add ? *to + acc[i][j][e] : acc[i][j][e];
                    const uint32_t u = __float_as_uint(v) << 1;
                    // (two terms of A: a zero sum is taken as it is, as in gemm_qbf.hip)
                    w = max(w, (COR || u != 0 ? u : least2) - least2);
                    any |= u;
                    *to = v;
                }
                if (COR && (zeros[i] >> (4 * g + e) & 1) && any == 0) w = 0;
                worst = max(worst, 16 * i + e < rows ? w : 0u);
            }
    };
    if constexpr (KW == 1) {
        put(false);
    } else {
        if (kg == 1) {
            put(false);
#pragma unroll
            for (int i = 0; i < TM && COR; ++i)
                if (lane == 0) flags[NW + sw * TM + i] = zeros[i];
        }
        worst = 0;
        __syncthreads();
        if (kg == 0) {
#pragma unroll
            for (int i = 0; i < TM && COR; ++i) zeros[i] &= flags[NW + sw * TM + i];
            put(true);
        }
    }
    float top = top_b;
#pragma unroll
    for (int i = 0; i < TM && TOP; ++i) top = fmaxf(top, top_a[i]);
    const bool suspect = worst >= 0xFF000000u - least2 || (TOP && top > 0x1p28f / kk);
    // (each wave's flag in LDS past sbf_repair's floats: one barrier, where __syncthreads_or has two)
    const bool mine = __any(suspect);
    if (lane == 0) flags[wave] = mine;
    __syncthreads();
    uint32_t any = 0;
#pragma unroll
    for (int w = 0; w < NW; ++w) any |= flags[w];
    if (__builtin_expect(__builtin_amdgcn_readfirstlane(any) != 0, 0))
        sbf_repair<FMT, BM, BN, NW>(a, ct, ct + BM * CS, top, m0, n0, kbase, kend);
    constexpr int CH = BN / 4, RPP = NT / CH;  // 16-byte pieces of a tile row; rows a pass
    const int pc = 4 * (tid % CH), tr0 = tid / CH, col = n0 + pc;  // a thread's pieces lie in one column of pieces
    if (tr0 >= RPP || col >= a.N) return;
    const int tr_end = min(BM, a.M - m0);
    if (a.nsplit > 1) {
        // raw partial of this split; launch_splitk_reduce adds the splits in
        // order and runs the epilogue
        float *const part = a.ws + ((size_t)split * a.M + m0) * a.N + col;
#pragma unroll 1
        for (int tr = tr0; tr < tr_end; tr += RPP) {
            const floatx4 v = *(const floatx4 *)&ct[tr * CS + pc];
            float *const to = part + (size_t)tr * a.N;
            if (a.N % 4 == 0) *(floatx4 *)to = v;
            else
                for (int q = 0; q < 4 && col + q < a.N; ++q) to[q] = v[q];
        }
        return;
    }
    auto factor = [&](int n) __attribute__((always_inline)) { return a.colscale ? a.alpha * a.colscale[n] : a.alpha; };
    auto scalar_piece = [&](int tr) {
        const size_t o = (size_t)(m0 + tr) * a.N + col;
#pragma unroll 1
        for (int q = 0; q < 4 && col + q < a.N; ++q) {
            float v = factor(col + q) * ct[tr * CS + pc + q];
            if (a.beta != 0.0f) v += a.beta * a.C[o + q];
            if (a.bias) v += a.bias[col + q];
            if (a.res) v += a.res[o + q];
            tml_store_c(a.C + o + q, tml_apply_act(v, a.act, (long long)o + q, a.tail0));
        }
    };
    // UN rows' loads in flight together
    auto finish = [&](auto act_tag, auto un_tag) __attribute__((always_inline)) {
        constexpr int ACT = decltype(act_tag)::value, UN = decltype(un_tag)::value;
        floatx4 bias4 = {0.f, 0.f, 0.f, 0.f};
        if (a.bias) bias4 = *(const floatx4 *)(a.bias + col);
        const floatx4 alpha4 = {factor(col), factor(col + 1), factor(col + 2), factor(col + 3)};
#pragma unroll 1
        for (int tr = tr0; tr < tr_end; tr += UN * RPP) {
            floatx4 v4[UN], cv[UN], rv[UN];
#pragma unroll
            for (int p = 0; p < UN; ++p) {
                const int t = min(tr + p * RPP, tr_end - 1);
                const size_t o = (size_t)(m0 + t) * a.N + col;
                v4[p] = *(const floatx4 *)&ct[t * CS + pc];
                if (a.beta != 0.0f) cv[p] = *(const floatx4 *)(a.C + o);
                if (a.res) rv[p] = *(const floatx4 *)(a.res + o);
            }
#pragma unroll
            for (int p = 0; p < UN; ++p) {
                const int t = tr + p * RPP;
                if (t >= tr_end) break;
                const size_t o = (size_t)(m0 + t) * a.N + col;
                if (ACT == TML_ACT_GELU_TANH && (long long)o + 4 > a.tail0) {  // the exact tanh of the flat tail
                    scalar_piece(t);
                    continue;
                }
                floatx4 out;
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    float v = alpha4[q] * v4[p][q];
                    if (a.beta != 0.0f) v += a.beta * cv[p][q];
                    if (a.bias) v += bias4[q];
                    if (a.res) v += rv[p][q];
                    out[q] = tml_apply_act(v, ACT, 0, 1);
                }
                tml_store_c(a.C + o, out);
            }
        }
    };
    using un4 = std::integral_constant<int, 4>;
    using un2 = std::integral_constant<int, 2>;
    if (!a.vec_epi) {
#pragma unroll 1
        for (int tr = tr0; tr < tr_end; tr += RPP) scalar_piece(tr);
    } else if (a.act == TML_ACT_GELU_ERF) {
        finish(std::integral_constant<int, TML_ACT_GELU_ERF>{}, un2{});
    } else if (a.act == TML_ACT_GELU_TANH) {
        finish(std::integral_constant<int, TML_ACT_GELU_TANH>{}, un2{});
    } else {
        finish(std::integral_constant<int, TML_ACT_NONE>{}, un4{});
    }
}

// Tile configs (index = TML_GEMM_SBF_TILE - 1) and the terms of pick_sbf's
// model: a launch with one tile a CU at most takes fixed + slices * (one +
// busy * the share of busy CUs past 0.4), a slice being bk deep.
struct SbfCfg {
    int bm, bn, bk;
    double fixed, one, busy;
    double f16, q8k, exact;  // the slice's cost in F16, Q8_K and exact int8 / int4, relative to f32 (0: not used)
};
constexpr SbfCfg kSbfCfgs[] = {
    {256, 128, 32, 9.7, 1.58, 1.25, 0.86, 0.0, 0.0},  // eight waves of 32 x 128
    {256, 96, 32, 8.9, 1.33, 0.95, 0.86, 1.05, 0.65},  // eight waves of 32 x 96
    {128, 64, 64, 8.2, 1.13, 0.37, 0.91, 1.09, 0.65},  // two wave groups of four 32 x 64
    {128, 64, 32, 6.4, 0.67, 0.13, 0.86, 1.12, 0.0},  // four waves of 32 x 64, two workgroups a CU
    {64, 64, 32, 5.1, 0.49, 0.03, 0.83, 1.22, 0.65},   // four waves of 16 x 64, three workgroups a CU
};
constexpr int kSbfNumCfgs = (int)(sizeof(kSbfCfgs) / sizeof(kSbfCfgs[0]));
// int8 / int4 run the first two only, with these terms
constexpr SbfCfg kSbfIntCfgs[] = {{256, 128, 32, 6.2, 0.93, 0.32, 0.0, 0.0, 0.0}, {256, 96, 32, 5.1, 0.83, 0.30, 0.0, 0.0, 0.0}};
constexpr int kSbfNumIntCfgs = (int)(sizeof(kSbfIntCfgs) / sizeof(kSbfIntCfgs[0]));
bool sbf_int(int fmt) { return fmt == TML_FMT_Q8_0 || fmt == TML_FMT_Q4_0; }
// Int8 / int4 outside gemm_qbf.hip's layouts (odd N, K % 8 != 0, an A on no 16-byte
// boundary), where the fp32 matrix cores' general kernel ran: at its precision.
bool sbf_exact(const MatmulArgs &m) { return sbf_int(m.fmt) && !gemm_qbf_supported(m); }
bool sbf_fast(const MatmulArgs &m) { return sbf_int(m.fmt) && gemm_qbf_supported(m); }
// A slice's cost in m's format, relative to f32; 0 where the tile has no kernel for it.
double sbf_cost(const MatmulArgs &m, const SbfCfg &t) {
    return m.fmt == TML_FMT_F16 ? t.f16 : m.fmt == TML_FMT_Q8_K ? t.q8k : sbf_exact(m) ? t.exact : 1.0;
}
bool sbf_cfg_ok(const MatmulArgs &m, int c) {
    if (sbf_fast(m)) return c >= 0 && c < kSbfNumIntCfgs;
    return c >= 0 && c < kSbfNumCfgs && sbf_cost(m, kSbfCfgs[c]) > 0.0;
}

template <int FMT>
void launch_sbf_cfg(int cfg, unsigned grid, const SbfArgs &a, hipStream_t s) {
    if constexpr (kSbfInt<FMT>) {
        // two slices of loads ahead; four measured the same
        if (cfg == 0) gemm_sbf_kernel<FMT, 256, 128, 32, 128, 32, 1, 8, 2><<<grid, 512, 0, s>>>(a);
        else gemm_sbf_kernel<FMT, 256, 96, 32, 96, 32, 1, 8, 2><<<grid, 512, 0, s>>>(a);
    } else if constexpr (FMT >= kSbfExact) {
        switch (cfg) {
            case 1: gemm_sbf_kernel<FMT, 256, 96, 32, 96, 32, 1, 8, 1><<<grid, 512, 0, s>>>(a); break;
            case 2: gemm_sbf_kernel<FMT, 128, 64, 32, 64, 64, 2, 8, 2><<<grid, 512, 0, s>>>(a); break;
            default: gemm_sbf_kernel<FMT, 64, 64, 16, 64, 32, 1, 4, 2><<<grid, 256, 0, s>>>(a); break;
        }
    } else {
        switch (cfg) {  // (the large tiles' registers hold one slice of loads ahead)
            case 0:  // (Q8_K: more registers than there are)
                if constexpr (FMT != TML_FMT_Q8_K)
                    gemm_sbf_kernel<FMT, 256, 128, 32, 128, 32, 1, 8, 1><<<grid, 512, 0, s>>>(a);
                break;
            case 1: gemm_sbf_kernel<FMT, 256, 96, 32, 96, 32, 1, 8, 1><<<grid, 512, 0, s>>>(a); break;
            case 2: gemm_sbf_kernel<FMT, 128, 64, 32, 64, 64, 2, 8, 2><<<grid, 512, 0, s>>>(a); break;
            case 3: gemm_sbf_kernel<FMT, 128, 64, 32, 64, 32, 1, 4, 2><<<grid, 256, 0, s>>>(a); break;
            default: gemm_sbf_kernel<FMT, 64, 64, 16, 64, 32, 1, 4, 2><<<grid, 256, 0, s>>>(a); break;
        }
    }
}

}  // namespace

bool gemm_sbf_supported(const MatmulArgs &m) {
    if (m.fmt == TML_FMT_Q4_0 && m.N % 2 != 0) return false;
    if (m.M <= kGemvMaxM || m.K <= 0) return false;
    // A's 16-byte loads need 4-byte alignment only, and a load that crosses the end
    // of A is checked dword by dword: any K serves.
    if (((uintptr_t)m.A % 4) != 0) return false;
    const uint64_t esz = m.fmt == TML_FMT_F32 ? 4 : m.fmt == TML_FMT_F16 ? 2 : 1;  // (int4: half, bounded as a byte)
    if ((uintptr_t)m.B % esz != 0) return false;
    if (m.fmt == TML_FMT_Q8_K && (m.block != 32 || m.N % 32 != 0 || ((uintptr_t)m.scales % 4) != 0)) return false;
    if (env_int("TML_GEMM_SBF", 1) == 0) return false;
    // every buffer offset below 2^31: A rows up to M + 256, B k-rows up to K + 512
    const uint64_t lim = (uint64_t)1 << 31;
    return (uint64_t)(m.M + 256) * (uint64_t)m.K * 4u < lim && (uint64_t)(m.K + 512) * (uint64_t)m.N * esz < lim &&
           m.M < ((int64_t)1 << 30) && m.N < ((int64_t)1 << 30);
}

// The tile of least modelled time, if that is below `other_us`, the modelled
// time of the other kernels' plan (0.95 of it for Q8_K; 1.1 for f32, int8 and int4,
// whose models run 5-20 % low at these sizes: f32 512x1024x4096 32.4 modelled, 42.8
// measured, Q8_0 1500x1280x5120 57.6 / 69-73).  The
// terms were fitted to a sweep of the five tiles on MI355X over
// M = 200-2048 and N, K = 384-5120 in the three formats (22 shapes; every launch
// reading one of 8 weight copies).  Measured, us, fp32 MFMA / this kernel's pick:
//   f32  1500x3840x1280 137 / 80 (256x96), 1500x5120x1280 165 / 95 (256x128),
//        1500x1280x5120 162 / 115 and 1500x1280x1280 51 / 33 (128x64x64),
//        512x4096x1024 40.0 / 29.5, 1024x3072x768 47.1 / 35.3 (64x64),
//        2048x768x3072 83 / 62; where it loses and stays unpicked: 512x1024x1024
//        13.4 / 21, 512x1536x384 9.5 / 11.0, 512x384x384 5.1 / 10.5, 256x3072x1024
//        18.5 / 21 (few tiles); unpicked though level by now: 1500x1536x384 20.4 - 21.2 /
//        19.7 (64x64);
//   F16  1500x3840x1280 140 / 69, 1500x1280x5120 169 / 105, 512x4096x1024 40.1 /
//        27.1, 1500x1536x384 19.7 / 17.8, 391x1536x384 11.2 / 9.8;
//   Q8_K 1500x3840x1280 159 / 82, 1500x1280x5120 185 / 127, 512x4096x1024 44.7 /
//        31.9, 1024x3072x768 50.2 / 39.7.
// 2-norm error against 64 bits, the same shapes: 3.7e-7 - 9.9e-7 / 0.9e-7 - 4.5e-7.
// int8 / int4 (other_us: the plan of gemm_qbf.hip), us: Q8_0 1500x3840x1280 54-58 /
// 45.3 (256x96), 1500x5120x1280 57-60 / 50.3, 1500x1280x5120 69-73 / 59.6 (256x128, K
// split 4); back to back 42.5 / 39.5, 49.2 / 45.4 and 61.5 / 52.0; where it stays unpicked: 1024x4096x1024 28.0 / 32.7, 1500x1280x1280 25.1 / 38.
//
// Layouts no other kernel has wide loads for (K % 4 != 0, odd N, A on a 4-byte
// boundary) always come here: the register-staged kernel reads them element by
// element and does not split K.  Measured, us, that kernel / this one: f32
// 9x4001x401 19.1 / 12.2, 60x401x399 20.6 / 15.3, 278x1340x2235 92 / 22.9,
// 1500x1537x383 45.9 / 30.3, 2500x3001x1999 501 / 186, 30x777x4999 188 / 30.3; F16
// 700x1111x1777 134 / 32.9, 20x3333x501 32.3 / 11.7; Q8_0 278x1341x2235 148 / 24.8,
// 20x3333x501 31.5 / 11.7, per-column 2000x2999x1500 325 / 102.  2-norm error against
// 64 bits 3.4e-7 - 1.3e-6 / 0.6e-7 - 2.8e-7.
//
// K is split s ways where the tiles leave CUs idle, at least eight slices a split;
// the reduce launch costs 2.5 us and the partials' traffic, s M N 8 bytes at 6
// TB/s (fp32 512x1024x4096, 128x64x64: 77.9 / 47.7 / 39.3 / 33.4 us at s = 1 - 4,
// the unsplit fp32-MFMA plan 42.8).  A split needs workspace that the other
// kernel's plan may not: int8 / int4 split at most as often as that plan does
// (other_split), f32, F16 and Q8_K within the allocation-free entry point's
// scratch, and not where the caller cannot grow the workspace (m.sbf_split), so a
// call keeps being served under stream capture and without allocation.
bool pick_sbf(const MatmulArgs &m, double other_us, int other_split, GemmPlan *p) {
    constexpr double kCus = 256.0;
    constexpr int kMaxSplit = 4;
    const bool is_int = sbf_fast(m);
    const double mn = (double)m.M * (double)m.N;
    double best = other_us * (m.fmt == TML_FMT_F32 || is_int ? 1.1 : m.fmt == TML_FMT_Q8_K ? 0.95 : 1.0);
    int cfg = -1, nsplit = 1;
    for (int c = 0; c < (is_int ? kSbfNumIntCfgs : kSbfNumCfgs); ++c) {
        const SbfCfg &t = is_int ? kSbfIntCfgs[c] : kSbfCfgs[c];
        const double rel = is_int ? 1.0 : sbf_cost(m, t);
        if (rel == 0.0) continue;
        const int64_t tiles = ((m.M + t.bm - 1) / t.bm) * ((m.N + t.bn - 1) / t.bn);
        const int64_t slices = (m.K + t.bk - 1) / t.bk;
        for (int s = 1; s <= kMaxSplit; ++s) {
            if (s > 1 && (tiles * s > 256 || slices / s < 8 || !m.sbf_split)) break;
            if (s > 1 && (is_int ? s > other_split : (double)s * mn > (double)kNoallocPartialFloats)) break;
            const double w = (double)(tiles * s) / kCus;  // tiles a CU
            const double busy = std::max(0.0, std::min(w, 1.0) - 0.4) * t.busy;
            double us = t.fixed, slice = t.one + busy;  // one tile a CU
            if (w > 1.0 && c < 3) {         // one workgroup a CU: whole rounds, each with its own fill and end
                us += 4.0 * (std::ceil(w) - 1.0);
                slice *= std::ceil(w);
            } else if (w > 1.0) {
                // two (config 3) or three (4) share a CU: whole rounds of that many, then the rest
                const double share = c == 3 ? 2.0 : 3.0, rest = w - share * std::floor(w / share);
                const double whole = std::floor(w / share) * (c == 3 ? 1.50 : 1.32);
                const double last = rest == 0.0 ? 0.0 : rest <= 1.0 ? t.one : c == 3 ? 1.25 + 0.2 * (rest - 1.0)
                                    : rest <= 2.0 ? 0.72 + 0.14 * (rest - 1.0) : 1.17 + 0.09 * (rest - 2.0);
                slice = whole + last;
            }
            us += slice * rel * (double)((slices + s - 1) / s);
            if (s > 1) us += 2.5 + (double)s * mn * 8.0 / 6.0e6;
            if (us < best) {
                best = us;
                cfg = c;
                nsplit = s;
            }
        }
    }
    const int forced = env_int("TML_GEMM_SBF_TILE", 0) - 1;
    if (sbf_cfg_ok(m, forced)) {
        cfg = forced;
        nsplit = m.sbf_split ? std::min(std::max(env_int("TML_GEMM_SBF_SPLIT", 1), 1), kMaxSplit) : 1;
    }
    if (cfg < 0) return false;
    const int64_t bk = kSbfCfgs[cfg].bk, slices = (m.K + bk - 1) / bk;
    p->spl = (int)((slices + nsplit - 1) / nsplit * bk);
    p->cfg = cfg;
    p->nsplit = (int)((m.K + p->spl - 1) / p->spl);
    p->tiles = (int)(((m.M + kSbfCfgs[cfg].bm - 1) / kSbfCfgs[cfg].bm) * ((m.N + kSbfCfgs[cfg].bn - 1) / kSbfCfgs[cfg].bn));
    return true;
}

Status launch_gemm_sbf(const MatmulArgs &m, const GemmPlan &p, const Workspace &ws, hipStream_t s) {
    if (!gemm_sbf_supported(m) || !sbf_cfg_ok(m, p.cfg))
        return Status::Err(TML_ERR_INVALID_ARG, "split-bf16 GEMM: operands or tile config not supported");
    SbfArgs a;
    a.M = (int)m.M; a.N = (int)m.N; a.K = (int)m.K;
    a.A = m.A; a.B = (const uint8_t *)m.B; a.scales = m.scales;
    a.ldb = (int)(m.fmt == TML_FMT_Q4_0 ? m.N / 2 : m.N * (m.fmt == TML_FMT_F32 ? 4 : m.fmt == TML_FMT_F16 ? 2 : 1));
    a.colscale = m.colscale;
    a.bias = m.bias; a.res = m.res; a.C = m.C;
    a.alpha = m.alpha_eff; a.beta = m.beta;
    a.act = m.act;
    a.tail0 = tml_act_tail0((long long)m.M * m.N);
    a.a_bytes = (unsigned)((uint64_t)m.M * (uint64_t)m.K * 4u);
    a.s_bytes = m.fmt == TML_FMT_Q8_K ? (unsigned)((uint64_t)m.K * (uint64_t)m.N / 32u * 4u) : 0u;
    a.tiles_m = (int)((m.M + kSbfCfgs[p.cfg].bm - 1) / kSbfCfgs[p.cfg].bm);
    a.tiles_n = (int)((m.N + kSbfCfgs[p.cfg].bn - 1) / kSbfCfgs[p.cfg].bn);
    a.vec_epi = m.N % 4 == 0 && ((uintptr_t)m.C % 16) == 0 && (m.bias == nullptr || ((uintptr_t)m.bias % 16) == 0) &&
                (m.res == nullptr || ((uintptr_t)m.res % 16) == 0) &&
                (m.colscale == nullptr || ((uintptr_t)m.colscale % 16) == 0);
    if (p.nsplit < 1 || p.spl < 1 || p.spl % kSbfCfgs[p.cfg].bk != 0 || (int64_t)p.spl * p.nsplit < m.K ||
        (int64_t)p.spl * (p.nsplit - 1) >= m.K)
        return Status::Err(TML_ERR_INVALID_ARG, "split-bf16 GEMM: split plan does not cover K");
    if (p.nsplit > 1 && (ws.partials == nullptr || ws.partial_floats < (size_t)p.nsplit * (size_t)m.M * (size_t)m.N))
        return Status::Err(TML_ERR_INVALID_ARG, "split-bf16 GEMM: split-K workspace too small");
    a.nsplit = p.nsplit;
    a.spl = p.spl;
    a.ws = p.nsplit > 1 ? ws.partials : nullptr;
    const int64_t grid = (int64_t)a.tiles_m * a.tiles_n * p.nsplit;
    if (grid >= ((int64_t)1 << 31)) return Status::Err(TML_ERR_INVALID_SHAPE, "split-bf16 GEMM: grid too large");
    switch (m.fmt) {
        case TML_FMT_F32: launch_sbf_cfg<TML_FMT_F32>(p.cfg, (unsigned)grid, a, s); break;
        case TML_FMT_F16: launch_sbf_cfg<TML_FMT_F16>(p.cfg, (unsigned)grid, a, s); break;
        case TML_FMT_Q8_K: launch_sbf_cfg<TML_FMT_Q8_K>(p.cfg, (unsigned)grid, a, s); break;
        case TML_FMT_Q8_0:
            if (sbf_exact(m)) launch_sbf_cfg<TML_FMT_Q8_0 + kSbfExact>(p.cfg, (unsigned)grid, a, s);
            else launch_sbf_cfg<TML_FMT_Q8_0>(p.cfg, (unsigned)grid, a, s);
            break;
        case TML_FMT_Q4_0:
            if (sbf_exact(m)) launch_sbf_cfg<TML_FMT_Q4_0 + kSbfExact>(p.cfg, (unsigned)grid, a, s);
            else launch_sbf_cfg<TML_FMT_Q4_0>(p.cfg, (unsigned)grid, a, s);
            break;
        default: return Status::Err(TML_ERR_INVALID_FORMAT, "unknown weight format");
    }
    TML_HIP_TRY(hipGetLastError());
    if (p.nsplit > 1) TML_TRY(launch_splitk_reduce(ws.partials, p.nsplit, m, s));
    return Status::Ok();
}

}  // namespace tml
