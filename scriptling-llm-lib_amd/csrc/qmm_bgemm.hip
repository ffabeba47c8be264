// Prefill GEMM of the formats whose activations stay fp32 (Q5_0, Q2_K, Q3_K)
// on the bf16 matrix cores, with exact products.
//
// The reference multiplies these weights with float32 activations: Q5_0 sums
// v_j x_j over a 32-element block (v = q5 - 16, float32_ops.go:335-367, :427-436)
// and scales the sum by d; Q2_K / Q3_K rebuild dense float32 weights
// (kquants.go:147-245) and multiply those (float32_ops.go:462-482). In every
// format a weight is scale * small integer (- min) over 16 or 32 elements, and
// the integer is exact in bf16, so
// * split_frag_kernel splits each activation exactly into three bf16 parts, x =
//   hi + mid + lo (hi the top 8 significand bits, mid the next 8 of the
//   remainder, lo the rest, at most 8 bits), in the order the MFMA's A operand
//   wants: 1 KB per (32 rows, 16 elements, part), lane l's 16 bytes at 16 l;
// * v_mfma_f32_32x32x16_bf16 over the three parts forms every product exactly
//   and sums a 16- or 32-element group in fp32;
// * the epilogue adds scale * sum with one fused multiply-add.
// * a Q2_K weight dl q - ml is taken as dl (q - b) + w_b, b the code whose weight w_b
//   = dl b - ml is nearest zero (rounded once: the reference's float32): the two
//   terms are never more than three times the weight, so where dl q and ml nearly
//   cancel nothing is lost, and a weight of 0 gives 0. The second term, w_b * (sum
//   of the group's x), goes through v_mfma_f32_32x32x2_f32 into the same accumulator
//   (the group sums are formed in fp64 and rounded once).
// Against the reference's per-element order this is reassociation and fewer
// roundings; measured against 64 bits the error is no larger than the GEMV's
// (gemm_kquant tests).
//
// What bounds it: from about 100 rows the matrix cores with what runs beside them (192
// cycles per 32 x 32 tile and 32 elements, three part products: busy 36 % of the 51.5 us
// of Q5_0 14336x4096 at M = 100, VALU 33 %, both at once 11 %); below, neither (Q3_K 14336x4096
// at M = 64, 46 us: matrix cores 19 %, VALU 32 %): the waves decode, write LDS (conflicts in
// 64-row tiles as many cycles as accesses) and wait at a barrier every two blocks. A wave
// owns 32 rows x 32 CT columns; its activation fragments go from L2 straight to registers
// (they are stored in lane order, so each load is 1 KB contiguous), one block ahead;
// only the decoded weights pass through LDS, in MFMA order, KB blocks per stage,
// double-buffered, decoded once per workgroup of 32 WM rows.
#include <hip/hip_runtime.h>

#include "qmm_device.hpp"
#include "qmm_internal.hpp"

namespace sllm {

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));

// Activations outside this range (or not finite) take the per-element path in
// Q2_K / Q3_K: there scale * sum could overflow, or the low parts underflow,
// where the reference's x * w does not.
constexpr float kBigX = 0x1p96f, kTinyX = 0x1p-90f;

// Scales per 32-element block and column: Q5_0 one, the k-quants one per
// 16-element sub-block.
__host__ __device__ constexpr int groups_of(int fmt) { return fmt == SLLM_Q5_0 ? 1 : 2; }

// The order of a 16-element group inside the MFMA's K: both operands use the
// same one, so it is free. k-quants: position p holds element p / 4 + 4 (p %
// 4), the order in which a word of 2-bit codes gives bytes.
template <int FMT>
__device__ __forceinline__ constexpr int elem_at(int p) {
    return kq_native(FMT) ? (p >> 2) + 4 * (p & 3) : p;
}

__device__ __forceinline__ void split3(float f, uint32_t &hi, uint32_t &mid, uint32_t &lo) {
    const uint32_t ub = __float_as_uint(f);
    hi = ub >> 16;
    if ((ub & 0x7f800000u) == 0x7f800000u) {  // Inf / NaN: the value itself, no remainder
        mid = lo = 0;
        // a NaN whose payload lies in the low half stays a NaN
        if ((ub & 0x007fffffu) && !(hi & 0x7fu)) hi |= 1u;
        return;
    }
    const float r1 = f - __uint_as_float(ub & 0xffff0000u);  // exact
    const uint32_t um = __float_as_uint(r1) & 0xffff0000u;
    const float r2 = r1 - __uint_as_float(um);  // exact, and a bf16
    mid = um >> 16;
    lo = __float_as_uint(r2) >> 16;
}

// x [M][K] fp32 -> fragments [rt][g][ks][part][lane][8] bf16, one wave per (32
// rows, block). Q2_K: also xsum [rt][g][lane], the sums of sub-block ks = lane
// / 32 of row lane % 32. k-quants: flag [rt][g] = 1 where a value needs the
// per-element path. Rows past M and blocks past G (up to Gp) are zeros.
template <int FMT>
__global__ void __launch_bounds__(256) split_frag_kernel(const float *__restrict__ x, int M, int G, int Gp, int nfrag,
                                                         uint16_t *__restrict__ frag, float *__restrict__ xsum,
                                                         uint8_t *__restrict__ flag) {
    const int w = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (w >= nfrag) return;
    const int lane = threadIdx.x & 63, r = lane & 31, h = lane >> 5;
    const int rt = w / Gp, g = w - rt * Gp;
    const int row = rt * 32 + r;
    const bool live = row < M && g < G;
    const float4 *src = (const float4 *)(x + ((size_t)min(row, M - 1) * G + min(g, G - 1)) * 32);
    float amax = 0.0f;
    bool bad = false;
    float sum[2];
#pragma unroll
    for (int ks = 0; ks < 2; ks++) {
        float v[8];
        if (kq_native(FMT)) {
            // positions 8 h .. 8 h + 7: elements 2 h + 4 k (k = 0..3), then 2 h + 1 + 4 k
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const float4 u = src[4 * ks + k];
                v[k] = h ? u.z : u.x;
                v[4 + k] = h ? u.w : u.y;
            }
        } else {
            const float4 u0 = src[4 * ks + 2 * h], u1 = src[4 * ks + 2 * h + 1];
            v[0] = u0.x; v[1] = u0.y; v[2] = u0.z; v[3] = u0.w;
            v[4] = u1.x; v[5] = u1.y; v[6] = u1.z; v[7] = u1.w;
        }
        uint32_t o[3][4];
        double s = 0.0;
#pragma unroll
        for (int k = 0; k < 8; k += 2) {
            uint32_t p[2][3];
#pragma unroll
            for (int e = 0; e < 2; e++) {
                const float f = live ? v[k + e] : 0.0f;
                split3(f, p[e][0], p[e][1], p[e][2]);
                if (kq_native(FMT)) {
                    const float a = __builtin_fabsf(f);
                    bad |= !(a < kBigX);
                    amax = a > amax ? a : amax;
                    if (FMT == SLLM_Q2K) s += (double)f;
                }
            }
#pragma unroll
            for (int part = 0; part < 3; part++) o[part][k >> 1] = p[0][part] | (p[1][part] << 16);
        }
        if (FMT == SLLM_Q2K) sum[ks] = (float)(s + __shfl_xor(s, 32, 64));
        uint16_t *dst = frag + ((size_t)w * 6 + ks * 3) * 512 + lane * 8;
#pragma unroll
        for (int part = 0; part < 3; part++)
            *(uint4 *)(dst + part * 512) = make_uint4(o[part][0], o[part][1], o[part][2], o[part][3]);
    }
    if (FMT == SLLM_Q2K) xsum[(size_t)w * 64 + lane] = h ? sum[1] : sum[0];
    if (kq_native(FMT)) {
        const float o = __shfl_xor(amax, 32, 64);
        amax = o > amax ? o : amax;
        bad |= amax > 0.0f && amax < kTinyX;
        const unsigned long long any = __ballot(bad);
        if (lane == 0) flag[w] = any ? 1 : 0;
    }
}

// A thread's share of one stage's weights: units (column, block).
template <int FMT>
struct WUnit {
    v4i qs;       // Q5_0: the nibble bytes
    uint2 q2;     // k-quants: the 2-bit codes
    uint32_t qh;  // Q5_0, Q3K: high bits
    uint32_t sb;  // k-quants: the super-block's scale word
    uint16_t d;
};

template <int FMT>
__device__ __forceinline__ void load_unit(WUnit<FMT> &u, const Planes &P, size_t idx) {
    if (FMT == SLLM_Q5_0) {
        u.qs = *(const v4i *)(P.qs + idx);
        u.qh = P.qh[idx];
    } else {
        u.q2 = P.q2[idx];
        u.sb = P.sb[idx >> 3];
        if (FMT == SLLM_Q3K) u.qh = P.qh[idx];
    }
    u.d = P.d[idx];
}

// Two floats' top halves: bf16 pair (values exact in bf16).
__device__ __forceinline__ uint32_t pack_bf(float a, float b) {
    return __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302u);
}

// The two 16-byte pieces (h = 0, 1) of group ks of a block's codes as bf16;
// neg 0x80: negated (0: not). The matrix cores' bf16 sums round down by a part
// of an ulp, which adds up over a row where every scale is positive: odd blocks
// go in with codes and scale negated, so that the two halves' drifts cancel
// (Q2_K over 4096 / 14336 columns 1.9e-7 / 2.9e-7 from the 64-bit result
// without, Q5_0 1.24e-7 / 1.8e-7).
// base: Q2_K's b (codes q - b).
template <int FMT>
__device__ __forceinline__ void decode_half(const WUnit<FMT> &u, int ks, uint32_t neg, uint32_t base, uint4 (&p)[2]) {
    if constexpr (FMT == SLLM_Q5_0) {
        const uint32_t w[4] = {(uint32_t)u.qs.x, (uint32_t)u.qs.y, (uint32_t)u.qs.z, (uint32_t)u.qs.w};
#pragma unroll
        for (int h = 0; h < 2; h++) {
            uint32_t o[4];
#pragma unroll
            for (int q = 0; q < 2; q++) {
                // four signed codes q5 - 16 as bytes (elements 16 ks + 8 h + 4 q ..)
                const int j = 2 * h + q;
                const uint32_t c = q5_codes(ks ? w[j] >> 4 : w[j], ~u.qh >> (16 * ks + 4 * j));
                float f[4];
#pragma unroll
                for (int k = 0; k < 4; k++) f[k] = (float)(int)(int8_t)((c >> (8 * k)) & 0xffu);
                o[2 * q] = pack_bf(f[0], f[1]) ^ neg * 0x01000100u;
                o[2 * q + 1] = pack_bf(f[2], f[3]) ^ neg * 0x01000100u;
            }
            p[h] = make_uint4(o[0], o[1], o[2], o[3]);
        }
    } else {
        // bf16 high and low bytes of the values -4 .. 3 at index 0 .. 7 (Q3K: code + 4 *
        // high bit; Q2K: code + 4 - b), looked up four at a time with v_perm
        constexpr uint32_t lo0 = 0x80004080u, lo1 = 0x40008000u;
        const uint32_t sgn = neg * 0x01010101u;
        const uint32_t hi0 = 0xBFC0C0C0u ^ sgn, hi1 = 0x40403F00u ^ sgn;
        const uint32_t shift = FMT == SLLM_Q2K ? (4u - base) * 0x01010101u : 0u;
        const uint32_t w = ks ? u.q2.y : u.q2.x;
        uint32_t o[8];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            uint32_t sel = (w >> (2 * j)) & 0x03030303u;  // elements j, j + 4, j + 8, j + 12
            if (FMT == SLLM_Q3K) {
                uint32_t t = (u.qh >> (16 * ks + j)) & 0x1111u;    // bits 0, 4, 8, 12
                t = (t & 0x0011u) | ((t & 0x1100u) << 8);          // bits 0, 4, 16, 20
                t = (t & 0x00010001u) | ((t & 0x00100010u) << 4);  // bits 0, 8, 16, 24
                sel |= t << 2;
            } else {
                sel += shift;
            }
            const uint32_t l = __builtin_amdgcn_perm(lo1, lo0, sel), hh = __builtin_amdgcn_perm(hi1, hi0, sel);
            o[2 * j] = __builtin_amdgcn_perm(hh, l, 0x05010400u);
            o[2 * j + 1] = __builtin_amdgcn_perm(hh, l, 0x07030602u);
        }
        p[0] = make_uint4(o[0], o[1], o[2], o[3]);
        p[1] = make_uint4(o[4], o[5], o[6], o[7]);
    }
}

// Scale (and Q2K min) of sub-block i of a unit: a weight is scale * code - min.
template <int FMT>
__device__ __forceinline__ void unit_scale(const WUnit<FMT> &u, int i, float &sc, float &mn) {
    mn = 0.0f;
    if (FMT == SLLM_Q5_0) {
        sc = f16_lut(u.d);
    } else if (FMT == SLLM_Q2K) {
        const uint32_t b = ((uint32_t)u.d >> (8 * i)) & 0xffu;
        sc = f16_exact((uint16_t)(u.sb & 0xffffu)) * (float)(b & 0xfu);
        mn = f16_exact((uint16_t)(u.sb >> 16)) * (float)(b >> 4);
    } else {
        sc = f16_exact((uint16_t)(u.sb & 0xffffu)) * (float)(int)(int8_t)(((uint32_t)u.d >> (8 * i)) & 0xffu);
    }
}

// Q2_K: the code whose weight is nearest zero, ml / dl rounded to 0 .. 3 (at dl = 0
// any: the codes do not matter).
__device__ __forceinline__ uint32_t q2k_base(float sc, float mn) {
    const float s = __builtin_fabsf(sc), t = sc < 0.0f ? -mn : mn;
    return (t > 0.5f * s) + (t > 1.5f * s) + (t > 2.5f * s);
}

// One LDS stage: KB blocks of BN columns. b: [blk][column tile][ks][lane][16
// bytes], a block's region padded by 32 bytes so that the four lanes that
// decode the blocks of one column write distinct banks.
template <int FMT, int KB, int BN>
struct alignas(16) BStage {
    static constexpr int BLK = BN * 64 + 32;  // bytes of one block's fragments
    static constexpr int NG = groups_of(FMT);
    unsigned char b[KB * BLK];
    float sc[KB * NG][BN];
    float mn[FMT == SLLM_Q2K ? KB * NG : 1][BN];
};

// The per-element path of one block for the k-quants (flagged activations):
// every weight rebuilt as the reference's float32, one product and one add per
// element, in element order.
template <int FMT, int CT>
__device__ __forceinline__ void slow_block(const Planes &P, const float *__restrict__ x, int M, int N, int G, int g,
                                           int mrow0, int ncol0, int lane, v16f (&acc)[CT]) {
    const int r32 = lane & 31, h = lane >> 5;
    const float *xr = x + ((size_t)min(mrow0 + r32, M - 1) * G + g) * 32;  // this lane's row, handed round below
#pragma unroll
    for (int j = 0; j < CT; j++) {
        const int n = min(ncol0 + 32 * j + r32, N - 1);
        WUnit<FMT> u;
        load_unit<FMT>(u, P, (size_t)n * G + g);
#pragma unroll 1
        for (int e = 0; e < 32; e++) {
            const int ks = e >> 4;
            float sc, mn;
            unit_scale<FMT>(u, ks, sc, mn);
            int q = (int)(((ks ? u.q2.y : u.q2.x) >> (2 * (e & 15))) & 3u);
            if (FMT == SLLM_Q3K) q += ((u.qh >> e) & 1u) ? 0 : -4;
            const float w = FMT == SLLM_Q2K ? __builtin_fmaf(sc, (float)q, -mn) : sc * (float)q;
            const float xv = xr[e];
#pragma unroll
            for (int v = 0; v < 16; v++) {
                const float xm = __shfl(xv, 8 * (v >> 2) + 4 * h + (v & 3), 64);
                acc[j][v] = acc[j][v] + xm * w;
            }
        }
    }
}

// Blocks whose terms are added one by one before they join the total (0: one
// chain over the whole range). One chain rounds at the total's size at every
// group: relative error against 64 bits over K = 4096 / 14336, Q3_K in one chain
// 2.9e-7 / 5.3e-7, in runs 0.98e-7 / 1.04e-7, the GEMV 1.25e-7 / 1.33e-7. Q5_0
// on 128-row tiles keeps one chain: its runs spill (14336x4096 at M = 512 180
// -> 358 us).
constexpr int run_of(int fmt, int ct) { return fmt == SLLM_Q5_0 ? (ct == 4 ? 0 : 16) : 8; }

// Workgroup = WM x WN waves, tile (32 WM) x (32 CT WN); stages [sp * sps, ...)
// of KB blocks. RA: blocks of activation fragments held in registers (RA - 1
// of them in flight); WA: stages of weights in flight. Gp: G rounded up to a
// multiple of 4, the blocks the fragments are laid out for (zeros past G).
template <int FMT, int WM, int WN, int CT, int KB, int RA, int WA, bool ADD>
__global__ void __launch_bounds__(64 * WM * WN) __attribute__((amdgpu_waves_per_eu(2)))
bgemm_kernel(Planes P, const uint16_t *__restrict__ frag, const float *__restrict__ xsum,
             const uint8_t *__restrict__ flag, const float *__restrict__ x, float *__restrict__ out, int M, int N,
             int G, int mtiles, int ntiles, int splits, int sps) {
    constexpr int BN = 32 * CT * WN, T = 64 * WM * WN;
    constexpr int UNITS = BN * KB, PER = UNITS / T;
    constexpr int HPB = PER * 2 / KB;  // half units decoded beside each block
    constexpr int RUN = run_of(FMT, CT);
    constexpr int SU = RA / KB > WA ? RA / KB : WA;  // stages per loop iteration: ring indices are constants
    static_assert(UNITS % T == 0 && PER * 2 % KB == 0, "every thread decodes as much beside every block");
    static_assert((SU * KB) % RA == 0 && SU % WA == 0, "rings close over an iteration");
    using St = BStage<FMT, KB, BN>;
    extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
    St *st = (St *)lds_raw;

    // XCD-aware order: the M-tiles of one weight tile and split run on one XCD,
    // so the weight tile is read from HBM once into its L2
    const int total = mtiles * ntiles * splits;
    const int per_xcd = (total + 7) / 8;
    const int lin = (blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
    if (lin >= total) return;
    const int mt = lin % mtiles;
    const int rest = lin / mtiles;
    const int sp = rest % splits, nt = rest / splits;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave % WM, wn = wave / WM;
    const int n0 = nt * BN;
    const int Gp = (G + 3) & ~3;
    const int nst = Gp / KB;
    const int st0 = sp * sps, st1 = min(nst, st0 + sps);
    const int RT = (M + 31) / 32;
    const int rt = mt * WM + wm;
    const int rtc = min(rt, RT - 1);  // a wave past the rows repeats the last ones and stores nothing
    const int g_end = st1 * KB;

    // tot: the sums of whole runs; acc: the current run
    v16f acc[CT], tot[RUN ? CT : 1];
#pragma unroll
    for (int j = 0; j < CT; j++)
#pragma unroll
        for (int v = 0; v < 16; v++) {
            acc[j][v] = 0.0f;
            if (RUN) tot[RUN ? j : 0][v] = 0.0f;
        }
    auto close_run = [&]() {
#pragma unroll
        for (int j = 0; j < CT; j++)
#pragma unroll
            for (int v = 0; v < 16; v++) {
                tot[RUN ? j : 0][v] = tot[RUN ? j : 0][v] + acc[j][v];
                acc[j][v] = 0.0f;
            }
    };

    // does any block of these rows need the per-element path? (k-quants)
    bool slow = false;
    if (kq_native(FMT)) {
        bool f = false;
        for (int g = st0 * KB + lane; g < g_end; g += 64) f |= flag[(size_t)rtc * Gp + g] != 0;
        slow = __ballot(f) != 0;
        if (lane == 0) lds_raw[wave] = slow;
        __syncthreads();
        slow = false;
#pragma unroll
        for (int w = 0; w < WM * WN; w++) slow |= lds_raw[w] != 0;
        __syncthreads();
    }
    if (slow) {
        for (int g = st0 * KB; g < g_end; g++)
            slow_block<FMT, CT>(P, x, M, N, G, g, rtc * 32, n0 + wn * 32 * CT, lane, acc);
    } else {
        WUnit<FMT> wu[WA][PER];
        auto fetch = [&](WUnit<FMT> (&u)[PER], int s) {
#pragma unroll
            for (int i = 0; i < PER; i++) {
                const int e = threadIdx.x + T * i;
                const int n = min(n0 + e / KB, N - 1), g = min(min(s, st1 - 1) * KB + e % KB, G - 1);
                load_unit<FMT>(u[i], P, (size_t)n * G + g);
            }
        };
        // half unit hu (unit hu / 2, group hu % 2) of stage s into LDS
        auto store = [&](St &S, const WUnit<FMT> (&u)[PER], int hu, int s) {
            const int i = hu >> 1, ks = hu & 1;
            const int e = threadIdx.x + T * i;
            const int c = e / KB, blk = e % KB;
            uint4 p[2];
            const uint32_t neg = blk & 1 ? 0x80u : 0u;  // odd blocks negated, codes and scale
            float sc, mn;
            unit_scale<FMT>(u[i], ks, sc, mn);
            const uint32_t base = FMT == SLLM_Q2K ? q2k_base(sc, mn) : 0u;
            decode_half<FMT>(u[i], ks, neg, base, p);
            unsigned char *b = S.b + blk * St::BLK + (c >> 5) * 2048 + (c & 31) * 16 + ks * 1024;
            *(uint4 *)b = p[0];
            *(uint4 *)(b + 512) = p[1];
            if (kq_native(FMT) || ks == 0) {
                const float wb = __builtin_fmaf(sc, (float)base, -mn);
                sc = __uint_as_float(__float_as_uint(sc) ^ neg << 24);
                // blocks past the row's end repeat its last one with scale 0 (their activations are zeros)
                S.sc[blk * St::NG + (kq_native(FMT) ? ks : 0)][c] = kq_native(FMT) || s * KB + blk < G ? sc : 0.0f;
                if (FMT == SLLM_Q2K) S.mn[FMT == SLLM_Q2K ? blk * St::NG + ks : 0][c] = wb;
            }
        };
        // activation fragments of a block: [ks][part]
        v4i a[RA][2][3];
        float xs[RA];
        const uint16_t *fb = frag + (size_t)rtc * Gp * 3072 + lane * 8;
        const float *xb = xsum + (size_t)rtc * Gp * 64 + lane;
        auto load_a = [&](int r, int g) {
            g = min(g, g_end - 1);
#pragma unroll
            for (int ks = 0; ks < 2; ks++)
#pragma unroll
                for (int part = 0; part < 3; part++)
                    a[r][ks][part] = *(const v4i *)(fb + (size_t)g * 3072 + (ks * 3 + part) * 512);
            if (FMT == SLLM_Q2K) xs[r] = xb[(size_t)g * 64];
        };
        auto block = [&](const St &S, int blk, int r) {
            const unsigned char *b = S.b + blk * St::BLK + wn * CT * 2048 + lane * 16;
            const int c0 = wn * 32 * CT + (lane & 31);
#pragma unroll
            for (int j = 0; j < CT; j++) {
                v16f sum = {};
#pragma unroll
                for (int ks = 0; ks < 2; ks++) {
                    const v8bf bf = __builtin_bit_cast(v8bf, *(const v4i *)(b + j * 2048 + ks * 1024));
                    if (kq_native(FMT)) sum = v16f{};
#pragma unroll
                    for (int part = 2; part >= 0; part--)  // the small parts first
                        sum = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf, a[r][ks][part]), bf, sum,
                                                                      0, 0, 0);
                    if (kq_native(FMT) || ks == 1) {
                        const float sc = S.sc[blk * St::NG + (kq_native(FMT) ? ks : 0)][c0 + 32 * j];
#pragma unroll
                        for (int v = 0; v < 16; v++) acc[j][v] = __builtin_fmaf(sc, sum[v], acc[j][v]);
                    }
                }
                if (FMT == SLLM_Q2K) {
                    // w_b * (group sum) of both sub-blocks: k slot = lane / 32
                    const float mn = S.mn[FMT == SLLM_Q2K ? blk * St::NG + (lane >> 5) : 0][c0 + 32 * j];
                    acc[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(xs[r], mn, acc[j], 0, 0, 0);
                }
            }
        };

        fetch(wu[0], st0);
#pragma unroll
        for (int r = 0; r < RA - 1; r++) load_a(r, st0 * KB + r);
        if (WA > 1) fetch(wu[WA - 1], st0 + 1);
#pragma unroll
        for (int hu = 0; hu < 2 * PER; hu++) store(st[0], wu[0], hu, st0);
        __syncthreads();
        for (int s0 = st0; s0 < st1; s0 += SU) {
#pragma unroll
            for (int u = 0; u < SU; u++) {
                const int s = s0 + u;
                if (SU > 1 && s >= st1) break;
                const St &S = st[(s - st0) & 1];
                St &Sn = st[(s + 1 - st0) & 1];
                // the registers of stage s (already in LDS) take stage s + WA
                fetch(wu[u % WA], s + WA);
#pragma unroll
                for (int blk = 0; blk < KB; blk++) {
                    const int gi = u * KB + blk;  // block within the iteration
                    load_a((gi + RA - 1) % RA, s * KB + blk + RA - 1);
                    block(S, blk, gi % RA);
                    // stage s + 1 decoded beside the products (past the last stage: never read)
#pragma unroll
                    for (int k = 0; k < HPB; k++) store(Sn, wu[(u + 1) % WA], blk * HPB + k, s + 1);
                }
                __syncthreads();
                if (RUN && (s + 1 - st0) % ((RUN ? RUN : KB) / KB) == 0) close_run();
            }
        }
    }

    if (RUN) close_run();
    if (rt >= RT) return;
    const int r32 = lane & 31, h = lane >> 5;
    float *o = out + (size_t)sp * M * N;  // splits > 1: partial tile of split sp
#pragma unroll
    for (int j = 0; j < CT; j++) {
        const int n = n0 + wn * 32 * CT + 32 * j + r32;
#pragma unroll
        for (int v = 0; v < 16; v++) {
            const int m = rt * 32 + 8 * (v >> 2) + 4 * h + (v & 3);
            if (m < M && n < N) {
                float &d = o[(size_t)m * N + n];
                const float r = RUN ? tot[RUN ? j : 0][v] : acc[j][v];
                d = ADD ? d + r : r;  // ADD: the residual add, one float32 add
            }
        }
    }
}

// Workgroup shapes, rows x columns: 32 x 256, 64 x 128 (both four waves, two workgroups
// per CU), 128 x 256 (eight waves).
enum BShape { kRows32 = 0, kRows64 = 1, kRows128 = 2 };

struct BPlan {
    int shape, wm, bn, kb, mtiles, ntiles, splits, sps;
};

// Blocks per stage of the 128-row shape
constexpr int kKb128(int fmt) { return fmt == SLLM_Q5_0 ? 4 : 2; }

BPlan plan(int fmt, int M, int N, int G) {
    BPlan p{};
    const int RT = (M + 31) / 32;
    const int64_t w = (int64_t)N * G * 32;
    // 32 x 256 up to 32 rows of a weight of 2^25 elements; 128 x 256 above 64 rows of
    // 1.5e9 products (the k-quants: 3e9, and a last row tile at least three quarters
    // full or the only one); else 64 x 128, whose many small workgroups fill the device
    // from a small weight. Best time over the K splits (us, 32 x 256 / 64 x 128 / 128 x
    // 256): Q5_0 1024x4096 at M = 32 17.9 / 16.1, M = 100 - / 21.1 / 26.5; 4096x4096 M =
    // 32 23.9 / 22.0, M = 100 - / 31.4 / 29.5; 14336x4096 M = 32 38.3 / 41.8, M = 96 - /
    // 70.5 / 57.4, M = 512 - / 254 / 171; Q3_K 4096x4096 M = 128 - / 35.5 / 35.4, 8192x4096
    // M = 160 - / 69.7 / 72.9, M = 256 - / 85.9 / 76.0. (64 x 256, one workgroup per CU:
    // Q5_0 1024x4096 at M = 64 20.5 against 18.8, 14336x4096 47.2 against 44.8.)
    const bool kq = kq_native(fmt);
    const bool wide = RT > 2 && w * M >= (kq ? (int64_t)3000000000 : 1500000000) &&
                      (!kq || RT <= 4 || (RT + 3) / 4 * 80 <= RT * 23);
    p.shape = RT == 1 && w >= ((int64_t)1 << 25) ? kRows32 : (wide ? kRows128 : kRows64);
    if (tuning().gemm_shape >= 1 && tuning().gemm_shape <= 3) p.shape = tuning().gemm_shape - 1;
    p.wm = p.shape == kRows32 ? 1 : (p.shape == kRows64 ? 2 : 4);
    p.bn = p.shape == kRows64 ? 128 : 256;
    p.kb = p.shape == kRows128 ? kKb128(fmt) : 2;
    p.mtiles = (RT + p.wm - 1) / p.wm;
    p.ntiles = (N + p.bn - 1) / p.bn;
    const int nst = ((G + 3) & ~3) / p.kb;
    // K splits: the count of least cost, in blocks of K that a workgroup alone on its CU
    // takes the time of: its blocks, times co for each workgroup where the CU has
    // several, and a fixed part for each; then the reduction's megabytes. Fitted to 477
    // (format, weight, rows), every split count timed: shape and count together are 1.2 %
    // above the best on average.
    static constexpr struct { double co, fix, mb; } kCost[4] = {{0.7, 0.5, 1}, {0.65, 2, 1}, {1, 8, 0.1}, {0.7, 8, 0.1}};
    const auto &c = kCost[kq && p.shape == kRows32 ? 3 : p.shape];
    int best = 1;
    double bc = 1e30;
    for (int S = 1; S <= 32 && S <= nst; S++) {
        const int sps = (nst + S - 1) / S;
        if ((nst + sps - 1) / sps != S) continue;
        const int64_t n = ((int64_t)p.mtiles * p.ntiles * S + 255) / 256;
        double t = sps * p.kb * (n == 1 ? 1.0 : c.co * n) + c.fix * n;
        if (S > 1) t += c.mb * S * M * (double)N * 4e-6;
        if (t < bc) {
            bc = t;
            best = S;
        }
    }
    if (tuning().gemm_splits) best = tuning().gemm_splits < nst ? tuning().gemm_splits : nst;
    p.sps = (nst + best - 1) / best;
    p.splits = (nst + p.sps - 1) / p.sps;
    return p;
}

size_t align256(size_t v) { return (v + 255) & ~(size_t)255; }

// Workspace: fragments, group sums, flags, split partials.
struct BWs {
    size_t frag, xsum, flag, part;
};
BWs layout(int fmt, int M, int N, int G, const BPlan &p) {
    const size_t nfrag = (size_t)((M + 31) / 32) * ((G + 3) & ~3);
    BWs w;
    w.frag = align256(nfrag * 6144);
    w.xsum = fmt == SLLM_Q2K ? align256(nfrag * 256) : 0;
    w.flag = kq_native(fmt) ? align256(nfrag) : 0;
    w.part = p.splits > 1 ? align256((size_t)p.splits * M * N * sizeof(float)) : 0;
    return w;
}

template <int FMT, int WM, int WN, int CT, int KB, int RA, int WA>
sllm_status launch_shape(const Planes &P, const uint16_t *frag, const float *xsum, const uint8_t *flag,
                         const float *x, float *out, int M, int N, int G, const BPlan &p, int add, hipStream_t s) {
    const int total = p.mtiles * p.ntiles * p.splits;
    constexpr size_t lds = 2 * sizeof(BStage<FMT, KB, 32 * CT * WN>);
    static_assert(lds <= 160 * 1024, "LDS");
    const auto kernel = add ? bgemm_kernel<FMT, WM, WN, CT, KB, RA, WA, true> : bgemm_kernel<FMT, WM, WN, CT, KB, RA, WA, false>;
    hipLaunchKernelGGL(kernel, dim3((total + 7) / 8 * 8), dim3(64 * WM * WN), lds, s, P, frag, xsum, flag, x, out, M, N, G,
                       p.mtiles, p.ntiles, p.splits, p.sps);
    SLLM_HIP(hipGetLastError());
    return SLLM_OK;
}

template <int FMT>
sllm_status launch_fmt(const Planes &P, const float *x, float *dst, int M, int N, int G, const BPlan &p, char *ws,
                       bool add, hipStream_t s) {
    const int ea = add && p.splits == 1;  // the add in the kernel's epilogue, else in the reduction
    const BWs L = layout(FMT, M, N, G, p);
    uint16_t *frag = (uint16_t *)ws;
    float *xsum = (float *)(ws + L.frag);
    uint8_t *flag = (uint8_t *)(ws + L.frag + L.xsum);
    float *out = p.splits > 1 ? (float *)(ws + L.frag + L.xsum + L.flag) : dst;
    const int Gp = (G + 3) & ~3, nfrag = (M + 31) / 32 * Gp;
    hipLaunchKernelGGL(split_frag_kernel<FMT>, dim3((nfrag + 3) / 4), dim3(256), 0, s, x, M, G, Gp, nfrag, frag,
                       xsum,
                       flag);
    SLLM_HIP(hipGetLastError());
    switch (p.shape) {
    case kRows32: return launch_shape<FMT, 1, 4, 2, 2, 2, 2>(P, frag, xsum, flag, x, out, M, N, G, p, ea, s);
    case kRows64: return launch_shape<FMT, 2, 2, 2, 2, 4, 2>(P, frag, xsum, flag, x, out, M, N, G, p, ea, s);
    default: return launch_shape<FMT, 4, 2, 4, kKb128(FMT), 2, 2>(P, frag, xsum, flag, x, out, M, N, G, p, ea, s);
    }
}

}  // namespace

size_t bgemm_workspace_bytes(int fmt, int N, int G, int M) {
    const BWs L = layout(fmt, M, N, G, plan(fmt, M, N, G));
    return L.frag + L.xsum + L.flag + L.part;
}

sllm_status launch_bgemm(int fmt, const Planes &P, const float *x, float *dst, int N, int G, int M, void *ws, bool add,
                         hipStream_t s) {
    const BPlan p = plan(fmt, M, N, G);
    sllm_status st;
    switch (fmt) {
    case SLLM_Q5_0: st = launch_fmt<SLLM_Q5_0>(P, x, dst, M, N, G, p, (char *)ws, add, s); break;
    case SLLM_Q2K: st = launch_fmt<SLLM_Q2K>(P, x, dst, M, N, G, p, (char *)ws, add, s); break;
    case SLLM_Q3K: st = launch_fmt<SLLM_Q3K>(P, x, dst, M, N, G, p, (char *)ws, add, s); break;
    default: return set_error(SLLM_ERR_QTYPE, "gemm: format has no bf16 MFMA path");
    }
    if (st != SLLM_OK || p.splits == 1) return st;
    const BWs L = layout(fmt, M, N, G, p);
    return launch_reduce_splits((const float *)((char *)ws + L.frag + L.xsum + L.flag), dst, (size_t)M * N, p.splits,
                                add, true, s);
}

}  // namespace sllm
