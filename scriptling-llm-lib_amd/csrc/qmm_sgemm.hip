// Short-prompt GEMM (up to 32 activation rows) of the int8 formats: Q8_0, Q4_0,
// Q4_1, Q5K1 on the int8 matrix cores, several weights that share their input in
// one launch, the residual add or the SwiGLU in its epilogue.
//
// What bounds a short prompt: the weight stream (each weight is read once), and
// before that the launches around it. The tiled GEMM (qmm_gemm.hip) staged
// weights through LDS with a barrier per 128 columns of K and needed a quantize
// pass per weight, a split reduction per weight and an elementwise pass after.
// Here
// * sact_kernel (sact_norm_kernel: normed) quantizes the rows once per input, with
//   the GEMV prologue's routines, into MFMA lane order;
// * a wave streams 32 weight rows over its share of K, eight blocks (one 128-byte
//   line of a row's codes) at a time: eight lanes load a row's line, a wave-private
//   LDS image hands every lane its own row, the next eight blocks in flight, no
//   barrier. (Each lane loading its own row's line read it in pieces: 14336x4096
//   Q4_1 at M = 32 25.3 us, 34.9 with non-temporal loads, which fetch the line
//   again for every piece.)
// * the W waves of a workgroup split K between them and meet in LDS once, where
//   the epilogue is applied: one launch, no partials in memory. K is cut into 8 or
//   16 parts whose sums are added as a binary tree, whichever waves form them:
//   an output's order depends on K alone, so a weight gives the same bits alone,
//   beside others and in a gate / up pair.
// The per-block arithmetic: v_mfma_i32_32x32x32_i8 gives a block's exact dots (on top of
// 1.5 * 2^23 as the tiled GEMM has them, or as integers), t = d dot with one rounding,
// acc = fma(t, xs, acc). A min joins its block's term before the scale, t = fma(Σxq, m,
// t), as the reference and the GEMV have it: d dot and m Σxq nearly cancel, and apart, as
// the tiled GEMM adds them, they enter the sum at their own size (error against 64 bits
// over K = 768 / 4096: Q4_1 6.4e-8 / 7.7e-8, apart 1.1e-7 / 1.2e-7, the GEMV 6.4e-8 / 7.8e-8;
// Q5K1 6.7e-8 / 7.9e-8, apart 9.5e-8 / 1.0e-7, the GEMV 8.4e-8 / 9.5e-8; it costs Q5K1
// 4096x4096 at M = 16 14.1 -> 15.0 us, Q4_1 12.8 -> 13.4). Eight blocks that hold a
// non-finite scale, or an activation scale from 2^90, are computed in the reference's
// operation order (qmm_gemm.hip has the reasons).
//
// Counters (RMSNorm + q / k / v, Q5K1 4096 / 1024, M = 30, 12.5 us for 20 MB of weights):
// matrix cores busy 3 %, VALU 16 %, waves issuing 30 %, waiting on loads and LDS 37 %: the
// chain of a wave's two chunks.
#include <hip/hip_runtime.h>

#include "qmm_device.hpp"
#include "qmm_internal.hpp"

namespace sllm {

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef unsigned v2u __attribute__((ext_vector_type(2)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));

constexpr int kMagicBits = 0x4B400000;  // 1.5 * 2^23
constexpr float kMagic = 12582912.0f;
constexpr float kHugeXs = 0x1p90f;
constexpr int kCh = 8;      // blocks per chunk
constexpr int kSplits = 8;  // K splits of a narrow weight's launch
// Parts of K, each summed by itself: a wave's in a narrow weight's launch, one
// chunk up to 4096 columns.
__host__ __device__ constexpr int parts_of(int G) { return G > 64 ? 16 : 8; }

__host__ __device__ constexpr bool has_min(int f) { return f == SLLM_Q4_1 || f == SLLM_Q5K1 || f == SLLM_Q5K1F; }
__host__ __device__ constexpr bool dual(int f) { return f == SLLM_Q5K1; }
__host__ __device__ constexpr bool has_hb(int f) { return f == SLLM_Q5K1 || f == SLLM_Q5K1F; }

// Quantized activations, 32 rows (rows past M: zeros):
//   xq [g][lane][16]  codes: lane r + 32 h, elements 16 h .. of row r
//   xs, sx [g][32]  scale, Σxq (exact in float32)
struct SAct {
    int8_t *xq;
    float *xs, *sx;
};

__host__ inline size_t sact_bytes(int G) { return (size_t)G * (1024 + 2 * 128); }
__host__ inline SAct carve_sact(void *ws, int G) {
    const size_t n = (size_t)G;
    SAct a;
    a.xq = (int8_t *)ws;
    a.xs = (float *)(a.xq + n * 1024);
    a.sx = a.xs + n * 32;
    return a;
}

// Statistics of rmsNormFlatF32 as the GEMV prologue forms them (qmm_gemv_kernel.hpp
// rms_load / rms_finish): 256 slots, slot s adds v * v over x[s], x[s + 256], ... in
// order, wave sums of 64 slots, added left to right.
__device__ __forceinline__ float row_inv(const float *xr, int K, float eps, float *red) {
    const int t = threadIdx.x;
    float p = 0.0f;
    for (int i = t; i < K; i += 16 * 256) {
        float v[16];
#pragma unroll
        for (int k = 0; k < 16; k++) v[k] = i + k * 256 < K ? xr[i + k * 256] : 0.0f;
#pragma unroll
        for (int k = 0; k < 16; k++) p = p + v[k] * v[k];
    }
    const float w = wave_sum(p);
    if ((t & 63) == 0) red[t >> 6] = w;
    __syncthreads();
    const float ss = ((red[0] + red[1]) + red[2]) + red[3];
    const double q = (K & (K - 1)) == 0 ? (double)ss * (1.0 / (double)K) : (double)ss / (double)K;
    return 1.0f / (float)sqrt(q + (double)eps);
}

// Eight lanes quantize a block. Rows past M (of 32) are zeros.
// A block's part u of row r: quantized into place.
__device__ __forceinline__ void put_part(const SAct &a, int r, int g, int sub, const float4 &u) {
    int q[1];
    float s;
    int sm;
    quantize_part<8>(&u, q, s, sm);
    const size_t t = (size_t)g;
    // word sub of the block: lane half sub / 4, word sub % 4 of its 16 bytes
    ((int *)(a.xq + t * 1024 + (r + 32 * (sub >> 2)) * 16))[sub & 3] = q[0];
    if (sub == 0) {
        a.xs[t * 32 + r] = s;
        a.sx[t * 32 + r] = (float)sm;
    }
}

// Without the norm: grid (32 rows, 32 blocks each). (One workgroup per row, its parts in
// turn: every call 0.8-1 us longer, Q4_1 4096x4096 at M = 16 13.8 against 12.8 us.)
__global__ void __launch_bounds__(256) sact_kernel(const float *__restrict__ x, int M, int G, SAct a) {
    const int r = blockIdx.x, sub = threadIdx.x & 7, g = blockIdx.y * 32 + (threadIdx.x >> 3);
    if (g >= G) return;  // eight lanes alike
    put_part(a, r, g, sub, r < M ? ((const float4 *)x)[((size_t)r * G + g) * 8 + sub] : make_float4(0.0f, 0.0f, 0.0f, 0.0f));
}

// RMSNormed rows: one workgroup per row. The first four blocks of a lane's group are
// loaded before the row's statistics are waited for (one memory round trip up to K =
// 4096).
__global__ void __launch_bounds__(256) sact_norm_kernel(const float *__restrict__ x, const float *__restrict__ nw,
                                                        float eps, int M, int G, SAct a) {
    __shared__ float red[4];
    const int r = blockIdx.x;
    const bool live = r < M;
    const float *xr = x + (size_t)(live ? r : M - 1) * G * 32;
    const int sub = threadIdx.x & 7, b0 = threadIdx.x >> 3;
    float4 v[4], w[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int g = min(b0 + 32 * i, G - 1);
        v[i] = ((const float4 *)(xr + (size_t)g * 32))[sub];
        w[i] = ((const float4 *)(nw + (size_t)g * 32))[sub];
    }
    const float inv = row_inv(xr, G * 32, eps, red);
    auto put = [&](int g, const float4 &u, const float4 &c) {
        put_part(a, r, g, sub, live ? make_float4((u.x * inv) * c.x, (u.y * inv) * c.y, (u.z * inv) * c.z, (u.w * inv) * c.w)
                                    : make_float4(0.0f, 0.0f, 0.0f, 0.0f));
    };
#pragma unroll
    for (int i = 0; i < 4; i++)
        if (b0 + 32 * i < G) put(b0 + 32 * i, v[i], w[i]);
    for (int g = b0 + 128; g < G; g += 32)
        put(g, ((const float4 *)(xr + (size_t)g * 32))[sub], ((const float4 *)(nw + (size_t)g * 32))[sub]);
}

// The weights of one launch: segment s owns the column tiles [tile0[s], tile0[s +
// 1]). Mode kPair: P[0] / P[1] are gate / up of one FFN, dst[0] receives the SwiGLU,
// dst[1] / dst[2] (optional) the two products.
enum SMode { kStore = 0, kAdd = 1, kPair = 2 };
struct SegG {
    Planes P[kMaxSegs];
    float *dst[kMaxSegs];
    int N[kMaxSegs];
    int tile0[kMaxSegs + 1];
    int n, mode;
};

// One chunk (kCh blocks x 32 weight rows) as a wave loads it: codes, lane l block
// l % 8 of rows 8 i + l / 8; high bits, lane l words 4 (l % 2) .. of row l / 2;
// scales, lanes 0..31 d and 32..63 m of row l % 32.
template <int FMT>
struct Chunk {
    static constexpr bool Q8 = FMT == SLLM_Q8_0;
    v4i q[Q8 ? 8 : 4];
    v4i sc, dh, hb;
};
// Its wave-private LDS image; rows padded so that lanes reading their own rows hit
// distinct banks.
template <int FMT>
struct alignas(16) Image {
    static constexpr int PL = FMT == SLLM_Q8_0 ? 2 : 1;
    v4i q[PL][32][kCh + 1];
    v4i sc[2][32];
    v4i dh[dual(FMT) ? 32 : 1];
    v4i hb[has_hb(FMT) ? 32 : 1][3];
    v4i a[kCh][64];  // the activation codes, lane's own
    float xs[kCh][32];
    float sx[has_min(FMT) ? kCh : 1][32];
};

template <int FMT>
__device__ __forceinline__ void load_chunk(Chunk<FMT> &c, const Planes &P, int n0, int N, int G, int g, int lane) {
    const int b = lane & 7;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const size_t at = (size_t)min(n0 + 8 * i + (lane >> 3), N - 1) * G + g + b;
        c.q[i] = *(const v4i *)(P.qs + at);
        if (FMT == SLLM_Q8_0) c.q[FMT == SLLM_Q8_0 ? 4 + i : 0] = *(const v4i *)(P.qs2 + at);
    }
    const size_t row = (size_t)min(n0 + (lane & 31), N - 1) * G + g;
    c.sc = *(const v4i *)((has_min(FMT) && lane >= 32 ? P.m : P.d) + row);
    if (dual(FMT)) c.dh = *(const v4i *)(P.dh + row);
    if (has_hb(FMT)) c.hb = *(const v4i *)(P.qh + (size_t)min(n0 + (lane >> 1), N - 1) * G + g + 4 * (lane & 1));
}

template <int FMT>
__device__ __forceinline__ void put_chunk(const Chunk<FMT> &c, Image<FMT> &I, int lane) {
#pragma unroll
    for (int i = 0; i < 4; i++) {
        I.q[0][8 * i + (lane >> 3)][lane & 7] = c.q[i];
        if (FMT == SLLM_Q8_0) I.q[FMT == SLLM_Q8_0 ? 1 : 0][8 * i + (lane >> 3)][lane & 7] = c.q[FMT == SLLM_Q8_0 ? 4 + i : 0];
    }
    I.sc[lane >> 5][lane & 31] = c.sc;
    if (dual(FMT)) I.dh[dual(FMT) ? lane & 31 : 0] = c.dh;
    if (has_hb(FMT)) I.hb[has_hb(FMT) ? lane >> 1 : 0][lane & 1] = c.hb;
}

__device__ __forceinline__ uint16_t half_of(const v2u &v, int b) { return (uint16_t)(v[b >> 1] >> (16 * (b & 1))); }
// any of the eight f16 values not finite
__device__ __forceinline__ bool any_nonfinite(const v4i &v) {
    bool bad = false;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const uint32_t u = (uint32_t)v[i];
        bad |= (u & 0x7c00u) == 0x7c00u || (u & 0x7c000000u) == 0x7c000000u;
    }
    return bad;
}

// Block b's codes as the MFMA's B operand (lane half h: elements 16 h ..).
template <int FMT>
__device__ __forceinline__ void operand(const Image<FMT> &I, int b, int r32, int h, v4i &q, v4i &qh) {
    if (FMT == SLLM_Q8_0) {
        q = I.q[FMT == SLLM_Q8_0 ? h : 0][r32][b];
        return;
    }
    const v4i w = I.q[0][r32][b];
    const int sh = 4 * h;
    const uint32_t hb = has_hb(FMT) ? (uint32_t)((const int *)I.hb[has_hb(FMT) ? r32 : 0])[b] >> sh : 0u;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        int t = (int)((uint32_t)w[k] >> sh) & 0x0f0f0f0f;
        if (FMT == SLLM_Q4_0) t = ((t | (int)0x80808080) - 0x08080808) ^ (int)0x80808080;  // nib - 8 per byte
        if (has_hb(FMT)) {
            // high bits in group order: (hb >> k) & 0x01010101 are elements 4 k ..
            const int bits = (int)((hb >> k) & 0x01010101u);
            if (FMT == SLLM_Q5K1F) t |= bits << 4;
            else qh[k] = bits;
        }
        q[k] = t;
    }
}

// The activation scales (or sums) of a lane's 16 rows of a block.
__device__ __forceinline__ void read_rows(const float *x, int h, float (&xv)[16]) {
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const v4f u = *(const v4f *)(x + 8 * i + 4 * h);
#pragma unroll
        for (int k = 0; k < 4; k++) xv[4 * i + k] = u[k];
    }
}

// The sum of n (1, 2, 4 or 8) values, at(0) .. at(n - 1), as a binary tree.
template <class F>
__device__ __forceinline__ float tree_sum(int n, F at) {
    float s = at(0);
    if (n >= 2) s = s + at(1);
    if (n >= 4) s = s + (at(2) + at(3));
    if (n >= 8) s = s + ((at(4) + at(5)) + (at(6) + at(7)));
    return s;
}

// Grid: column tiles of 32, K splits (1, or kSplits with W = 2: one weight, its partial
// sums to S.dst[0] as [split][M][N]); W waves.
// LDS: every wave's image of its current chunk, then (after a barrier) the waves'
// sums.
template <int FMT, int W>
__global__ void __launch_bounds__(64 * W) __attribute__((amdgpu_waves_per_eu(2)))
sgemm_kernel(SegG S, SAct A, int M, int G) {
    extern __shared__ __attribute__((aligned(16))) float lds[];
    const int lane = threadIdx.x & 63, r32 = lane & 31, h = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const bool pair = S.mode == kPair;
    const int KW = pair ? W / 2 : W;              // waves that split K
    const int kw = pair ? wave % (W / 2) : wave;  // this wave's place among them
    // the workgroup's segment (uniform)
    int seg = 0;
#pragma unroll
    for (int s = 1; s < kMaxSegs; s++)
        if (s < S.n && (int)blockIdx.x >= S.tile0[s]) seg = s;
    Planes P = S.P[0];
    int N = S.N[0];
#pragma unroll
    for (int s = 1; s < kMaxSegs; s++)
        if (s == (pair ? wave / (W / 2) : seg)) {
            P = S.P[s];
            N = S.N[s];
        }
    const int n0 = ((int)blockIdx.x - S.tile0[seg]) * 32;
    // this wave's parts of K: per (1, 2 or 4) of them, chunks [c0, c1)
    const int nch = G / kCh, parts = parts_of(G);
    const int per = parts / (KW * (int)gridDim.y);
    const int p0 = ((int)blockIdx.y * KW + kw) * per;
    const int c0 = nch * p0 / parts, c1 = nch * (p0 + per) / parts;

    v16f acc;
#pragma unroll
    for (int v = 0; v < 16; v++) acc[v] = 0.0f;
    // a dot comes on top of 1.5 * 2^23 as a float, or (has_hb: registers are short) as an
    // integer, converted
    v16i cmag;
#pragma unroll
    for (int v = 0; v < 16; v++) cmag[v] = has_hb(FMT) ? 0 : kMagicBits;
    auto dot_of = [](int d) { return has_hb(FMT) ? (float)d : __int_as_float(d) - kMagic; };  // exact

    // acc: the current part's sum; ones, twos: finished parts that wait for their
    // neighbours in the tree
    v16f ones, twos;
    auto close_part = [&](int i) {
        if (i & 1) {
#pragma unroll
            for (int v = 0; v < 16; v++) acc[v] = ones[v] + acc[v];
            if (i & 2) {
#pragma unroll
                for (int v = 0; v < 16; v++) acc[v] = twos[v] + acc[v];
            }
        }
        if (i + 1 < per) {
            if (i & 1) twos = acc;
            else ones = acc;
#pragma unroll
            for (int v = 0; v < 16; v++) acc[v] = 0.0f;
        }
    };
    if (c0 < c1) {
        Image<FMT> &I = ((Image<FMT> *)lds)[wave];
        Chunk<FMT> ck;
        v4f xr, sr;
        // Everything a chunk needs is requested a whole chunk ahead, the weights
        // last: loads return in order, so a load issued behind the next weights and
        // needed before them would wait for memory in every chunk.
        v4i a[kCh];
        auto load = [&](int c) {
#pragma unroll
            for (int i = 0; i < kCh; i++) a[i] = *(const v4i *)(A.xq + ((size_t)c * kCh + i) * 1024 + lane * 16);
            // kCh x 32 scales are contiguous, four per lane
            xr = *(const v4f *)(A.xs + (size_t)c * kCh * 32 + 4 * lane);
            if (has_min(FMT)) sr = *(const v4f *)(A.sx + (size_t)c * kCh * 32 + 4 * lane);
            load_chunk<FMT>(ck, P, n0, N, G, c * kCh, lane);
        };
        load(c0);
        int part = 0, cend = nch * (p0 + 1) / parts;
        for (int c = c0; c < c1; c++) {
            while (c == cend) {  // parts may be empty
                close_part(part++);
                cend = nch * (p0 + part + 1) / parts;
            }
            const int cnx = min(c + 1, c1 - 1);
            bool slow = any_nonfinite(ck.sc);
            if (dual(FMT)) slow |= any_nonfinite(ck.dh);
            put_chunk<FMT>(ck, I, lane);
#pragma unroll
            for (int i = 0; i < kCh; i++) I.a[i][lane] = a[i];
            *(v4f *)((float *)I.xs + 4 * lane) = xr;
            if (has_min(FMT)) *(v4f *)((float *)I.sx + 4 * lane) = sr;
#pragma unroll
            for (int k = 0; k < 4; k++) slow |= !(xr[k] < kHugeXs);
            const bool exact = __ballot(slow) != 0;
            load(cnx);
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
            __builtin_amdgcn_wave_barrier();
            if (!exact) {
#pragma unroll
                for (int b0 = 0; b0 < kCh; b0 += 4) {
                    const v2u du = *(const v2u *)((const uint16_t *)&I.sc[0][r32] + b0);
                    const v2u mu = *(const v2u *)((const uint16_t *)&I.sc[1][r32] + b0);
                    v2u hu = {};
                    if (dual(FMT)) hu = *(const v2u *)((const uint16_t *)&I.dh[dual(FMT) ? r32 : 0] + b0);
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const int b = b0 + i;
                        v4i q, qh;
                        operand<FMT>(I, b, r32, h, q, qh);
                        const float wd = FMT == SLLM_Q8_0 ? f16_lut(half_of(du, i)) : f16_exact(half_of(du, i));
                        const float wdh = dual(FMT) ? f16_exact(half_of(hu, i)) : 0.0f;
                        const float cd = -kMagic * wd;  // exact
                        const float wm = has_min(FMT) ? f16_exact(half_of(mu, i)) : 0.0f;
                        const v16i D = __builtin_amdgcn_mfma_i32_32x32x32_i8(I.a[b][lane], q, cmag, 0, 0, 0);
                        v16i Dh = {};
                        if (dual(FMT)) Dh = __builtin_amdgcn_mfma_i32_32x32x32_i8(I.a[b][lane], qh, cmag, 0, 0, 0);
#pragma unroll
                        for (int r = 0; r < 4; r++) {
                            // four rows' scales and sums
                            const v4f xv = *(const v4f *)(I.xs[b] + 8 * r + 4 * h);
                            v4f sv = {};
                            if (has_min(FMT)) sv = *(const v4f *)(I.sx[has_min(FMT) ? b : 0] + 8 * r + 4 * h);
#pragma unroll
                            for (int k = 0; k < 4; k++) {
                                const int v = 4 * r + k;
                                float f = has_hb(FMT) ? dot_of(D[v]) * wd : __builtin_fmaf(__int_as_float(D[v]), wd, cd);
                                if (has_min(FMT)) f = __builtin_fmaf(sv[k], wm, f);
                                if (dual(FMT)) f = __builtin_fmaf(dot_of(Dh[v]), wdh, f);
                                acc[v] = __builtin_fmaf(f, xv[k], acc[v]);
                            }
                        }
                    }
                }
            } else {
                // the reference's operation order (no contraction)
#pragma unroll 1
                for (int b = 0; b < kCh; b++) {
                    v4i q, qh, hq = {};
                    operand<FMT>(I, b, r32, h, q, qh);
                    if (FMT == SLLM_Q5K1F) {
                        // the two halves apart: low nibbles and high bits of the 5-bit codes
#pragma unroll
                        for (int k = 0; k < 4; k++) {
                            hq[k] = (q[k] >> 4) & 0x01010101;
                            q[k] = q[k] & 0x0f0f0f0f;
                        }
                    } else if (dual(FMT)) {
                        hq = qh;
                    }
                    const uint16_t db = ((const uint16_t *)&I.sc[0][r32])[b];
                    const float wd = FMT == SLLM_Q8_0 ? f16_lut(db) : f16_exact(db);
                    const float wm = has_min(FMT) ? f16_exact(((const uint16_t *)&I.sc[1][r32])[b]) : 0.0f;
                    const float wdh = dual(FMT) ? f16_exact(((const uint16_t *)&I.dh[dual(FMT) ? r32 : 0])[b]) : 16.0f * wd;
                    const v4i av = I.a[b][lane];
                    float xv[16], sv[16];
                    read_rows(I.xs[b], h, xv);
                    if (has_min(FMT)) read_rows(I.sx[has_min(FMT) ? b : 0], h, sv);
                    const v16i D = __builtin_amdgcn_mfma_i32_32x32x32_i8(av, q, cmag, 0, 0, 0);
                    v16i Dh = {};
                    if (has_hb(FMT)) Dh = __builtin_amdgcn_mfma_i32_32x32x32_i8(av, hq, cmag, 0, 0, 0);
#pragma unroll
                    for (int v = 0; v < 16; v++) {
                        const float dot = dot_of(D[v]);
                        if (!has_min(FMT)) {
                            // q8q8.go:193-195 + vnni_amd64.s:70-73; q4q8.go:37-43
                            const float cmb = wd * xv[v];
                            const float term = cmb * dot;
                            acc[v] = acc[v] + term;
                        } else {
                            // q41q8_row_amd64.s:65-71; the high half of Q5K1 has min +0
                            const float t1 = dot * wd;
                            const float t2 = sv[v] * wm;
                            float tt = t1 + t2;
                            tt = tt * xv[v];
                            acc[v] = acc[v] + tt;
                            if (has_hb(FMT)) {
                                const float h1 = dot_of(Dh[v]) * wdh;
                                const float hh = h1 * xv[v];
                                acc[v] = acc[v] + hh;
                            }
                        }
                    }
                }
            }
            // the image is read before the next chunk is written into it
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
            __builtin_amdgcn_wave_barrier();
        }
        for (; part < per; part++) close_part(part);
    }

    // the waves' sums meet in LDS: [wave][16][64]
    __syncthreads();
#pragma unroll
    for (int v = 0; v < 16; v++) lds[(wave * 16 + v) * 64 + lane] = acc[v];
    __syncthreads();
    constexpr int E = 16 * 64;  // elements of the tile
    float *dst = S.dst[0];
#pragma unroll
    for (int s = 1; s < kMaxSegs; s++)
        if (s == seg) dst = S.dst[s];
    const int Ns = pair ? S.N[0] : N;
    dst += (size_t)blockIdx.y * M * Ns;
#pragma unroll
    for (int i = 0; i < E / (64 * W); i++) {
        const int e = threadIdx.x + 64 * W * i;
        const int l = e & 63, v = e >> 6;
        const int m = 8 * (v >> 2) + 4 * (l >> 5) + (v & 3), col = n0 + (l & 31);
        const float s = tree_sum(KW, [&](int w) { return lds[w * E + e]; });
        if (m >= M || col >= Ns) continue;
        const size_t o = (size_t)m * Ns + col;
        if (pair) {
            const float u = tree_sum(KW, [&](int w) { return lds[(KW + w) * E + e]; });
            if (S.dst[1]) S.dst[1][o] = s;
            if (S.dst[2]) S.dst[2][o] = u;
            dst[o] = swiglu(s, u);  // last: h may lie over gate or up, as for the tiled GEMM
        } else {
            dst[o] = S.mode == kAdd ? dst[o] + s : s;
        }
    }
}

// The upper levels of the tree over a narrow weight's K splits.
__global__ void __launch_bounds__(256) split_sum_kernel(const float *__restrict__ part, float *__restrict__ dst, int n,
                                                        int add) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const float s = tree_sum(kSplits, [&](int k) { return part[(size_t)k * n + i]; });
    dst[i] = add ? dst[i] + s : s;
}

// A weight of 64 tiles or fewer and more than 64 blocks of K, launched by itself, is cut
// into K splits, one chunk of K to a wave; while the partial sums stay small also one of up
// to 96 tiles, 128 for the formats with high bits, whose waves take longest. The bits are
// the same. Measured (us, in splits / in one launch): Q5K1 1024x4096 at M = 32 11.3 / 14.8,
// 3072x3072 at M = 8 12.2 / 14.1, M = 16 12.6 / 13.8, M = 32 13.9 / 14.5, 4096x4096 at M = 16
// 14.5 / 15.0, M = 24 15.5 / 15.1; Q4_0 2560x2560 at M = 16 10.6 / 12.0; Q8_0 3072x4096 at
// M = 24 12.8 / 13.1, M = 32 13.6 / 13.2, 4096x4096 at M = 8 13.6 / 12.5.
bool narrow(bool high_bits, int64_t rows, int G, int M) {
    if (G <= 64) return false;
    if (rows <= 3072) return rows <= 2048 || rows * M <= (high_bits ? 100000 : 75000);
    return high_bits && rows <= 4096 && rows * M <= 75000;
}

template <int FMT, int W>
sllm_status launch_w(const SegG &S, const SAct &A, int M, int G, hipStream_t s, int splits = 1) {
    constexpr size_t img = W * sizeof(Image<FMT>), red = (size_t)W * 1024 * sizeof(float);
    static_assert((img > red ? img : red) <= 160 * 1024, "LDS");
    hipLaunchKernelGGL((sgemm_kernel<FMT, W>), dim3(S.tile0[S.n], splits), dim3(64 * W), img > red ? img : red, s, S, A, M, G);
    SLLM_HIP(hipGetLastError());
    return SLLM_OK;
}

// Eight waves per tile, one tile per CU; with more tiles than CUs four, two
// tiles per CU (14336x4096 at M = 30: eight waves run in two rounds, 21.4 against
// 19.6 us), but not for a pair of more than 64 blocks of K, where a wave would have
// eight parts to hold sums of.
template <int FMT>
sllm_status launch_f(const SegG &S, const SAct &A, int M, int G, hipStream_t s) {
    if (S.n == 1 && S.mode != kPair && narrow(has_hb(FMT), S.N[0], G, M)) {
        SegG T = S;
        T.mode = kStore;
        T.dst[0] = (float *)((char *)A.xq + ((sact_bytes(G) + 255) & ~(size_t)255));
        const sllm_status st = launch_w<FMT, 2>(T, A, M, G, s, kSplits);
        if (st != SLLM_OK) return st;
        const int n = M * S.N[0];
        hipLaunchKernelGGL(split_sum_kernel, dim3((n + 255) / 256), dim3(256), 0, s, T.dst[0], S.dst[0], n, S.mode == kAdd);
        SLLM_HIP(hipGetLastError());
        return SLLM_OK;
    }
    return S.tile0[S.n] > 256 && (S.mode != kPair || G <= 64) ? launch_w<FMT, 4>(S, A, M, G, s) : launch_w<FMT, 8>(S, A, M, G, s);
}

}  // namespace

// Up to 32 rows, and 8192 columns above 4096 weight rows, else 4096 (fewer tiles than
// waves' chunks of K in turn), whatever else the call holds: a weight's bits do not
// depend on its company. Measured (us, with the quantize pass; this / the tiled GEMM, M =
// 16 and 32): Q4_1 14336x4096 22.2 / 29.6 (M = 16), 4096x4096 13.4 / 15.9 and 13.6 / 18.9,
// 1024x4096 10.1 / 11.7 and 10.5 / 12.5, 4608x8192 21.0 / 27.3 and 21.3 / 29.3, 1536x768 7.6 /
// 12.1 (M = 16); Q5K1 4096x4096 14.6 / 14.9 and 15.4 / 16.9, 1024x4096 10.7 / 11.3 and 11.3 /
// 12.2, 3072x3072 12.6 / 13.0 and 13.9 / 14.2; but Q5K1 4096x8192 24.2 / 20.0 and 24.5 / 21.6,
// 2304x4608 17.4 / 14.5 and 17.5 / 15.9, Q4_1 4096x8192 22.1 / 21.5, Q8_0 4096x14336 37.2 /
// 26.2 (a wave's seven chunks of K in turn), and with two row tiles (33 to 64 rows) Q4_1
// 14336x4096 39.4 / 28.8.
bool sgemm_supported(int fmt, int G, int M, int64_t rows) {
    return !act_f32(fmt) && G % kCh == 0 && M <= 32 && G <= (rows <= 4096 ? 128 : 256);
}

// The codes, and the partial sums of a weight of so many rows that is launched by
// itself.
size_t sgemm_ws_bytes(int G, int M, int64_t rows) {
    const size_t act = (sact_bytes(G) + 255) & ~(size_t)255;
    return act + (narrow(true, rows, G, M) ? (size_t)kSplits * M * rows * sizeof(float) : 0);
}

sllm_status launch_sact(const float *x, const float *norm_w, float eps, int M, int G, void *act, hipStream_t s) {
    const SAct a = carve_sact(act, G);
    if (norm_w) hipLaunchKernelGGL(sact_norm_kernel, dim3(32), dim3(256), 0, s, x, norm_w, eps, M, G, a);
    else hipLaunchKernelGGL(sact_kernel, dim3(32, (G + 31) / 32), dim3(256), 0, s, x, M, G, a);
    SLLM_HIP(hipGetLastError());
    return SLLM_OK;
}

sllm_status launch_sgemm(int fmt, const Planes *P, float *const *dst, const int *N, int nseg, int mode, int G, int M,
                         const void *act, hipStream_t s) {
    SegG S{};
    S.mode = mode;
    const bool pair = mode == kPair;
    S.n = pair ? 1 : nseg;
    S.tile0[0] = 0;
    for (int i = 0; i < nseg; i++) {
        S.P[i] = P[i];
        S.N[i] = N[i];
    }
    for (int i = 0; i < (pair ? 3 : nseg); i++) S.dst[i] = dst[i];
    for (int i = 0; i < S.n; i++) S.tile0[i + 1] = S.tile0[i] + (N[i] + 31) / 32;
    const SAct A = carve_sact((void *)act, G);
    switch (fmt) {
    case SLLM_Q8_0: return launch_f<SLLM_Q8_0>(S, A, M, G, s);
    case SLLM_Q4_0: return launch_f<SLLM_Q4_0>(S, A, M, G, s);
    case SLLM_Q4_1: return launch_f<SLLM_Q4_1>(S, A, M, G, s);
    case SLLM_Q5K1: return launch_f<SLLM_Q5K1>(S, A, M, G, s);
    case SLLM_Q5K1F: return launch_f<SLLM_Q5K1F>(S, A, M, G, s);
    }
    return set_error(SLLM_ERR_QTYPE, "short-prompt gemm: format has no int8 MFMA path");
}

}  // namespace sllm
