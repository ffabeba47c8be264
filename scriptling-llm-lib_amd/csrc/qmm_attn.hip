// The attention section of a decode / prefill step (forwardBlock,
// model_f32.go:398-466) on device buffers: bias adds, per-head QK RMSNorm,
// RoPE, the KV-cache append and the causal GQA attention with merged heads.
//
// attn_split_kernel: one workgroup per (split, row, kv head, head slice). A
//   split is a range of cached positions in tiles of 64 (one per lane),
//   shared by up to three tile groups of waves that run side by side; a group
//   stages its tile's K and V rows in LDS once for the q heads of its slice
//   (GQA: the kv head is read from HBM once, through L2 by each slice) and
//   each owning wave takes one q head. The groups' softmax states are merged in LDS; with one split the
//   workgroup writes the attention output itself, otherwise the split's
//   state goes to the workspace. Scores are the reference's sequential
//   float32 dots. For one query row (decode) it also does the bias / norm /
//   RoPE / append work itself.
// attn_prep_kernel / attn_prep_rows_kernel (several rows): that work.
// attn_flash_kernel / attn_flash_combine_kernel (prompts): below.
// attn_combine_kernel (more than one split), attn_combine_long_kernel (more than
//   kShortSplits): merge the splits of every (row, head). Separate launches instead of a last-workgroup combine: on
//   this multi-XCD part a device-scope fence writes back and invalidates the
//   L2, which costs more than the launch.
#include <hip/hip_runtime.h>

#include <cmath>

#include "qmm_device.hpp"
#include "qmm_internal.hpp"

namespace sllm {

namespace {

constexpr int kTile = 64;     // positions per tile: one per lane
constexpr int kChunk = 128;   // K columns staged per pass (LDS: 64 x 132 floats)
constexpr int kMaxDk = 256;   // head size limit (o: 4 values per lane)
constexpr int kMaxWaves = 12; // split workgroup: up to three tile groups of four waves (168 VGPRs each)
constexpr int kDotSteps = 4;  // 4-element steps of a score's LDS reads issued together

// Native 4-float vector: arrays of it stay in registers (HIP's float4, a
// union type, can keep a register array in scratch memory).
typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v2f __attribute__((ext_vector_type(2)));
typedef float v16f __attribute__((ext_vector_type(16)));

__device__ __forceinline__ float lane_bcast(float v, int lane) {
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), lane));
}

// Bias (model_f32.go:398-420), per-head RMSNorm (:424-435; rmsNormFlatF32,
// float32_ops.go:159-172, the sum of squares in the library's association:
// slot s < 256 adds x[s]^2, x[s+256]^2, ..., the four groups of 64 slots are
// wave sums added left to right) and RoPE (applyRopeInPlaceF32,
// float32_ops.go:174-188) of one head row, by one wave, into row (LDS).
// j0: the row's offset in the full q / k row (the bias index).
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
}
__device__ void prep_row(float *row, const float *src, int dk, const float *bias, int j0, int blen,
                         const float *nw, float eps, const float *freqs, int half, int pos, int lane) {
    // this lane's first rotation frequency and its norm weights (d = lane +
    // 64 j, dk <= 256), loaded with the row: one memory round trip in all
    const float f0 = lane < half ? freqs[lane] : 0.0f;
    float wv[4];
#pragma unroll
    for (int j = 0; j < 4; j++) wv[j] = nw && lane + 64 * j < dk ? nw[lane + 64 * j] : 0.0f;
    for (int d = lane; d < dk; d += 64) {
        float x = src[d];
        if (bias && j0 + d < blen) x = x + bias[j0 + d];
        row[d] = x;
    }
    wave_lds_sync();
    if (nw) {
        float w[4];
#pragma unroll
        for (int q4 = 0; q4 < 4; q4++) {
            float p = 0.0f;
            for (int i = q4 * 64 + lane; i < dk; i += 256) p = p + row[i] * row[i];
            w[q4] = wave_sum(p);
        }
        const float ss = ((w[0] + w[1]) + w[2]) + w[3];
        const float inv = 1.0f / (float)sqrt((double)ss / (double)dk + (double)eps);
        wave_lds_sync();
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int d = lane + 64 * j;
            if (d < dk) row[d] = (row[d] * inv) * wv[j];
        }
        wave_lds_sync();
    }
    for (int i = lane; i < half; i += 64) {
        const float ang = (i == lane ? f0 : freqs[i]) * (float)pos;
        double sd, cd;
        sincos((double)ang, &sd, &cd);
        const float c = (float)cd, sn = (float)sd;
        const float x0 = row[2 * i], x1 = row[2 * i + 1];
        row[2 * i] = x0 * c - x1 * sn;
        row[2 * i + 1] = x0 * sn + x1 * c;
    }
    wave_lds_sync();
}

// Several rows (prefill): q heads go to the workspace, kv heads into the cache (k:
// bias, norm, RoPE; v: bias) at rows cache_len + s (the append, model_f32.go:445-448).
// Few rows before the split kernel: one wave per (row, head).
__global__ void __launch_bounds__(64) attn_prep_kernel(AttnArgs a) {
    __shared__ float row[kMaxDk];
    const int s = blockIdx.x, t = blockIdx.y, lane = threadIdx.x;
    const int dk = a.d_k;
    const bool isq = t < a.n_heads;
    const int h = isq ? t : t - a.n_heads;
    const int cols = (isq ? a.n_heads : a.n_kv) * dk;
    prep_row(row, (isq ? a.q : a.k) + (size_t)s * cols + (size_t)h * dk, dk, isq ? a.q_bias : a.k_bias, h * dk,
             isq ? a.qb_len : a.kb_len, isq ? a.q_norm : a.k_norm, a.eps, a.freqs, a.half_dim, a.start_pos + s,
             lane);
    if (isq) {
        float *dst = a.qrot + ((size_t)s * a.n_heads + h) * dk;
        for (int d = lane; d < dk; d += 64) dst[d] = row[d];
        return;
    }
    const size_t at = ((size_t)h * a.cap + (size_t)(a.cache_len + s)) * dk;
    const float *vs = a.v + (size_t)s * cols + (size_t)h * dk;
    for (int d = lane; d < dk; d += 64) {
        a.cache_k[at + d] = row[d];
        float x = vs[d];
        if (a.v_bias && h * dk + d < a.vb_len) x = x + a.v_bias[h * dk + d];
        a.cache_v[at + d] = x;
    }
}

// Prompts: gridDim.y workgroups per row. The row's rotation (the same for every head)
// is formed once per workgroup in LDS, then a wave takes every eighth head of the
// workgroup's: with a workgroup and an fp64 sincos of its own for every head, 1024
// rows of 32 + 8 heads took 15.9 us (now 13.0). Below kPrepRows rows a row has a
// workgroup for every eight heads, so that no wave takes two in turn. (Whole calls,
// us, one wave per head / one workgroup per row: 32/8/128 20 rows 10.3 / 12.1, 64
// 10.9 / 13.6, 200 32.0 / 33.7, 512 62.6 / 62.8, 700 96.6 / 95.7.)
constexpr int kPrepRows = 512;
constexpr int kPrepWaves = 8;
__global__ void __launch_bounds__(64 * kPrepWaves) attn_prep_rows_kernel(AttnArgs a) {
    __shared__ float rows[kPrepWaves][kMaxDk];
    __shared__ float rc[kMaxDk / 2], rs[kMaxDk / 2];
    const int s = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int dk = a.d_k;
    float *row = rows[wave];
    auto prep = [&](int t) {
        const bool isq = t < a.n_heads;
        const int h = isq ? t : t - a.n_heads;
        const int cols = (isq ? a.n_heads : a.n_kv) * dk;
        prep_row(row, (isq ? a.q : a.k) + (size_t)s * cols + (size_t)h * dk, dk, isq ? a.q_bias : a.k_bias, h * dk,
                 isq ? a.qb_len : a.kb_len, isq ? a.q_norm : a.k_norm, a.eps, nullptr, 0, 0, lane);
    };
    // the first head's row is loaded with the frequency (half_dim is below the
    // workgroup's threads), not behind the rotation's barrier
    const int first = blockIdx.y * kPrepWaves + wave;
    const float fr = (int)threadIdx.x < a.half_dim ? a.freqs[threadIdx.x] : 0.0f;
    if (first < a.n_heads + a.n_kv) prep(first);
    static_assert(kMaxDk / 2 <= 64 * kPrepWaves, "a thread per frequency");
    if ((int)threadIdx.x < a.half_dim) {
        const float ang = fr * (float)(a.start_pos + s);
        double sd, cd;
        sincos((double)ang, &sd, &cd);
        rc[threadIdx.x] = (float)cd;
        rs[threadIdx.x] = (float)sd;
    }
    __syncthreads();
    for (int t = first; t < a.n_heads + a.n_kv; t += gridDim.y * kPrepWaves) {
        const bool isq = t < a.n_heads;
        const int h = isq ? t : t - a.n_heads;
        const int cols = (isq ? a.n_heads : a.n_kv) * dk;
        if (t != first) prep(t);
        // RoPE (applyRopeInPlaceF32, float32_ops.go:174-188)
        for (int i = lane; i < a.half_dim; i += 64) {
            const float c = rc[i], sn = rs[i];
            const float x0 = row[2 * i], x1 = row[2 * i + 1];
            row[2 * i] = x0 * c - x1 * sn;
            row[2 * i + 1] = x0 * sn + x1 * c;
        }
        wave_lds_sync();
        if (isq) {
            float *dst = a.qrot + ((size_t)s * a.n_heads + h) * dk;
            for (int d = lane; d < dk; d += 64) dst[d] = row[d];
        } else {
            const size_t at = ((size_t)h * a.cap + (size_t)(a.cache_len + s)) * dk;
            const float *vs = a.v + (size_t)s * cols + (size_t)h * dk;
            for (int d = lane; d < dk; d += 64) {
                a.cache_k[at + d] = row[d];
                float x = vs[d];
                if (a.v_bias && h * dk + d < a.vb_len) x = x + a.v_bias[h * dk + d];
                a.cache_v[at + d] = x;
            }
        }
        wave_lds_sync();  // the row is read before the next head's is written
    }
}

// fusedAttentionHeadF32 (float32_ops.go:190-235) for the q heads of one kv
// head (repeatKVDataF32, float32_ops.go:252-260: q head g*rep + r reads kv
// head g) and one query row, over one split of the positions the causal mask
// leaves (0 .. cache_len + qi). Score = (sequential float32 dot) * scale, as
// the reference computes it; the exponentials are float32(exp(float64(score
// - running max))), rescaled by the same form when the running max grows.
//
// The split is a.tw tile groups of nh = max(4, rep) waves (at most
// kMaxWaves waves in all); group t takes a.tps consecutive tiles of the
// split's range (every group runs the same number of steps, so the
// workgroup barriers line up; a tile past the range has no positions). The
// kv group's q heads are shared by a.hs workgroups (head slices) of hp =
// rep / hs heads each; in group t, wave r owns slice head hr = (r - t hp)
// mod nh if hr < hp (the owning waves of successive groups start on
// successive SIMDs), and keeps the value sums of d_k / 64 (rounded up)
// dimensions per lane: d = 2 lane + j when d_k is 128 (one 8-byte LDS read
// per position), d = lane + 64 j otherwise. FULL: d_k is exactly 64 DKL.
// Every head's arithmetic is the same whatever hs is.
// PREP (one query row): group 0's waves first build the q heads (bias, norm,
// RoPE) in LDS, and in the workgroup whose range holds the new position the
// last wave builds the new k / v row, appends it to the cache and the groups
// use it from LDS; otherwise the preparation has done both. Per tile the K
// and V rows are loaded together (K straight to LDS, V to registers while
// the scores are computed, then to the same LDS buffer): one memory latency
// per tile, overlapped with the q preparation for the first tile (FULL; the
// other head sizes issue its V rows after the preparation, whose registers
// they would share). LDS reads are issued in groups. At the end each wave
// leaves its (max, sum, values) state in LDS and group 0 merges the groups'
// states in group order exactly as attn_combine_kernel merges splits.
template <bool PREP, int DKL, bool FULL>
__global__ void __launch_bounds__(kMaxWaves * 64) attn_split_kernel(AttnArgs a) {

    extern __shared__ __attribute__((aligned(16))) float lds[];
    constexpr int ks = kChunk + 4;
    const int dk = FULL ? 64 * DKL : a.d_k;
    // o[j] of a lane holds value dof(j): d = 2 lane + j (PAIRED: one 8-byte
    // LDS read per position) or d = lane + 64 j
    constexpr bool PAIRED = FULL && DKL == 2;
    const int nh = a.rep > 4 ? a.rep : 4;  // waves per tile group
    const int hp = a.rep / a.hs;           // q heads per workgroup
    const int ng = 64 * nh;                // threads per tile group
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int grp = wave / nh;
    const int r = wave - grp * nh;
    const int hr = (r + nh - (grp * hp) % nh) % nh;  // this wave's q head in the slice, if < hp
    const int tg = tid - grp * ng;                   // thread index within the group
    const bool head = hr < hp;
    auto dof = [&](int j) { return PAIRED ? 2 * lane + j : lane + 64 * j; };
    float *kt = lds + (size_t)grp * kTile * ks;  // kTile x ks: a K chunk, then a V chunk
    float *qs = lds + (size_t)a.tw * kTile * ks; // hp x d_k: the slice's rotated q heads
    float *nk = qs + hp * dk;                    // PREP: the new k and v rows (2 x d_k)
    float *mg = nk + 2 * dk;                     // hp x tw x (d_k + 2): the groups' states
    float *ew = mg + (size_t)hp * a.tw * (dk + 2) + (size_t)wave * kTile;  // this wave's tile weights
    const int split = blockIdx.x;
    const int ys = blockIdx.y / a.hs, sl = blockIdx.y - ys * a.hs;  // (row, kv head), head slice
    const int qi = a.row0 + ys / a.n_kv, g = ys - (ys / a.n_kv) * a.n_kv;
    const int h0 = g * a.rep + sl * hp;  // the slice's first q head
    const int limit = a.cache_len + qi + 1;
    const int w0 = split * a.tw * a.tps * kTile;  // the workgroup's range [w0, w1)
    const int w1 = min(w0 + a.tw * a.tps * kTile, limit);
    const int p0 = w0 + grp * a.tps * kTile;      // this group's range [p0, p1) (may be empty)
    const int p1 = min(p0 + a.tps * kTile, limit);
    // rows read from the cache: PREP builds the new one (position cache_len) itself
    const int have = PREP ? a.cache_len : limit;
    const bool owns_new = PREP && a.cache_len >= w0 && a.cache_len < w1;
    const float *kb = a.cache_k + (size_t)g * a.cap * dk;
    const float *vb = a.cache_v + (size_t)g * a.cap * dk;
    constexpr bool one_chunk = DKL <= 2;  // d_k <= kChunk

    v4f kreg[8], vreg[8];
    auto load_chunk = [&](int t0, int n, int c0, bool k_too, bool v_too) {
        const int q4 = FULL ? 16 * DKL : min(kChunk, dk - c0) / 4;
#pragma unroll
        for (int u = 0; u < 8; u++) {
            const int i = tg + ng * u;
            if (i < n * q4) {
                const int p = (int)((unsigned)i / (unsigned)q4), c = (i - p * q4) * 4;
                if (t0 + p < have) {
                    // 32-bit byte offset from the head's base (SGPR base + VGPR offset)
                    const uint32_t at = ((uint32_t)(t0 + p) * (uint32_t)dk + (uint32_t)(c0 + c)) * 4u;
                    if (k_too) kreg[u] = *(const v4f *)((const char *)kb + at);
                    if (v_too) vreg[u] = *(const v4f *)((const char *)vb + at);
                }
            }
        }
    };
    // rows n .. n rounded up to 8 are written as zeros (the value loop reads
    // whole groups of eight rows)
    auto store_chunk = [&](const v4f *reg, int n, int c0, int newp, const float *newrow) {
        const int q4 = FULL ? 16 * DKL : min(kChunk, dk - c0) / 4;
        const int n8 = (n + 7) & ~7;
#pragma unroll
        for (int u = 0; u < 8; u++) {
            const int i = tg + ng * u;
            if (i < n8 * q4) {
                const int p = (int)((unsigned)i / (unsigned)q4), c = (i - p * q4) * 4;
                const v4f z = {0.0f, 0.0f, 0.0f, 0.0f};
                *(v4f *)(kt + p * ks + c) = p >= n ? z : ((p == newp) ? *(const v4f *)(newrow + c0 + c) : reg[u]);
            }
        }
    };
    // the first tile's K rows (FULL: and V rows) are issued before anything
    // waits; otherwise its V rows after the q preparation, whose registers
    // they would share
    if (p0 < p1) load_chunk(p0, min(kTile, p1 - p0), 0, true, FULL && one_chunk);

    if (PREP) {
        const int pos = a.start_pos + qi;
        if (head && grp == 0) {
            const int h = h0 + hr;
            prep_row(qs + hr * dk, a.q + (size_t)qi * a.n_heads * dk + (size_t)h * dk, dk, a.q_bias, h * dk, a.qb_len,
                     a.q_norm, a.eps, a.freqs, a.half_dim, pos, lane);
        }
        // the first wave of group 0 that prepares no q head (waves 0 .. nh - 1
        // start first; with every group-0 wave on a q head, the workgroup's
        // last wave); every head slice builds the row for itself, slice 0
        // appends it to the cache
        const int kwave = hp < nh ? hp : (int)(blockDim.x >> 6) - 1;
        if (owns_new && wave == kwave) {
            const size_t off = (size_t)qi * a.n_kv * dk + (size_t)g * dk;
            // the v row (d = lane + 64 j, dk <= 256) is loaded before the k
            // row is prepared, so its memory round trip overlaps that work
            float vv[4];
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int d = lane + 64 * j;
                vv[j] = 0.0f;
                if (d < dk) {
                    vv[j] = a.v[off + d];
                    if (a.v_bias && g * dk + d < a.vb_len) vv[j] = vv[j] + a.v_bias[g * dk + d];
                }
            }
            prep_row(nk, a.k + off, dk, a.k_bias, g * dk, a.kb_len, a.k_norm, a.eps, a.freqs, a.half_dim, pos, lane);
            const size_t at = ((size_t)g * a.cap + (size_t)a.cache_len) * dk;
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int d = lane + 64 * j;
                if (d < dk) {
                    nk[dk + d] = vv[j];
                    if (sl == 0) {
                        a.cache_k[at + d] = nk[d];
                        a.cache_v[at + d] = vv[j];
                    }
                }
            }
        }
    } else {
        const float4 *qq = (const float4 *)(a.qrot + ((size_t)qi * a.n_heads + (size_t)h0) * dk);
        for (int i = tid; i < hp * dk / 4; i += (int)blockDim.x) ((float4 *)qs)[i] = qq[i];
    }

    if (!FULL && one_chunk && p0 < p1) load_chunk(p0, min(kTile, p1 - p0), 0, false, true);

    float m = -INFINITY, l = 0.0f, o[DKL];
#pragma unroll
    for (int j = 0; j < DKL; j++) o[j] = 0.0f;
    for (int it = 0; it < a.tps; it++) {
        const int t0 = p0 + it * kTile;
        const int n = max(0, min(kTile, p1 - t0));  // valid positions of this tile (lanes < n)
        const int newp = owns_new ? a.cache_len - t0 : -1;  // row of the new position in this tile
        float dot = 0.0f;
        for (int c0 = 0; c0 < dk; c0 += kChunk) {
            const int cw = min(kChunk, dk - c0);
            if (it != 0 || c0 != 0) load_chunk(t0, n, c0, true, one_chunk);
            __syncthreads();  // the previous users of kt are done (and qs / nk are written)
            store_chunk(kreg, n, c0, newp, nk);
            __syncthreads();
            if (head && lane < n) {
                const float *qr = qs + hr * dk + c0;
                const float *kr = kt + lane * ks;
                for (int d0 = 0; d0 < cw; d0 += 4 * kDotSteps) {
                    // kDotSteps 4-element steps: their LDS reads issue together,
                    // the products are added one by one in element order
                    v4f kv[kDotSteps], qv[kDotSteps];
#pragma unroll
                    for (int u = 0; u < kDotSteps; u++) {
                        kv[u] = *(const v4f *)(kr + d0 + 4 * u);
                        qv[u] = *(const v4f *)(qr + d0 + 4 * u);
                    }
                    const int steps = min(kDotSteps, (cw - d0) / 4);
#pragma unroll
                    for (int u = 0; u < kDotSteps; u++) {
                        if (u < steps) {
                            dot += qv[u].x * kv[u].x;
                            dot += qv[u].y * kv[u].y;
                            dot += qv[u].z * kv[u].z;
                            dot += qv[u].w * kv[u].w;
                        }
                    }
                }
            }
        }
        // online softmax of this tile (a tile without positions changes nothing)
        float e = 0.0f;
        if (head && n > 0) {
            const float sc = lane < n ? dot * a.scale : -INFINITY;
            float mt = sc;
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) mt = fmaxf(mt, __shfl_xor(mt, off, 64));
            const float mn = fmaxf(m, mt);
            // a group's first tile (running max still -inf) against a finite
            // max: exp(-inf) = 0 exactly, without the fp64 exp on the chain
            const float alpha = (m == -INFINITY && mn > -INFINITY && mn < INFINITY) ? 0.0f
                                                                                  : (float)exp((double)(m - mn));
            e = lane < n ? (float)exp((double)(sc - mn)) : 0.0f;
            l = l * alpha + wave_sum(e);
            m = mn;
#pragma unroll
            for (int j = 0; j < DKL; j++) o[j] = o[j] * alpha;
        }
        // o += sum over the tile's positions of e_p * V[p], V chunk by chunk in LDS
        for (int c0 = 0; c0 < dk; c0 += kChunk) {
            const int cw = min(kChunk, dk - c0);
            if (!one_chunk) load_chunk(t0, n, c0, false, true);
            __syncthreads();  // the score readers of kt are done
            store_chunk(vreg, n, c0, newp, nk + dk);
            __syncthreads();
            if (head) {
                // the weights go through LDS: eight per group of positions in two
                // broadcast reads (0 past the tile's end, where the rows are zeros)
                if (c0 == 0) {
                    ew[lane] = e;
                    wave_lds_sync();
                }
                for (int q0 = 0; q0 < n; q0 += 8) {
                    const v4f ea = *(const v4f *)(ew + q0), eb = *(const v4f *)(ew + q0 + 4);
                    const float ev[8] = {ea.x, ea.y, ea.z, ea.w, eb.x, eb.y, eb.z, eb.w};
                    if (PAIRED) {
                        // eight positions' values read together, then accumulated in
                        // order (fused multiply-add: one rounding per step)
                        v2f vv[8];
#pragma unroll
                        for (int pp = 0; pp < 8; pp++) vv[pp] = *(const v2f *)(kt + (q0 + pp) * ks + 2 * lane);
#pragma unroll
                        for (int pp = 0; pp < 8; pp++) {
                            o[0] = __builtin_fmaf(ev[pp], vv[pp].x, o[0]);
                            o[PAIRED ? 1 : 0] = __builtin_fmaf(ev[pp], vv[pp].y, o[PAIRED ? 1 : 0]);
                        }
                    } else {
                        float vv[8][DKL];
#pragma unroll
                        for (int pp = 0; pp < 8; pp++) {
                            const float *vr = kt + (q0 + pp) * ks - c0;
#pragma unroll
                            for (int j = 0; j < DKL; j++) {
                                const int d = dof(j);
                                vv[pp][j] = (d >= c0 && d < c0 + cw) ? vr[d] : 0.0f;
                            }
                        }
#pragma unroll
                        for (int pp = 0; pp < 8; pp++) {
#pragma unroll
                            for (int j = 0; j < DKL; j++) {
                                const int d = dof(j);
                                if (d >= c0 && d < c0 + cw) o[j] = __builtin_fmaf(ev[pp], vv[pp][j], o[j]);
                            }
                        }
                    }
                }
            }
        }
    }

    // the groups' states meet in LDS; group 0 merges them (M = max, weights
    // w_t = float32(exp(float64(m_t - M))), L = wave_sum over lanes t of
    // l_t * w_t, O = sum over t in order of o_t * w_t), as attn_combine_kernel does
    const int sst = dk + 2;
    if (head) {
        float *st = mg + ((size_t)hr * a.tw + grp) * sst;
        if (lane == 0) {
            st[0] = m;
            st[1] = l;
        }
#pragma unroll
        for (int j = 0; j < DKL; j++) {
            const int d = dof(j);
            if (d < dk) st[2 + d] = o[j];
        }
    }
    __syncthreads();
    if (!head || grp != 0) return;
    const float *sb = mg + (size_t)hr * a.tw * sst;
    float M = -INFINITY;
    for (int t = 0; t < a.tw; t++) M = fmaxf(M, sb[t * sst]);
    const bool mine = lane < a.tw;
    const float ml = mine ? sb[lane * sst] : -INFINITY;
    const float ll = mine ? sb[lane * sst + 1] : 0.0f;
    // a group without positions weighs 0 (also when no group has any: a split
    // of a causal row can lie wholly past it, and then leaves (-inf, 0, 0))
    const float wl = (mine && ml != -INFINITY) ? (float)exp((double)(ml - M)) : 0.0f;
    const float L = wave_sum(0.0f + ll * wl);
    float O[DKL];
#pragma unroll
    for (int j = 0; j < DKL; j++) O[j] = 0.0f;
    for (int t = 0; t < a.tw; t++) {
        const float w = lane_bcast(wl, t);
#pragma unroll
        for (int j = 0; j < DKL; j++) {
            const int d = dof(j);
            O[j] = O[j] + (d < dk ? sb[t * sst + 2 + d] : 0.0f) * w;
        }
    }
    const int h = h0 + hr;
    if (a.splits == 1) {
        const float inv = 1.0f / L;
        float *dst = a.out + ((size_t)qi * a.n_heads + h) * dk;  // mergeHeadsDataF32 layout
#pragma unroll
        for (int j = 0; j < DKL; j++) {
            const int d = dof(j);
            if (d < dk) dst[d] = O[j] * inv;
        }
    } else {
        // this split's partial of the head: running max, sum, weighted values
        float *pp = a.part + (((size_t)qi * a.n_heads + h) * a.splits + split) * sst;
        if (lane == 0) {
            pp[0] = M;
            pp[1] = L;
        }
#pragma unroll
        for (int j = 0; j < DKL; j++) {
            const int d = dof(j);
            if (d < dk) pp[2 + d] = O[j];
        }
    }
}

// The merge of the splits of one (row, head): M = max of the split maxima, weights
// w_t = float32(exp(float64(m_t - M))), L = sum of l_t * w_t (lane t % 16 adds its
// splits' terms in order, then the wave's tree), out[d] = (sum over t, in order, of
// o_t[d] * w_t) * (1 / L), written in mergeHeadsDataF32's layout
// (float32_ops.go:262-273). A split without positions (max -inf) weighs 0. Both
// kernels below form every output in that one order.

// Up to kShortSplits splits: one wave per (row, head), everything loaded together.
constexpr int kShortSplits = 16;
__global__ void __launch_bounds__(256) attn_combine_kernel(AttnArgs a) {
    const int lane = threadIdx.x & 63;
    const int pair = blockIdx.x * 4 + (threadIdx.x >> 6);  // qi * n_heads + h
    if (pair >= a.seq * a.n_heads) return;                 // wave-uniform
    const int dk = a.d_k, nt = a.splits;
    const size_t stride = (size_t)dk + 2;
    const float *pb = a.part + (size_t)pair * nt * stride;
    const bool mine = lane < nt;  // lane t holds m_t and l_t
    const float ml = mine ? pb[lane * stride] : -INFINITY;
    const float ll = mine ? pb[lane * stride + 1] : 0.0f;
    float ov[kShortSplits][4];
#pragma unroll
    for (int u = 0; u < kShortSplits; u++) {
        const float *ob = pb + (size_t)u * stride + 2;
#pragma unroll
        for (int jj = 0; jj < 4; jj++) {
            const int d = lane + 64 * jj;
            ov[u][jj] = (u < nt && d < dk) ? ob[d] : 0.0f;
        }
    }
    float M = ml;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) M = fmaxf(M, __shfl_xor(M, off, 64));
    const float wl = (mine && ml != -INFINITY) ? (float)exp((double)(ml - M)) : 0.0f;
    float O[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int u = 0; u < kShortSplits; u++) {
        const float w = lane_bcast(wl, u);  // 0 past the last split, where the values are zeros
#pragma unroll
        for (int jj = 0; jj < 4; jj++) O[jj] = O[jj] + ov[u][jj] * w;
    }
    const float inv = 1.0f / wave_sum(0.0f + ll * wl);
    float *dst = a.out + (size_t)pair * dk;  // mergeHeadsDataF32 layout
#pragma unroll
    for (int jj = 0; jj < 4; jj++) {
        const int d = lane + 64 * jj;
        if (d < dk) dst[d] = O[jj] * inv;
    }
}

// More splits: one workgroup of eight waves per (row, head). In a round a wave takes
// up to eight splits, all its loads issued together, and leaves their weighted values
// in LDS; a thread per dimension then adds the round's in split order. (One wave per
// head left 32 waves on the device for a decode step, each with a round of memory
// per 16 splits: 9.0 us at 63 splits. One decode step, whole call, one wave / this:
// 32/8/128 at 8000 cached 31.2 / 27.5 us, 4000 18.3 / 16.5; 8/1/256 at 8000 40.1 /
// 32.0. Sums by wave, in another order, would take 26.1 at 8000.)
constexpr int kLongWaves = 8, kRound = 8 * kLongWaves;
__global__ void __launch_bounds__(64 * kLongWaves) attn_combine_long_kernel(AttnArgs a) {
    extern __shared__ __attribute__((aligned(16))) float lds[];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int pair = blockIdx.x;  // qi * n_heads + h
    const int dk = a.d_k;
    float *P = lds, *T = lds + kRound * dk;  // [split of the round][d]; l_t * w_t
    const size_t stride = (size_t)dk + 2;
    const float *pb = a.part + (size_t)pair * a.splits * stride;
    // this wave's splits of the round from t0: u0 .. u0 + nu - 1 (none if nu <= 0);
    // lane u holds split u0 + u's max and sum
    int n, u0, nu;
    float ov[8][4], ml, ll;
    auto load = [&](int t0) {
        n = min(kRound, a.splits - t0);
        const int per = (n + kLongWaves - 1) / kLongWaves;
        u0 = wave * per;
        nu = min(per, n - u0);
        const float *rb = pb + (size_t)(t0 + min(u0, n - 1)) * stride;
        const int last = max(nu, 1) - 1;
        ml = rb[min(lane, last) * stride];
        ll = rb[min(lane, last) * stride + 1];
#pragma unroll
        for (int u = 0; u < 8; u++) {
            const float *ob = rb + min(u, last) * stride + 2;
#pragma unroll
            for (int jj = 0; jj < 4; jj++) {
                const int d = lane + 64 * jj;
                ov[u][jj] = d < dk ? ob[d] : 0.0f;
            }
        }
    };
    load(0);  // before the maxima are waited for
    float M = -INFINITY;
    for (int t = lane; t < a.splits; t += 64) M = fmaxf(M, pb[t * stride]);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) M = fmaxf(M, __shfl_xor(M, off, 64));
    static_assert(kMaxDk <= 64 * kLongWaves, "a thread per dimension");
    float O = 0.0f, Lp = 0.0f;
    for (int t0 = 0; t0 < a.splits; t0 += kRound) {
        if (t0 > 0) load(t0);
        const float wl = ml != -INFINITY ? (float)exp((double)(ml - M)) : 0.0f;
        if (lane < nu) T[u0 + lane] = ll * wl;
#pragma unroll
        for (int u = 0; u < 8; u++) {
            const float w = lane_bcast(wl, u);
#pragma unroll
            for (int jj = 0; jj < 4; jj++) {
                const int d = lane + 64 * jj;
                if (u < nu && d < dk) P[(u0 + u) * dk + d] = ov[u][jj] * w;
            }
        }
        __syncthreads();
        for (int t = lane & 15; t < n; t += 16) Lp = Lp + T[t];
        if ((int)threadIdx.x < dk) {
            int t = 0;
            for (; t + 16 <= n; t += 16) {
                float v[16];
#pragma unroll
                for (int u = 0; u < 16; u++) v[u] = P[(t + u) * dk + threadIdx.x];
#pragma unroll
                for (int u = 0; u < 16; u++) O = O + v[u];
            }
            for (; t < n; t++) O = O + P[t * dk + threadIdx.x];
        }
        if (t0 + kRound < a.splits) __syncthreads();  // read before the next round is written
    }
    const float inv = 1.0f / wave_sum(lane < 16 ? Lp : 0.0f);
    if ((int)threadIdx.x < dk) a.out[(size_t)pair * dk + threadIdx.x] = O * inv;  // mergeHeadsDataF32 layout
}

// ---------------------------------------------------------- prompts ----
//
// attn_flash_kernel: several query rows (more than flash_pairs pairs of row and kv
// head, d_k up to 128) on the fp32 matrix cores. A wave owns 32 query rows of one q head; the four
// waves of a workgroup share one kv head's K and V tiles of 32 positions in LDS
// (GQA: the q heads of the group; otherwise further row blocks). Both products
// are taken transposed, so that a lane is a query row throughout:
//   S^T = K Q^T: A = K (LDS), B = Q (registers for the whole kernel). Lane half h
//     takes the head's dimensions DK / 2 h .. (the order of the MFMA's k is
//     free), so K is read with 16-byte LDS reads;
//   softmax: a lane holds 16 of the tile's positions of its row, lane ^ 32 the
//     other 16: no reduction over lanes but one exchange;
//   O^T = V^T P^T: accumulator v of S^T is position 8 (v / 4) + 4 h + v % 4, so as
//     B operand of a two-deep MFMA it pairs positions p and p + 4: P goes from
//     accumulator to operand without leaving its registers, V is read to match.
// Scores are fp32 dots of the same products as the reference's (in two halves,
// added by the MFMA), the exponentials float32(exp(float64(x))) as the reference's
// (exp_neg), the sums fp32, in another association than the split kernel's.
//
// What bounds it: the fp32 matrix cores (64 cycles per 32 x 32 x 2, DK of them per tile:
// busy for 47 % of 126 us) and what they wait on, issue behind each other and the
// softmax between the two products (waves ready for 65 % of their cycles, VALU busy 18
// %). The split kernel spent 64-lane VALU dots and one pass over K and V per query row
// (1024 rows of 32 / 8 heads, d_k 128, whole call: 882 us, now 152).
// Causal rows differ in length: a row block's tiles are cut into chunks of C
// tiles (workgroups of their own; heaviest first) whose states
// attn_flash_combine_kernel merges; C is about the tiles one workgroup slot gets
// in all, so that no workgroup outlasts the rest.
// Positions past a row's limit get weight 0 by selection. A non-finite V
// element would still turn the earlier rows' 0 into NaN inside the MFMA: such
// elements are staged as 0, their positions noted, and their products added to
// the rows that see them on the VALU.
constexpr int kFlashTile = 32;
constexpr int kFlashWaves = 4;

struct FlashPlan {
    int groups;   // workgroups of units per kv head
    int chunk;    // most tiles per chunk
    int chunks;   // most chunks of a group
};
// Tiles of each chunk of a group with so many tiles: chunks of one group are even.
__host__ __device__ inline int flash_chunk(const FlashPlan &f, int tiles) {
    const int n = (tiles + f.chunk - 1) / f.chunk;
    return (tiles + n - 1) / n;
}

// float32(exp(float64(x))) for a float32 x <= 0 (or NaN): the exponential in 64 bits,
// rounded to float32 once. r = x - n ln 2 in two parts (the first product exact: n
// has at most 8 bits, the first constant 42), |r| <= 0.35, the Taylor polynomial of
// exp(r) to r^11 (remainder below 2^-46 of the value). Below -104 the float32 is 0.
__device__ __forceinline__ float exp_neg(float x) {
    const double xd = (double)x;
    const double n = __builtin_rint(xd * 1.4426950408889634);
    double r = __builtin_fma(n, -0x1.62e42fefa38p-1, xd);
    r = __builtin_fma(n, -0x1.ef35793c7673p-45, r);
    double p = 1.0 / 39916800.0;
    p = __builtin_fma(p, r, 1.0 / 3628800.0);
    p = __builtin_fma(p, r, 1.0 / 362880.0);
    p = __builtin_fma(p, r, 1.0 / 40320.0);
    p = __builtin_fma(p, r, 1.0 / 5040.0);
    p = __builtin_fma(p, r, 1.0 / 720.0);
    p = __builtin_fma(p, r, 1.0 / 120.0);
    p = __builtin_fma(p, r, 1.0 / 24.0);
    p = __builtin_fma(p, r, 1.0 / 6.0);
    p = __builtin_fma(p, r, 0.5);
    p = __builtin_fma(p, r, 1.0);
    p = __builtin_fma(p, r, 1.0);
    const float y = (float)__builtin_ldexp(p, (int)n);
    return x < -104.0f ? 0.0f : y;
}

template <int DT, bool FULL>
__global__ void __launch_bounds__(64 * kFlashWaves) __attribute__((amdgpu_waves_per_eu(2)))
attn_flash_kernel(AttnArgs a, FlashPlan f) {
    constexpr int DK = 32 * DT, HD = DK / 2;  // padded head size; dimensions per lane half
    constexpr int KS = DK + 4;                // LDS row stride: 16-byte reads of successive rows hit distinct banks
    constexpr int T = 64 * kFlashWaves;
    constexpr int PER = kFlashTile * (DK / 4) / T;  // 16-byte pieces of K (and of V) per thread
    extern __shared__ __attribute__((aligned(16))) float lds[];
    // [2 buffers][K tile, V tile], then the masks
    auto ktile = [&](int b) { return lds + b * 2 * kFlashTile * KS; };
    auto vtile = [&](int b) { return lds + (b * 2 + 1) * kFlashTile * KS; };
    // masks of the tile's positions with non-finite V elements, one for each of
    // three successive tiles: read, filled and cleared in the same step
    unsigned *badm = (unsigned *)(lds + 4 * kFlashTile * KS);

    const int dk = FULL ? DK : a.d_k;
    const int g = blockIdx.x;                           // kv head (fastest: one head per XCD)
    const int ug = (int)gridDim.y - 1 - (int)blockIdx.y;  // longest rows first
    const int ch = blockIdx.z;
    const int lane = threadIdx.x & 63, r32 = lane & 31, h = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nrb = (a.seq + 31) / 32, U = nrb * a.rep;
    auto kv_of = [&](int rb) { return a.cache_len + min(a.seq, 32 * (rb + 1)); };  // positions a row block sees
    const int last = min(ug * kFlashWaves + kFlashWaves - 1, U - 1);
    const int tiles = (kv_of(last / a.rep) + kFlashTile - 1) / kFlashTile;
    const int clen = flash_chunk(f, tiles);
    const int t0 = ch * clen, t1 = min(tiles, t0 + clen);
    if (t0 >= tiles) return;
    const int unit = min(ug * kFlashWaves + wave, U - 1);
    const bool mine = ug * kFlashWaves + wave < U;
    const int rb = unit / a.rep, hq = g * a.rep + unit % a.rep;
    const int wkv = kv_of(rb);
    const int row = min(rb * 32 + r32, a.seq - 1);  // rows past seq repeat the last one, never stored
    const int limit = a.cache_len + row + 1;        // positions this lane's row sees

    const float *kb = a.cache_k + (size_t)g * a.cap * dk;
    const float *vb = a.cache_v + (size_t)g * a.cap * dk;
    const int kvmax = kv_of(last / a.rep);

    // A thread stages pieces of 16 bytes (dimensions c .. c + 3) of positions p0, p0
    // + PS, ... of K, then of V (the same registers). Positions past the last
    // repeat it: their weights are 0 and V is staged finite.
    constexpr int PS = T / (DK / 4);
    static_assert(T % (DK / 4) == 0 || DK == 96, "a thread's pieces share their dimensions");
    v4f st[PER];
    auto piece = [&](int i, int &p, int &c) {
        if (DK == 96) {
            const int e = threadIdx.x + T * i;
            p = e / (DK / 4);
            c = e % (DK / 4) * 4;
        } else {
            p = (int)threadIdx.x / (DK / 4) + PS * i;
            c = (int)threadIdx.x % (DK / 4) * 4;
        }
    };
    auto load_tile = [&](const float *src, int t) {
#pragma unroll
        for (int i = 0; i < PER; i++) {
            int p, c;
            piece(i, p, c);
            const uint32_t pos = (uint32_t)min(t * kFlashTile + p, kvmax - 1);
            // 32-bit byte offsets: one head's rows stay below 4 GiB
            st[i] = *(const v4f *)((const char *)src + (pos * (uint32_t)dk + (uint32_t)(FULL ? c : min(c, dk - 4))) * 4u);
        }
    };
    auto store_k = [&](int b) {
#pragma unroll
        for (int i = 0; i < PER; i++) {
            int p, c;
            piece(i, p, c);
            const v4f z = {0.0f, 0.0f, 0.0f, 0.0f};
            *(v4f *)(ktile(b) + p * KS + c) = FULL || c < dk ? st[i] : z;
        }
    };
    auto store_v = [&](int b, unsigned *bm) {
#pragma unroll
        for (int i = 0; i < PER; i++) {
            int p, c;
            piece(i, p, c);
            bool bad = false;
            v4f v = st[i];
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const bool fin = __builtin_isfinite(v[k]);
                bad |= !fin;
                v[k] = fin ? v[k] : 0.0f;
            }
            *(v4f *)(vtile(b) + p * KS + c) = v;
            if (bad) atomicOr(bm, 1u << p);
        }
    };

    // this lane's half of its query row
    v4f q[HD / 4];
    {
        const float *qr = a.qrot + ((size_t)row * a.n_heads + hq) * dk + HD * h;
#pragma unroll
        for (int j = 0; j < HD / 4; j++) {
            const v4f z = {0.0f, 0.0f, 0.0f, 0.0f};
            q[j] = FULL || HD * h + 4 * j < dk ? *(const v4f *)(qr + 4 * j) : z;
        }
    }
    v16f o[DT];
#pragma unroll
    for (int t = 0; t < DT; t++)
#pragma unroll
        for (int v = 0; v < 16; v++) o[t][v] = 0.0f;
    float m = -INFINITY, l = 0.0f;

    if (threadIdx.x < 3) badm[threadIdx.x] = 0;
    load_tile(kb, t0);
    store_k(0);
    load_tile(vb, t0);
    __syncthreads();
    store_v(0, badm);
    __syncthreads();
    int b3 = 0;  // (t - t0) % 3
    for (int t = t0; t < t1; t++, b3 = b3 == 2 ? 0 : b3 + 1) {
        const int b = (t - t0) & 1;
        if (threadIdx.x == 0) badm[b3 == 0 ? 2 : b3 - 1] = 0;  // the tile before's, read by all
        const bool more = t + 1 < t1, work = t * kFlashTile < wkv;
        v16f s = {};
        if (more) load_tile(kb, t + 1);
        if (work) {
            // S^T: rows = positions, columns = query rows
            const float *kt = ktile(b) + r32 * KS + HD * h;
#pragma unroll
            for (int j = 0; j < HD / 4; j++) {
                const v4f kv = *(const v4f *)(kt + 4 * j);
#pragma unroll
                for (int k = 0; k < 4; k++) s = __builtin_amdgcn_mfma_f32_32x32x2f32(kv[k], q[j][k], s, 0, 0, 0);
            }
            // online softmax over the lane's 16 positions and lane ^ 32's
            const int left = limit - t * kFlashTile - 4 * h;  // position index 8 (v / 4) + v % 4 counts if below
            float mt = -INFINITY;
#pragma unroll
            for (int v = 0; v < 16; v++) {
                s[v] = s[v] * a.scale;
                if (8 * (v >> 2) + (v & 3) < left) mt = fmaxf(mt, s[v]);
            }
            mt = fmaxf(mt, __shfl_xor(mt, 32, 64));
            const float mn = fmaxf(m, mt);
            const bool any = limit > t * kFlashTile;  // this row sees some position of the tile
            // the first positions a row meets: exp(-inf) = 0 exactly
            float alpha = 1.0f;
            if (any && !(m == mn)) alpha = (m == -INFINITY && mn < INFINITY) ? 0.0f : (float)exp((double)(m - mn));
            // while every score so far is -inf a position weighs exp(-inf) = 0 (not exp(-inf + inf))
            const float ref = mn == -INFINITY ? 0.0f : mn;
            float es = 0.0f;
#pragma unroll
            for (int v = 0; v < 16; v++) {
                const bool in = 8 * (v >> 2) + (v & 3) < left;
                const float e = exp_neg(s[v] - ref);
                s[v] = in ? e : 0.0f;
                es = es + s[v];
            }
            es = es + __shfl_xor(es, 32, 64);
            if (any) {
                l = l * alpha + es;
                m = mn;
            }
            if (__ballot(alpha != 1.0f)) {
#pragma unroll
                for (int tt = 0; tt < DT; tt++)
#pragma unroll
                    for (int v = 0; v < 16; v++) o[tt][v] = o[tt][v] * alpha;
            }
        }
        // the other buffer is free since the barrier at the end of the tile before
        if (more) {
            store_k(b ^ 1);
            load_tile(vb, t + 1);
        }
        if (work) {
            // O^T += V^T P^T
            const float *vt = vtile(b) + 4 * h * KS + r32;
#pragma unroll
            for (int v = 0; v < 16; v++) {
                const float *vp = vt + (8 * (v >> 2) + (v & 3)) * KS;
#pragma unroll
                for (int tt = 0; tt < DT; tt++)
                    o[tt] = __builtin_amdgcn_mfma_f32_32x32x2f32(vp[32 * tt], s[v], o[tt], 0, 0, 0);
            }
            // non-finite V elements of the tile, for the rows that see them
            unsigned bad = badm[b3];
            while (bad) {
                const int p = __builtin_ctz(bad);
                bad &= bad - 1;
                const int want = (p & 3) + 4 * (p >> 3), ph = (p >> 2) & 1;  // accumulator and lane half of position p
                float w = 0.0f;
#pragma unroll
                for (int v = 0; v < 16; v++) w = v == want ? s[v] : w;
                w = __shfl(w, r32 + 32 * ph, 64);
                const float *vrow = vb + (size_t)(t * kFlashTile + p) * dk;
                if (t * kFlashTile + p < limit) {
#pragma unroll
                    for (int tt = 0; tt < DT; tt++)
#pragma unroll
                        for (int v = 0; v < 16; v++) {
                            const int d = 32 * tt + 8 * (v >> 2) + 4 * h + (v & 3);
                            const float x = d < dk ? vrow[d] : 0.0f;
                            if (!__builtin_isfinite(x)) o[tt][v] = __builtin_fmaf(w, x, o[tt][v]);
                            __builtin_amdgcn_sched_barrier(0);  // rare path: one load at a time, few registers
                        }
                }
            }
        }
        if (more) store_v(b ^ 1, &badm[b3 == 2 ? 0 : b3 + 1]);
        __syncthreads();
    }

    if (!mine) return;
    const int qi = rb * 32 + r32;
    const bool live = qi < a.seq;
    if (tiles <= f.chunk) {
        const float inv = 1.0f / l;
        float *dst = a.out + ((size_t)min(qi, a.seq - 1) * a.n_heads + hq) * dk;
#pragma unroll
        for (int tt = 0; tt < DT; tt++)
#pragma unroll
            for (int v = 0; v < 16; v += 4) {
                const int d = 32 * tt + 2 * v + 4 * h;
                const v4f w = {o[tt][v] * inv, o[tt][v + 1] * inv, o[tt][v + 2] * inv, o[tt][v + 3] * inv};
                if (live && d < dk) *(v4f *)(dst + d) = w;
            }
    } else {
        // this chunk's state: [kv head][group][chunk][wave][row]: d_k values; (max, sum) behind all of them
        const size_t at = ((((size_t)g * f.groups + ug) * f.chunks + ch) * kFlashWaves + wave) * 32 + r32;
        const size_t all = (size_t)a.n_kv * f.groups * f.chunks * kFlashWaves * 32;
        float *dst = a.part + at * dk;
#pragma unroll
        for (int tt = 0; tt < DT; tt++)
#pragma unroll
            for (int v = 0; v < 16; v += 4) {
                const int d = 32 * tt + 2 * v + 4 * h;
                const v4f w = {o[tt][v], o[tt][v + 1], o[tt][v + 2], o[tt][v + 3]};
                if (d < dk) *(v4f *)(dst + d) = w;
            }
        if (h == 0) {
            a.part[all * dk + at * 2] = m;
            a.part[all * dk + at * 2 + 1] = l;
        }
    }
}

// The chunks of one (row, head), half a wave each (four dimensions per lane),
// merged in chunk order as attn_combine_kernel merges splits (rows with one
// chunk are written already). VALU-bound: every lane forms the few chunk weights
// for itself, which is cheaper than one lane forming and handing them round
// (1024 rows of 32 heads, d_k 128: 24.6 us with a wave per pair).
__global__ void __launch_bounds__(256) attn_flash_combine_kernel(AttnArgs a, FlashPlan f) {
    const int lane = threadIdx.x & 31;
    const int pair = blockIdx.x * 8 + (threadIdx.x >> 5);  // qi * n_heads + head
    if (pair >= a.seq * a.n_heads) return;
    const int qi = pair / a.n_heads, hq = pair - qi * a.n_heads;
    const int g = hq / a.rep, dk = a.d_k;
    const int U = (a.seq + 31) / 32 * a.rep;
    const int unit = qi / 32 * a.rep + hq % a.rep;
    const int ug = unit / kFlashWaves, wave = unit % kFlashWaves;
    const int last = min(ug * kFlashWaves + kFlashWaves - 1, U - 1);
    const int kv = a.cache_len + min(a.seq, 32 * (last / a.rep + 1));
    const int tiles = (kv + kFlashTile - 1) / kFlashTile;
    if (tiles <= f.chunk) return;
    // chunks this row sees anything of
    const int n = (a.cache_len + qi) / (flash_chunk(f, tiles) * kFlashTile) + 1;
    const size_t base = (((size_t)g * f.groups + ug) * f.chunks * kFlashWaves + wave) * 32 + qi % 32;
    const size_t step = (size_t)kFlashWaves * 32;  // between chunks
    const v2f *ml = (const v2f *)(a.part + (size_t)a.n_kv * f.groups * f.chunks * step * dk) + base;
    const int d = 4 * lane, dc = d < dk ? d : 0;
    const float *pv = a.part + base * dk + dc;
    float M = -INFINITY;
#pragma unroll 4
    for (int c = 0; c < n; c++) M = fmaxf(M, ml[c * step].x);
    float L = 0.0f;
    v4f O = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 4
    for (int c = 0; c < n; c++) {
        const v2f s = ml[c * step];
        const v4f v = *(const v4f *)(pv + c * step * dk);
        const float w = s.x != -INFINITY ? exp_neg(s.x - M) : 0.0f;
        L = L + s.y * w;
        O = O + v * w;
    }
    const float inv = 1.0f / L;
    if (d < dk) *(v4f *)(a.out + (size_t)pair * dk + d) = O * inv;
}

}  // namespace

namespace {
// hp: q heads per workgroup (rep / head slices)
size_t attn_lds_bytes(int tw, int rep, int hp, int d_k) {
    const int nh = rep > 4 ? rep : 4;
    return ((size_t)tw * kTile * (kChunk + 4) + (size_t)(hp + 2) * d_k + (size_t)tw * hp * (d_k + 2) +
            (size_t)tw * nh * kTile) *
           sizeof(float);
}
// the device's LDS per workgroup (read once)
size_t lds_per_block() {
    static const size_t v = [] {
        int dev = 0, b = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&b, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess || b <= 0)
            return (size_t)64 * 1024;
        return (size_t)b;
    }();
    return v;
}
// the device's CU count (read once)
int cus_per_device() {
    static const int v = [] {
        int dev = 0, c = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&c, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || c <= 0)
            return 256;
        return c;
    }();
    return v;
}
}  // namespace

void attention_plan(int seq, int n_heads, int n_kv, int d_k, int kv_len, int *splits, int *tps, int *tw, int *hs,
                    size_t *ws_bytes) {
    const int tiles = (kv_len + kTile - 1) / kTile;
    const int pairs = seq * n_kv;
    const int rep = n_heads / n_kv, nh = rep > 4 ? rep : 4;
    const Tuning &T = tuning();
    // tile groups per workgroup: at most kMaxWaves waves, and what LDS holds
    int G = kMaxWaves / nh;
    G = G < T.attn_tile_groups ? G : T.attn_tile_groups;
    G = G < tiles ? G : tiles;
    while (G > 1 && attn_lds_bytes(G, rep, rep, d_k) > lds_per_block()) G--;
    G = G < 1 ? 1 : G;
    int S, t;
    if (tiles <= G) {
        // one workgroup per (row, kv head), a tile per group: no combine launch
        S = 1;
        t = 1;
        G = tiles;
    } else {
        // splits of at most two groups (waves that share a SIMD share its
        // VALU), about attn_target_blocks workgroups over the (row, kv head)
        // pairs; more tiles per group only past that
        G = G < 2 ? G : 2;
        S = (T.attn_target_blocks + pairs - 1) / pairs;
        const int smax = (tiles + G - 1) / G;
        S = S < 1 ? 1 : (S > smax ? smax : S);
        t = (tiles + S * G - 1) / (S * G);
        S = (tiles + t * G - 1) / (t * G);
    }
    // head slices (the plan above does not depend on them, so neither do the
    // results): while there are fewer workgroups than CUs, the q heads of a
    // kv head are spread over up to rep / 2 workgroups (two heads or more
    // each), every one reading the kv head's rows for its own heads; a
    // divisor of rep. Measured (decode, 32 q / 8 kv heads, d_k 128): KV 128
    // 10.2 -> 8.8 µs, KV 2047 15.4 -> 14.8 µs; one head per workgroup was
    // slower (9.1 and 21.4 µs)
    int H = T.attn_head_slices;
    if (H <= 0) {
        const int64_t wgs = (int64_t)pairs * S;
        H = (int)((cus_per_device() + wgs - 1) / wgs);
        H = H < rep / 2 ? H : rep / 2;
    }
    H = H < 1 ? 1 : (H > rep ? rep : H);
    while (H > 1 && (rep % H || (int64_t)pairs * H > 65535)) H--;  // grid y: pairs x H
    *splits = S;
    *tps = t;
    *tw = G;
    *hs = H;
    const size_t qrot = (size_t)seq * n_heads * d_k * sizeof(float);
    const size_t part = S > 1 ? (size_t)seq * n_heads * S * (d_k + 2) * sizeof(float) : 0;
    *ws_bytes = ((qrot + 255) & ~(size_t)255) + part;
}

template <bool PREP>
void launch_split(const AttnArgs &a, dim3 grid, size_t lds, hipStream_t s) {
    const dim3 block(64 * (a.rep > 4 ? a.rep : 4) * a.tw);
    switch ((a.d_k + 63) / 64) {
    case 1:
        if (a.d_k == 64) hipLaunchKernelGGL((attn_split_kernel<PREP, 1, true>), grid, block, lds, s, a);
        else hipLaunchKernelGGL((attn_split_kernel<PREP, 1, false>), grid, block, lds, s, a);
        break;
    case 2:
        if (a.d_k == 128) hipLaunchKernelGGL((attn_split_kernel<PREP, 2, true>), grid, block, lds, s, a);
        else hipLaunchKernelGGL((attn_split_kernel<PREP, 2, false>), grid, block, lds, s, a);
        break;
    case 3: hipLaunchKernelGGL((attn_split_kernel<PREP, 3, false>), grid, block, lds, s, a); break;
    default: hipLaunchKernelGGL((attn_split_kernel<PREP, 4, false>), grid, block, lds, s, a); break;
    }
}

namespace {
sllm_status launch_prep(const AttnArgs &a, bool flash, hipStream_t s) {
    const int heads = a.n_heads + a.n_kv;
    if (flash || a.seq >= kPrepRows)
        hipLaunchKernelGGL(attn_prep_rows_kernel,
                           dim3(a.seq, a.seq >= kPrepRows ? 1 : (heads + kPrepWaves - 1) / kPrepWaves),
                           dim3(64 * kPrepWaves), 0, s, a);
    else
        hipLaunchKernelGGL(attn_prep_kernel, dim3(a.seq, heads), dim3(64), 0, s, a);
    SLLM_HIP(hipGetLastError());
    return SLLM_OK;
}
}  // namespace

namespace {
// (query row, kv head) pairs above which a prompt takes attn_flash_kernel: up to
// there the split kernel's one workgroup per pair all run at once, and its shorter
// chain wins. The fewer tiles of positions a row sees, the fewer tile groups (waves,
// LDS) a workgroup has and the more run side by side; q heads above four per kv head
// make it larger. Head sizes that are no multiple of 64 have the slower form of the
// split kernel. Measured (us, split / matrix cores; q heads / kv heads / d_k, rows +
// cached): 32/32/64 40 12.8 / 13.9, 48 13.9 / 14.1, 64 18.4 / 14.6; 16/16/128 48 10.3
// / 17.5, 64 14.0 / 18.3; 40/40/128 13 + 30 10.3 / 16.9; 32/8/128 72 17.8 / 19.7, 96
// 19.7 / 20.4, 112 25.4 / 21.2, 65 + 100 26.8 / 27.0; 24/8/128 96 19.2 / 20.9; 64/8/128
// 65 25.2 / 21.1; 16/16/80 48 13.5 / 16.0, 64 19.2 / 16.6, 33 + 64 28.5 / 17.0;
// 9/3/64 160 18.8 (split), 171 23.0 / 17.1; 32/4/128 128 22.4 (split), 129 32.8 / 22.6.
int64_t flash_pairs(int rep, int d_k, int kv_len) {
    const bool full = d_k % 64 == 0;
    const int64_t one_tile = full ? 1536 : 768, two = full ? 768 : 512;
    const int64_t n = (kv_len <= kTile ? one_tile : kv_len <= 2 * kTile ? two : 512) * 4 / (rep > 4 ? rep : 4);
    return n > 512 ? n : 512;
}

size_t qrot_bytes(int seq, int n_heads, int d_k) {
    return ((size_t)seq * n_heads * d_k * sizeof(float) + 255) & ~(size_t)255;
}

FlashPlan flash_plan(int seq, int n_heads, int n_kv, int d_k, int cache_len, size_t *part) {
    const int rep = n_heads / n_kv, U = (seq + 31) / 32 * rep;
    FlashPlan f;
    f.groups = (U + kFlashWaves - 1) / kFlashWaves;
    int64_t total = 0;
    int most = 0;
    for (int ug = 0; ug < f.groups; ug++) {
        const int last = ug * kFlashWaves + kFlashWaves - 1 < U - 1 ? ug * kFlashWaves + kFlashWaves - 1 : U - 1;
        const int rows = 32 * (last / rep + 1) < seq ? 32 * (last / rep + 1) : seq;
        most = (cache_len + rows + kFlashTile - 1) / kFlashTile;
        total += most;
    }
    // about two workgroups per resident one (two per CU); few tiles in all are cut
    // to one, two or three each, where a workgroup's fixed cost (first loads, the
    // merge) weighs against the idle CUs. Measured (us, with the exponential in 32 bits;
    // in 64 bits each takes 3 to 5 % more): 32/8/128, 128 rows
    // with chunks of 1 / 3 24.7 / 35.2; 200 rows 1 / 2 / 3 36.7 / 32.2 / 37.8; 512
    // rows 2 / 3 / 5 66.0 / 59.8 / 75.5; 1024 rows 3 / 5 / 9 148 / 139 / 149.7
    const int64_t all = total * n_kv, slots = 2 * (int64_t)tuning().attn_target_blocks;
    const int64_t c = (all + slots - 1) / slots, least = all > 1024 ? 3 : (all > 128 ? 2 : 1);
    f.chunk = (int)(c < least ? least : c);
    // the states' most bytes; calls that the static scratch takes get what it holds
    // beside the q rows, also on a stream's workspace: both give the same bits
    const size_t most_part = qrot_bytes(seq, n_heads, d_k) <= kNoallocBytes ? kStaticScratchBytes - kNoallocBytes
                                                                            : (size_t)256 << 20;
    for (;; f.chunk *= 2) {
        f.chunks = (most + f.chunk - 1) / f.chunk;
        *part = f.chunks > 1 ? (size_t)n_kv * f.groups * f.chunks * kFlashWaves * 32 * (d_k + 2) * sizeof(float) : 0;
        if (*part <= most_part) return f;
    }
}

template <int DT>
void launch_flash_dt(const AttnArgs &a, const FlashPlan &f, hipStream_t s) {
    constexpr size_t lds = (size_t)(4 * kFlashTile * (32 * DT + 4) + 4) * sizeof(float);
    const dim3 grid(a.n_kv, f.groups, f.chunks), block(64 * kFlashWaves);
    if (a.d_k == 32 * DT) hipLaunchKernelGGL((attn_flash_kernel<DT, true>), grid, block, lds, s, a, f);
    else hipLaunchKernelGGL((attn_flash_kernel<DT, false>), grid, block, lds, s, a, f);
}
}  // namespace

bool attention_flash(int seq, int n_heads, int n_kv, int d_k, int cache_len, const float *out, size_t *ws_bytes) {
    if ((int64_t)seq * n_kv <= flash_pairs(n_heads / n_kv, d_k, cache_len + seq) || d_k > 128 || ((uintptr_t)out & 15) != 0) return false;
    size_t part = 0;
    const FlashPlan f = flash_plan(seq, n_heads, n_kv, d_k, cache_len, &part);
    if (f.groups > 65535 || f.chunks > 65535) return false;  // grid y, z
    *ws_bytes = qrot_bytes(seq, n_heads, d_k) + part;
    return true;
}

sllm_status launch_attention_flash(const AttnArgs &a, hipStream_t s) {
    size_t part = 0;
    const FlashPlan f = flash_plan(a.seq, a.n_heads, a.n_kv, a.d_k, a.cache_len, &part);
    const sllm_status st = launch_prep(a, true, s);
    if (st != SLLM_OK) return st;
    switch ((a.d_k + 31) / 32) {
    case 1: launch_flash_dt<1>(a, f, s); break;
    case 2: launch_flash_dt<2>(a, f, s); break;
    case 3: launch_flash_dt<3>(a, f, s); break;
    default: launch_flash_dt<4>(a, f, s); break;
    }
    SLLM_HIP(hipGetLastError());
    if (f.chunks > 1) {
        hipLaunchKernelGGL(attn_flash_combine_kernel, dim3((a.seq * a.n_heads + 7) / 8), dim3(256), 0, s, a, f);
        SLLM_HIP(hipGetLastError());
    }
    return SLLM_OK;
}

sllm_status launch_attention(const AttnArgs &a, hipStream_t s) {
    if (a.hs < 1 || a.rep % a.hs) return set_error(SLLM_ERR_ARG, "attention: head slices must divide rep");
    const size_t lds = attn_lds_bytes(a.tw, a.rep, a.rep / a.hs, a.d_k);
    if (a.seq == 1) {
        AttnArgs b = a;
        b.row0 = 0;
        launch_split<true>(b, dim3(a.splits, a.n_kv * a.hs), lds, s);
        SLLM_HIP(hipGetLastError());
    } else {
        const sllm_status st = launch_prep(a, false, s);
        if (st != SLLM_OK) return st;
        // grid y is (row, kv head, head slice), at most 65535: long prefills
        // run in chunks of rows (every row's k / v is already in the cache)
        const int per = 65535 / (a.n_kv * a.hs);
        if (per < 1) return set_error(SLLM_ERR_SHAPE, "attention: n_kv_heads x head slices exceeds the grid");
        for (int r0 = 0; r0 < a.seq; r0 += per) {
            AttnArgs b = a;
            b.row0 = r0;
            const int rows = a.seq - r0 < per ? a.seq - r0 : per;
            launch_split<false>(b, dim3(a.splits, rows * a.n_kv * a.hs), lds, s);
            SLLM_HIP(hipGetLastError());
        }
    }
    if (a.splits > 1) {
        const int pairs = a.seq * a.n_heads;
        if (a.splits <= kShortSplits)
            hipLaunchKernelGGL(attn_combine_kernel, dim3((pairs + 3) / 4), dim3(256), 0, s, a);
        else
            hipLaunchKernelGGL(attn_combine_long_kernel, dim3(pairs), dim3(64 * kLongWaves),
                               (size_t)kRound * (a.d_k + 1) * sizeof(float), s, a);
        SLLM_HIP(hipGetLastError());
    }
    return SLLM_OK;
}

}  // namespace sllm
