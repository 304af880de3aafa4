// ScaledDotProductAttention / FlashAttention: one head, Q/K [seq, depth],
// V/O [seq, valueDim].
// Reference: device/cpu/attention/ops.go:9-31 (FlashAttention calls
// ScaledDotProductAttention), compute.go:10-29,54-68 (zero seqQ or seqK is a
// no-op; scale = float32(1/sqrt(float64(depth)))), typed_compute.go:31-97 and
// select_flash_amd64.go:133-177 (per row: online softmax over the visible keys
// in order, causal hides key > row, i.e. top-left aligned; exponentials through
// flashExpFloat32, flash_attention.go:171-189, which is FastExp32 with -inf and
// anything below -88 mapped to 0; output acc * (1/normalizer), zeros when the
// normalizer is 0).  16-bit dots are rounded to the 16-bit format.
//
// General kernel: one wave64 per query row.  Each lane scores one key of a
// 64-key chunk; the chunk's keys are then folded into the running (max,
// normalizer, acc) one at a time, in key order, with the reference's exact
// sequence of exponentials (FastExp32's error is ~1e-5 relative, so regrouping
// the rescales would move f32 results by more than their tolerance); lanes own
// the output dims.  bf16 / f16 with depth = valueDim a multiple of 8 up to 256 runs
// on the MFMA prefill kernel with one head and shift 0 (hardware exp2 in place of
// FastExp32; the difference is far below bf16 / f16 resolution).
#include "attention.hpp"
#include <algorithm>

namespace puter {

struct FlashArgs {
    const void *q, *k, *v;
    void *o;
    int64_t seq_q, seq_k, depth, value_dim;
    int causal;
    float scale;
};

constexpr int64_t kFlashMaxDepth = 8192;     // Q row staged in LDS as f32 (32 KB)
constexpr int64_t kFlashMaxValueDim = 1024;  // 16 output dims per lane

__device__ __forceinline__ float flash_exp(float v) {
    if (v != v) return v;
    if (v < -88.0f) return 0.0f;  // includes -inf
    if (isinf(v)) return INFINITY;
    return fast_exp32(v);
}

template <int DT>
__global__ __launch_bounds__(64) void flash_generic_kernel(FlashArgs a) {
    using T = typename Elem<DT>::T;
    constexpr int NV = kFlashMaxValueDim / kWave;
    extern __shared__ float qrow[];
    const int64_t r = blockIdx.x;
    const int lane = threadIdx.x;
    const T *Q = reinterpret_cast<const T *>(a.q) + r * a.depth;
    const T *K = reinterpret_cast<const T *>(a.k);
    const T *V = reinterpret_cast<const T *>(a.v);
    T *O = reinterpret_cast<T *>(a.o) + r * a.value_dim;
    for (int64_t d = lane; d < a.depth; d += kWave) qrow[d] = Elem<DT>::load(Q[d]);
    __syncthreads();
    const int64_t k_hi = a.causal ? min(a.seq_k, r + 1) : a.seq_k;
    float m = -INFINITY, l = 0.0f;
    float acc[NV];
#pragma unroll
    for (int j = 0; j < NV; ++j) acc[j] = 0.0f;
    for (int64_t c0 = 0; c0 < k_hi; c0 += kWave) {
        // lane t scores key c0 + t (sequential f32 dot over depth)
        float s = -INFINITY;
        if (c0 + lane < k_hi) {
            const T *kr = K + (c0 + lane) * a.depth;
            float dot = 0.0f;
            for (int64_t d = 0; d < a.depth; ++d) dot += qrow[d] * Elem<DT>::load(kr[d]);
            s = round_reduction<DT>(dot) * a.scale;
        }
        // the keys of the chunk, in order, exactly as the reference's per-key loop
        const int n = (int)min((int64_t)kWave, k_hi - c0);
        for (int t = 0; t < n; ++t) {
            const float score = __shfl(s, t, kWave);
            const float old = m;
            if (score > m) m = score;
            const float alpha = flash_exp(old - m);
            const float shifted = flash_exp(score - m);
            l = l * alpha + shifted;
            const T *vr = V + (c0 + t) * a.value_dim;
#pragma unroll
            for (int j = 0; j < NV; ++j) {
                const int64_t d = lane + kWave * j;
                if (d < a.value_dim) acc[j] = acc[j] * alpha + Elem<DT>::load(vr[d]) * shifted;
            }
        }
    }
    const float inv = l != 0.0f ? 1.0f / l : 0.0f;
#pragma unroll
    for (int j = 0; j < NV; ++j) {
        const int64_t d = lane + kWave * j;
        if (d < a.value_dim) O[d] = Elem<DT>::store(l != 0.0f ? acc[j] * inv : 0.0f);
    }
}

// ------------------------------------------------- three-pass form (MFMA) --
// f32, and the 16-bit head sizes that the MFMA prefill kernel does not take: the scores of
// a block of query rows in the library's scratch, the rows turned into weights, the weights
// times V.  The general kernel above walks one row's keys one at a time (2048 x 2048 x 64
// f32 1246 us); here the two products run on v_mfma_f32_32x32x2_f32 and a row's keys are
// spread over a block.  The exponentials are the reference's own, each evaluated at the
// same argument: with M_j the running maximum after key j and alpha_j = exp(M_(j-1) - M_j)
// the reference's rescale, key j ends up with the weight
//     exp(s_j - M_j) * product of alpha_i over i > j,
// so a prefix maximum and a suffix product over the row give the weights in any order of
// evaluation (only the rounding of the products and of the sum differs).  Measured, the
// error against float64 unchanged in each: f32 2048 x 2048 x 64 1249 -> 41 us (scores 16.5,
// weights 12, product 13.5; the three are bound by their passes over the 16 MB of scores,
// which are written non-temporally, 44.3 -> 41, and by the float32 MFMA rate, 3.5 us a
// product), 1000 x 1000 x 512 f32 2488 -> 59, bf16 2334 -> 88; 64 x 64 x 64 38 -> 13; below
// 64 keys the general kernel runs.  Scores from a tile staged in LDS: 43.5 against 44.3 at
// depth 64, but 74 against 60 at 1000 x 1000 x 512.

// S[r, k] = Q[q0 + r] . K[k] for 32 query rows and 4 x 64 keys a block: wave w owns keys
// 64 w .. + 63 of the block's as two 32 x 32 accumulators.  A lane's operands for four
// MFMA steps are 4 consecutive elements of its row (half h = lane / 32 takes d = 8 g + 4 h
// .. + 3), read straight from memory: Q and K of one head stay in the caches.  VEC: rows
// are whole 4-element pieces at their natural alignment.
typedef float fl_f32x4 __attribute__((ext_vector_type(4)));
typedef float fl_f32x16 __attribute__((ext_vector_type(16)));

template <int DT, bool VEC>
__device__ __forceinline__ float4 flash_load4(const void *row, int64_t d, int64_t depth) {
    using T = typename Elem<DT>::T;
    const T *p = static_cast<const T *>(row) + d;
    if constexpr (VEC) {
        if (d >= depth) return make_float4(0, 0, 0, 0);
        if constexpr (DT == PUTER_F32) return *reinterpret_cast<const float4 *>(p);
        else {
            const uint2 v = *reinterpret_cast<const uint2 *>(p);
            return make_float4(Elem<DT>::load((T)v.x), Elem<DT>::load((T)(v.x >> 16)), Elem<DT>::load((T)v.y),
                               Elem<DT>::load((T)(v.y >> 16)));
        }
    } else {
        float f[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) f[i] = d + i < depth ? Elem<DT>::load(p[i]) : 0.0f;
        return make_float4(f[0], f[1], f[2], f[3]);
    }
}

template <int DT, bool VEC>
__global__ __launch_bounds__(256) void flash_score_kernel(FlashArgs a, float *S, int64_t ld, int64_t q0, int64_t rows) {
    using T = typename Elem<DT>::T;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, l32 = lane & 31, h = lane >> 5;
    const int64_t r0 = (int64_t)blockIdx.y * 32, k0 = ((int64_t)blockIdx.x * 4 + wave) * 64;
    // (causal: keys past the block's last row are masked in all of it)
    if (k0 >= a.seq_k || (a.causal && k0 > q0 + std::min(r0 + 31, rows - 1))) return;
    const int64_t depth = a.depth;
    const T *q = static_cast<const T *>(a.q) + (q0 + std::min(r0 + l32, rows - 1)) * depth;
    const T *k[2];
#pragma unroll
    for (int n = 0; n < 2; ++n) k[n] = static_cast<const T *>(a.k) + std::min(k0 + 32 * n + l32, a.seq_k - 1) * depth;
    fl_f32x16 acc[2] = {(fl_f32x16){}, (fl_f32x16){}};
    constexpr int U = 4;   // groups of 8 d's in flight
    for (int64_t d0 = 0; d0 < depth; d0 += 8 * U) {
        float4 qv[U], kv[U][2];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int64_t d = d0 + 8 * u + 4 * h;
            qv[u] = flash_load4<DT, VEC>(q, d, depth);
#pragma unroll
            for (int n = 0; n < 2; ++n) kv[u][n] = flash_load4<DT, VEC>(k[n], d, depth);
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int n = 0; n < 2; ++n)
                    acc[n] = __builtin_amdgcn_mfma_f32_32x32x2f32((&qv[u].x)[i], (&kv[u][n].x)[i], acc[n], 0, 0, 0);
    }
    // register j of lane (l32, h): row 8 (j / 4) + 4 h + j % 4, key l32
#pragma unroll
    for (int n = 0; n < 2; ++n) {
        const int64_t key = k0 + 32 * n + l32;
        if (key >= a.seq_k) continue;
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            const int64_t r = r0 + 8 * (j >> 2) + 4 * h + (j & 3);
            if (r < rows) __builtin_nontemporal_store(acc[n][j], S + r * ld + key);
        }
    }
}

// flash_exp for x <= 0 or NaN, without a branch
__device__ __forceinline__ float flash_exp_neg(float x) {
    const float y = fast_exp32_body(x);
    return x < -87.33654f ? 0.0f : x != x ? x : y;
}

// Row r of S becomes its normalised weights, zeros on masked keys and on the columns
// [seq_k, ld).  One block per row; thread t holds the E keys E t .. + E - 1 (E T >= ld).
template <int DT, int E>
__global__ __launch_bounds__(1024) void flash_weights_kernel(FlashArgs a, float *S, int64_t ld, int64_t q0) {
    __shared__ float part[3][16];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6, nw = blockDim.x >> 6;
    float *row = S + (int64_t)blockIdx.x * ld;
    const int64_t k0 = (int64_t)t * E;
    const int64_t k_hi = a.causal ? min(a.seq_k, q0 + (int64_t)blockIdx.x + 1) : a.seq_k;
    float s[E];
#pragma unroll
    for (int j = 0; j < E; j += 4) {   // ld % 4 == 0
        const float4 v = k0 + j < k_hi ? *reinterpret_cast<const float4 *>(row + k0 + j) : make_float4(0, 0, 0, 0);
        s[j] = v.x; s[j + 1] = v.y; s[j + 2] = v.z; s[j + 3] = v.w;
    }
    // the running maximum before this thread's keys (NaN scores never raise it)
    float top = -INFINITY;
#pragma unroll
    for (int j = 0; j < E; ++j) {
        s[j] = round_reduction<DT>(s[j]) * a.scale;
        if (k0 + j < k_hi && s[j] > top) top = s[j];
    }
    float incl = top;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const float up = __shfl_up(incl, o, kWave);
        if (lane >= o) incl = fmaxf(incl, up);
    }
    if (lane == 63) part[0][wave] = incl;
    __syncthreads();
    float m = __shfl_up(incl, 1, kWave);
    if (lane == 0) m = -INFINITY;
    for (int w = 0; w < wave; ++w) m = fmaxf(m, part[0][w]);
    // this thread's keys in order: weight against the running maximum, then the later
    // rescales of its own keys (alpha is 1 wherever the maximum stays)
    float alpha[E];
#pragma unroll
    for (int j = 0; j < E; ++j) {
        const bool seen = k0 + j < k_hi;
        const float old = m;
        if (seen && s[j] > m) m = s[j];
        const bool rescale = seen && (old != m || m == -INFINITY);
        alpha[j] = 1.0f;
        if (__any(rescale)) alpha[j] = rescale ? flash_exp_neg(old - m) : 1.0f;
        s[j] = seen ? flash_exp_neg(s[j] - m) : 0.0f;
    }
    float after = 1.0f;
#pragma unroll
    for (int j = E - 1; j >= 0; --j) {
        s[j] *= after;
        after *= alpha[j];
    }
    // the rescales of all later threads: a suffix product
    float suf = after;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const float dn = __shfl_down(suf, o, kWave);
        if (lane + o < 64) suf *= dn;
    }
    if (lane == 0) part[1][wave] = suf;
    float later = __shfl_down(suf, 1, kWave);
    if (lane == 63) later = 1.0f;
    __syncthreads();
    float all = 1.0f;   // the product of every rescale, which the empty sum at the start gets
    for (int w = 0; w < nw; ++w) {
        all *= part[1][w];
        if (w > wave) later *= part[1][w];
    }
    float l = 0.0f;
#pragma unroll
    for (int j = 0; j < E; ++j) {
        s[j] *= later;
        l += s[j];
    }
    l = wave_sum(l);
    if (lane == 0) part[2][wave] = l;
    __syncthreads();
    l = 0.0f * all;
    for (int w = 0; w < nw; ++w) l += part[2][w];
    const float inv = l != 0.0f ? 1.0f / l : 0.0f;
#pragma unroll
    for (int j = 0; j < E; j += 4)
        if (k0 + j < ld)
            __builtin_nontemporal_store((fl_f32x4){s[j] * inv, s[j + 1] * inv, s[j + 2] * inv, s[j + 3] * inv}, reinterpret_cast<fl_f32x4 *>(row + k0 + j));
}

// O[r, d] = sum over k of W[r, k] V[k, d] for 16 rows and 32 dims a block, its 8 waves
// taking the 16-key groups w, w + 8, .. on v_mfma_f32_16x16x4_f32 and adding their sums in
// LDS in wave order.  Lane (i = lane % 16, q = lane / 16) holds W[r0 + i][k + 4 q .. + 3] (one
// 16-byte load a group) and V[k + 4 q + e][2 i, 2 i + 1] (e < 4), and MFMA (e, j) multiplies
// k + 4 q + e into dim 2 i + j.  A causal block stops at its last row's key; a masked key's
// zero weight times an infinite value is NaN in its products, while the general kernel
// never reads that row, so an output that is not finite is summed again over the row's
// own keys.  (The f32 Matmul in its place, with V widened or padded for it and the result
// narrowed afterwards: 18.5 us against 13.5 at 2048 x 2048 x 64, 19 -> 13 the whole call at 64.)
template <int DT>
__global__ __launch_bounds__(512) void flash_product_kernel(FlashArgs a, const float *W, int64_t ld, int64_t q0, int64_t rows) {
    using T = typename Elem<DT>::T;
    __shared__ float part[8][16][33];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, i = lane & 15, q = lane >> 4;
    const int64_t r0 = (int64_t)blockIdx.x * 16, d0 = (int64_t)blockIdx.y * 32 + 2 * i, vd = a.value_dim;
    const int64_t kend = a.causal ? std::min(a.seq_k, q0 + std::min(r0 + 16, rows)) : a.seq_k;
    const float *w = W + std::min(r0 + i, rows - 1) * ld;
    const T *V = static_cast<const T *>(a.v);
    const bool pair = d0 + 1 < vd, one = d0 < vd;
    fl_f32x4 acc[2] = {(fl_f32x4){}, (fl_f32x4){}};
    constexpr int U = 4;   // groups in flight
    for (int64_t k0 = (int64_t)wave * 16; k0 < kend; k0 += 8 * 16 * U) {
        float4 wv[U];
        float v[U][4][2];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int64_t k = k0 + u * 128 + 4 * q;
            wv[u] = k < kend ? *reinterpret_cast<const float4 *>(w + k) : make_float4(0, 0, 0, 0);   // ld % 4 == 0
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                v[u][e][0] = v[u][e][1] = 0.0f;
                if (k + e < kend) {
                    const T *p = V + (k + e) * vd + d0;
                    if (pair) {   // (8 or 4 bytes at any element)
                        T t[2];
                        __builtin_memcpy(t, p, sizeof(t));
                        v[u][e][0] = Elem<DT>::load(t[0]);
                        v[u][e][1] = Elem<DT>::load(t[1]);
                    } else if (one) v[u][e][0] = Elem<DT>::load(p[0]);
                }
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    // (keys past kend: their weights count as zero against zero values)
                    const float x = k0 + u * 128 + 4 * q + e < kend ? (&wv[u].x)[e] : 0.0f;
                    acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(x, v[u][e][j], acc[j], 0, 0, 0);
                }
    }
    // register g of acc[j]: row 4 q + g, dim 2 i + j
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int g = 0; g < 4; ++g) part[wave][4 * q + g][2 * i + j] = acc[j][g];
    __syncthreads();
    const int row = threadIdx.x >> 5, col = threadIdx.x & 31;
    float t = part[0][row][col];
#pragma unroll
    for (int x = 1; x < 8; ++x) t += part[x][row][col];
    const int64_t r = r0 + row, d = (int64_t)blockIdx.y * 32 + col;
    if (r >= rows || d >= vd) return;
    if (a.causal && t * 0.0f != 0.0f) {
        t = 0.0f;
        const int64_t k_hi = std::min(a.seq_k, q0 + r + 1);
        for (int64_t k = 0; k < k_hi; ++k) t += W[r * ld + k] * Elem<DT>::load(V[k * vd + d]);
    }
    static_cast<T *>(a.o)[(q0 + r) * vd + d] = Elem<DT>::store(t);
}

constexpr int64_t kFlashScores = (int64_t)64 << 20;   // bytes of scores held at once
constexpr int64_t kFlashMaxKeys = 16384;              // a row's keys in one block's registers

// The most keys that a row sees.
static int64_t flash_visible(const FlashArgs &a) { return a.causal ? std::min(a.seq_k, a.seq_q) : a.seq_k; }

// Returns false when the general kernel is to run: few keys (a step of its key loop is 0.55 us
// at 64 dims, three launches about 10: causal 4 x 1000 x 64 f32 4.9 us against 11.8, 16 x 1000
// level, 24 x 1000 15.8 against 12.5; in bf16, whose large heads cost the scores more, level at
// 30 keys), rows past a block, a stream capture (graphs of these calls may replay side by
// side), or no room.
template <int DT>
static bool run_flash_passes(const FlashArgs &a, hipStream_t s, int *status) {
    if (a.seq_k < 64 || a.seq_k > kFlashMaxKeys || flash_visible(a) < (DT == PUTER_BF16 ? 30 : 18)) return false;
    const int64_t ld = (a.seq_k + 3) / 4 * 4;
    const int64_t chunk = std::min<int64_t>(a.seq_q, std::max<int64_t>(32, kFlashScores / (ld * 4) / 32 * 32));
    const size_t need = (size_t)(chunk * ld) * sizeof(float);
    if (scratch_capturing(s)) return false;
    ScratchLease lease(need, s, true);
    if (lease.status()) return false;
    float *S = static_cast<float *>(lease.ptr());
    const uintptr_t align = DT == PUTER_F32 ? 15 : 7;
    const bool vec = a.depth % 4 == 0 && ((reinterpret_cast<uintptr_t>(a.q) | reinterpret_cast<uintptr_t>(a.k)) & align) == 0;
    for (int64_t q0 = 0; q0 < a.seq_q; q0 += chunk) {
        const int64_t rows = std::min(chunk, a.seq_q - q0);
        const dim3 grid((unsigned)((a.seq_k + 255) / 256), (unsigned)((rows + 31) / 32));
        if (vec) flash_score_kernel<DT, true><<<grid, 256, 0, s>>>(a, S, ld, q0, rows);
        else flash_score_kernel<DT, false><<<grid, 256, 0, s>>>(a, S, ld, q0, rows);
        const int E = ld <= 256 * 4 ? 4 : ld <= 1024 * 8 ? 8 : 16;
        const unsigned T = (unsigned)((ld + E - 1) / E + 63) / 64 * 64;
        if (E == 4) flash_weights_kernel<DT, 4><<<(unsigned)rows, T, 0, s>>>(a, S, ld, q0);
        else if (E == 8) flash_weights_kernel<DT, 8><<<(unsigned)rows, T, 0, s>>>(a, S, ld, q0);
        else flash_weights_kernel<DT, 16><<<(unsigned)rows, T, 0, s>>>(a, S, ld, q0);
        flash_product_kernel<DT><<<dim3((unsigned)((rows + 15) / 16), (unsigned)((a.value_dim + 31) / 32)), 512, 0, s>>>(a, S, ld, q0, rows);
    }
    const int rc = check_launch("flash attention");
    const int fin = lease.finish();
    *status = rc ? rc : fin;
    return true;
}

static int run_flash(const puter_flash_config *config, const void *q, const void *k,
                     const void *v, void *o, int64_t seq_q, int64_t seq_k, int64_t depth,
                     int64_t value_dim, int dtype, hipStream_t s) {
    if (!config) return fail(PUTER_ERR_NIL, "flash attention: nil config");
    if (!is_norm_dtype(dtype)) return fail(PUTER_ERR_INVALID, "flash attention: unsupported dtype %d", dtype);
    if (seq_q < 0 || seq_k < 0 || depth < 0 || value_dim < 0)
        return fail(PUTER_ERR_INVALID, "flash attention: negative shape");
    if (seq_q == 0 || seq_k == 0 || value_dim == 0) return PUTER_OK;
    if (depth == 0) return fail(PUTER_ERR_INVALID, "flash attention: depth must be positive");
    if (depth > kFlashMaxDepth || value_dim > kFlashMaxValueDim)
        return fail(PUTER_ERR_INVALID, "flash attention: depth %lld / value dim %lld above %lld / %lld",
                    (long long)depth, (long long)value_dim, (long long)kFlashMaxDepth,
                    (long long)kFlashMaxValueDim);
    if (seq_q > 0x7FFFFFFF) return fail(PUTER_ERR_INVALID, "flash attention: grid too large");
    if (!q || !k || !v || !o) return fail(PUTER_ERR_NIL, "flash attention: nil buffer");
    const float scale = (float)(1.0 / sqrt((double)depth));
    FlashArgs a{q, k, v, o, seq_q, seq_k, depth, value_dim, config->causal ? 1 : 0, scale};
    // (bf16 head sizes other than 64 and 128 over one to three keys: a padded tile costs more
    // than the general kernel's few steps, 2 x 1 x 40 3.2 us against 3.8, 2 x 3 x 256 8.5 against 8.7)
    const bool few = dtype == PUTER_BF16 && depth != 64 && depth != 128 && flash_visible(a) <= (depth > 128 ? 3 : 2);
    if ((dtype == PUTER_BF16 || dtype == PUTER_F16) && value_dim == depth && !few) {
        MhaArgs m{q, k, v, o, 1, seq_q, seq_k, 1, 1, depth, config->causal ? 1 : 0, 0, 0.0f, scale, 0};
        m.nan_rows = 1;
        int status = PUTER_OK;
        if (launch_prefill_mfma(m, dtype, s, &status)) return status;
    }
    const size_t lds = sizeof(float) * (size_t)depth;
    {
        int status = PUTER_OK;
        const bool done = dtype == PUTER_F32   ? run_flash_passes<PUTER_F32>(a, s, &status)
                          : dtype == PUTER_BF16 ? run_flash_passes<PUTER_BF16>(a, s, &status)
                                                : run_flash_passes<PUTER_F16>(a, s, &status);
        if (done) return status;
    }
    switch (dtype) {
    case PUTER_F32: flash_generic_kernel<PUTER_F32><<<(unsigned)seq_q, kWave, lds, s>>>(a); break;
    case PUTER_BF16: flash_generic_kernel<PUTER_BF16><<<(unsigned)seq_q, kWave, lds, s>>>(a); break;
    case PUTER_F16: flash_generic_kernel<PUTER_F16><<<(unsigned)seq_q, kWave, lds, s>>>(a); break;
    }
    return check_launch("flash attention");
}

}  // namespace puter

using namespace puter;

extern "C" {

int puter_hip_scaled_dot_product_attention(const puter_flash_config *config, const void *query,
                                           const void *key, const void *value, void *output,
                                           int64_t seq_q, int64_t seq_k, int64_t depth,
                                           int64_t value_dim, int dtype, void *stream) {
    return run_flash(config, query, key, value, output, seq_q, seq_k, depth, value_dim, dtype,
                     as_stream(stream));
}

int puter_hip_flash_attention(const puter_flash_config *config, const void *query,
                              const void *key, const void *value, void *output, int64_t seq_q,
                              int64_t seq_k, int64_t depth, int64_t value_dim, int dtype,
                              void *stream) {
    return run_flash(config, query, key, value, output, seq_q, seq_k, depth, value_dim, dtype,
                     as_stream(stream));
}

}  // extern "C"
