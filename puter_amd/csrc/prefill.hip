// MFMA flash-attention prefill: bf16 or f16 Q/K/V (prefill_kernel<dtype, head
// dim, window>; f32 Q/K/V on prefill_f32_kernel, described where it is defined),
// f32 accumulation, output in the input format, head_dim 128 or 64 (tuned) or any multiple
// of 8 up to 256 (4 in f32; rows padded with zero chunks in LDS, see PfDim), GQA,
// optional causal mask: key k is visible to query q when
// k <= q + shift.  MultiHeadAttention passes shift = seqK - seqQ (bottom-right
// aligned, device/cpu/attention/typed_compute.go:166-168);
// ScaledDotProductAttention passes 0 (typed_compute.go:60-62).  Optional
// sliding window: key k is visible to query q only when q - k < window
// (typed_compute.go:172); a block skips the key tiles below its first query's
// window and masks those below its last query's.  Optional ALiBi: the score
// gains slope * (k - q) (typed_compute.go:176-178); every tile then takes the
// masked step.
//
// Work split: one 256-thread block (4 wave64s) per (128-query tile, head,
// batch); wave w owns 32 queries; two blocks share a CU (2 waves per SIMD, so
// one wave's softmax VALU work overlaps the other's MFMAs).  K/V stream
// through LDS in 64-key tiles, double buffered.  The tiles are copied
// straight from HBM into LDS by buffer_load ... lds (no register staging, no
// LDS write instructions): the next tile's copy is issued while the current
// tile's first MFMAs run and waited for (vmcnt) only at the tile's closing barrier.
// The buffer descriptors' range ends with the last row of the sequence, so
// rows past the end arrive as zeros.  The wave index is read through
// readfirstlane so all per-wave control flow is scalar.
//
// LDS layouts (one tile of 64 key rows each, no padding; 256-byte rows at head
// dim 128, 128-byte rows at 64): K row r keeps its 16-byte chunk c at position
// c ^ kswz(r) and V row r at c ^ vswz(r) (PfDim below); both swizzles make the
// fragment reads below bank-conflict free.  The V^T
// operand is read from the row-major V tile with ds_read_b64_tr_b16: within a
// 16-lane group, result lane i gets element i%4 of the 8 bytes addressed by
// lane 4j + i/4 as its element j, so lanes 4j..4j+3 pointing at four 4-dim
// runs of key row j deliver dims 0..15 of keys 0..3 transposed.
//
// Everything is computed transposed so the softmax needs no cross-lane
// reductions beyond one permlane32 swap between the two half-waves:
//   S^T[key, q] = K . Q^T        (v_mfma_f32_32x32x16_bf16, A = K from LDS,
//                                 B = Q^T held in registers for the whole loop)
// The 32x32 accumulator puts query q = lane%32 in every register of a lane,
// so a row max / row sum is an in-lane reduction over the lane's 16 keys plus
// one swap.  exp2 runs on the scaled scores; P^T, narrowed to bf16 in
// registers, is already in the B-operand layout of
//   O^T[d, q] += V^T . P^T       (A = V^T read from a transposed LDS tile)
// because the accumulator's key order (8*(r/4) + 4*(lane/32) + r%4) is used as
// the k-order of both operands.
//
// Online softmax with a lazy rescale: each query keeps a reference maximum m
// (scaled log2 domain) and p = exp2(s*c - m).  O and l are rescaled only when
// some query of the wave sees a score more than 2^8 above its reference
// (wave-uniform branch, rare after the first tiles); otherwise p may exceed 1
// by at most 2^8, which f32 accumulation and bf16 P absorb exactly as well.
// The tile max is not even computed on the common path: p is evaluated against
// the current reference and, as every p is at most its lane's partial row sum,
// a sum <= 2^8 proves no score crossed the threshold; only otherwise is the max
// taken and p redone.  The final O / l is the same softmax.
//
// The mask-free tiles are software-pipelined inside each wave
// (prefill_step_pipelined): the softmax VALU work of one 32-key chunk is
// interleaved with the MFMAs of the next phase (S of the other chunk, or P.V),
// and the K / V^T fragment reads run ahead of the MFMAs that use them, so a
// wave keeps the matrix core busy through its own softmax instead of leaving
// that to the SIMD's other wave (+8-9% on B4 S4096 causal bf16 against the
// unpipelined step, both timed in one process).
//
// Causal blocks visit only the key tiles at or below their diagonal.  Tiles
// that no query of the block needs masked run a mask-free loop; the few tiles
// on the diagonal (and the sequence tail) run a masked loop.  Blocks are
// dispatched heaviest-first, and the block -> (batch, head) map puts the query
// heads that share a kv head on the same XCD (consecutive block ids go
// round-robin over the 8 XCDs), so the K/V tiles they re-read hit that XCD's L2.
#include "attention.hpp"

#include <climits>
#include <cmath>
#include <type_traits>

namespace puter {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));

// element, fragment types and MFMA of the two 16-bit formats
template <int DT> struct PfFormat;
template <> struct PfFormat<PUTER_BF16> {
    using E = __bf16;
    using V8 = bf16x8;
    using V4 = bf16x4;
};
template <> struct PfFormat<PUTER_F16> {
    using E = _Float16;
    using V8 = f16x8;
    using V4 = f16x4;
};
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

namespace fa {
constexpr int BM = 128;       // queries per block (4 waves x 32)
constexpr int BN = 64;        // keys per tile
constexpr float RESCALE_SLACK = 8.0f;   // log2 headroom before O and l are rescaled
constexpr float RESCALE_LIMIT = 256.0f; // 2^RESCALE_SLACK: the largest p allowed
// buffer descriptor word 3 for raw (untyped, stride 0) dword access on gfx9
constexpr int BUF_WORD3 = 0x00020000;
constexpr int OOB = 0x7FFFFFF0;  // an offset past every descriptor's range
}  // namespace fa

// Layout of the K / V tiles for head dims up to D (D = 64, 96, 128 or 256; 16-bit
// elements).  Rows are 128, 256 or 512 bytes (8, 16 or 32 chunks of 16 bytes), the
// power of two that holds D, so a lane's row and chunk are a shift and a mask; a head
// dim below D (any multiple of 8) leaves the chunks past it zero, and 96 computes 6 of
// a 128-row's 8 k-steps and 3 of its 4 output blocks.  K row r keeps chunk c at
// c ^ kswz(r): with rows of 256 bytes or more kswz = r % 16, with 128-byte rows (two
// rows per 64-bank line) kswz = (r / 2) % 8, so the 16 rows a fragment read touches
// fall on distinct banks either way.  V row r keeps chunk c at c ^ vswz(r): 4 (r % 4)
// for rows of 256 bytes or more, 4 ((r / 2) % 2) for 128-byte rows, so the four rows x 32
// bytes of each transposing read (and the rows two apart that share a bank
// line) do not collide.  Both swizzles are unchanged by row offsets of 8, 16
// and 32, which the fragment reads add to a base row.
template <int D> struct PfDim {
    static_assert(D == 256 || D == 128 || D == 96 || D == 64, "head dim 256, 128, 96 or 64");
    static constexpr int RB = D > 128 ? 512 : D > 64 ? 256 : 128;   // row bytes
    static constexpr int NC = RB / 16;         // 16-byte chunks per row
    static constexpr int TILE = fa::BN * RB;   // one K or V tile: 32, 16 or 8 KB
    static constexpr int KS = D / 16;          // S MFMA k-steps (16 dims each)
    static constexpr int DB = D / 32;          // O^T blocks of 32 dims
    static constexpr int RPI = 64 / NC;        // rows per copy instruction (64 lanes x 16 B)
    static constexpr int NI = 16 / RPI;        // copy instructions per wave and tensor
    static constexpr int kswz(int r) { return RB >= 256 ? (r & 15) : ((r >> 1) & 7); }
    static constexpr int vswz(int r) { return RB >= 256 ? ((r & 3) << 2) : (((r >> 1) & 1) << 2); }
};

typedef short i16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void lds_void;
typedef __attribute__((address_space(3))) i16x4 lds_i16x4;

struct PrefillArgs {
    const uint16_t *q, *k, *v;
    uint16_t *o;
    int batch, seq_q, seq_k, heads, kv_heads, qtiles;
    int nan_rows;      // padded kernels: a row with a NaN score is NaN (else zeros)
    int dim;           // head dim: a multiple of 8 (16-bit) or 4 (f32), at most the kernel's D
    int causal, xcd_map;
    int shift;         // causal: key k visible to query q iff k <= q + shift
    int window;        // > 0: key k visible to query q only if k > q - window
    float alibi_s;     // ALiBi slope / scale: the dot gains alibi_s * (k - q) before scaling
    float scale_log2;  // softmax scale * log2(e)
    float scale_log2_lo = 0.0f;  // what scale_log2's rounding left (padded f32 head dims)
    // f32 kernel, key range split over blockIdx.y (split_tiles key tiles each): per
    // split, query row and head the (max, sum) and the unnormalised output row, in
    // [split][batch][query][head] order; null when unsplit
    int split_tiles = 0;
    float2 *part_ml = nullptr;
    float *part_o = nullptr;
};

template <int D> struct PrefillState {
    f32x16 o[D / 32];  // O^T accumulators: lane's query, dims 32d + 8*(r/4) + 4*(lane/32) + r%4
    float m;      // reference max, scaled log2 domain (-inf: none yet)
    float l;      // this lane's half of the row sum
};

__device__ __forceinline__ float swap_halves_max(float t) {
    const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(t), __float_as_uint(t), false, false);
    return fmaxf(__uint_as_float(sw[0]), __uint_as_float(sw[1]));
}
__device__ __forceinline__ float swap_halves_sum(float t) {
    const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(t), __float_as_uint(t), false, false);
    return __uint_as_float(sw[0]) + __uint_as_float(sw[1]);
}

__device__ __forceinline__ void wait_tile_copies() {
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): this wave's HBM -> LDS copies landed
}

// Copy K/V rows [kv0, kv0 + 64) of this head into LDS.  Each copy instruction
// fills RPI consecutive rows (64 lanes x 16 bytes): wave w copies rows
// 4 RPI i + RPI w + lane / NC (i < NI), lane L filling chunk L % NC of its row
// with the row's chunk (L % NC) ^ swizzle(row) (kg / vg hold those byte offsets).
template <int D, bool PAD>
__device__ __forceinline__ void prefill_copy_tile(const PrefillArgs &a, const uint16_t *kbase,
                                                  const uint16_t *vbase, int kv0, const int *kg,
                                                  const int *vg, char *kdst, char *vdst, int wave) {
    using namespace fa;
    using T = PfDim<D>;
    const int dim = PAD ? a.dim : D;
    const int rs2 = a.kv_heads * dim * 2;  // K/V row stride in bytes
    const int rows = min(a.seq_k - kv0, BN);   // <= 0: an empty range, every lane reads zeros
    const int bytes = rows > 0 ? (rows - 1) * rs2 + dim * 2 : 0;
    const int64_t base = rows > 0 ? (int64_t)kv0 * a.kv_heads * dim : 0;
    const __amdgpu_buffer_rsrc_t kd =
        __builtin_amdgcn_make_buffer_rsrc((void *)(kbase + base), (short)0, bytes, BUF_WORD3);
    const __amdgpu_buffer_rsrc_t vd =
        __builtin_amdgcn_make_buffer_rsrc((void *)(vbase + base), (short)0, bytes, BUF_WORD3);
#pragma unroll
    for (int i = 0; i < T::NI; ++i)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(kd, (lds_void *)(kdst + (4 * T::RPI * i + T::RPI * wave) * T::RB), 16,
                                                 kg[i], 0, 0, 0);
#pragma unroll
    for (int i = 0; i < T::NI; ++i)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(vd, (lds_void *)(vdst + (4 * T::RPI * i + T::RPI * wave) * T::RB), 16,
                                                 vg[i], 0, 0, 0);
}

// One 64-key tile for this wave's 32 queries.  masked applies the causal and
// sequence-end mask (diagonal and tail tiles only).  ka / va: this lane's byte
// offsets of its K fragments (per 16-dim step t) and V^T fragments (per
// 32-dim block d) inside a tile.
template <int DT>
__device__ __forceinline__ f32x16 pf_mfma(typename PfFormat<DT>::V8 a, typename PfFormat<DT>::V8 b, f32x16 c) {
    if constexpr (DT == PUTER_BF16) return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
    else return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

// P as MFMA operands: its 16-bit rounding and, with LO, what the rounding left, so that
// hi + lo carries 16 (bf16) or 22 (f16) bits of p.  The head dims that padded rows serve
// take both: their products with V keep the f32 probabilities of the general kernel, which
// is what served these dims before, at half as many MFMAs again (64 and 128 round P once).
template <int DT, bool LO> struct PfLow {
    typename PfFormat<DT>::V8 v;
};
template <int DT> struct PfLow<DT, false> {};
template <int DT, bool LO>
__device__ __forceinline__ void pf_set(typename PfFormat<DT>::V8 &hi, PfLow<DT, LO> &lo, int j, float p) {
    using E = typename PfFormat<DT>::E;
    hi[j] = (E)p;
    if constexpr (LO) lo.v[j] = (E)(p - (float)hi[j]);
}
template <int DT, bool LO>
__device__ __forceinline__ f32x16 pf_pv(typename PfFormat<DT>::V8 v, typename PfFormat<DT>::V8 hi,
                                        const PfLow<DT, LO> &lo, f32x16 c) {
    c = pf_mfma<DT>(v, hi, c);
    if constexpr (LO) c = pf_mfma<DT>(v, lo.v, c);
    return c;
}

template <int DT, int D, bool GEN, bool LO>
__device__ __forceinline__ void prefill_step(const PrefillArgs &a, const char *ks, const char *vs,
                                             const typename PfFormat<DT>::V8 (&qf)[PfDim<D>::KS], PrefillState<D> &st,
                                             int qi, int kv0, const int (&ka)[PfDim<D>::KS],
                                             const int (&va)[PfDim<D>::DB], int g, bool masked) {
    using namespace fa;
    using T = PfDim<D>;
    using V8 = typename PfFormat<DT>::V8;
    // S^T chunks: keys kv0 + 32c + (8*(r/4) + 4g + r%4), query qi; two
    // independent accumulation chains interleaved
    f32x16 s[2] = {(f32x16){}, (f32x16){}};
#pragma unroll
    for (int t = 0; t < T::KS; ++t)
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            const V8 kf = *reinterpret_cast<const V8 *>(ks + c * 32 * T::RB + ka[t]);
            s[c] = pf_mfma<DT>(kf, qf[t], s[c]);
        }
    if constexpr (DT == PUTER_F16) {
        // f16 dots are rounded to f16 as the reference's typed row dot does
        // (attention/typed_compute.go:16-20); bf16 keeps the f32 dot
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int r = 0; r < 16; ++r) s[c][r] = (float)(_Float16)s[c][r];
    }
    if (masked) {
        // key kv0 + 32c + 8(r/4) + 4g + r%4 is visible iff its offset past
        // kv0 + 4g lies in [lo, lim] (the query's first and last visible keys,
        // relative; the first is the sliding window's lower edge, GEN only).  GEN
        // also adds the ALiBi bias slope * (k - q) (as alibi_s * (k - q) before the
        // scale), after the f16 rounding of the dot, as the reference adds it to
        // the scaled score (typed_compute.go:176-178)
        const int last = a.causal ? min(qi + a.shift, a.seq_k - 1) : a.seq_k - 1;
        const int lim = last - kv0 - 4 * g;
        const bool win = GEN && a.window > 0;
        const int lo = win ? qi - a.window + 1 - kv0 - 4 * g : 0;
        if (GEN && a.alibi_s != 0.0f) {
            const float base = (float)(kv0 + 4 * g - qi);
#pragma unroll
            for (int c = 0; c < 2; ++c)
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    s[c][r] += a.alibi_s * (base + (float)(32 * c + 8 * (r >> 2) + (r & 3)));
        }
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int off = 32 * c + 8 * (r >> 2) + (r & 3);
                s[c][r] = (off > lim || (win && off < lo)) ? -INFINITY : s[c][r];
            }
    }
    // Fast path: every lane already has a reference and p = exp2(s*c - m) is
    // evaluated without the tile max; since every p <= the row sum, a sum <= 2^8
    // bounds every p as the max test would.  Otherwise (first tile, or a score
    // far above the reference) the max is taken, O and l rescaled, p redone.
    float psum = 0.0f;
    V8 pf[2][2];
    PfLow<DT, LO> pl[2][2];
    bool done = false;
    if (!__any(st.m == -INFINITY)) {
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(s[c][8 * h + j], a.scale_log2, -st.m));
                    psum += p;
                    pf_set<DT, LO>(pf[c][h], pl[c][h], j, p);
                }
        done = !__any(psum > RESCALE_LIMIT);  // each p of this lane <= its partial sum
    }
    if (!done) {
        float tmax = -INFINITY;
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int r = 0; r < 16; ++r) tmax = fmaxf(tmax, s[c][r]);
        tmax = swap_halves_max(tmax) * a.scale_log2;
        if (__any(tmax > st.m + RESCALE_SLACK)) {
            const float mnew = fmaxf(st.m, tmax);
            const float alpha = st.m == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(st.m - mnew);
            st.m = mnew;
            st.l *= alpha;
#pragma unroll
            for (int d = 0; d < D / 32; ++d)
#pragma unroll
                for (int r = 0; r < 16; ++r) st.o[d][r] *= alpha;
        }
        const float mref = st.m == -INFINITY ? 0.0f : st.m;
        psum = 0.0f;
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(s[c][8 * h + j], a.scale_log2, -mref));
                    psum += p;
                    pf_set<DT, LO>(pf[c][h], pl[c][h], j, p);
                }
    }
    st.l += psum;
    // O^T[d, q] += V^T[d, keys] . P^T[keys, q]: the V^T fragment (dims 32d +
    // lane%32, keys 32c + 16h + 4g + 0..3 and + 8) is two transposing reads
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int d = 0; d < T::DB; ++d) {
                const char *p = vs + (32 * c + 16 * h) * T::RB + va[d];
                const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4 *)(p));
                const i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4 *)(p + 8 * T::RB));
                const V8 vf = __builtin_bit_cast(V8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
                st.o[d] = pf_pv<DT, LO>(vf, pf[c][h], pl[c][h], st.o[d]);
            }
}

// a score dot as the reference's typed row dot leaves it: f16 dots rounded to
// f16 (attention/typed_compute.go:16-20); bf16 keeps the f32 dot
template <int DT> __device__ __forceinline__ float pf_score(float x) {
    if constexpr (DT == PUTER_F16) return (float)(_Float16)x;
    else return x;
}

// Online-softmax update for one 32-key chunk that needs the slow path (first
// tile, or a score more than 2^8 above the reference): take the chunk max,
// rescale O and l if the reference moves, and redo p against it.
template <int DT, int D, bool LO>
__device__ __forceinline__ float prefill_chunk_slow(const PrefillArgs &a, const f32x16 &s, PrefillState<D> &st,
                                                    typename PfFormat<DT>::V8 (&pf)[2], PfLow<DT, LO> (&pl)[2]) {
    using namespace fa;
    float tmax = -INFINITY;
#pragma unroll
    for (int r = 0; r < 16; ++r) tmax = fmaxf(tmax, pf_score<DT>(s[r]));
    tmax = swap_halves_max(tmax) * a.scale_log2;
    if (__any(tmax > st.m + RESCALE_SLACK)) {
        const float mnew = fmaxf(st.m, tmax);
        const float alpha = st.m == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(st.m - mnew);
        st.m = mnew;
        st.l *= alpha;
#pragma unroll
        for (int d = 0; d < D / 32; ++d)
#pragma unroll
            for (int r = 0; r < 16; ++r) st.o[d][r] *= alpha;
    }
    const float mref = st.m == -INFINITY ? 0.0f : st.m;
    float psum = 0.0f;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(pf_score<DT>(s[8 * h + j]), a.scale_log2, -mref));
            psum += p;
            pf_set<DT, LO>(pf[h], pl[h], j, p);
        }
    return psum;
}

// One mask-free 64-key tile, software-pipelined inside the wave so the softmax
// VALU work runs under MFMAs instead of between them:
//   phase 1: S chunk 0 (keys 0..31), 8 MFMAs;
//   phase 2: S chunk 1 MFMAs, each followed by a share of chunk 0's p = exp2(s c - m);
//   phase 3: O += V^T P^T for chunk 0 (8 MFMAs), each followed by a share of chunk 1's p;
//   phase 4: O += V^T P^T for chunk 1.
// The p of a chunk are evaluated against the current reference m; the chunk's
// row-sum check (every p <= its lane's partial sum, so a sum <= 2^8 bounds them
// all) sends it to prefill_chunk_slow otherwise.  Chunk 1's check comes after
// chunk 0's contribution is in O and l, so a rescale there covers it.
// sched_group_barrier fixes the interleave (the scheduler would otherwise
// cluster the MFMAs and the VALU work apart).  The next tile's HBM -> LDS copy
// (rows kvn.., into kn / vn; kvn = seq_k for none) is issued in phases 1 and 2,
// one copy instruction beside every other MFMA, instead of as one burst before
// them (bit-identical; +1-2.5% on B4 S4096 / S2048 causal and non-causal, timed
// interleaved in one process).
template <int DT, int D, bool PAD>
__device__ __forceinline__ void prefill_step_pipelined(const PrefillArgs &a, const char *ks, const char *vs,
                                                       const typename PfFormat<DT>::V8 (&qf)[PfDim<D>::KS],
                                                       PrefillState<D> &st, const int (&ka)[PfDim<D>::KS],
                                                       const int (&va)[PfDim<D>::DB], const uint16_t *kbase,
                                                       const uint16_t *vbase, int kvn, const int (&kg)[PfDim<D>::NI],
                                                       const int (&vg)[PfDim<D>::NI], char *kn, char *vn, int wave) {
    using namespace fa;
    prefill_copy_tile<D, PAD>(a, kbase, vbase, kvn, kg, vg, kn, vn, wave);
    using T = PfDim<D>;
    using V8 = typename PfFormat<DT>::V8;
    constexpr bool LO = PAD;
    constexpr int KS = T::KS, NM = 2 * T::DB;   // S MFMAs per chunk, P.V MFMAs per chunk
    // p values evaluated beside MFMA t of phases 2 and 3: [16 t / KS, 16 (t + 1) / KS) and
    // the same over NM; copy instructions: one where NI (t + 1) / KS steps up
    auto e2 = [](int t) { return 16 * t / KS; };
    auto e3 = [](int t) { return 16 * t / NM; };
    auto cp = [](int t) { return T::NI * (t + 1) / KS - T::NI * t / KS; };
    constexpr int PV = LO ? 6 : 3;              // VALU instructions per p value
    constexpr int RA = KS < 4 ? KS : 4;         // K reads issued ahead of the first S MFMA
    f32x16 s0 = (f32x16){}, s1 = (f32x16){};
    V8 p0[2], p1[2];
    PfLow<DT, LO> l0[2], l1[2];
    const float m = st.m, c = a.scale_log2;
    // phase 1 + 2
#pragma unroll
    for (int t = 0; t < KS; ++t) {
        const V8 kf = *reinterpret_cast<const V8 *>(ks + ka[t]);
        s0 = pf_mfma<DT>(kf, qf[t], s0);
    }
    float ps0 = 0.0f;
#pragma unroll
    for (int t = 0; t < KS; ++t) {
        const V8 kf = *reinterpret_cast<const V8 *>(ks + 32 * T::RB + ka[t]);
        s1 = pf_mfma<DT>(kf, qf[t], s1);
#pragma unroll
        for (int r = e2(t); r < e2(t + 1); ++r) {
            const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(pf_score<DT>(s0[r]), c, -m));
            ps0 += p;
            pf_set<DT, LO>(p0[r >> 3], l0[r >> 3], r & 7, p);
        }
    }
    // K fragment reads run RA ahead of the MFMAs that use them (LDS latency
    // hidden behind the MFMAs in flight)
    __builtin_amdgcn_sched_group_barrier(0x100, RA, 0);      // K reads c0 t0 ..
#pragma unroll
    for (int t = 0; t < KS; ++t) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // S chunk 0 MFMA t
        if (cp(t)) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);   // a K copy
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // next K read (c0, then c1)
    }
#pragma unroll
    for (int t = 0; t < KS; ++t) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // S chunk 1 MFMA t
        if (cp(t)) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);   // a V copy
        if (t < KS - RA) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // remaining K reads of c1
        __builtin_amdgcn_sched_group_barrier(0x002, PV * ((16 + KS - 1) / KS), 0);  // chunk 0 softmax share
    }
    if (__any(ps0 > RESCALE_LIMIT)) ps0 = prefill_chunk_slow<DT, D, LO>(a, s0, st, p0, l0);
    st.l += ps0;
    // phase 3: chunk 0's P.V with chunk 1's softmax between the MFMAs
    const float m1 = st.m;
    float ps1 = 0.0f;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int d = 0; d < T::DB; ++d) {
            const char *p = vs + 16 * h * T::RB + va[d];
            const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4 *)(p));
            const i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4 *)(p + 8 * T::RB));
            const V8 vf = __builtin_bit_cast(V8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
            st.o[d] = pf_pv<DT, LO>(vf, p0[h], l0[h], st.o[d]);
            const int t = T::DB * h + d;
#pragma unroll
            for (int r = e3(t); r < e3(t + 1); ++r) {
                const float pv = __builtin_amdgcn_exp2f(__builtin_fmaf(pf_score<DT>(s1[r]), c, -m1));
                ps1 += pv;
                pf_set<DT, LO>(p1[r >> 3], l1[r >> 3], r & 7, pv);
            }
        }
    // V^T fragment reads (two per MFMA) run two MFMAs ahead
    __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
#pragma unroll
    for (int t = 0; t < NM; ++t) {
        __builtin_amdgcn_sched_group_barrier(0x008, LO ? 2 : 1, 0);  // P.V MFMA (chunk 0)
        if (t < NM - 2) __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, PV * ((16 + NM - 1) / NM), 0);  // chunk 1 softmax share
    }
    if (__any(ps1 > RESCALE_LIMIT)) ps1 = prefill_chunk_slow<DT, D, LO>(a, s1, st, p1, l1);
    st.l += ps1;
    // phase 4: chunk 1's P.V
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int d = 0; d < T::DB; ++d) {
            const char *p = vs + (32 + 16 * h) * T::RB + va[d];
            const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4 *)(p));
            const i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4 *)(p + 8 * T::RB));
            const V8 vf = __builtin_bit_cast(V8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
            st.o[d] = pf_pv<DT, LO>(vf, p1[h], l1[h], st.o[d]);
        }
    __builtin_amdgcn_sched_group_barrier(0x100, 6, 0);
#pragma unroll
    for (int t = 0; t < NM; ++t) {
        __builtin_amdgcn_sched_group_barrier(0x008, LO ? 2 : 1, 0);
        if (t < NM - 3) __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
    }
}

// Byte offsets of a lane's tile copies (source side, swizzled; chunks past the head dim: an
// offset past the buffer's range, read as zeros) and of its fragment reads: K row l32 (+32c),
// chunk (2t + g) ^ kswz(l32); V: lane group q = lane/16, i = lane%16 = 4j + m reads key row
// 4(q/2) + j, dims 16(q%2) + 4m .. +3 of dim block d: chunk (4d + 2(q%2) + m/2) ^ vswz(row),
// half m%2
template <int D>
__device__ __forceinline__ void prefill_offsets(int kv_heads, int dim, int lane, int wave, int (&kg)[PfDim<D>::NI],
                                                int (&vg)[PfDim<D>::NI], int (&ka)[PfDim<D>::KS], int (&va)[PfDim<D>::DB]) {
    using T = PfDim<D>;
    const int rs2 = kv_heads * dim * 2;
    const int pos = lane % T::NC;
#pragma unroll
    for (int i = 0; i < T::NI; ++i) {
        const int row = 4 * T::RPI * i + T::RPI * wave + lane / T::NC;
        const int kc = pos ^ T::kswz(row), vc = pos ^ T::vswz(row);
        kg[i] = 8 * kc < dim ? row * rs2 + (kc << 4) : fa::OOB;
        vg[i] = 8 * vc < dim ? row * rs2 + (vc << 4) : fa::OOB;
    }
    const int l32 = lane & 31, g = lane >> 5;
#pragma unroll
    for (int t = 0; t < T::KS; ++t) ka[t] = l32 * T::RB + (((2 * t + g) ^ T::kswz(l32)) << 4);
    const int q = lane >> 4, i = lane & 15, j = i >> 2, m = i & 3;
    const int row = 4 * (q >> 1) + j;
#pragma unroll
    for (int d = 0; d < T::DB; ++d) {
        const int chunk = (4 * d + 2 * (q & 1) + (m >> 1)) ^ T::vswz(row);
        va[d] = row * T::RB + (chunk << 4) + 8 * (m & 1);
    }
}

// The padded kernels' outputs where an infinity or NaN of V met a P of zero (a masked key
// of a computed tile, or P's low half): 0 * inf is NaN in the MFMA, while the general
// kernel, which served these head dims before, never reads a masked key's row.  A block
// with such outputs (a finite row sum, some output not finite) walks its key tiles once more
// against the final reference m: values that are not finite count as zero in the products,
// and what a row sees of them is counted on the MFMA too, per tile, by products of 0 / 1
// with a value's class (a visible key of probability zero makes an infinity a NaN, as 0 *
// inf does).  Only outputs that were not finite are replaced.  The second walk costs what the
// first does and is never taken on finite values; a lane summing its row key by key took
// 18 ms for bf16 2 x 700 of 1500 keys x 16 heads of 96 with a NaN in V, the general kernel 1.0; now
// 110 us, 36 without the NaN.
// It runs after the first walk's outputs are stored, loads Q again and finds the lane's offsets
// again: with more alive the first walk of 129 to 256 dims slowed by 2 to 9% (one register more and
// its V reads no longer ran ahead; not inlined, by the stack that a call needs: 34 -> 38 us).
constexpr float kPfPos = 1.0f, kPfNeg = 128.0f, kPfNan = 16384.0f;   // up to 64 keys a tile: digits that stay apart
// a lane's outputs that are not finite: bit 16 (d % 2) + r of word d / 2; whether there are any
template <int NO> __device__ __forceinline__ bool prefill_spoiled(const f32x16 (&o)[NO], uint32_t (&bits)[(NO + 1) / 2]) {
    float t = 0.0f;
#pragma unroll
    for (int d = 0; d < NO; ++d)
#pragma unroll
        for (int r = 0; r < 16; ++r) t = __builtin_fmaf(o[d][r], 0.0f, t);
    if (t == 0.0f) return false;   // (0 * x is NaN for an infinite or NaN x)
#pragma unroll
    for (int d = 0; d < NO; ++d)
#pragma unroll
        for (int r = 0; r < 16; ++r)
            if (!(__builtin_fabsf(o[d][r]) < INFINITY)) bits[d >> 1] |= 1u << (16 * (d & 1) + r);
    return true;
}
// adds the infinities and NaNs that were counted
__device__ __forceinline__ void prefill_add_classes(f32x16 &o, const f32x16 &count) {
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const uint32_t n = (uint32_t)count[r];
        if (n & 127) o[r] += INFINITY;
        if (n >> 7 & 127) o[r] -= INFINITY;
        if (n >> 14) o[r] = NAN;
    }
}
template <int DT, int D, bool GEN>
__device__ __forceinline__ void prefill_redo(const PrefillArgs &a, const uint16_t *qrow, const uint16_t *kbase,
                                             const uint16_t *vbase, char *ks, char *vs, const int (&kg)[PfDim<D>::NI],
                                             const int (&vg)[PfDim<D>::NI], const int (&ka)[PfDim<D>::KS],
                                             const int (&va)[PfDim<D>::DB], int tlo, int ntiles, int qi, int g,
                                             int wave, float m, float inv, const uint32_t (&bits)[(PfDim<D>::DB + 1) / 2], uint16_t *orow) {
    using namespace fa;
    using T = PfDim<D>;
    using V8 = typename PfFormat<DT>::V8;
    using E = typename PfFormat<DT>::E;
    constexpr uint32_t EXP = DT == PUTER_BF16 ? 0x7F80u : 0x7C00u;
    typedef uint16_t u16x8 __attribute__((ext_vector_type(8)));
    const int first = GEN && a.window > 0 ? qi - a.window + 1 : 0;
    const int last = a.causal ? min(qi + a.shift, a.seq_k - 1) : a.seq_k - 1;
    const float mref = m == -INFINITY ? 0.0f : m;
    bool spoiled = false;
#pragma unroll
    for (int w = 0; w < (T::DB + 1) / 2; ++w) spoiled |= bits[w] != 0;
    const bool mine = __any(spoiled);
    V8 qf[T::KS];
#pragma unroll
    for (int t = 0; t < T::KS; ++t)
        qf[t] = 16 * t + 8 * g < a.dim ? __builtin_bit_cast(V8, *reinterpret_cast<const uint4 *>(qrow + 16 * t + 8 * g)) : (V8){};
    f32x16 o[T::DB];
#pragma unroll
    for (int d = 0; d < T::DB; ++d) o[d] = (f32x16){};
    for (int it = tlo; it < ntiles; ++it) {
        const int kv0 = it * BN;
        prefill_copy_tile<D, true>(a, kbase, vbase, kv0, kg, vg, ks, vs, wave);
        wait_tile_copies();
        __syncthreads();
        if (mine) {
#pragma unroll 1
            for (int c = 0; c < 2; ++c) {
                f32x16 s = (f32x16){};
#pragma unroll
                for (int t = 0; t < T::KS; ++t)
                    s = pf_mfma<DT>(*reinterpret_cast<const V8 *>(ks + c * 32 * T::RB + ka[t]), qf[t], s);
                V8 p[2], seen[2], zero[2];
                PfLow<DT, true> low[2];
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int key = kv0 + 32 * c + 8 * (r >> 2) + 4 * g + (r & 3);
                    float dot = s[r];
                    if constexpr (DT == PUTER_F16) dot = (float)(_Float16)dot;
                    if (GEN) dot += a.alibi_s * (float)(key - qi);
                    const bool vis = key >= first && key <= last;
                    const float e = vis ? __builtin_amdgcn_exp2f(__builtin_fmaf(dot, a.scale_log2, -mref)) : 0.0f;
                    pf_set<DT, true>(p[r >> 3], low[r >> 3], r & 7, e);
                    seen[r >> 3][r & 7] = (E)(vis ? 1.0f : 0.0f);
                    zero[r >> 3][r & 7] = (E)(vis && e == 0.0f ? 1.0f : 0.0f);
                }
#pragma unroll
                for (int d = 0; d < T::DB; ++d) {
                    u16x8 v[2];
                    bool bad = false;
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        const char *q = vs + va[d] + (32 * c + 16 * h) * T::RB;
                        const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4 *)(q));
                        const i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4 *)(q + 8 * T::RB));
                        v[h] = __builtin_bit_cast(u16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
                        u16x8 fin;
#pragma unroll
                        for (int j = 0; j < 8; ++j) {
                            const bool f = (v[h][j] & EXP) != EXP;
                            bad |= !f;
                            fin[j] = f ? v[h][j] : (uint16_t)0;
                        }
                        o[d] = pf_pv<DT, true>(__builtin_bit_cast(V8, fin), p[h], low[h], o[d]);
                    }
                    if (!__any(bad)) continue;
                    f32x16 count = (f32x16){};
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        V8 cls, inf;
#pragma unroll
                        for (int j = 0; j < 8; ++j) {
                            const uint32_t x = v[h][j], mag = x & 0x7FFFu;
                            cls[j] = (E)(mag < EXP ? 0.0f : mag > EXP ? kPfNan : x >> 15 ? kPfNeg : kPfPos);
                            inf[j] = (E)(mag == EXP ? kPfNan : 0.0f);
                        }
                        count = pf_mfma<DT>(cls, seen[h], count);
                        count = pf_mfma<DT>(inf, zero[h], count);
                    }
                    prefill_add_classes(o[d], count);
                }
            }
        }
        __syncthreads();
    }
    if (!spoiled) return;
#pragma unroll
    for (int d = 0; d < T::DB; ++d)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int at = 32 * d + 8 * (r >> 2) + 4 * g + (r & 3);
            if ((bits[d >> 1] >> (16 * (d & 1) + r) & 1) && at < a.dim)
                orow[at] = __builtin_bit_cast(uint16_t, (E)(o[d][r] * inv));
        }
}

// GEN: a sliding window (a.window > 0) or an ALiBi slope is set; without either
// that code compiles away.  With ALiBi every tile takes the masked step, which
// adds the bias.  PAD: the head dim is below D and read from the arguments (per-lane copy
// offsets that the exact kernels derive from one register cost the f32 one spills).
template <int DT, int D, bool GEN, bool PAD>
__global__ __launch_bounds__(256, D > 128 ? 1 : 2) void prefill_kernel(PrefillArgs a) {
    using namespace fa;
    using T = PfDim<D>;
    using V8 = typename PfFormat<DT>::V8;
    using V4 = typename PfFormat<DT>::V4;
    using E = typename PfFormat<DT>::E;
    // four separate arrays (not one indexed by parity) so the compiler can
    // tell the tile being copied from the tile being read and does not wait
    // for the copy before the reads
    __shared__ __attribute__((aligned(1024))) char k0s[T::TILE];
    __shared__ __attribute__((aligned(1024))) char k1s[T::TILE];
    __shared__ __attribute__((aligned(1024))) char v0s[T::TILE];
    __shared__ __attribute__((aligned(1024))) char v1s[T::TILE];
    __shared__ int redo;   // PAD: bit w: some output of dims 64 w .. + 63 is not finite

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, g = lane >> 5;
    if (PAD && tid == 0) redo = 0;

    // block -> (query tile, batch, head)
    const int id = blockIdx.x;
    const int bh = a.batch * a.heads;
    const int qt = a.causal ? (a.qtiles - 1 - id / bh) : (id / bh);  // heaviest tiles first
    int b, h;
    if (a.xcd_map) {
        // Inside one tile index, consecutive block ids (dispatched round-robin
        // over the 8 XCDs) are mapped so the G query heads of a kv group
        // (batch, kv head) land on the same XCD and share its L2 for their K/V
        // tiles.  (Walking one group at a time per XCD measured slower: it
        // loses the global heaviest-first order.)
        const int G = a.heads / a.kv_heads;
        const int j = id % bh;
        const int xcd = j & 7, slot = j >> 3;
        const int grp = (slot / G) * 8 + xcd;
        b = grp / a.kv_heads;
        h = (grp % a.kv_heads) * G + slot % G;
    } else {
        b = (id % bh) / a.heads;
        h = id % a.heads;
    }
    const int kvh = h / (a.heads / a.kv_heads);
    const int q0 = qt * BM;
    const int dim = PAD ? a.dim : D;
    const int64_t qrs = (int64_t)a.heads * dim, krs = (int64_t)a.kv_heads * dim;
    const uint16_t *qbase = a.q + (int64_t)b * a.seq_q * qrs + (int64_t)h * dim;
    const uint16_t *kbase = a.k + (int64_t)b * a.seq_k * krs + (int64_t)kvh * dim;
    const uint16_t *vbase = a.v + (int64_t)b * a.seq_k * krs + (int64_t)kvh * dim;

    // this lane's query and its Q^T operand fragments (KS k-steps of 16 dims)
    const int qfirst = q0 + 32 * wave;
    const int qlast = min(qfirst + 31, a.seq_q - 1);
    const int qi = qfirst + l32;
    V8 qf[T::KS];
    {
        const int qload = min(qi, a.seq_q - 1);  // rows past the end compute garbage, never stored
#pragma unroll
        for (int t = 0; t < T::KS; ++t)
            qf[t] = 16 * t + 8 * g < dim   // dims past the head dim: zeros
                        ? __builtin_bit_cast(V8, *reinterpret_cast<const uint4 *>(qbase + (int64_t)qload * qrs + 16 * t + 8 * g))
                        : (V8){};
    }

    // key tiles of the block: [tlo, ntiles); tiles [tfree, nfree) need no mask for
    // any query of it.  Without a window tlo = tfree = 0; with one, the tiles below
    // the first query's window are skipped and those below the last query's window
    // edge are masked.
    int kend = a.seq_k;
    if (a.causal) kend = min(kend, min(q0 + BM, a.seq_q) + a.shift);
    const int ntiles = kend > 0 ? (kend + BN - 1) / BN : 0;
    int nfree = a.seq_k / BN;
    if (a.causal) nfree = min(nfree, q0 + a.shift + 1 > 0 ? (q0 + a.shift + 1) / BN : 0);
    nfree = min(nfree, ntiles);
    if (GEN && a.alibi_s != 0.0f) nfree = 0;   // the bias is added by the masked step only
    int tlo = 0, tfree = 0;
    if (GEN && a.window > 0) {
        const int qmax = min(q0 + BM, a.seq_q) - 1;
        tlo = min(max(0, q0 - a.window + 1) / BN, ntiles);
        tfree = max(tlo, (max(0, qmax - a.window + 1) + BN - 1) / BN);
    }

    int kg[T::NI], vg[T::NI], ka[T::KS], va[T::DB];
    prefill_offsets<D>(a.kv_heads, dim, lane, wave, kg, vg, ka, va);
    PrefillState<D> st;
#pragma unroll
    for (int d = 0; d < T::DB; ++d) st.o[d] = (f32x16){};
    st.m = -INFINITY;
    st.l = 0.0f;

    // tile t lives in buffer t % 2
    if (tlo < ntiles)
        prefill_copy_tile<D, PAD>(a, kbase, vbase, tlo * BN, kg, vg, (tlo & 1) ? k1s : k0s, (tlo & 1) ? v1s : v0s, wave);
    wait_tile_copies();
    __syncthreads();
    // One tile: copy the next tile into the other buffers, compute this one, then
    // wait for the copy and meet at the barrier.  The mask-free tiles [0, nfree)
    // come first and run in a loop of their own (two tiles per iteration so the
    // buffer roles are fixed at compile time); the masked tiles (diagonal, tail)
    // follow in a second loop, so the O accumulators never pass through a merge
    // of the two paths (which cost a register copy of O per tile).
    auto tile_free = [&](int it, const char *kc, const char *vc, char *kn, char *vn) __attribute__((always_inline)) {
        // the next tile's copy runs inside the step (past the last tile: an empty one
        // into the free buffers, so the step has no branch around it)
        const int kvn = it + 1 < ntiles ? (it + 1) * BN : a.seq_k;
        prefill_step_pipelined<DT, D, PAD>(a, kc, vc, qf, st, ka, va, kbase, vbase, kvn, kg, vg, kn, vn, wave);
        wait_tile_copies();
        __syncthreads();
    };
    auto tile_masked = [&](int it) __attribute__((always_inline)) {
        const int kv0 = it * BN;
        const bool odd = it & 1;
        if (it + 1 < ntiles)
            prefill_copy_tile<D, PAD>(a, kbase, vbase, kv0 + BN, kg, vg, odd ? k0s : k1s, odd ? v0s : v1s, wave);
        // waves whose queries all precede this tile, or whose windows all start
        // past it, skip it
        if ((!a.causal || kv0 <= qlast + a.shift) && (!GEN || a.window <= 0 || kv0 + BN - 1 >= qfirst - a.window + 1))
            prefill_step<DT, D, GEN, PAD>(a, odd ? k1s : k0s, odd ? v1s : v0s, qf, st, qi, kv0, ka, va, g, true);
        wait_tile_copies();
        __syncthreads();
    };
    int it = tlo;
    for (; it < tfree && it < ntiles; ++it) tile_masked(it);   // the window's lower edge
    if (it < nfree && (it & 1)) {   // the paired loop below starts on an even tile
        tile_free(it, k1s, v1s, k0s, v0s);
        ++it;
    }
    for (; it + 1 < nfree; it += 2) {
        tile_free(it, k0s, v0s, k1s, v1s);
        tile_free(it + 1, k1s, v1s, k0s, v0s);
    }
    if (it < nfree) {
        tile_free(it, k0s, v0s, k1s, v1s);
        ++it;
    }
    for (; it < ntiles; ++it) tile_masked(it);

    // normalise and store: lane holds O[qi][32d + 8*(r/4) + 4g + r%4]
    const float ltot = swap_halves_sum(st.l);
    const float inv = ltot > 0.0f ? 1.0f / ltot : 0.0f;
    uint32_t bits[(T::DB + 1) / 2] = {};
    bool spoiled = false;
    if constexpr (PAD) {
        spoiled = ltot > 0.0f && qi < a.seq_q && prefill_spoiled(st.o, bits);
        if (spoiled) {
#pragma unroll
            for (int w = 0; w < (T::DB + 1) / 2; ++w)
                if (bits[w]) atomicOr(&redo, 1 << w);
        }
        // a NaN row sum (a NaN score): zeros, or NaN from FlashAttention, as the general kernels
        if (!(ltot > 0.0f)) {
            const float z = a.nan_rows ? ltot : 0.0f;
#pragma unroll
            for (int d = 0; d < T::DB; ++d)
#pragma unroll
                for (int r = 0; r < 16; ++r) st.o[d][r] = z;
        }
    }
    if (qi < a.seq_q) {
        uint16_t *orow = a.o + (int64_t)b * a.seq_q * qrs + (int64_t)qi * qrs + (int64_t)h * dim;
#pragma unroll
        for (int d = 0; d < T::DB; ++d)
#pragma unroll
            for (int rb = 0; rb < 4; ++rb) {
                if (32 * d + 8 * rb >= dim) continue;   // dim % 8 == 0: an 8-dim run is whole or absent
                V4 v;
#pragma unroll
                for (int i = 0; i < 4; ++i) v[i] = (E)(PAD && !(ltot > 0.0f) ? st.o[d][4 * rb + i] : st.o[d][4 * rb + i] * inv);
                *reinterpret_cast<V4 *>(orow + 32 * d + 8 * rb + 4 * g) = v;
            }
    }
    if constexpr (PAD) {
        __syncthreads();
        if (__builtin_expect(!redo, 1)) return;
        // (the lane and its offsets afresh, so that none of them is alive for this in the first walk)
        const int lane = (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)), g = lane >> 5;
        const int qi = qfirst + (lane & 31);
        int kg[T::NI], vg[T::NI], ka[T::KS], va[T::DB];
        prefill_offsets<D>(a.kv_heads, dim, lane, wave, kg, vg, ka, va);
        const int64_t row = (int64_t)min(qi, a.seq_q - 1) * qrs;
        prefill_redo<DT, D, GEN>(a, qbase + row, kbase, vbase, k0s, v0s, kg, vg, ka, va, tlo, ntiles, qi, g, wave, st.m, inv, bits,
                                 a.o + (qbase - a.q) + row);
    }
}

// ------------------------------------------------------------ f32 prefill --
// f32 MultiHeadAttention (head dim 128 or 64, or any multiple of 4 up to 256; causal or not, sliding window, ALiBi) on
// v_mfma_f32_32x32x2_f32: exact f32 products, f32 sums, softmax in f32 against a
// running maximum (the reference's stableSoftmaxRow takes the row max, exp in
// float64 and a sequential f32 sum; the order of the sums differs, the f32 bar
// holds).  One 256-thread block per (128-query tile, head, batch), wave w owning 32
// queries; K/V stream through LDS in 32-key tiles (16 KB each at D = 128), double
// buffered, copied HBM -> LDS by buffer_load ... lds; two blocks per CU.
//   S^T[key, q] = K . Q^T: MFMA step s of 4-step group g gives half h = lane / 32 of
//     the wave d = 8 g + 4 h + s, so a lane's K operands for a group are one 16-byte
//     LDS read of its key row (chunk c of row r at c ^ (r % 16): the 16 rows an LDS
//     cycle serves on distinct banks) and Q^T sits in registers for the whole loop.
//   The accumulator's register r = 4 g + s of lane (q, h) holds key 8 g + 4 h + s, so
//     P^T is already the B operand of O^T[d, q] += V^T . P^T for the same k order;
//     V^T's operand is one float per lane and step from the row-major V tile (row k
//     keeps column d at d ^ 32 (k / 4 % 2), so the two half-waves, rows k and k + 4,
//     read opposite halves of the bank line).
template <int D> struct PfF32Dim {
    static_assert(D == 256 || D == 128 || D == 96 || D == 64, "head dim 256, 128, 96 or 64");
    static constexpr int BN = 32;               // keys per tile
    static constexpr int RB = D > 128 ? 1024 : D > 64 ? 512 : 256;   // row bytes (the power of two that holds D)
    static constexpr int NC = RB / 16;          // 16-byte chunks per row
    static constexpr int TILE = BN * RB;        // 32, 16 or 8 KB
    static constexpr int KG = D / 8;            // 4-step groups over d
    static constexpr int DB = D / 32;           // O^T blocks of 32 dims
    static constexpr int RPI = 64 / NC;         // rows per copy instruction
    static constexpr int NI = BN / RPI / 4;     // copy instructions per wave and tensor
    static constexpr int kswz(int r) { return r & 15; }
    static constexpr int vswz(int r) { return ((r >> 2) & 1) << 3; }   // in chunks (8 = 32 floats)
};

// prefill_redo for f32 (a value is one float per lane and MFMA step).  Beyond 128 dims two blocks
// of 32 a walk, those that need it: with all of them alive the first walk spilled (129 -> 136 us
// for 2 x 512 x 8 of 256, now 128).
constexpr int redo_blocks(int D) { return D > 128 ? 2 : D / 32; }
constexpr int redo_words(int D) { return (redo_blocks(D) + 1) / 2; }
template <int D, bool GEN, typename Copy>
__device__ __forceinline__ void prefill_f32_redo(const PrefillArgs &a, Copy copy_tile, const float *qrow, char *ks, char *vs,
                                                 int kr, const int (&vr)[redo_blocks(D)], int d0, int tlo, int thi, int qi,
                                                 int l32, int h, float m, float inv, const uint32_t (&bits)[redo_words(D)],
                                                 float *orow) {
    using T = PfF32Dim<D>;
    const int first = GEN && a.window > 0 ? qi - a.window + 1 : 0;
    const int last = a.causal ? min(qi + a.shift, a.seq_k - 1) : a.seq_k - 1;
    const float mref = m == -INFINITY ? 0.0f : m;
    constexpr int NB = redo_blocks(D);
    bool spoiled = false;
#pragma unroll
    for (int w = 0; w < redo_words(D); ++w) spoiled |= bits[w] != 0;
    const bool mine = __any(spoiled);
    f32x4 qf[T::KG];
#pragma unroll
    for (int g = 0; g < T::KG; ++g)
        qf[g] = 8 * g + 4 * h < a.dim ? *reinterpret_cast<const f32x4 *>(qrow + 8 * g + 4 * h) : (f32x4){};
    f32x16 o[NB];
#pragma unroll
    for (int db = 0; db < NB; ++db) o[db] = (f32x16){};
    for (int it = tlo; it < thi; ++it) {
        const int kv0 = it * T::BN;
        copy_tile(kv0, ks, vs);
        __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0)
        __syncthreads();
        if (mine) {
            f32x16 p = (f32x16){};
#pragma unroll
            for (int g = 0; g < T::KG; ++g) {
                const f32x4 kv = *reinterpret_cast<const f32x4 *>(ks + kr + (((2 * g + h) ^ T::kswz(l32)) << 4));
#pragma unroll
                for (int s4 = 0; s4 < 4; ++s4) p = __builtin_amdgcn_mfma_f32_32x32x2f32(kv[s4], qf[g][s4], p, 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);   // as in the first walk
            }
            uint32_t seen = 0, zero = 0;   // register r's key: visible, and of probability zero
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int key = kv0 + 8 * (r >> 2) + 4 * h + (r & 3);
                float dot = p[r];
                if (GEN) dot += a.alibi_s * (float)(key - qi);
                const bool vis = key >= first && key <= last;
                p[r] = vis ? __builtin_amdgcn_exp2f(__builtin_fmaf(dot, a.scale_log2_lo, __builtin_fmaf(dot, a.scale_log2, -mref))) : 0.0f;
                seen |= (uint32_t)vis << r;
                zero |= (uint32_t)(vis && p[r] == 0.0f) << r;
            }
#pragma unroll
            for (int db = 0; db < NB; ++db) {
                f32x16 t = (f32x16){};
                bool bad = false;
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const float v = *reinterpret_cast<const float *>(vs + (8 * (r >> 2) + (r & 3)) * T::RB + vr[db]);
                    const bool f = __builtin_fabsf(v) < INFINITY;
                    bad |= !f;
                    t = __builtin_amdgcn_mfma_f32_32x32x2f32(f ? v : 0.0f, p[r], t, 0, 0, 0);
                }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int r = 0; r < 16; ++r) o[db][r] += t[r];
                if (!__any(bad)) continue;
                t = (f32x16){};
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const float v = *reinterpret_cast<const float *>(vs + (8 * (r >> 2) + (r & 3)) * T::RB + vr[db]);
                    const float cls = v != v ? kPfNan : v == INFINITY ? kPfPos : v == -INFINITY ? kPfNeg : 0.0f;
                    const float inf = __builtin_fabsf(v) == INFINITY ? kPfNan : 0.0f;
                    t = __builtin_amdgcn_mfma_f32_32x32x2f32(cls, (float)(seen >> r & 1), t, 0, 0, 0);
                    t = __builtin_amdgcn_mfma_f32_32x32x2f32(inf, (float)(zero >> r & 1), t, 0, 0, 0);
                }
                prefill_add_classes(o[db], t);
            }
        }
        __syncthreads();
    }
    if (!spoiled) return;
#pragma unroll
    for (int db = 0; db < NB; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int at = 32 * (d0 + db) + 8 * (r >> 2) + 4 * h + (r & 3);
            if ((bits[db >> 1] >> (16 * (db & 1) + r) & 1) && at < a.dim) orow[at] = o[db][r] * inv;
        }
}

template <int D, bool GEN, bool PAD>
__global__ __launch_bounds__(256, D > 128 ? 1 : 2) void prefill_f32_kernel(PrefillArgs a) {
    using T = PfF32Dim<D>;
    constexpr int BM = fa::BM, BN = T::BN;
    __shared__ __attribute__((aligned(1024))) char k0s[T::TILE];
    __shared__ __attribute__((aligned(1024))) char k1s[T::TILE];
    __shared__ __attribute__((aligned(1024))) char v0s[T::TILE];
    __shared__ __attribute__((aligned(1024))) char v1s[T::TILE];
    __shared__ int redo;   // PAD: bit w: some output of dims 64 w .. + 63 is not finite

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, h = lane >> 5;
    if (PAD && tid == 0) redo = 0;

    // block -> (query tile, batch, head), heaviest tiles first, a kv group's query
    // heads on one XCD (as prefill_kernel)
    const int id = blockIdx.x;
    const int bh = a.batch * a.heads;
    const int qt = a.causal ? (a.qtiles - 1 - id / bh) : (id / bh);
    int b, hd;
    if (a.xcd_map) {
        const int G = a.heads / a.kv_heads;
        const int j = id % bh;
        const int xcd = j & 7, slot = j >> 3;
        const int grp = (slot / G) * 8 + xcd;
        b = grp / a.kv_heads;
        hd = (grp % a.kv_heads) * G + slot % G;
    } else {
        b = (id % bh) / a.heads;
        hd = id % a.heads;
    }
    const int kvh = hd / (a.heads / a.kv_heads);
    const int q0 = qt * BM;
    const float *const qp = reinterpret_cast<const float *>(a.q);
    const float *const kp = reinterpret_cast<const float *>(a.k);
    const float *const vp = reinterpret_cast<const float *>(a.v);
    const int dim = PAD ? a.dim : D;
    const int64_t qrs = (int64_t)a.heads * dim, krs = (int64_t)a.kv_heads * dim;
    const float *qbase = qp + (int64_t)b * a.seq_q * qrs + (int64_t)hd * dim;
    const float *kbase = kp + (int64_t)b * a.seq_k * krs + (int64_t)kvh * dim;
    const float *vbase = vp + (int64_t)b * a.seq_k * krs + (int64_t)kvh * dim;

    // this lane's query and its Q^T operands: qf[g] = Q[qi][8 g + 4 h .. + 3]
    const int qfirst = q0 + 32 * wave;
    const int qlast = min(qfirst + 31, a.seq_q - 1);
    const int qi = qfirst + l32;
    f32x4 qf[T::KG];
    {
        const int qload = min(qi, a.seq_q - 1);   // rows past the end compute garbage, never stored
#pragma unroll
        for (int g = 0; g < T::KG; ++g)
            qf[g] = 8 * g + 4 * h < dim   // dims past the head dim: zeros
                        ? *reinterpret_cast<const f32x4 *>(qbase + (int64_t)qload * qrs + 8 * g + 4 * h)
                        : (f32x4){};
    }

    int kend = a.seq_k;
    if (a.causal) kend = min(kend, min(q0 + BM, a.seq_q) + a.shift);
    const int ntiles = kend > 0 ? (kend + BN - 1) / BN : 0;
    int nfree = a.seq_k / BN;
    if (a.causal) nfree = min(nfree, q0 + a.shift + 1 > 0 ? (q0 + a.shift + 1) / BN : 0);
    nfree = min(nfree, ntiles);
    if (GEN && a.alibi_s != 0.0f) nfree = 0;   // the bias is added by the masked step only
    // a sliding window: the tiles below the block's first query's window are skipped,
    // those below its last query's window edge masked ([wlo, wfree))
    int wlo = 0, wfree = 0;
    if (GEN && a.window > 0) {
        const int qmax = min(q0 + BM, a.seq_q) - 1;
        wlo = min(max(0, q0 - a.window + 1) / BN, ntiles);
        wfree = max(wlo, (max(0, qmax - a.window + 1) + BN - 1) / BN);
    }

    // copy offsets (source side, swizzled): wave w fills rows 4 RPI i + RPI w + lane / NC
    int kg[8], vg[8];
    {
        // chunks past the head dim: an offset past the buffer's range, read as zeros
        const int rs4 = a.kv_heads * dim * 4;
        const int pos = lane % T::NC;
#pragma unroll
        for (int i = 0; i < T::NI; ++i) {
            const int row = 4 * T::RPI * i + T::RPI * wave + lane / T::NC;
            const int kc = pos ^ T::kswz(row), vc = pos ^ T::vswz(row);
            kg[i] = 4 * kc < dim ? row * rs4 + (kc << 4) : fa::OOB;
            vg[i] = 4 * vc < dim ? row * rs4 + (vc << 4) : fa::OOB;
        }
    }
    auto copy_tile = [&](int kv0, char *kdst, char *vdst) __attribute__((always_inline)) {
        const int rs4 = a.kv_heads * dim * 4;
        const int rows = min(a.seq_k - kv0, BN);
        const int bytes = (rows - 1) * rs4 + dim * 4;
        const int64_t base = (int64_t)kv0 * a.kv_heads * dim;
        const __amdgpu_buffer_rsrc_t kd =
            __builtin_amdgcn_make_buffer_rsrc((void *)(kbase + base), (short)0, bytes, fa::BUF_WORD3);
        const __amdgpu_buffer_rsrc_t vd =
            __builtin_amdgcn_make_buffer_rsrc((void *)(vbase + base), (short)0, bytes, fa::BUF_WORD3);
        // (constant trip counts with a guard: a loop bound that depends on the template
        // arguments inside a lambda loses the kernel's host stub)
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if (i < T::NI)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(kd, (lds_void *)(kdst + (4 * T::RPI * i + T::RPI * wave) * T::RB),
                                                         16, kg[i], 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if (i < T::NI)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(vd, (lds_void *)(vdst + (4 * T::RPI * i + T::RPI * wave) * T::RB),
                                                         16, vg[i], 0, 0, 0);
    };
    // fragment reads: K row l32, group g at chunk (2 g + h) ^ kswz(l32); V row
    // 8 g + 4 h + s, column (32 db + l32) ^ 32 h (vswz(row) = 8 chunks iff h = 1)
    const int kr = l32 * T::RB;
    int vr[T::DB];
#pragma unroll
    for (int db = 0; db < T::DB; ++db) vr[db] = 4 * h * T::RB + (((32 * db + l32) ^ (32 * h)) << 2);

    f32x16 o[T::DB];
#pragma unroll
    for (int db = 0; db < T::DB; ++db) o[db] = (f32x16){};
    float m = -INFINITY, l = 0.0f;
    const float c = a.scale_log2;

    auto step = [&](const char *ks, const char *vs, int kv0, bool masked) __attribute__((always_inline)) {
        f32x16 sacc = (f32x16){};
#pragma unroll
        for (int g = 0; g < 32; ++g) {
            if (g >= T::KG) break;
            const f32x4 kv = *reinterpret_cast<const f32x4 *>(ks + kr + (((2 * g + h) ^ T::kswz(l32)) << 4));
#pragma unroll
            for (int s4 = 0; s4 < 4; ++s4) sacc = __builtin_amdgcn_mfma_f32_32x32x2f32(kv[s4], qf[g][s4], sacc, 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);   // one group's K read live at a time
        }
        // register r: key kv0 + 8 (r / 4) + 4 h + r % 4, query qi.  The masked step
        // also adds ALiBi's alibi_s * (k - q) (before the scale: slope * (k - q) on the
        // scaled score, typed_compute.go:176-178) and hides keys below the window
        if (masked) {
            const int last = a.causal ? min(qi + a.shift, a.seq_k - 1) : a.seq_k - 1;
            const int lim = last - kv0 - 4 * h;
            const int lo = GEN && a.window > 0 ? qi - a.window + 1 - kv0 - 4 * h : INT_MIN;
            if (GEN && a.alibi_s != 0.0f) {
                const float base = (float)(kv0 + 4 * h - qi);
#pragma unroll
                for (int r = 0; r < 16; ++r) sacc[r] += a.alibi_s * (base + (float)(8 * (r >> 2) + (r & 3)));
            }
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int off = 8 * (r >> 2) + (r & 3);
                if (off > lim || off < lo) sacc[r] = -INFINITY;
            }
        }
        float tmax = -INFINITY;
#pragma unroll
        for (int r = 0; r < 16; ++r) tmax = fmaxf(tmax, sacc[r]);
        tmax = swap_halves_max(tmax) * c;
        if (__any(tmax > m)) {   // a new maximum: rescale O and l (wave-uniform branch)
            const float mnew = fmaxf(m, tmax);
            const float alpha = m == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m - mnew);
            m = mnew;
            l *= alpha;
#pragma unroll
            for (int db = 0; db < 8; ++db) {
                if (db >= T::DB) break;
#pragma unroll
                for (int r = 0; r < 16; ++r) o[db][r] *= alpha;
            }
        }
        const float mref = m == -INFINITY ? 0.0f : m;
        float psum = 0.0f;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            float e = __builtin_fmaf(sacc[r], c, -mref);
            if constexpr (PAD) e = __builtin_fmaf(sacc[r], a.scale_log2_lo, e);
            sacc[r] = __builtin_amdgcn_exp2f(e);
            psum += sacc[r];
        }
        l += psum;
        if constexpr (PAD) {
            // (the general kernel, which served these head dims before, sums the keys in
            // short runs: each tile's product starts from zero here and is added to O once,
            // so the error stays below its own)
#pragma unroll
            for (int db = 0; db < 8; ++db) {
                if (db >= T::DB) break;
                f32x16 t = (f32x16){};
#pragma unroll
                for (int g = 0; g < BN / 8; ++g)
#pragma unroll
                    for (int s4 = 0; s4 < 4; ++s4) {
                        const float vv = *reinterpret_cast<const float *>(vs + (8 * g + s4) * T::RB + vr[db]);
                        t = __builtin_amdgcn_mfma_f32_32x32x2f32(vv, sacc[4 * g + s4], t, 0, 0, 0);
                    }
#pragma unroll
                for (int r = 0; r < 16; ++r) o[db][r] += t[r];
            }
            return;
        }
        // O^T += V^T . P^T, step (g, s4): V row 8 g + 4 h + s4, P^T register 4 g + s4; a
        // scheduling barrier per group keeps one group's V reads live at a time
#pragma unroll
        for (int g = 0; g < BN / 8; ++g) {
#pragma unroll
            for (int s4 = 0; s4 < 4; ++s4)
#pragma unroll
                for (int db = 0; db < 8; ++db) {
                    if (db >= T::DB) break;
                    const float vv = *reinterpret_cast<const float *>(vs + (8 * g + s4) * T::RB + vr[db]);
                    o[db] = __builtin_amdgcn_mfma_f32_32x32x2f32(vv, sacc[4 * g + s4], o[db], 0, 0, 0);
                }
            __builtin_amdgcn_sched_barrier(0);
        }
    };

    // this block's key tiles: from the window's lower edge on, all of them or split
    // blockIdx.y's run of split_tiles
    int tlo = wlo, thi = ntiles;
    if (a.split_tiles > 0) {
        const int ylo = min(ntiles, (int)blockIdx.y * a.split_tiles);
        tlo = max(tlo, ylo);
        thi = min(ntiles, ylo + a.split_tiles);
    }
    if (tlo < thi) copy_tile(tlo * BN, k0s, v0s);
    __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0)
    __syncthreads();
    auto tile = [&](int it, const char *kc, const char *vc, char *kn, char *vn) __attribute__((always_inline)) {
        const int kv0 = it * BN;
        if (it + 1 < thi) copy_tile(kv0 + BN, kn, vn);
        // waves whose queries all precede the tile, or whose windows all start past it,
        // skip it
        const bool seen = (!a.causal || kv0 <= qlast + a.shift) && (!GEN || a.window <= 0 || kv0 + BN - 1 >= qfirst - a.window + 1);
        if (it >= wfree && it < nfree) step(kc, vc, kv0, false);
        else if (seen) step(kc, vc, kv0, true);
        __builtin_amdgcn_s_waitcnt(0x0F70);
        __syncthreads();
    };
    int it = tlo;
    for (; it + 1 < thi; it += 2) {
        tile(it, k0s, v0s, k1s, v1s);
        tile(it + 1, k1s, v1s, k0s, v0s);
    }
    if (it < thi) tile(it, k0s, v0s, k1s, v1s);

    const float ltot = swap_halves_sum(l);
    uint32_t bits[(T::DB + 1) / 2] = {};
    bool spoiled = false;
    if constexpr (PAD) {
        spoiled = ltot > 0.0f && qi < a.seq_q && prefill_spoiled(o, bits);
        if (spoiled) {
#pragma unroll
            for (int w = 0; w < (T::DB + 1) / 2; ++w)
                if (bits[w]) atomicOr(&redo, 1 << w);
        }
        if (!(ltot > 0.0f)) {   // a NaN score: zeros, as the general kernel
#pragma unroll
            for (int db = 0; db < 8; ++db)
                if (db < T::DB) o[db] = (f32x16){};
        }
    }
    float *orow;
    float inv = 1.0f;
    if (a.part_ml) {
        // split: the row's (max, sum) and unnormalised output to the partials
        const int64_t prow = (((int64_t)blockIdx.y * a.batch + b) * a.seq_q + qi) * a.heads + hd;
        orow = a.part_o + prow * dim;
        if (qi < a.seq_q) {
            if (h == 0) a.part_ml[prow] = make_float2(m, ltot);
#pragma unroll
            for (int db = 0; db < 8; ++db) {
                if (db >= T::DB) break;
#pragma unroll
                for (int rb = 0; rb < 4; ++rb) {
                    if (32 * db + 8 * rb + 4 * h >= dim) continue;
                    f32x4 v;
#pragma unroll
                    for (int i = 0; i < 4; ++i) v[i] = o[db][4 * rb + i];
                    *reinterpret_cast<f32x4 *>(orow + 32 * db + 8 * rb + 4 * h) = v;
                }
            }
        }
    } else {
        // normalise and store: lane holds O[qi][32 db + 8 (r/4) + 4 h + r%4]
        inv = ltot > 0.0f ? 1.0f / ltot : 0.0f;
        orow = reinterpret_cast<float *>(a.o) + (int64_t)b * a.seq_q * qrs + (int64_t)qi * qrs + (int64_t)hd * dim;
        if (qi < a.seq_q) {
#pragma unroll
            for (int db = 0; db < 8; ++db) {
                if (db >= T::DB) break;
#pragma unroll
                for (int rb = 0; rb < 4; ++rb) {
                    if (32 * db + 8 * rb + 4 * h >= dim) continue;   // dim % 4 == 0
                    f32x4 v;
#pragma unroll
                    for (int i = 0; i < 4; ++i) v[i] = o[db][4 * rb + i] * inv;
                    *reinterpret_cast<f32x4 *>(orow + 32 * db + 8 * rb + 4 * h) = v;
                }
            }
        }
    }
    if constexpr (PAD) {   // outputs that are not finite, once they are stored
        __syncthreads();
        if (!redo) return;
        const float *qrow = qbase + (int64_t)min(qi, a.seq_q - 1) * qrs;
        if constexpr (D <= 128) {
            prefill_f32_redo<D, GEN>(a, copy_tile, qrow, k0s, v0s, kr, vr, 0, tlo, thi, qi, l32, h, m, inv, bits, orow);
        } else {
            const int groups = __builtin_amdgcn_readfirstlane(redo);
#pragma unroll 1
            for (int w = 0; w < T::DB / 2; ++w) {
                if (!(groups >> w & 1)) continue;
                const int at = 4 * h * T::RB, vd[2] = {at + (((64 * w + l32) ^ (32 * h)) << 2), at + (((64 * w + 32 + l32) ^ (32 * h)) << 2)};
                const uint32_t mine[1] = {w == 0 ? bits[0] : w == 1 ? bits[1] : w == 2 ? bits[2] : bits[3]};
                prefill_f32_redo<D, GEN>(a, copy_tile, qrow, k0s, v0s, kr, vd, 2 * w, tlo, thi, qi, l32, h, m, inv, mine, orow);
            }
        }
    }
}

// Merges the key splits of prefill_f32_kernel: one wave per (batch, query, head) row,
// lanes over the head dims; the splits are folded in order with weights
// exp2(m_s - M) (m in the scaled log2 domain), O = sum w_s O_s / sum w_s l_s; a row
// with no visible key (every m = -inf) is 0, as in the unsplit kernel.
template <int D, bool PAD>
__global__ __launch_bounds__(256) void prefill_f32_combine_kernel(PrefillArgs a, int splits, int64_t rows) {
    constexpr int J = (D + 63) / 64;
    const int dim = PAD ? a.dim : D;
    const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= rows) return;
    const int lane = threadIdx.x & 63;
    float M = -INFINITY;
    for (int s = 0; s < splits; ++s) M = fmaxf(M, a.part_ml[s * rows + row].x);
    float acc[J] = {}, lsum = 0.0f;   // dims lane, lane + 64, ..
    if (M != -INFINITY) {
        for (int s = 0; s < splits; ++s) {
            const float2 ml = a.part_ml[s * rows + row];
            const float w = ml.x == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(ml.x - M);
            lsum += w * ml.y;
            const float *po = a.part_o + (s * rows + row) * dim;
#pragma unroll
            for (int j = 0; j < J; ++j)   // (past a padded row's end: its last dim, not stored)
                acc[j] += w * po[PAD ? min(64 * j + lane, dim - 1) : 64 * j + lane];
        }
    }
    const float inv = lsum > 0.0f ? 1.0f / lsum : 0.0f;
    // row = (batch, query, head): the output row of the same index, dim floats
    float *out = reinterpret_cast<float *>(a.o) + row * dim;
#pragma unroll
    for (int j = 0; j < J; ++j)
        if (!PAD || 64 * j + lane < dim) out[64 * j + lane] = acc[j] * inv;
}

// The head dim D of the kernel that serves a head dim: the least that holds it.  A dim of
// 96 runs on the kernel of 96 (6 of 8 k-steps, 3 of 4 output blocks) rather than padded
// to 128; between 129 and 255 the padding of 256 still beats the general kernel.  Bound
// by the S, softmax and P.V phases of a tile as at 128, plus the P low halves' MFMAs; before,
// the general kernel (a thread per key, row-strided 2-byte loads, no MFMA): f16 2 x 700 of
// 1500 x 16 heads of 96 causal 9680 -> 33 us, bf16 1014 -> 34, f32 1473 -> 150; 2 x 512 x 8
// of 256 f16 2068 -> 34, bf16 221 -> 34, f32 333 -> 135; FlashAttention 1000 x 1000 of 80
// f16 929 -> 22, bf16 639 -> 22.  Errors against float64 are no larger than the general
// kernel's in any of them (f16 2.1e-4, bf16 1.7e-3, f32 2.2e-7 -> 1.5e-7).
template <int D_, bool PAD_> struct PfHeadDim {
    static constexpr int D = D_;
    static constexpr bool PAD = PAD_;
};
template <typename F> static void with_head_dim(int64_t dim, F f) {
    if (dim == 64) f(PfHeadDim<64, false>{});
    else if (dim == 128) f(PfHeadDim<128, false>{});
    else if (dim < 64) f(PfHeadDim<64, true>{});
    else if (dim <= 96) f(PfHeadDim<96, true>{});
    else if (dim < 128) f(PfHeadDim<128, true>{});
    else f(PfHeadDim<256, true>{});
}

// The general kernel or the padded one?  Estimates in us, fitted to 2900 bf16 and 1200 f32
// shapes (1 to 32 heads, 2 to 300 queries over 40 to 3000 keys, dims 16 to 256; 6% off for the padded
// kernels, 15% for the general one).  The general kernel has a block per query row and
// head: a row's keys in steps, 1.7 times slower where the heads that an XCD's rows see overflow
// its L2, or, once rows fill the chip, all rows' keys at a rate.  f16 needs no such rule: its
// general kernel widens in software and never wins.
static double general_us(const MhaArgs &m, bool f32) {
    const double rows = (double)m.batch * m.seq_q * m.heads, dim = (double)m.dim;
    double most = (double)m.seq_k, mean = most;   // keys that a row sees
    if (m.causal) mean = (double)m.shift + 0.5 * (double)(m.seq_q + 1);
    if (m.window > 0) most = std::min(most, (double)m.window);
    mean = std::min(std::max(mean, 1.0), most);
    const double heads = std::max(1.0, std::min((double)m.batch * m.kv_heads, rows / 8));
    const bool overflows = heads * (double)m.seq_k * dim * (f32 ? 8 : 4) > 4.2e6;
    const double steps = most * (f32 ? 0.0078 + 0.000162 * dim : 0.0082 + 0.000145 * dim) * (overflows ? 1.7 : 1.0);
    return (f32 ? 3.9 : 3.7) + std::hypot(steps, rows * mean * (f32 ? 1.3e-5 + 6.6e-7 * dim : 1.8e-5 + 4.4e-7 * dim));
}
// The padded kernels: the key tiles of the longest block, in rounds of blocks.
static double padded_us(const MhaArgs &m, int64_t blocks, int64_t tiles, int64_t splits, bool f32) {
    const int i = m.dim <= 64 ? 0 : m.dim <= 96 ? 1 : m.dim <= 128 ? 2 : 3;
    constexpr double base[2][4] = {{3.5, 4.2, 4.6, 7.4}, {3.7, 4.5, 6.2, 8.0}};
    constexpr double tile[2][4] = {{0.94, 1.14, 1.3, 2.85}, {2.5, 3.7, 6.3, 13.0}};
    const int64_t room = (int64_t)device_cus() * (m.dim > 128 ? 1 : 2), rounds = (blocks * splits + room - 1) / room;
    const double sums = splits > 1 ? 1.2 + 0.53 * (double)splits + 4.3e-6 * (double)(splits * m.batch * m.seq_q * m.heads * m.dim) : 0.0;
    return base[f32][i] + tile[f32][i] * (double)(tiles * rounds) + sums;
}
static int64_t prefill_tiles(const MhaArgs &m, int64_t bn) {   // key tiles of the longest block
    const int64_t keys = m.window > 0 ? std::min(m.seq_k, m.window + fa::BM + bn) : m.seq_k;
    return (keys + bn - 1) / bn;
}

// f32 MultiHeadAttention on prefill_f32_kernel: head dims of 4 n up to 256, at least 16 query
// rows, causal or not, with or without a sliding window and ALiBi.
static bool launch_prefill_f32(const MhaArgs &m, hipStream_t s, int *status) {
    if (m.dim % 4 || m.dim > 256) return false;
    if (m.seq_q < 16) return false;
    if (m.seq_q > 0x3FFFFFFF || m.seq_k > 0x3FFFFFFF || m.shift > 0x3FFFFFFF || m.shift < -0x3FFFFFFF) return false;
    if (m.kv_heads * m.dim > 32768 * 128) return false;   // a 32-row K/V tile spans < 2^30 bytes
    const uintptr_t mask = 15;
    if ((reinterpret_cast<uintptr_t>(m.q) | reinterpret_cast<uintptr_t>(m.k) |
         reinterpret_cast<uintptr_t>(m.v) | reinterpret_cast<uintptr_t>(m.o)) & mask)
        return false;
    PrefillArgs a;
    a.q = static_cast<const uint16_t *>(m.q);
    a.k = static_cast<const uint16_t *>(m.k);
    a.v = static_cast<const uint16_t *>(m.v);
    a.o = static_cast<uint16_t *>(m.o);
    a.batch = (int)m.batch;
    a.seq_q = (int)m.seq_q;
    a.seq_k = (int)m.seq_k;
    a.heads = (int)m.heads;
    a.kv_heads = (int)m.kv_heads;
    a.dim = (int)m.dim;
    a.nan_rows = m.nan_rows;
    a.qtiles = (int)((m.seq_q + fa::BM - 1) / fa::BM);
    a.causal = m.causal;
    a.shift = (int)m.shift;
    // a window of seq_q or more hides no key (a query's distance to a visible key is
    // below seq_q): run it as no window
    a.window = (m.window > 0 && m.window < m.seq_q) ? (int)m.window : 0;
    a.alibi_s = m.alibi != 0.0f ? m.alibi / m.scale : 0.0f;
    a.xcd_map = ((a.batch * a.kv_heads) % 8 == 0) ? 1 : 0;
    a.scale_log2 = m.scale * 1.4426950408889634f;
    if (m.dim != 64 && m.dim != 128) {
        // the padded kernels add the scale's low part; it is kept positive, so a masked
        // score's -inf stays -inf through both products
        const double exact = (double)m.scale * 1.4426950408889634;
        a.scale_log2 = (float)exact;
        if ((double)a.scale_log2 >= exact) a.scale_log2 = std::nextafter(a.scale_log2, 0.0f);
        a.scale_log2_lo = (float)(exact - (double)a.scale_log2);
    }
    const bool gen = a.window > 0 || a.alibi_s != 0.0f;   // the kernel with the window / ALiBi code
    const int64_t blocks = (int64_t)a.qtiles * a.batch * a.heads;
    if (blocks > 0x7FFFFFFF) return false;
    const int64_t cus = device_cus();
    const int64_t ktiles = (m.seq_k + 31) / 32;
    hipStreamCaptureStatus cst = hipStreamCaptureStatusNone;
    const bool capturing = hipStreamIsCapturing(s, &cst) != hipSuccess || cst != hipStreamCaptureStatusNone;
    // Grids of fewer than 24 blocks stay on the general kernel (one block per query
    // row and head) unless they are causal over at least 8 key tiles and can split
    // them (below): config 1's 128 queries x 8 heads of 64 (8 blocks) 9.2 us there
    // against 14.2 here even split; 256 x 8 x 128 (16 blocks) 33.1 against 24.1 split
    // (43 unsplit), 640 x 4 x 64 47.5 against 22.1.  From 24 blocks this kernel wins
    // unsplit too (384 x 8 x 64: 32.9 against 36.0, 4 x 128 x 8 x 64: 15.0 against 24.5)
    if (blocks < 24 && (!a.causal || ktiles < 8 || capturing)) return false;
    // other head dims than 64 and 128: from 2048 rows (batch x queries x heads) or 512 keys on
    // (2 x 21 x 12 rows over 173 keys of 96: 10.6 there against 24.9 here; 2 x 60 x 8 over 1500
    // keys of 256: 218 against 107, 2 x 200 x 16 over 200 keys of 40: 75 against 21), and there
    // by the estimates above (16 x 32 heads over 700 keys of 256: 77 there against 152)
    if (m.dim != 64 && m.dim != 128 && m.batch * m.seq_q * m.heads < 2048 && ktiles < 16) return false;
    // Small grids split each block's key range over blockIdx.y, partials in the
    // library's scratch: the longest block's key loop, the critical path, shrinks with
    // the split count.  Causal grids of under two blocks per CU aim at four blocks per
    // CU in runs of at least 8 key tiles (2 under 24 blocks) (the triangle leaves most
    // CUs idle while the last query tiles run: B1 S4096 8 x 64 causal 296 -> 221 us,
    // S2048 8 x 128 154 -> 146 us), other grids of under one block per CU at two, in
    // runs of at least 16 (B1 S2048 8 x 64, 150 -> 88 us; more splits lose there).  A
    // stream that is capturing a graph keeps the unsplit kernel (the scratch cannot
    // grow there)
    int64_t splits = 1;
    if (a.causal && blocks < 2 * cus)
        splits = std::max<int64_t>(1, std::min<int64_t>((4 * cus + blocks - 1) / blocks, ktiles / (blocks < 24 ? 2 : 8)));
    else if (!a.causal && blocks < cus)
        splits = std::max<int64_t>(1, std::min<int64_t>((2 * cus + blocks - 1) / blocks, ktiles / 16));
    if (capturing) splits = 1;
    if (m.dim != 64 && m.dim != 128 &&
        general_us(m, true) < padded_us(m, blocks, (prefill_tiles(m, 32) + splits - 1) / splits, splits, true))
        return false;
    auto launch = [&](dim3 grid) {
        with_head_dim(m.dim, [&](auto d) {
            if (gen) prefill_f32_kernel<d.D, true, d.PAD><<<grid, 256, 0, s>>>(a);
            else prefill_f32_kernel<d.D, false, d.PAD><<<grid, 256, 0, s>>>(a);
        });
    };
    if (splits > 1) {
        a.split_tiles = (int)((ktiles + splits - 1) / splits);
        splits = (ktiles + a.split_tiles - 1) / a.split_tiles;
        const int64_t rows = m.batch * m.seq_q * m.heads;
        const size_t need = (size_t)(splits * rows) * (sizeof(float2) + (size_t)m.dim * sizeof(float));
        ScratchLease lease(need, s, true);
        if (!lease.status()) {
            // outputs first: splits * rows * D floats keep the (max, sum) pairs 16-byte aligned
            a.part_o = static_cast<float *>(lease.ptr());
            a.part_ml = reinterpret_cast<float2 *>(a.part_o + splits * rows * m.dim);
            const dim3 grid((unsigned)blocks, (unsigned)splits);
            const unsigned cblocks = (unsigned)((rows + 3) / 4);
            launch(grid);
            with_head_dim(m.dim, [&](auto d) {
                prefill_f32_combine_kernel<d.D, d.PAD><<<cblocks, 256, 0, s>>>(a, (int)splits, rows);
            });
            const int rc = check_launch("prefill f32 mfma split");
            const int fin = lease.finish();
            *status = rc ? rc : fin;
            return true;
        }
        a.split_tiles = 0;   // no room: unsplit
    }
    launch(dim3((unsigned)blocks));
    *status = check_launch("prefill f32 mfma");
    return true;
}

bool launch_prefill_mfma(const MhaArgs &m, int dtype, hipStream_t s, int *status) {
    if (dtype == PUTER_F32) return launch_prefill_f32(m, s, status);
    if ((dtype != PUTER_BF16 && dtype != PUTER_F16) || m.dim % 8 || m.dim > 256) return false;
    if (m.dim != 128 && m.seq_q == 1) return false;   // one query row: the general kernel (no 127 padding rows)
    if (m.seq_q > 0x3FFFFFFF || m.seq_k > 0x3FFFFFFF || m.shift > 0x3FFFFFFF || m.shift < -0x3FFFFFFF)
        return false;
    // 32-bit buffer offsets: one 64-row tile of K/V must span at most 2^30 bytes
    if (m.kv_heads * m.dim > 65536 * 128) return false;
    const uintptr_t mask = 15;
    if ((reinterpret_cast<uintptr_t>(m.q) | reinterpret_cast<uintptr_t>(m.k) |
         reinterpret_cast<uintptr_t>(m.v) | reinterpret_cast<uintptr_t>(m.o)) & mask)
        return false;
    PrefillArgs a;
    a.q = static_cast<const uint16_t *>(m.q);
    a.k = static_cast<const uint16_t *>(m.k);
    a.v = static_cast<const uint16_t *>(m.v);
    a.o = static_cast<uint16_t *>(m.o);
    a.batch = (int)m.batch;
    a.seq_q = (int)m.seq_q;
    a.seq_k = (int)m.seq_k;
    a.heads = (int)m.heads;
    a.kv_heads = (int)m.kv_heads;
    a.dim = (int)m.dim;
    a.nan_rows = m.nan_rows;
    a.qtiles = (int)((m.seq_q + fa::BM - 1) / fa::BM);
    a.causal = m.causal;
    a.shift = (int)m.shift;
    // a window of seq_q or more hides no key (a query's distance to a visible key
    // is below seq_q): run it as no window
    a.window = (m.window > 0 && m.window < m.seq_q) ? (int)m.window : 0;
    a.alibi_s = m.alibi != 0.0f ? m.alibi / m.scale : 0.0f;
    a.xcd_map = ((a.batch * a.kv_heads) % 8 == 0) ? 1 : 0;
    a.scale_log2 = m.scale * 1.4426950408889634f;
    const int64_t blocks = (int64_t)a.qtiles * a.batch * a.heads;
    if (blocks > 0x7FFFFFFF) return false;
    const bool bf = dtype == PUTER_BF16, win = a.window > 0 || a.alibi_s != 0.0f;
    // few rows of other head dims, by the estimates above (8 x 8 heads over 200 keys of 256: 11.9
    // us on the general kernel against 18.4; one tile of keys is the padded kernel's up to 128
    // dims).  FlashAttention has another general kernel, slower than the padded one.
    if (bf && !m.nan_rows && m.dim != 64 && m.dim != 128 && (m.seq_k > 64 || m.dim > 128) &&
        general_us(m, false) < padded_us(m, blocks, prefill_tiles(m, 64), 1, false))
        return false;
    const dim3 grid((unsigned)blocks);
    with_head_dim(m.dim, [&](auto d) {
        if (win) {
            if (bf) prefill_kernel<PUTER_BF16, d.D, true, d.PAD><<<grid, 256, 0, s>>>(a);
            else prefill_kernel<PUTER_F16, d.D, true, d.PAD><<<grid, 256, 0, s>>>(a);
        } else {
            if (bf) prefill_kernel<PUTER_BF16, d.D, false, d.PAD><<<grid, 256, 0, s>>>(a);
            else prefill_kernel<PUTER_F16, d.D, false, d.PAD><<<grid, 256, 0, s>>>(a);
        }
    });
    *status = check_launch("prefill mfma");
    return true;
}

}  // namespace puter
