// Full attention of the verify step: M <= 16 new tokens against a KV cache, GQA.
//
// Reference behaviour: the full-attention layers of the mlx_lm decoder the reference
// patches (skinny_mlx/spec.py:24-29 runs them through `model(...)`; KVCache append/trim at
// spec.py:78, 93 and rollback.py:71-73), with per-head q/k RMSNorm and rotate-half RoPE.
//
// Cache layout (per layer): K [Hkv][maxlen][D] and V transposed, Vt [Hkv][D][maxlen], bf16.
// The transposed V makes eight consecutive keys of one dimension contiguous — exactly the
// B operand of the P.V MFMA. The number of tokens already cached (`pos0`) is read from
// device memory, so a launch sequence can be captured once and replayed at any length.
//
// Every query row is computed from its own data only and every reduction runs in a fixed
// order over absolute key positions (chunks of 128 keys), so a token's output
// does not depend on how many tokens share the step.
#include <mutex>

#include "attn_chunk.h"

namespace {

// --- q/k RMSNorm + RoPE + cache store ---------------------------------------------------------

// One wave per (head, token). Heads [0, Hq) are queries (written to q_out), [Hq, Hq+Hkv) keys
// (written to the K cache at slot pos0 + t), [Hq+Hkv, Hq+2Hkv) values (to Vt). Token t is rotated
// to position pos0 + t, or pos0 + rpos[t] for a draft tree (its depth).
__global__ __launch_bounds__(64) void qk_rope_store_kernel(const uint16_t* __restrict__ qkv, int ldq, int Hq, int Hkv,
                                                           const uint16_t* __restrict__ qn, const uint16_t* __restrict__ kn,
                                                           float eps, const int32_t* __restrict__ pos0, float theta,
                                                           const int32_t* __restrict__ tree, int M,
                                                           uint16_t* __restrict__ q_out, uint16_t* __restrict__ kc,
                                                           uint16_t* __restrict__ vt, int maxlen) {
  const int head = blockIdx.x, t = blockIdx.y, lane = threadIdx.x;
  const int slot = pos0[0] + t;                                 // cache slot of token t
  const int pos = pos0[0] + (tree ? tree[1 + M + t] : t);       // its RoPE position
  const uint16_t* src = qkv + (size_t)t * ldq + (size_t)head * kD;
  float a = bf16_bits_to_f32(src[lane]), b = bf16_bits_to_f32(src[lane + 64]);
  if (head >= Hq + Hkv) {  // value: straight into the transposed cache
    const int h = head - Hq - Hkv;
    vt[((size_t)h * kD + lane) * maxlen + slot] = src[lane];
    vt[((size_t)h * kD + lane + 64) * maxlen + slot] = src[lane + 64];
    return;
  }
  const uint16_t* nw = head < Hq ? qn : kn;
  if (nw) {
    const float ss = wave_sum(fmaf(b, b, a * a));
    const float inv = rsqrtf(ss / (float)kD + eps);
    a = bf16_bits_to_f32(f32_to_bf16_bits(a * inv * bf16_bits_to_f32(nw[lane])));
    b = bf16_bits_to_f32(f32_to_bf16_bits(b * inv * bf16_bits_to_f32(nw[lane + 64])));
  }
  // rotate-half RoPE on the pair (i, i + D/2), frequency theta^(-2i/D)
  const float inv_freq = powf(theta, -2.0f * (float)lane / (float)kD);
  float sn, cs;
  sincosf((float)pos * inv_freq, &sn, &cs);
  // explicit fused multiply-adds, the same in the fused attention kernel: its key rows are these bits
  const uint16_t ra = f32_to_bf16_bits(fmaf(a, cs, -(b * sn)));
  const uint16_t rb = f32_to_bf16_bits(fmaf(b, cs, a * sn));
  if (head < Hq) {
    uint16_t* dst = q_out + ((size_t)t * Hq + head) * kD;
    dst[lane] = ra;
    dst[lane + 64] = rb;
  } else {
    uint16_t* dst = kc + ((size_t)(head - Hq) * maxlen + slot) * kD;
    dst[lane] = ra;
    dst[lane + 64] = rb;
  }
}


// The device position comes first among the arguments: it is the kernel's first read, and the
// leading argument dwords arrive preloaded in SGPRs.
template <bool kFused>
__global__ __launch_bounds__(64 * kWaves) void attn_chunk_kernel(const int32_t* __restrict__ pos0,
                                                                 const uint16_t* __restrict__ q, FusedArgs fa, int M,
                                                                 int Hq, int Hkv, uint16_t* __restrict__ kc,
                                                                 uint16_t* __restrict__ vt, int maxlen, float scale,
                                                                 const int32_t* __restrict__ tree,
                                                                 float* __restrict__ part_o, float* __restrict__ part_ml,
                                                                 int nchunk_max) {
  attn_chunk_body<kFused>((int)blockIdx.x, (int)blockIdx.y, pos0, q, fa, M, Hq, Hkv, kc, vt, maxlen, scale, tree, part_o,
                          part_ml, nchunk_max);
}

// The fused chunk stage of a step of at most 16 query rows per kv head (one token, or a short draft):
// there only one wave of a chunk's workgroup has rows, so instead of staging the chunk in LDS for four,
// each wave takes a chunk of its own, its K and V^T fragments straight from memory into registers (the
// same fragments, MFMAs and softmax, so the partials are bitwise attn_chunk_body's). Nothing waits at a
// barrier, and a CU holds 8 chunks' loads in flight instead of 2. Only chunks without new tokens are taken
// this way: the first workgroups of a head run attn_chunk_body over the one or two chunks that hold the new slots, the
// others the chunks below them, 1, 2 or 4 each. The grid is sized for a full cache; how many of its waves a workgroup
// uses goes by the context, so that a short context's chunks in a long cache are on CUs of their own, and the grid's
// workgroups are dealt to the heads anew, the idle ones last: workgroups that end at once between the busy ones left some
// CUs two chunks and others none (4000 keys of 4096 slots, 256 busy of 272: 11.5 us a layer, dealt 10.1). What bounds it at
// a long context is the read of K and V^T; at a short one the chain position, chunk, partial, merge.
// Measured on MI355X, one token, chunk stage and merge of a layer, staged against this: 32768 keys 41.5 / 36.4 us
// (3.69 TB/s of KV; with it, partials of the live rows only and eight merge waves); 8000 keys of 8192 slots 14.0 / 13.1; 1000
// of 8192 10.6 / 9.0; 4000 of 32896 13.6 / 10.4; 4000 of 4096 10.9 / 10.2; 2000 of 2048 9.4 / 9.3; 60 in 2048 or 4096 8.7 / 8.7
// and 9.2 / 9.0. Caches of 256 / 512 / 1280 slots were 1% slower so: up to kFewChunks chunks stay staged. With more rows per
// kv head several waves of a staged chunk have work, and staging serves them all.
constexpr int kFewRows = 16;
constexpr int kFewChunks = 12;        // caches of up to this many chunks stay staged
constexpr int kFewMaxlen = 1 << 22;  // V^T of a head within a buffer descriptor

__device__ __forceinline__ void attn_direct_chunk(int c, int h, int p0, const uint16_t* __restrict__ q, const FusedArgs& fa,
                                                  int M, int Hq, int Hkv, const uint16_t* __restrict__ kc,
                                                  const uint16_t* __restrict__ vt, int maxlen, float scale,
                                                  const int32_t* __restrict__ tree, float* __restrict__ part_o,
                                                  float* __restrict__ part_ml, int nchunk_max) {
  const int lane = threadIdx.x & 63, col = lane & 15, quad = lane >> 4;
  const int G = Hq / Hkv, rows = G * M, key0 = c * kChunk;
  const bool live = col < rows;
  const int t = live ? col / G : 0, qg = live ? col % G : 0;
  // The query side first, then K and V^T: buffer loads whose lane offset is fixed, the tile's in an SGPR.
  const uint16_t* qr = q + (size_t)t * fa.ldq + ((size_t)h * G + qg) * kD;
  const uint16_t* qn = fa.qn ? fa.qn : qr;
  const int pos = p0 + (tree ? tree[1 + M + t] : t);
  u32x4_t raw[4], wq[4];
  f32x4_t cs[2][4];
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) {
    raw[ks] = *reinterpret_cast<const u32x4_t*>(qr + ks * 32 + quad * 8);
    wq[ks] = *reinterpret_cast<const u32x4_t*>(qn + ks * 32 + quad * 8);
  }
  const f32x4_t* rp = reinterpret_cast<const f32x4_t*>(fa.rope + (size_t)pos * 128);
#pragma unroll
  for (int ks = 0; ks < 2; ++ks)
#pragma unroll
    for (int j = 0; j < 4; ++j) cs[ks][j] = rp[(ks * 32 + quad * 8) / 2 + j];
  int tbase = key0;
  uint32_t tmask = 0;
  const int tree0 = tree ? tree[0] : 0;
  const uint32_t mask = tree ? (uint32_t)tree[1 + t] : 0u;
  if (live) {
    tbase = tree ? p0 - tree0 : p0 + t + 1;
    tmask = mask;
  }
  const __amdgpu_buffer_rsrc_t rk = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t*>(kc) + ((size_t)h * maxlen + key0) * kD, (short)0, kChunk * kD * 2, 0x00020000);
  const __amdgpu_buffer_rsrc_t rv = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t*>(vt) + (size_t)h * kD * maxlen + key0, (short)0, ((kD - 1) * maxlen + kChunk) * 2, 0x00020000);
  const uint32_t koff = (uint32_t)((8 * (col >> 2) + (col & 3)) * kD + quad * 8) * 2u;
  const uint32_t voff = (uint32_t)(col * maxlen + quad * 8) * 2u;
  bf16x8_t kf[8][4], vf[8][4];
#pragma unroll
  for (int kt = 0; kt < 8; ++kt)
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
      kf[kt][ks] = __builtin_bit_cast(bf16x8_t, __builtin_amdgcn_raw_buffer_load_b128(
                                                    rk, koff, ((32 * (kt >> 1) + 4 * (kt & 1)) * kD + ks * 32) * 2, 0));
  bf16x8_t qf[4] = {};
  if (live) rotate_query(raw, wq, cs, fa.qn != nullptr, fa.eps, qf);
  const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
  float s[8][4];
#pragma unroll
  for (int kt = 0; kt < 8; ++kt) {
    f32x4_t acc = zero;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) acc = mfma16x16x32(kf[kt][ks], qf[ks], acc);
#pragma unroll
    for (int i = 0; i < 4; ++i) s[kt][i] = acc[i];
    // the V^T fragments follow the K tiles into flight, in the registers those leave
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
      vf[kt][ks] = __builtin_bit_cast(bf16x8_t, __builtin_amdgcn_raw_buffer_load_b128(rv, voff, (kt * 16 * maxlen + ks * 32) * 2, 0));
    __builtin_amdgcn_sched_barrier(0);
  }
  u32x4_t pa[4];
  float mx, sum;
  attn_softmax(s, key0, tbase, tmask, scale, pa, mx, sum);
  f32x4_t o[8];
#pragma unroll
  for (int dt = 0; dt < 8; ++dt) {
    o[dt] = zero;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) o[dt] = mfma16x16x32(__builtin_bit_cast(bf16x8_t, pa[ks]), vf[dt][ks], o[dt]);
  }
  const size_t base = ((size_t)h * nchunk_max + c) * kRowsMax;
  attn_store_rows(o, mx, sum, rows, part_o + base * kD, part_ml + base * 2);
}

__global__ __launch_bounds__(64 * kWaves) void attn_few_kernel(const int32_t* __restrict__ pos0,
                                                               const uint16_t* __restrict__ q, FusedArgs fa, int M, int Hq,
                                                               int Hkv, uint16_t* __restrict__ kc, uint16_t* __restrict__ vt,
                                                               int maxlen, float scale, const int32_t* __restrict__ tree,
                                                               float* __restrict__ part_o, float* __restrict__ part_ml,
                                                               int nchunk_max, int n) {
  const int wave = wave_id(), p0 = pos0[0];
  const int fresh = max(p0, 0) / kChunk;  // the first chunk with new slots
  const int last = min((p0 + M - 1) / kChunk, nchunk_max - 1);  // and the last (slots past the cache are dropped)
  const int old = min(fresh, nchunk_max);
  const int sh = old > 2 * n ? 2 : old > n ? 1 : 0;
  const int staged = max(0, last - fresh + 1), used = max(1, staged + ((old + (1 << sh) - 1) >> sh));  // of each head
  int h = blockIdx.y, b = blockIdx.x, first = 2;  // workgroup of the head, and the first with a chunk per wave
  if (sh < 2) {  // (with four chunks each the grid is at least half used, and as it stands no slower)
    const auto [quot, rem] = work_index(h * (2 + n) + b, used);
    if (quot >= Hkv) return;
    h = quot;
    b = rem;
    first = staged;
  }
  if (b < first) {
    if (b < staged)
      attn_chunk_body<true>(fresh + b, h, pos0, q, fa, M, Hq, Hkv, kc, vt, maxlen, scale, tree, part_o, part_ml, nchunk_max);
    return;
  }
  const int c = ((b - first) << sh) + wave;
  if ((wave >> sh) || c >= old) return;
  attn_direct_chunk(c, h, p0, q, fa, M, Hq, Hkv, kc, vt, maxlen, scale, tree, part_o, part_ml, nchunk_max);
}

// One workgroup per (q head, token): merge the chunk partials, normalise, store bf16. Chunks are
// taken in blocks of 32 by absolute index: all of a block's loads are issued together (lane c holds
// chunk c's statistics, every lane its two dims of every chunk's partial row), then the block is
// folded into running sums in chunk order, rescaled when the running maximum grows. A block past
// a row's position holds only empty chunks and rescales by exactly 1, so the result does not
// depend on how many tokens share the step. With W waves (caches of more than one block), wave v
// folds blocks v, v + W, ... into sums of its own, and wave 0 then folds waves 1 .. W-1 into its
// sums in that order, a wave without keys for the row by exactly 1 and 0: W is fixed by the cache
// size, so every step over one cache merges a row's blocks the same way.
constexpr int kCombineBlock = 32;
constexpr int kCombineWaves = 4;      // waves of the merge for caches of more than kCombineBlock chunks
constexpr int kCombineWavesLong = 8;  // and of more than kCombineLong chunks
constexpr int kCombineLong = 128;

// The merge of one row (chunk c's partial at head_base + c * kRowsMax; pos0[0] + tokens keys) into
// dst[128]; false in the waves that only helped. kPrompt reads the chunk count first, since a prompt's
// early tokens see few of the chunk slots.
template <int W, bool kPrompt>
__device__ __forceinline__ bool combine_row(const float* __restrict__ part_o, const float* __restrict__ part_ml,
                                            size_t head_base, const int32_t* __restrict__ pos0, int tokens,
                                            int nchunk_max, uint16_t* __restrict__ dst) {
  const int lane = threadIdx.x & 63, v = W > 1 ? wave_id() : 0;
  const int first = v * kCombineBlock;                                // this wave's first block
  // The first block's partials are loaded before the chunk count is known (it needs *pos0):
  // every chunk the workspace holds up to kCombineBlock, the ones past the context discarded below
  // by selection (their stale values never enter an arithmetic operation). Waves past the fourth (of a long cache,
  // which the context seldom fills) take the count first: 16 tokens over 60 / 4000 keys in 32896 slots 20.3 / 25.4 us a
  // layer when all eight load ahead, 14.5 / 21.2 so, 14.0 / 20.9 with four waves in all; 32768 keys the same.
  int pre = kPrompt ? 0 : max(0, min(kCombineBlock, nchunk_max - first));
  if constexpr (!kPrompt && W > kCombineWaves)
    if (v >= kCombineWaves) pre = max(0, min(pre, (pos0[0] + tokens + kChunk - 1) / kChunk - first));
  float mc_pre = -INFINITY, lc_pre = 0.f;
  float o0[kCombineBlock], o1[kCombineBlock];
  if (lane < pre) {
    mc_pre = part_ml[(head_base + (size_t)(first + lane) * kRowsMax) * 2];
    lc_pre = part_ml[(head_base + (size_t)(first + lane) * kRowsMax) * 2 + 1];
  }
#pragma unroll
  for (int j = 0; j < kCombineBlock; ++j) {
    o0[j] = o1[j] = 0.f;
    if (j < pre) {
      const float* po = part_o + (head_base + (size_t)(first + j) * kRowsMax) * kD;
      o0[j] = po[lane];
      o1[j] = po[lane + 64];
    }
  }
  const int total = pos0[0] + tokens;
  // (the workspace holds nchunk_max chunks; no read past them whatever *pos0 says)
  const int nch = min((total + kChunk - 1) / kChunk, nchunk_max);
  float run_m = -INFINITY, run_l = 0.f, a0 = 0.f, a1 = 0.f;
  for (int c0 = first; c0 < nch; c0 += W * kCombineBlock) {
    const int nb = min(kCombineBlock, nch - c0);
    float mc = -INFINITY, lc = 0.f;
    if (!kPrompt && c0 == first) {
      mc = lane < nb ? mc_pre : -INFINITY;
      lc = lane < nb ? lc_pre : 0.f;
#pragma unroll
      for (int j = 0; j < kCombineBlock; ++j) {
        o0[j] = j < nb ? o0[j] : 0.f;
        o1[j] = j < nb ? o1[j] : 0.f;
      }
    } else {
      if (lane < nb) {
        mc = part_ml[(head_base + (size_t)(c0 + lane) * kRowsMax) * 2];
        lc = part_ml[(head_base + (size_t)(c0 + lane) * kRowsMax) * 2 + 1];
      }
#pragma unroll
      for (int j = 0; j < kCombineBlock; ++j) {
        o0[j] = o1[j] = 0.f;
        if (j < nb) {
          const float* po = part_o + (head_base + (size_t)(c0 + j) * kRowsMax) * kD;
          o0[j] = po[lane];
          o1[j] = po[lane + 64];
        }
      }
    }
    float bm = mc;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) bm = fmaxf(bm, __shfl_xor(bm, off, 64));
    const float new_m = fmaxf(run_m, bm);
    const float keep = run_m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(run_m - new_m);
    run_l *= keep;
    a0 *= keep;
    a1 *= keep;
    const float wgt = mc == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mc - new_m);
#pragma unroll
    for (int j = 0; j < kCombineBlock; ++j) {
      if (j < nb) {  // lane j's weight and sum, broadcast by v_readlane (j is a constant here)
        const float wj = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(wgt), j));
        run_l = fmaf(__int_as_float(__builtin_amdgcn_readlane(__float_as_int(lc), j)), wj, run_l);
        a0 = fmaf(o0[j], wj, a0);
        a1 = fmaf(o1[j], wj, a1);
      }
    }
    run_m = new_m;
  }
  if constexpr (W > 1) {
    // A context of one block (up to 4096 keys): no other wave has keys, and none is waited for. One token over 60 keys
    // in 32896 slots 9.47 -> 9.15 us a layer (9.25 with the four waves and their barrier that it had before eight).
    if (nch <= kCombineBlock) {
      if (v > 0) return false;
      a0 += 0.f;  // as adding them would: no zero keeps a sign
      a1 += 0.f;
    } else {
      __shared__ float sm[W], sl[W], sa[W][2][64];
      if (lane == 0) {
        sm[v] = run_m;
        sl[v] = run_l;
      }
      sa[v][0][lane] = a0;
      sa[v][1][lane] = a1;
      __syncthreads();
      if (v > 0) return false;
#pragma unroll
      for (int u = 1; u < W; ++u) {
        const float mu = sm[u], lu = sl[u];
        const float new_m = fmaxf(run_m, mu);
        const float k0 = run_m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(run_m - new_m);
        const float ku = mu == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mu - new_m);
        run_l = fmaf(lu, ku, run_l * k0);
        a0 = fmaf(sa[u][0][lane], ku, a0 * k0);
        a1 = fmaf(sa[u][1][lane], ku, a1 * k0);
        run_m = new_m;
      }
    }
  }
  const float inv = run_l > 0.f ? 1.0f / run_l : 0.f;
  dst[lane] = f32_to_bf16_bits(a0 * inv);
  dst[lane + 64] = f32_to_bf16_bits(a1 * inv);
  return true;
}

template <int W>
__global__ __launch_bounds__(64 * W) void attn_combine_kernel(const float* __restrict__ part_o,
                                                              const float* __restrict__ part_ml, int M, int Hq, int Hkv,
                                                              const int32_t* __restrict__ pos0, int nchunk_max,
                                                              uint16_t* __restrict__ out, uint32_t* __restrict__ reset,
                                                              int reset_ld, int reset_words) {
  const int hq = blockIdx.x, t = blockIdx.y, lane = threadIdx.x & 63;
  const int G = Hq / Hkv, h = hq / G, row = t * G + hq % G;
  const size_t head_base = (size_t)h * nchunk_max * kRowsMax + row;  // chunk c at + c * kRowsMax
  if (!combine_row<W, false>(part_o, part_ml, head_base, pos0, M, nchunk_max, out + ((size_t)t * Hq + hq) * kD)) return;
  if (reset) {  // every chunk workgroup has read the hand-off rows: back to "not yet written"
    const int per = (reset_words + Hq - 1) / Hq;
    const int w1 = min(reset_words, (hq + 1) * per);
    uint32_t* r = reset + (size_t)t * reset_ld;
    for (int w = hq * per + lane; w < w1; w += 64)
      __hip_atomic_store(r + w, 0xffffffffu, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

// --- the attention of a prompt: more tokens than one step holds ---------------------------------
//
// The prompt's tokens are taken in pieces of kPiece, and every row's arithmetic is that of the fused
// step kernels over its piece (the same query and key rows, chunk partials and merge, which depend on
// absolute key positions only), so a prompt's rows and cache entries are bitwise those of 16-token steps.
// Three launches instead of two per piece: (1) queries into a workspace, keys and values into the
// caches; (2) one workgroup per (kPieceGroup pieces, chunk, kv head), which stages the chunk once for all
// of them; (3) one workgroup per (query head, token) for the merge.
constexpr int kPiece = 16;      // tokens per piece
constexpr int kPieceGroup = 4;  // pieces that share a staged chunk

struct PromptArgs {
  int M, Hq, Hkv;
  const uint16_t* qn;
  const uint16_t* kn;
  float eps;
  const float* rope;  // [positions][64] (cos, sin)
  uint16_t* q_out;    // [M][Hq][128]
  uint16_t* kc;
  uint16_t* vt;
  int maxlen;
};

// (1) Workgroups [0, nq): 64 query rows each, a wave per 16 (lane (col, quad) as in the chunk kernel);
// [nq, nq + nk): a key row per wave (lanes d and d + 64); the rest: 64 tokens of one value head, turned in
// LDS so that the stores into V^T run along the cache slots.
__global__ __launch_bounds__(256) void prompt_qkv_kernel(const int32_t* __restrict__ pos0, const uint16_t* __restrict__ qkv,
                                                         int ldq, int nq, int nk, const PromptArgs pa) {
  __shared__ uint16_t vl[64][kD + 2];
  const int lane = threadIdx.x & 63, wave = wave_id();
  const int p0 = pos0[0];
  const int M = pa.M, Hq = pa.Hq, Hkv = pa.Hkv;
  const int b = blockIdx.x;
  if (b < nq) {
    const int col = lane & 15, quad = lane >> 4;
    const int r = b * 64 + wave * 16 + col;
    const bool live = r < M * Hq;
    const int t = live ? r / Hq : 0, hq = live ? r % Hq : 0;
    const uint16_t* src = qkv + (size_t)t * ldq + (size_t)hq * kD;
    const uint16_t* qn = pa.qn ? pa.qn : src;
    const f32x4_t* rp = reinterpret_cast<const f32x4_t*>(pa.rope + (size_t)(p0 + t) * 128);
    u32x4_t raw[4], wq[4];
    f32x4_t cs[2][4];
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      raw[ks] = *reinterpret_cast<const u32x4_t*>(src + ks * 32 + quad * 8);
      wq[ks] = *reinterpret_cast<const u32x4_t*>(qn + ks * 32 + quad * 8);
    }
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int j = 0; j < 4; ++j) cs[ks][j] = rp[(ks * 32 + quad * 8) / 2 + j];
    bf16x8_t qf[4];
    rotate_query(raw, wq, cs, pa.qn != nullptr, pa.eps, qf);
    if (live) {
      uint16_t* dst = pa.q_out + (size_t)r * kD;
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) *reinterpret_cast<bf16x8_t*>(dst + ks * 32 + quad * 8) = qf[ks];
    }
  } else if (b < nq + nk) {
    const int r = (b - nq) * 4 + wave;
    if (r >= M * Hkv) return;
    const int t = r / Hkv, h = r % Hkv, slot = p0 + t;
    if (slot >= pa.maxlen) return;  // tokens past the cache are dropped, as the steps drop them
    const uint16_t* src = qkv + (size_t)t * ldq + (size_t)(Hq + h) * kD;
    float ka = bf16_bits_to_f32(src[lane]), kb = bf16_bits_to_f32(src[lane + 64]);
    const float2 cs = reinterpret_cast<const float2*>(pa.rope)[(size_t)slot * 64 + lane];
    if (pa.kn) {
      const float w0 = bf16_bits_to_f32(pa.kn[lane]), w1 = bf16_bits_to_f32(pa.kn[lane + 64]);
      const float inv = rsqrtf(wave_sum(fmaf(kb, kb, ka * ka)) / (float)kD + pa.eps);
      ka = bf16_bits_to_f32(f32_to_bf16_bits(ka * inv * w0));
      kb = bf16_bits_to_f32(f32_to_bf16_bits(kb * inv * w1));
    }
    uint16_t* dst = pa.kc + ((size_t)h * pa.maxlen + slot) * kD;
    dst[lane] = f32_to_bf16_bits(fmaf(ka, cs.x, -(kb * cs.y)));
    dst[lane + 64] = f32_to_bf16_bits(fmaf(kb, cs.x, ka * cs.y));
  } else {
    const int i = b - nq - nk, h = i % Hkv, t0 = i / Hkv * 64;
    for (int e = threadIdx.x; e < 64 * (kD / 8); e += 256) {
      const int t = e / (kD / 8), piece = e % (kD / 8);
      const u32x4_t v = *reinterpret_cast<const u32x4_t*>(qkv + (size_t)min(t0 + t, M - 1) * ldq + (size_t)(Hq + Hkv + h) * kD + piece * 8);
#pragma unroll
      for (int k = 0; k < 4; ++k) *reinterpret_cast<uint32_t*>(&vl[t][piece * 8 + 2 * k]) = v[k];
    }
    __syncthreads();
    if (t0 + lane < M && p0 + t0 + lane < pa.maxlen)
      for (int d = wave; d < kD; d += 4) pa.vt[((size_t)h * kD + d) * pa.maxlen + p0 + t0 + lane] = vl[lane][d];
  }
}

// (2) Workgroup (chunk c, kv head h, group g of pieces): pieces z0 + kPieceGroup g .. of the launch's
// pieces [z0, z1); piece z's partials at (z - z0) * Hkv * nch chunk slots. The caches hold all of the prompt's keys and
// values already, of which a step would see those up to its own. The others' weights are 0, but 0 times an infinity or a NaN
// is a NaN: in a chunk with such a value the pieces, which run from the last to the first, clear what they do not see. (In
// every chunk at the prompt's edge that took 6% of 100 tokens' attention; looking for such values takes less than 1%.)
__global__ __launch_bounds__(64 * kWaves) void prompt_chunk_kernel(const int32_t* __restrict__ pos0,
                                                                   const uint16_t* __restrict__ q, int M, int Hq, int Hkv,
                                                                   const uint16_t* __restrict__ kc,
                                                                   const uint16_t* __restrict__ vt, int maxlen, float scale,
                                                                   int z0, int z1, int nch, float* __restrict__ part_o,
                                                                   float* __restrict__ part_ml) {
  __shared__ __attribute__((aligned(16))) uint16_t ks_lds[kChunk * kPitch];
  __shared__ __attribute__((aligned(16))) uint16_t vs_lds[kD * kPitch];
  __shared__ int odd_lds[kWaves];
  const int lane = threadIdx.x & 63, wave = wave_id();
  const int c = blockIdx.x, h = blockIdx.y, p0 = pos0[0], G = Hq / Hkv;
  const int za = z0 + (int)blockIdx.z * kPieceGroup, zb = min(za + kPieceGroup, z1);
  const int key0 = c * kChunk;
  if (key0 >= p0 + min(M, zb * kPiece)) return;  // past the last piece's keys
  const u32x4_t* kh = reinterpret_cast<const u32x4_t*>(kc + ((size_t)h * maxlen + key0) * kD);
  const uint16_t* vh = vt + (size_t)h * kD * maxlen + key0;
  u32x4_t kr[8], vr[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int e = threadIdx.x + i * 64 * kWaves;  // piece e: row e / 16, column piece e % 16
    kr[i] = kh[e];
    vr[i] = *reinterpret_cast<const u32x4_t*>(vh + (size_t)(e >> 4) * maxlen + (e & 15) * 8);
  }
  const int col = lane & 15, quad = lane >> 4, qrow = wave * 16 + col;
  bf16x8_t qf[kPieceGroup][4];
#pragma unroll
  for (int i = 0; i < kPieceGroup; ++i) {
    const int t0 = (za + i) * kPiece, rows = G * min(kPiece, M - t0);
    const bool live = za + i < zb && qrow < rows;
    const uint16_t* qr = q + ((size_t)(live ? t0 + qrow / G : 0) * Hq + h * G + (live ? qrow % G : 0)) * kD;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      qf[i][ks] = *reinterpret_cast<const bf16x8_t*>(qr + ks * 32 + quad * 8);
      if (!live) qf[i][ks] = bf16x8_t{};
    }
  }
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int e = threadIdx.x + i * 64 * kWaves;
    *reinterpret_cast<u32x4_t*>(&ks_lds[(e >> 4) * kPitch + (e & 15) * 8]) = kr[i];
    *reinterpret_cast<u32x4_t*>(&vs_lds[(e >> 4) * kPitch + (e & 15) * 8]) = vr[i];
  }
  const bool edge = key0 + kChunk > p0 + min(M, (za + 1) * kPiece);  // holds slots that the first piece does not see
  if (edge) odd_lds[wave] = any_not_finite(vr);
  __syncthreads();
  bool odd = false;
  if (edge) {
#pragma unroll
    for (int w = 0; w < kWaves; ++w) odd |= __builtin_amdgcn_readfirstlane(odd_lds[w]) != 0;
  }
  int seen = kChunk;
#pragma unroll
  for (int i = kPieceGroup - 1; i >= 0; --i) {
    const int z = za + i, t0 = z * kPiece;
    if (z >= zb) continue;
    const int mb = min(kPiece, M - t0), end = min(p0 + t0 + mb - key0, kChunk);
    if (end <= 0) break;
    if (odd && end < seen) {
      __syncthreads();
      for (int e = threadIdx.x; e < kD * (seen - end); e += 64 * kWaves) vs_lds[e % kD * kPitch + end + e / kD] = 0;
      __syncthreads();
      seen = end;
    }
    if (wave * 16 >= G * mb) continue;
    const int tbase = qrow < G * mb ? p0 + t0 + qrow / G + 1 : key0;
    const size_t base = (((size_t)(z - z0) * Hkv + h) * nch + c) * kRowsMax + wave * 16;
    attn_rows(ks_lds, vs_lds, qf[i], key0, tbase, 0u, scale, G * mb - wave * 16, part_o + base * kD, part_ml + base * 2);
  }
}

// (3) Token t0 + blockIdx.y (t0 = kPiece z0).
template <int W>
__global__ __launch_bounds__(64 * W) void prompt_combine_kernel(const float* __restrict__ part_o,
                                                                const float* __restrict__ part_ml, int M, int Hq, int Hkv,
                                                                const int32_t* __restrict__ pos0, int z0, int nch,
                                                                uint16_t* __restrict__ out) {
  const int hq = blockIdx.x, t = z0 * kPiece + (int)blockIdx.y, z = t / kPiece;
  const int G = Hq / Hkv, h = hq / G, row = (t % kPiece) * G + hq % G;
  const size_t head_base = (((size_t)(z - z0) * Hkv + h) * nch) * kRowsMax + row;
  combine_row<W, true>(part_o, part_ml, head_base, pos0, min(M, (z + 1) * kPiece), nch, out + ((size_t)t * Hq + hq) * kD);
}

// cos/sin table of rotate-half RoPE: table[pos][i] = (cos, sin)(pos * theta^(-2i/128)), i < 64,
// by the same expressions as qk_rope_store_kernel.
__global__ void rope_table_kernel(float theta, int positions, float* __restrict__ table) {
  const int idx = blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= positions * 64) return;
  const int pos = idx >> 6, i = idx & 63;
  const float inv_freq = powf(theta, -2.0f * (float)i / (float)kD);
  float sn, cs;
  sincosf((float)pos * inv_freq, &sn, &cs);
  table[2 * idx] = cs;
  table[2 * idx + 1] = sn;
}

}  // namespace

int attn_combine_launch(const float* part_o, const float* part_ml, int M, int Hq, int Hkv, const int32_t* pos0,
                        int nchunk_max, uint16_t* out, uint32_t* reset, int reset_ld, int reset_words,
                        hipStream_t stream) {
  if (nchunk_max > kCombineLong)
    hipLaunchKernelGGL(attn_combine_kernel<kCombineWavesLong>, dim3(Hq, M), dim3(64 * kCombineWavesLong), 0, stream, part_o,
                       part_ml, M, Hq, Hkv, pos0, nchunk_max, out, reset, reset_ld, reset_words);
  else if (nchunk_max > kCombineBlock)
    hipLaunchKernelGGL(attn_combine_kernel<kCombineWaves>, dim3(Hq, M), dim3(64 * kCombineWaves), 0, stream, part_o,
                       part_ml, M, Hq, Hkv, pos0, nchunk_max, out, reset, reset_ld, reset_words);
  else
    hipLaunchKernelGGL(attn_combine_kernel<1>, dim3(Hq, M), dim3(64), 0, stream, part_o, part_ml, M, Hq, Hkv, pos0,
                       nchunk_max, out, reset, reset_ld, reset_words);
  return skinny_check_launch("attention combine");
}

extern "C" int skinny_rope_table(float theta, int positions, float* table, void* stream) {
  SKINNY_CHECK_ARG(table && positions >= 1 && theta > 1.f, "rope_table: bad arguments");
  hipLaunchKernelGGL(rope_table_kernel, dim3((positions * 64 + 255) / 256), dim3(256), 0, (hipStream_t)stream, theta,
                     positions, table);
  return skinny_check_launch("rope_table");
}

extern "C" int skinny_qk_rope_store(const uint16_t* qkv, int ldq, int M, int Hq, int Hkv, int D,
                                    const uint16_t* q_norm, const uint16_t* k_norm, float eps, const int32_t* pos0,
                                    float theta, const int32_t* tree, uint16_t* q_out, uint16_t* k_cache,
                                    uint16_t* vt_cache, int maxlen, void* stream) {
  SKINNY_CHECK_ARG(qkv && pos0 && q_out && k_cache && vt_cache, "qk_rope_store: null pointer");
  SKINNY_CHECK_ARG(D == kD, "qk_rope_store: head dim %d unsupported (only %d)", D, kD);
  SKINNY_CHECK_ARG(M >= 1 && M <= 65535 && Hq >= 1 && Hkv >= 1 && Hq % Hkv == 0, "qk_rope_store: bad heads/tokens");
  SKINNY_CHECK_ARG(ldq >= (Hq + 2 * Hkv) * D, "qk_rope_store: ldq=%d too small", ldq);
  SKINNY_CHECK_ARG(maxlen >= 1, "qk_rope_store: bad maxlen");
  SKINNY_CHECK_ARG(!tree || M <= 32, "qk_rope_store: a draft tree holds at most 32 tokens (M=%d)", M);
  hipLaunchKernelGGL(qk_rope_store_kernel, dim3(Hq + 2 * Hkv, M), dim3(64), 0, (hipStream_t)stream, qkv, ldq, Hq, Hkv,
                     q_norm, k_norm, eps, pos0, theta, tree, M, q_out, k_cache, vt_cache, maxlen);
  return skinny_check_launch("qk_rope_store");
}

extern "C" size_t skinny_attn_workspace_bytes(int Hkv, int maxlen) {
  const size_t nch = (size_t)((maxlen + kChunk - 1) / kChunk);
  return (size_t)Hkv * nch * kRowsMax * (kD + 2) * sizeof(float);
}

extern "C" int skinny_attention_bf16(const uint16_t* q, int M, int Hq, int Hkv, int D, const uint16_t* k_cache,
                                     const uint16_t* vt_cache, int maxlen, const int32_t* pos0, float scale,
                                     const int32_t* tree, float* workspace, size_t workspace_bytes, uint16_t* out,
                                     void* stream) {
  SKINNY_CHECK_ARG(q && k_cache && vt_cache && pos0 && workspace && out, "attention: null pointer");
  SKINNY_CHECK_ARG(D == kD, "attention: head dim %d unsupported (only %d)", D, kD);
  SKINNY_CHECK_ARG(Hkv >= 1 && Hq % Hkv == 0, "attention: Hq=%d not a multiple of Hkv=%d", Hq, Hkv);
  SKINNY_CHECK_ARG(M >= 1 && (Hq / Hkv) * M <= kRowsMax, "attention: %d query rows per kv head exceed %d",
                   (Hq / Hkv) * M, kRowsMax);
  SKINNY_CHECK_ARG(maxlen >= kChunk && maxlen % kChunk == 0, "attention: maxlen=%d must be a multiple of %d", maxlen,
                   kChunk);
  SKINNY_CHECK_ARG(workspace_bytes >= skinny_attn_workspace_bytes(Hkv, maxlen), "attention: workspace too small");
  SKINNY_CHECK_ARG(skinny_aligned(q, 16) && skinny_aligned(k_cache, 16) && skinny_aligned(vt_cache, 16),
                   "attention: q and caches must be 16-byte aligned");
  const int nch = maxlen / kChunk;
  float* part_o = workspace;
  float* part_ml = workspace + (size_t)Hkv * nch * kRowsMax * kD;
  const FusedArgs none{0, nullptr, nullptr, 0.f, nullptr};
  hipLaunchKernelGGL(attn_chunk_kernel<false>, dim3(nch, Hkv), dim3(64 * kWaves), 0, (hipStream_t)stream, pos0, q, none, M,
                     Hq, Hkv, const_cast<uint16_t*>(k_cache), const_cast<uint16_t*>(vt_cache), maxlen, scale, tree,
                     part_o, part_ml, nch);
  int rc = skinny_check_launch("attention");
  if (rc) return rc;
  return attn_combine_launch(part_o, part_ml, M, Hq, Hkv, pos0, nch, out, nullptr, 0, 0, (hipStream_t)stream);
}

// Validation and launches of the fused attention, given the chunk-partial workspace.
static int attention_fused(const uint16_t* qkv, int ldq, int M, int Hq, int Hkv, int D, const uint16_t* q_norm,
                           const uint16_t* k_norm, float eps, const float* rope_table, int rope_positions,
                           const int32_t* pos0, const int32_t* tree, uint16_t* k_cache, uint16_t* vt_cache,
                           int maxlen, float scale, float* workspace, size_t workspace_bytes, uint16_t* out,
                           void* stream) {
  SKINNY_CHECK_ARG(qkv && rope_table && k_cache && vt_cache && pos0 && workspace && out, "attention: null pointer");
  SKINNY_CHECK_ARG(D == kD, "attention: head dim %d unsupported (only %d)", D, kD);
  SKINNY_CHECK_ARG(Hkv >= 1 && Hq % Hkv == 0, "attention: Hq=%d not a multiple of Hkv=%d", Hq, Hkv);
  SKINNY_CHECK_ARG(M >= 1 && M <= kFusedMaxTokens && (Hq / Hkv) * M <= kRowsMax,
                   "attention: M=%d (at most %d) with %d query rows per kv head (at most %d)", M, kFusedMaxTokens,
                   (Hq / Hkv) * M, kRowsMax);
  SKINNY_CHECK_ARG(ldq >= (Hq + 2 * Hkv) * D && ldq % 8 == 0, "attention: ldq=%d too small or not a multiple of 8",
                   ldq);
  SKINNY_CHECK_ARG(maxlen >= kChunk && maxlen % kChunk == 0 && rope_positions >= maxlen,
                   "attention: maxlen=%d must be a multiple of %d and within the RoPE table (%d)", maxlen, kChunk,
                   rope_positions);
  SKINNY_CHECK_ARG(workspace_bytes >= skinny_attn_workspace_bytes(Hkv, maxlen), "attention: workspace too small");
  SKINNY_CHECK_ARG(skinny_aligned(qkv, 16) && skinny_aligned(k_cache, 16) && skinny_aligned(vt_cache, 16) &&
                       skinny_aligned(rope_table, 16) && (!q_norm || skinny_aligned(q_norm, 16)),
                   "attention: qkv, caches, table and q_norm must be 16-byte aligned");
  const int nch = maxlen / kChunk;
  float* part_o = workspace;
  float* part_ml = workspace + (size_t)Hkv * nch * kRowsMax * kD;
  const FusedArgs fa{ldq, q_norm, k_norm, eps, rope_table};
  if ((Hq / Hkv) * M <= kFewRows && nch > kFewChunks && maxlen <= kFewMaxlen) {
    const int per = nch * Hkv <= 512 ? 1 : nch * Hkv <= 1024 ? 2 : kWaves, n = (nch + per - 1) / per;
    hipLaunchKernelGGL(attn_few_kernel, dim3(2 + n, Hkv), dim3(64 * kWaves), 0, (hipStream_t)stream, pos0, qkv, fa, M, Hq, Hkv,
                       k_cache, vt_cache, maxlen, scale, tree, part_o, part_ml, nch, n);
  } else {
    hipLaunchKernelGGL(attn_chunk_kernel<true>, dim3(nch, Hkv), dim3(64 * kWaves), 0, (hipStream_t)stream, pos0, qkv, fa, M,
                       Hq, Hkv, k_cache, vt_cache, maxlen, scale, tree, part_o, part_ml, nch);
  }
  int rc = skinny_check_launch("attention");
  if (rc) return rc;
  return attn_combine_launch(part_o, part_ml, M, Hq, Hkv, pos0, nch, out, nullptr, 0, 0, (hipStream_t)stream);
}

extern "C" int skinny_attention_fused_bf16(const uint16_t* qkv, int ldq, int M, int Hq, int Hkv, int D,
                                           const uint16_t* q_norm, const uint16_t* k_norm, float eps,
                                           const float* rope_table, int rope_positions, const int32_t* pos0,
                                           const int32_t* tree, uint16_t* k_cache, uint16_t* vt_cache, int maxlen,
                                           float scale, float* workspace, size_t workspace_bytes, uint16_t* out,
                                           void* stream) {
  return attention_fused(qkv, ldq, M, Hq, Hkv, D, q_norm, k_norm, eps, rope_table, rope_positions, pos0, tree,
                         k_cache, vt_cache, maxlen, scale, workspace, workspace_bytes, out, stream);
}

// Workspace of a prompt's attention: the rotated queries, then the partials of as many pieces as fit
// kPromptPartBytes (at least one group of pieces).
constexpr size_t kPromptPartBytes = (size_t)256 << 20;

static size_t prompt_piece_bytes(int Hkv, int nch) { return (size_t)Hkv * nch * kRowsMax * (kD + 2) * sizeof(float); }

static size_t prompt_query_bytes(int M, int Hq) { return ((size_t)M * Hq * kD * 2 + 255) & ~(size_t)255; }

extern "C" size_t skinny_attn_prompt_workspace_bytes(int M, int Hq, int Hkv, int keys) {
  if (M < 1 || Hq < 1 || Hkv < 1 || keys < 1) return 0;
  const size_t piece = prompt_piece_bytes(Hkv, (keys + kChunk - 1) / kChunk);
  const size_t all = (size_t)((M + kPiece - 1) / kPiece) * piece, group = kPieceGroup * piece;
  const size_t most = kPromptPartBytes / group * group;
  return prompt_query_bytes(M, Hq) + (all <= most ? all : most > group ? most : group < all ? group : all);
}

extern "C" int skinny_attention_prompt_bf16(const uint16_t* qkv, int ldq, int M, int Hq, int Hkv, int D,
                                            const uint16_t* q_norm, const uint16_t* k_norm, float eps,
                                            const float* rope_table, int rope_positions, const int32_t* pos0, int keys,
                                            uint16_t* k_cache, uint16_t* vt_cache, int maxlen, float scale,
                                            void* workspace, size_t workspace_bytes, uint16_t* out, void* stream) {
  SKINNY_CHECK_ARG(qkv && rope_table && k_cache && vt_cache && pos0 && workspace && out, "attention prompt: null pointer");
  SKINNY_CHECK_ARG(D == kD, "attention prompt: head dim %d unsupported (only %d)", D, kD);
  SKINNY_CHECK_ARG(Hkv >= 1 && Hq % Hkv == 0 && (Hq / Hkv) * kPiece <= kRowsMax,
                   "attention prompt: Hq=%d must be a multiple of Hkv=%d, at most %d query heads each", Hq, Hkv,
                   kRowsMax / kPiece);
  SKINNY_CHECK_ARG(M >= 1 && M <= 65535 && keys >= M && keys <= maxlen, "attention prompt: M=%d (at most 65535), keys=%d in [M, maxlen=%d]",
                   M, keys, maxlen);
  SKINNY_CHECK_ARG(ldq >= (Hq + 2 * Hkv) * D && ldq % 8 == 0, "attention prompt: ldq=%d too small or not a multiple of 8", ldq);
  SKINNY_CHECK_ARG(maxlen >= kChunk && maxlen % kChunk == 0 && rope_positions >= maxlen,
                   "attention prompt: maxlen=%d must be a multiple of %d and within the RoPE table (%d)", maxlen, kChunk,
                   rope_positions);
  SKINNY_CHECK_ARG(skinny_aligned(qkv, 16) && skinny_aligned(k_cache, 16) && skinny_aligned(vt_cache, 16) &&
                       skinny_aligned(rope_table, 16) && (!q_norm || skinny_aligned(q_norm, 16)) && skinny_aligned(workspace, 16),
                   "attention prompt: qkv, caches, table, q_norm and workspace must be 16-byte aligned");
  const int nch = (keys + kChunk - 1) / kChunk, pieces = (M + kPiece - 1) / kPiece;
  const size_t piece = prompt_piece_bytes(Hkv, nch), qbytes = prompt_query_bytes(M, Hq);
  const size_t room = workspace_bytes > qbytes ? (workspace_bytes - qbytes) / piece : 0;
  const int fit = room < (size_t)pieces ? (int)room / kPieceGroup * kPieceGroup : pieces;
  SKINNY_CHECK_ARG(fit >= 1, "attention prompt: workspace of %zu bytes, needs %zu", workspace_bytes,
                   skinny_attn_prompt_workspace_bytes(M, Hq, Hkv, keys));
  uint16_t* q = static_cast<uint16_t*>(workspace);
  float* part_o = reinterpret_cast<float*>(static_cast<char*>(workspace) + qbytes);
  float* part_ml = part_o + (size_t)fit * Hkv * nch * kRowsMax * kD;
  const hipStream_t s = (hipStream_t)stream;
  const PromptArgs pa{M, Hq, Hkv, q_norm, k_norm, eps, rope_table, q, k_cache, vt_cache, maxlen};
  const int nq = (M * Hq + 63) / 64, nk = (M * Hkv + 3) / 4, nv = Hkv * ((M + 63) / 64);
  hipLaunchKernelGGL(prompt_qkv_kernel, dim3(nq + nk + nv), dim3(256), 0, s, pos0, qkv, ldq, nq, nk, pa);
  if (int rc = skinny_check_launch("attention prompt q/k/v")) return rc;
  for (int z0 = 0; z0 < pieces; z0 += fit) {
    const int z1 = z0 + fit < pieces ? z0 + fit : pieces;
    const int last = z1 * kPiece < M ? z1 * kPiece : M;             // tokens up to this launch's end
    const int n = (keys - M + last + kChunk - 1) / kChunk;          // chunks its last piece sees
    hipLaunchKernelGGL(prompt_chunk_kernel, dim3(n, Hkv, (z1 - z0 + kPieceGroup - 1) / kPieceGroup), dim3(64 * kWaves), 0, s,
                       pos0, q, M, Hq, Hkv, k_cache, vt_cache, maxlen, scale, z0, z1, nch, part_o, part_ml);
    if (int rc = skinny_check_launch("attention prompt chunks")) return rc;
    // the wave count of the merge goes by the cache size, as in the step kernels
    const int W = maxlen / kChunk > kCombineLong ? kCombineWavesLong : maxlen / kChunk > kCombineBlock ? kCombineWaves : 1;
    const auto merge = W == kCombineWavesLong ? prompt_combine_kernel<kCombineWavesLong>
                       : W == kCombineWaves   ? prompt_combine_kernel<kCombineWaves>
                                              : prompt_combine_kernel<1>;
    hipLaunchKernelGGL(merge, dim3(Hq, last - z0 * kPiece), dim3(64 * W), 0, s, part_o, part_ml, M, Hq, Hkv, pos0, z0, nch,
                       out);
    if (int rc = skinny_check_launch("attention prompt merge")) return rc;
  }
  return SKINNY_OK;
}

// --- the allocation-free form -----------------------------------------------------------------

// The chunk partials of skinny_attention_fused_noalloc_bf16: a file-scope device array (one copy
// per GPU, held until the process ends) instead of a caller workspace, sized for at most
// kScratchChunks (kv head, 128-key chunk) pairs — 8 kv heads over 4096 cached positions, 8.1 MiB.
// No entry needs it cleared: the chunk kernel writes every partial the combine kernel reads.
constexpr int kScratchChunks = 256;
constexpr size_t kScratchFloats = (size_t)kScratchChunks * kRowsMax * (kD + 2);
static __device__ __align__(256) float scratch[kScratchFloats];

constexpr int kMaxDevices = 64;
static std::mutex g_scratch_mu;
static float* g_scratch_ptr[kMaxDevices] = {};

// Device address of `scratch` on the current device, looked up once per device: in host code the
// array's name is only a stand-in, and every GPU holds its copy at its own address.
static int scratch_of_current_device(void* stream, float** out) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return skinny_set_error(SKINNY_ELAUNCH, "attention (no alloc): hipGetDevice: %s", hipGetErrorString(e));
  if (stream) {
    hipDevice_t sdev = 0;
    e = hipStreamGetDevice((hipStream_t)stream, &sdev);
    if (e != hipSuccess)
      return skinny_set_error(SKINNY_ELAUNCH, "attention (no alloc): hipStreamGetDevice: %s", hipGetErrorString(e));
    SKINNY_CHECK_ARG((int)sdev == dev, "attention (no alloc): the stream is on device %d, the current device is %d",
                     (int)sdev, dev);
  }
  SKINNY_CHECK_ARG(dev >= 0 && dev < kMaxDevices, "attention (no alloc): device %d beyond %d", dev, kMaxDevices);
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p)
      return skinny_set_error(SKINNY_ELAUNCH, "attention (no alloc): hipGetSymbolAddress(scratch) on device %d: %s", dev,
                              hipGetErrorString(e));
    g_scratch_ptr[dev] = static_cast<float*>(p);
  }
  *out = g_scratch_ptr[dev];
  return SKINNY_OK;
}

extern "C" int skinny_attention_fused_noalloc_bf16(const uint16_t* qkv, int ldq, int M, int Hq, int Hkv, int D,
                                                   const uint16_t* q_norm, const uint16_t* k_norm, float eps,
                                                   const float* rope_table, int rope_positions, const int32_t* pos0,
                                                   const int32_t* tree, uint16_t* k_cache, uint16_t* vt_cache,
                                                   int maxlen, float scale, uint16_t* out, void* stream) {
  SKINNY_CHECK_ARG(Hkv >= 1 && maxlen >= kChunk && maxlen % kChunk == 0,
                   "attention (no alloc): Hkv=%d, maxlen=%d must be a multiple of %d", Hkv, maxlen, kChunk);
  SKINNY_CHECK_ARG((size_t)Hkv * (maxlen / kChunk) <= (size_t)kScratchChunks,
                   "attention (no alloc): %d kv heads x %d cached positions exceed the scratch maximum of %d "
                   "(kv head, %d-position chunk) pairs",
                   Hkv, maxlen, kScratchChunks, kChunk);
  float* ws = nullptr;
  if (int rc = scratch_of_current_device(stream, &ws)) return rc;
  return attention_fused(qkv, ldq, M, Hq, Hkv, D, q_norm, k_norm, eps, rope_table, rope_positions, pos0, tree,
                         k_cache, vt_cache, maxlen, scale, ws, kScratchFloats * sizeof(float), out, stream);
}
