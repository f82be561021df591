// W4A16 affine group-64 matmul for many rows (prompts): weights read once per block of rows, with the
// bits of the 1..16-token kernels of qmm.hip.
//
// Reference behaviour: skinny_mlx/qmm.py:132-152 runs its kernel for up to 16 rows and hands more to
// mx.quantized_matmul; here more rows once ran as 16-row pieces, each reading every weight again.
//
// A piece's bits follow from its cut of K and from the order in which the cut's sums are added: S splits
// of G groups of consecutive 128-wide pairs, each group accumulated from zero in pair order
// (acc += s g; acc += (b - 128 s) x, per 64-wide scale group, g and x from the same two MFMAs), the group
// sums added in group order from zero, the split sums in split order. This kernel walks the same cut in
// one wave, so each row's output is bitwise that of the piece it would have been part of.
//
// Layout. A workgroup of 4 waves holds 16 MT rows x 64 NT weight rows: the waves share the X block (staged
// in LDS in MFMA fragment order, two buffers of one 128-wide pair) and own 16 NT weight rows each, whose
// packed blocks go straight to registers, so a weight crosses the memory path once per 16 MT rows. What
// bounds it is the issue of one SIMD's waves: per 16x16 tile and scale group two MFMAs (32 cycles) stand
// against 8 FMAs (32 cycles; the scale and bias terms in fp32, which the bits fix) and the nibble unpacking
// (17 instructions per 16 weight rows, shared by MT tiles), so everything else has to be hidden: X's LDS reads
// run half a pair ahead of their MFMAs, X's rows are loaded in whole 128-byte lines, and the loop's loads stand
// in the same order on every path, as a wait counts the loads issued after the one it is for. So VALU instructions issue in
// 86% of the CUs' busy cycles (2560x19456 gate|up, 501 rows: 77.4 us). All figures here and at pick_rows: one launch over
// weights that are in no cache (400 MB of them in turn). MT = 4 saves a fifth of the instructions but leaves two waves per
// SIMD (the same case 81.5 us with NT = 2; with NT = 4 it spills).
// MT = 3 serves grids that fit the CUs with blocks of 48 rows and not with 32 (pick_rows).
#include "qmm_frag.h"

namespace {

enum RowsEpi { kRowsPlain = 0, kRowsGluSplit = 1, kRowsSwiGlu = 2 };

// X of one pair for this wave's share of the 16 MT rows: MT loads of 16 bytes per lane. Staged, fragment
// 4 mt + 2 j + h of the pair holds rows 16 mt + tok and columns 64 j + 32 h + 8 quad ... for lane 16 quad + tok.
template <int MT>
struct XPart {
  u32x4_t v[MT];
};

template <int MT>
__device__ __forceinline__ void load_xpart(XPart<MT>& xp, __amdgpu_buffer_rsrc_t rx, const uint32_t (&xoff)[MT], int pair) {
#pragma unroll
  for (int i = 0; i < MT; ++i)
    xp.v[i] = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rx, xoff[i], pair * 256, 0));
}

template <int V>
struct IntTag {
  static constexpr int value = V;
};

// The cut of K walked by one wave of the kernel below.
struct RowsArgs {
  const uint16_t* x;
  int M, K, ldx;
  const uint32_t* w;
  int N, S, G;              // S splits of G groups
  int row_blocks, per_xcd;  // blocks of rows; workgroups per XCD
  uint16_t* y;
  int ldy, vec;             // vec: y's rows take 16-byte stores
};

// KS parts of 4 waves each share the workgroup's output tile: with KS = 1 one part walks all of K; with
// KS > 1 (a grid too small to fill the chip, or a deep K) part p walks split p (S = KS > 1) or the groups
// [p G / KS, (p + 1) G / KS) of the one split, and leaves its split's sum, or each of its groups' sums, in
// LDS; part 0 then adds them in the cut's order, so the bits do not depend on KS. NACC: sums a wave keeps
// apart (1 = one group in all, 2 = groups, 3 = groups and splits).
//
// The wide wave (NT = 4) and several parts keep one pair of weights per wave in flight, loaded again as soon
// as its second half is unpacked: half a pair of time, which the other waves of the SIMD fill; one part of
// NT = 2 has registers for two (9728x2560, 1024 rows: level with one, 94.7 us). The wide wave also keeps its group sums in
// LDS, each lane its own words: in registers they spill within the loop at three waves per SIMD (2560x19456,
// 501 rows: 83.5 against 77.4 us).
template <int MT, int NT, int NACC, int KS, int EPI>
__global__ __launch_bounds__(256 * KS, NT == 4 ? 3 : 1) void qmm_rows_kernel(const RowsArgs ra) {
  static_assert(EPI == kRowsPlain || NT % 2 == 0, "gate|up epilogues pair two row tiles per wave");
  static_assert(KS == 1 || NACC == 2, "several parts: the groups of one split each");
  static_assert(NT < 4 || NACC < 3, "the wide wave's registers hold two sums at most");
  constexpr bool kGrpLds = NT == 4 && NACC == 2;     // the group sums live in LDS
  constexpr bool kGrp = NACC >= 2 && !kGrpLds;
  constexpr int kStages = NT == 4 || KS > 1 ? 1 : 2;  // pairs of weights in flight
  constexpr int kXWords = MT * 4 * 64;  // 16-byte words of one staged pair
  constexpr int kOutCols = EPI == kRowsSwiGlu ? 8 * NT : 16 * NT;
  constexpr int kOutPitch = kOutCols + 8;
  static_assert(2 * kXWords * 16 * KS >= 4 * 16 * kOutPitch * 2, "the output rows fit the staging buffers");
  extern __shared__ __attribute__((aligned(16))) char lds[];  // [KS][2] staged pairs, then the parts' sums
  const int M = ra.M, K = ra.K, ldx = ra.ldx, N = ra.N, S = ra.S, G = ra.G;
  const int GP = K >> 7, T = N >> 4;
  const int lane = threadIdx.x & 63, wv = wave_id();
  const int wave = wv & 3, part = KS > 1 ? wv >> 2 : 0;
  const int tok = lane & 15, quad = lane >> 4;
  // Workgroup i runs on XCD i % 8: each XCD takes a contiguous run of (weight block, row block) pairs,
  // row blocks fastest, so the workgroups in flight on one L2 share their weights.
  const int id = ((int)blockIdx.x & 7) * ra.per_xcd + ((int)blockIdx.x >> 3);
  const int nblk = id / ra.row_blocks, rblk = id % ra.row_blocks;
  const int tile0 = (nblk * 4 + wave) * NT;
  if (nblk * 4 * NT >= T) return;  // the grid's padding: the whole workgroup
  const int row0 = rblk * 16 * MT;
  const int rows = min(16 * MT, M - row0);
  // (min and max of scalars may become a vector med3; a descriptor word in a vector register would wrap
  // every load in a waterfall loop)
  const int mytiles = __builtin_amdgcn_readfirstlane(max(0, min(NT, T - tile0)));
  const __amdgpu_buffer_rsrc_t rx = make_rsrc(ra.x + (size_t)row0 * ldx, ((uint32_t)(rows - 1) * ldx + K) * 2u);
  const __amdgpu_buffer_rsrc_t rw = make_rsrc(
      reinterpret_cast<const char*>(ra.w) + (size_t)min(tile0, T - 1) * GP * kBlockBytes, (uint32_t)(mytiles * GP * kBlockBytes));
  const uint32_t woff = (uint32_t)lane * 16u;
  const uint32_t sboff = kSbOffsetBytes + (uint32_t)tok * 8u;
  const bf16x8_t ones = ones_operand();
  u32x4_t* const xl = reinterpret_cast<u32x4_t*>(lds) + part * 2 * kXWords;
  float* const sums = reinterpret_cast<float*>(lds + (size_t)KS * 2 * kXWords * 16);
  // A load takes 8 rows of a scale group's 64 columns, 128 bytes each: half the rows of two fragments (load f: row tile
  // f / 4, group f / 2 % 2). This wave does loads wave MT .. + MT - 1. Rows past M carry an out-of-range offset and
  // read as zeros.
  // Lane group g = lane / 8 takes rows 4 (g % 4) + g / 4 and two below, and a fragment's quad holds its rows in
  // the order t ^ quad ^ 12 h: so both the 16 lanes of a read and any 16 of a write fall on different banks.
  auto slot_of = [](int t, int qd, int h) { return qd * 16 + (t ^ qd ^ (12 * h)); };
  const int srow = ((lane >> 3) & 3) * 4 + (lane >> 5);
  uint32_t xoff[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    const int f = wave * MT + i, r = (f >> 2) * 16 + (f & 1) * 2 + srow;
    xoff[i] = r < rows ? (uint32_t)(r * ldx + (f & 2) * 32 + (lane & 7) * 8) * 2u : 0x7ffffff0u;
  }

  f32x4_t acc[MT][NT], grp[kGrp ? MT : 1][kGrp ? NT : 1], spl[NACC >= 3 ? MT : 1][NACC >= 3 ? NT : 1];
  const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int n = 0; n < NT; ++n) {
      acc[m][n] = zero;
      if constexpr (kGrp) grp[m][n] = zero;
      if constexpr (NACC >= 3) spl[m][n] = zero;
    }

  // The cut: split sp holds pairs [pb, pe), its group g ends before pair gend. Part p > 0 of a single split
  // keeps its groups apart in the slots of `sums`, slot s of wave w at (4 s + w) MT NT 256.
  int sp = KS > 1 && S > 1 ? part : 0;
  int pb = sp * GP / S, pe = (sp + 1) * GP / S;
  int g = 0, first = 0, stop = GP;  // this part's pairs [first, stop)
  if constexpr (KS > 1) {
    if (S > 1) {
      first = pb;
      stop = pe;
    } else {
      g = part * G / KS;
      first = g * GP / G;
      stop = ((part + 1) * G / KS) * GP / G;
    }
  }
  int gend = pb + (g + 1) * (pe - pb) / G;
  int slot = KS > 1 ? (S > 1 ? part - 1 : g - G / KS) : 0;
  auto dump = [&](f32x4_t (&v)[MT][NT]) {
    float* d = sums + (size_t)(4 * slot + wave) * MT * NT * 256 + lane;
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int i = 0; i < 4; ++i) d[((m * NT + n) * 4 + i) * 64] = v[m][n][i];
    ++slot;
  };
  auto close = [&](int p) {  // after pair p
    if constexpr (NACC >= 2) {
      if (p + 1 != gend) return;
      if constexpr (kGrpLds) {  // this lane's own words; the last group's sum stays in acc
        f32x4_t* d = reinterpret_cast<f32x4_t*>(sums) + wave * MT * NT * 64 + lane;
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
          for (int n = 0; n < NT; ++n) {
            const f32x4_t v = (g > 0 ? d[(m * NT + n) * 64] : zero) + acc[m][n];
            if (g + 1 < G) d[(m * NT + n) * 64] = v;
            acc[m][n] = g + 1 < G ? zero : v;
          }
        ++g;
        gend = (g + 1) * GP / G;
        return;
      }
      if (KS > 1 && S == 1 && part > 0) {
        dump(acc);
      } else if constexpr (kGrp) {
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
          for (int n = 0; n < NT; ++n) grp[m][n] += acc[m][n];
      }
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int n = 0; n < NT; ++n) acc[m][n] = zero;
      ++g;
      if constexpr (NACC >= 3) {
        if (g == G && sp + 1 < S) {
#pragma unroll
          for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int n = 0; n < NT; ++n) {
              spl[m][n] = sp == 0 ? grp[m][n] : spl[m][n] + grp[m][n];
              grp[m][n] = zero;
            }
          ++sp;
          g = 0;
          pb = pe;
          pe = (sp + 1) * GP / S;
        }
      }
      gend = pb + (g + 1) * (pe - pb) / G;
    }
  };

  using XOps = bf16x8_t[MT][2];  // X's operands of one scale group
  auto fetch = [&](XOps& o, int buf, int j) {
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int h = 0; h < 2; ++h)
        o[m][h] = __builtin_bit_cast(bf16x8_t, xl[buf * kXWords + (m * 4 + j * 2 + h) * 64 + slot_of(tok, quad, h)]);
  };
  auto load_w1 = [&](WStage<NT>& ws, int n, int p) {
    const int blk = (n * GP + p) * kBlockBytes;
    ws.w[n] = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rw, woff, blk, 0));
    ws.sb[n] = __builtin_bit_cast(u32x2_t, __builtin_amdgcn_raw_buffer_load_b64(rw, sboff, blk, 0));
  };
  // Scale group j of a pair; with one stage the second group's tiles make way for those of pair `next`.
  auto compute = [&](const XOps& xa, WStage<NT>& ws, int j, int next) {
    f32x4_t xsum[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) xsum[m] = mfma16x16x32(xa[m][0], ones, zero);
#pragma unroll
    for (int m = 0; m < MT; ++m) xsum[m] = mfma16x16x32(xa[m][1], ones, xsum[m]);
#pragma unroll
    for (int n = 0; n < NT; ++n) {
      const bf16x8_t b0 = unpack_nibbles(j ? ws.w[n].z : ws.w[n].x), b1 = unpack_nibbles(j ? ws.w[n].w : ws.w[n].y);
      const float s = __uint_as_float(j ? (ws.sb[n].x & 0xffff0000u) : (ws.sb[n].x << 16));
      const float b = __uint_as_float(j ? (ws.sb[n].y & 0xffff0000u) : (ws.sb[n].y << 16));
      const float bp = fmaf(-128.0f, s, b);
      if (kStages == 1 && j == 1) load_w1(ws, n, next);
      f32x4_t gm[MT];
#pragma unroll
      for (int m = 0; m < MT; ++m) gm[m] = mfma16x16x32(xa[m][0], b0, zero);
#pragma unroll
      for (int m = 0; m < MT; ++m) gm[m] = mfma16x16x32(xa[m][1], b1, gm[m]);
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          acc[m][n][i] = fmaf(s, gm[m][i], acc[m][n][i]);
          acc[m][n][i] = fmaf(bp, xsum[m][i], acc[m][n][i]);
        }
    }
  };

  // Pair q of the part (counted from `first`): its X is in LDS buffer q % 2, stored while pair q - 1's first
  // group runs, from registers loaded a pair before. One barrier per pair, between its groups: then pair q + 1
  // is staged and this pair's operands are read, and each group's operands are fetched while the other group
  // runs. Every part runs the longest part's count of rounds.
  int rounds = stop - first;
  if constexpr (KS > 1) {
#pragma unroll
    for (int p = 0; p < KS; ++p) {
      const int n = S > 1 ? (p + 1) * GP / S - p * GP / S : ((p + 1) * G / KS) * GP / G - (p * G / KS) * GP / G;
      rounds = max(rounds, n);
    }
  }
  WStage<NT> ws[kStages];
  XPart<MT> xp;
  const int last = stop - 1;
  auto store_x = [&](int buf) {
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      const int f = wave * MT + i, h = (lane >> 2) & 1;
      xl[buf * kXWords + ((f & ~1) + h) * 64 + slot_of((f & 1) * 2 + srow, lane & 3, h)] = xp.v[i];
    }
  };
  XOps xo[2];
  // u: the parity of q. The loads stand in this order on every path into and round the loop (see above): no
  // branch skips them (past the end they repeat the last pair), and the scheduler keeps the prologue's order.
  auto step = [&](auto uc, int q) {
    constexpr int u = decltype(uc)::value;
    const bool mine = KS == 1 || q <= last;
    if (mine) {
      fetch(xo[1], u, 1);
      __builtin_amdgcn_sched_barrier(0);
      store_x(u ^ 1);
      load_xpart<MT>(xp, rx, xoff, min(q + 2, last));
      compute(xo[0], ws[u & (kStages - 1)], 0, 0);
    }
    lds_barrier();
    if (mine) {
      fetch(xo[0], u ^ 1, 0);
      __builtin_amdgcn_sched_barrier(0);
      compute(xo[1], ws[u & (kStages - 1)], 1, min(q + 1, last));
      if constexpr (kStages == 2) load_w<NT>(ws[u], rw, woff, sboff, min(q + 2, last), GP);
      close(q);
    }
  };
  load_xpart<MT>(xp, rx, xoff, first);
  __builtin_amdgcn_sched_barrier(0);
  load_w<NT>(ws[0], rw, woff, sboff, first, GP);
  __builtin_amdgcn_sched_barrier(0);
  store_x(0);
  load_xpart<MT>(xp, rx, xoff, min(first + 1, last));
  __builtin_amdgcn_sched_barrier(0);
  if constexpr (kStages == 2) load_w<NT>(ws[1], rw, woff, sboff, min(first + 1, last), GP);
  __builtin_amdgcn_sched_barrier(0);
  lds_barrier();
  fetch(xo[0], 0, 0);
  int q = first;
  for (const int even = first + (rounds & ~1); q < even; q += 2) {
    step(IntTag<0>{}, q);
    step(IntTag<1>{}, q + 1);
  }
  if (rounds & 1) step(IntTag<0>{}, q);
  if constexpr (KS > 1) {
    if (S > 1 && part > 0) dump(grp);
    __syncthreads();
    if (part == 0) {  // the other parts' sums in the cut's order
      const int slots = S > 1 ? S - 1 : G - G / KS;
      for (int s = 0; s < slots; ++s) {
        const float* d = sums + (size_t)(4 * s + wave) * MT * NT * 256 + lane;
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
          for (int n = 0; n < NT; ++n)
#pragma unroll
            for (int i = 0; i < 4; ++i) grp[m][n][i] += d[((m * NT + n) * 4 + i) * 64];
      }
    }
  }

  // Output through LDS (the staging buffers), 16 rows of every wave of part 0 at a time: lane (col, quad)
  // holds rows 4 quad + i of weight row col of each tile; the stores then run along rows in 16-byte pieces.
  uint16_t* const ol = reinterpret_cast<uint16_t*>(lds) + wave * 16 * kOutPitch;
  __syncthreads();
  if (part > 0) return;
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    if (m * 16 >= rows) break;
    auto val = [&](int n, int i) {
      if constexpr (NACC == 1 || kGrpLds) return acc[m][n][i];
      if constexpr (NACC == 2 && kGrp) return grp[m][n][i];
      if constexpr (NACC == 3) return spl[m][n][i] + grp[m][n][i];
    };
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      uint16_t* o = ol + (quad * 4 + i) * kOutPitch + tok;
      if constexpr (EPI == kRowsSwiGlu) {
#pragma unroll
        for (int n = 0; n < NT; n += 2)
          o[n * 8] = silu_mul_bf16(bf16_bits_to_f32(f32_to_bf16_bits(val(n, i))),
                                   bf16_bits_to_f32(f32_to_bf16_bits(val(n + 1, i))));
      } else {
#pragma unroll
        for (int n = 0; n < NT; ++n) o[n * 16] = f32_to_bf16_bits(val(n, i));
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // each wave reads back only its own rows
    constexpr int kPieces = kOutCols / 8;               // 16-byte pieces per row of this wave
    for (int e = lane; e < 16 * kPieces; e += 64) {
      const int r = e / kPieces, c = (e % kPieces) * 8;
      const int row = m * 16 + r;
      const int til = EPI == kRowsSwiGlu ? (c >> 4) * 2 : c >> 4;  // the tile (pair) this piece lies in
      if (row >= rows || til >= mytiles) continue;
      size_t col;
      if constexpr (EPI == kRowsSwiGlu) col = (size_t)(tile0 >> 1) * 16 + c;
      else if constexpr (EPI == kRowsGluSplit) col = (size_t)(til & 1) * (N >> 1) + (size_t)((tile0 + til) >> 1) * 16 + (c & 15);
      else col = (size_t)tile0 * 16 + c;
      const u32x4_t v = *reinterpret_cast<const u32x4_t*>(ol + r * kOutPitch + c);
      uint16_t* dst = ra.y + (size_t)(row0 + row) * ra.ldy + col;
      if (ra.vec) {
        *reinterpret_cast<u32x4_t*>(dst) = v;
      } else {
#pragma unroll
        for (int k = 0; k < 8; ++k) dst[k] = (uint16_t)(v[k >> 1] >> (16 * (k & 1)));
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the rows are read before the next 16 replace them
  }
}

using RowsKernel = void (*)(const RowsArgs);

struct RowsForm {
  RowsKernel kern;
  int mt, nt, ks;  // row tiles, weight tiles per wave, parts of a workgroup
};

constexpr size_t kRowsMaxLds = 160 * 1024;
constexpr int kCus = 256;

// LDS slots of the parts' sums, or of the wide wave's group sums (16 MT rows x 64 NT weight rows of fp32 each).
int rows_slots(int S, int G, const RowsForm& f) {
  if (f.ks == 1) return f.nt == 4 && G > 1 ? 1 : 0;
  return S > 1 ? S - 1 : G - G / f.ks;
}

size_t rows_lds(const RowsForm& f, int S, int G) {
  return (size_t)f.ks * 2 * f.mt * 4096 + (size_t)rows_slots(S, G, f) * 4 * f.mt * f.nt * 1024;
}

int rows_blocks(int M, int N, int mt, int nt) { return ((M + 16 * mt - 1) / (16 * mt)) * ((N / 16 + 4 * nt - 1) / (4 * nt)); }

template <int NT, int EPI>
RowsForm rows_one_part(int S, int G) {
  if constexpr (NT < 4)
    if (S > 1) return {qmm_rows_kernel<2, NT, 3, 1, EPI>, 2, NT, 1};
  return {G > 1 ? qmm_rows_kernel<2, NT, 2, 1, EPI> : qmm_rows_kernel<2, NT, 1, 1, EPI>, 2, NT, 1};
}

template <int NT, int EPI>
RowsForm rows_parts(int S, int G) {
  if (S == 3) return {qmm_rows_kernel<2, NT, 2, 3, EPI>, 2, NT, 3};
  if (S == 1 && G >= 4) return {qmm_rows_kernel<2, NT, 2, 4, EPI>, 2, NT, 4};
  return {};
}

// As rows_parts with 48 rows a block; one split's groups in two parts, whose eight waves have the registers of two
// per SIMD.
template <int EPI>
RowsForm rows_parts48(int S, int G) {
  if (S == 3) return {qmm_rows_kernel<3, 2, 2, 3, EPI>, 3, 2, 3};
  if (S == 1 && G >= 2) return {qmm_rows_kernel<3, 2, 2, 2, EPI>, 3, 2, 2};
  return {};
}

// Which form. A grid of at most one workgroup per CU leaves its 4 waves alone on their CUs, where a pair
// takes about 0.7 us however few rows there are, so K is cut over the parts of a workgroup (3 for a cut of
// 3 splits, else 4), with the narrowest block whose grid still fits the CUs: 16 NT = 16 and 32, then 48 rows of 32
// (a second workgroup on some CUs would double the time). Larger grids take one part; the
// busiest CU holds ceil(blocks / CUs) of them, and a wide block (64 weight rows a wave instead of 32) costs
// 1.72 times a narrow one: it amortises its X reads over twice the weights, and is taken where that count comes
// out lower (from two wide blocks per CU on: alone on its CU a wide block is slower than two narrow ones).
// Measured on MI355X in us (K x N, M: one part / parts, chosen width; see the top): 4096x2560, 64: 22.3 / 14.9 (16 NT =
// 16); 256: 22.2 / 18.1 (32); 509: 28.9 / 25.5 (48 rows). 9728x2560, 96: 50.1 / 31.1 (16); 300: 50.5 / 38.8 (32); 400: 63.4 /
// 44.0 (48 rows); 509: 63.8 / 45.9 (48 rows). 2048x2560, 509: 16.7 / 15.5 (48 rows). 2560x6144, 64: 15.2 / 11.5 (16); 77:
// 15.1 / 13.5 (32); 160: 15.2 / 13.7 (32). Wide block against narrow, one part: 2560x19456 gate|up, 96: 29.4 / 22.3; 256: 47.5 /
// 46.2; 320: 50.3 / 54.4; 501: 77.7 / 84.8; 1024: 152 / 174; 2560x8224, 509: 44.1 / 42.7; 2560x12352, 256: 34.6 / 36.4; 509:
// 61.3 / 58.3; 2560x151936, 20: 50.8 / 51.4; 64: 85.2 / 91.0. A wide block of these takes 1.66 to 1.83 times a narrow one.
template <int EPI>
RowsForm pick_rows(int M, int N, int S, int G) {
  if constexpr (EPI != kRowsGluSplit) {
    if constexpr (EPI == kRowsPlain) {
      const RowsForm f = rows_parts<1, EPI>(S, G);
      if (f.kern && rows_blocks(M, N, f.mt, f.nt) <= kCus && rows_lds(f, S, G) <= kRowsMaxLds) return f;
    }
    const RowsForm f = rows_parts<2, EPI>(S, G);
    if (f.kern && rows_blocks(M, N, f.mt, f.nt) <= kCus && rows_lds(f, S, G) <= kRowsMaxLds) return f;
    const RowsForm f48 = rows_parts48<EPI>(S, G);
    if (f48.kern && rows_blocks(M, N, f48.mt, f48.nt) <= kCus && rows_lds(f48, S, G) <= kRowsMaxLds) return f48;
    const int wide = (rows_blocks(M, N, 2, 4) + kCus - 1) / kCus, narrow = (rows_blocks(M, N, 2, 2) + kCus - 1) / kCus;
    if (S == 1 && wide > 1 && (long long)wide * 172 < (long long)narrow * 100) return rows_one_part<4, EPI>(S, G);
  }
  return rows_one_part<2, EPI>(S, G);
}

}  // namespace

extern "C" int skinny_qmm_w4g64_rows_bf16(const uint16_t* x, int M, int K, int ldx, const uint32_t* w_frag, int N,
                                          uint16_t* y, int ldy, int splits, int groups, int epilogue, void* stream) {
  SKINNY_CHECK_ARG(x && w_frag && y, "qmm rows: null pointer");
  SKINNY_CHECK_ARG(M >= 1, "qmm rows: M=%d must be positive", M);
  SKINNY_CHECK_ARG(K > 0 && K % 128 == 0, "qmm rows: K=%d must be a positive multiple of 128", K);
  SKINNY_CHECK_ARG(epilogue >= kRowsPlain && epilogue <= kRowsSwiGlu, "qmm rows: unknown epilogue %d", epilogue);
  SKINNY_CHECK_ARG(N > 0 && N % (epilogue == kRowsPlain ? 16 : 32) == 0, "qmm rows: N=%d must be a positive multiple of %d", N,
                   epilogue == kRowsPlain ? 16 : 32);
  SKINNY_CHECK_ARG(ldx >= K && ldx % 8 == 0, "qmm rows: ldx=%d must be >= K and a multiple of 8", ldx);
  SKINNY_CHECK_ARG(ldy >= (epilogue == kRowsSwiGlu ? N / 2 : N), "qmm rows: ldy=%d too small", ldy);
  SKINNY_CHECK_ARG(splits >= 1 && groups >= 1 && (K / 128) / splits >= groups,
                   "qmm rows: %d splits of %d groups need a pair of 128 each (K=%d)", splits, groups, K);
  SKINNY_CHECK_ARG(skinny_aligned(x, 16) && skinny_aligned(w_frag, 16) && skinny_aligned(y, 2), "qmm rows: misaligned buffer");
  SKINNY_CHECK_ARG((size_t)48 * ldx * 2 < 0x7ff00000u && (size_t)4 * (K / 128) * kBlockBytes < 0x40000000u,
                   "qmm rows: rows too long for a buffer descriptor");
  // 32-row x 128-weight blocks of 256 threads: the grid stays below 2^32 threads
  SKINNY_CHECK_ARG(((size_t)M / 32 + 1) * ((size_t)N / 128 + 1) < (1u << 23), "qmm rows: M=%d x N=%d is too large for one launch",
                   M, N);
  const RowsForm f = epilogue == kRowsSwiGlu     ? pick_rows<kRowsSwiGlu>(M, N, splits, groups)
                     : epilogue == kRowsGluSplit ? pick_rows<kRowsGluSplit>(M, N, splits, groups)
                                                 : pick_rows<kRowsPlain>(M, N, splits, groups);
  const int row_blocks = (M + 16 * f.mt - 1) / (16 * f.mt);
  const size_t total = (size_t)row_blocks * ((N / 16 + 4 * f.nt - 1) / (4 * f.nt));
  const size_t lds = rows_lds(f, splits, groups);
  if (lds > 64 * 1024) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(f.kern),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return skinny_set_error(SKINNY_ELAUNCH, "qmm rows: %zu bytes of LDS: %s", lds, hipGetErrorString(e));
  }
  const int per_xcd = (int)((total + 7) / 8);
  const RowsArgs ra{x, M, K, ldx, w_frag, N, splits, groups, row_blocks, per_xcd, y, ldy,
                    ldy % 8 == 0 && skinny_aligned(y, 16) ? 1 : 0};
  hipLaunchKernelGGL(f.kern, dim3(8 * per_xcd), dim3(256 * f.ks), lds, (hipStream_t)stream, ra);
  return skinny_check_launch("qmm rows");
}
