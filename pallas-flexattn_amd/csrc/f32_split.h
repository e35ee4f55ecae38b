// float32 FlexAttention kernels for gfx950 on the bf16 matrix cores.
//
// A float32 value x is exactly x0 + x1 + x2 with x0 = bf16(x), x1 = bf16(x -
// x0), x2 = bf16(x - x0 - x1) (8 significant bits each, round to nearest:
// |x1| <= 2^-9 |x|, |x2| <= 2^-18 |x|).  A product of two such values is taken
// as the six partial products x_i y_j with i + j <= 2; the three left out are
// below 2^-26 of it, a quarter of a float32 rounding.  The six are exact in
// the matrix core and its float32 accumulation rounds once per 16 terms and
// partial product instead of once per 2 terms (v_mfma_f32_32x32x2f32), so the
// results are closer to float64 than the float32 matrix instructions':
// relative error of O, dQ, dK, dV at B4 H8 S1000 D64 causal 2.7 / 4.2 / 5.3 /
// 4.8e-7 against 3.3 / 5.0 / 6.4 / 5.7e-7 (the same order at D 32 and 128, S
// 393 to 4096).  Six v_mfma_f32_32x32x16_bf16 take 192 matrix-core cycles for a
// 32 x 32 x 16 block, the eight v_mfma_f32_32x32x2f32 they replace 512.
//
// Times (us; forward, dK/dV, dQ; float32 instructions -> this file):
//   B4 H8  S1000 D64  causal   150, 190, 163  ->   42,  90,  58
//   B4 H16 S4096 D64  causal  1287, 2982, 1770 -> 732, 1530, 982
//   B2 H16 S2048 D128 causal   474, 680, 460  ->  231,  428, 277
// Bound by the chain of a tile (products, exponentials, splitting, products):
// the large shape runs at 178 to 209 TFLOP/s, 1.07 to 1.25 PFLOP/s of bf16
// products, what the library's bf16 GEMM reaches on this board.
//
// What is split: Q, K, V, dO as they are staged (each element once per
// workgroup that stages it), P and dS in registers.  Everything else (softmax,
// sums, Delta, the accumulators) is float32 as before.
//
// Small values: bf16 has float32's exponents, so the low pieces of a value
// below 2^-110 would fall off the end of them (2^-133).  Operands are therefore
// scaled by 2^16 as they are split, which makes the pieces of every float32
// exact, subnormal ones too, and the sums are scaled back (exactly) by 2^-32
// where they are used: in the exponent's FMA, in dP - Delta, at the end.  Only
// the forward's Q and K stay as they are: what their scores lose is below 2^-84
// before the exponential.  Same results bit for bit at ordinary magnitudes;
// unscaled / scaled, one board (us; forward, dK/dV, dQ): 45.5, 94, 59 / 47, 95, 61
// at the first shape above, 711, 1497, 982 / 733, 1506, 987 at the second.
//
// Large values: partial products of infinities differ from the float32 product
// (inf times an exact zero piece), and sums of 2^32 times their value overflow
// before float32 ones do.  A work item that meets an element of Q or K of
// magnitude >= 2^43 (below that the scores stay finite), or whose O, dQ, dK or
// dV sums are not finite at the end (which V, dO and everything after the
// exponential shows up in), discards what it has and runs again on the float32
// matrix instructions (fwd_item, dq_item, dkdv_item: the general kernels' code,
// same results as a call without the split).
//
// One structure for all three kernels: NW waves, 32 rows (or keys) per wave
// with their split operands in registers, tiles of 32 rows of the two streamed
// tensors in LDS as three bf16 planes each, double-buffered.  A tile's rows are
// loaded into registers a tile ahead, split into the other buffer between the
// MFMAs of the current tile's first products (VALU work passes under them) and
// published by the one barrier per tile; the second half of P / dS is computed
// and split between the first half's products.  The planes are read both ways
// (rows; transposed with ds_read_b64_tr_b16), so no transposed copy is written.
// With NG = 2 groups of NW waves take alternate tiles of one work item and add
// up through LDS at its end (problem.h: f32_groups).
#pragma once
#include "bwd.h"

namespace fa {

struct Frag3 {  // eight consecutive k of a matrix operand, as three bf16 pieces
  u32x4 p[3];
};

constexpr float kSplitMax = 8796093022208.0f;  // 2^43
constexpr float kUp = 65536.0f;                // 2^16: the scale of every split operand
constexpr float kDown = 1.0f / kUp, kDown2 = kDown * kDown;

// Word j (elements 2 j, 2 j + 1) of the three pieces.  The packed words are
// opaque to the compiler, which would otherwise convert each low element a
// second time instead of shifting it out of the word.
__device__ __forceinline__ void split2(Frag3& f, int j, float a, float b) {
  uint32_t w0 = pack_bf16x2(a, b);
  asm("" : "+v"(w0));
  const float a1 = a - bf16_lo(w0), b1 = b - bf16_hi(w0);
  uint32_t w1 = pack_bf16x2(a1, b1);
  asm("" : "+v"(w1));
  f.p[0][j] = w0;
  f.p[1][j] = w1;
  f.p[2][j] = pack_bf16x2(a1 - bf16_lo(w1), b1 - bf16_hi(w1));
}
__device__ __forceinline__ Frag3 split8(const float* x) {
  Frag3 f;
#pragma unroll
  for (int j = 0; j < 4; ++j) split2(f, j, x[2 * j], x[2 * j + 1]);
  return f;
}

// the largest of m, |a| and |b| (a NaN is passed over: it stays NaN through
// the pieces); fmaxf would first canonicalise each operand
__device__ __forceinline__ float max_mag(float m, float a, float b) {
  asm("v_max3_f32 %0, %0, |%1|, |%2|" : "+v"(m) : "v"(a), "v"(b));
  return m;
}

__device__ __forceinline__ f32x16 mma1(u32x4 a, u32x4 b, f32x16 c) { return Elt<uint16_t>::mma(a, b, c); }

// c += A B over 16 k: the six partial products, small ones first
__device__ __forceinline__ f32x16 mma6(const Frag3& a, const Frag3& b, f32x16 c) {
  c = mma1(a.p[2], b.p[0], c);
  c = mma1(a.p[0], b.p[2], c);
  c = mma1(a.p[1], b.p[1], c);
  c = mma1(a.p[1], b.p[0], c);
  c = mma1(a.p[0], b.p[1], c);
  return mma1(a.p[0], b.p[0], c);
}

// N MFMAs with the VALU work of their scheduling region spread between them:
// an MFMA occupies the matrix core for 32 cycles and its wave's issue for a
// quarter of that, so V other instructions after each one pass under it.
template <int N, int V>
__device__ __forceinline__ void mix_mfma_valu() {
#pragma unroll
  for (int i = 0; i < N; ++i) {
    __builtin_amdgcn_sched_group_barrier(kSchedMfma, 1, 0);
    __builtin_amdgcn_sched_group_barrier(kSchedValu, V, 0);
  }
}

__device__ __forceinline__ void zero16(f32x16& x) {
#pragma unroll
  for (int e = 0; e < 16; ++e) x[e] = 0.f;
}

// A 32-row tile of a float32 (rows, D) tensor in LDS: three planes of 32 rows
// of D bf16, 16-byte chunk c of row r in slot c ^ chunk_swz(r) (the bf16
// kernels' layout: conflict-free for row reads and transposing reads).
template <int D, int NW>
struct SplitTile : RowTileOffsets<D> {
  using RowTileOffsets<D>::RB;
  using RowTileOffsets<D>::KCH;
  using RowTileOffsets<D>::aoff;
  using RowTileOffsets<D>::tr;
  static constexpr int kRows = 32;
  static constexpr int kPlane = kRows * RB;
  static constexpr int kBytes = 3 * kPlane;
  static constexpr int kChunks = kRows * KCH;  // 8-element chunks of a tile
  static constexpr int kPer = (kChunks + NW * 64 - 1) / (NW * 64);  // chunks per thread
  static constexpr bool kAll = kChunks % (NW * 64) == 0;

  // row fragment: rows perm23(lane % 32), k = 16 s + 8 (lane / 32) + [0..7]
  __device__ __forceinline__ Frag3 rows(const char* t, int s) const {
    Frag3 f;
#pragma unroll
    for (int i = 0; i < 3; ++i) f.p[i] = *reinterpret_cast<const u32x4*>(t + i * kPlane + aoff[s]);
    return f;
  }
  // transposed fragment: row d = 32 dt + lane % 32, k = tile rows 16 c + 8 (lane / 32) + [0..7]
  __device__ __forceinline__ Frag3 cols(const char* t, int dt, int c) const {
    Frag3 f;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const uint2 lo = lds_read_tr16(t + i * kPlane + 16 * c * RB + tr[0][dt]);
      const uint2 hi = lds_read_tr16(t + i * kPlane + 16 * c * RB + tr[1][dt]);
      f.p[i] = u32x4{lo.x, lo.y, hi.x, hi.y};
    }
    return f;
  }
};

// acc += A(tile ta) * ba (and acc2 += A(tile tb) * bb) over all k steps, the
// row fragments one (AH) step ahead, the MFMAs of the two chains alternating;
// work(s) is VALU and LDS-write work issued between step s's MFMAs.
template <int D, int NW, class Work>
__device__ __forceinline__ void mma6_rows(const SplitTile<D, NW>& t, const char* ta, const Frag3* ba, f32x16& acc,
                                          const Work& work) {
  constexpr int KS = D / 16;
  Frag3 fa[2];
  fa[0] = t.rows(ta, 0);
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    if (s + 1 < KS) fa[(s + 1) & 1] = t.rows(ta, s + 1);
    __builtin_amdgcn_sched_barrier(0);
    acc = mma6(fa[s & 1], ba[s], acc);
    work(s);
    mix_mfma_valu<6, 8>();
    __builtin_amdgcn_sched_barrier(0);
  }
}
template <int D, int NW, int AH = 1, class Work>
__device__ __forceinline__ void mma6_rows2(const SplitTile<D, NW>& t, const char* ta, const char* tb, const Frag3* ba,
                                           const Frag3* bb, f32x16& acc, f32x16& acc2, const Work& work) {
  constexpr int KS = D / 16;
  constexpr int ia[6] = {2, 0, 1, 1, 0, 0}, ib[6] = {0, 2, 1, 0, 1, 0};  // small products first
  Frag3 fa[AH + 1], fb[AH + 1];
#pragma unroll
  for (int s = 0; s < KS + AH; ++s) {
    if (s < KS) {
      fa[s % (AH + 1)] = t.rows(ta, s);
      fb[s % (AH + 1)] = t.rows(tb, s);
    }
    __builtin_amdgcn_sched_barrier(0);
    if (s >= AH) {
      const int r = s - AH;
#pragma unroll
      for (int x = 0; x < 6; ++x) {
        acc = mma1(fa[r % (AH + 1)].p[ia[x]], ba[r].p[ib[x]], acc);
        acc2 = mma1(fb[r % (AH + 1)].p[ia[x]], bb[r].p[ib[x]], acc2);
      }
      work(r);
      mix_mfma_valu<12, 4>();
      __builtin_amdgcn_sched_barrier(0);
    }
  }
}

// One streamed tensor of a tile on its way to LDS: kPer chunks of eight
// floats per thread (chunk g of the tile is bytes [32 g, 32 g + 32) of its
// rows, which are contiguous in memory).
template <int D, int NW>
struct SplitStage {
  using Tile = SplitTile<D, NW>;
  u32x4 v[Tile::kPer][2];
  // rows [row0, row0 + 32) of a tensor of `rows` rows at base; rows past the
  // end (and row0 >= rows) read as zero
  __device__ __forceinline__ void load(const float* base, int row0, int rows, int tid) {
    const int r0 = row0 < rows ? row0 : rows;
    const int n = rows - r0 < Tile::kRows ? rows - r0 : Tile::kRows;
    const i32x4 rs = make_rsrc(base + (size_t)r0 * D, (uint32_t)n * D * 4);
#pragma unroll
    for (int u = 0; u < Tile::kPer; ++u) {
      const int off = (tid + u * NW * 64) * 32;
      v[u][0] = buf_load16(rs, off);
      v[u][1] = buf_load16(rs, off + 16);
    }
  }
  // half h (four floats) of chunk u split into its three planes; kMag: returns
  // the largest magnitude seen (else mag)
  template <bool kScaled, bool kMag>
  __device__ __forceinline__ float store(char* tile, int u, int h, int tid, float mag) const {
    const int g = tid + u * NW * 64;
    // (keeps the compiler from splitting the chunk, and so waiting for its
    // load, ahead of the products it is issued between)
    u32x4 raw = v[u][h];
    asm volatile("" : "+v"(raw));
    float x[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const uint32_t word = raw[t];
      x[t] = __uint_as_float(word);
    }
    Frag3 f;
    const float up = kScaled ? kUp : 1.0f;
    split2(f, 0, x[0] * up, x[1] * up);
    split2(f, 1, x[2] * up, x[3] * up);
    if (Tile::kAll || g < Tile::kChunks) {
      const int row = g / Tile::KCH, c = g % Tile::KCH;
      char* p = tile + row * Tile::RB + ((c ^ chunk_swz<Tile::KCH>(row)) * 16) + 8 * h;
#pragma unroll
      for (int i = 0; i < 3; ++i) *reinterpret_cast<u32x2*>(p + i * Tile::kPlane) = u32x2{f.p[i][0], f.p[i][1]};
    }
    return kMag ? max_mag(max_mag(mag, x[0], x[1]), x[2], x[3]) : mag;
  }
};

// The halves of both streamed tensors that a tile's k step s splits (all of
// them over the KS steps); x is the score's factor, whose magnitudes count, and
// is scaled with kScaledX.
template <int D, int NW, bool kScaledX = true>
__device__ __forceinline__ float stage_step(const SplitStage<D, NW>& x, const SplitStage<D, NW>& y, char* xt, char* yt,
                                            int s, int tid, float mag) {
  constexpr int PER = SplitTile<D, NW>::kPer, N = 4 * PER, KS = D / 16;
  static_assert(N % KS == 0 || KS % N == 0, "halves over steps");
#pragma unroll
  for (int u = s * N / KS; u < (s + 1) * N / KS; ++u) {
    if (u < 2 * PER) mag = x.template store<kScaledX, true>(xt, u >> 1, u & 1, tid, mag);
    else mag = y.template store<true, false>(yt, (u - 2 * PER) >> 1, u & 1, tid, mag);
  }
  return mag;
}

// A row operand kept in registers: row `row` of a (rows, D) tensor at base;
// returns the largest magnitude seen.
template <int D, bool kScaled = true>
__device__ __forceinline__ float load_rows3(Frag3* f, const float* base, int row, bool ok, int hh, float mag) {
#pragma unroll
  for (int s = 0; s < D / 16; ++s) {
    const f32x8 v = ld_frag<float>(base + (size_t)row * D + 16 * s + 8 * hh, ok);
    float x[8];
#pragma unroll
    for (int t = 0; t < 8; ++t) x[t] = v[t] * (kScaled ? kUp : 1.0f);
    f[s] = split8(x);
#pragma unroll
    for (int t = 0; t < 8; t += 2) mag = max_mag(mag, v[t], v[t + 1]);
  }
  return mag;
}

// Whether any lane of the workgroup met a score factor that the split does not
// take, or sums that are not finite (`probe`: their products with 0, added up);
// `flag` is a word of LDS.  Ends with a barrier.
__device__ __forceinline__ bool any_large(float mag, float probe, uint32_t* flag) {
  __syncthreads();
  if (threadIdx.x == 0) *flag = 0u;
  __syncthreads();
  if (mag >= kSplitMax || !(probe == 0.f)) *flag = 1u;
  __syncthreads();
  return *flag != 0u;
}

// 0 where every accumulator is finite, else NaN.
template <int N>
__device__ __forceinline__ float finite_probe(const f32x16* acc, float z) {
#pragma unroll
  for (int i = 0; i < N; ++i)
#pragma unroll
    for (int e = 0; e < 16; ++e) z = fmaf(acc[i][e], 0.f, z);
  return z;
}

// A gradient's last factors (2^-32 and the softmax scale), the smaller first:
// the product neither overflows before it is due nor rounds twice unless it is
// subnormal.
struct GradScale {
  float a, b;
  __device__ __forceinline__ explicit GradScale(float scale)
      : a(scale > 1.0f ? kDown2 : scale), b(scale > 1.0f ? scale : kDown2) {}
  __device__ __forceinline__ float operator()(float x) const { return x * a * b; }
};

// A group's accumulators in LDS, one column per thread: x = base + thread.
template <int N, int NW>
__device__ __forceinline__ void put_acc(float* x, const f32x16* acc) {
#pragma unroll
  for (int i = 0; i < N; ++i)
#pragma unroll
    for (int e = 0; e < 16; ++e) x[(i * 16 + e) * NW * 64] = acc[i][e];
}
template <int N, int NW>
__device__ __forceinline__ void add_acc(const float* x, f32x16* acc) {
#pragma unroll
  for (int i = 0; i < N; ++i)
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[i][e] += x[(i * 16 + e) * NW * 64];
}

// Element mask of the generic kernels with the interval form where the masks
// are intervals (no document reads per element).
struct ElemMask {
  bool interval;
  int lo, hi;  // visible positions of this lane's row (interval masks)
  int doc;     // its document label (others)
};

// ------------------------------------------------------------- forward ----
// LDS: K 0, K 1, V 0, V 1 (12 KiB each at D = 64), a flag word.
template <int D>
constexpr int f32_lds_bytes() {
  return 4 * 3 * 32 * D * 2;
}

template <int D, int NW, bool kMods, class Mod, int NG>
__device__ __forceinline__ bool fwd_split_item(const FwdArgs& a, char* lds, uint32_t* flag) {
  using Tile = SplitTile<D, NW>;
  constexpr int BM = 32 * NW, BN = 32, KS = D / 16, DT = D / 32, TB = Tile::kBytes;
  const Problem& P = a.p;
  const int grp = NG > 1 ? __builtin_amdgcn_readfirstlane((int)threadIdx.x / (NW * 64)) : 0;
  const int tid = threadIdx.x - grp * NW * 64, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 31, hh = lane >> 5;
  const int nqt = (P.Sq + BM - 1) / BM;
  int head, qt;
  work_item(blockIdx.x, P.B * P.Hq, nqt, P.xcd_remap, P.head_group_q, false, &head, &qt);
  const int b = head / P.Hq, h = head - b * P.Hq;
  const int hk = h / (P.Hq / P.Hkv);
  const int q0 = qt * BM;
  const int qw = q0 + 32 * w + lr;
  const bool qvalid = qw < P.Sq;
  const float* kp = static_cast<const float*>(a.k) + (size_t)(b * P.Hkv + hk) * P.Skv * D;
  const float* vp = static_cast<const float*>(a.v) + (size_t)(b * P.Hkv + hk) * P.Skv * D;

  KvWalk walk = make_kv_walk(P, b, h, q0, BN);
  const int n_it = walk.count(), n_full = walk.count_full();
  const int sub_log2 = log2_if_pow2(walk.sub);
  KvTab tab;
  // group grp takes tiles grp, grp + NG, ..; one past the walk is a tile of
  // no rows (skipped, zeros into the idle buffer)
  auto kbase_of = [&](int it) { return it < n_it ? tab.kbase(walk, it, sub_log2, lane) : kPastEnd; };
  char* const tiles = lds + grp * f32_lds_bytes<D>();

  // The rows of tile it + 1 are split into LDS during tile it's S products and
  // were loaded during tile it - 1: kb_c, kb_s, the starts of the current tile
  // and of the staged one.
  SplitStage<D, NW> ks, vs;
  int kb_c = kbase_of(grp), kb_s = kPastEnd;
  auto load_tile = [&](int kb) {
    ks.load(kp, kb, P.Skv, tid);
    vs.load(vp, kb, P.Skv, tid);
  };
  load_tile(kb_c);
  Frag3 qf[KS];
  float mag = load_rows3<D, false>(qf, static_cast<const float*>(a.q) + (size_t)head * P.Sq * D, qw, qvalid, hh, 0.f);
  const float slope = P.alibi ? P.alibi[h] : 0.f;
  ElemMask em;
  em.interval = interval_mask(P);
  key_interval(P, b, qw, &em.lo, &em.hi);
  em.doc = (!em.interval && qvalid) ? P.q_doc[(size_t)b * P.Sq + qw] : 0;
  Tile kt;
  kt.init(lane);

  f32x16 oacc[DT];
#pragma unroll
  for (int i = 0; i < DT; ++i) zero16(oacc[i]);
  float m = -INFINITY, l = 0.f;

  auto stage_kv = [&](int buf, int st) {
    mag = stage_step<D, NW, false>(ks, vs, tiles + buf * TB, tiles + (2 + buf) * TB, st, tid, mag);
  };
#pragma unroll
  for (int st = 0; st < KS; ++st) stage_kv(0, st);
  kb_s = kbase_of(grp + NG);
  load_tile(kb_s);
  __syncthreads();
  auto tile_step = [&](int it, auto buf_c) {
    constexpr int buf = decltype(buf_c)::value;
    const int kbase = kb_c;
    kb_c = kb_s;
    // a tile past the keys (or the walk) is all masked
    const bool masked = it >= n_full || kbase + BN > P.Skv;
    const char* kl = tiles + buf * TB;
    const char* vl = tiles + (2 + buf) * TB;
    f32x16 sacc;
    zero16(sacc);
    mma6_rows<D, NW>(kt, kl, qf, sacc, [&](int st) { stage_kv(buf ^ 1, st); });
    kb_s = kbase_of(it + 2 * NG);  // (scalar work, behind the products just issued)
    load_tile(kb_s);
    Frag3 va[2];
    va[0] = kt.cols(vl, 0, 0);
    if constexpr (kMods) {  // log2-domain logits; without mods raw q.k, scaled in the exponent's FMA
#pragma unroll
      for (int e = 0; e < 16; ++e)
        sacc[e] = mod_score_t<Mod, kMods>(P, sacc[e], slope, b, h, qw, kbase + acc_row(e, hh), nullptr);
    }
    if (masked) {
      if (em.interval) {
        // (nothing to drop where every row of the wave sees the whole tile)
        if (Mod::kMask || !__all(!qvalid || (em.lo <= kbase && em.hi >= kbase + 31))) {
          const int base = kbase + 8 * hh;
          uint32_t bits = interval_bits(em.lo - base, em.hi - base);
          if constexpr (Mod::kMask) {
            uint32_t user = 0u;
#pragma unroll
            for (int e = 0; e < 16; ++e) {
              const int r = acc_row(e, 0);
              user |= Mod::mask(P, b, h, qw, base + r) ? (1u << r) : 0u;
            }
            bits &= user;
          }
#pragma unroll
          for (int e = 0; e < 16; ++e) sacc[e] = keep_bit(sacc[e], bits, acc_row(e, 0), -INFINITY);
        }
      } else {
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int key = kbase + acc_row(e, hh);
          if (!(key < P.Skv && mod_mask_ok<Mod>(P, b, h, qw, key, em.doc, kv_doc_of(P, b, key)))) sacc[e] = -INFINITY;
        }
      }
    }
    const float sc = kMods ? 1.0f : P.scale_log2;
    float mx = -INFINITY;
#pragma unroll
    for (int e = 0; e < 16; ++e) mx = fmaxf(mx, sacc[e]);
    mx = pair_max(mx) * sc;
    // the reference maximum m only follows a row's maximum once that is more
    // than 2^8 above it (P <= 2^8, far from overflow; O / l does not depend on m)
    if (__any(mx > m + 8.0f)) {
      const float mnew = fmaxf(m, mx);
      const float alpha = fast_exp2(m - (mnew == -INFINITY ? 0.f : mnew));
      l *= alpha;
      m = mnew;
#pragma unroll
      for (int i = 0; i < DT; ++i)
#pragma unroll
        for (int e = 0; e < 16; ++e) oacc[i][e] *= alpha;
    }
    const float muse = m == -INFINITY ? 0.f : m;
    // P of rows 16 c + .. (elements 8 c + 2 j, + 1), split; the second half
    // between the first one's products
    float r0 = 0.f, r1 = 0.f;
    Frag3 pf[2];
    auto exps = [&](int c, int j) {
      const float x = fast_exp2(fmaf(sacc[8 * c + 2 * j], sc, -muse));
      const float y = fast_exp2(fmaf(sacc[8 * c + 2 * j + 1], sc, -muse));
      r0 += x;
      r1 += y;
      split2(pf[c], j, x * kUp, y * kUp);
    };
#pragma unroll
    for (int j = 0; j < 4; ++j) exps(0, j);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int x = 0; x < 2 * DT; ++x) {
      if (x + 1 < 2 * DT) va[(x + 1) & 1] = kt.cols(vl, (x + 1) % DT, (x + 1) / DT);
      __builtin_amdgcn_sched_barrier(0);
      oacc[x % DT] = mma6(va[x & 1], pf[x / DT], oacc[x % DT]);
      if (x < DT) {
#pragma unroll
        for (int j = 4 * x / DT; j < 4 * (x + 1) / DT; ++j) exps(1, j);
      }
      mix_mfma_valu<6, 6>();
      __builtin_amdgcn_sched_barrier(0);
    }
    l += r0 + r1;
    __syncthreads();
  };
  // (the trip count is the workgroup's, not the group's: a tile is a barrier)
  int it = 0;
  for (; it + NG < n_it; it += 2 * NG) {
    tile_step(it + grp, Int<0>{});
    tile_step(it + NG + grp, Int<1>{});
  }
  if (it < n_it) tile_step(it + grp, Int<0>{});

  if (any_large(mag, qvalid ? finite_probe<DT>(oacc, 0.f) : 0.f, flag)) return false;
  if constexpr (NG > 1) {  // group 1's (m, l, O) through LDS, merged by group 0
    float* x = reinterpret_cast<float*>(lds) + tid;
    if (grp) {
      put_acc<DT, NW>(x, oacc);
      x[DT * 16 * NW * 64] = m;
      x[(DT * 16 + 1) * NW * 64] = l;
    }
    __syncthreads();
    if (grp) return true;
    const float m1 = x[DT * 16 * NW * 64], l1 = x[(DT * 16 + 1) * NW * 64];
    const float mm = fmaxf(m, m1), mu = mm == -INFINITY ? 0.f : mm;
    const float c0 = fast_exp2(m - mu), c1 = fast_exp2(m1 - mu);
    l = l * c0 + l1 * c1;
    m = mm;
#pragma unroll
    for (int i = 0; i < DT; ++i)
#pragma unroll
      for (int e = 0; e < 16; ++e) oacc[i][e] = oacc[i][e] * c0 + x[(i * 16 + e) * NW * 64] * c1;
  }
  const float lt = pair_sum(l);
  const float inv = lt > 0.f ? kDown2 / lt : 0.f;
  if (qvalid) {
    float* op = static_cast<float*>(a.o) + ((size_t)head * P.Sq + qw) * D;
#pragma unroll
    for (int i = 0; i < DT; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        *reinterpret_cast<f32x4*>(op + 32 * i + 8 * j + 4 * hh) =
            f32x4{oacc[i][4 * j] * inv, oacc[i][4 * j + 1] * inv, oacc[i][4 * j + 2] * inv, oacc[i][4 * j + 3] * inv};
    if (hh == 0) a.lse[(size_t)head * P.Sq + qw] = lt > 0.f ? (m + log2f(lt)) * kLn2 : -INFINITY;
  }
  return true;
}

template <int D, int NW, bool kMods, class Mod = BuiltinMod, int NG = 1>
__global__ __launch_bounds__(NG * NW * 64) __attribute__((amdgpu_waves_per_eu(D == 128 ? 1 : 2)))
void fwd_f32_kernel(FwdArgs a) {
  __shared__ __attribute__((aligned(1024))) char lds[NG * f32_lds_bytes<D>()];
  static_assert(fwd_item_lds<float, D, 32>() <= f32_lds_bytes<D>(), "shared by both paths");
  __shared__ uint32_t flag;
  if (fwd_split_item<D, NW, kMods, Mod, NG>(a, lds, &flag)) return;
  __syncthreads();
  // the general code has no groups: it counts on NW waves
  if (NG > 1 && threadIdx.x >= NW * 64) return;
  fwd_item<float, D, 32, NW, kMods, Mod>(a, lds);
}

// ------------------------------------------------------------------- dQ ----
template <int D, int NW, bool kMods, class Mod, int NG>
__device__ __forceinline__ bool dq_split_item(const BwdArgs& a, char* lds, uint32_t* flag) {
  using Tile = SplitTile<D, NW>;
  constexpr int BM = 32 * NW, BN = 32, KS = D / 16, DT = D / 32, TB = Tile::kBytes;
  const Problem& P = a.p;
  const int grp = NG > 1 ? __builtin_amdgcn_readfirstlane((int)threadIdx.x / (NW * 64)) : 0;
  const int tid = threadIdx.x - grp * NW * 64, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 31, hh = lane >> 5;
  const int nqt = (P.Sq + BM - 1) / BM;
  int head, qt;
  work_item(blockIdx.x, P.B * P.Hq, nqt, P.xcd_remap, P.head_group_q, false, &head, &qt);
  const int b = head / P.Hq, h = head - b * P.Hq;
  const int hk = h / (P.Hq / P.Hkv);
  const int q0 = qt * BM;
  const int qw = q0 + 32 * w + lr;
  const bool qvalid = qw < P.Sq;
  const float* kp = static_cast<const float*>(a.k) + (size_t)(b * P.Hkv + hk) * P.Skv * D;
  const float* vp = static_cast<const float*>(a.v) + (size_t)(b * P.Hkv + hk) * P.Skv * D;

  KvWalk walk = make_kv_walk(P, b, h, q0, BN);
  const int n_it = walk.count(), n_full = walk.count_full();
  const int sub_log2 = log2_if_pow2(walk.sub);
  KvTab tab;
  // group grp takes tiles grp, grp + NG, ..; one past the walk is a tile of
  // no rows (skipped, zeros into the idle buffer)
  auto kbase_of = [&](int it) { return it < n_it ? tab.kbase(walk, it, sub_log2, lane) : kPastEnd; };
  char* const tiles = lds + grp * f32_lds_bytes<D>();

  // The rows of tile it + 1 are split into LDS during tile it's S products and
  // were loaded during tile it - 1: kb_c, kb_s, the starts of the current tile
  // and of the staged one.
  SplitStage<D, NW> ks, vs;
  int kb_c = kbase_of(grp), kb_s = kPastEnd;
  auto load_tile = [&](int kb) {
    ks.load(kp, kb, P.Skv, tid);
    vs.load(vp, kb, P.Skv, tid);
  };
  load_tile(kb_c);
  Frag3 qf[KS], df[KS];
  const size_t qoff = (size_t)head * P.Sq * D;
  float mag = load_rows3<D>(qf, static_cast<const float*>(a.q) + qoff, qw, qvalid, hh, 0.f);
  load_rows3<D>(df, static_cast<const float*>(a.dout) + qoff, qw, qvalid, hh, 0.f);
  const size_t rowi = (size_t)head * P.Sq + qw;
  // a row with no live key (LSE = -inf) gets P = 0 everywhere, like rows past Sq
  const float lse_row = qvalid ? a.lse[rowi] : -INFINITY;
  const float lse2 = lse_row > -INFINITY ? lse_row * kLog2e : INFINITY;
  const float dl = qvalid ? a.delta[rowi] * kUp : 0.f;
  const float slope = P.alibi ? P.alibi[h] : 0.f;
  ElemMask em;
  em.interval = interval_mask(P);
  key_interval(P, b, qw, &em.lo, &em.hi);
  em.doc = (!em.interval && qvalid) ? P.q_doc[(size_t)b * P.Sq + qw] : 0;
  Tile kt;
  kt.init(lane);

  f32x16 dqa[DT];
#pragma unroll
  for (int i = 0; i < DT; ++i) zero16(dqa[i]);

  auto stage_kv = [&](int buf, int st) {
    mag = stage_step<D, NW>(ks, vs, tiles + buf * TB, tiles + (2 + buf) * TB, st, tid, mag);
  };
#pragma unroll
  for (int st = 0; st < KS; ++st) stage_kv(0, st);
  kb_s = kbase_of(grp + NG);
  load_tile(kb_s);
  __syncthreads();
  auto tile_step = [&](int it, auto buf_c) {
    constexpr int buf = decltype(buf_c)::value;
    const int kbase = kb_c;
    kb_c = kb_s;
    const bool masked = it >= n_full || kbase + BN > P.Skv;
    const char* kl = tiles + buf * TB;
    const char* vl = tiles + (2 + buf) * TB;
    f32x16 sacc, pacc;
    zero16(sacc);
    zero16(pacc);
    mma6_rows2<D, NW>(kt, kl, vl, qf, df, sacc, pacc, [&](int st) { stage_kv(buf ^ 1, st); });
    kb_s = kbase_of(it + 2 * NG);  // (scalar work, behind the products just issued)
    load_tile(kb_s);
    Frag3 ka[2];
    ka[0] = kt.cols(kl, 0, 0);
    float dsdx[16];
    if constexpr (kMods) {
#pragma unroll
      for (int e = 0; e < 16; ++e)
        sacc[e] = mod_score_t<Mod, kMods>(P, sacc[e] * kDown2, slope, b, h, qw, kbase + acc_row(e, hh), &dsdx[e]);
    }
    if (masked) {
      if (em.interval) {
        // (nothing to drop where every row of the wave sees the whole tile)
        if (Mod::kMask || !__all(!qvalid || (em.lo <= kbase && em.hi >= kbase + 31))) {
          const int base = kbase + 8 * hh;
          uint32_t bits = interval_bits(em.lo - base, em.hi - base);
          if constexpr (Mod::kMask) {
            uint32_t user = 0u;
#pragma unroll
            for (int e = 0; e < 16; ++e) {
              const int r = acc_row(e, 0);
              user |= Mod::mask(P, b, h, qw, base + r) ? (1u << r) : 0u;
            }
            bits &= user;
          }
#pragma unroll
          for (int e = 0; e < 16; ++e) {
            sacc[e] = keep_bit(sacc[e], bits, acc_row(e, 0), -INFINITY);
            if constexpr (kMods) dsdx[e] = keep_bit(dsdx[e], bits, acc_row(e, 0), 0.f);
          }
        }
      } else {
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int key = kbase + acc_row(e, hh);
          const bool keep = key < P.Skv && mod_mask_ok<Mod>(P, b, h, qw, key, em.doc, kv_doc_of(P, b, key));
          sacc[e] = keep ? sacc[e] : -INFINITY;
          if constexpr (kMods) dsdx[e] = keep ? dsdx[e] : 0.f;
        }
      }
    }
    const float sc = kMods ? 1.0f : P.scale_log2 * kDown2;
    Frag3 sf[2];
    auto grads = [&](int c, int j) {  // 2^16 dS of elements 8 c + 2 j, + 1, split
      float y[2];
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const int e = 8 * c + 2 * j + t;
        y[t] = fast_exp2(fmaf(sacc[e], sc, -lse2)) * fmaf(pacc[e], kDown, -dl);
        if constexpr (kMods) y[t] *= dsdx[e];
      }
      split2(sf[c], j, y[0], y[1]);
    };
#pragma unroll
    for (int j = 0; j < 4; ++j) grads(0, j);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int x = 0; x < 2 * DT; ++x) {
      if (x + 1 < 2 * DT) ka[(x + 1) & 1] = kt.cols(kl, (x + 1) % DT, (x + 1) / DT);
      __builtin_amdgcn_sched_barrier(0);
      dqa[x % DT] = mma6(ka[x & 1], sf[x / DT], dqa[x % DT]);
      if (x < DT) {
#pragma unroll
        for (int j = 4 * x / DT; j < 4 * (x + 1) / DT; ++j) grads(1, j);
      }
      mix_mfma_valu<6, 6>();
      __builtin_amdgcn_sched_barrier(0);
    }
    __syncthreads();
  };
  // (the trip count is the workgroup's, not the group's: a tile is a barrier)
  int it = 0;
  for (; it + NG < n_it; it += 2 * NG) {
    tile_step(it + grp, Int<0>{});
    tile_step(it + NG + grp, Int<1>{});
  }
  if (it < n_it) tile_step(it + grp, Int<0>{});

  if (any_large(mag, qvalid ? finite_probe<DT>(dqa, 0.f) : 0.f, flag)) return false;
  if constexpr (NG > 1) {
    float* x = reinterpret_cast<float*>(lds) + tid;
    if (grp) put_acc<DT, NW>(x, dqa);
    __syncthreads();
    if (grp) return true;
    add_acc<DT, NW>(x, dqa);
  }
  if (qvalid) {
    float* dqp = static_cast<float*>(a.dq) + rowi * D;
    const GradScale gs(P.scale);
#pragma unroll
    for (int i = 0; i < DT; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        *reinterpret_cast<f32x4*>(dqp + 32 * i + 8 * j + 4 * hh) =
            f32x4{gs(dqa[i][4 * j]), gs(dqa[i][4 * j + 1]), gs(dqa[i][4 * j + 2]), gs(dqa[i][4 * j + 3])};
  }
  return true;
}

template <int D, int NW, bool kMods, class Mod = BuiltinMod, int NG = 1>
__global__ __launch_bounds__(NG * NW * 64) __attribute__((amdgpu_waves_per_eu(D == 128 ? 1 : 2)))
void dq_f32_kernel(BwdArgs a) {
  __shared__ __attribute__((aligned(1024))) char lds[NG * f32_lds_bytes<D>()];
  static_assert(dq_item_lds<float, D, 32>() <= f32_lds_bytes<D>(), "shared by both paths");
  __shared__ uint32_t flag;
  if (dq_split_item<D, NW, kMods, Mod, NG>(a, lds, &flag)) return;
  __syncthreads();
  // the general code has no groups: it counts on NW waves
  if (NG > 1 && threadIdx.x >= NW * 64) return;
  dq_item<float, D, 32, NW, kMods, Mod>(a, lds);
}

// ---------------------------------------------------------------- dK dV ----
template <int D, int NW, bool kMods, class Mod, int NG>
__device__ __forceinline__ bool dkdv_split_item(const BwdArgs& a, char* lds, float* stat, uint32_t* flag) {
  using Tile = SplitTile<D, NW>;
  constexpr int BKV = 32 * NW, BQ = 32, KS = D / 16, DT = D / 32, TB = Tile::kBytes;
  // At D = 128 the K and V pieces and the accumulators take 320 registers:
  // operands are read when they are due and each half of P and dS is used up
  // before the next (the overlapped form spills).
  constexpr bool kLean = D == 128;
  const Problem& P = a.p;
  const int grp = NG > 1 ? __builtin_amdgcn_readfirstlane((int)threadIdx.x / (NW * 64)) : 0;
  const int tid = threadIdx.x - grp * NW * 64, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 31, hh = lane >> 5;
  const int nkt = (P.Skv + BKV - 1) / BKV;
  const int g = P.Hq / P.Hkv;
  int head, kt0;
  work_item(blockIdx.x, P.B * P.Hkv, nkt, P.xcd_remap, P.head_group_kv, true, &head, &kt0);
  const int b = head / P.Hkv, hk = head - b * P.Hkv;
  const int k0 = kt0 * BKV;
  const int kw = k0 + 32 * w + lr;  // this lane's key
  const bool kvalid = kw < P.Skv;

  QWalk walk;
  walk.P = &P;
  walk.b = b;
  walk.hq0 = hk * g;
  walk.g = g;
  walk.kvrow = k0 / P.mblk_kv;
  walk.sub = P.mblk_q / BQ;
  walk.bq = BQ;
  walk.dense = !P.has_tables;
  walk.ntiles_dense = (P.Sq + BQ - 1) / BQ;
  walk.init();
  const int n_it = walk.count(), n_full = walk.count_full();

  char* const tiles = lds + grp * f32_lds_bytes<D>();
  stat += grp * 128;

  SplitStage<D, NW> qs, ds;
  float lse_in = 0.f, dl_in = 0.f;
  auto gload = [&](int hq, int qb) {
    const size_t hoff = (size_t)(b * P.Hq + hq) * P.Sq;
    qs.load(static_cast<const float*>(a.q) + hoff * D, qb, P.Sq, tid);
    ds.load(static_cast<const float*>(a.dout) + hoff * D, qb, P.Sq, tid);
    if (tid < BQ) {
      const int qi = qb + tid;
      lse_in = qi < P.Sq ? a.lse[hoff + qi] : -INFINITY;
      dl_in = qi < P.Sq ? a.delta[hoff + qi] : 0.f;
    }
  };
  auto stat_store = [&](int buf) {  // rows past Sq and rows with no live key (LSE = -inf): P = 0
    if (tid < BQ) {
      stat[buf * 64 + tid] = lse_in > -INFINITY ? lse_in * kLog2e : INFINITY;
      stat[buf * 64 + 32 + tid] = dl_in;
    }
  };
  // As in the forward, tile it + 1 is split into LDS during tile it's first
  // products, tile it + 2 is loaded after them, and its table entry is fetched
  // a tile before that.  A tile past the walk starts at Sq: no rows.
  int hq_c = walk.hq0, qb_c = P.Sq, hq_s = walk.hq0, qb_s = P.Sq;
  TileRef ref{0, 0, walk.hq0};
  auto resolve = [&](int it, int& hq, int& qb) {  // tile it, fetched before
    hq = it < n_it ? ref.hq : walk.hq0;
    qb = it < n_it ? walk.qbase(ref) : P.Sq;
  };
  auto fetch = [&](int it) {
    if (it < n_it) ref = walk.fetch(it);
  };
  fetch(grp);
  resolve(grp, hq_c, qb_c);
  gload(hq_c, qb_c);
  fetch(grp + NG);
  Frag3 kf[KS], vf[KS];
  float mag = load_rows3<D>(kf, static_cast<const float*>(a.k) + (size_t)head * P.Skv * D, kw, kvalid, hh, 0.f);
  load_rows3<D>(vf, static_cast<const float*>(a.v) + (size_t)head * P.Skv * D, kw, kvalid, hh, 0.f);
  ElemMask em;
  em.interval = interval_mask(P);
  query_interval(P, b, kw, &em.lo, &em.hi);
  em.doc = (!em.interval && kvalid) ? P.kv_doc[(size_t)b * P.Skv + kw] : 0;
  Tile qt;
  qt.init(lane);

  f32x16 dka[DT], dva[DT];
#pragma unroll
  for (int i = 0; i < DT; ++i) {
    zero16(dka[i]);
    zero16(dva[i]);
  }
  auto stage_q = [&](int buf, int st) {
    mag = stage_step<D, NW>(qs, ds, tiles + buf * TB, tiles + (2 + buf) * TB, st, tid, mag);
  };
#pragma unroll
  for (int st = 0; st < KS; ++st) stage_q(0, st);
  stat_store(0);
  resolve(grp + NG, hq_s, qb_s);
  gload(hq_s, qb_s);
  fetch(grp + 2 * NG);
  __syncthreads();
  auto tile_step = [&](int it, auto buf_c) {
    constexpr int buf = decltype(buf_c)::value;
    const int hq = hq_c, qbase = qb_c;
    hq_c = hq_s;
    qb_c = qb_s;
    const bool masked = it >= n_full || qbase >= P.Sq;
    const float slope = P.alibi ? P.alibi[hq] : 0.f;
    const char* ql = tiles + buf * TB;
    const char* dl = tiles + (2 + buf) * TB;
    f32x16 sacc, pacc;
    zero16(sacc);
    zero16(pacc);
    mma6_rows2<D, NW, kLean ? 0 : 1>(qt, ql, dl, kf, vf, sacc, pacc, [&](int st) { stage_q(buf ^ 1, st); });
    stat_store(buf ^ 1);
    resolve(it + 2 * NG, hq_s, qb_s);
    fetch(it + 3 * NG);
    gload(hq_s, qb_s);
    constexpr int R = kLean ? 1 : 2;
    Frag3 da[R], qa[R];
    if constexpr (!kLean) {
      da[0] = qt.cols(dl, 0, 0);
      qa[0] = qt.cols(ql, 0, 0);
    }
    f32x4 ls[4], dd[4];  // LSE and Delta of rows acc_row(4 q ..)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      ls[q] = *reinterpret_cast<const f32x4*>(stat + buf * 64 + acc_row(4 * q, hh));
      dd[q] = *reinterpret_cast<const f32x4*>(stat + buf * 64 + 32 + acc_row(4 * q, hh));
    }
    float dsdx[16];
    if constexpr (kMods) {
#pragma unroll
      for (int e = 0; e < 16; ++e)
        sacc[e] = mod_score_t<Mod, kMods>(P, sacc[e] * kDown2, slope, b, hq, qbase + acc_row(e, hh), kw, &dsdx[e]);
    }
    if (masked) {
      if (em.interval) {
        // (nothing to drop where every row of the wave sees the whole tile)
        if (Mod::kMask || !__all(!kvalid || (em.lo <= qbase && em.hi >= qbase + 31))) {
          const int base = qbase + 8 * hh;
          uint32_t bits = interval_bits(em.lo - base, em.hi - base);
          if constexpr (Mod::kMask) {
            uint32_t user = 0u;
#pragma unroll
            for (int e = 0; e < 16; ++e) {
              const int r = acc_row(e, 0);
              user |= Mod::mask(P, b, hq, base + r, kw) ? (1u << r) : 0u;
            }
            bits &= user;
          }
#pragma unroll
          for (int e = 0; e < 16; ++e) {
            sacc[e] = keep_bit(sacc[e], bits, acc_row(e, 0), -INFINITY);
            if constexpr (kMods) dsdx[e] = keep_bit(dsdx[e], bits, acc_row(e, 0), 0.f);
          }
        }
      } else {
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int qi = qbase + acc_row(e, hh);
          const bool keep = kvalid && qi < P.Sq && mod_mask_ok<Mod>(P, b, hq, qi, kw, q_doc_of(P, b, qi), em.doc);
          sacc[e] = keep ? sacc[e] : -INFINITY;
          if constexpr (kMods) dsdx[e] = keep ? dsdx[e] : 0.f;
        }
      }
    }
    const float sc = kMods ? 1.0f : P.scale_log2 * kDown2;
    Frag3 pf[R], sf[R];
    auto grads = [&](int c, int j) {  // 2^16 P and 2^16 dS (rows = queries, column = this lane's key), split
      float x[2], y[2];
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const int e = 8 * c + 2 * j + t;
        x[t] = fast_exp2(fmaf(sacc[e], sc, -ls[e >> 2][e & 3])) * kUp;
        y[t] = x[t] * fmaf(pacc[e], kDown2, -dd[e >> 2][e & 3]);
        if constexpr (kMods) y[t] *= dsdx[e];
      }
      split2(pf[c % R], j, x[0], x[1]);
      split2(sf[c % R], j, y[0], y[1]);
    };
    if constexpr (!kLean) {
#pragma unroll
      for (int j = 0; j < 4; ++j) grads(0, j);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int x = 0; x < 2 * DT; ++x) {
      const int c = x / DT, i = x % DT;
      if constexpr (kLean) {
        if (i == 0) {
#pragma unroll
          for (int j = 0; j < 4; ++j) grads(c, j);
        }
        da[0] = qt.cols(dl, i, c);
        qa[0] = qt.cols(ql, i, c);
      } else if (x + 1 < 2 * DT) {
        da[(x + 1) % R] = qt.cols(dl, (x + 1) % DT, (x + 1) / DT);
        qa[(x + 1) % R] = qt.cols(ql, (x + 1) % DT, (x + 1) / DT);
      }
      __builtin_amdgcn_sched_barrier(0);
      dva[i] = mma6(da[x % R], pf[c % R], dva[i]);
      dka[i] = mma6(qa[x % R], sf[c % R], dka[i]);
      if (!kLean && x < DT) {
#pragma unroll
        for (int j = 4 * x / DT; j < 4 * (x + 1) / DT; ++j) grads(1, j);
      }
      mix_mfma_valu<12, 6>();
      __builtin_amdgcn_sched_barrier(0);
    }
    __syncthreads();
  };
  // (the trip count is the workgroup's, not the group's: a tile is a barrier)
  int it = 0;
  for (; it + NG < n_it; it += 2 * NG) {
    tile_step(it + grp, Int<0>{});
    tile_step(it + NG + grp, Int<1>{});
  }
  if (it < n_it) tile_step(it + grp, Int<0>{});

  if (any_large(mag, kvalid ? finite_probe<DT>(dva, finite_probe<DT>(dka, 0.f)) : 0.f, flag)) return false;
  if constexpr (NG > 1) {
    float* x = reinterpret_cast<float*>(lds) + tid;
    if (grp) {
      put_acc<DT, NW>(x, dka);
      put_acc<DT, NW>(x + DT * 16 * NW * 64, dva);
    }
    __syncthreads();
    if (grp) return true;
    add_acc<DT, NW>(x, dka);
    add_acc<DT, NW>(x + DT * 16 * NW * 64, dva);
  }
  if (kvalid) {
    float* dkp = static_cast<float*>(a.dk) + ((size_t)head * P.Skv + kw) * D;
    float* dvp = static_cast<float*>(a.dv) + ((size_t)head * P.Skv + kw) * D;
    const GradScale gs(P.scale), gv(1.0f);
#pragma unroll
    for (int i = 0; i < DT; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int d0 = 32 * i + 8 * j + 4 * hh;
        *reinterpret_cast<f32x4*>(dkp + d0) =
            f32x4{gs(dka[i][4 * j]), gs(dka[i][4 * j + 1]), gs(dka[i][4 * j + 2]), gs(dka[i][4 * j + 3])};
        *reinterpret_cast<f32x4*>(dvp + d0) =
            f32x4{gv(dva[i][4 * j]), gv(dva[i][4 * j + 1]), gv(dva[i][4 * j + 2]), gv(dva[i][4 * j + 3])};
      }
  }
  return true;
}

template <int D, int NW, bool kMods, class Mod = BuiltinMod, int NG = 1>
__global__ __launch_bounds__(NG * NW * 64) __attribute__((amdgpu_waves_per_eu(NG)))
void dkdv_f32_kernel(BwdArgs a) {
  __shared__ __attribute__((aligned(1024))) char lds[NG * f32_lds_bytes<D>()];
  static_assert(dkdv_item_lds<float, D, 32>() <= f32_lds_bytes<D>(), "shared by both paths");
  __shared__ __attribute__((aligned(16))) float stat[NG * 128];  // per group and buffer: LSE log2(e), Delta of 32 rows
  __shared__ uint32_t flag;
  if (dkdv_split_item<D, NW, kMods, Mod, NG>(a, lds, stat, &flag)) return;
  __syncthreads();
  // the general code has no groups: it counts on NW waves
  if (NG > 1 && threadIdx.x >= NW * 64) return;
  dkdv_item<float, D, 32, NW, kMods, Mod>(a, lds);
}

}  // namespace fa
