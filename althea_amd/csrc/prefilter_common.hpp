// GGX prefilter of texel pairs, or single texels, shared by the single-map and
// the batched (persistent) kernels, so both produce bit-identical texels.
#pragma once

#include <type_traits>

#include "device_math.hpp"
#include "precise_lookup.hpp"

namespace althea {

// Sample-table entry (one per Hammersley sample with NdotL > 0, in sample
// order): L in the texel frame (T, B, N), the source LOD split into levels
// (l0, l1) and fraction delta, and the sample's weight in the NdotL-weighted
// mean (NdotL = lz, or the summed weight of coinciding samples) with its
// shares of the two levels, w0 = weight (1 - delta) and w1 = weight delta
// (rounded once from FP64; w1 = 0 where the sample reads one level).
// 32 bytes, one scalar load.
struct GgxEntry {
  float lx, ly, lz, w0;
  int l0, l1;
  float w1, weight;
};
static_assert(sizeof(GgxEntry) == 32, "one scalar load per entry");

constexpr int kBlockSums = 32;  // FP32 partial sums flushed to FP64 every 32 samples

// Two texels share every sample's direction and angles.  A texel n and its
// partner F n on the opposite face, F a half turn about the axis that the
// frame's |x| > |y| branch (Sampling.glsl:58-70) leaves in place, have frames
// that are each other's image under F, so sample by sample L' = F L:
//   kTurnY (|x| > |y|): F = (-x, y, -z), yaw' = yaw + pi, pitch' = pitch (the
//     precompute's pole branch, yaw 0, stays where it is);
//   kTurnX (otherwise):  F = (x, -y, -z), yaw' = -yaw, pitch' = -pitch.
// Both act on a level's texel lattice exactly (an even or unit width), so the
// partner's lookup takes the same fractions and weights at a shifted, or
// mirrored, cell.  kAlone: a texel by itself (prefilter_alone).
enum PairTurn { kTurnY, kTurnX, kAlone };

// Partner of texel (face, x, y) of an S x S face, face +X, +Y or +Z.
__device__ __forceinline__ void pair_partner(int face, int x, int y, int S, bool turn_y, int& face2, int& x2,
                                             int& y2) {
  face2 = face + 1;
  const bool mirror = face == 4 && !turn_y;
  x2 = mirror ? S - 1 - x : x;
  y2 = mirror ? S - 1 - y : y;
}

// Sums of the NdotL-weighted source for a pair of texels (kN = 6: RGB of the
// texel, RGB of its partner) or one (3): FP64 (kF64Sums) or FP32 totals, and the
// FP32 weight sum of the all-FP32 variant.
template <bool kF64Sums, int kN>
struct PrefilterSums {
  using T = typename std::conditional<kF64Sums, double, float>::type;
  T v[kN] = {};
  float w = 0.0f;
};

// Source lookups of the sample loop: add<turn> adds an entry's weighted bilinear
// values into s[0..2] for the texel and s[3..5] for its partner.  `turn` is
// +1 / -1 where yaw < 0 / yaw >= 0 (kTurnY: the half turn that stays in
// [-pi, pi]) and 0 in the pole branch.  Levels from `first` on are staged in
// LDS; finer ones, which few samples name, are read from the pyramid.  Both
// read the same texels with the same weights in the same order.
struct PairTaps {
  LevelTaps a, b;  // the texel's cell, its partner's
};
template <bool kTogether>
struct StagedAcc {
  const char* lds;
  const StagedLevel* __restrict__ slv;
  const char* __restrict__ pyr;
  const LevelC* __restrict__ lv;
  int first;

  template <PairTurn kTurn>
  __device__ __forceinline__ PairTaps staged(int l, float yaw, float pitch, int turn) const {
    const StagedLevel& g = slv[l];
    const TexelCoord q = texel_coord(g, yaw, pitch);
    const uint32_t o = staged_offset(g, q.ix, q.iy);
    PairTaps t;
    staged_texels(lds, g, o, t.a);
    if (kTurn != kAlone)
      staged_texels(lds, g,
                    kTurn == kTurnY ? o + static_cast<uint32_t>(__mul24(turn, static_cast<int>(g.half))) : g.mirror - o,
                    t.b);
    t.a.ax = q.ax, t.a.ay = q.ay;
    return t;
  }
  template <PairTurn kTurn>
  __device__ __forceinline__ PairTaps pyramid(int l, float yaw, float pitch, int turn) const {
    const LevelC& c = lv[l];
    const TexelCoord q = texel_coord(c, yaw, pitch);
    const int W = static_cast<int>(c.wmask) + 1, H = static_cast<int>(c.hmask) + 1;
    PairTaps t;
    level_texels(pyr, c, q.ix, q.iy, t.a);
    if (kTurn == kTurnY)
      level_texels(pyr, c, q.ix + __mul24(turn, W >> 1), q.iy, t.b);
    else if (kTurn == kTurnX)
      level_texels(pyr, c, W - 2 - q.ix, H - 2 - q.iy, t.b);
    t.a.ax = q.ax, t.a.ay = q.ay;
    return t;
  }
  template <PairTurn kTurn>
  __device__ __forceinline__ static void sum(const PairTaps& t, float w, float* s) {
    const TapWeights k = tap_weights(t.a.ax, t.a.ay, w);
    taps_acc(t.a, k, s[0], s[1], s[2]);
    if (kTurn != kAlone)
      taps_acc(t.b, kTurn == kTurnY ? k : TapWeights{k.w11, k.w01, k.w10, k.w00}, s[3], s[4], s[5]);
  }
  // A table entry's two levels.  kTogether: the reads of both are in flight
  // together where both are staged (48 registers of texels), for four waves a
  // SIMD; with six, a level at a time.
  template <PairTurn kTurn>
  __device__ __forceinline__ void add(const GgxEntry& e, float yaw, float pitch, int turn, float* s) const {
    const bool two = __float_as_uint(e.w1) != 0u;
    if (kTogether && two && e.l0 >= first) {
      const PairTaps t0 = staged<kTurn>(e.l0, yaw, pitch, turn), t1 = staged<kTurn>(e.l1, yaw, pitch, turn);
      sum<kTurn>(t0, e.w0, s);
      sum<kTurn>(t1, e.w1, s);
      return;
    }
    if (e.l0 >= first)
      sum<kTurn>(staged<kTurn>(e.l0, yaw, pitch, turn), e.w0, s);
    else
      sum<kTurn>(pyramid<kTurn>(e.l0, yaw, pitch, turn), e.w0, s);
    if (!two) return;
    if (e.l1 >= first)
      sum<kTurn>(staged<kTurn>(e.l1, yaw, pitch, turn), e.w1, s);
    else
      sum<kTurn>(pyramid<kTurn>(e.l1, yaw, pitch, turn), e.w1, s);
  }
};

// Table entries [lo, hi) for one pair, or texel (PreFilterEnvMap.comp:147-169): the
// FP32 per-sample body (each level's bilinear in weight form, added into
// running FP32 sums); kF64Sums flushes the FP32 sums into FP64 every
// kBlockSums entries (blocks aligned at multiples of kBlockSums).
template <bool kF64Sums, PairTurn kTurn, int kN, class Acc>
__device__ __forceinline__ PrefilterSums<kF64Sums, kN> prefilter_pair_range(const Acc& acc,
                                                                            const GgxEntry* __restrict__ tab, int lo,
                                                                            int hi, const Frame& fr) {
  static_assert(kN == (kTurn == kAlone ? 3 : 6), "three sums a texel");
  PrefilterSums<kF64Sums, kN> t;
  float s[kN] = {};
  GgxEntry next = tab[lo < hi ? lo : 0];
  for (int e = lo; e < hi; ++e) {
    const GgxEntry en = next;
    next = tab[e + 1 < hi ? e + 1 : e];
    const f3 L = mk(fmaf(fr.t.x, en.lx, fmaf(fr.b.x, en.ly, fr.n.x * en.lz)),
                    fmaf(fr.t.y, en.lx, fmaf(fr.b.y, en.ly, fr.n.y * en.lz)),
                    fmaf(fr.t.z, en.lx, fmaf(fr.b.z, en.ly, fr.n.z * en.lz)));
    // equirect_angles; the pole branch's selects only where some lane needs it.
    const float len_xz = sqrt_fast(fmaf(L.x, L.x, L.z * L.z));
    float yaw = atan2_fast(L.z, L.x), pitch = atan2_xpos(L.y, len_xz);
    int turn = kTurn == kTurnY ? (__float_as_uint(L.z) >> 31 ? 1 : -1) : 0;
    const bool pole = !(len_xz > 0.001f);
    if (__builtin_amdgcn_ballot_w64(pole)) {
      yaw = pole ? 0.0f : yaw;
      pitch = pole ? (L.y > 0.0f ? 0.5f * kPi : -0.5f * kPi) : pitch;
      turn = pole ? 0 : turn;
    }
    acc.template add<kTurn>(en, yaw, pitch, turn, s);
    if (kF64Sums) {
      if ((e & (kBlockSums - 1)) == kBlockSums - 1) {
#pragma unroll
        for (int c = 0; c < kN; ++c) t.v[c] += s[c], s[c] = 0.0f;
      }
    } else {
      t.w += en.weight;
    }
  }
#pragma unroll
  for (int c = 0; c < kN; ++c) t.v[c] += s[c];
  return t;
}

// The pair's values from its sums: FP64 sums over the FP64 weight sum, or
// all-FP32 sums over their own weight sum.
template <bool kF64Sums, int kN>
__device__ __forceinline__ float4 prefilter_value(const PrefilterSums<kF64Sums, kN>& t, int texel, double wsum) {
  const int c = 3 * texel;
  if (kF64Sums) {
    const double inv = 1.0 / wsum;
    return make_float4(static_cast<float>(t.v[c] * inv), static_cast<float>(t.v[c + 1] * inv),
                       static_cast<float>(t.v[c + 2] * inv), 1.0f);
  }
  return make_float4(static_cast<float>(t.v[c]) / t.w, static_cast<float>(t.v[c + 1]) / t.w,
                     static_cast<float>(t.v[c + 2]) / t.w, 1.0f);
}

// Roughness 0 (PreFilterEnvMap.comp:139-161 with a = 0): every half vector
// is N, so every kept sample is the mirror lookup at N, LOD 0, and the
// NdotL-weighted mean is that one lookup.  It reads the full texel contrast
// of the source, so it is addressed in df32 from the texel's exact lattice
// direction (yaw and pitch do not depend on the direction's length); the pole
// branch (|xz| <= 0.001 of the unit direction, PreFilterEnvMap.comp:104-112)
// is decided in FP32 as the sampled path decides it.
template <class LevelOf>
__device__ __forceinline__ float4 prefilter_texel_mirror(const char* __restrict__ pyr, const LevelOf& level, int face,
                                                         int x, int y, int S) {
  const f3 raw = cube_texel_raw_dir(face, x, y, S);
  const f3 n = normalize(raw);
  const float len_xz = sqrtf(fmaf(n.x, n.x, n.z * n.z));
  const int pole = len_xz > 0.001f ? 0 : (n.y > 0.0f ? 1 : -1);
  const LevelC& c = level(0);
  df32 tx, ty;
  equirect_coords_df(df3{df_of(raw.x), df_of(raw.y), df_of(raw.z)}, static_cast<int>(c.wmask + 1),
                     static_cast<int>(c.hmask + 1), pole, tx, ty);
  const f3 v = level_bilinear_df(pyr, c, tx, ty);
  return make_float4(v.x, v.y, v.z, 1.0f);
}

// ------------------------------------------------------------ block of work
// What the blocks of one map share.
struct PrefilterMap {
  const char* pyr;
  float4* cube;            // [mip][face][y][x]
  const GgxEntry* tables;  // [mip][samples]
  const int* counts;
  const double* wsum;
  const LevelC* lv;         // source pyramid levels
  const StagedLevel* slv;   // levels from `first` on, as staged in LDS
  int first, levels;
  int size, mips, samples;
  int split;  // chunks of a rough mip's table, a power of two
  int chunk;  // table entries per chunk, a multiple of kBlockSums
  int waves;  // waves per tile of a rough mip: split, or half of it
  int alone;  // texels by themselves (prefilter_alone)
};

constexpr int kPrefilterMaxSplit = 16;
constexpr int kPrefilterPart = 6 * 64 + 1;  // sums of a chunk: a tile's six (or three), the weight

// LDS texels of levels first..levels - 1, block-cooperative; the caller
// synchronises the block.
template <int kWaves>
__device__ __forceinline__ void stage_levels(const char* __restrict__ pyr, const LevelC* __restrict__ lv,
                                             const StagedLevel* __restrict__ slv, int first, int levels, char* lds) {
  for (int l = first; l < levels; ++l) {
    const LevelC& c = lv[l];
    const int w = static_cast<int>(c.wmask) + 1, h = static_cast<int>(c.hmask) + 1;
    const float4* src = reinterpret_cast<const float4*>(pyr) + c.off;
    float* dst = reinterpret_cast<float*>(lds + slv[l].off);
    const int n = (w + 2) * (h + 2);
    for (int i = threadIdx.x; i < n; i += 64 * kWaves) {
      const int r = i / (w + 2), col = i - r * (w + 2);
      const float4 v = src[((static_cast<uint32_t>(r - 1) & c.hmask) << c.wshift) +
                           (static_cast<uint32_t>(col - 1) & c.wmask)];
      dst[3 * i] = v.x, dst[3 * i + 1] = v.y, dst[3 * i + 2] = v.z;
    }
  }
}

// Units of a rough mip: the tiles of +X (turn about y) and +Y (about x), and
// those of +Z once for either turn, a unit's lanes of the other turn idle.  The
// Z tiles off the diagonals have one turn; their other unit ends at once.
constexpr int kPairUnits = 4;

// Blocks of mip m: a wave per tile of a roughness-0 mip (all six faces),
// `waves` waves per unit of a rough one (of texels alone: per tile).
__host__ __device__ inline int prefilter_blocks(int size, int mips, int m, int waves, bool alone,
                                                int tw, int th, int block_waves) {
  const int S = size >> m > 1 ? size >> m : 1;
  const int tiles = ((S + tw - 1) / tw) * ((S + th - 1) / th);
  const bool mirror = m == 0 || mips == 1;
  const int per = mirror ? block_waves : block_waves / waves;
  return ((mirror || alone ? 6 : kPairUnits) * tiles + per - 1) / per;
}

// One block of mip m, the levels staged by the caller.  A rough mip's table is
// cut into `split` chunks, one for each of the tile's waves or (kTwoChunks,
// where the block has half as many waves as the table has chunks) two; the
// chunks' partials are added in chunk order, so the bits are the same.
//
// Bound: VALU (the nominal issue rate, one wave instruction a SIMD per 4 cycles,
// is reached).  A sample costs a pair of texels about 160 VALU (66 for the shared
// direction and angles; 173 over the launch) and 24 ds_read2_b32; one texel
// alone, gathering from global memory, took 115 VALU and eight gathers at 16
// cycles of the texture data return, which was 98 % busy.  2048 x 1024 source to
// 512^2 x 6 mips at 1024 samples: 1.83 ms -> 0.95.  Measured beside it: 48-byte
// records of a cell's four texels in global memory (three gathers a lookup) 2.7
// ms, the records of neighbouring lanes spreading over more lines than their
// texels.
template <bool kF64Sums, int kTW, int kTH, int kWaves, bool kTogether, bool kTwoChunks, bool kSingle>
__device__ __forceinline__ void prefilter_block(const PrefilterMap& p, int m, int block, char* lds) {
  static_assert(kTW * kTH == 64, "one wave per tile");
  constexpr int kN = kSingle ? 3 : 6;
  using Sums = PrefilterSums<kF64Sums, kN>;
  using T = typename Sums::T;
  const int S = max(1, p.size >> m);
  const int tpr = (S + kTW - 1) / kTW, tiles = tpr * ((S + kTH - 1) / kTH);
  const int wave = static_cast<int>(threadIdx.x >> 6), lane = static_cast<int>(threadIdx.x & 63);
  const bool mirror = m == 0 || p.mips == 1;  // roughness m / (mips - 1) == 0 (block-uniform)
  const int waves = mirror ? 1 : p.waves;
  const int local = (block * kWaves + wave) / waves;
  const int lt = min(local, (mirror || kSingle ? 6 : kPairUnits) * tiles - 1);
  const int f = lt / tiles, t = lt - f * tiles;
  const int x = (t % tpr) * kTW + (lane % kTW);
  const int y = (t / tpr) * kTH + (lane / kTW);
  const bool active = local == lt && x < S && y < S;
  const int xc = min(x, S - 1), yc = min(y, S - 1);
  float4* out = p.cube;
  for (int k = 0; k < m; ++k) {
    const size_t s = static_cast<size_t>(max(1, p.size >> k));
    out += 6 * s * s;
  }
  if (mirror) {
    const auto level = [&](int l) -> const LevelC& { return p.lv[l]; };
    const float4 v = prefilter_texel_mirror(p.pyr, level, f, xc, yc, S);
    if (active) out[(static_cast<size_t>(f) * S + y) * S + x] = v;
    return;
  }
  const int face = kSingle ? f : 2 * min(f, 2);
  const bool turn_y = (f & 1) == 0;
  const f3 raw = cube_texel_raw_dir(face, xc, yc, S);
  const Frame fr = local_to_world(raw);
  const bool mine = kSingle || (fabsf(raw.x) > fabsf(raw.y)) == turn_y;
  const bool any = __builtin_amdgcn_ballot_w64(mine) != 0;  // the same for every wave of the unit
  const int count = p.counts[m], part = __builtin_amdgcn_readfirstlane(wave & (waves - 1));
  const StagedAcc<kTogether> acc{lds, p.slv, p.pyr, p.lv, p.first};
  const GgxEntry* tab = p.tables + static_cast<size_t>(m) * p.samples;
  Sums tot, first;
  for (int k = part;;) {
    const int lo = min(count, k * min(p.chunk, count)), hi = any ? min(count, lo + min(p.chunk, count)) : lo;
    if constexpr (kSingle)
      tot = prefilter_pair_range<kF64Sums, kAlone, kN>(acc, tab, lo, hi, fr);
    else if (turn_y)
      tot = prefilter_pair_range<kF64Sums, kTurnY, kN>(acc, tab, lo, hi, fr);
    else
      tot = prefilter_pair_range<kF64Sums, kTurnX, kN>(acc, tab, lo, hi, fr);
    if (!kTwoChunks || (k += waves) >= p.split) break;
    first = tot;
  }
  if (p.split > 1) {
    // The partials take the staged texels' place.
    T* s_part = reinterpret_cast<T*>(lds) + static_cast<size_t>(wave / waves) * p.split * kPrefilterPart;
    const auto store = [&](int k, const Sums& t) {
#pragma unroll
      for (int c = 0; c < kN; ++c) s_part[k * kPrefilterPart + 64 * c + lane] = t.v[c];
      if (lane == 0) s_part[k * kPrefilterPart + 6 * 64] = static_cast<T>(t.w);
    };
    __syncthreads();
    if (kTwoChunks && p.split > waves) {
      store(part, first);
      store(part + waves, tot);
    } else {
      store(part, tot);
    }
    __syncthreads();
    if (part != 0) return;
    tot = Sums();
    for (int k = 0; k < p.split; ++k) {
#pragma unroll
      for (int c = 0; c < kN; ++c) tot.v[c] += s_part[k * kPrefilterPart + 64 * c + lane];
      tot.w += static_cast<float>(s_part[k * kPrefilterPart + 6 * 64]);
    }
  }
  if (!active || !mine) return;
  out[(static_cast<size_t>(face) * S + y) * S + x] = prefilter_value<kF64Sums>(tot, 0, p.wsum[m]);
  if (kSingle) return;
  int face2, x2, y2;
  pair_partner(face, x, y, S, turn_y, face2, x2, y2);
  out[(static_cast<size_t>(face2) * S + y2) * S + x2] = prefilter_value<kF64Sums>(tot, kSingle ? 0 : 1, p.wsum[m]);
}

}  // namespace althea
