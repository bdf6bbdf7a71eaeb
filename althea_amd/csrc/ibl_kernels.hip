// IBL precompute kernels for gfx950: Hammersley, the environment pyramid, the
// per-roughness GGX sample tables, the prefiltered cube, the irradiance cube,
// the split-sum BRDF LUT, point prefiltering and sampler probes.
//
// The GGX prefilter (Shaders/IBL_Precompute/PreFilterEnvMap.comp:126-177)
// evaluated at a cube texel with N = V = R has every per-sample quantity except
// the frame rotation independent of the texel: with h the local half vector,
// V.H = h.z, so L = frame * (2 h.z h.x, 2 h.z h.y, 2 h.z^2 - 1), NdotL = the z
// term and the source LOD depends on h.z only.  A one-block kernel per
// roughness builds these entries in FP64 (rounded once to FP32), drops samples
// with NdotL <= 0 in sample order, and sums the weights in FP64.  The texel
// kernel then reads one wave-uniform entry per sample (scalar loads), rotates
// it by its frame and filters the source in software.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <mutex>
#include <vector>

#include "device_math.hpp"
#include "internal.hpp"
#include "irradiance_launch.hpp"
#include "point_launch.hpp"
#include "precise_lookup.hpp"
#include "prefilter_common.hpp"

namespace althea {

// -------------------------------------------------------------- Hammersley
__global__ void hammersley_kernel(uint32_t n, uint32_t first, uint32_t count, uint32_t* __restrict__ bits,
                                  float2* __restrict__ xi) {
  uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= count) return;
  uint32_t i = first + k;
  if (bits) bits[k] = vdc_bits(i);
  if (xi) {
    float x1, x2;
    hammersley(i, n, x1, x2);
    xi[k] = make_float2(x1, x2);
  }
}

althea_status launch_hammersley(uint32_t n, uint32_t first, uint32_t count, uint32_t* bits, float* xi,
                                hipStream_t s) {
  if (count == 0) return ALTHEA_OK;
  dim3 grid((count + 255) / 256);
  hipLaunchKernelGGL(hammersley_kernel, grid, dim3(256), 0, s, n, first, count, bits,
                     reinterpret_cast<float2*>(xi));
  return check_launch("hammersley_kernel");
}

// ----------------------------------------------------------------- pyramid
// Level l = mean of the 2x2 (2x1 / 1x2 at unit extents) block of level l-1,
// the LINEAR half-size blit of Image::generateMipMaps (Src/Image.cpp:135-239).
//
// One pass reads a 32 x 32 tile of a level and writes its part of the next five
// (and, for level 0, the copy of the source), each formed in LDS from the one
// above, so a map takes two or three launches and its source is read once:
// 4096 x 2048 98 -> 66 us (4.8 TB/s of the source read and the pyramid written),
// 512 x 256 35 -> 12 us.  Bound: HBM on large sources, launches on small ones.
constexpr int kPyrTile = 32, kPyrSteps = 5;

static int pyramid_tiles(const PyramidJob& j, int level) {
  const int w = std::max(1, j.w >> level), h = std::max(1, j.h >> level);
  return ((w + kPyrTile - 1) / kPyrTile) * ((h + kPyrTile - 1) / kPyrTile);
}

__device__ __forceinline__ float4 pyramid_mean(const float4* p, int stride, int fx, int fy) {
  const float4 a = p[0];
  if (fx == 2 && fy == 2) {
    const float4 b = p[1], c = p[stride], d = p[stride + 1];
    return make_float4(((a.x + b.x) + (c.x + d.x)) * 0.25f, ((a.y + b.y) + (c.y + d.y)) * 0.25f,
                       ((a.z + b.z) + (c.z + d.z)) * 0.25f, ((a.w + b.w) + (c.w + d.w)) * 0.25f);
  }
  const float4 b = fx == 2 ? p[1] : p[stride];  // one of the extents is 1
  return make_float4((a.x + b.x) * 0.5f, (a.y + b.y) * 0.5f, (a.z + b.z) * 0.5f, (a.w + b.w) * 0.5f);
}

__device__ __forceinline__ void pyramid_tile(const PyramidJob& j, int level, int tile) {
  __shared__ float4 s_a[kPyrTile * kPyrTile], s_b[kPyrTile * kPyrTile / 4];
  int w = max(1, j.w >> level), h = max(1, j.h >> level);
  const int tiles_x = (w + kPyrTile - 1) / kPyrTile;
  // Extents are powers of two: a tile is whole, or the level's whole extent.
  int tw = min(w, kPyrTile), th = min(h, kPyrTile);
  int x0 = (tile % tiles_x) * tw, y0 = (tile / tiles_x) * th;
  const float4* src = level == 0 ? j.src : j.pyr + j.off[level];
  const bool copy = level == 0 && j.src != j.pyr;
  for (int i = threadIdx.x; i < tw * th; i += 256) {
    const size_t at = static_cast<size_t>(y0 + i / tw) * w + x0 + i % tw;
    const float4 v = src[at];
    s_a[i] = v;
    if (copy) j.pyr[at] = v;
  }
  float4 *from = s_a, *to = s_b;
  const int last = min(level + kPyrSteps, j.levels - 1);
  for (int l = level + 1; l <= last; ++l) {
    __syncthreads();
    const int nw = max(1, tw >> 1), nh = max(1, th >> 1);
    const int fx = tw > nw ? 2 : 1, fy = th > nh ? 2 : 1;
    w = max(1, w >> 1), h = max(1, h >> 1), x0 /= fx, y0 /= fy;
    float4* dst = j.pyr + j.off[l];
    for (int i = threadIdx.x; i < nw * nh; i += 256) {
      const int x = i % nw, y = i / nw;
      const float4 v = pyramid_mean(from + (y * fy) * tw + x * fx, tw, fx, fy);
      to[i] = v;
      dst[static_cast<size_t>(y0 + y) * w + x0 + x] = v;
    }
    tw = nw, th = nh;
    float4* t = from;
    from = to, to = t;
  }
}

__global__ __launch_bounds__(256) void pyramid_kernel(const PyramidJob job, int level) {
  pyramid_tile(job, level, blockIdx.x);
}

// The same pass for many maps: block b works on the last job whose first block
// of the pass is at most b.
__global__ __launch_bounds__(256) void pyramid_batch_kernel(const PyramidJob* __restrict__ jobs, int count, int pass) {
  const int b = blockIdx.x;
  int lo = 0, hi = count;
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (jobs[mid].first_block[pass] <= b)
      lo = mid;
    else
      hi = mid;
  }
  pyramid_tile(jobs[lo], pass * kPyrSteps, b - jobs[lo].first_block[pass]);
}

PyramidJob pyramid_job(const float* level0, int w, int h, float* pyr) {
  const PyramidGeometry g = pyramid_geometry(w, h);
  PyramidJob j{};
  j.src = reinterpret_cast<const float4*>(level0);
  j.pyr = reinterpret_cast<float4*>(pyr);
  j.w = w;
  j.h = h;
  j.levels = g.levels;
  for (int l = 0; l < g.levels; ++l) j.off[l] = g.off[l];
  return j;
}

// A pass is needed from level 0 (the copy) and from every fifth level that has
// one above it.
static bool pyramid_pass(const PyramidJob& j, int level) {
  return level + 1 < j.levels || (level == 0 && j.src != j.pyr);
}

althea_status launch_pyramid(const float* level0, int w, int h, float* pyr, hipStream_t s) {
  const PyramidJob j = pyramid_job(level0, w, h, pyr);
  for (int level = 0; pyramid_pass(j, level); level += kPyrSteps) {
    hipLaunchKernelGGL(pyramid_kernel, dim3(pyramid_tiles(j, level)), dim3(256), 0, s, j, level);
    const althea_status st = check_launch("pyramid_kernel");
    if (st != ALTHEA_OK) return st;
  }
  return ALTHEA_OK;
}

// Fills the jobs' first blocks; blocks[p] = the blocks of pass p.
void pyramid_schedule(std::vector<PyramidJob>& jobs, int blocks[kPyramidPasses]) {
  for (int p = 0; p < kPyramidPasses; ++p) {
    blocks[p] = 0;
    for (PyramidJob& j : jobs) {
      j.first_block[p] = blocks[p];
      if (pyramid_pass(j, p * kPyrSteps)) blocks[p] += pyramid_tiles(j, p * kPyrSteps);
    }
  }
}

althea_status launch_pyramid_batch(const PyramidJob* jobs, int count, const int blocks[kPyramidPasses], hipStream_t s) {
  for (int p = 0; p < kPyramidPasses; ++p) {
    if (blocks[p] == 0) continue;
    hipLaunchKernelGGL(pyramid_batch_kernel, dim3(blocks[p]), dim3(256), 0, s, jobs, count, p);
    const althea_status st = check_launch("pyramid_batch_kernel");
    if (st != ALTHEA_OK) return st;
  }
  return ALTHEA_OK;
}

// ------------------------------------------------------- GGX sample tables
// One block per roughness level.  Entry e (in sample order, NdotL > 0 only):
// L in the frame (T, B, N), and the source LOD clamped to the pyramid's
// [0, levels-1] split into (l0, l1 = min(l0+1, levels-1), delta).
// counts[m] = kept entries, wsum[m] = FP64 sum of L.n.  Kept entries are placed
// by a ballot per wave and the waves' counts.
struct TableParams {
  int samples;
  int mips;
  int env_levels;
  double sa_texel;  // 4 pi / (6 W H)  (PreFilterEnvMap.comp:158)
};

constexpr int kTableThreads = 1024;

__global__ __launch_bounds__(kTableThreads) void ggx_table_kernel(TableParams p, GgxEntry* __restrict__ tables,
                                                                  int* __restrict__ counts,
                                                                  double* __restrict__ wsum) {
  const int m = blockIdx.x;
  const int tid = threadIdx.x;
  const double rough = p.mips > 1 ? static_cast<double>(m) / (p.mips - 1) : 0.0;
  const double a2 = rough * rough;  // alpha = roughness (PreFilterEnvMap.comp:139-140)
  const double two_pi = 6.283185307179586476925;
  __shared__ int s_kept[kTableThreads / 64];
  __shared__ double s_sum[kTableThreads / 64];
  const int wave = tid >> 6, lane = tid & 63;
  int placed = 0;  // entries of the earlier chunks
  double my_sum = 0.0;
  GgxEntry* tab = tables + static_cast<size_t>(m) * p.samples;
  for (int chunk = 0; chunk < p.samples; chunk += kTableThreads) {
    int s = chunk + tid;
    bool keep = false;
    GgxEntry entry{};
    if (s < p.samples) {
      double x1 = static_cast<double>(s) / p.samples;
      double x2 = static_cast<double>(__builtin_bitreverse32(static_cast<uint32_t>(s))) * (1.0 / 4294967296.0);
      double den = 1.0 + (a2 - 1.0) * x2;
      double cos_t = sqrt((1.0 - x2) / den);
      double sin_t = sqrt(a2 * x2 / den);  // = sqrt(1 - cos_t^2) without cancellation
      double phi = two_pi * x1;
      double hx = cos(phi) * sin_t, hy = sin(phi) * sin_t, hz = cos_t;
      double lz = 2.0 * hz * hz - 1.0;
      if (lz > 0.0) {
        keep = true;
        double lod = 0.0;
        if (rough != 0.0) {
          double t = hz * hz * (a2 - 1.0) + 1.0;
          double D = a2 / (3.14159265358979323846 * t * t);
          double pdf = D * hz / (4.0 * hz + 0.00001);
          double sa_sample = 1.0 / (p.samples * pdf + 0.0001);
          lod = 0.5 * log2(sa_sample / p.sa_texel);
        }
        lod = fmin(fmax(lod, 0.0), static_cast<double>(p.env_levels - 1));
        // Rounded to FP32 as a sampler LOD would be, then split.
        const float lodf = static_cast<float>(lod);
        const float fl = floorf(lodf);
        entry.lx = static_cast<float>(2.0 * hz * hx);
        entry.ly = static_cast<float>(2.0 * hz * hy);
        entry.lz = static_cast<float>(lz);
        const double delta = static_cast<double>(lodf - fl);
        entry.l0 = static_cast<int>(fl);
        entry.l1 = min(entry.l0 + 1, p.env_levels - 1);
        entry.w0 = static_cast<float>(lz * (1.0 - delta));
        entry.w1 = static_cast<float>(lz * delta);
        entry.weight = static_cast<float>(lz);
        my_sum += lz;
      }
    }
    const uint64_t kept = __builtin_amdgcn_ballot_w64(keep);
    if (lane == 0) s_kept[wave] = __popcll(kept);
    __syncthreads();
    int at = placed, all = 0;
    for (int k = 0; k < kTableThreads / 64; ++k) {
      if (k < wave) at += s_kept[k];
      all += s_kept[k];
    }
    if (keep) tab[at + __popcll(kept & ((1ull << lane) - 1ull))] = entry;
    placed += all;
    __syncthreads();  // s_kept is read
  }
  my_sum = wave_sum_f64(my_sum);
  if (lane == 0) s_sum[wave] = my_sum;
  __syncthreads();
  if (tid == 0) {
    double sum = 0.0;
    for (int k = 0; k < kTableThreads / 64; ++k) sum += s_sum[k];
    counts[m] = placed;
    wsum[m] = sum;
    // Roughness 0 (alpha = 0): every half vector is N, so every kept sample
    // is L = N at LOD 0 with NdotL = 1 and the entries are bit-identical.  One
    // entry carrying their summed weight gives the same weighted mean (v * n /
    // n, exact for n <= 2^24) with one lookup instead of n.
    if (rough == 0.0 && placed > 1) {
      tab[0].weight = tab[0].w0 = static_cast<float>(placed);
      counts[m] = 1;
    }
  }
}

// ------------------------------------------------------------ prefilter
struct PrefilterParams {
  LevelC lv[kMaxLevels];
  StagedLevel slv[kMaxLevels];
  PrefilterMap map;  // lv and slv set by the kernel
  int block_start[kMaxLevels + 1];  // blocks before each mip
};

constexpr int kPrefilterTile = 8;

// 16 waves a block where a tile's table is cut into 16 chunks (few tiles: one
// block a CU, four waves a SIMD), else 8, held to six waves a SIMD (three
// blocks of at most 52 KB of LDS a CU, so one block's staging and last waves
// run beside another's samples): 512^2 x 6 cube 0.95 ms, against 1.09 at four
// waves a SIMD.
constexpr int kPrefilterWide = 16, kPrefilterNarrow = 8;

template <bool kF64Sums, int kWaves, bool kTogether, bool kSingle>
__device__ __forceinline__ void prefilter_cube(const PrefilterParams& p, float* s_levels) {
  const int b = blockIdx.x;
  int m = 0;
  while (m + 1 < p.map.mips && b >= p.block_start[m + 1]) ++m;
  PrefilterMap map = p.map;
  map.lv = p.lv;
  map.slv = p.slv;
  char* lds = reinterpret_cast<char*>(s_levels);
  if (m > 0) {
    stage_levels<kWaves>(map.pyr, map.lv, map.slv, map.first, map.levels, lds);
    __syncthreads();
  }
  prefilter_block<kF64Sums, kPrefilterTile, kPrefilterTile, kWaves, kTogether, false, kSingle>(
      map, m, b - p.block_start[m], lds);
}

template <bool kF64Sums>
__global__ __launch_bounds__(64 * kPrefilterWide) void prefilter_wide_kernel(const PrefilterParams p) {
  extern __shared__ float s_levels[];
  prefilter_cube<kF64Sums, kPrefilterWide, true, false>(p, s_levels);
}

template <bool kF64Sums>
__global__ __launch_bounds__(64 * kPrefilterNarrow) __attribute__((amdgpu_waves_per_eu(6))) void prefilter_cube_kernel(
    const PrefilterParams p) {
  extern __shared__ float s_levels[];
  prefilter_cube<kF64Sums, kPrefilterNarrow, false, false>(p, s_levels);
}

template <bool kF64Sums, int kWaves>
__global__ __launch_bounds__(64 * kWaves) __attribute__((amdgpu_waves_per_eu(4))) void prefilter_alone_kernel(
    const PrefilterParams p) {
  extern __shared__ float s_levels[];
  prefilter_cube<kF64Sums, kWaves, false, true>(p, s_levels);
}

// Pairs of 8 x 8 tiles of the rough mips.
static long long prefilter_pair_tiles(int size, int mips) {
  long long rough = 0;
  for (int m = 1; m < mips; ++m) {
    const int S = std::max(1, size >> m);
    const int tpf = (S + kPrefilterTile - 1) / kPrefilterTile;
    rough += 3ll * tpf * tpf;
  }
  return rough;
}

// Chunks of a rough mip's table: doubled while the pairs of tiles times the
// chunks stay under 4096 waves (to 16), or to 8 while they stay under 32 768
// (finer blocks level the last round, the roughest tiles having half the kept
// samples of the smoothest), as long as a chunk keeps 32 entries.  Chunks are
// multiples of the 32-entry FP32 blocks; one chunk is longer than any table.
// The batched kernel cuts each map's sums the same way.
int prefilter_split(int size, int mips, int samples, int& chunk) {
  const long long rough = prefilter_pair_tiles(size, mips);
  int k = 1;
  while (k < kPrefilterMaxSplit && rough > 0 && rough * k < (k < 8 ? 32768 : 4096) && samples / (2 * k) >= kBlockSums) k *= 2;
  chunk = k == 1 ? (1 << 30) : ((samples + k - 1) / k + kBlockSums - 1) / kBlockSums * kBlockSums;
  return k;
}

static size_t align256(size_t v) { return (v + 255) & ~static_cast<size_t>(255); }

void pyramid_levels(int w, int h, LevelC* out) {
  PyramidGeometry g = pyramid_geometry(w, h);
  for (int l = 0; l < g.levels; ++l) out[l] = make_level(g.w[l], g.h[l], g.off[l]);
}

// ------------------------------------------------------------ staged levels
// Source LOD of sample 0 (the half vector N) at a roughness, not clamped to the
// pyramid.
static double prefilter_lod(int w, int h, double rough, int samples) {
  const double a2 = rough * rough;
  const double pdf = 1.0 / (M_PI * a2 * (4.0 + 0.00001));
  const double sa_texel = 4.0 * M_PI / (6.0 * static_cast<double>(w) * h);
  return 0.5 * std::log2(1.0 / (samples * pdf + 0.0001) / sa_texel);
}

// The lowest source level the sample tables name: the source LOD grows with
// roughness and away from the lobe's centre, so it is that of sample 0 (the
// half vector N) at the lowest sampled roughness, 1 / (mips - 1); a margin of
// 1e-4 level covers the device's rounding.
int prefilter_first_level(int w, int h, int mips, int samples) {
  const double lod = prefilter_lod(w, h, mips > 1 ? 1.0 / (mips - 1) : 1.0, samples);
  return std::min(std::max(static_cast<int>(std::floor(lod - 1e-4)), 0), althea_env_levels(w, h) - 1);
}

// The levels of a map that a prefilter block stages in LDS: the coarsest ones,
// from `lowest` on, as many as kStagedMaxBytes holds (from 64 x 32 on for a
// 2:1 source, 38 KB; three blocks a CU).  At 1024 samples the lobes of roughness
// 1/4 and up read finer levels for a seventh of their samples or less, whatever
// the source's extent; staging 128 x 64 too (140 KB, one block a CU) measured
// 1.21 ms against 0.95 on the 512^2 x 6 cube.
constexpr size_t kStagedMaxBytes = 52 * 1024;

int staged_levels(int w, int h, int lowest, StagedLevel* out, size_t* bytes) {
  const PyramidGeometry g = pyramid_geometry(w, h);
  size_t total = 0;
  int first = g.levels;
  while (first > lowest) {
    const size_t level = 12 * static_cast<size_t>(g.w[first - 1] + 2) * (g.h[first - 1] + 2);
    if (total + level > kStagedMaxBytes) break;
    --first;
    out[first] = make_staged_level(g.w[first], g.h[first], static_cast<uint32_t>(total));
    total += level;
  }
  *bytes = total;
  return first;
}

// Whether a call's texels are summed by themselves instead of in pairs.  Where the
// samples' levels are mostly finer than the staged ones, the lines that the
// lookups touch in global memory bound a CU, as many for a pair as for two texels,
// and the pairs' half as many blocks leave CUs idle.  The measure is the level of
// sample 0 at roughness 1 against the first staged level.  Us a cube, pairs and
// alone (texels gathered from a padded copy of the pyramid took the third):
//   512 x 256 source,  32^2 x 6, 5 mips,  32 768 samples (0.7 finer)  8 121  4 027  5 761
//   512 x 256,         64^2, 4 mips,     131 072 (1.7)               32 188 15 606 20 949
//   64 x 1024,         64^2, 4 mips,       4 096 (-0.3)                 764    374    616
//   64 x 1024,        128^2, 5 mips,       8 192 (0.2)                2 674  1 979  2 331
//   64 x 1024,        512^2, 4 mips,       4 096 (-0.3)               5 059  4 794  6 955
//   512 x 512,        512^2, 4 mips,       4 096 (-0.3)               4 217  4 374  6 634
//   16 x 2048,        256^2, 6 mips,       8 192 (0.7)               10 000  9 156  8 334
bool prefilter_alone(int w, int h, int size, int mips, int samples) {
  StagedLevel staged[kMaxLevels];
  size_t bytes = 0;
  const int first = staged_levels(w, h, 0, staged, &bytes);
  if (mips < 2 || first == 0) return false;
  const double finer = first - std::max(prefilter_lod(w, h, 1.0, samples), 0.0);
  return finer > 0.0 || (finer > -0.5 && prefilter_pair_tiles(size, mips) < 256);
}

size_t prefilter_lds_bytes(size_t staged, int split, int waves, int block_waves) {
  return std::max(staged, split > 1 ? sizeof(double) * kPrefilterPart * split * (block_waves / waves) : size_t{0});
}

// ------------------------------------------------------ split gather copy
// Levels first..last of a pyramid, each padded with its REPEAT neighbours
// ((w + 2) x (h + 2) texels, SplitLevel), concatenated from texel 0.
struct GatherGeometry {
  int first, last;
  uint32_t off[kMaxLevels];
  size_t texels;
};
static GatherGeometry gather_geometry(int w, int h, int first, int last) {
  const PyramidGeometry g = pyramid_geometry(w, h);
  GatherGeometry out{};
  out.first = first;
  out.last = last;
  size_t total = 0;
  for (int l = first; l <= last; ++l) {
    out.off[l] = static_cast<uint32_t>(total);
    total += static_cast<size_t>(g.w[l] + 2) * (g.h[l] + 2);
  }
  out.texels = total;
  return out;
}

struct PadParams {
  int first, last;
  int w[kMaxLevels], h[kMaxLevels];
  uint32_t src[kMaxLevels];      // pyramid texel offset of each level
  uint32_t dst[kMaxLevels + 1];  // gather texel offset of each level; dst[last + 1] = total
};

// Texels of a split gather copy's RG plane (the B plane starts 8 times this
// many bytes in): the total rounded up to 64, so both planes start 256-byte
// aligned.
static size_t split_plane_texels(const GatherGeometry& gg) { return (gg.texels + 63) & ~static_cast<size_t>(63); }

static size_t split_gather_bytes(int w, int h, int first, int last) {
  if (w <= 0 || h <= 0) return 0;
  return 12 * split_plane_texels(gather_geometry(w, h, first, last));
}

static SplitLevel split_level(int w, int h, const GatherGeometry& gg, int l) {
  const PyramidGeometry g = pyramid_geometry(w, h);
  const LevelC c = make_level(g.w[l], g.h[l], 0);
  SplitLevel s{};
  s.kx = c.kx;
  s.cx = c.cx;
  s.ky = c.ky;
  s.cy = c.cy;
  s.rowbytes = static_cast<uint32_t>(g.w[l] + 2) * 8u;
  s.rg = 8u * gg.off[l];
  s.b = static_cast<uint32_t>(8 * split_plane_texels(gg)) + 4u * gg.off[l];
  return s;
}

// One thread per padded texel: padded (r, c) of level l is the pyramid texel
// ((r - 1) mod h, (c - 1) mod w), into the RG and B planes (plane_texels apart).
__global__ __launch_bounds__(256) void gather_pad_kernel(const float4* __restrict__ pyr, const PadParams p,
                                                         float2* __restrict__ rg, size_t plane_texels) {
  const uint32_t i = blockIdx.x * 256u + threadIdx.x;
  if (i >= p.dst[p.last + 1]) return;
  int l = p.first;
  while (l < p.last && i >= p.dst[l + 1]) ++l;
  const int w = p.w[l], h = p.h[l];
  const uint32_t k = i - p.dst[l];
  const int r = static_cast<int>(k / static_cast<uint32_t>(w + 2));
  const int c = static_cast<int>(k) - r * (w + 2);
  const int sr = r == 0 ? h - 1 : (r == h + 1 ? 0 : r - 1);
  const int sc = c == 0 ? w - 1 : (c == w + 1 ? 0 : c - 1);
  const float4 v = pyr[p.src[l] + static_cast<size_t>(sr) * w + sc];
  rg[i] = make_float2(v.x, v.y);
  reinterpret_cast<float*>(rg + plane_texels)[i] = v.z;
}

static althea_status launch_split_gather(const float* pyr, int w, int h, const GatherGeometry& gg, float* gpyr,
                                         hipStream_t s) {
  const PyramidGeometry g = pyramid_geometry(w, h);
  PadParams p{};
  p.first = gg.first;
  p.last = gg.last;
  for (int l = gg.first; l <= gg.last; ++l) {
    p.w[l] = g.w[l];
    p.h[l] = g.h[l];
    p.src[l] = g.off[l];
    p.dst[l] = gg.off[l];
  }
  p.dst[gg.last + 1] = static_cast<uint32_t>(gg.texels);
  const uint32_t blocks = static_cast<uint32_t>((gg.texels + 255) / 256);
  hipLaunchKernelGGL(gather_pad_kernel, dim3(blocks), dim3(256), 0, s, reinterpret_cast<const float4*>(pyr), p,
                     reinterpret_cast<float2*>(gpyr), split_plane_texels(gg));
  return check_launch("gather_pad_kernel");
}

static CubeMips cube_mips_of(int size, int mips) {
  CubeMips c{};
  c.size = size;
  c.mips = mips;
  for (int m = 0; m < mips; ++m) c.off[m] = static_cast<uint32_t>(cube_mip_offset(size, m));
  return c;
}


althea_status launch_ggx_tables(int samples, int mips, int env_w, int env_h, GgxEntry* tables, int* counts,
                                double* wsum, hipStream_t s) {
  TableParams tp;
  tp.samples = samples;
  tp.mips = mips;
  tp.env_levels = althea_env_levels(env_w, env_h);
  tp.sa_texel = 4.0 * M_PI / (6.0 * static_cast<double>(env_w) * env_h);
  hipLaunchKernelGGL(ggx_table_kernel, dim3(mips), dim3(kTableThreads), 0, s, tp, tables, counts, wsum);
  return check_launch("ggx_table_kernel");
}

// Entries, counts and weight sums (and a part that no kernel reads: the size is
// the one the allocation-free entry point's limit has always been stated in).
size_t prefilter_table_bytes(int mips, int samples) {
  return align256(sizeof(GgxEntry) * static_cast<size_t>(mips) * samples) + align256(sizeof(int) * mips) +
         align256(sizeof(double) * mips) + align256(sizeof(float) * mips);
}

// The sample tables.
size_t prefilter_workspace_bytes(int, int, int, int mips, int samples) { return prefilter_table_bytes(mips, samples); }

// ------------------------------------------- allocation-free prefilter
// The sample tables of althea_prefilter_cube_noalloc: a fixed device array,
// one copy per GPU, held until the process ends.  In host code `scratch`
// names a host-side stand-in, so its device address is looked up once per
// device with hipGetSymbolAddress and only that address is handed to kernels.
static_assert(ALTHEA_PREFILTER_SCRATCH_MAX_BYTES % 256 == 0, "scratch size");
static __device__ __align__(256) unsigned char scratch[ALTHEA_PREFILTER_SCRATCH_MAX_BYTES];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mutex;
void* g_scratch_ptr[kMaxDevices] = {};
}  // namespace

// Device address of `scratch` on the current device.
static althea_status prefilter_scratch(void** out) {
  int dev = 0;
  ALTHEA_TRY_HIP(hipGetDevice(&dev));
  if (dev < 0 || dev >= kMaxDevices) {
    set_error("prefilter_cube_noalloc: device %d beyond the %d supported", dev, kMaxDevices);
    return ALTHEA_ERROR_UNSUPPORTED;
  }
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (!g_scratch_ptr[dev]) {
    void* ptr = nullptr;
    ALTHEA_TRY_HIP(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
    g_scratch_ptr[dev] = ptr;
  }
  *out = g_scratch_ptr[dev];
  return ALTHEA_OK;
}

// Every table entry, count and weight sum the prefilter reads is written by
// the table kernel of the same call before the texel kernel runs, so nothing
// left in the array by an earlier call is read and nothing needs clearing.
althea_status launch_prefilter_cube_noalloc(const float* pyr, int env_w, int env_h, int size, int mips,
                                            int samples, unsigned flags, float* cube, hipStream_t s) {
  void* ws = nullptr;
  althea_status st = prefilter_scratch(&ws);
  if (st != ALTHEA_OK) return st;
  return launch_prefilter_cube(pyr, env_w, env_h, size, mips, samples, flags, cube, ws, s);
}

althea_status launch_prefilter_cube(const float* pyr, int env_w, int env_h, int size, int mips, int samples,
                                    unsigned flags, float* cube, void* workspace, hipStream_t s) {
  char* ws = static_cast<char*>(workspace);
  GgxEntry* tables = reinterpret_cast<GgxEntry*>(ws);
  ws += align256(sizeof(GgxEntry) * static_cast<size_t>(mips) * samples);
  int* counts = reinterpret_cast<int*>(ws);
  ws += align256(sizeof(int) * mips);
  double* wsum = reinterpret_cast<double*>(ws);

  althea_status st = launch_ggx_tables(samples, mips, env_w, env_h, tables, counts, wsum, s);
  if (st != ALTHEA_OK) return st;

  PrefilterParams p{};
  pyramid_levels(env_w, env_h, p.lv);
  size_t staged = 0;
  p.map.first = staged_levels(env_w, env_h, prefilter_first_level(env_w, env_h, mips, samples), p.slv, &staged);
  p.map.levels = althea_env_levels(env_w, env_h);
  p.map.pyr = reinterpret_cast<const char*>(pyr);
  p.map.cube = reinterpret_cast<float4*>(cube);
  p.map.tables = tables;
  p.map.counts = counts;
  p.map.wsum = wsum;
  p.map.size = size;
  p.map.mips = mips;
  p.map.samples = samples;
  p.map.split = p.map.waves = prefilter_split(size, mips, samples, p.map.chunk);
  p.map.alone = prefilter_alone(env_w, env_h, size, mips, samples) ? 1 : 0;
  const bool wide = p.map.waves > kPrefilterNarrow;
  const int waves = wide ? kPrefilterWide : kPrefilterNarrow;
  for (int m = 0; m < mips; ++m)
    p.block_start[m + 1] = p.block_start[m] + prefilter_blocks(size, mips, m, p.map.waves, p.map.alone, kPrefilterTile,
                                                               kPrefilterTile, waves);
  const int variant = (flags & ALTHEA_PRECOMPUTE_FP32_SUMS ? 0 : 1) | (wide ? 2 : 0) | (p.map.alone ? 4 : 0);
  auto kernel = variant == 0   ? prefilter_cube_kernel<false>
                : variant == 1 ? prefilter_cube_kernel<true>
                : variant == 2 ? prefilter_wide_kernel<false>
                : variant == 3 ? prefilter_wide_kernel<true>
                : variant == 4 ? prefilter_alone_kernel<false, kPrefilterNarrow>
                : variant == 5 ? prefilter_alone_kernel<true, kPrefilterNarrow>
                : variant == 6 ? prefilter_alone_kernel<false, kPrefilterWide>
                               : prefilter_alone_kernel<true, kPrefilterWide>;
  hipLaunchKernelGGL(kernel, dim3(p.block_start[mips]), dim3(64 * waves),
                     mips > 1 ? prefilter_lds_bytes(staged, p.map.split, p.map.waves, waves) : 0, s, p);
  return check_launch("prefilter_cube_kernel");
}

// -------------------------------------------------------- point prefilter
// Same estimator at a query's (direction, roughness r).  kLanes lanes of a wave
// take a query, each its samples: lane l takes samples l C + t, t = 0..C - 1
// (C = n / kLanes rounded up), so with C a power of two the lanes of a step have
// radical inverses within 1 / C: nearly one source LOD, spread around a ring of
// the lobe, and with the whole wave on a query the steps outside the hemisphere
// are skipped whole.  point_lanes says which kLanes a call takes.
//
// With x2 the radical inverse and den = 1 + (r^2 - 1) x2, the GGX half vector
// has cos^2 = (1 - x2) / den and sin^2 = r^2 x2 / den, so L in the frame is
//   (r q cos phi, r q sin phi, 1 - (1 + r^2) x2) / den, q = 2 sqrt(x2 (1 - x2)),
// whose r-free parts are a table of the sample set, and D = den^2 / (pi r^2):
// one reciprocal a sample, no square root.  pdf = D cos / (4 cos + 1e-5)
// (PreFilterEnvMap.comp:155-161) takes D (1/4 - 1e-5 / (16 cos)) with 1 / cos =
// 1.415 - 0.425 L.z on the kept range, off by up to 0.05: 1.3e-7 of the pdf.
//
// Bound: VALU (about 140 a step with the wave on a query, 0.93 of the nominal
// issue rate).  One lane per query walked its samples alone, 250 VALU each with
// IEEE roots and quotients, its lookups unrelated to its neighbours': 2^18 queries
// of 1024 samples from 1024 x 512, 2.06 ms, here 0.91; 1 394 queries of 605
// samples, 598 us (a wave's latency of all samples), here 18.  The error against
// 64 bits went from 2.1e-5 (sin and cos of theta by FP32 roots) to 4.8e-7.
struct PointParams {
  LevelC lv[kMaxLevels];
  StagedLevel slv[kMaxLevels];
  const char* pyr;
  int first, levels;
  int samples, steps;  // steps = ceil(samples / kLanes)
  int count;
  int level_off, table_off;  // byte offsets in LDS of the level records and the sample table
  float log2_sa_texel;
};

// A level's constants as a lane reads them from LDS (its levels are its own).
struct PointLevel {
  float kx, cx, ky, cy;
  uint32_t rowbytes, off;          // staged
  uint32_t wmask, hmask;
  uint32_t wshift, src, pad0, pad1;  // pyramid texel offset
};

// Sample i of n: (q cos phi, q sin phi, x2); x2 = 2 beyond the set (never kept).
__device__ __forceinline__ f3 point_sample(int i, int n) {
  if (i >= n) return mk(0.0f, 0.0f, 2.0f);
  float x1, x2, sp, cp;
  hammersley(static_cast<uint32_t>(i), static_cast<uint32_t>(n), x1, x2);
  sincospif(2.0f * x1, &sp, &cp);
  const float q = 2.0f * sqrtf(x2 * (1.0f - x2));
  return mk(q * cp, q * sp, x2);
}

// Adds w times the bilinear value of level l at (yaw, pitch).
__device__ __forceinline__ void point_lookup(const char* __restrict__ pyr, const char* lds, const PointLevel& g,
                                             bool staged, float yaw, float pitch, float w, float s[3]) {
  const TexelCoord q = texel_coord(g, yaw, pitch);
  LevelTaps t;
  if (staged) {
    // off + (iy + 1) rowbytes + (ix + 1) 12
    const uint32_t o = g.off + static_cast<uint32_t>(__mul24(q.iy + 1, static_cast<int>(g.rowbytes)) + 12 * (q.ix + 1));
    StagedLevel sl{};
    sl.rowbytes = g.rowbytes;
    staged_texels(lds, sl, o, t);
  } else {
    LevelC c{};
    c.wmask = g.wmask;
    c.hmask = g.hmask;
    c.wshift = g.wshift;
    level_texels(pyr + (static_cast<size_t>(g.src) << 4), c, q.ix, q.iy, t);
  }
  taps_acc(t, tap_weights(q.ax, q.ay, w), s[0], s[1], s[2]);
}

constexpr int kPointWaves = 8;
constexpr int kPointBlocks = 768;  // three a CU walk the queries: the staging and the table are per block
constexpr int kPointTableMax = 2048;  // samples whose table stays in LDS (24 KB)

template <int kLanes, bool kTable>
__global__ __launch_bounds__(64 * kPointWaves) void prefilter_points_kernel(const PointParams p,
                                                                            const float4* __restrict__ dir_rough,
                                                                            float* __restrict__ out) {
  constexpr int kQueries = 64 / kLanes;
  extern __shared__ float s_levels[];
  char* lds = reinterpret_cast<char*>(s_levels);
  PointLevel* levels = reinterpret_cast<PointLevel*>(lds + p.level_off);
  float* table = reinterpret_cast<float*>(lds + p.table_off);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  stage_levels<kPointWaves>(p.pyr, p.lv, p.slv, p.first, p.levels, lds);
  if (static_cast<int>(threadIdx.x) < p.levels) {
    const LevelC& c = p.lv[threadIdx.x];
    const StagedLevel& g = p.slv[threadIdx.x];
    levels[threadIdx.x] = PointLevel{c.kx, c.cx, c.ky, c.cy, g.rowbytes, g.off, c.wmask, c.hmask, c.wshift, c.off, 0, 0};
  }
  if (kTable) {
    // Step t's lanes side by side.
    for (int i = threadIdx.x; i < kLanes * p.steps; i += 64 * kPointWaves) {
      const f3 v = point_sample(i % kLanes * p.steps + i / kLanes, p.samples);
      table[3 * i] = v.x, table[3 * i + 1] = v.y, table[3 * i + 2] = v.z;
    }
  }
  __syncthreads();
  const float max_lod = static_cast<float>(p.levels - 1);
  const float half_sa = -0.5f * p.log2_sa_texel;
  const int sub = lane % kLanes;
  const size_t count = static_cast<size_t>(p.count);
  const PointWalk walk = point_walk(blockIdx.x, gridDim.x, wave, kPointWaves, kQueries);
  for (size_t base = walk.first; base < count; base += walk.stride) {
    const size_t query = base + lane / kLanes;  // lanes past the count repeat the last query
    const float4 q = dir_rough[query < count ? query : count - 1];
    const Frame fr = local_to_world(mk(q.x, q.y, q.z));
    const float rough = fabsf(q.w), a2 = rough * rough, a2m1 = a2 - 1.0f, a2p1 = a2 + 1.0f;
    const float kd = static_cast<float>(p.samples) * kInvPi / a2;  // n D = kd den^2
    double ar = 0.0, ag = 0.0, ab = 0.0, aw = 0.0;
    float s[3] = {0.0f, 0.0f, 0.0f}, sw = 0.0f;
    for (int t = 0; t < p.steps; ++t) {
      f3 e;
      if (kTable) {
        const float* v = table + 3 * (kLanes * t + sub);
        e = mk(v[0], v[1], v[2]);
      } else {
        e = point_sample(sub * p.steps + t, p.samples);
      }
      const float num = fmaf(-e.z, a2p1, 1.0f);
      if (num > 0.0f) {
        const float den = fmaf(e.z, a2m1, 1.0f);
        const float rden = rcp_fast(den);
        const float lz = num * rden, k = rough * rden;
        const float lx = e.x * k, ly = e.y * k;
        float lod = 0.0f;
        if (rough != 0.0f) {
          const float f = fmaf(lz, 2.65625e-7f, 0.249999116f);
          lod = fmaf(__builtin_amdgcn_logf(fmaf(den * den * f, kd, 0.0001f)), -0.5f, half_sa);
        }
        lod = fminf(fmaxf(lod, 0.0f), max_lod);
        const float fl = floorf(lod), delta = lod - fl;
        const int l0 = static_cast<int>(fl);
        const f3 L = mk(fmaf(fr.t.x, lx, fmaf(fr.b.x, ly, fr.n.x * lz)), fmaf(fr.t.y, lx, fmaf(fr.b.y, ly, fr.n.y * lz)),
                        fmaf(fr.t.z, lx, fmaf(fr.b.z, ly, fr.n.z * lz)));
        float yaw, pitch;
        equirect_angles(L, yaw, pitch);
        point_lookup(p.pyr, lds, levels[l0], l0 >= p.first, yaw, pitch, fmaf(-delta, lz, lz), s);
        if (delta != 0.0f) {
          const int l1 = min(l0 + 1, p.levels - 1);
          point_lookup(p.pyr, lds, levels[l1], l1 >= p.first, yaw, pitch, delta * lz, s);
        }
        sw += lz;
      }
      if ((t & (kBlockSums - 1)) == kBlockSums - 1) {
        ar += s[0], ag += s[1], ab += s[2], aw += sw;
        s[0] = s[1] = s[2] = sw = 0.0f;
      }
    }
    ar += s[0], ag += s[1], ab += s[2], aw += sw;
    if constexpr (kLanes == 1) {
      if (query < count)
        reinterpret_cast<float4*>(out)[query] = make_float4(static_cast<float>(ar / aw), static_cast<float>(ag / aw),
                                                            static_cast<float>(ab / aw), 1.0f);
    } else {
      // Four sums over the query's lanes: halves exchange two sums, quarters
      // one, then one value is summed over a quarter (first r, then g, b, w).
      constexpr int kHalf = kLanes / 2, kQuarter = kLanes / 4;
      const bool hi = lane & kHalf, hi2 = lane & kQuarter;
      double k0 = hi ? ab : ar, k1 = hi ? aw : ag;
      k0 += __shfl_xor(hi ? ar : ab, kHalf, 64);
      k1 += __shfl_xor(hi ? ag : aw, kHalf, 64);
      double v = hi2 ? k1 : k0;
      v += __shfl_xor(hi2 ? k0 : k1, kQuarter, 64);
#pragma unroll
      for (int o = kQuarter / 2; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
      const double w = __shfl(v, lane | kHalf | kQuarter, 64);
      const int component = sub / kQuarter;
      if (sub % kQuarter == 0 && query < count)
        out[4 * query + component] = component == 3 ? 1.0f : static_cast<float>(v / w);
    }
  }
}

althea_status launch_prefilter_points(const float* pyr, int env_w, int env_h, int samples, const float* dir_rough,
                                      int count, float* out, void*, hipStream_t s) {
  if (count == 0) return ALTHEA_OK;
  PointParams p{};
  pyramid_levels(env_w, env_h, p.lv);
  const bool table = samples <= kPointTableMax;
  const int lanes = point_lanes(samples, count);
  size_t staged = 0;
  p.levels = althea_env_levels(env_w, env_h);
  p.first = p.levels;
  if (point_stages(samples, lanes)) p.first = staged_levels(env_w, env_h, 0, p.slv, &staged);
  p.pyr = reinterpret_cast<const char*>(pyr);
  p.samples = samples;
  p.steps = (samples + lanes - 1) / lanes;
  p.count = count;
  p.level_off = static_cast<int>((staged + 15) & ~size_t{15});
  p.table_off = p.level_off + static_cast<int>(sizeof(PointLevel)) * kMaxLevels;
  p.log2_sa_texel = static_cast<float>(std::log2(4.0 * M_PI / (6.0 * static_cast<double>(env_w) * env_h)));
  const size_t lds = p.table_off + (table ? sizeof(float) * 3 * lanes * p.steps : size_t{0});
  auto kernel = !table        ? prefilter_points_kernel<64, false>
                : lanes == 1  ? prefilter_points_kernel<1, true>
                : lanes == 4  ? prefilter_points_kernel<4, true>
                : lanes == 16 ? prefilter_points_kernel<16, true>
                              : prefilter_points_kernel<64, true>;
  hipLaunchKernelGGL(kernel, dim3(point_blocks(count, kPointWaves, 64 / lanes, kPointBlocks)), dim3(64 * kPointWaves), lds, s,
                     p, reinterpret_cast<const float4*>(dir_rough), out);
  return check_launch("prefilter_points_kernel");
}

// ------------------------------------------------------------ irradiance
// GenIrradianceMap.comp:106-155 per cube texel: the Riemann sum over
// theta_samples azimuths x phi_samples polar angles of radiance(d) cos sin,
// read at the fixed source LOD log2(W / theta_samples), times
// pi / (theta_samples phi_samples).  An even azimuth count over a source
// whose level is at least 8 x 4 takes the folded kernel below; the kernel
// here, one wave per texel, serves odd azimuth counts, smaller levels, few
// samples (kFoldMinSteps), and two levels that are not an exact halving.
struct IrradianceParams {
  SplitLevel lv0, lv1;  // the two source levels around LOD log2(W / theta_samples), split gather copies
  SplitLevel grid;      // their blend grid (blend)
  int blend;
  int levels;
  int size;
  int theta_samples;
  int phi_samples;
  int l0, l1;
  float delta;
  double scale;  // pi / theta_samples / phi_samples
};

// phi_tab[j] = (cos, sin, cos sin (1 - delta), cos sin delta): the sample
// weight split over the two source levels (delta = the LOD's fraction);
// with the blend grid, whose values carry the split, (cos, sin, cos sin, 0).
__global__ void irradiance_tables_kernel(int theta_samples, int phi_samples, float delta, int blend,
                                         float2* __restrict__ theta_tab, float4* __restrict__ phi_tab) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  const double pi = 3.14159265358979323846;
  if (i < theta_samples) {
    double th = i * 2.0 * pi / theta_samples;
    theta_tab[i] = make_float2(static_cast<float>(cos(th)), static_cast<float>(sin(th)));
  }
  if (i < phi_samples) {
    double ph = i * 0.5 * pi / phi_samples;
    double c = cos(ph), s = sin(ph), d = static_cast<double>(delta);
    phi_tab[i] = blend ? make_float4(static_cast<float>(c), static_cast<float>(s), static_cast<float>(c * s), 0.0f)
                       : make_float4(static_cast<float>(c), static_cast<float>(s),
                                     static_cast<float>(c * s * (1.0 - d)), static_cast<float>(c * s * d));
  }
}

// One wave per output texel.  A lane owns one polar column (phi index
// 8 k + lane / 8) per pass and walks the azimuth rows theta = 8 s + lane % 8,
// so for a fixed step the wave's 64 lookups cover a compact patch of 8 polar
// by 8 azimuth samples (4.8 degrees of polar angle by at most 9.6 degrees,
// times sin(phi), of azimuth at the configured 300 x 150) and the gathers of
// a step share cache lines; a ring of 64 azimuths reaches 77 degrees.  Of
// the patches 4 x 16, 8 x 8, 16 x 4 and 32 x 2 (polar x azimuth), 8 x 8
// wastes the fewest lanes on the configured 150 x 300 samples: 19 passes of
// 38 steps (722 wave-steps) against 10 of 75 (750) for 16 x 4.  Each lane sums its column's samples over theta in FP32 in theta
// order and flushes the column into FP64 (kF64Sums) or FP32; the lanes are
// combined by a fixed xor tree across the wave.
constexpr int kIrrPhiLanes = 8, kIrrThetaLanes = 8;
static_assert(kIrrPhiLanes * kIrrThetaLanes == 64, "one wave per texel");

// kLevels: 1 (one source level), 2 (two levels, each its own lookup) or 3
// (the two levels' blend grid, one lookup of weight w0).
template <int kLevels>
__device__ __forceinline__ void irradiance_column(const char* __restrict__ gpyr, const float2* __restrict__ theta_tab,
                                                  const IrradianceParams& p, f3 u, f3 v, f3 w, float w0, float w1,
                                                  int a, float& sr, float& sg, float& sb) {
  for (int i = a; i < p.theta_samples; i += kIrrThetaLanes) {
    const float2 th = theta_tab[i];
    // n cos(phi) + (t cos(theta) + b sin(theta)) sin(phi), with u = t sin(phi),
    // v = b sin(phi), w = n cos(phi).
    const f3 d = mk(fmaf(u.x, th.x, fmaf(v.x, th.y, w.x)), fmaf(u.y, th.x, fmaf(v.y, th.y, w.y)),
                    fmaf(u.z, th.x, fmaf(v.z, th.y, w.z)));
    float yaw, pitch;
    equirect_angles(d, yaw, pitch);
    if (kLevels == 3) {
      blend_bilinear_acc(gpyr, p.grid, yaw, pitch, w0, sr, sg, sb);
    } else {
      split_bilinear_acc(gpyr, p.lv0, yaw, pitch, w0, sr, sg, sb);
      if (kLevels == 2) split_bilinear_acc(gpyr, p.lv1, yaw, pitch, w1, sr, sg, sb);
    }
  }
}

// Azimuth tables of up to this many rows are read from LDS (kLds): the
// table's loads then leave the texture data return, which bounds the kernel.
constexpr int kIrrThetaLdsMax = 4096;
constexpr int kIrrWaves = 4;

template <bool kF64Sums, bool kLds>
__global__ __launch_bounds__(64 * kIrrWaves) void irradiance_cube_kernel(const char* __restrict__ gpyr,
                                                                         const float2* __restrict__ theta_glob,
                                                                         const float4* __restrict__ phi_tab,
                                                                         const IrradianceParams p, float4* __restrict__ cube) {
  extern __shared__ float2 s_theta[];  // theta_samples rows when kLds
  if (kLds) {
    for (int i = threadIdx.x; i < p.theta_samples; i += 64 * kIrrWaves) s_theta[i] = theta_glob[i];
    __syncthreads();
  }
  const float2* theta_tab = kLds ? s_theta : theta_glob;
  const int S = p.size;
  const int rem = blockIdx.x * kIrrWaves + static_cast<int>(threadIdx.x >> 6);
  if (rem >= S * S) return;  // whole waves; no block barrier follows
  const int lane = threadIdx.x & 63;
  const int face = blockIdx.y;
  const int y = rem / S, x = rem - y * S;
  const size_t texel = static_cast<size_t>(face) * S * S + rem;
  const Frame fr = local_to_world(cube_texel_raw_dir(face, x, y, S));
  const int a = lane % kIrrThetaLanes, b = lane / kIrrThetaLanes;
  double ar = 0.0, ag = 0.0, ab = 0.0;
  float fr32 = 0.0f, fg32 = 0.0f, fb32 = 0.0f;
  for (int j = b; j < p.phi_samples; j += kIrrPhiLanes) {
    const float4 ph = phi_tab[j];
    const f3 u = fr.t * ph.y, v = fr.b * ph.y, w = fr.n * ph.x;
    float sr = 0.0f, sg = 0.0f, sb = 0.0f;
    if (p.blend)
      irradiance_column<3>(gpyr, theta_tab, p, u, v, w, ph.z, ph.w, a, sr, sg, sb);
    else if (p.delta != 0.0f)
      irradiance_column<2>(gpyr, theta_tab, p, u, v, w, ph.z, ph.w, a, sr, sg, sb);
    else
      irradiance_column<1>(gpyr, theta_tab, p, u, v, w, ph.z, ph.w, a, sr, sg, sb);
    if (kF64Sums) {
      ar += sr;
      ag += sg;
      ab += sb;
    } else {
      fr32 += sr;
      fg32 += sg;
      fb32 += sb;
    }
  }
  if (kF64Sums) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      ar += __shfl_xor(ar, o, 64);
      ag += __shfl_xor(ag, o, 64);
      ab += __shfl_xor(ab, o, 64);
    }
    if (lane == 0)
      cube[texel] = make_float4(static_cast<float>(ar * p.scale), static_cast<float>(ag * p.scale),
                                static_cast<float>(ab * p.scale), 1.0f);
  } else {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      fr32 += __shfl_xor(fr32, o, 64);
      fg32 += __shfl_xor(fg32, o, 64);
      fb32 += __shfl_xor(fb32, o, 64);
    }
    const float sc = static_cast<float>(p.scale);
    if (lane == 0) cube[texel] = make_float4(fr32 * sc, fg32 * sc, fb32 * sc, 1.0f);
  }
}

static int irradiance_phi_samples(int w, int h, int theta) {
  // int(pushConstants.height * thetaSamples / pushConstants.width) in FP32
  // (GenIrradianceMap.comp:135-136).
  return static_cast<int>(static_cast<float>(h) * static_cast<float>(theta) / static_cast<float>(w));
}

// Source LOD log2(W / thetaSamples) (GenIrradianceMap.comp:139) in FP32 as
// the shader computes it, clamped to the pyramid: levels l0, l1 and the
// fraction delta.
struct IrradianceLod {
  int l0, l1;
  float delta;
};
static IrradianceLod irradiance_lod(int w, int h, int theta) {
  const int levels = althea_env_levels(w, h);
  float lod = std::log2(static_cast<float>(w) / static_cast<float>(theta));
  lod = std::min(std::max(lod, 0.0f), static_cast<float>(levels - 1));
  IrradianceLod r;
  r.l0 = static_cast<int>(std::floor(lod));
  r.l1 = std::min(r.l0 + 1, levels - 1);
  r.delta = lod - static_cast<float>(r.l0);
  return r;
}

// Blend grid of levels l0 and l1 = l0 + 1 (two levels, each extent of l0
// even and l1 exactly half of it): nodes per axis 3 w0 / 2, plus the REPEAT
// border; RG plane texels rounded up to 64.
struct BlendGrid {
  bool ok;
  int w0, h0, nx, ny;
  size_t plane;
};
static BlendGrid blend_grid(int w, int h, const IrradianceLod& lod) {
  const PyramidGeometry g = pyramid_geometry(w, h);
  BlendGrid b{};
  if (lod.delta == 0.0f || lod.l1 != lod.l0 + 1) return b;
  b.w0 = g.w[lod.l0];
  b.h0 = g.h[lod.l0];
  b.ok = b.w0 >= 2 && b.h0 >= 2 && b.w0 % 2 == 0 && b.h0 % 2 == 0 && g.w[lod.l1] == b.w0 / 2 &&
         g.h[lod.l1] == b.h0 / 2;
  b.nx = 3 * b.w0 / 2;
  b.ny = 3 * b.h0 / 2;
  b.plane = (static_cast<size_t>(b.nx + 2) * (b.ny + 2) + 63) & ~static_cast<size_t>(63);
  return b;
}

struct BlendGridParams {
  int w0, h0, nx, ny;
  uint32_t off0, off1;  // pyramid texel offsets of the two levels
  double delta;
  size_t plane;
};

// Bilinear REPEAT value of the level at `off` (w x h) at texel coordinates
// (x, y), in FP64.
__device__ __forceinline__ void level_bilinear_f64(const float4* __restrict__ pyr, uint32_t off, int w, int h, double x,
                                                   double y, double* v) {
  const double fx = floor(x), fy = floor(y), ax = x - fx, ay = y - fy;
  const int i0 = static_cast<int>(fx), j0 = static_cast<int>(fy);
  auto at = [&](int i, int j) {
    return pyr[off + static_cast<size_t>((j % h + h) % h) * w + (i % w + w) % w];
  };
  const float4 t00 = at(i0, j0), t10 = at(i0 + 1, j0), t01 = at(i0, j0 + 1), t11 = at(i0 + 1, j0 + 1);
  const float a[4][3] = {{t00.x, t00.y, t00.z}, {t10.x, t10.y, t10.z}, {t01.x, t01.y, t01.z}, {t11.x, t11.y, t11.z}};
  for (int k = 0; k < 3; ++k)
    v[k] = (1.0 - ay) * ((1.0 - ax) * a[0][k] + ax * a[1][k]) + ay * ((1.0 - ax) * a[2][k] + ax * a[3][k]);
}

// The blend (1 - delta) B0 + delta B1 at fine coordinates (x0, y0), B1 at
// x0 / 2 - 1/4 of the half-size level.
__device__ __forceinline__ void blend_value(const float4* __restrict__ pyr, const BlendGridParams& p, double x0,
                                            double y0, float f[3]) {
  double b0[3], b1[3];
  level_bilinear_f64(pyr, p.off0, p.w0, p.h0, x0, y0, b0);
  level_bilinear_f64(pyr, p.off1, p.w0 / 2, p.h0 / 2, 0.5 * x0 - 0.25, 0.5 * y0 - 0.25, b1);
  for (int k = 0; k < 3; ++k) f[k] = static_cast<float>((1.0 - p.delta) * b0[k] + p.delta * b1[k]);
}

// One thread per padded node (r, c): node (c - 1, r - 1) wrapped to the
// grid, at fine coordinates (2 (n / 3) + (n % 3) / 2) per axis; its value
// (1 - delta) B0 + delta B1 in FP64 (B1 at x0 / 2 - 1/4, REPEAT), rounded
// once, into the RG and B planes.
__global__ __launch_bounds__(256) void blend_grid_kernel(const float4* __restrict__ pyr, const BlendGridParams p,
                                                         float* __restrict__ out) {
  const size_t W = static_cast<size_t>(p.nx) + 2, i = static_cast<size_t>(blockIdx.x) * 256 + threadIdx.x;
  if (i >= W * (p.ny + 2)) return;
  const int r = static_cast<int>(i / W), c = static_cast<int>(i - r * W);
  auto wrap = [](int k, int n) { return k < 0 ? k + n : (k >= n ? k - n : k); };
  const int n = wrap(c - 1, p.nx), m = wrap(r - 1, p.ny);
  float f[3];
  blend_value(pyr, p, 2.0 * (n / 3) + 0.5 * (n % 3), 2.0 * (m / 3) + 0.5 * (m % 3), f);
  reinterpret_cast<float2*>(out)[i] = make_float2(f[0], f[1]);
  out[2 * p.plane + i] = f[2];
}

// ------------------------------------------------- irradiance, folded source
// The equirect map, the texel lattice and (with an even azimuth count) the
// azimuth set are all symmetric under the eight sign flips F of (x, y, z):
// the frame of texel direction F n is F times the frame of n up to a half
// turn and a reflection of the azimuth, so the samples of the eight texels
// F n are F times the samples of n, and a flip acts on a lookup as yaw ->
// pi - yaw (x), yaw -> -yaw (z), pitch -> -pitch (y).  One evaluation of a
// sample's direction, angles, cell and weights serves eight texels, whose
// lookups read the same node of the source folded onto yaw and pitch in
// [0, pi/2]: a folded node holds its eight images (x bit 0, z bit 1, y bit 2
// of the slot) as eight 12-byte slots.
//
// Folded coordinates (either axis, E the extent): x' = angle E / 2pi + 3/2
// (pitch: angle H / pi + 3/2), which is the source coordinate minus E / 2 - 2,
// so the node pattern of the blend grid keeps its phase (E % 4 == 0).  Column
// 0 is the node at x' = 1, just across the fold.  Two more columns hold the
// precompute's pole branch (|xz| <= 0.001 reads yaw 0 whatever the signs of
// x and z): the nodes beside yaw 0 in every slot, without the x and z flips.
// The row after the last, all zeros, is what the lanes past the last azimuth
// or polar row read (an infinite texel times their weight 0 would be NaN).
struct FoldGrid {
  bool ok;
  int w0, h0, blend;
  int cols, rows;  // columns without the two pole columns
  size_t cells;    // nodes of the grid, pole columns included
  size_t nodes;    // stored nodes: the grid and, after it, a row and two nodes of zeros
};
constexpr int kFoldNodeBytes = 96;
constexpr size_t kFoldMaxBytes = size_t{1} << 30;

// Steps of an orbit from which the folded kernel takes a call.  Its block of 16
// waves stands idle for the rest of them, and orders its waves and adds their sums
// whatever the steps: 128^2 x 6 texels of a 512 x 256 source take 53 us by texel
// and 126 folded at 1 step (8 azimuths), 118 and 180 at 6 (24), 152 and 197 at 8
// (30), 286 and 280 at 15 (40), 360 and 309 at 18 (48).
constexpr int kFoldMinSteps = 14;

static FoldGrid fold_grid(int w, int h, int theta, const IrradianceLod& lod) {
  FoldGrid f{};
  if (w <= 0 || h <= 0 || theta % 2 != 0) return f;
  const long long polar = (irradiance_phi_samples(w, h, theta) + 7) / 8, azimuth = (theta + 7) / 8;
  if (polar * azimuth < kFoldMinSteps) return f;
  const PyramidGeometry g = pyramid_geometry(w, h);
  f.blend = lod.delta != 0.0f ? 1 : 0;
  if (f.blend && !blend_grid(w, h, lod).ok) return f;
  f.w0 = g.w[lod.l0];
  f.h0 = g.h[lod.l0];
  if (f.w0 % 8 != 0 || f.h0 % 4 != 0) return f;
  f.cols = (f.blend ? 3 * f.w0 / 8 : f.w0 / 4) + 2;
  f.rows = (f.blend ? 3 * f.h0 / 4 : f.h0 / 2) + 2;
  f.cells = static_cast<size_t>(f.cols + 2) * f.rows;
  f.nodes = f.cells + (f.cols + 2) + 2;
  f.ok = kFoldNodeBytes * f.nodes <= kFoldMaxBytes;
  return f;
}

// The theta and phi tables, then the folded grid, the blend grid of levels
// l0, l1 or their split gather copy.
size_t irradiance_workspace_bytes(int w, int h, int, int theta) {
  int phi = irradiance_phi_samples(w, h, theta);
  const size_t tables = align256(sizeof(float2) * theta) + align256(sizeof(float4) * std::max(phi, 1));
  if (w <= 0 || h <= 0 || theta <= 0) return tables;
  const IrradianceLod lod = irradiance_lod(w, h, theta);
  const FoldGrid f = fold_grid(w, h, theta, lod);
  if (f.ok) return tables + align256(kFoldNodeBytes * f.nodes);
  const BlendGrid b = blend_grid(w, h, lod);
  if (b.ok) return tables + 12 * b.plane;
  return tables + split_gather_bytes(w, h, lod.l0, lod.l1);
}

struct FoldGridParams {
  BlendGridParams src;  // w0, h0, off0, off1, delta
  int blend, cols, rows;
};

// One thread per slot of a folded node, in storage order.
__global__ __launch_bounds__(256) void fold_grid_kernel(const float4* __restrict__ pyr, const FoldGridParams p,
                                                        float* __restrict__ out) {
  const uint32_t i = blockIdx.x * 256u + threadIdx.x;
  const uint32_t cols = static_cast<uint32_t>(p.cols) + 2u;
  const uint32_t cells = cols * static_cast<uint32_t>(p.rows);
  if (i >= 8u * (cells + cols + 2u)) return;
  if (i >= 8u * cells) {
    for (int k = 0; k < 3; ++k) out[3 * static_cast<size_t>(i) + k] = 0.0f;
    return;
  }
  const int slot = static_cast<int>(i & 7u);
  const int r = static_cast<int>((i >> 3) / cols), c = static_cast<int>((i >> 3) - static_cast<uint32_t>(r) * cols);
  const int W = p.src.w0, H = p.src.h0;
  const bool pole = c >= p.cols;
  // Column k of the stored grid as x' (column 0: the node at x' = 1).
  auto at = [&](int k) { return p.blend ? 2.0 * ((k + 2) / 3) + 0.5 * ((k + 2) % 3) : k + 1.0; };
  double x0 = (pole ? 1.0 + (c - p.cols) : at(c)) + (0.5 * W - 2.0);
  double y0 = at(r) + (0.5 * H - 2.0);  // the row of negative pitch
  if (!pole && (slot & 1)) x0 = 1.5 * W - 1.0 - x0;
  if (!pole && (slot & 2)) x0 = W - 1.0 - x0;
  if (!(slot & 4)) y0 = H - 1.0 - y0;
  float f[3];
  if (p.blend) {
    blend_value(pyr, p.src, x0, y0, f);
  } else {
    const int i0 = (static_cast<int>(x0) + 2 * W) % W, j0 = (static_cast<int>(y0) + 2 * H) % H;
    const float4 t = pyr[p.src.off0 + static_cast<size_t>(j0) * W + i0];
    f[0] = t.x, f[1] = t.y, f[2] = t.z;
  }
  for (int k = 0; k < 3; ++k) out[3 * static_cast<size_t>(i) + k] = f[k];
}

struct FoldParams {
  float kx, ky;  // x' = yaw kx + 3/2, y' = pitch ky + 3/2
  int cols;
  uint32_t rowbytes;  // kFoldNodeBytes (cols + 2)
  uint32_t zeros;     // byte offset of the row of zeros
  int size;
  int theta_samples, phi_samples;
  int theta_steps, polar_steps;  // groups of 8 azimuths and of 8 polar rows
  double scale;            // pi / theta_samples / phi_samples
};

// Lower node (stored column or row) of folded coordinate x' and the fraction.
template <bool kBlend>
__device__ __forceinline__ int fold_cell(float x, float& t) {
  if (kBlend) return blend_cell(x, t) - 2;
  t = __builtin_amdgcn_fractf(x);
  return cvt_floor(x) - 1;
}

// A block of 16 waves per orbit of eight texels F n; the waves take the
// orbit's steps in turn, a step being a patch of 8 polar by 8 azimuth samples.
// Each lane evaluates one sample of the step for n = |n| and leaves (node
// offset with the sample's own signs as slot bits, fractions, weight) in LDS;
// then in eight rounds lane (s, F) adds sample 8 k + s into texel F.
// FP32 sums of 32 lookups are flushed into FP64 (kF64Sums); lanes and waves
// combine in a fixed order.
//
// Bound: the gathers. A gather instruction whose lanes each read 12 or 16
// bytes takes 16 cycles of the texture data return; the eight lanes of a
// sample read one node's 96 bytes, so a round's loads stay at 16.4 cycles
// (31 for 64 unrelated lookups, irradiance_cube_kernel) and the return is 94 %
// busy, and a lookup costs 36 VALU in all instead of 115.  512 x 256 source,
// 32^2 x 6 texels, 300 x 150 samples: 1.09 -> 0.51 ms.  Measured beside it
// for the whole precompute (0.816 ms): 16-byte slots 0.84 (4.8 MB of nodes
// against 3.6 MB in a 4 MB L2), RG and B planes (eight narrower loads a
// lookup) 1.05, six waves per SIMD instead of four 0.91; 4, 8 or 16 waves
// per orbit alike, and 16 keep the GPU filled on the smallest cubes.
constexpr int kFoldWaves = 16;
// Azimuth and polar tables of up to this many bytes are read from LDS.
constexpr size_t kFoldTableMax = 32768;

template <bool kF64Sums, bool kBlend, bool kLds>
__global__ __launch_bounds__(64 * kFoldWaves) void irradiance_fold_kernel(const char* __restrict__ grid,
                                                                          const float2* __restrict__ theta_glob,
                                                                          const float4* __restrict__ phi_glob,
                                                                          const FoldParams p,
                                                                          float4* __restrict__ cube) {
  using T = typename std::conditional<kF64Sums, double, float>::type;
  typedef const __attribute__((address_space(1))) char gchar;
  typedef const __attribute__((address_space(1))) float gfloat;
  extern __shared__ float4 s_tab[];  // the polar rows, then the azimuth rows (kLds)
  __shared__ float4 s_rec[kFoldWaves][64];
  __shared__ T s_part[kFoldWaves][3][8];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  float2* s_theta = reinterpret_cast<float2*>(s_tab + p.phi_samples);
  if (kLds) {
    for (int i = threadIdx.x; i < p.phi_samples; i += 64 * kFoldWaves) s_tab[i] = phi_glob[i];
    for (int i = threadIdx.x; i < p.theta_samples; i += 64 * kFoldWaves) s_theta[i] = theta_glob[i];
    __syncthreads();
  }
  const float4* phi_tab = kLds ? s_tab : phi_glob;
  const float2* theta_tab = kLds ? s_theta : theta_glob;
  const int S = p.size, half = (S + 1) / 2;
  // The orbit's representative with no negative component, on the lattice of
  // half-texels (cube_texel_raw_dir): the major component is S.
  const int axis = blockIdx.y / half;
  const int even = 1 - (S & 1);
  const int cu = 2 * (static_cast<int>(blockIdx.y) - axis * half) + even, cv = 2 * static_cast<int>(blockIdx.x) + even;
  const int nx = axis == 0 ? S : cu, ny = axis == 1 ? S : (axis == 0 ? cu : cv), nz = axis == 2 ? S : cv;
  const Frame fr = local_to_world(mk(static_cast<float>(nx), static_cast<float>(ny), static_cast<float>(nz)));
  const uint32_t flip = static_cast<uint32_t>(lane & 7);
  float4* rec = s_rec[wave];
  T ar = 0, ag = 0, ab = 0;
  float sr = 0.0f, sg = 0.0f, sb = 0.0f;
  unsigned done = 0;
  for (FoldStep st = fold_advance({0, 0}, wave, p.theta_steps); st.polar < p.polar_steps;
       st = fold_advance(st, kFoldWaves, p.theta_steps)) {
    const int i = st.azimuth * 8 + (lane & 7), j = st.polar * 8 + (lane >> 3);
    const bool valid = i < p.theta_samples && j < p.phi_samples;
    const float2 th = theta_tab[min(i, p.theta_samples - 1)];
    const float4 ph = phi_tab[min(j, p.phi_samples - 1)];
    const f3 u = fr.t * ph.y, v = fr.b * ph.y, w = fr.n * ph.x;
    const f3 d = mk(fmaf(u.x, th.x, fmaf(v.x, th.y, w.x)), fmaf(u.y, th.x, fmaf(v.y, th.y, w.y)),
                    fmaf(u.z, th.x, fmaf(v.z, th.y, w.z)));
    const float len_xz = sqrt_fast(fmaf(d.x, d.x, d.z * d.z));
    const bool off_pole = len_xz > 0.001f;  // equirect_angles' branch
    float fx, fy;
    int col = fold_cell<kBlend>(fmaf(atan2_first(fabsf(d.z), fabsf(d.x)), p.kx, 1.5f), fx);
    const int row =
        fold_cell<kBlend>(fmaf(off_pole ? atan2_first(fabsf(d.y), len_xz) : 0.5f * kPi, p.ky, 1.5f), fy);
    if (!off_pole) col = p.cols, fx = 0.5f;
    const uint32_t signs = (__float_as_uint(d.x) >> 31) | (__float_as_uint(d.z) >> 31 << 1) |
                           (__float_as_uint(d.y) >> 31 << 2);
    const uint32_t off = static_cast<uint32_t>(row) * p.rowbytes + static_cast<uint32_t>(col * kFoldNodeBytes);
    rec[lane] = make_float4(__uint_as_float(valid ? off | signs : p.zeros), fx, fy, valid ? ph.z : 0.0f);
    wave_lds_sync();
#pragma unroll 4
    for (int k = 0; k < 8; ++k) {
      const float4 q = rec[8 * k + (lane >> 3)];
      const uint32_t node = __float_as_uint(q.x);  // a multiple of 32, plus the sample's sign bits
      const uint32_t o0 = (node & ~7u) + ((node ^ flip) & 7u) * 12u;
      gfloat* r0 = (gfloat*)((gchar*)grid + o0);
      gfloat* r1 = (gfloat*)((gchar*)grid + (o0 + p.rowbytes));
      LevelTaps t;
      t.t00 = mk(r0[0], r0[1], r0[2]);
      t.t10 = mk(r0[24], r0[25], r0[26]);
      t.t01 = mk(r1[0], r1[1], r1[2]);
      t.t11 = mk(r1[24], r1[25], r1[26]);
      t.ax = q.y;
      t.ay = q.z;
      taps_acc(t, q.w, sr, sg, sb);
    }
    wave_lds_sync();  // the rounds' reads before the next step's records
    if ((++done & 3) == 0) {
      ar += sr, ag += sg, ab += sb;
      sr = sg = sb = 0.0f;
    }
  }
  ar += sr, ag += sg, ab += sb;
#pragma unroll
  for (int o = 8; o < 64; o <<= 1) {
    ar += __shfl_xor(ar, o, 64);
    ag += __shfl_xor(ag, o, 64);
    ab += __shfl_xor(ab, o, 64);
  }
  if (lane < 8) s_part[wave][0][lane] = ar, s_part[wave][1][lane] = ag, s_part[wave][2][lane] = ab;
  __syncthreads();
  if (threadIdx.x >= 8) return;
  // Texel F n; a flip of a zero component names the same texel again.
  if (((lane & 1) && nx == 0) || ((lane & 2) && nz == 0) || ((lane & 4) && ny == 0)) return;
  T v[3] = {0, 0, 0};
  for (int k = 0; k < kFoldWaves; ++k)
    for (int c = 0; c < 3; ++c) v[c] += s_part[k][c][lane];
  const int px = (lane & 1) ? -nx : nx, py = (lane & 4) ? -ny : ny, pz = (lane & 2) ? -nz : nz;
  int face, sc, tc;
  if (axis == 0)
    face = px > 0 ? 0 : 1, sc = px > 0 ? -pz : pz, tc = -py;
  else if (axis == 1)
    face = py > 0 ? 2 : 3, sc = px, tc = py > 0 ? pz : -pz;
  else
    face = pz > 0 ? 4 : 5, sc = pz > 0 ? px : -px, tc = -py;
  const T scale = static_cast<T>(p.scale);
  cube[(static_cast<size_t>(face) * S + (tc + S - 1) / 2) * S + (sc + S - 1) / 2] =
      make_float4(static_cast<float>(v[0] * scale), static_cast<float>(v[1] * scale), static_cast<float>(v[2] * scale),
                  1.0f);
}

// One lookup per sample (a blend grid, folded or not): the polar weights are
// not split over two levels.
static int irradiance_one_lookup(int w, int h, int theta, const IrradianceLod& lod) {
  return fold_grid(w, h, theta, lod).ok || blend_grid(w, h, lod).ok ? 1 : 0;
}

// The folded grid, then one block per orbit.
static althea_status launch_irradiance_fold(const float* pyr, const PyramidGeometry& g, const FoldGrid& fg,
                                            const IrradianceLod& lod, int size, int theta_samples, int phi,
                                            unsigned flags, float* cube, const float2* theta_tab,
                                            const float4* phi_tab, float* grid, hipStream_t s) {
  FoldGridParams q{};
  q.src.w0 = fg.w0;
  q.src.h0 = fg.h0;
  q.src.off0 = g.off[lod.l0];
  q.src.off1 = g.off[lod.l1];
  q.src.delta = static_cast<double>(lod.delta);
  q.blend = fg.blend;
  q.cols = fg.cols;
  q.rows = fg.rows;
  hipLaunchKernelGGL(fold_grid_kernel, dim3(static_cast<unsigned>((8 * fg.nodes + 255) / 256)), dim3(256), 0, s,
                     reinterpret_cast<const float4*>(pyr), q, grid);
  const althea_status st = check_launch("fold_grid_kernel");
  if (st != ALTHEA_OK) return st;
  const LevelC c0 = make_level(fg.w0, fg.h0, 0);
  FoldParams p{};
  p.kx = c0.kx;
  p.ky = -c0.ky;
  p.cols = fg.cols;
  p.rowbytes = static_cast<uint32_t>(kFoldNodeBytes * (fg.cols + 2));
  p.zeros = static_cast<uint32_t>(kFoldNodeBytes * fg.cells);
  p.size = size;
  p.theta_samples = theta_samples;
  p.phi_samples = phi;
  p.theta_steps = (theta_samples + 7) / 8;
  p.polar_steps = (phi + 7) / 8;
  p.scale = M_PI / theta_samples / phi;
  const IrradianceGrid blocks = fold_blocks(size);
  const bool f64 = !(flags & ALTHEA_PRECOMPUTE_FP32_SUMS);
  const size_t tables = sizeof(float4) * static_cast<size_t>(phi) + sizeof(float2) * static_cast<size_t>(theta_samples);
  const bool lds = tables <= kFoldTableMax;
  const int variant = (f64 ? 1 : 0) | (fg.blend ? 2 : 0) | (lds ? 4 : 0);
  auto kernel = variant == 0   ? irradiance_fold_kernel<false, false, false>
                : variant == 1 ? irradiance_fold_kernel<true, false, false>
                : variant == 2 ? irradiance_fold_kernel<false, true, false>
                : variant == 3 ? irradiance_fold_kernel<true, true, false>
                : variant == 4 ? irradiance_fold_kernel<false, false, true>
                : variant == 5 ? irradiance_fold_kernel<true, false, true>
                : variant == 6 ? irradiance_fold_kernel<false, true, true>
                               : irradiance_fold_kernel<true, true, true>;
  hipLaunchKernelGGL(kernel, dim3(blocks.x, blocks.y), dim3(64 * kFoldWaves), lds ? tables : 0, s,
                     reinterpret_cast<const char*>(grid), theta_tab, phi_tab, p, reinterpret_cast<float4*>(cube));
  return check_launch("irradiance_fold_kernel");
}

althea_status launch_irradiance(const float* pyr, int env_w, int env_h, int size, int theta_samples,
                                unsigned flags, float* cube, void* workspace, hipStream_t s) {
  const int phi = irradiance_phi_samples(env_w, env_h, theta_samples);
  ALTHEA_REQUIRE(phi >= 1, "irradiance: int(H*theta/W) = %d phi samples", phi);
  char* ws = static_cast<char*>(workspace);
  float2* theta_tab = reinterpret_cast<float2*>(ws);
  ws += align256(sizeof(float2) * theta_samples);
  float4* phi_tab = reinterpret_cast<float4*>(ws);
  ws += align256(sizeof(float4) * phi);
  float* gather = reinterpret_cast<float*>(ws);

  IrradianceParams p{};
  PyramidGeometry g = pyramid_geometry(env_w, env_h);
  p.levels = g.levels;
  p.size = size;
  p.theta_samples = theta_samples;
  p.phi_samples = phi;
  const IrradianceLod lod = irradiance_lod(env_w, env_h, theta_samples);
  p.l0 = lod.l0;
  p.l1 = lod.l1;
  p.delta = lod.delta;
  const int tab = std::max(theta_samples, phi);
  hipLaunchKernelGGL(irradiance_tables_kernel, dim3((tab + 255) / 256), dim3(256), 0, s, theta_samples, phi, p.delta,
                     irradiance_one_lookup(env_w, env_h, theta_samples, lod), theta_tab, phi_tab);
  althea_status st = check_launch("irradiance_tables_kernel");
  if (st != ALTHEA_OK) return st;
  const FoldGrid fg = fold_grid(env_w, env_h, theta_samples, lod);
  if (fg.ok) return launch_irradiance_fold(pyr, g, fg, lod, size, theta_samples, phi, flags, cube, theta_tab, phi_tab, gather, s);
  const BlendGrid bg = blend_grid(env_w, env_h, lod);
  if (bg.ok) {
    BlendGridParams q{};
    q.w0 = bg.w0;
    q.h0 = bg.h0;
    q.nx = bg.nx;
    q.ny = bg.ny;
    q.off0 = g.off[p.l0];
    q.off1 = g.off[p.l1];
    q.delta = static_cast<double>(lod.delta);
    q.plane = bg.plane;
    const size_t nodes = static_cast<size_t>(bg.nx + 2) * (bg.ny + 2);
    hipLaunchKernelGGL(blend_grid_kernel, dim3(static_cast<unsigned>((nodes + 255) / 256)), dim3(256), 0, s,
                       reinterpret_cast<const float4*>(pyr), q, gather);
    st = check_launch("blend_grid_kernel");
    if (st != ALTHEA_OK) return st;
    const LevelC c0 = make_level(bg.w0, bg.h0, 0);
    p.grid.kx = c0.kx;
    p.grid.cx = c0.cx;
    p.grid.ky = c0.ky;
    p.grid.cy = c0.cy;
    p.grid.rowbytes = static_cast<uint32_t>(bg.nx + 2) * 8u;
    p.grid.rg = 0;
    p.grid.b = static_cast<uint32_t>(8 * bg.plane);
    p.blend = 1;
  } else {
    const GatherGeometry gg = gather_geometry(env_w, env_h, p.l0, p.l1);
    st = launch_split_gather(pyr, env_w, env_h, gg, gather, s);
    if (st != ALTHEA_OK) return st;
    p.lv0 = split_level(env_w, env_h, gg, p.l0);
    p.lv1 = split_level(env_w, env_h, gg, p.l1);
  }
  p.scale = M_PI / theta_samples / phi;
  const IrradianceGrid blocks = texel_blocks(size, kIrrWaves);
  const dim3 grid(blocks.x, blocks.y), block(64 * kIrrWaves);
  const char* g4 = reinterpret_cast<const char*>(gather);
  float4* cube4 = reinterpret_cast<float4*>(cube);
  const bool f64 = !(flags & ALTHEA_PRECOMPUTE_FP32_SUMS);
  if (theta_samples <= kIrrThetaLdsMax) {
    const size_t lds = sizeof(float2) * static_cast<size_t>(theta_samples);
    if (f64)
      hipLaunchKernelGGL((irradiance_cube_kernel<true, true>), grid, block, lds, s, g4, theta_tab, phi_tab, p,
                         cube4);
    else
      hipLaunchKernelGGL((irradiance_cube_kernel<false, true>), grid, block, lds, s, g4, theta_tab, phi_tab, p,
                         cube4);
  } else if (f64) {
    hipLaunchKernelGGL((irradiance_cube_kernel<true, false>), grid, block, 0, s, g4, theta_tab, phi_tab, p, cube4);
  } else {
    hipLaunchKernelGGL((irradiance_cube_kernel<false, false>), grid, block, 0, s, g4, theta_tab, phi_tab, p,
                       cube4);
  }
  return check_launch("irradiance_cube_kernel");
}

// --------------------------------------------------------------- BRDF LUT
// Karis split-sum (A, B) at texel centre (NdotV, roughness).  A block covers
// 64 NdotV columns of one roughness row with kLutWaves waves, each owning a
// contiguous range of samples that is a whole number of 32-sample blocks.  The
// half vectors depend on the row only: a wave's lanes form 64 of them (correctly
// rounded roots and quotients, sincospi), leave them in LDS and then all read
// each in turn.  32-sample FP32 block sums flushed into FP64, the waves' FP64
// partials combined in wave order, FP64 normalisation.
//
// Bound: VALU, 30 a column and sample in all, 19 of them the loop's (about 120
// with the half vector formed by every lane), at 0.87 of the nominal issue rate:
// 128^2 x 1024 samples, 62 -> 14 us.
constexpr int kLutWaves = 16;

__global__ __launch_bounds__(64 * kLutWaves) void brdf_lut_kernel(int size, int samples, int chunk,
                                                                  float2* __restrict__ rg) {
  __shared__ double s_a[kLutWaves][64], s_b[kLutWaves][64];
  __shared__ float4 s_half[kLutWaves][64];  // h.x, h.z, 2 h.z, 1 / h.z
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int x = blockIdx.x * 64 + lane;
  const int y = blockIdx.y;
  const float nv = (static_cast<float>(x) + 0.5f) / static_cast<float>(size);
  const float r = (static_cast<float>(y) + 0.5f) / static_cast<float>(size);
  const float alpha = r * r;
  const float a2 = alpha * alpha;
  const float k = 0.5f * alpha, om_k = 1.0f - k;
  const float vx = sqrtf(fmaxf(0.0f, fmaf(-nv, nv, 1.0f)));
  double sa = 0.0, sb = 0.0;
  float fa = 0.0f, fb = 0.0f;
  const int s0 = wave * chunk, s1 = min(samples, s0 + chunk);
  for (int base = s0; base < s1; base += 64) {
    float x1, x2, sp, cp;
    hammersley(static_cast<uint32_t>(base + lane), static_cast<uint32_t>(samples), x1, x2);
    const float den = fmaf(a2 - 1.0f, x2, 1.0f);
    const float cos_t = sqrtf((1.0f - x2) / den);
    sincospif(2.0f * x1, &sp, &cp);
    wave_lds_sync();  // the last 64 are read
    s_half[wave][lane] = make_float4(cp * sqrtf(a2 * x2 / den), cos_t, 2.0f * cos_t, 1.0f / cos_t);
    wave_lds_sync();
    const int n = min(64, s1 - base);
    for (int j = 0; j < n; ++j) {
      const float4 h = s_half[wave][j];
      const float vdh = fmaf(vx, h.x, nv * h.y);
      const float ndl = fmaf(vdh, h.z, -nv);
      const float om = 1.0f - vdh;
      const float om2 = om * om;
      const float fc = om2 * om2 * om;
      // gl VdotH / NdotH (the view term over NdotV once, after the sums);
      // nothing below the horizon.
      const float dl = fmaf(ndl, om_k, k), rl = rcp_fast(dl);
      const float g = (ndl * vdh) * h.w * fmaf(rl, fmaf(-dl, rl, 1.0f), rl);
      const float g_vis = ndl > 0.0f ? g : 0.0f;
      fa = fmaf(1.0f - fc, g_vis, fa);
      fb = fmaf(fc, g_vis, fb);
      if (((base + j) & (kBlockSums - 1)) == kBlockSums - 1) {
        sa += fa;
        sb += fb;
        fa = fb = 0.0f;
      }
    }
  }
  sa += fa;
  sb += fb;
  s_a[wave][lane] = sa;
  s_b[wave][lane] = sb;
  __syncthreads();
  if (wave != 0 || x >= size) return;
  double ta = 0.0, tb = 0.0;
#pragma unroll
  for (int w = 0; w < kLutWaves; ++w) {
    ta += s_a[w][lane];
    tb += s_b[w][lane];
  }
  const double gv = 1.0 / ((static_cast<double>(nv) * (1.0 - k) + k) * samples);  // Smith's view term over NdotV
  rg[y * size + x] = make_float2(static_cast<float>(ta * gv), static_cast<float>(tb * gv));
}

althea_status launch_brdf_lut(int size, int samples, float* rg, hipStream_t s) {
  dim3 grid((size + 63) / 64, size);
  const int per_wave = (samples + kLutWaves - 1) / kLutWaves;
  const int chunk = (per_wave + kBlockSums - 1) / kBlockSums * kBlockSums;
  hipLaunchKernelGGL(brdf_lut_kernel, grid, dim3(64 * kLutWaves), 0, s, size, samples, chunk,
                     reinterpret_cast<float2*>(rg));
  return check_launch("brdf_lut_kernel");
}

// ---------------------------------------------------------- sampler probes
__global__ void cube_sample_kernel(const float4* __restrict__ cube, const CubeMips cm,
                                   const float4* __restrict__ dir_lod, int count, float4* __restrict__ out) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= count) return;
  float4 q = dir_lod[i];
  f3 v = cube_sample(cube, cm, mk(q.x, q.y, q.z), q.w);
  out[i] = make_float4(v.x, v.y, v.z, 1.0f);
}

althea_status launch_cube_sample(const float* cube, int size, int mips, const float* dir_lod, int count,
                                 float* out, void*, hipStream_t s) {
  if (count == 0) return ALTHEA_OK;
  CubeMips cm = cube_mips_of(size, mips);
  hipLaunchKernelGGL(cube_sample_kernel, dim3((count + 255) / 256), dim3(256), 0, s,
                     reinterpret_cast<const float4*>(cube), cm, reinterpret_cast<const float4*>(dir_lod), count,
                     reinterpret_cast<float4*>(out));
  return check_launch("cube_sample_kernel");
}

// --------------------------------------------------- seamless-bordered cubes
BorderedCube bordered_cube_of(int size, int mips) {
  BorderedCube c{};
  c.size = size;
  c.mips = mips;
  size_t off = 0;
  for (int m = 0; m < mips; ++m) {
    c.off[m] = static_cast<uint32_t>(off);
    const size_t w = static_cast<size_t>(std::max(1, size >> m)) + 2;
    off += 6 * w * w;
  }
  return c;
}

size_t cube_bordered_texels(int size, int mips) {
  size_t n = 0;
  for (int m = 0; m < mips; ++m) {
    const size_t w = static_cast<size_t>(std::max(1, size >> m)) + 2;
    n += 6 * w * w;
  }
  return n;
}

// One thread per bordered texel: bordered (r, c) of face f at mip m is
// cube_tap(f, c - 1, r - 1), the tap a seamless bilinear lookup reads there.
__global__ __launch_bounds__(256) void cube_border_kernel(const float4* __restrict__ cube, const CubeMips cm,
                                                          const BorderedCube bc, uint32_t total,
                                                          float4* __restrict__ out) {
  const uint32_t i = blockIdx.x * 256u + threadIdx.x;
  if (i >= total) return;
  int m = 0;
  while (m + 1 < bc.mips && i >= bc.off[m + 1]) ++m;
  const int S = max(1, bc.size >> m), W = S + 2;
  const uint32_t k = i - bc.off[m];
  const int face = static_cast<int>(k / static_cast<uint32_t>(W * W));
  const int rem = static_cast<int>(k) - face * W * W;
  const int r = rem / W, c = rem - r * W;
  const f3 v = cube_tap(cube + cm.off[m], S, face, c - 1, r - 1);
  out[i] = make_float4(v.x, v.y, v.z, 1.0f);
}

althea_status launch_cube_border(const float* cube, int size, int mips, float* bordered, hipStream_t s) {
  const CubeMips cm = cube_mips_of(size, mips);
  const BorderedCube bc = bordered_cube_of(size, mips);
  const uint32_t total = static_cast<uint32_t>(cube_bordered_texels(size, mips));
  hipLaunchKernelGGL(cube_border_kernel, dim3((total + 255) / 256), dim3(256), 0, s,
                     reinterpret_cast<const float4*>(cube), cm, bc, total, reinterpret_cast<float4*>(bordered));
  return check_launch("cube_border_kernel");
}

struct EnvSampleParams {
  LevelC lv[kMaxLevels];
  int levels;
  int count;
};

__global__ __launch_bounds__(256) void env_sample_kernel(const char* __restrict__ pyr, const EnvSampleParams p,
                                                         const float4* __restrict__ dir_lod,
                                                         float4* __restrict__ out) {
  __shared__ LevelC s_lv[kMaxLevels];
  if (threadIdx.x < kMaxLevels) s_lv[threadIdx.x] = p.lv[threadIdx.x];
  __syncthreads();
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= p.count) return;
  // The mirror-lookup path: angles and texel coordinates in df32 (the
  // addressing of the roughness-0 prefilter), the two levels blended with
  // weights 1 - delta and delta.
  const float4 q = dir_lod[i];
  const float len_xz = sqrtf(fmaf(q.x, q.x, q.z * q.z));
  const int pole = len_xz > 0.001f ? 0 : (q.y > 0.0f ? 1 : -1);
  df32 yaw, pitch;
  equirect_angles_df(df3{df_of(q.x), df_of(q.y), df_of(q.z)}, pole, yaw, pitch);
  const float d = fminf(fmaxf(q.w, 0.0f), static_cast<float>(p.levels - 1));
  const float fl = floorf(d);
  const int l0 = static_cast<int>(fl);
  const float delta = d - fl;
  auto at = [&](int l) {
    const LevelC& c = s_lv[l];
    df32 x, y;
    equirect_texel_df(yaw, pitch, static_cast<int>(c.wmask + 1), static_cast<int>(c.hmask + 1), x, y);
    return level_bilinear_df(pyr, c, x, y);
  };
  f3 v = at(l0);
  if (delta != 0.0f) {
    const f3 b = at(min(l0 + 1, p.levels - 1));
    const float w0 = 1.0f - delta;
    v = mk(fmaf(b.x, delta, v.x * w0), fmaf(b.y, delta, v.y * w0), fmaf(b.z, delta, v.z * w0));
  }
  out[i] = make_float4(v.x, v.y, v.z, 1.0f);
}

althea_status launch_env_sample(const float* pyr, int w, int h, const float* dir_lod, int count, float* out, void*,
                                hipStream_t s) {
  if (count == 0) return ALTHEA_OK;
  EnvSampleParams p{};
  pyramid_levels(w, h, p.lv);
  p.levels = althea_env_levels(w, h);
  p.count = count;
  hipLaunchKernelGGL(env_sample_kernel, dim3((count + 255) / 256), dim3(256), 0, s,
                     reinterpret_cast<const char*>(pyr), p, reinterpret_cast<const float4*>(dir_lod),
                     reinterpret_cast<float4*>(out));
  return check_launch("env_sample_kernel");
}

}  // namespace althea
