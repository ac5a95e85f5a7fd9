// Decode projections for gfx950: y[M, N] = x[M, K] . W[N, K]^T (+ bias) with M <= 16.
//
// In a decode step every projection of the batched engine multiplies a few
// token rows by a large weight, so the weight read is the whole cost: the
// kernel is an HBM stream of W.  Tiles are v_mfma_f32_16x16x32_{bf16,f16} with
// 16 weight rows as the MFMA's M dimension and the (padded) token rows as its
// N dimension, so the MFMA's output tile is 16 weight rows x 16 tokens.
//
// A workgroup (4 or 8 waves) owns 16 to 32 weight rows and one K slice; wave w
// takes k-steps (of 32) in groups of GU consecutive steps, round-robin over
// the waves, so within a round the waves read GU * 64 contiguous bytes of every
// row each.  Per round a lane issues all of its loads (GU weight fragments of
// every row tile, GU token fragments) before the first MFMA.  The waves'
// partial tiles are summed in LDS.  With one K slice the workgroup adds the
// bias and writes y; with several (split-K, for tall-K shapes that would
// otherwise give too few workgroups) it writes partials and
// the last workgroup of each row tile to arrive sums them in slice order
// (deterministic), adds the bias and rounds: tagged partial words and an arrival
// counter per tile (arrive.h), so the launch needs no second kernel
// (HS_GEMM_FUSED_MERGE=0: fp32 partials summed the same way by
// gemm_finalize_kernel, a second launch).  The argmax form (the LM head of a greedy step) keeps, per
// workgroup and token, only the best rounded logit and its index as one ordered
// 64-bit key, and argmax_finalize_kernel takes the largest key per token.
#include <math.h>
#include <stdlib.h>

#include "arrive.h"
#include "hs_common.h"

namespace hs {

constexpr int GM_T = 256;  // threads per workgroup of gemm_finalize_kernel
constexpr int GM_SLICES = 8;  // most K slices of a plan

template <int DT>
__device__ __forceinline__ f32x4 gemm_mfma(u32x4 a, u32x4 b, f32x4 c) {
  if constexpr (DT == HS_DTYPE_BF16) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c,
                                                   0, 0, 0);
  } else {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0,
                                                  0, 0);
  }
}

struct GemmArgs {
  const unsigned short* x;
  int64_t x_stride;
  const unsigned short* w;
  int64_t K, N, M;
  const unsigned short* bias;  // nullable
  void* out;
  int64_t out_stride;
  float* part;  // [splits, M, N] when splits > 1
  int64_t splits, slice_steps;
  int64_t rows;  // WINDOW: weight rows of a workgroup
  int64_t F;  // SWIGLU: output features (N = 2 * 16 * ceil(F / 16) interleaved weight rows)
  unsigned long long* keys;  // ARGMAX: [M, gridDim.x] best key per token and workgroup
  // split-K merged in-kernel (epoch != 0): tagged partial words [splits, M, N] and one
  // arrival counter per row tile
  unsigned long long* words;
  unsigned long long* counters;
  unsigned long long epoch;
};

// Ordered key of logit v at vocabulary index n: a larger key is a larger value, or
// the same value at a smaller index, so the largest key is torch.argmax's answer
// (the first maximal index).  -0 counts as +0 (they compare equal); a NaN sits
// above every number (torch's argmax returns the first NaN).  Every key is above
// 0, the key of "no row".
__device__ __forceinline__ unsigned long long argmax_key(float v, int64_t n) {
  const uint32_t u = v == 0.f ? 0u : __float_as_uint(v);
  uint32_t ord = (u & 0x80000000u) ? ~u : (u | 0x80000000u);
  if (v != v) ord = 0xffffffffu;
  return (static_cast<unsigned long long>(ord) << 32) | (0xffffffffu - static_cast<uint32_t>(n));
}

template <int DT>
__device__ __forceinline__ float gemm_round(float v) {
  if constexpr (DT == HS_DTYPE_BF16) return bf16_bits_to_f32(f32_to_bf16_bits(v));
  else return f16_bits_to_f32(f32_to_f16_bits(v));
}

// GM_TILES row tiles of 16 per workgroup, shared by its NW waves, which split
// the slice's k-steps in rounds of GU.  (Measured on MI355X: splitting rows
// over the waves instead, or double-buffering the rounds in registers, is
// slower at every decode shape of the Qwen2.5 0.5B/7B/32B projections.)
// TILED: W is stored tile-major, [ceil(N/16)][K/32][16][32] (each 16-row x 32-k
// block of MFMA A fragments contiguous, rows past N zero-padded), so one wave's
// load of a block reads 1 KB of consecutive bytes instead of 16 rows x 64 bytes
// a row stride apart.
// SWIGLU (with TILED and two tiles per workgroup): the weight interleaves the
// gate and up projections tile by tile (tile 2i = gate rows 16i.., 2i+1 = up rows
// 16i..), and the workgroup writes silu(gate) * up for its 16 features with the
// arithmetic of the separate path: each projection rounded to the dtype, then
// SiLU rounded, then the product (hs_silu_mul).
// ARGMAX (one K slice): per token the workgroup's best key over its rows, each
// logit rounded to the dtype after the bias as the plain form stores it.
// WINDOW: the workgroup's a.rows weight rows start anywhere in its first tile (plan_gemm).
template <int DT, int GM_TILES, int NW, bool TILED, bool NT, bool SWIGLU = false, bool ARGMAX = false, bool WINDOW = false>
__global__ __launch_bounds__(64 * NW) void skinny_gemm_kernel(GemmArgs a) {
  constexpr int GU = 8;  // k-steps of a wave's round
  constexpr int GM_T = 64 * NW;
  constexpr int GM_ROWS = 16 * GM_TILES;  // weight rows of the workgroup's tiles
  __shared__ float red[NW][GM_ROWS][17];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int c = lane & 15, j = lane >> 4;
  // weight rows n0 .. n1, in the tiles from nb
  const int64_t n0 = static_cast<int64_t>(blockIdx.x) * (WINDOW ? a.rows : GM_ROWS);
  const int64_t nb = WINDOW ? n0 & ~static_cast<int64_t>(15) : n0;
  const int64_t n1 = WINDOW && n0 + a.rows < a.N ? n0 + a.rows : a.N;
  auto dropped = [&](int64_t n) -> bool { return n >= n1 || (WINDOW && n < n0); };
  const int64_t split = blockIdx.y;
  const int64_t steps = a.K / 32;
  const int64_t s0 = split * a.slice_steps;
  int64_t s1 = s0 + a.slice_steps;
  if (s1 > steps) s1 = steps;
  // lane (c, j): weight rows nb + 16t + c, token row c, k offset 8j within a step
  const unsigned short* wrow[GM_TILES];
#pragma unroll
  for (int t = 0; t < GM_TILES; ++t) {
    if constexpr (WINDOW) {
      // a lane outside the rows reads the first or the last one again, a tile past them the
      // last tile (no more bytes of the weight); their outputs are dropped
      const int64_t last = (n1 - 1) >> 4;
      const int64_t nt = (nb >> 4) + t < last ? (nb >> 4) + t : last;
      const int lo = n0 > 16 * nt ? static_cast<int>(n0 - 16 * nt) : 0;
      const int hi = n1 - 1 - 16 * nt < 15 ? static_cast<int>(n1 - 1 - 16 * nt) : 15;
      const int row = c < lo ? lo : c > hi ? hi : c;
      wrow[t] = TILED ? a.w + nt * steps * 512 + row * 32 + 8 * j : a.w + (16 * nt + row) * a.K + 8 * j;
    } else if constexpr (TILED) {
      const int64_t tiles = (a.N + 15) / 16;
      int64_t nt = n0 / 16 + t;
      if (nt >= tiles) nt = tiles - 1;  // tiles past N read the last one; their outputs are dropped
      wrow[t] = a.w + nt * steps * 512 + c * 32 + 8 * j;
    } else {
      int64_t n = n0 + 16 * t + c;
      if (n >= a.N) n = a.N - 1;  // rows past N read the last row; their outputs are dropped
      wrow[t] = a.w + n * a.K + 8 * j;
    }
  }
  const unsigned short* xrow = a.x + (c < a.M ? c : a.M - 1) * a.x_stride + 8 * j;
  // the tile's arrival counter, read with the first loads: its round tags the partials
  const unsigned long long c0 = (a.splits > 1 && a.epoch != 0)
                                    ? __hip_atomic_load(a.counters + blockIdx.x, __ATOMIC_RELAXED,
                                                        __HIP_MEMORY_SCOPE_AGENT)
                                    : 0ull;
  f32x4 acc[GM_TILES];
#pragma unroll
  for (int t = 0; t < GM_TILES; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int64_t base = s0 + static_cast<int64_t>(wave) * GU; base < s1; base += NW * GU) {
    // every load of the round before the first MFMA; steps past the slice
    // reload its last step (in bounds) and are skipped
    u32x4 wf[GU][GM_TILES], xf[GU];
#pragma unroll
    for (int u = 0; u < GU; ++u) {
      int64_t s = base + u;
      if (s >= s1) s = s1 - 1;
      const int64_t k = 32 * s;                   // x is row-major
      const int64_t wk = TILED ? 512 * s : k;      // a 16 x 32 block per k-step when tiled
#pragma unroll
      for (int t = 0; t < GM_TILES; ++t) {
        const u32x4* at = reinterpret_cast<const u32x4*>(wrow[t] + wk);
        wf[u][t] = NT ? __builtin_nontemporal_load(at) : *at;
      }
      xf[u] = *reinterpret_cast<const u32x4*>(xrow + k);
    }
#pragma unroll
    for (int u = 0; u < GU; ++u) {
      if (base + u < s1) {  // uniform per wave
#pragma unroll
        for (int t = 0; t < GM_TILES; ++t) acc[t] = gemm_mfma<DT>(wf[u][t], xf[u], acc[t]);
      }
    }
  }
  // lane holds C[row 16t + 4j + i][token c]; the waves' partials summed in wave order
#pragma unroll
  for (int t = 0; t < GM_TILES; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) red[wave][16 * t + 4 * j + i][c] = acc[t][i];
  __syncthreads();
  auto sum_of = [&](int r, int m) -> float {
    float v = red[0][r][m];
#pragma unroll
    for (int w = 1; w < NW; ++w) v += red[w][r][m];
    return v;
  };
  if constexpr (SWIGLU) {
    static_assert(TILED && GM_TILES == 2, "the fused gate/up product takes a gate tile and an up tile");
    for (int idx = threadIdx.x; idx < 16 * 16; idx += GM_T) {
      const int r = idx >> 4, m = idx & 15;
      const int64_t f = static_cast<int64_t>(blockIdx.x) * 16 + r;
      if (m >= a.M || f >= a.F) continue;
      const float g = gemm_round<DT>(sum_of(r, m) + 0.f);
      const float u = gemm_round<DT>(sum_of(16 + r, m) + 0.f);
      const float act = gemm_round<DT>(g / (1.f + expf(-g)));
      store_elem<DT>(a.out, m * a.out_stride + f, act * u);
    }
    return;
  }
  if constexpr (ARGMAX) {
    __shared__ unsigned long long best[GM_ROWS][16];
    for (int idx = threadIdx.x; idx < GM_ROWS * 16; idx += GM_T) {
      const int r = idx >> 4, m = idx & 15;
      const int64_t n = nb + r;
      unsigned long long key = 0;
      if (!dropped(n)) {
        const float b = a.bias != nullptr ? load_elem<DT>(a.bias, n) : 0.f;
        key = argmax_key(gemm_round<DT>(sum_of(r, m) + b), n);
      }
      best[r][m] = key;
    }
    __syncthreads();
    if (threadIdx.x < a.M) {
      const int m = threadIdx.x;
      unsigned long long key = 0;
      for (int r = 0; r < GM_ROWS; ++r) key = best[r][m] > key ? best[r][m] : key;
      a.keys[static_cast<int64_t>(m) * gridDim.x + blockIdx.x] = key;
    }
    return;
  }
  if (a.splits > 1 && a.epoch != 0) {
    // this slice's partial words, then the arrival; the tile's last workgroup sums
    // every slice's word in slice order (reading again a word whose tag has not
    // landed yet), adds the bias, rounds, and leaves the counter to the next round
    const uint32_t round = counter_round(c0, a.epoch);
    const uint32_t tag = group_tag(a.epoch, round);
    for (int idx = threadIdx.x; idx < GM_ROWS * 16; idx += GM_T) {
      const int r = idx >> 4, m = idx & 15;
      const int64_t n = nb + r;
      if (m >= a.M || dropped(n)) continue;
      store_partial(a.words + (split * a.M + m) * a.N + n, sum_of(r, m), tag);
    }
    __shared__ int s_last;
    __syncthreads();
    if (threadIdx.x == 0) s_last = arrive_last(a.counters + blockIdx.x, c0, a.epoch, a.splits) ? 1 : 0;
    __syncthreads();
    if (!s_last) return;
    const int64_t sstride = a.M * a.N;
    for (int idx = threadIdx.x; idx < GM_ROWS * 16; idx += GM_T) {
      const int r = idx >> 4, m = idx & 15;
      const int64_t n = nb + r;
      if (m >= a.M || dropped(n)) continue;
      const unsigned long long* w0 = a.words + m * a.N + n;
      float v = 0.f;
      unsigned long long w[GM_SLICES];  // every slice's word, loaded together
#pragma unroll
      for (int u = 0; u < GM_SLICES; ++u)
        if (u < a.splits)
          w[u] = __hip_atomic_load(w0 + u * sstride, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
      for (int u = 0; u < GM_SLICES; ++u) {
        if (u >= a.splits) break;
        if (static_cast<uint32_t>(w[u] >> 32) != tag) w[u] = partial_reread(w0 + u * sstride, tag);
        v += partial_value(w[u]);
      }
      const float b = a.bias != nullptr ? load_elem<DT>(a.bias, n) : 0.f;
      store_elem<DT>(a.out, m * a.out_stride + n, v + b);
    }
    if (threadIdx.x == 0)
      __hip_atomic_store(a.counters + blockIdx.x,
                         (static_cast<unsigned long long>(counter_id(a.epoch)) << 32) |
                             (static_cast<unsigned long long>((round + 1) & 0xffffu) << 16),
                         __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return;
  }
  for (int idx = threadIdx.x; idx < GM_ROWS * 16; idx += GM_T) {
    const int r = idx >> 4, m = idx & 15;
    const int64_t n = nb + r;
    if (m >= a.M || dropped(n)) continue;
    const float v = sum_of(r, m);
    if (a.splits > 1) {
      a.part[(split * a.M + m) * a.N + n] = v;
    } else {
      const float b = a.bias != nullptr ? load_elem<DT>(a.bias, n) : 0.f;
      store_elem<DT>(a.out, m * a.out_stride + n, v + b);
    }
  }
}

template <int DT>
__global__ __launch_bounds__(GM_T) void gemm_finalize_kernel(const float* part, int64_t splits, int64_t M, int64_t N,
                                                             const unsigned short* bias, void* out,
                                                             int64_t out_stride) {
  const int64_t idx = static_cast<int64_t>(blockIdx.x) * GM_T + threadIdx.x;
  if (idx >= M * N) return;
  const int64_t m = idx / N, n = idx - m * N;
  float v = 0.f;
  for (int64_t s = 0; s < splits; ++s) v += part[(s * M + m) * N + n];
  if (bias != nullptr) v += load_elem<DT>(bias, n);
  store_elem<DT>(out, m * out_stride + n, v);
}

// One workgroup per token: the largest of its `blocks` keys, as the vocabulary index.
// Bound by the round trips of its loads: FIN_KEYS keys per thread are loaded together
// (4752 keys a token: 4.8 us, 9.2 us with 256 threads of one load at a time).  Up to 1024
// keys take 256 threads, whose fewer waves start and meet sooner, and up to 256 one load each
// (16 keys, with the product of 256 x 128: 5.1 us with 1024 threads, 4.8 with 256 of 8 loads,
// 4.7 with 256 of one).
template <int FIN_T, int FIN_KEYS>
__global__ __launch_bounds__(FIN_T) void argmax_finalize_kernel(const unsigned long long* keys, int64_t blocks,
                                                                int64_t* tokens) {
  __shared__ unsigned long long wave_best[FIN_T / 64];
  const int64_t m = blockIdx.x;
  unsigned long long key = 0;
  for (int64_t b0 = threadIdx.x; b0 < blocks; b0 += FIN_T * FIN_KEYS) {
    unsigned long long v[FIN_KEYS];
#pragma unroll
    for (int i = 0; i < FIN_KEYS; ++i) {
      const int64_t b = b0 + i * FIN_T;
      v[i] = keys[m * blocks + (b < blocks ? b : b0)];
    }
#pragma unroll
    for (int i = 0; i < FIN_KEYS; ++i) key = v[i] > key ? v[i] : key;
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const unsigned long long o = __shfl_xor(key, off, 64);
    key = o > key ? o : key;
  }
  if ((threadIdx.x & 63) == 0) wave_best[threadIdx.x >> 6] = key;
  __syncthreads();
  if (threadIdx.x == 0) {
#pragma unroll
    for (int w = 1; w < FIN_T / 64; ++w) key = wave_best[w] > key ? wave_best[w] : key;
    tokens[m] = static_cast<int64_t>(0xffffffffu - static_cast<uint32_t>(key));
  }
}

struct GemmPlan {
  int tiles, waves;
  bool stream;  // non-temporal weight loads
  int64_t rows;  // weight rows per workgroup where they cross tile edges, else 0
  int64_t blocks, splits, slice_steps;
};

static int64_t gemm_ceil(int64_t a, int64_t b) { return (a + b - 1) / b; }

// Waves of a workgroup: 8 where a wave of 4 would read its k-steps in more than one round
// (each round is a memory round trip, and a CU with one workgroup has only its own waves'
// loads in flight), unless there are so many rows that every CU holds several workgroups
// (then only for a long K).
// 8 rows, us with 4 and with 8 waves: 3584 x 3584 9.8 and 8.5, 896 x 4864 10.5 and 8.3,
// 3584 x 18944 39.4 and 30.0; 1152 x 896 (7 steps a wave of 4) 3.60 and 3.65; 12288 x
// 1536 9.3 and 10.9, 12288 x 3584, one row, 17.2 and 18.1.  The same for a projection in one K slice and its fused forms,
// so their sums agree.
static int gemm_waves(int64_t N, int64_t slice_steps) {
  return slice_steps > 32 && (N <= 8192 || (slice_steps > 112 && N <= 16384)) ? 8 : 4;
}

// Row tiles of 16 per workgroup and K slices.  The weight's stream bounds the launch, a CU
// reads about 23 bytes per ns, and the launch ends with the CU that reads most: the cost of
// a plan is the rounds of its workgroups over the 256 CUs times a workgroup's tile-steps
// (1 KB each) and its x reads: 1/20 tile-step per token row and step, of which a second tile
// has no more.  A second tile costs about 28 tile-steps (over 1 us of loads, LDS sums and stores)
// whatever K is.  Merging K slices costs about 48 (2 us), and pays only within one round or for
// long slices; more than three only while each keeps 80 k-steps (few rows of a long K).  The
// slices are chosen without the token rows (an eighth of the tile-steps for one tile's x, no
// charge for the second), so a row's sums are the same in every batch.
// Measured, 8 rows, us with at least 512 workgroups of 4 waves (one tile up to 16384 rows) and
// with these plans: 3584 x 18944 34.2 and 28.5 (two tiles in two slices instead of one in
// three), 7168 x 5120 21.6 and 15.7, 5120 x 27648 64.9 and 53.3 (two tiles in three slices),
// 896 x 4864 9.6 and 7.5 (three slices); without the second tile's share 8192 x 512 takes two
// tiles, 4.4 and 5.1, with it one, 4.4; with at most three slices 16 x 27648 12.0 instead of
// 8.1, with eight 7.5.  The argmax of 152064 x 896, one tile and two: 42.7 and 46.0 for one token
// row, 51.3 and 47.5 for 8, 66.2 and 52.7 for 16.
static GemmPlan plan_gemm(int64_t rows, int64_t N, int64_t K, bool one_slice = false) {
  // unsigned, with constant divisors: every projection call plans, on the host's time
  constexpr uint64_t CUS = 256, X_SHARE = 8, X_ROWS = 20, TILE2 = 28, MERGE = 48, LONG_SLICE = 256, MORE_SLICES = 80;
  const uint64_t M = static_cast<uint64_t>(rows), steps = static_cast<uint64_t>(K) / 32;
  const uint64_t n[2] = {(static_cast<uint64_t>(N) + 15) / 16, (static_cast<uint64_t>(N) + 31) / 32};
  const uint64_t slices[GM_SLICES] = {steps, (steps + 1) / 2, (steps + 2) / 3, (steps + 3) / 4, (steps + 4) / 5,
                                      (steps + 5) / 6, (steps + 6) / 7, (steps + 7) / 8};
  // the tile-steps of the busiest CU
  auto stream_of = [&](uint64_t s, uint64_t tiles) { return (n[tiles - 1] * s + CUS - 1) / CUS * slices[s - 1] * tiles; };
  auto sliced = [&](uint64_t s, uint64_t tiles) { return s == 1 || n[tiles - 1] * s <= CUS || slices[s - 1] >= LONG_SLICE; };
  uint64_t splits = 1, best = UINT64_MAX;
  for (uint64_t s = 1; s <= (one_slice ? 1 : GM_SLICES); ++s) {
    const uint64_t slice = slices[s - 1];
    if (slice * (s - 1) >= steps || (s > 3 && slice < MORE_SLICES)) break;  // one would be empty, or too short
    for (uint64_t tiles = s > 3 ? 1 : 2; tiles >= 1; --tiles) {
      if (!sliced(s, tiles)) continue;
      const uint64_t stream = stream_of(s, tiles);
      const uint64_t cost = stream + (tiles == 1 ? stream / X_SHARE : 0) + (s > 1 ? MERGE : 0);
      if (cost >= best) continue;
      best = cost;
      splits = s;
    }
  }
  // Where two tiles per workgroup leave CUs idle (4096 < N <= 6144), the rows are dealt evenly
  // instead: an even count (two are a 128-byte line of a k-step) of 18, 20 or 24, which two
  // tiles hold wherever it starts.  us, two whole tiles and this, 8 rows (16 rows): 4608 x 3584
  // 12.2 and 10.3 (14.2 and 12.2), 5120 x 5120 15.9 and 13.6 (19.2 and 16.9), 6144 x 4096 13.2
  // and 12.6 (15.9 and 14.5).  Fewer rows than a tile's, or two rounds, do not pay: the second
  // tile's loads cost more than the bytes they leave out (3584 x 3584 in one tile 8.0, in
  // 14 rows of two 9.7; 9216 x 4096 19.0 and 20.7), so they are charged 44 here, which leaves
  // a short K to one tile (5120 x 512 4.2, even rows 4.9; 4608 x 1024 5.2 and 5.5).  Longer
  // K stays in slices: 5120 x 27648 in three 50.1, in 20 rows 53.3 (but 4608 x 18944, here two
  // whole tiles and one slice, 41.0 and in 18 rows 36.1).
  constexpr uint64_t EVEN = 44;
  uint64_t even = 2 * ((static_cast<uint64_t>(N) + 2 * CUS - 1) / (2 * CUS));
  if (even == 22) even = 24;  // starts at multiples of 2: 22 rows could touch a third tile
  const bool dealt = !one_slice && even > 16 && even <= 24 && steps <= 2 * LONG_SLICE;
  if (dealt && steps * even / 16 < best) splits = 1;
  GemmPlan p{};
  p.splits = static_cast<int64_t>(splits);
  p.slice_steps = static_cast<int64_t>(slices[splits - 1]);
  // Many rows of a short K in two tiles as long as all of these workgroups run at once: 20480 x 128
  // in one tile 5.9 us, in two 5.0; 27648 x 128 6.2 and 7.4
  const bool two_tiles = N > 16384 && n[1] <= 3 * CUS && steps <= 16;
  best = UINT64_MAX;
  for (uint64_t tiles = 2; tiles >= (two_tiles ? 2u : 1u); --tiles) {
    if (!sliced(splits, tiles)) continue;
    const uint64_t stream = stream_of(splits, tiles);
    const uint64_t cost = stream + stream * M / (X_ROWS * tiles) + (tiles == 2 ? TILE2 : 0);
    if (cost >= best) continue;
    best = cost;
    p.tiles = static_cast<int>(tiles);
    p.blocks = static_cast<int64_t>(n[tiles - 1]);
  }
  if (dealt && splits == 1 && steps * even / 16 + steps * M / X_ROWS + EVEN < best) {
    p.tiles = 2;
    p.rows = static_cast<int64_t>(even);
    p.blocks = gemm_ceil(N, p.rows);
  }
  p.waves = gemm_waves(N, p.slice_steps);
  // A weight is read once per step.  Above the 4 MB of an XCD's L2 nothing of it is left
  // for the next step, and keeping it costs: 2 x 18944 x 3584 52.4 us, non-temporal 48.2;
  // 3584 x 18944 30.0 and 28.9; 896 x 4864 8.3 and 8.1.  Below, it may still be in a cache:
  // 1152 x 896 (2 MB) 3.6 us, non-temporal 3.8.
  p.stream = N * K * 2 > (4 << 20);
  return p;
}

template <int DT, int TILES, bool TILED, bool NT, bool ARGMAX>
static void launch_gemm_waves(const GemmPlan& p, dim3 grid, const GemmArgs& a, hipStream_t s) {
  if (p.waves == 8) hipLaunchKernelGGL((skinny_gemm_kernel<DT, TILES, 8, TILED, NT, false, ARGMAX>), grid, dim3(512), 0, s, a);
  else hipLaunchKernelGGL((skinny_gemm_kernel<DT, TILES, 4, TILED, NT, false, ARGMAX>), grid, dim3(256), 0, s, a);
}

template <int DT, bool TILED, bool NT, bool ARGMAX>
static void launch_gemm_tiles(const GemmPlan& p, dim3 grid, const GemmArgs& a, hipStream_t s) {
  if constexpr (!ARGMAX) {
    if (p.rows > 0) {
      if (p.waves == 8) hipLaunchKernelGGL((skinny_gemm_kernel<DT, 2, 8, TILED, NT, false, false, true>), grid, dim3(512), 0, s, a);
      else hipLaunchKernelGGL((skinny_gemm_kernel<DT, 2, 4, TILED, NT, false, false, true>), grid, dim3(256), 0, s, a);
      return;
    }
  }
  if (p.tiles == 1) launch_gemm_waves<DT, 1, TILED, NT, ARGMAX>(p, grid, a, s);
  else launch_gemm_waves<DT, 2, TILED, NT, ARGMAX>(p, grid, a, s);
}

template <int DT, bool TILED, bool ARGMAX = false>
static void launch_gemm(const GemmPlan& p, dim3 grid, const GemmArgs& a, hipStream_t s) {
  if constexpr (TILED) {  // a row-major weight's loads take half lines: the other half is read later
    if (p.stream) return launch_gemm_tiles<DT, TILED, true, ARGMAX>(p, grid, a, s);
  }
  launch_gemm_tiles<DT, TILED, false, ARGMAX>(p, grid, a, s);
}

template <int DT>
static void launch_swiglu(const GemmPlan& p, dim3 grid, const GemmArgs& a, hipStream_t s) {
  if (p.waves == 8) {
    if (p.stream) hipLaunchKernelGGL((skinny_gemm_kernel<DT, 2, 8, true, true, true>), grid, dim3(512), 0, s, a);
    else hipLaunchKernelGGL((skinny_gemm_kernel<DT, 2, 8, true, false, true>), grid, dim3(512), 0, s, a);
  } else {
    if (p.stream) hipLaunchKernelGGL((skinny_gemm_kernel<DT, 2, 4, true, true, true>), grid, dim3(256), 0, s, a);
    else hipLaunchKernelGGL((skinny_gemm_kernel<DT, 2, 4, true, false, true>), grid, dim3(256), 0, s, a);
  }
}

}  // namespace hs

using namespace hs;

extern "C" int64_t hs_skinny_gemm_workspace_bytes(int64_t rows, int64_t n, int64_t k) {
  if (rows < 1 || n < 1 || k < 32) return 256;
  const GemmPlan p = plan_gemm(rows, n, k);
  // tagged 64-bit partial words and a counter per row tile (the fp32 partials of the
  // two-launch form fit in the same bytes)
  return p.splits > 1 ? p.splits * rows * n * 8 + p.blocks * 8 + 256 : 256;
}

static int run_gemm(const void* x, int64_t x_stride, const void* weight, int64_t n, int64_t k, const void* bias,
                    void* out, int64_t out_stride, int64_t rows, int32_t dtype, void* workspace,
                    int64_t workspace_bytes, hipStream_t stream, bool tiled) {
  HS_CHECK_ARG(dtype == HS_DTYPE_BF16 || dtype == HS_DTYPE_F16, "the decode GEMM takes bf16 or f16");
  HS_CHECK_ARG(rows >= 1 && rows <= 16, "the decode GEMM takes 1 to 16 rows");
  HS_CHECK_ARG(n >= 1 && k >= 32 && k % 32 == 0, "K must be a positive multiple of 32");
  HS_CHECK_ARG(x_stride >= k && x_stride % 8 == 0 && out_stride >= n, "invalid row strides");
  HS_CHECK_ARG(x && weight && out, "null GEMM pointer");
  HS_CHECK_ARG((reinterpret_cast<uintptr_t>(x) & 15) == 0 && (reinterpret_cast<uintptr_t>(weight) & 15) == 0,
               "x and weight must be 16-byte aligned");
  const GemmPlan p = plan_gemm(rows, n, k);
  HS_CHECK_ARG(p.blocks <= 0x7fffffff && p.splits <= 65535, "GEMM too large");
  GemmArgs a{};
  a.x = static_cast<const unsigned short*>(x);
  a.x_stride = x_stride;
  a.w = static_cast<const unsigned short*>(weight);
  a.K = k;
  a.N = n;
  a.M = rows;
  a.bias = static_cast<const unsigned short*>(bias);
  a.out = out;
  a.out_stride = out_stride;
  a.splits = p.splits;
  a.rows = p.rows;
  a.slice_steps = p.slice_steps;
  bool fused = true;
  if (p.splits > 1) {
    // the split-K partials merged in-kernel unless HS_GEMM_FUSED_MERGE=0 (read per call)
    const char* fused_env = getenv("HS_GEMM_FUSED_MERGE");
    fused = !(fused_env && atoi(fused_env) == 0);
    const int64_t need = fused ? p.splits * rows * n * 8 + p.blocks * 8 : p.splits * rows * n * 4;
    HS_CHECK_ARG(workspace != nullptr && workspace_bytes >= need && (reinterpret_cast<uintptr_t>(workspace) & 7) == 0,
                 "GEMM workspace too small or misaligned: need %lld bytes", static_cast<long long>(need));
    if (fused) {
      a.words = static_cast<unsigned long long*>(workspace);
      a.counters = a.words + p.splits * rows * n;
      a.epoch = next_epoch();
    } else {
      a.part = static_cast<float*>(workspace);
    }
  }
  const dim3 grid(static_cast<unsigned>(p.blocks), static_cast<unsigned>(p.splits));
  if (dtype == HS_DTYPE_BF16) {
    if (tiled) launch_gemm<HS_DTYPE_BF16, true>(p, grid, a, stream);
    else launch_gemm<HS_DTYPE_BF16, false>(p, grid, a, stream);
  } else {
    if (tiled) launch_gemm<HS_DTYPE_F16, true>(p, grid, a, stream);
    else launch_gemm<HS_DTYPE_F16, false>(p, grid, a, stream);
  }
  HS_CHECK_LAUNCH("skinny GEMM");
  if (p.splits > 1 && !fused) {
    const unsigned blocks = static_cast<unsigned>(gemm_ceil(rows * n, GM_T));
    if (dtype == HS_DTYPE_BF16)
      hipLaunchKernelGGL((gemm_finalize_kernel<HS_DTYPE_BF16>), dim3(blocks), dim3(GM_T), 0, stream, a.part, p.splits,
                         rows, n, a.bias, out, out_stride);
    else
      hipLaunchKernelGGL((gemm_finalize_kernel<HS_DTYPE_F16>), dim3(blocks), dim3(GM_T), 0, stream, a.part, p.splits,
                         rows, n, a.bias, out, out_stride);
    HS_CHECK_LAUNCH("skinny GEMM finalize");
  }
  return HS_OK;
}

extern "C" int hs_skinny_gemm(const void* x, int64_t x_stride, const void* weight, int64_t n, int64_t k,
                              const void* bias, void* out, int64_t out_stride, int64_t rows, int32_t dtype,
                              void* workspace, int64_t workspace_bytes, hipStream_t stream) {
  return run_gemm(x, x_stride, weight, n, k, bias, out, out_stride, rows, dtype, workspace, workspace_bytes, stream,
                  false);
}

extern "C" int hs_skinny_gemm_tiled(const void* x, int64_t x_stride, const void* weight_tiles, int64_t n, int64_t k,
                                    const void* bias, void* out, int64_t out_stride, int64_t rows, int32_t dtype,
                                    void* workspace, int64_t workspace_bytes, hipStream_t stream) {
  return run_gemm(x, x_stride, weight_tiles, n, k, bias, out, out_stride, rows, dtype, workspace, workspace_bytes,
                  stream, true);
}

extern "C" int hs_skinny_gemm_swiglu_tiled(const void* x, int64_t x_stride, const void* gate_up_tiles, int64_t ffn,
                                           int64_t k, void* out, int64_t out_stride, int64_t rows, int32_t dtype,
                                           hipStream_t stream) {
  HS_CHECK_ARG(dtype == HS_DTYPE_BF16 || dtype == HS_DTYPE_F16, "the decode GEMM takes bf16 or f16");
  HS_CHECK_ARG(rows >= 1 && rows <= 16, "the decode GEMM takes 1 to 16 rows");
  HS_CHECK_ARG(ffn >= 1 && k >= 32 && k % 32 == 0, "K must be a positive multiple of 32");
  HS_CHECK_ARG(x_stride >= k && x_stride % 8 == 0 && out_stride >= ffn, "invalid row strides");
  HS_CHECK_ARG(x && gate_up_tiles && out, "null GEMM pointer");
  HS_CHECK_ARG((reinterpret_cast<uintptr_t>(x) & 15) == 0 && (reinterpret_cast<uintptr_t>(gate_up_tiles) & 15) == 0,
               "x and weight must be 16-byte aligned");
  const int64_t blocks = gemm_ceil(ffn, 16);
  HS_CHECK_ARG(blocks <= 0x7fffffff, "GEMM too large");
  GemmArgs a{};
  a.x = static_cast<const unsigned short*>(x);
  a.x_stride = x_stride;
  a.w = static_cast<const unsigned short*>(gate_up_tiles);
  a.K = k;
  a.N = 2 * 16 * blocks;  // interleaved weight rows, padded
  a.M = rows;
  a.out = out;
  a.out_stride = out_stride;
  a.splits = 1;  // one K slice: the workgroup sees whole sums before the product
  a.slice_steps = k / 32;
  a.F = ffn;
  const dim3 grid(static_cast<unsigned>(blocks));
  const GemmPlan p = plan_gemm(rows, 2 * ffn, k, true);  // the plain projection's waves
  if (dtype == HS_DTYPE_BF16) launch_swiglu<HS_DTYPE_BF16>(p, grid, a, stream);
  else launch_swiglu<HS_DTYPE_F16>(p, grid, a, stream);
  HS_CHECK_LAUNCH("skinny GEMM swiglu");
  return HS_OK;
}

extern "C" int64_t hs_skinny_gemm_argmax_workspace_bytes(int64_t rows, int64_t n, int64_t k) {
  if (rows < 1 || n < 1 || k < 32) return 256;
  // one tile per workgroup, the most keys of any row count: a workspace serves fewer rows too, whose
  // plan may have the smaller workgroups
  return gemm_ceil(n, 16) * rows * 8 + 256;
}

extern "C" int hs_skinny_gemm_argmax_tiled(const void* x, int64_t x_stride, const void* weight_tiles, int64_t n,
                                           int64_t k, const void* bias, int64_t* tokens, int64_t rows, int32_t dtype,
                                           void* workspace, int64_t workspace_bytes, hipStream_t stream) {
  HS_CHECK_ARG(dtype == HS_DTYPE_BF16 || dtype == HS_DTYPE_F16, "the decode GEMM takes bf16 or f16");
  HS_CHECK_ARG(rows >= 1 && rows <= 16, "the decode GEMM takes 1 to 16 rows");
  HS_CHECK_ARG(n >= 1 && n <= 0x7fffffff && k >= 32 && k % 32 == 0,
               "n must be in [1, 2^31) and K a positive multiple of 32");
  HS_CHECK_ARG(x_stride >= k && x_stride % 8 == 0, "invalid row stride");
  HS_CHECK_ARG(x && weight_tiles && tokens, "null GEMM pointer");
  HS_CHECK_ARG((reinterpret_cast<uintptr_t>(x) & 15) == 0 && (reinterpret_cast<uintptr_t>(weight_tiles) & 15) == 0,
               "x and weight must be 16-byte aligned");
  const GemmPlan p = plan_gemm(rows, n, k, true);
  HS_CHECK_ARG(p.blocks <= 0x7fffffff, "GEMM too large");
  const int64_t need = p.blocks * rows * 8;
  HS_CHECK_ARG(workspace != nullptr && workspace_bytes >= need && (reinterpret_cast<uintptr_t>(workspace) & 7) == 0,
               "argmax workspace too small or misaligned: need %lld bytes", static_cast<long long>(need));
  GemmArgs a{};
  a.x = static_cast<const unsigned short*>(x);
  a.x_stride = x_stride;
  a.w = static_cast<const unsigned short*>(weight_tiles);
  a.K = k;
  a.N = n;
  a.M = rows;
  a.bias = static_cast<const unsigned short*>(bias);
  a.splits = 1;
  a.slice_steps = p.slice_steps;
  a.keys = static_cast<unsigned long long*>(workspace);
  const dim3 grid(static_cast<unsigned>(p.blocks));
  if (dtype == HS_DTYPE_BF16) launch_gemm<HS_DTYPE_BF16, true, true>(p, grid, a, stream);
  else launch_gemm<HS_DTYPE_F16, true, true>(p, grid, a, stream);
  HS_CHECK_LAUNCH("skinny GEMM argmax");
  const dim3 fin(static_cast<unsigned>(rows));
  auto finalize = [&](auto kernel, unsigned threads) {
    hipLaunchKernelGGL(kernel, fin, dim3(threads), 0, stream, a.keys, p.blocks, tokens);
  };
  if (p.blocks <= 256) finalize(argmax_finalize_kernel<256, 1>, 256);
  else if (p.blocks <= 1024) finalize(argmax_finalize_kernel<256, 4>, 256);
  else finalize(argmax_finalize_kernel<1024, 8>, 1024);
  HS_CHECK_LAUNCH("argmax finalize");
  return HS_OK;
}
