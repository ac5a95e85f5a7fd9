// Quest page scorer, per-head top-k and the device-side union builder for gfx950.
//
// Scorer + top-k replace `quest_selection` (selection.py:80-101): for query
// head h with KV head h // g, page p scores
//     s = sum_d max(q_d * lo_d, q_d * hi_d)
// over the page's K minimum/maximum bounds; the tail page and (optionally)
// page 0 are forced; the `top` best pages per head are kept.  The sum runs over
// d in ascending order with one float32 rounding per step (for 16-bit inputs
// the product is exact, so a fused multiply-add gives the same value); ties
// go to the lower page index.  Since max(q*lo, q*hi) is q*hi for q >= 0 and
// q*lo otherwise (hi >= lo), the kernel selects the bound before multiplying.
//
// The union builder replaces the host adapter Selection -> LogicalTopK
// (row_index.py:20-31, selection.py:43-60): from the chosen pages it writes the
// ascending union of selected tokens (padded with -1), each head's union
// columns, and per KV head the deduplicated union columns its query heads read
// with a bit mask of those heads (the entry lists of the group attention).
#include <algorithm>
#include <stdlib.h>
#include <string.h>

#include "hs_common.h"

namespace hs {

constexpr int QMAXB = 16;       // requests per launch
constexpr int QHEADS = 8;       // query heads per scorer thread
constexpr int QT = 256;         // scorer / top-k threads
constexpr int UT = 1024;        // union builder threads
constexpr int64_t UMAXPAGES = 65536;

struct QuestArgs {
  const void* q;                // [B, Hq, D] in q_dtype (f32, bf16 or f16)
  int q_dtype;
  int64_t q_sb, q_sh;
  const void* kmin[QMAXB];      // per request [pages, Hkv, D]
  const void* kmax[QMAXB];
  int64_t count[QMAXB];         // ceil(length / P)
  int64_t Hq, Hkv, g, D, top;
  int keep_sink;
  float* scores;                // [B, Hq, cmax]
  int64_t cmax;
  int32_t* pages;               // [B, Hq, top]
  int64_t p_sb;
};

// Query element i widened to fp32 (exact for every query dtype).
__device__ __forceinline__ float query_value(const QuestArgs& a, int64_t i) {
  if (a.q_dtype == HS_DTYPE_BF16) return load_elem<HS_DTYPE_BF16>(a.q, i);
  if (a.q_dtype == HS_DTYPE_F16) return load_elem<HS_DTYPE_F16>(a.q, i);
  return load_elem<HS_DTYPE_F32>(a.q, i);
}

template <int DT, bool FUSED>
__global__ __launch_bounds__(QT) void quest_score_kernel(QuestArgs a) {
#pragma clang fp contract(off)
  extern __shared__ float sq[];  // [QHEADS][D]
  const int64_t b = blockIdx.z;
  const int64_t kv = blockIdx.y / ((a.g + QHEADS - 1) / QHEADS);
  const int64_t hc = blockIdx.y % ((a.g + QHEADS - 1) / QHEADS);
  const int64_t count = a.count[b];
  if (a.top >= count) return;
  const int64_t h0 = kv * a.g + hc * QHEADS;
  int64_t nh = a.g - hc * QHEADS;
  if (nh > QHEADS) nh = QHEADS;
  const int64_t D = a.D;
  for (int64_t i = threadIdx.x; i < QHEADS * D; i += QT) {
    const int64_t hl = i / D, d = i - hl * D;
    sq[i] = hl < nh ? query_value(a, b * a.q_sb + (h0 + hl) * a.q_sh + d) : 0.f;
  }
  __syncthreads();
  const int64_t p = static_cast<int64_t>(blockIdx.x) * QT + threadIdx.x;
  if (p >= count) return;
  const int64_t row = (p * a.Hkv + kv) * D;
  const void* lo = a.kmin[b];
  const void* hi = a.kmax[b];
  float acc[QHEADS];
#pragma unroll
  for (int hl = 0; hl < QHEADS; ++hl) acc[hl] = 0.f;
  auto step = [&](int64_t d, float l, float u) {
#pragma unroll
    for (int hl = 0; hl < QHEADS; ++hl) {
      const float qv = sq[hl * D + d];
      const float bound = qv >= 0.f ? u : l;
      if constexpr (FUSED) {
        acc[hl] = __builtin_fmaf(qv, bound, acc[hl]);
      } else {
        const float prod = qv * bound;
        acc[hl] = acc[hl] + prod;
      }
    }
  };
  constexpr int EPV = DT == HS_DTYPE_F32 ? 4 : 8;  // elements per 16-byte load
  const bool vec = (D % EPV) == 0;
  if (vec) {
    for (int64_t d0 = 0; d0 < D; d0 += EPV) {
      const u32x4 L = *reinterpret_cast<const u32x4*>(static_cast<const char*>(lo) + (row + d0) * (DT == HS_DTYPE_F32 ? 4 : 2));
      const u32x4 U = *reinterpret_cast<const u32x4*>(static_cast<const char*>(hi) + (row + d0) * (DT == HS_DTYPE_F32 ? 4 : 2));
#pragma unroll
      for (int e = 0; e < EPV; ++e) {
        float l, u;
        if constexpr (DT == HS_DTYPE_F32) {
          l = __uint_as_float(L[e]);
          u = __uint_as_float(U[e]);
        } else {
          const unsigned short lb = static_cast<unsigned short>(L[e >> 1] >> (16 * (e & 1)));
          const unsigned short ub = static_cast<unsigned short>(U[e >> 1] >> (16 * (e & 1)));
          if constexpr (DT == HS_DTYPE_BF16) {
            l = bf16_bits_to_f32(lb);
            u = bf16_bits_to_f32(ub);
          } else {
            l = f16_bits_to_f32(lb);
            u = f16_bits_to_f32(ub);
          }
        }
        step(d0 + e, l, u);
      }
    }
  } else {
    for (int64_t d = 0; d < D; ++d) step(d, load_elem<DT>(lo, row + d), load_elem<DT>(hi, row + d));
  }
  for (int hl = 0; hl < nh; ++hl) a.scores[(b * a.Hq + h0 + hl) * a.cmax + p] = acc[hl];
}

// LDS-tiled scorer for the common shapes.  One workgroup scores QS_PAGES pages
// of one KV head for a chunk of up to QHEADS query heads.  The pages' lower and
// upper bound rows (D elements each, 2 KB apart in HBM for Hkv = 8, D = 128
// bf16) are staged in LDS with full-line loads (consecutive lanes read
// consecutive 16-byte units, every unit of a fetched line is used); then lane
// l of wave w scores page l for query heads 2w and 2w+1 of the chunk, reading
// its row from LDS (row stride padded by 16 bytes: conflict-free 16-byte
// reads) and the query values as wave-wide broadcasts.  The per-score
// arithmetic is that of quest_score_kernel: d ascending, one float32 rounding
// per step.
constexpr int QS_PAGES = 64;
constexpr int QS_UNITS = 8;                  // 16-byte units per thread per bound
constexpr int64_t QS_MAX_ROW_BYTES = QS_UNITS * QT * 16 / QS_PAGES;  // 512

__host__ __device__ constexpr int64_t qs_lds_bytes(int64_t row_bytes, int64_t D) {
  return 2 * QS_PAGES * (row_bytes + 16) + QHEADS * D * 4;
}

template <int DT, bool FUSED>
__global__ __launch_bounds__(QT) void quest_score_tile_kernel(QuestArgs a) {
#pragma clang fp contract(off)
  extern __shared__ __attribute__((aligned(16))) unsigned char qs_smem[];
  constexpr int ESZ = DT == HS_DTYPE_F32 ? 4 : 2;
  constexpr int EPV = 16 / ESZ;  // elements per 16-byte unit
  const int64_t b = blockIdx.z;
  const int64_t hchunks = (a.g + QHEADS - 1) / QHEADS;
  const int64_t kv = blockIdx.y / hchunks, hc = blockIdx.y - kv * hchunks;
  const int64_t count = a.count[b];
  const int64_t p0 = static_cast<int64_t>(blockIdx.x) * QS_PAGES;
  if (a.top >= count || p0 >= count) return;
  const int64_t D = a.D, Hkv = a.Hkv;
  const int64_t rb = D * ESZ, rs = rb + 16, upr = rb / 16;
  unsigned char* tlo = qs_smem;
  unsigned char* thi = qs_smem + QS_PAGES * rs;
  float* sq = reinterpret_cast<float*>(qs_smem + 2 * QS_PAGES * rs);  // [QHEADS][D]
  int64_t nh = a.g - hc * QHEADS;
  if (nh > QHEADS) nh = QHEADS;
  const int64_t h0 = kv * a.g + hc * QHEADS;
  for (int64_t i = threadIdx.x; i < QHEADS * D; i += QT) {
    const int64_t hl = i / D, d = i - hl * D;
    sq[i] = hl < nh ? query_value(a, b * a.q_sb + (h0 + hl) * a.q_sh + d) : 0.f;
  }
  int64_t npg = count - p0;
  if (npg > QS_PAGES) npg = QS_PAGES;
  const char* lo = static_cast<const char*>(a.kmin[b]);
  const char* hi = static_cast<const char*>(a.kmax[b]);
  // 32-bit tile indexing: at most QS_PAGES * 32 units per bound
  const uint32_t units = static_cast<uint32_t>(npg * upr), upr32 = static_cast<uint32_t>(upr);
  const uint32_t rb32 = static_cast<uint32_t>(rb), rs32 = static_cast<uint32_t>(rs);
  const char* lo_t = lo + (p0 * Hkv + kv) * rb;
  const char* hi_t = hi + (p0 * Hkv + kv) * rb;
  const uint32_t gstride = static_cast<uint32_t>(Hkv) * rb32;  // bytes between consecutive pages
  // every thread issues all of its loads before the first LDS store; a unit
  // past the tile reloads unit 0 (in bounds) and is not stored
  u32x4 L[QS_UNITS], U[QS_UNITS];
#pragma unroll
  for (int k = 0; k < QS_UNITS; ++k) {
    uint32_t u = threadIdx.x + static_cast<uint32_t>(k) * QT;
    if (u >= units) u = 0;
    const uint32_t r = u / upr32, c = u - r * upr32;
    const uint64_t off = static_cast<uint64_t>(r) * gstride + c * 16u;
    L[k] = *reinterpret_cast<const u32x4*>(lo_t + off);
    U[k] = *reinterpret_cast<const u32x4*>(hi_t + off);
  }
#pragma unroll
  for (int k = 0; k < QS_UNITS; ++k) {
    const uint32_t u = threadIdx.x + static_cast<uint32_t>(k) * QT;
    const uint32_t r = u / upr32, c = u - r * upr32;
    if (u < units) {
      *reinterpret_cast<u32x4*>(tlo + r * rs32 + c * 16u) = L[k];
      *reinterpret_cast<u32x4*>(thi + r * rs32 + c * 16u) = U[k];
    }
  }
  __syncthreads();
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int hA = 2 * wave, hB = 2 * wave + 1;
  if (lane >= npg || hA >= nh) return;  // no barrier follows
  const float* qa = sq + hA * D;
  const float* qb = sq + hB * D;
  const unsigned char* rlo = tlo + lane * rs;
  const unsigned char* rhi = thi + lane * rs;
  float accA = 0.f, accB = 0.f;
  auto step = [&](float qv, float l, float u, float& acc) {
    const float bound = qv >= 0.f ? u : l;
    if constexpr (FUSED) {
      acc = __builtin_fmaf(qv, bound, acc);
    } else {
      const float prod = qv * bound;
      acc = acc + prod;
    }
  };
  for (int64_t d0 = 0; d0 < D; d0 += EPV) {
    const u32x4 Lv = *reinterpret_cast<const u32x4*>(rlo + d0 * ESZ);
    const u32x4 Uv = *reinterpret_cast<const u32x4*>(rhi + d0 * ESZ);
#pragma unroll
    for (int e = 0; e < EPV; ++e) {
      float l, u;
      if constexpr (DT == HS_DTYPE_F32) {
        l = __uint_as_float(Lv[e]);
        u = __uint_as_float(Uv[e]);
      } else {
        const unsigned short lb = static_cast<unsigned short>(Lv[e >> 1] >> (16 * (e & 1)));
        const unsigned short ub = static_cast<unsigned short>(Uv[e >> 1] >> (16 * (e & 1)));
        if constexpr (DT == HS_DTYPE_BF16) {
          l = bf16_bits_to_f32(lb);
          u = bf16_bits_to_f32(ub);
        } else {
          l = f16_bits_to_f32(lb);
          u = f16_bits_to_f32(ub);
        }
      }
      step(qa[d0 + e], l, u, accA);
      step(qb[d0 + e], l, u, accB);
    }
  }
  const int64_t p = p0 + lane;
  a.scores[(b * a.Hq + h0 + hA) * a.cmax + p] = accA;
  if (hB < nh) a.scores[(b * a.Hq + h0 + hB) * a.cmax + p] = accB;
}

// Scorer for bf16 bounds with the bound selection taken off the vector ALU.
// For query head h and element d, max(q*lo, q*hi) is q*hi when q >= 0 and q*lo
// otherwise, and that choice is the same for every page a wave scores: each
// wave scores one query head, reads its query words with uniform (scalar) loads
// and turns each sign into a byte selector.  One v_perm_b32 per (page, element)
// then picks the bf16 half of the chosen bound and widens it to fp32 (the bf16
// bits become the high half of the word, the low half zero), leaving one fused
// multiply-add per element for bf16 queries (their product with a bf16 bound is
// exact) and a multiply and an add for fp32 queries.  A query of -0 picks the
// lower bound here and the upper one in quest_score_kernel; both products are
// zeros, and a sum started at +0 is never -0, so adding either zero leaves it
// unchanged.  One workgroup scores QP_PAGES pages of one KV head for a chunk of
// up to QHEADS query heads (wave w: head w, lane l: pages l and l + 64), the
// bound rows staged in LDS as in quest_score_tile_kernel.  The KV head is the fastest grid
// dimension, so the workgroups running together read whole page rows.
// The launch is bound by the bounds' HBM stream: what it needs is loads in flight while
// other waves score.  A 256-byte row (D = 128) is staged in PARTS = 2 halves of 128 bytes,
// so a workgroup holds 36.9 KB of LDS, four share a CU instead of two, and the second
// half's loads are in flight while the first is scored.  16 requests of 8192 pages, 28 heads,
// 4 KV heads (268 MB): 66.2 us with whole rows, 55.4 us in halves (page tiles the fastest grid
// dimension: 54.0).
// NT, non-temporal loads, where one workgroup is the only reader of its lines (rows of whole
// lines, D = 64 or 128, and one head chunk per KV head) and the bounds are too many to be in an
// L2 still: the same 50.7 us = 5.3 TB/s; 8, 4 and 2 requests: 32.0, 19.7 and 13.0 us without,
// 29.4, 18.6 and 12.3 us with.  Elsewhere they cost (us with the top-k of one page, 16 requests of
// 8192 pages, without and with): 32 heads on one KV head, four chunks, 63.8 and 70.4; 8 KV heads
// of D = 32, two rows to a line, 48.8 and 54.7; a megabyte (1 request of 2048 pages, 2 KV heads of
// D = 64) 7.4 and 8.3.  Same arithmetic and order as quest_score_kernel.
constexpr int QP_PAGES = 128;                // pages per workgroup: two per lane
constexpr int QP_T = 64 * QHEADS;            // one wave per query head of the chunk
constexpr int QP_UNITS = 4;                  // 16-byte units per thread, bound and staging round
constexpr int64_t QP_NT_BYTES = 2 << 20;     // least bounds of a launch that are read non-temporally
constexpr int64_t QP_MAX_ROW_BYTES = 256;    // D <= 128: one staging round per part

__host__ __device__ constexpr int64_t qp_lds_bytes(int64_t row_bytes, int parts) {
  return 2 * QP_PAGES * (row_bytes / parts + 16);
}

template <bool QF32, int DK, int PARTS, bool NT>
__global__ __launch_bounds__(QP_T, 4 * PARTS) void quest_score_perm_kernel(QuestArgs a) {
#pragma clang fp contract(off)
  extern __shared__ __attribute__((aligned(16))) unsigned char qp_smem[];
  const int64_t b = blockIdx.z;
  const int64_t hchunks = (a.g + QHEADS - 1) / QHEADS;
  const int64_t kv = blockIdx.x / hchunks, hc = blockIdx.x - kv * hchunks;
  const int64_t count = a.count[b];
  const int64_t p0 = static_cast<int64_t>(blockIdx.y) * QP_PAGES;
  if (a.top >= count || p0 >= count) return;
  const int64_t Hkv = a.Hkv;
  const uint32_t D = DK ? static_cast<uint32_t>(DK) : static_cast<uint32_t>(a.D);
  const uint32_t rb = D * 2u, upr = rb / 16u / PARTS, rs = upr * 16u + 16u;  // units of a row's part, staged row stride
  constexpr int UNITS = QP_UNITS / PARTS;
  unsigned char* tlo = qp_smem;
  unsigned char* thi = qp_smem + QP_PAGES * rs;
  int64_t npg = count - p0;
  if (npg > QP_PAGES) npg = QP_PAGES;
  const uint32_t units = static_cast<uint32_t>(npg) * upr;
  const char* lo_t = static_cast<const char*>(a.kmin[b]) + (p0 * Hkv + kv) * rb;
  const char* hi_t = static_cast<const char*>(a.kmax[b]) + (p0 * Hkv + kv) * rb;
  const uint32_t gstride = static_cast<uint32_t>(Hkv) * rb;  // bytes between consecutive pages
  // one staging round per part (row_bytes <= 256: at most QP_UNITS * QP_T units in all): a
  // thread's loads are issued together; a unit past the tile reloads unit 0 (in bounds) and
  // is not stored
  u32x4 Ls[UNITS], Us[UNITS];
  auto load = [&](int part) {
#pragma unroll
    for (int k = 0; k < UNITS; ++k) {
      uint32_t u = threadIdx.x + static_cast<uint32_t>(k) * QP_T;
      if (u >= units) u = 0;
      const uint32_t r = u / upr, c = u - r * upr;
      const uint64_t off = static_cast<uint64_t>(r) * gstride + (part * upr + c) * 16u;
      const u32x4* lo_at = reinterpret_cast<const u32x4*>(lo_t + off);
      const u32x4* hi_at = reinterpret_cast<const u32x4*>(hi_t + off);
      Ls[k] = NT ? __builtin_nontemporal_load(lo_at) : *lo_at;
      Us[k] = NT ? __builtin_nontemporal_load(hi_at) : *hi_at;
    }
  };
  auto stage = [&]() {
#pragma unroll
    for (int k = 0; k < UNITS; ++k) {
      const uint32_t u = threadIdx.x + static_cast<uint32_t>(k) * QP_T;
      const uint32_t r = u / upr, c = u - r * upr;
      if (u < units) {
        *reinterpret_cast<u32x4*>(tlo + r * rs + c * 16u) = Ls[k];
        *reinterpret_cast<u32x4*>(thi + r * rs + c * 16u) = Us[k];
      }
    }
  };
  load(0);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // uniform: scalar query loads
  int64_t nh = a.g - hc * QHEADS;
  if (nh > QHEADS) nh = QHEADS;
  const int64_t h = kv * a.g + hc * QHEADS + (wave < nh ? wave : 0);
  constexpr int QESZ = QF32 ? 4 : 2;
  constexpr int WPU = QF32 ? 8 : 4;  // query words per 16-byte unit of the bounds (8 elements)
  const uint32_t* qw = reinterpret_cast<const uint32_t*>(static_cast<const char*>(a.q) + (b * a.q_sb + h * a.q_sh) * QESZ);
  const unsigned char* l0 = tlo + lane * rs;
  const unsigned char* l1 = tlo + (lane + 64) * rs;
  const unsigned char* u0 = thi + lane * rs;
  const unsigned char* u1 = thi + (lane + 64) * rs;
  float acc0 = 0.f, acc1 = 0.f;  // pages l and l + 64
  // selector of bound element e (half e & 1 of word e >> 1): bytes 0-3 come from
  // the lower bound's word, 4-7 from the upper's, 0x0c is a zero byte
  auto selector = [](uint32_t qbits, int half) -> uint32_t {
    const bool neg = static_cast<int32_t>(qbits) < 0;
    return half ? (neg ? 0x03020c0cu : 0x07060c0cu) : (neg ? 0x01000c0cu : 0x05040c0cu);
  };
#pragma unroll
  for (int part = 0; part < PARTS; ++part) {
    if (part > 0) __syncthreads();  // every wave has read the part before
    stage();
    if (part + 1 < PARTS) load(part + 1);  // in flight while this part is scored
    __syncthreads();
    if (wave < nh) {
#pragma unroll 2
      for (uint32_t c = 0; c < upr; ++c) {
        const u32x4 L0 = *reinterpret_cast<const u32x4*>(l0 + c * 16u);
        const u32x4 L1 = *reinterpret_cast<const u32x4*>(l1 + c * 16u);
        const u32x4 U0 = *reinterpret_cast<const u32x4*>(u0 + c * 16u);
        const u32x4 U1 = *reinterpret_cast<const u32x4*>(u1 + c * 16u);
        uint32_t wq[WPU];
#pragma unroll
        for (int i = 0; i < WPU; ++i) wq[i] = qw[(part * upr + c) * WPU + i];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const uint32_t qbits = QF32 ? wq[e] : ((e & 1) ? (wq[e >> 1] & 0xffff0000u) : (wq[e >> 1] << 16));
          const float qf = __uint_as_float(qbits);
          const uint32_t sel = selector(qbits, e & 1);
          const float b0 = __uint_as_float(__builtin_amdgcn_perm(U0[e >> 1], L0[e >> 1], sel));
          const float b1 = __uint_as_float(__builtin_amdgcn_perm(U1[e >> 1], L1[e >> 1], sel));
          if constexpr (QF32) {
            const float p0v = qf * b0, p1v = qf * b1;
            acc0 = acc0 + p0v;
            acc1 = acc1 + p1v;
          } else {
            acc0 = __builtin_fmaf(qf, b0, acc0);
            acc1 = __builtin_fmaf(qf, b1, acc1);
          }
        }
      }
    }
  }
  if (wave >= nh) return;
  float* out = a.scores + (b * a.Hq + h) * a.cmax + p0;
  if (lane < npg) out[lane] = acc0;
  if (lane + 64 < npg) out[lane + 64] = acc1;
}

__device__ __forceinline__ uint32_t score_key(float s) {
  if (s == 0.f) s = 0.f;  // -0 and +0 compare equal
  const uint32_t u = __float_as_uint(s);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

// The top keys of one (query head, request) per workgroup, ties to the lower page,
// pages written ascending; the tail page and the sink are always taken.
//
// A thread holds its keys in registers (page j * TT + thread), so the scores are read
// once.  What bounds the launch is its chain of block-wide steps, so there are few: a lower
// bound of the last taken key and the largest key give a range that one histogram of 2048
// equal bins covers (a head's scores crowd into a few powers of two, where fixed top digits
// of the key put most pages into a handful of bins and a lane's LDS atomics behind each
// other's), the bin holding the last taken key is found by one scan from the top, and usually
// holds few keys: they are ranked among themselves.  A bin of more than FEW keys is cut
// into 2048 again; equal keys are ranked by page.  Every wave's taken pages are a ballot, and
// the ballots of (j, wave) follow the pages' order, so one scan of their counts places
// each page.
// The bound: of `need` or more groups of keys, each holds a key at or above the least of the
// groups' largest, so that many keys lie there and the last taken one does.  From the least
// key instead, scores of both signs spread the bins over all powers of two down to zero.
// us of the scorer and the top-k (28 heads, D = 128, top 64), radix select of four 8-bit digits
// over keys in LDS / this from the least key, 64 keys ranked by a thread each / now:
//   4 requests of 300 pages    one sign 14.4 / 10.6 / 10.8    both signs 14.4 / 15.3 / 12.2
//   4 requests of 2048 pages            16.8 / 11.7 / 11.7               16.9 / 17.9 / 11.6
//   4 requests of 8192 pages            32.6 / 22.0 / 21.5               33.1 / 28.6 / 21.3
//   16 requests of 12000 pages, all scores equal 99.8 / 106.7 / 84.5
constexpr int TOPK_BINS = 2048;
constexpr int TOPK_GROUP = 8;  // threads

// cnt[0 .. N) -> its exclusive prefix sum, by the first wave.
template <int N>
__device__ __forceinline__ void prefix_counts(int32_t* cnt) {
  constexpr int PER = (N + 63) / 64;
  const int lane = threadIdx.x;
  if (threadIdx.x < 64) {
    int32_t v[PER], own = 0;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      v[i] = lane * PER + i < N ? cnt[lane * PER + i] : 0;
      own += v[i];
    }
    int32_t at = wave_inclusive_sum(own) - own;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      if (lane * PER + i < N) cnt[lane * PER + i] = at;
      at += v[i];
    }
  }
}

template <int TT, int KPT>
__global__ __launch_bounds__(TT, 4) void quest_topk_kernel(QuestArgs a) {  // at most 128 VGPRs
  constexpr int NW = TT / 64, PB = TOPK_BINS / TT;
  // Keys ranked among themselves: more where few keys per thread leave no closer bound (300 pages,
  // both signs, as above with 64: 15.6 us).
  constexpr int FEW = KPT <= 2 ? 128 : 64;
  static_assert(KPT * TT <= 32 * TOPK_BINS, "the histogram also holds a bitmap of the pages");
  __shared__ uint32_t hist[TOPK_BINS];
  __shared__ uint32_t red[2 * NW];
  __shared__ uint32_t few_key[FEW], few_page[FEW];
  __shared__ int32_t cnt[KPT * NW];
  __shared__ uint32_t s_bin, s_above, s_held, s_few;
  const int64_t h = blockIdx.x, b = blockIdx.y;
  const int32_t T = threadIdx.x, lane = T & 63, wave = T >> 6;
  int32_t* out = a.pages + b * a.p_sb + h * a.top;
  if (a.top >= a.count[b]) {
    for (int64_t j = T; j < a.count[b]; j += TT) out[j] = static_cast<int32_t>(j);
    return;
  }
  const int32_t count = static_cast<int32_t>(a.count[b]);  // at most TT * KPT
  const float* sc = a.scores + (b * a.Hq + h) * a.cmax;
  const bool sink = a.keep_sink && a.top > 1;  // top < count: another page than the tail
  float v[KPT];
#pragma unroll
  for (int j = 0; j < KPT; ++j) v[j] = sc[j * TT + T < count ? j * TT + T : 0];
#pragma unroll
  for (int i = 0; i < PB; ++i) hist[i * TT + T] = 0u;
  if (T == 0) s_few = 0u;
  uint32_t key[KPT];
  uint32_t live = 0u, taken = 0u;  // bit j: key j may still be taken / is taken
  uint32_t lo = 0xffffffffu, hi = 0u;
#pragma unroll
  for (int j = 0; j < KPT; ++j) {
    const int32_t p = j * TT + T;
    key[j] = score_key(v[j]);
    const bool forced = p == count - 1 || (sink && p == 0);
    if (forced) taken |= 1u << j;
    if (p < count && !forced) {
      live |= 1u << j;
      lo = key[j] < lo ? key[j] : lo;
      hi = key[j] > hi ? key[j] : hi;
    }
  }
  // still to take among the live keys
  uint32_t need = static_cast<uint32_t>(a.top) - (sink ? 2u : 1u);
  // The least of the largest keys of `need` or more groups of keys is a lower bound of the last
  // taken key, and a far closer one than the least key: groups of TOPK_GROUP threads, or single
  // threads (a group without a live key makes the bound 0).
  const bool by_group = need <= TT / TOPK_GROUP && count >= TT;
  const bool by_thread = need <= TT && count >= 2 * TT;
  if (by_group || by_thread) lo = hi;
#pragma unroll
  for (int off = 1; off <= 32; off <<= 1) {
    const uint32_t u = __shfl_xor(hi, off, 64);
    hi = u > hi ? u : hi;
    if (by_group && off < TOPK_GROUP) {
      lo = hi;
    } else {
      const uint32_t l = __shfl_xor(lo, off, 64);
      lo = l < lo ? l : lo;
    }
  }
  if (lane == 0) {
    red[wave] = lo;
    red[NW + wave] = hi;
  }
  __syncthreads();
#pragma unroll
  for (int w = 0; w < NW; ++w) {
    lo = red[w] < lo ? red[w] : lo;
    hi = red[NW + w] > hi ? red[NW + w] : hi;
  }
  // the keys that may still be taken lie in [lo, hi]
#pragma unroll
  for (int j = 0; j < KPT; ++j)
    if (key[j] < lo) live &= ~(1u << j);
  uint32_t span = hi > lo ? hi - lo : 0u;
  while (need > 0) {  // the same for the whole workgroup
    if (span == 0u) {  // equal keys: the lowest pages
#pragma unroll 1
      for (int j = 0; j < KPT; ++j) {
        const uint64_t m = __ballot((live >> j) & 1u);
        if (lane == 0) cnt[j * NW + wave] = __popcll(m);
      }
      __syncthreads();
      prefix_counts<KPT * NW>(cnt);
      __syncthreads();
#pragma unroll 1
      for (int j = 0; j < KPT; ++j) {
        const uint64_t m = __ballot((live >> j) & 1u);
        if (((live >> j) & 1u) && static_cast<uint32_t>(cnt[j * NW + wave] + lanes_below(m)) < need) taken |= 1u << j;
      }
      __syncthreads();  // cnt is written again below
      break;
    }
    const int bits = 32 - __clz(static_cast<int>(span));  // __clz(0) == 32
    const int shift = bits > 11 ? bits - 11 : 0;
#pragma unroll
    for (int j = 0; j < KPT; ++j)
      if ((live >> j) & 1u) atomicAdd(&hist[(key[j] - lo) >> shift], 1u);
    __syncthreads();
    // thread T owns the PB bins below those of the threads before it
    uint32_t own[PB], sum = 0u;
    const int32_t first = TOPK_BINS - 1 - T * PB;
#pragma unroll
    for (int i = 0; i < PB; ++i) {
      own[i] = hist[first - i];
      sum += own[i];
    }
    const uint32_t inc = wave_inclusive_sum(sum);
    if (lane == 63) red[wave] = inc;
    __syncthreads();
    uint32_t above = inc - sum;
#pragma unroll
    for (int w = 0; w < NW; ++w) above += w < wave ? red[w] : 0u;
#pragma unroll
    for (int i = 0; i < PB; ++i) {
      if (above < need && above + own[i] >= need) {  // one bin of one thread
        s_bin = static_cast<uint32_t>(first - i);
        s_above = above;
        s_held = own[i];
      }
      above += own[i];
      hist[first - i] = 0u;
    }
    __syncthreads();
    const uint32_t bin = s_bin, held = s_held;
    need -= s_above;
    asm volatile("" : "+v"(lo));  // the keys' bins are taken again: kept, 18 keys a thread spill
#pragma unroll
    for (int j = 0; j < KPT; ++j) {
      const uint32_t k = (key[j] - lo) >> shift;
      if (((live >> j) & 1u) && k >= bin && (k > bin || held == need)) taken |= 1u << j;
      if (k != bin) live &= ~(1u << j);
    }
    if (held == need) break;
    if (held <= FEW) {  // rank the bin's keys among themselves
#pragma unroll
      for (int j = 0; j < KPT; ++j)
        if ((live >> j) & 1u) {
          const uint32_t i = atomicAdd(&s_few, 1u);
          few_key[i] = key[j];
          few_page[i] = static_cast<uint32_t>(j * TT + T);
        }
      __syncthreads();
      // every wave holds them all, and ranks every NW-th of them by ballots
      constexpr int FJ = FEW / 64;
      uint32_t fk[FJ], fp[FJ];
#pragma unroll
      for (int i = 0; i < FJ; ++i) {
        fk[i] = few_key[i * 64 + lane];
        fp[i] = few_page[i * 64 + lane];
      }
      const int32_t mine = wave + NW * lane < FEW ? wave + NW * lane : 0;
      const uint32_t mk = few_key[mine], mp = few_page[mine];
      for (int32_t c = 0; wave + NW * c < static_cast<int32_t>(held); ++c) {
        const uint32_t k = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(mk), c));
        const uint32_t p = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(mp), c));
        uint32_t rank = 0;
#pragma unroll
        for (int i = 0; i < FJ; ++i) {
          const bool before = fk[i] > k || (fk[i] == k && fp[i] < p);
          rank += static_cast<uint32_t>(__popcll(__ballot(i * 64u + lane < held && before)));
        }
        if (lane == 0 && rank < need) atomicOr(&hist[p >> 5], 1u << (p & 31));  // cleared above: a bitmap of the pages
      }
      __syncthreads();
#pragma unroll
      for (int j = 0; j < KPT; ++j) taken |= ((hist[(j * TT + T) >> 5] >> (T & 31)) & 1u) << j;
      break;
    }
    lo += bin << shift;
    span = (1u << shift) - 1u;
  }
  uint64_t m[KPT];
#pragma unroll
  for (int j = 0; j < KPT; ++j) {
    m[j] = __ballot((taken >> j) & 1u);
    if (lane == 0) cnt[j * NW + wave] = __popcll(m[j]);
  }
  __syncthreads();
  prefix_counts<KPT * NW>(cnt);
  __syncthreads();
#pragma unroll
  for (int j = 0; j < KPT; ++j)
    if ((taken >> j) & 1u) out[cnt[j * NW + wave] + lanes_below(m[j])] = j * TT + T;
}

// The same for histories of more pages than a workgroup's registers hold: a radix
// select of four 8-bit passes over the scores in memory, each pass's digit found by
// the first wave with a suffix scan over the histogram.
__global__ __launch_bounds__(1024) void quest_topk_long_kernel(QuestArgs a) {
  constexpr int TT = 1024;
  __shared__ uint32_t hist[256];
  __shared__ uint32_t s_prefix, s_mask, s_need;
  __shared__ int64_t scan64[16];
  const int64_t h = blockIdx.x, b = blockIdx.y;
  const int64_t count = a.count[b];
  int32_t* out = a.pages + b * a.p_sb + h * a.top;
  if (a.top >= count) {
    for (int64_t j = threadIdx.x; j < count; j += TT) out[j] = static_cast<int32_t>(j);
    return;
  }
  const float* sc = a.scores + (b * a.Hq + h) * a.cmax;
  const bool sink = a.keep_sink && a.top > 1 && count > 1;
  auto key_from_scores = [&](int64_t p) -> uint32_t {
    if (p == count - 1 || (sink && p == 0)) return 0xffffffffu;
    return score_key(sc[p]);
  };
  if (threadIdx.x == 0) {
    s_prefix = 0u;
    s_mask = 0u;
    s_need = static_cast<uint32_t>(a.top);
  }
  const int lane = threadIdx.x & 63;
  for (int shift = 24; shift >= 0; shift -= 8) {
    for (int i = threadIdx.x; i < 256; i += TT) hist[i] = 0u;
    __syncthreads();
    const uint32_t prefix = s_prefix, mask = s_mask;
    for (int64_t p0 = threadIdx.x - lane; p0 < count; p0 += TT) {  // wave-uniform trip count
      const int64_t p = p0 + lane;
      const uint32_t k = p < count ? key_from_scores(p) : 0u;
      const uint32_t digit = (k >> shift) & 255u;
      bool pending = p < count && (k & mask) == prefix;
      // Scores of one magnitude share their top digits, so most lanes of a wave
      // would add to one bin (an LDS atomic conflicting 64 ways).  Twice, the
      // lanes holding the first pending lane's digit add their count in one
      // atomic; the lanes left add their own.
#pragma unroll
      for (int r = 0; r < 2; ++r) {
        const uint64_t live = __ballot(pending);
        if (live == 0) break;
        const int leader = __ffsll(static_cast<unsigned long long>(live)) - 1;
        const uint32_t ld = __shfl(digit, leader, 64);
        const bool same = pending && digit == ld;
        const uint64_t group = __ballot(same);
        if (lane == leader) atomicAdd(&hist[ld], static_cast<uint32_t>(__popcll(group)));
        pending = pending && !same;
      }
      if (pending) atomicAdd(&hist[digit], 1u);
    }
    __syncthreads();
    if (threadIdx.x < 64) {
      // lane l owns digits 4l .. 4l+3; keys with a digit above d number
      // above(d) = (sum over lanes > l) + (own digits above d)
      const uint32_t h0 = hist[4 * lane], h1 = hist[4 * lane + 1], h2 = hist[4 * lane + 2],
                     h3 = hist[4 * lane + 3];
      const uint32_t own = h0 + h1 + h2 + h3;
      uint32_t suffix = own;  // inclusive suffix sum over lanes >= l
#pragma unroll
      for (int off = 1; off < 64; off <<= 1) {
        const uint32_t o = __shfl_down(suffix, off, 64);
        if (lane + off < 64) suffix += o;
      }
      const uint32_t need = s_need;
      uint32_t above = suffix - own;
      const uint32_t hv[4] = {h0, h1, h2, h3};
#pragma unroll
      for (int i = 3; i >= 0; --i) {
        if (above < need && above + hv[i] >= need) {
          // exactly one (lane, digit) satisfies this
          s_need = need - above;
          s_prefix = prefix | (static_cast<uint32_t>(4 * lane + i) << shift);
          s_mask = mask | (255u << shift);
        }
        above += hv[i];
      }
    }
    __syncthreads();
  }
  const uint32_t kth = s_prefix, need_eq = s_need;
  // ordered compaction over contiguous page ranges
  const int64_t per = (count + TT - 1) / TT;
  const int64_t p0 = threadIdx.x * per;
  int64_t p1 = p0 + per;
  if (p1 > count) p1 = count;
  int64_t eq = 0;
  for (int64_t p = p0; p < p1; ++p) eq += key_from_scores(p) == kth;
  int64_t tot;
  const int64_t eq_before = block_exclusive_sum<int64_t>(eq, scan64, &tot);
  int64_t sel = 0, e = eq_before;
  for (int64_t p = p0; p < p1; ++p) {
    const uint32_t k = key_from_scores(p);
    if (k > kth) ++sel;
    else if (k == kth && e++ < static_cast<int64_t>(need_eq)) ++sel;
  }
  const int64_t sel_before = block_exclusive_sum<int64_t>(sel, scan64, &tot);
  int64_t o = sel_before;
  e = eq_before;
  for (int64_t p = p0; p < p1; ++p) {
    const uint32_t k = key_from_scores(p);
    bool take = k > kth;
    if (!take && k == kth) take = e++ < static_cast<int64_t>(need_eq);
    if (take) out[o++] = static_cast<int32_t>(p);
  }
}

// Uniform page resampling (the miss-heavy stress workload's selector): per
// (layer, request) the tail page and top - 1 other pages drawn uniformly without
// replacement by Floyd's algorithm -- for j = n - k .. n - 1, t uniform in
// [0, j]; take t unless taken, else j -- over the count - 1 non-tail pages, with
// a counter-based generator (splitmix64 of seed, step, layer, request, j), so the
// draw depends on nothing but those.  Lane 0 draws into an LDS bitmap; the wave
// then writes the pages in ascending order (tail last) to every head's row, and
// -1 past min(top, count).  One wave per (layer, request).
struct UniformArgs {
  uint64_t seed, step;
  int64_t count[QMAXB];  // of requests b0 .. b0 + gridDim.y - 1
  int64_t b0, B, layers, top, heads;
  int32_t* out;  // [layers, B, heads, top]
};

__host__ __device__ __forceinline__ uint64_t splitmix64(uint64_t x) {
  x += 0x9e3779b97f4a7c15ull;
  x = (x ^ (x >> 30)) * 0xbf58476d1ce4e5b9ull;
  x = (x ^ (x >> 27)) * 0x94d049bb133111ebull;
  return x ^ (x >> 31);
}

// Uniform in [0, bound) from a 64-bit draw: the high half of draw_hi32 * bound.
__host__ __device__ __forceinline__ uint32_t uniform_below(uint64_t draw, uint32_t bound) {
  return static_cast<uint32_t>(((draw >> 32) * static_cast<uint64_t>(bound)) >> 32);
}

constexpr int UNIFORM_MAX_PAGES = 1 << 16;

__global__ __launch_bounds__(64) void uniform_pages_kernel(UniformArgs a) {
  __shared__ uint32_t bits[UNIFORM_MAX_PAGES / 32];
  const int64_t layer = blockIdx.x, b = a.b0 + blockIdx.y;
  const int lane = threadIdx.x;
  const int64_t count = a.count[blockIdx.y];
  const int64_t n = count - 1;  // non-tail pages
  const int64_t k = a.top - 1;  // of them drawn
  const int64_t words = (count + 31) / 32;
  for (int64_t w = lane; w < words; w += 64) bits[w] = 0u;
  __syncthreads();
  if (count <= a.top) {
    for (int64_t w = lane; w < words; w += 64) {
      const int64_t rest = count - 32 * w;
      bits[w] = rest >= 32 ? 0xffffffffu : ((1u << rest) - 1u);
    }
  } else if (lane == 0) {
    const uint64_t base = splitmix64(splitmix64(splitmix64(a.seed) ^ a.step) ^
                                     static_cast<uint64_t>(layer * a.B + b));
    for (int64_t j = n - k; j < n; ++j) {
      const uint32_t t = uniform_below(splitmix64(base ^ static_cast<uint64_t>(j)), static_cast<uint32_t>(j + 1));
      const bool taken = (bits[t >> 5] >> (t & 31)) & 1u;
      const uint32_t pick = taken ? static_cast<uint32_t>(j) : t;
      bits[pick >> 5] |= 1u << (pick & 31);
    }
    bits[n >> 5] |= 1u << (n & 31);  // the tail page
  }
  __syncthreads();
  // ascending write: lane l owns words l, l + 64, ...; a running base per round
  int32_t* row = a.out + (layer * a.B + b) * a.heads * a.top;
  int64_t written = 0;
  for (int64_t w0 = 0; w0 < words; w0 += 64) {
    const int64_t w = w0 + lane;
    uint32_t word = w < words ? bits[w] : 0u;
    const int c = __popc(word);
    int inc = c;  // inclusive prefix over the wave
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int o = __shfl_up(inc, off, 64);
      if (lane >= off) inc += o;
    }
    int64_t at = written + inc - c;
    while (word) {
      const int bit = __ffs(word) - 1;
      word &= word - 1;
      for (int64_t h = 0; h < a.heads; ++h) row[h * a.top + at] = static_cast<int32_t>(32 * w + bit);
      ++at;
    }
    written += __shfl(inc, 63, 64);
  }
  for (int64_t i = written + lane; i < a.top; i += 64)
    for (int64_t h = 0; h < a.heads; ++h) row[h * a.top + i] = -1;
}

struct UnionArgs {
  const int32_t* pages;  // [B, Hq, top], first min(top, count) ascending
  int64_t p_sb, top;
  int64_t length[QMAXB];
  int64_t P, Hq, Hkv, g;
  int32_t* positions;    // [B, cap]
  int64_t pos_cap;
  int64_t* head_columns; // [B, Hq, width]
  int64_t width;
  int32_t* union_count;  // [B]
  int32_t* ecol;         // [B, Hkv, ecap]
  uint32_t* emask;
  int64_t ecap;
  int32_t* ecount;       // [B, Hkv]
  unsigned long long* estats;  // nullable: the clamped entry counts are added here
  int32_t* status;       // nonzero on overflow
  uint32_t* page_bits;   // nullable [B, pb_stride]: the union's page bitmap
  int64_t pb_stride;
  int64_t words;         // bitmap words of the longest history
  int64_t maxcount;      // pages of the longest history
  int use_map;           // rank -> page map in LDS (maxcount <= UMAPPAGES)
  int pshift;            // log2 P, or -1
  int chunk, part_heads;  // positions or entries, and heads, of a workgroup
  int parts, pos_parts, entry_parts;  // workgroups in all, of the positions, of a KV head's entries
};

__device__ __forceinline__ bool head_has_page(const int32_t* row, int64_t k, int32_t p) {
  int64_t lo = 0, hi = k;
  while (lo < hi) {
    const int64_t mid = (lo + hi) >> 1;
    if (row[mid] < p) lo = mid + 1;
    else hi = mid;
  }
  return lo < k && row[lo] == p;
}

// Workgroups of one request (blockIdx.y), by blockIdx.x: a chunk of union positions each;
// then, per KV head, a chunk of its group entries each; then the union columns of up
// to UCHUNK / UT query heads each, one after the other.  Every workgroup rebuilds the selected-page bitmap and its
// word prefix popcounts in LDS (a few hundred words) from the heads' pages, so none waits for
// another; one whose chunk no list of the request reaches ends before that.  The launch is
// bound by that chain of steps and by what the longest workgroup writes after it: equal
// chunks keep the second part short, and indexes are 32-bit with pages of a power of two
// taken by shifts (a 64-bit division by a runtime page size costs more than the store it
// serves).  Positions and entries are written one output element per thread through an LDS
// map from a page's rank to the page, a group entry's head mask comes from an LDS array
// indexed by the page's rank among the group's pages.
// A chunk is UCHUNK while a CU has one workgroup at most, and doubles up to UCHUNK_MAX while
// they have more: rebuilding the bitmap then costs more than a chunk's stores.
// us per launch with one workgroup per head, KV head and position list and 64-bit indexes, with
// chunks of 4096 and heads of 4096 columns whatever they cost, and now (heads x pages of the
// history's, requests): 28 x 64 of 8192, 16: 20.0, 9.4 and 8.2; 64 x 4 of 13, 1: 5.8, 17.1 and
// 4.8; 64 x 512 of 8192, 16: 114, 146 and 78; 64 x 2000 of 4096, 16: 601, 1097 and 480; 64 x 32
// of 125 with lists for 64 times as many, 16: 26.5, 43.9 and 9.1.
constexpr int64_t UMAXMASK = 4096;  // group pages (g * top) with an LDS mask slot
constexpr int64_t UMAPPAGES = 24576;  // longest history (pages) with an LDS rank -> page map
constexpr int64_t UCHUNK = 4096;
constexpr int64_t UCHUNK_MAX = 16384;
constexpr int64_t UGRID = 1 << 20;  // workgroups of one grid row: the next ones are in the third dimension
constexpr int64_t UMAXHEADS = 1 << 22;
constexpr int64_t UCUS = 256;

// prefix[w] = set bits of bits[0 .. w), by one wave; returns all set bits.
__device__ __forceinline__ void prefix_popcounts(const uint32_t* bits, uint32_t* prefix, int32_t words) {
  const int32_t lane = threadIdx.x & 63;
  const int32_t per = (words + 63) / 64;
  const int32_t w0 = lane * per;
  const int32_t w1 = w0 + per < words ? w0 + per : words;
  int32_t own = 0;
  for (int32_t w = w0; w < w1; ++w) own += __popc(bits[w]);
  int32_t at = wave_inclusive_sum(own) - own;
  for (int32_t w = w0; w < w1; ++w) {
    prefix[w] = static_cast<uint32_t>(at);
    at += __popc(bits[w]);
  }
}

// Both bitmaps' prefixes by the whole workgroup, two words a thread: for more words than a
// wave should walk.
__device__ __forceinline__ void block_prefix_popcounts(const uint32_t* ubits, uint32_t* uprefix, const uint32_t* gbits,
                                                       uint32_t* gprefix, int32_t words, uint64_t* scan) {
  static_assert(UMAXPAGES <= 2 * 32 * UT, "two words a thread");
  const int32_t w = 2 * static_cast<int32_t>(threadIdx.x), wave = threadIdx.x >> 6;
  auto both = [&](int32_t i) -> uint64_t {  // the group's count above the union's
    return i < words ? static_cast<uint64_t>(__popc(gbits[i])) << 32 | static_cast<uint64_t>(__popc(ubits[i])) : 0u;
  };
  const uint64_t c0 = both(w), c1 = both(w + 1);
  uint64_t at = wave_inclusive_sum(c0 + c1);
  if ((threadIdx.x & 63) == 63) scan[wave] = at;
  __syncthreads();
  at -= c0 + c1;
  for (int32_t u = 0; u < wave; ++u) at += scan[u];
  for (int32_t i = w; i < w + 2 && i < words; ++i, at += c0) {
    uprefix[i] = static_cast<uint32_t>(at);
    gprefix[i] = static_cast<uint32_t>(at >> 32);
  }
}

// Dynamic LDS: four bitmaps of `a.words` words and a rank -> page map of `a.maxcount`
// entries (longest history of the batch).  At most 80 SGPRs: with more a SIMD was seen to hold
// seven waves, so a CU one workgroup instead of two (16 requests, 64 heads x 512 pages: 78 us with
// 80, 106 with 81).
__global__ __launch_bounds__(UT) __attribute__((amdgpu_num_sgpr(80))) void build_union_kernel(UnionArgs a) {
  extern __shared__ uint32_t union_lds[];
  uint32_t* ubits = union_lds;
  uint32_t* uprefix = ubits + a.words;
  uint32_t* gbits = uprefix + a.words;
  uint32_t* gprefix = gbits + a.words;
  int32_t* rank_page = reinterpret_cast<int32_t*>(gprefix + a.words);  // [maxcount], or scan scratch [32]
  __shared__ uint32_t gmask[UMAXMASK];
  const int64_t b = blockIdx.y;
  const int32_t T = threadIdx.x;
  const int32_t L = static_cast<int32_t>(a.length[b]), P = static_cast<int32_t>(a.P);
  const int32_t Hq = static_cast<int32_t>(a.Hq), g = static_cast<int32_t>(a.g);
  const int64_t top = a.top;  // the pages' row stride; it and the capacities may pass 31 bits
  const int32_t count = (L - 1) / P + 1;
  const int32_t k = top < count ? static_cast<int32_t>(top) : count;
  const int32_t tail_len = L - (count - 1) * P;
  const int32_t words = (count + 31) / 32;
  const int32_t* pg = a.pages + b * a.p_sb;
  // the role and its chunk
  int32_t part = static_cast<int32_t>(blockIdx.z * gridDim.x + blockIdx.x);
  if (part >= a.parts) return;
  const bool position = part < a.pos_parts;
  if (!position) part -= a.pos_parts;
  const bool group = !position && part < static_cast<int32_t>(a.Hkv) * a.entry_parts;
  const int32_t kv = group ? part / a.entry_parts : 0;
  if (!position && !group) part -= static_cast<int32_t>(a.Hkv) * a.entry_parts;
  const int32_t chunk = group ? part - kv * a.entry_parts : part;
  const bool masks_in_lds = g * k <= UMAXMASK;
  // a list has at most the history's tokens and at most those of the pages its heads select
  const int64_t c0 = static_cast<int64_t>(chunk) * a.chunk;
  if (chunk > 0 && (position || group) && (c0 >= L || c0 >= static_cast<int64_t>(position ? Hq : g) * k * P)) {
    if (group) return;
    const int64_t end = c0 + a.chunk < a.pos_cap ? c0 + a.chunk : a.pos_cap;
    for (int64_t i = c0 + T; i < end; i += UT) a.positions[b * a.pos_cap + i] = -1;
    return;
  }
  // page and row of a token offset: a shift where the page size is a power of two
  auto page_of = [&](uint32_t i) { return static_cast<int32_t>(a.pshift >= 0 ? i >> a.pshift : i / static_cast<uint32_t>(P)); };

  for (int32_t i = T; i < words; i += UT) {
    ubits[i] = 0u;
    gbits[i] = 0u;
  }
  if (group && masks_in_lds)
    for (int32_t i = T; i < g * k; i += UT) gmask[i] = 0u;
  __syncthreads();
  // the thread's pages, UT apart; heads times pages may pass 31 bits, so head and page are stepped.
  // The quotients of up to UT by k come from a reciprocal of one ulp: half a step off the integers
  // is 2^-11 of them or more (an integer division of each took 0.2 us a launch).
  const float by_k = __builtin_amdgcn_rcpf(static_cast<float>(k));
  const int32_t step_h = static_cast<int32_t>((UT + 0.5f) * by_k), step_j = UT - step_h * k;
  for (int32_t h = static_cast<int32_t>((T + 0.5f) * by_k), j = T - h * k; h < Hq;) {
    const int32_t p = pg[h * top + j];
    if (p >= 0 && p < count) {
      atomicOr(&ubits[p >> 5], 1u << (p & 31));
      if (group && h / g == kv) atomicOr(&gbits[p >> 5], 1u << (p & 31));
    }
    h += step_h;
    j += step_j;
    if (j >= k) {
      j -= k;
      ++h;
    }
  }
  __syncthreads();
  if (!a.use_map) {
    block_prefix_popcounts(ubits, uprefix, gbits, gprefix, words, reinterpret_cast<uint64_t*>(rank_page));
  } else if (T < 64) {
    prefix_popcounts(ubits, uprefix, words);
  } else if (T < 128 && group) {
    prefix_popcounts(gbits, gprefix, words);
  }
  __syncthreads();
  auto rank_of = [&](const uint32_t* bits, const uint32_t* pre, int32_t p) -> int32_t {
    return static_cast<int32_t>(pre[p >> 5]) + __popc(bits[p >> 5] & ((1u << (p & 31)) - 1u));
  };

  if (position) {
    const int32_t upages = rank_of(ubits, uprefix, count - 1) + 1;  // the tail page is always selected
    const int32_t n = (upages - 1) * P + tail_len;
    if (chunk == 0) {
      if (T == 0) {
        a.union_count[b] = n;
        if (n > a.pos_cap) atomicOr(a.status, 1);
      }
      if (a.page_bits)
        for (int32_t w = T; w < words; w += UT) a.page_bits[b * a.pb_stride + w] = ubits[w];
    }
    // the chunk: `size` positions from c0, the first `held` of them union positions
    int32_t* pos = a.positions + b * a.pos_cap + c0;
    const int32_t size = a.pos_cap - c0 < a.chunk ? static_cast<int32_t>(a.pos_cap - c0) : a.chunk;
    const int32_t held = n <= c0 ? 0 : n - c0 < size ? static_cast<int32_t>(n - c0) : size;
    const int32_t i0 = static_cast<int32_t>(c0);  // used where held > 0: below n
    if (a.use_map) {
      for (int32_t p = T; p < count; p += UT)
        if ((ubits[p >> 5] >> (p & 31)) & 1u) rank_page[rank_of(ubits, uprefix, p)] = p;
      __syncthreads();
      // position i: token i % P of the (i / P)-th union page (the tail page is the last)
      for (int32_t i = T; i < held; i += UT) {
        const int32_t r = page_of(i0 + i);
        pos[i] = rank_page[r] * P + (i0 + i - r * P);
      }
    } else {
      for (int32_t p = T; p < count; p += UT) {
        if (!((ubits[p >> 5] >> (p & 31)) & 1u)) continue;
        const int32_t base = rank_of(ubits, uprefix, p) * P;
        const int32_t plen = p == count - 1 ? tail_len : P;
        // the page's tokens in the chunk
        const int64_t o0 = c0 - base > 0 ? c0 - base : 0;
        const int64_t o1 = c0 + held - base < plen ? c0 + held - base : plen;
        for (int64_t off = o0; off < o1; ++off) pos[base + off - c0] = static_cast<int32_t>(p * P + off);
      }
    }
    for (int32_t i = held + T; i < size; i += UT) pos[i] = -1;
  } else if (!group) {
    // union columns of the chunk's heads: a head's j-th token (its pages ascending, tail last)
    const int32_t W = (k - 1) * P + tail_len;
    for (int32_t h = chunk * a.part_heads; h < (chunk + 1) * a.part_heads && h < Hq; ++h) {
      int64_t* hc = a.head_columns + (b * a.Hq + h) * a.width;
      const int32_t* row = pg + h * top;
      // unsigned: the step past the last column of a history of 2^31 - 1 tokens passes 31 bits
      for (uint32_t jj = T; jj < static_cast<uint32_t>(W); jj += UT) {
        const int32_t j = page_of(jj);
        const int32_t p = j < k - 1 ? row[j] : count - 1;
        hc[jj] = rank_of(ubits, uprefix, p) * P + (static_cast<int32_t>(jj) - j * P);
      }
      for (int64_t jj = static_cast<int64_t>(W) + T; jj < a.width; jj += UT) hc[jj] = -1;
    }
  } else {
    const int32_t gpages = rank_of(gbits, gprefix, count - 1) + 1;
    const int32_t E = (gpages - 1) * P + tail_len;
    const int32_t held = E < a.ecap ? E : static_cast<int32_t>(a.ecap);
    if (chunk == 0 && T == 0) {
      a.ecount[b * a.Hkv + kv] = held;
      if (E > a.ecap) atomicOr(a.status, 2);
      if (a.estats) atomicAdd(a.estats, static_cast<unsigned long long>(held));
    }
    if (c0 >= held) return;
    const uint32_t i0 = static_cast<uint32_t>(c0);  // below held; the step past i1 may pass 31 bits
    const uint32_t i1 = held - c0 < a.chunk ? static_cast<uint32_t>(held) : i0 + a.chunk;
    if (masks_in_lds) {
      // head bits of each group page, indexed by the page's rank in the group
      for (int32_t i = T; i < g * k; i += UT) {
        const int32_t hl = i / k;
        const int32_t p = pg[(kv * g + hl) * top + (i - hl * k)];
        if (p < 0 || p >= count) continue;
        atomicOr(&gmask[rank_of(gbits, gprefix, p)], 1u << hl);
      }
    }
    int32_t* ec = a.ecol + (b * a.Hkv + kv) * a.ecap;
    uint32_t* em = a.emask + (b * a.Hkv + kv) * a.ecap;
    if (masks_in_lds && a.use_map) {
      for (int32_t p = T; p < count; p += UT)
        if ((gbits[p >> 5] >> (p & 31)) & 1u) rank_page[rank_of(gbits, gprefix, p)] = rank_of(ubits, uprefix, p);
      __syncthreads();
      // entry i: token i % P of the (i / P)-th group page, its union column and head mask
      for (uint32_t i = i0 + T; i < i1; i += UT) {
        const int32_t r = page_of(i);
        ec[i] = rank_page[r] * P + (static_cast<int32_t>(i) - r * P);
        em[i] = gmask[r];
      }
      return;
    }
    __syncthreads();
    for (int32_t p = T; p < count; p += UT) {
      if (!((gbits[p >> 5] >> (p & 31)) & 1u)) continue;
      const int32_t grank = rank_of(gbits, gprefix, p);
      const int32_t gbase = grank * P;
      const int32_t plen = p == count - 1 ? tail_len : P;
      // the page's tokens in the chunk
      const int64_t o0 = c0 - gbase > 0 ? c0 - gbase : 0;
      const int64_t o1 = static_cast<int64_t>(i1) - gbase < plen ? static_cast<int64_t>(i1) - gbase : plen;
      if (o0 >= o1) continue;
      uint32_t mask = 0u;
      if (masks_in_lds) {
        mask = gmask[grank];
      } else {
        for (int32_t hl = 0; hl < g; ++hl)
          if (head_has_page(pg + (kv * g + hl) * top, k, p)) mask |= 1u << hl;
      }
      const int32_t ubase = rank_of(ubits, uprefix, p) * P;
      for (int64_t off = o0; off < o1; ++off) {
        ec[gbase + off] = static_cast<int32_t>(ubase + off);
        em[gbase + off] = mask;
      }
    }
  }
}

static int64_t ceil_div(int64_t x, int64_t y) { return (x + y - 1) / y; }

}  // namespace hs

using namespace hs;

extern "C" int64_t hs_quest_workspace_bytes(int64_t batch, int64_t heads, int64_t max_pages) {
  if (batch < 1 || heads < 1 || max_pages < 1) return 256;
  return ((batch * heads * max_pages * 4) + 255) & ~static_cast<int64_t>(255);
}

// At most QMAXB requests (their bounds pointers and page counts travel in the
// kernel arguments); hs_quest_topk cuts larger batches into such chunks.
static int quest_topk_chunk(const void* query, int64_t q_stride_b, int64_t q_stride_h,
                            int32_t query_dtype, const void* const* minimum,
                            const void* const* maximum, int32_t kv_dtype,
                            const int64_t* page_counts, int64_t batch, int64_t heads,
                            int64_t kv_heads, int64_t head_dim, int64_t top, int32_t keep_sink,
                            int32_t* out_pages, int64_t out_stride_b, void* workspace,
                            int64_t workspace_bytes, hipStream_t stream) {
  HS_CHECK_ARG(top >= 1 && heads >= 1 && kv_heads >= 1 && heads % kv_heads == 0,
               "invalid page budget or GQA shape");
  HS_CHECK_ARG(batch >= 1 && batch <= QMAXB, "quest batch must be in [1, %d]", QMAXB);
  HS_CHECK_ARG(valid_dtype(kv_dtype), "invalid dtype code %d", kv_dtype);
  HS_CHECK_ARG(valid_dtype(query_dtype), "invalid query dtype code %d", query_dtype);
  HS_CHECK_ARG(head_dim >= 1 && head_dim <= 1024, "invalid head_dim");
  HS_CHECK_ARG(query && minimum && maximum && page_counts && out_pages, "null quest pointer");
  QuestArgs a{};
  a.q = query;
  a.q_dtype = query_dtype;
  a.q_sb = q_stride_b;
  a.q_sh = q_stride_h;
  int64_t cmax = 1;
  for (int64_t i = 0; i < batch; ++i) {
    HS_CHECK_ARG(page_counts[i] >= 1, "cannot select pages of an empty history");
    HS_CHECK_ARG(minimum[i] && maximum[i], "null bounds pointer");
    a.kmin[i] = minimum[i];
    a.kmax[i] = maximum[i];
    a.count[i] = page_counts[i];
    if (page_counts[i] > cmax) cmax = page_counts[i];
  }
  a.Hq = heads;
  a.Hkv = kv_heads;
  a.g = heads / kv_heads;
  a.D = head_dim;
  a.top = top;
  a.keep_sink = keep_sink;
  a.cmax = cmax;
  a.pages = out_pages;
  a.p_sb = out_stride_b;
  const int64_t need = hs_quest_workspace_bytes(batch, heads, cmax);
  HS_CHECK_ARG(workspace && workspace_bytes >= need, "quest workspace too small: need %lld bytes",
               static_cast<long long>(need));
  a.scores = static_cast<float*>(workspace);
  bool any_scored = false;
  for (int64_t i = 0; i < batch; ++i) any_scored |= top < page_counts[i];
  if (any_scored) {
    const int64_t hchunks = ceil_div(a.g, QHEADS);
    // 16-bit queries times 16-bit bounds: every product is exact in fp32, so an FMA
    // rounds like the reference's product-then-sum
    const bool fused = query_dtype != HS_DTYPE_F32 && kv_dtype != HS_DTYPE_F32;
    const int64_t epv = kv_dtype == HS_DTYPE_F32 ? 4 : 8;
    const int64_t row_bytes = head_dim * (kv_dtype == HS_DTYPE_F32 ? 4 : 2);
    bool aligned = true;
    for (int64_t i = 0; i < batch; ++i)
      aligned &= ((reinterpret_cast<uintptr_t>(minimum[i]) | reinterpret_cast<uintptr_t>(maximum[i])) & 15) == 0;
    // HS_QUEST_SCORER=tile keeps bf16 bounds on quest_score_tile_kernel (for comparisons)
    static const bool perm_off = [] {
      const char* env = getenv("HS_QUEST_SCORER");
      return env && strcmp(env, "tile") == 0;
    }();
    const bool query_words = (reinterpret_cast<uintptr_t>(query) & 3) == 0 &&
                             (query_dtype == HS_DTYPE_F32 || (q_stride_b % 2 == 0 && q_stride_h % 2 == 0));
    if (!perm_off && kv_dtype == HS_DTYPE_BF16 && (query_dtype == HS_DTYPE_BF16 || query_dtype == HS_DTYPE_F32) &&
        query_words && head_dim % 8 == 0 && aligned && row_bytes <= QP_MAX_ROW_BYTES) {
      dim3 grid(static_cast<unsigned>(kv_heads * hchunks), static_cast<unsigned>(ceil_div(cmax, QP_PAGES)),
                static_cast<unsigned>(batch));
      const size_t lds = static_cast<size_t>(qp_lds_bytes(row_bytes, head_dim == 128 ? 2 : 1));
      const bool f32q = query_dtype == HS_DTYPE_F32;
      int64_t bound_rows = 0;
      for (int64_t i = 0; i < batch; ++i) bound_rows += page_counts[i];
      const bool nt = hchunks == 1 && bound_rows * kv_heads * row_bytes * 2 >= QP_NT_BYTES;
      auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, dim3(QP_T), lds, stream, a); };
      if (head_dim == 128) {
        if (f32q) nt ? launch(quest_score_perm_kernel<true, 128, 2, true>) : launch(quest_score_perm_kernel<true, 128, 2, false>);
        else nt ? launch(quest_score_perm_kernel<false, 128, 2, true>) : launch(quest_score_perm_kernel<false, 128, 2, false>);
      } else if (head_dim == 64) {
        if (f32q) nt ? launch(quest_score_perm_kernel<true, 64, 1, true>) : launch(quest_score_perm_kernel<true, 64, 1, false>);
        else nt ? launch(quest_score_perm_kernel<false, 64, 1, true>) : launch(quest_score_perm_kernel<false, 64, 1, false>);
      } else {
        if (f32q) launch(quest_score_perm_kernel<true, 0, 1, false>);
        else launch(quest_score_perm_kernel<false, 0, 1, false>);
      }
      HS_CHECK_LAUNCH("quest scorer");
    } else if (head_dim % epv == 0 && aligned && row_bytes <= QS_MAX_ROW_BYTES) {
      dim3 grid(static_cast<unsigned>(ceil_div(cmax, QS_PAGES)), static_cast<unsigned>(kv_heads * hchunks),
                static_cast<unsigned>(batch));
      const size_t lds = static_cast<size_t>(qs_lds_bytes(row_bytes, head_dim));
      if (kv_dtype == HS_DTYPE_BF16) {
        if (fused) hipLaunchKernelGGL((quest_score_tile_kernel<HS_DTYPE_BF16, true>), grid, dim3(QT), lds, stream, a);
        else hipLaunchKernelGGL((quest_score_tile_kernel<HS_DTYPE_BF16, false>), grid, dim3(QT), lds, stream, a);
      } else if (kv_dtype == HS_DTYPE_F16) {
        if (fused) hipLaunchKernelGGL((quest_score_tile_kernel<HS_DTYPE_F16, true>), grid, dim3(QT), lds, stream, a);
        else hipLaunchKernelGGL((quest_score_tile_kernel<HS_DTYPE_F16, false>), grid, dim3(QT), lds, stream, a);
      } else {
        hipLaunchKernelGGL((quest_score_tile_kernel<HS_DTYPE_F32, false>), grid, dim3(QT), lds, stream, a);
      }
      HS_CHECK_LAUNCH("quest scorer");
    } else {
    dim3 grid(static_cast<unsigned>(ceil_div(cmax, QT)), static_cast<unsigned>(kv_heads * hchunks),
              static_cast<unsigned>(batch));
    const size_t lds = static_cast<size_t>(QHEADS * head_dim * 4);
    if (kv_dtype == HS_DTYPE_BF16) {
      if (fused) hipLaunchKernelGGL((quest_score_kernel<HS_DTYPE_BF16, true>), grid, dim3(QT), lds, stream, a);
      else hipLaunchKernelGGL((quest_score_kernel<HS_DTYPE_BF16, false>), grid, dim3(QT), lds, stream, a);
    } else if (kv_dtype == HS_DTYPE_F16) {
      if (fused) hipLaunchKernelGGL((quest_score_kernel<HS_DTYPE_F16, true>), grid, dim3(QT), lds, stream, a);
      else hipLaunchKernelGGL((quest_score_kernel<HS_DTYPE_F16, false>), grid, dim3(QT), lds, stream, a);
    } else {
      hipLaunchKernelGGL((quest_score_kernel<HS_DTYPE_F32, false>), grid, dim3(QT), lds, stream, a);
    }
    HS_CHECK_LAUNCH("quest scorer");
    }
  }
  const dim3 tgrid(static_cast<unsigned>(heads), static_cast<unsigned>(batch));
  // The thread count and the keys per thread, by the longest history.  512 threads take up
  // to 18 keys each in 128 VGPRs, so two workgroups share a CU (8192 pages, 448 heads: 11.6
  // us, against 13.7 us with 256 threads of 32 keys and 15.5 us with 1024 of 8, which leave
  // one; 2048 pages, 56 heads: 5.7, 6.3 and 6.2 us).  Longer ones take 1024 threads (8250
  // pages: 20.6 us, against 23.6 us for 512 threads of 32 keys), and past their registers
  // the scores are read again for each digit.
  auto launch = [&](auto kernel, int threads) {
    hipLaunchKernelGGL(kernel, tgrid, dim3(static_cast<unsigned>(threads)), 0, stream, a);
  };
  if (cmax <= 512) launch(quest_topk_kernel<512, 1>, 512);
  else if (cmax <= 512 * 2) launch(quest_topk_kernel<512, 2>, 512);
  else if (cmax <= 512 * 4) launch(quest_topk_kernel<512, 4>, 512);
  else if (cmax <= 512 * 8) launch(quest_topk_kernel<512, 8>, 512);
  else if (cmax <= 512 * 16) launch(quest_topk_kernel<512, 16>, 512);
  else if (cmax <= 512 * 18) launch(quest_topk_kernel<512, 18>, 512);
  else if (cmax <= 1024 * 16) launch(quest_topk_kernel<1024, 16>, 1024);
  else launch(quest_topk_long_kernel, 1024);
  HS_CHECK_LAUNCH("quest top-k");
  return HS_OK;
}

// At most QMAXB requests (their lengths travel in the kernel arguments);
// hs_build_union cuts larger batches into such chunks.
static int build_union_chunk(const int32_t* pages, int64_t p_stride_b, int64_t top,
                             const int64_t* lengths, int64_t page_size, int64_t batch,
                             int64_t heads, int64_t kv_heads, int32_t* positions,
                             int64_t pos_capacity, int64_t* head_columns, int64_t width,
                             int32_t* union_count, int32_t* entry_columns,
                             uint32_t* entry_masks, int64_t entry_capacity,
                             int32_t* entry_counts, int32_t* status, uint32_t* page_bits,
                             int64_t pb_stride, int64_t* entry_stats, hipStream_t stream) {
  HS_CHECK_ARG(batch >= 1 && batch <= QMAXB, "union batch must be in [1, %d]", QMAXB);
  HS_CHECK_ARG(top >= 1 && page_size >= 1 && heads >= 1 && kv_heads >= 1 && heads % kv_heads == 0,
               "invalid union shape");
  HS_CHECK_ARG(heads / kv_heads <= 32, "at most 32 query heads per KV head");
  HS_CHECK_ARG(heads <= UMAXHEADS, "too many query heads for the union builder");
  HS_CHECK_ARG(pages && lengths && positions && head_columns && union_count && entry_columns &&
                   entry_masks && entry_counts && status,
               "null union pointer");
  HS_CHECK_ARG(pos_capacity >= 1 && entry_capacity >= 1 && width >= 1, "union capacities must be positive");
  UnionArgs a{};
  a.pages = pages;
  a.p_sb = p_stride_b;
  a.top = top;
  for (int64_t i = 0; i < batch; ++i) {
    HS_CHECK_ARG(lengths[i] >= 1, "cannot build a union over an empty history");
    HS_CHECK_ARG(ceil_div(lengths[i], page_size) <= UMAXPAGES, "too many pages for the union builder");
    const int64_t count = ceil_div(lengths[i], page_size);
    const int64_t k = top < count ? top : count;
    const int64_t W = (k - 1) * page_size + (lengths[i] - (count - 1) * page_size);
    HS_CHECK_ARG(W <= width, "head column width %lld below the selection width %lld",
                 static_cast<long long>(width), static_cast<long long>(W));
    a.length[i] = lengths[i];
  }
  // a page of more tokens than the longest history holds what one of that many does
  a.P = std::min(page_size, *std::max_element(lengths, lengths + batch));
  a.Hq = heads;
  a.Hkv = kv_heads;
  a.g = heads / kv_heads;
  a.positions = positions;
  a.pos_cap = pos_capacity;
  a.page_bits = page_bits;
  a.pb_stride = pb_stride;
  a.head_columns = head_columns;
  a.width = width;
  a.union_count = union_count;
  a.ecol = entry_columns;
  a.emask = entry_masks;
  a.ecap = entry_capacity;
  a.ecount = entry_counts;
  a.estats = reinterpret_cast<unsigned long long*>(entry_stats);
  a.status = status;
  int64_t max_count = 1;
  for (int64_t i = 0; i < batch; ++i) max_count = std::max(max_count, ceil_div(lengths[i], page_size));
  a.words = (max_count + 31) / 32;
  a.maxcount = max_count;
  a.use_map = max_count <= UMAPPAGES;
  const size_t lds = static_cast<size_t>((4 * a.words + (a.use_map ? max_count : 32)) * 4);
  static bool lds_attr = false;
  if (!lds_attr) {  // up to 4 * 768 + 24576 words of dynamic LDS
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(build_union_kernel),
                              hipFuncAttributeMaxDynamicSharedMemorySize, 128 * 1024);
    (void)hipGetLastError();
    lds_attr = true;
  }
  a.pshift = (a.P & (a.P - 1)) == 0 ? __builtin_ctzll(static_cast<unsigned long long>(a.P)) : -1;
  // a list has at most one row per token of the longest history
  const int64_t longest = *std::max_element(lengths, lengths + batch);
  const int64_t most_pos = std::min(pos_capacity, longest), most_entries = std::min(entry_capacity, longest);
  a.part_heads = static_cast<int>(std::max<int64_t>(1, UCHUNK / std::max<int64_t>(width, UT)));
  const int64_t head_parts = ceil_div(heads, a.part_heads);
  int64_t chunk = UCHUNK;
  while (chunk < UCHUNK_MAX &&
         batch * (ceil_div(most_pos, chunk) + kv_heads * ceil_div(most_entries, chunk) + head_parts) > UCUS)
    chunk *= 2;
  a.chunk = static_cast<int>(chunk);
  const int64_t pos_parts = ceil_div(pos_capacity, chunk);  // what no history reaches is filled with -1
  const int64_t entry_parts = ceil_div(most_entries, chunk);
  const int64_t parts = pos_parts + kv_heads * entry_parts + head_parts;
  HS_CHECK_ARG(pos_parts <= INT32_MAX / 2 && parts <= INT32_MAX - UGRID, "union capacities too large");
  a.parts = static_cast<int>(parts);
  a.pos_parts = static_cast<int>(pos_parts);
  a.entry_parts = static_cast<int>(entry_parts);
  const dim3 grid(static_cast<unsigned>(std::min(parts, UGRID)), static_cast<unsigned>(batch),
                  static_cast<unsigned>(ceil_div(parts, UGRID)));
  hipLaunchKernelGGL(build_union_kernel, grid, dim3(UT), lds, stream, a);
  HS_CHECK_LAUNCH("union builder");
  return HS_OK;
}

extern "C" int hs_quest_topk(const void* query, int64_t q_stride_b, int64_t q_stride_h,
                             int32_t query_dtype, const void* const* minimum,
                             const void* const* maximum, int32_t kv_dtype,
                             const int64_t* page_counts, int64_t batch, int64_t heads,
                             int64_t kv_heads, int64_t head_dim, int64_t top, int32_t keep_sink,
                             int32_t* out_pages, int64_t out_stride_b, void* workspace,
                             int64_t workspace_bytes, hipStream_t stream) {
  HS_CHECK_ARG(batch >= 1, "quest batch must be positive");
  HS_CHECK_ARG(valid_dtype(query_dtype), "invalid query dtype code %d", query_dtype);
  HS_CHECK_ARG(valid_dtype(kv_dtype), "invalid dtype code %d", kv_dtype);
  HS_CHECK_ARG(top >= 1 && heads >= 1 && kv_heads >= 1 && heads % kv_heads == 0,
               "invalid page budget or GQA shape");
  HS_CHECK_ARG(head_dim >= 1 && head_dim <= 1024, "invalid head_dim");
  HS_CHECK_ARG(query && minimum && maximum && page_counts && out_pages, "null quest pointer");
  // every request and every chunk's workspace need are checked before the first
  // launch, so an invalid call launches nothing
  for (int64_t i = 0; i < batch; ++i) {
    HS_CHECK_ARG(page_counts[i] >= 1, "cannot select pages of an empty history");
    HS_CHECK_ARG(minimum[i] && maximum[i], "null bounds pointer");
  }
  for (int64_t s0 = 0; s0 < batch; s0 += QMAXB) {
    const int64_t n = batch - s0 < QMAXB ? batch - s0 : QMAXB;
    int64_t cmax = 1;
    for (int64_t i = s0; i < s0 + n; ++i) cmax = page_counts[i] > cmax ? page_counts[i] : cmax;
    const int64_t need = hs_quest_workspace_bytes(n, heads, cmax);
    HS_CHECK_ARG(workspace && workspace_bytes >= need, "quest workspace too small: need %lld bytes",
                 static_cast<long long>(need));
  }
  const int64_t qbytes = query_dtype == HS_DTYPE_F32 ? 4 : 2;
  // chunks run in stream order and each reuses the workspace, which holds the
  // scores of at most the whole batch
  for (int64_t s0 = 0; s0 < batch; s0 += QMAXB) {
    const int64_t n = batch - s0 < QMAXB ? batch - s0 : QMAXB;
    const int rc = quest_topk_chunk(static_cast<const char*>(query) + s0 * q_stride_b * qbytes, q_stride_b,
                                    q_stride_h, query_dtype, minimum + s0, maximum + s0, kv_dtype,
                                    page_counts + s0, n, heads, kv_heads, head_dim, top, keep_sink,
                                    out_pages + s0 * out_stride_b, out_stride_b, workspace, workspace_bytes,
                                    stream);
    if (rc != HS_OK) return rc;
  }
  return HS_OK;
}

extern "C" int hs_build_union(const int32_t* pages, int64_t p_stride_b, int64_t top,
                              const int64_t* lengths, int64_t page_size, int64_t batch,
                              int64_t heads, int64_t kv_heads, int32_t* positions,
                              int64_t pos_capacity, int64_t* head_columns, int64_t width,
                              int32_t* union_count, int32_t* entry_columns,
                              uint32_t* entry_masks, int64_t entry_capacity,
                              int32_t* entry_counts, int32_t* status, uint32_t* page_bits,
                              int64_t page_bits_stride, int64_t* entry_stats, hipStream_t stream) {
  HS_CHECK_ARG(batch >= 1, "union batch must be positive");
  HS_CHECK_ARG(top >= 1 && page_size >= 1 && lengths, "invalid union shape");
  HS_CHECK_ARG(heads >= 1 && kv_heads >= 1 && heads % kv_heads == 0, "invalid GQA shape");
  for (int64_t i = 0; i < batch; ++i) {  // every request, before the first launch
    HS_CHECK_ARG(lengths[i] >= 1, "cannot build a union over an empty history");
    HS_CHECK_ARG(lengths[i] <= INT32_MAX, "union positions are 32-bit: %lld tokens", static_cast<long long>(lengths[i]));
    HS_CHECK_ARG(ceil_div(lengths[i], page_size) <= UMAXPAGES, "too many pages for the union builder");
    const int64_t count = ceil_div(lengths[i], page_size);
    const int64_t k = top < count ? top : count;
    const int64_t W = (k - 1) * page_size + (lengths[i] - (count - 1) * page_size);
    HS_CHECK_ARG(W <= width, "head column width %lld below the selection width %lld",
                 static_cast<long long>(width), static_cast<long long>(W));
    HS_CHECK_ARG(!page_bits || page_bits_stride >= ceil_div(count, 32),
                 "page bitmap stride %lld below the %lld words of a history",
                 static_cast<long long>(page_bits_stride), static_cast<long long>(ceil_div(count, 32)));
  }
  for (int64_t s0 = 0; s0 < batch; s0 += QMAXB) {
    const int64_t n = batch - s0 < QMAXB ? batch - s0 : QMAXB;
    const int rc = build_union_chunk(
        pages + s0 * p_stride_b, p_stride_b, top, lengths + s0, page_size, n, heads, kv_heads,
        positions + s0 * pos_capacity, pos_capacity, head_columns + s0 * heads * width, width, union_count + s0,
        entry_columns + s0 * kv_heads * entry_capacity, entry_masks + s0 * kv_heads * entry_capacity,
        entry_capacity, entry_counts + s0 * kv_heads, status,
        page_bits ? page_bits + s0 * page_bits_stride : nullptr, page_bits_stride, entry_stats, stream);
    if (rc != HS_OK) return rc;
  }
  return HS_OK;
}

extern "C" int hs_uniform_pages(uint64_t seed, uint64_t step, const int64_t* page_counts, int64_t batch,
                                int64_t layers, int64_t top, int64_t heads, int32_t* out, hipStream_t stream) {
  HS_CHECK_ARG(batch >= 1 && layers >= 1 && layers <= 65535 && heads >= 1 && top >= 1,
               "invalid uniform pages shape");
  HS_CHECK_ARG(page_counts && out, "null uniform pages pointer");
  for (int64_t i = 0; i < batch; ++i)
    HS_CHECK_ARG(page_counts[i] >= 1 && page_counts[i] <= UNIFORM_MAX_PAGES, "page counts must be 1 to %d",
                 UNIFORM_MAX_PAGES);
  for (int64_t b0 = 0; b0 < batch; b0 += QMAXB) {  // launches of at most 16 requests, in order
    const int64_t nb = batch - b0 < QMAXB ? batch - b0 : QMAXB;
    UniformArgs a{};
    a.seed = seed;
    a.step = step;
    for (int64_t i = 0; i < nb; ++i) a.count[i] = page_counts[b0 + i];
    a.b0 = b0;
    a.B = batch;
    a.layers = layers;
    a.top = top;
    a.heads = heads;
    a.out = out;
    hipLaunchKernelGGL(uniform_pages_kernel, dim3(static_cast<unsigned>(layers), static_cast<unsigned>(nb)),
                       dim3(64), 0, stream, a);
    HS_CHECK_LAUNCH("uniform pages");
  }
  return HS_OK;
}
