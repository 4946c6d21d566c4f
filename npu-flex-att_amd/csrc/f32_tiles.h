// Building blocks of the fp32 matrix-core kernels (f32_mfma.hip, f32_split.hip):
// MFMA wrappers, padded LDS tiles, and the two kinds of products over them.  The
// operand layouts and step orders are described at the top of f32_mfma.hip.
#pragma once
#include "flexatt_device.h"

namespace flexatt {

namespace f32m {

constexpr int kTile = 32;  // rows per LDS tile (one MFMA block)

__device__ __forceinline__ f32x16 mma(float a, float b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

// Row of the 32-row block that lane half h takes at step r (and that holds
// accumulator element r).
__device__ __forceinline__ int blk_row(int r, int h) { return 8 * (r >> 2) + 4 * h + (r & 3); }

template <int D, int NW>
struct Cfg {
  static constexpr int NT = NW * 64;              // threads per workgroup
  static constexpr int P = D + 4;                 // LDS row pitch (floats)
  static constexpr int TILE = kTile * P;          // floats per LDS tile
  static constexpr int N4 = kTile * D / 4;        // 16-byte pieces per tile
  static constexpr int NL = (N4 + NT - 1) / NT;   // pieces per thread per tensor
  static constexpr int HD = D / 2;                // head-dim values per lane for the d-sums
  static constexpr int DB = D / 32;               // 32-wide head-dim blocks
};

// One 32-row tile of one tensor into an LDS tile of D + 4-float rows.
// fetch() starts the copy, commit() completes it in the issuing thread,
// settle() (before the barrier that publishes the tile) waits for it.  At
// D = 256 a row is 1 KB, one direct-to-LDS load of the wave (lane l's 16
// bytes at row offset 16 l), so the copy holds no registers.  Otherwise the
// copy passes through registers, which nothing reads before commit() (so
// the loads overlap the work between the two calls).  Either way rows past
// the tensor repeat its last row: their scores are masked, so the finite
// values drop out.
template <int D, int NW>
struct Tile {
  using C = Cfg<D, NW>;
  static constexpr bool kDirect = D == 256;
  f32x4 x[kDirect ? 1 : C::NL];
  float* dst = nullptr;
  __device__ __forceinline__ void fetch(float* lds, const float* xp, int64_t xs, int r0, int rows, int tid) {
    if constexpr (kDirect) {
      constexpr int RPW = kTile / NW;  // rows per wave
      const int w = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63;
#pragma unroll
      for (int i = 0; i < RPW; ++i) {
        const int r = w * RPW + i;
        const int n = min(r0 + r, rows - 1);
        load_lds16(xp + (int64_t)n * xs + 4 * l, lds_addr_of(lds + r * C::P));
      }
    } else {
      dst = lds;
#pragma unroll
      for (int i = 0; i < C::NL; ++i) {
        const int idx = tid + i * C::NT;
        const int r = idx / (D / 4), c = 4 * (idx % (D / 4));
        const int n = r0 + r;
        const int nc = n < rows ? n : rows - 1;
        x[i] = *(const f32x4*)(xp + (int64_t)nc * xs + c);
      }
    }
  }
  __device__ __forceinline__ void commit(int tid) const {
    if constexpr (!kDirect) {
#pragma unroll
      for (int i = 0; i < C::NL; ++i) {
        const int idx = tid + i * C::NT;
        if (C::N4 % C::NT == 0 || idx < C::N4) {
          const int r = idx / (D / 4), c = 4 * (idx % (D / 4));
          *(f32x4*)(dst + r * C::P + c) = x[i];
        }
      }
    }
  }
  __device__ static __forceinline__ void settle() {
    if constexpr (kDirect) wait_vmcnt<0>();
  }
};

__device__ __forceinline__ f32x4 lds4(const float* p) { return *(const f32x4*)p; }

// acc += A B^T over the head dim: A rows from LDS (row l32 of `t`, 16-byte
// reads one group of four MFMAs ahead), B from the lane's registers.
template <int HD, int P>
__device__ __forceinline__ void dsum(const float* t, const float (&b)[HD], f32x16& acc) {
  f32x4 cur = lds4(t);
#pragma unroll
  for (int k4 = 0; k4 < HD; k4 += 4) {
    f32x4 nxt = cur;
    if (k4 + 4 < HD) nxt = lds4(t + k4 + 4);
#pragma unroll
    for (int e = 0; e < 4; ++e) acc = mma(cur[e], b[k4 + e], acc);
    cur = nxt;
    __builtin_amdgcn_sched_barrier(0);
  }
}
// acc[db] += A^T x over 32 rows: A column 32 db + l32 of `t` read at the rows
// of step r (one group of four steps ahead), x = the lane's element r.
template <int DB, int P>
__device__ __forceinline__ void rsum(const float* t, int l32, int h, const f32x16& x, f32x16 (&acc)[DB]) {
  float cur[4], nxt[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) cur[i] = t[blk_row(i, h) * P + l32];
#pragma unroll
  for (int g = 0; g < 4 * DB; ++g) {
    const int db = g >> 2, r0 = 4 * (g & 3);
#pragma unroll
    for (int i = 0; i < 4; ++i) nxt[i] = cur[i];
    if (g + 1 < 4 * DB) {
      const int db1 = (g + 1) >> 2, r1 = 4 * ((g + 1) & 3);
#pragma unroll
      for (int i = 0; i < 4; ++i) nxt[i] = t[blk_row(r1 + i, h) * P + 32 * db1 + l32];
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[db] = mma(cur[i], x[r0 + i], acc[db]);
#pragma unroll
    for (int i = 0; i < 4; ++i) cur[i] = nxt[i];
    __builtin_amdgcn_sched_barrier(0);
  }
}
// --- 16 x 16 x 4 fp32 MFMA (16 accumulator columns per wave) -----------------
//   A operand  lane l holds A[row = l%16][k = l/16]
//   B operand  lane l holds B[k = l/16][col = l%16]
//   C/D        acc[r] = C[row = 4*(l/16) + r][col = l%16]
// Head-dim sums: lane group g = l/16 takes d = g*D/4 + s at step s.  16-row
// sums: at step s group g takes row 4g + s, the row of its accumulator
// element s.
__device__ __forceinline__ f32x4 mma16(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
// acc1 += A1 B1^T and acc2 += A2 B2^T over the head dim (A rows from LDS,
// 16-byte reads one group of four MFMAs ahead; B from registers).
template <int HD4>
__device__ __forceinline__ void dsum16x2(const float* t1, const float (&b1)[HD4], f32x4& acc1, const float* t2,
                                         const float (&b2)[HD4], f32x4& acc2) {
  f32x4 c1 = lds4(t1), c2 = lds4(t2);
#pragma unroll
  for (int k4 = 0; k4 < HD4; k4 += 4) {
    f32x4 n1 = c1, n2 = c2;
    if (k4 + 4 < HD4) {
      n1 = lds4(t1 + k4 + 4);
      n2 = lds4(t2 + k4 + 4);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      acc1 = mma16(c1[e], b1[k4 + e], acc1);
      acc2 = mma16(c2[e], b2[k4 + e], acc2);
    }
    c1 = n1;
    c2 = n2;
    __builtin_amdgcn_sched_barrier(0);
  }
}
// acc1[db] += A1^T x1 and acc2[db] += A2^T x2 over the 32 rows of a tile
// (two 16-row blocks qb): A column 16 db + l16 of t1 / t2 at row
// 16 qb + 4 g + s, x = the lane's element s of block qb.
template <int DB16, int P>
__device__ __forceinline__ void rsum16x2(const float* t1, const f32x4 (&x1)[2], f32x4 (&acc1)[DB16],
                                         const float* t2, const f32x4 (&x2)[2], f32x4 (&acc2)[DB16], int l16,
                                         int g) {
  constexpr int NG = 2 * DB16;  // groups of four MFMA steps: (db, qb)
  float c1[4], c2[4], n1[4], n2[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    c1[i] = t1[(4 * g + i) * P + l16];
    c2[i] = t2[(4 * g + i) * P + l16];
  }
#pragma unroll
  for (int q = 0; q < NG; ++q) {
    const int db = q >> 1, qb = q & 1;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      n1[i] = c1[i];
      n2[i] = c2[i];
    }
    if (q + 1 < NG) {
      const int db1 = (q + 1) >> 1, qb1 = (q + 1) & 1;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int off = (16 * qb1 + 4 * g + i) * P + 16 * db1 + l16;
        n1[i] = t1[off];
        n2[i] = t2[off];
      }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      acc1[db] = mma16(c1[i], x1[qb][i], acc1[db]);
      acc2[db] = mma16(c2[i], x2[qb][i], acc2[db]);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      c1[i] = n1[i];
      c2[i] = n2[i];
    }
    __builtin_amdgcn_sched_barrier(0);
  }
}

// acc[db] += A^T x over the 32 rows of a tile (two 16-row blocks qb): A
// column 16 db + l16 of t at row 16 qb + 4 g + s, x = the lane's element s
// of block qb.
template <int DB16, int P>
__device__ __forceinline__ void rsum16(const float* t, const f32x4 (&x)[2], f32x4 (&acc)[DB16], int l16, int g) {
  constexpr int NG = 2 * DB16;
  float c[4], n[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) c[i] = t[(4 * g + i) * P + l16];
#pragma unroll
  for (int q = 0; q < NG; ++q) {
    const int db = q >> 1, qb = q & 1;
#pragma unroll
    for (int i = 0; i < 4; ++i) n[i] = c[i];
    if (q + 1 < NG) {
      const int db1 = (q + 1) >> 1, qb1 = (q + 1) & 1;
#pragma unroll
      for (int i = 0; i < 4; ++i) n[i] = t[(16 * qb1 + 4 * g + i) * P + 16 * db1 + l16];
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[db] = mma16(c[i], x[qb][i], acc[db]);
#pragma unroll
    for (int i = 0; i < 4; ++i) c[i] = n[i];
    __builtin_amdgcn_sched_barrier(0);
  }
}

// Natural-domain transformed score (scale, soft-cap, ALiBi); t receives
// tanh(scale s / cap) for the soft-cap derivative.
template <bool SOFTCAP, bool ALIBI>
__device__ __forceinline__ float score(float s, const Shape& p, float slope, int i, int j, float& t) {
  float x = s * p.scale;
  if constexpr (SOFTCAP) {
    t = tanhf(x * p.inv_cap);
    x = p.cap * t;
  }
  if constexpr (ALIBI) x += slope * (float)(i - j);
  return x;
}

}  // namespace f32m

}  // namespace flexatt
