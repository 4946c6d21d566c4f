// fp32 forward and backward for problems whose tiles fill too few of the
// workgroups of f32_mfma.hip: the streams of tiles are split over the waves of
// a workgroup, and a long dK/dV stream over several workgroups.
//
// Semantics and arithmetic are those of f32_mfma.hip (npu_flash_attention.py
// :17-166, :298-402, :407-560 and the group sum at :734-737): fp32 products on the
// matrix cores (v_mfma_f32_32x32x2_f32), softmax in the natural domain with
// expf / logf / tanhf.  The decomposition is that of fwd_split.hip and
// bwd_split.hip (packed query rows, KV items and Q items in one grid, the waves'
// results combined in wave order through LDS, the splits' sums by a second
// kernel); here
//  * a wave owns 32 rows (or keys), with their fp32 values as B operands in
//    registers (D/2 per lane), and its own pair of padded LDS tiles: at D = 128
//    34 KB, so that one wave runs on each SIMD with up to 512 registers;
//  * the next tiles pass through registers: fetched before a product of 64 or
//    more MFMAs over the current tile, stored to LDS after it.
// What bounds it: the MFMAs of a wave's chain of tiles (at D = 128 4096 cycles a
// product: two products a tile forward, four for dK/dV, three for dQ), where
// f32_mfma.hip walks the whole stream in one wave.
#include "f32_tiles.h"
#include "flexatt_kernels.h"

#ifndef FLEXATT_D
#error "FLEXATT_D (head dim) must be defined"
#endif

namespace flexatt {

#if FLEXATT_D <= 128

namespace {
constexpr int kNW = 4;  // waves per workgroup

template <int D>
struct FSplitCfg {
  using C = f32m::Cfg<D, 1>;             // one wave's tiles
  static constexpr int WAVEF = 2 * C::TILE + 64;  // floats per wave: a tile pair, LSE and Delta of 32 rows
  static constexpr int COMBF = kNW * 64 * (2 + 32 * C::DB);  // the combine: m, l and two accumulators
  static constexpr int LDSF = kNW * WAVEF > COMBF ? kNW * WAVEF : COMBF;
  static_assert(LDSF * 4 <= 160 * 1024, "LDS");
};

// A lane's half of one row as a B operand: x[s] = row[h D/2 + s].
template <int HD>
__device__ __forceinline__ void load_half_row(float (&x)[HD], const float* row, int h) {
#pragma unroll
  for (int s = 0; s < HD; s += 4) {
    const f32x4 v = *(const f32x4*)(row + h * HD + s);
#pragma unroll
    for (int e = 0; e < 4; ++e) x[s + e] = v[e];
  }
}
}  // namespace

template <int D, bool SOFTCAP, bool ALIBI>
__global__ __launch_bounds__(kNW * 64) __attribute__((amdgpu_waves_per_eu(D == 128 ? 1 : 2)))
void fwd_split_f32_kernel(DecodeArgs a) {
  using namespace f32m;
  using F = FSplitCfg<D>;
  using C = typename F::C;
  __shared__ __attribute__((aligned(16))) float smem[F::LDSF];
  const Shape& p = a.p;
  const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // the last row tiles, which have the longest causal range, go first
  const int nbh = p.B * p.Hkv, rt = a.nrt - 1 - (int)blockIdx.x / nbh, bh = blockIdx.x % nbh;
  const int hk = bh % p.Hkv, b = bh / p.Hkv;
  const int R = p.G * p.Sq, r = min(32 * rt + l32, R - 1);
  const int qi = r / p.G, hq = hk * p.G + r % p.G;
  float q[C::HD];
  load_half_row(q, (const float*)a.q.data + b * a.q.sb + hq * a.q.sh + (int64_t)qi * a.q.ss, h);
  const float slope = ALIBI ? p.alibi[hq] : 0.f;

  const int i0 = 32 * rt / p.G, i1 = min(32 * rt + 31, R - 1) / p.G;
  int lo, hi, l0, h0, l1, h1;
  doc_bounds(p, b, qi, lo, hi);
  doc_bounds(p, b, i0, l0, h0);
  doc_bounds(p, b, i1, l1, h1);
  lo = max(lo, 0), hi = min(hi, p.Skv);
  int k_lo = max(l0, 0), k_hi = min(h1, p.Skv);
  if (p.causal) hi = min(hi, qi + 1), k_hi = min(k_hi, i1 + 1);
  if (p.window > 0) lo = max(lo, qi - p.window), k_lo = max(k_lo, i0 - p.window);
  const unsigned w = (unsigned)max(hi - lo, 0);
  const int t0 = __builtin_amdgcn_readfirstlane(k_lo / kTile + wave);
  const int nt = __builtin_amdgcn_readfirstlane(max(((k_hi + kTile - 1) / kTile - t0 + kNW - 1) / kNW, 0));
  const float* kp = (const float*)a.k.data + b * a.k.sb + hk * a.k.sh;
  const float* vp = (const float*)a.v.data + b * a.v.sb + hk * a.v.sh;
  float* sK = smem + wave * F::WAVEF;
  float* sV = sK + C::TILE;

  f32x16 acc[C::DB];
#pragma unroll
  for (int db = 0; db < C::DB; ++db) acc[db] = f32x16{};
  float m_run = kNegInf, l_run = 0.f;
  Tile<D, 1> st;
  if (nt > 0) {
    st.fetch(sK, kp, a.k.ss, t0 * kTile, p.Skv, lane);
    st.commit(lane);
    st.fetch(sV, vp, a.v.ss, t0 * kTile, p.Skv, lane);
    st.commit(lane);
  }
  for (int j = 0; j < nt; ++j) {
    const int n0 = (t0 + kNW * j) * kTile, n1 = n0 + kNW * kTile;
    const bool more = j + 1 < nt;
    if (more) st.fetch(sK, kp, a.k.ss, n1, p.Skv, lane);
    f32x16 s = f32x16{};
    dsum<C::HD, C::P>(sK + l32 * C::P + h * C::HD, q, s);
    if (more) {
      st.commit(lane);
      st.fetch(sV, vp, a.v.ss, n1, p.Skv, lane);
    }
    const int a0 = lo - n0 - 4 * h;
    float mx = kNegInf;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      float t;
      float x = score<SOFTCAP, ALIBI>(s[e], p, slope, qi, n0 + blk_row(e, h), t);
      if ((unsigned)(8 * (e >> 2) + (e & 3) - a0) >= w) x = kNegInf;
      s[e] = x;
      mx = fmaxf(mx, x);
    }
    mx = fmaxf(mx, swap_halves(mx));
    const float m_new = fmaxf(m_run, mx);
    const float m_use = m_new == kNegInf ? 0.f : m_new;
    const float alpha = expf(m_run - m_use);
    l_run *= alpha;
#pragma unroll
    for (int db = 0; db < C::DB; ++db)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[db][e] *= alpha;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      s[e] = expf(s[e] - m_use);
      l_run += s[e];
    }
    m_run = m_new;
    rsum<C::DB, C::P>(sV, l32, h, s, acc);
    if (more) st.commit(lane);
  }

  const float l_tot = l_run + swap_halves(l_run);
  __syncthreads();
  float* xm = smem;                // [kNW][64]
  float* xl = xm + kNW * 64;       // [kNW][64]
  float* xa = xl + kNW * 64;       // [kNW][DB][16][64]
  xm[wave * 64 + lane] = m_run;
  xl[wave * 64 + lane] = l_tot;
#pragma unroll
  for (int db = 0; db < C::DB; ++db)
#pragma unroll
    for (int e = 0; e < 16; ++e) xa[((wave * C::DB + db) * 16 + e) * 64 + lane] = acc[db][e];
  __syncthreads();
  float m = kNegInf, al[kNW], L = 0.f;
#pragma unroll
  for (int v = 0; v < kNW; ++v) m = fmaxf(m, xm[v * 64 + lane]);
#pragma unroll
  for (int v = 0; v < kNW; ++v) {
    const float mv = xm[v * 64 + lane];
    al[v] = mv == kNegInf ? 0.f : expf(mv - m);
    L = fmaf(al[v], xl[v * 64 + lane], L);
  }
  const bool empty = L == 0.f;  // no key; NaN (a NaN query row or key) is not
  if (32 * rt + l32 < R) {
    float* out = (float*)a.o.data + b * a.o.sb + hq * a.o.sh + (int64_t)qi * a.o.ss + 4 * h;
    for (int x = wave; x < 4 * C::DB; x += kNW) {
      f32x4 o = f32x4{};
#pragma unroll
      for (int v = 0; v < kNW; ++v)
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = fmaf(al[v], xa[(v * C::DB * 16 + 4 * x + e) * 64 + lane], o[e]);
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = empty ? 0.f : o[e] / L;
      *(f32x4*)(out + 8 * x) = o;
    }
    if (wave == 0 && h == 0) a.lse[((int64_t)b * p.Hq + hq) * p.Sq + qi] = empty ? kNegInf : m + logf(L);
  }
}

template <int D, bool SOFTCAP, bool ALIBI>
__global__ __launch_bounds__(kNW * 64) __attribute__((amdgpu_waves_per_eu(D == 128 ? 1 : 2)))
void bwd_split_f32_kernel(BwdSplitArgs a) {
  using namespace f32m;
  using F = FSplitCfg<D>;
  using C = typename F::C;
  __shared__ __attribute__((aligned(16))) float smem[F::LDSF];
  const Shape& p = a.p;
  const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nbh = p.B * p.Hkv, R = p.G * p.Sq;
  float* s1 = smem + wave * F::WAVEF;  // Q or K
  float* s2 = s1 + C::TILE;            // dO or V
  float* sr = s2 + C::TILE;            // LSE, Delta of the tile's rows (KV items)
  const int off1 = l32 * C::P + h * C::HD;
  Tile<D, 1> st;

  const int nkv = a.nkt * nbh * a.nsplit;
  if ((int)blockIdx.x < nkv) {
    // ---- KV item: 32 KV rows, one share of the group's query tiles ---------
    const int split = blockIdx.x % a.nsplit;
    const int bh = blockIdx.x / a.nsplit % nbh, kt = blockIdx.x / a.nsplit / nbh;
    const int hk = bh % p.Hkv, b = bh / p.Hkv;
    const int n0 = 32 * kt, n1 = min(n0 + 31, p.Skv - 1);
    const int my_kv = n0 + l32, row = min(my_kv, p.Skv - 1);
    float kr[C::HD], vr[C::HD];
    load_half_row(kr, (const float*)a.k.data + b * a.k.sb + hk * a.k.sh + (int64_t)row * a.k.ss, h);
    load_half_row(vr, (const float*)a.v.data + b * a.v.sb + hk * a.v.sh + (int64_t)row * a.v.ss, h);
    int lo, hi, l0, h0, l1, h1;
    col_bounds(p, b, row, lo, hi);
    col_bounds(p, b, n0, l0, h0);
    col_bounds(p, b, n1, l1, h1);
    lo = max(lo, 0), hi = min(hi, p.Sq);
    int q_lo = max(l0, 0), q_hi = min(h1, p.Sq);
    if (p.causal) lo = max(lo, my_kv), q_lo = max(q_lo, n0);
    if (p.window > 0) hi = min(hi, my_kv + p.window + 1), q_hi = min(q_hi, n1 + p.window + 1);
    if (my_kv >= p.Skv) hi = lo;
    const unsigned w = (unsigned)max(hi - lo, 0);
    const int qt_lo = q_lo / 32, total = p.G * max((q_hi + 31) / 32 - qt_lo, 0);
    const int u_lo = (int)((int64_t)total * split / a.nsplit), u_hi = (int)((int64_t)total * (split + 1) / a.nsplit);
    const int u0 = __builtin_amdgcn_readfirstlane(u_lo + wave);
    const int nt = __builtin_amdgcn_readfirstlane(max((u_hi - u0 + kNW - 1) / kNW, 0));
    auto qptr = [&](int u) { return (const float*)a.q.data + b * a.q.sb + (hk * p.G + u % p.G) * a.q.sh; };
    auto optr = [&](int u) { return (const float*)a.dout.data + b * a.dout.sb + (hk * p.G + u % p.G) * a.dout.sh; };
    auto m0_of = [&](int u) { return 32 * (qt_lo + u / p.G); };
    // LSE (half 0) or Delta (half 1) of row l32 of tile u
    auto row_value = [&](int u) {
      const float x = (h ? a.delta : a.lse)[(int64_t)(b * p.Hq + hk * p.G + u % p.G) * p.Sq + min(m0_of(u) + l32, p.Sq - 1)];
      return !h && x == kNegInf ? kPosInf : x;  // a row with no allowed key: P = 0
    };
    f32x16 acc[2][C::DB];  // dK^T, dV^T
#pragma unroll
    for (int db = 0; db < C::DB; ++db) acc[0][db] = acc[1][db] = f32x16{};
    float rv = 0.f;
    if (nt > 0) {
      st.fetch(s1, qptr(u0), a.q.ss, m0_of(u0), p.Sq, lane);
      rv = row_value(u0);
      st.commit(lane);
      st.fetch(s2, optr(u0), a.dout.ss, m0_of(u0), p.Sq, lane);
      st.commit(lane);
      sr[lane] = rv;
    }
    for (int j = 0; j < nt; ++j) {
      const int u = u0 + kNW * j, un = u + kNW, m0 = m0_of(u);
      const bool more = j + 1 < nt;
      if (more) {
        st.fetch(s1, qptr(un), a.q.ss, m0_of(un), p.Sq, lane);
        rv = row_value(un);
      }
      f32x16 s = f32x16{}, dp = f32x16{};
      dsum<C::HD, C::P>(s1 + off1, kr, s);
      dsum<C::HD, C::P>(s2 + off1, vr, dp);
      const float slope = ALIBI ? p.alibi[hk * p.G + u % p.G] : 0.f;
      const int a0 = lo - m0 - 4 * h;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const f32x4 l4 = lds4(sr + 8 * i + 4 * h), d4 = lds4(sr + 32 + 8 * i + 4 * h);
#pragma unroll
        for (int jj = 0; jj < 4; ++jj) {
          const int e = 4 * i + jj;
          float t = 0.f;
          const float x = score<SOFTCAP, ALIBI>(s[e], p, slope, m0 + blk_row(e, h), my_kv, t);
          const float pj = (unsigned)(8 * i + jj - a0) < w ? expf(x - l4[jj]) : 0.f;
          float d = pj * (dp[e] - d4[jj]) * p.scale;
          if constexpr (SOFTCAP) d *= (1.0f - t * t);
          s[e] = pj;
          dp[e] = d;
        }
      }
      rsum<C::DB, C::P>(s1, l32, h, dp, acc[0]);
      if (more) {
        st.commit(lane);
        sr[lane] = rv;
        st.fetch(s2, optr(un), a.dout.ss, m0_of(un), p.Sq, lane);
      }
      rsum<C::DB, C::P>(s2, l32, h, s, acc[1]);
      if (more) st.commit(lane);
    }
    const bool in = my_kv < p.Skv;
    const int64_t pn = (int64_t)nbh * p.Skv * D;
    const int64_t prow = ((int64_t)bh * p.Skv + row) * D + 4 * h;
    float* dk = (float*)a.dk.data + b * a.dk.sb + hk * a.dk.sh + (int64_t)row * a.dk.ss + 4 * h;
    float* dv = (float*)a.dv.data + b * a.dv.sb + hk * a.dv.sh + (int64_t)row * a.dv.ss + 4 * h;
    combine_waves<2, C::DB, kNW>((char*)smem, acc, wave, lane, [&](int i, int db, int qr, f32x4 v) {
      float* dst = a.nsplit > 1 ? a.part + (2 * split + i) * pn + prow : i ? dv : dk;
      if (in) *(f32x4*)(dst + 32 * db + 8 * qr) = v;
    });
  } else {
    // ---- Q item: 32 packed query rows, every key tile they meet ------------
    const int item = blockIdx.x - nkv;
    const int bh = item % nbh, rt = a.nrt - 1 - item / nbh;
    const int hk = bh % p.Hkv, b = bh / p.Hkv;
    const int r = min(32 * rt + l32, R - 1);
    const int qi = r / p.G, hq = hk * p.G + r % p.G;
    float q[C::HD], g[C::HD];
    load_half_row(q, (const float*)a.q.data + b * a.q.sb + hq * a.q.sh + (int64_t)qi * a.q.ss, h);
    load_half_row(g, (const float*)a.dout.data + b * a.dout.sb + hq * a.dout.sh + (int64_t)qi * a.dout.ss, h);
    const int64_t srow = (int64_t)(b * p.Hq + hq) * p.Sq + qi;
    const float lse = a.lse[srow] == kNegInf ? kPosInf : a.lse[srow], dl = a.delta[srow];
    const float slope = ALIBI ? p.alibi[hq] : 0.f;
    const int i0 = 32 * rt / p.G, i1 = min(32 * rt + 31, R - 1) / p.G;
    int lo, hi, l0, h0, l1, h1;
    doc_bounds(p, b, qi, lo, hi);
    doc_bounds(p, b, i0, l0, h0);
    doc_bounds(p, b, i1, l1, h1);
    lo = max(lo, 0), hi = min(hi, p.Skv);
    int k_lo = max(l0, 0), k_hi = min(h1, p.Skv);
    if (p.causal) hi = min(hi, qi + 1), k_hi = min(k_hi, i1 + 1);
    if (p.window > 0) lo = max(lo, qi - p.window), k_lo = max(k_lo, i0 - p.window);
    const unsigned w = (unsigned)max(hi - lo, 0);
    const int t0 = __builtin_amdgcn_readfirstlane(k_lo / kTile + wave);
    const int nt = __builtin_amdgcn_readfirstlane(max(((k_hi + kTile - 1) / kTile - t0 + kNW - 1) / kNW, 0));
    const float* kp = (const float*)a.k.data + b * a.k.sb + hk * a.k.sh;
    const float* vp = (const float*)a.v.data + b * a.v.sb + hk * a.v.sh;
    f32x16 acc[1][C::DB];
#pragma unroll
    for (int db = 0; db < C::DB; ++db) acc[0][db] = f32x16{};
    if (nt > 0) {
      st.fetch(s2, vp, a.v.ss, t0 * kTile, p.Skv, lane);
      st.commit(lane);
      st.fetch(s1, kp, a.k.ss, t0 * kTile, p.Skv, lane);
      st.commit(lane);
    }
    for (int j = 0; j < nt; ++j) {
      const int n0 = (t0 + kNW * j) * kTile, n1 = n0 + kNW * kTile;
      const bool more = j + 1 < nt;
      if (more) st.fetch(s2, vp, a.v.ss, n1, p.Skv, lane);
      f32x16 s = f32x16{}, dp = f32x16{};
      dsum<C::HD, C::P>(s2 + off1, g, dp);
      if (more) {
        st.commit(lane);
        st.fetch(s1, kp, a.k.ss, n1, p.Skv, lane);
      }
      dsum<C::HD, C::P>(s1 + off1, q, s);
      const int a0 = lo - n0 - 4 * h;
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        float t = 0.f;
        const float x = score<SOFTCAP, ALIBI>(s[e], p, slope, qi, n0 + blk_row(e, h), t);
        const float pj = (unsigned)(8 * (e >> 2) + (e & 3) - a0) < w ? expf(x - lse) : 0.f;
        float d = pj * (dp[e] - dl) * p.scale;
        if constexpr (SOFTCAP) d *= (1.0f - t * t);
        s[e] = d;
      }
      rsum<C::DB, C::P>(s1, l32, h, s, acc[0]);
      if (more) st.commit(lane);
    }
    const bool in = 32 * rt + l32 < R;
    float* out = (float*)a.dq.data + b * a.dq.sb + hq * a.dq.sh + (int64_t)qi * a.dq.ss + 4 * h;
    combine_waves<1, C::DB, kNW>((char*)smem, acc, wave, lane, [&](int, int db, int qr, f32x4 v) {
      if (in) *(f32x4*)(out + 32 * db + 8 * qr) = v;
    });
  }
}

// dK and dV from the splits' sums, in split order: four columns per thread.
template <int D>
__global__ __launch_bounds__(256) void bwd_split_sum_f32_kernel(BwdSplitArgs a) {
  const Shape& p = a.p;
  const int64_t n = (int64_t)p.B * p.Hkv * p.Skv * D;
  const int64_t x = 4 * ((int64_t)blockIdx.x * 256 + threadIdx.x);
  if (x >= 2 * n) return;
  const int which = x >= n;
  const int64_t y = x - which * n, row = y / D, bh = row / p.Skv;
  f32x4 v = f32x4{};
  for (int s = 0; s < a.nsplit; ++s) v += *(const f32x4*)(a.part + (2 * s + which) * n + y);
  const MutView& t = which ? a.dv : a.dk;
  *(f32x4*)((float*)t.data + bh / p.Hkv * t.sb + bh % p.Hkv * t.sh + row % p.Skv * t.ss + y % D) = v;
}

#define FLEXATT_CAT2(a, b) a##b
#define FLEXATT_CAT(a, b) FLEXATT_CAT2(a, b)
hipError_t FLEXATT_CAT(fwd_split_f32_d, FLEXATT_D)(const DecodeArgs& a, hipStream_t st) {
  constexpr int D = FLEXATT_D;
  DecodeArgs x = a;
  x.nrt = (int)(((int64_t)a.p.G * a.p.Sq + 31) / 32);
  const dim3 grid(x.nrt * a.p.B * a.p.Hkv), block(kNW * 64);
  const bool sc = a.p.cap > 0.f, al = a.p.alibi != nullptr;
  if (sc && al) hipLaunchKernelGGL((fwd_split_f32_kernel<D, true, true>), grid, block, 0, st, x);
  else if (sc) hipLaunchKernelGGL((fwd_split_f32_kernel<D, true, false>), grid, block, 0, st, x);
  else if (al) hipLaunchKernelGGL((fwd_split_f32_kernel<D, false, true>), grid, block, 0, st, x);
  else hipLaunchKernelGGL((fwd_split_f32_kernel<D, false, false>), grid, block, 0, st, x);
  return hipGetLastError();
}
hipError_t FLEXATT_CAT(bwd_split_f32_d, FLEXATT_D)(const BwdSplitArgs& a, hipStream_t st) {
  constexpr int D = FLEXATT_D;
  BwdSplitArgs x = a;
  x.nkt = (a.p.Skv + 31) / 32;
  x.nrt = (a.p.G * a.p.Sq + 31) / 32;
  const dim3 grid(a.p.B * a.p.Hkv * (x.nkt * x.nsplit + x.nrt)), block(kNW * 64);
  const bool sc = a.p.cap > 0.f, al = a.p.alibi != nullptr;
  if (sc && al) hipLaunchKernelGGL((bwd_split_f32_kernel<D, true, true>), grid, block, 0, st, x);
  else if (sc) hipLaunchKernelGGL((bwd_split_f32_kernel<D, true, false>), grid, block, 0, st, x);
  else if (al) hipLaunchKernelGGL((bwd_split_f32_kernel<D, false, true>), grid, block, 0, st, x);
  else hipLaunchKernelGGL((bwd_split_f32_kernel<D, false, false>), grid, block, 0, st, x);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess || x.nsplit == 1) return e;
  const int64_t n = 2 * (int64_t)a.p.B * a.p.Hkv * a.p.Skv * D / 4;
  hipLaunchKernelGGL((bwd_split_sum_f32_kernel<D>), dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, x);
  return hipGetLastError();
}

#endif  // FLEXATT_D <= 128

}  // namespace flexatt
