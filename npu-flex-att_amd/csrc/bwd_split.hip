// Flash-attention backward for fp16/bf16 problems whose tiles fill too few of
// the staged or recomputing kernels' workgroups (bwd_kv.hip, bwd_q.hip): dK/dV
// and dQ in one launch, each item's stream of tiles split over the waves of its
// workgroup, and a dK/dV stream over several workgroups where one is too long.
//
// Semantics: npu_flash_attention.py:298-402 (dQ) and :407-560 with the group
// sum at :734-737 (dK/dV): P recomputed from the forward LSE (including the
// ALiBi bias, which the reference's backward kernels omit), dP = dO V^T,
// dS = P (dP - Delta) scale (1 - tanh^2), dV = P^T dO, dK = dS^T Q, dQ = dS K.
// P and dS are rounded to the input dtype before their MFMAs, as the
// reference does before tl.dot: dS with the scale in it at D = 32 and without it
// above (the gradient is scaled instead), as the kernels that larger problems of
// each head dim take round it, so that the size does not change fp16's range.
//
// Decomposition
//  * Two kinds of items in one grid, so that neither waits for the other:
//      - a KV item owns 32 KV rows of one (b, hkv) (the columns of its MFMA
//        tiles; K and V rows as B operands in registers) and streams the 32-row
//        Q / dO tiles of the group's G heads that can meet them;
//      - a Q item owns 32 query rows of one (b, hkv), packed with the G heads
//        innermost as in fwd_split.hip (Q and dO rows in registers), and streams
//        the 32-row K / V tiles of their key range.
//  * Wave w of an item takes tiles w, w + NW, ... of the stream on its own (two
//    LDS stages of a tile pair, direct-to-LDS copies one tile ahead, no
//    barriers): S and dP from the tiles' rows, P and dS on the VALU, which leave
//    as MFMA B operands in the registers they were computed in, then the
//    gradient MFMAs with the same tiles read as columns (LDS transpose reads).
//    The waves' accumulators are added in wave order through LDS at the end.
//  * A KV item's stream may be split further over `nsplit` workgroups, whose
//    fp32 sums go to the caller's workspace and are added in split order by a
//    second kernel.  Deterministic.
//  * What bounds it: the serial chain of a wave's tiles (at D = 64 about 0.9 us a
//    tile: 16 MFMAs, 128 VALU operations of softmax, two LDS round trips),
//    where the tile-stream kernels walk the whole stream in one workgroup.
#include "flexatt_device.h"
#include "flexatt_kernels.h"

#ifndef FLEXATT_D
#error "FLEXATT_D (head dim) must be defined"
#endif

namespace flexatt {

// dK and dV from the splits' sums, in split order: four columns per thread.
template <class T, int D>
__global__ __launch_bounds__(256) void bwd_split_sum_kernel(BwdSplitArgs a) {
  const Shape& p = a.p;
  const int64_t n = (int64_t)p.B * p.Hkv * p.Skv * D;
  const int64_t x = 4 * ((int64_t)blockIdx.x * 256 + threadIdx.x);
  if (x >= 2 * n) return;
  const int which = x >= n;
  const int64_t y = x - which * n, row = y / D, bh = row / p.Skv;
  f32x4 v = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int s = 0; s < a.nsplit; ++s) v += *(const f32x4*)(a.part + (2 * s + which) * n + y);
  const MutView& t = which ? a.dv : a.dk;
  T* dst = (T*)t.data + bh / p.Hkv * t.sb + bh % p.Hkv * t.sh + row % p.Skv * t.ss + y % D;
  st_global8(dst, pack4<T>(v[0], v[1], v[2], v[3]));
}

template <class T, int D>
hipError_t launch_split_sum(const BwdSplitArgs& a, hipStream_t st) {
  const int64_t n = 2 * (int64_t)a.p.B * a.p.Hkv * a.p.Skv * D / 4;
  hipLaunchKernelGGL((bwd_split_sum_kernel<T, D>), dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, a);
  return hipGetLastError();
}

#define FLEXATT_CAT2(a, b) a##b
#define FLEXATT_CAT(a, b) FLEXATT_CAT2(a, b)
hipError_t FLEXATT_CAT(bwd_split_sum_bf16_d, FLEXATT_D)(const BwdSplitArgs& a, hipStream_t st) {
  return launch_split_sum<__bf16, FLEXATT_D>(a, st);
}
hipError_t FLEXATT_CAT(bwd_split_sum_f16_d, FLEXATT_D)(const BwdSplitArgs& a, hipStream_t st) {
  return launch_split_sum<_Float16, FLEXATT_D>(a, st);
}

#if FLEXATT_D <= 128

template <int D, int NW>
struct BSplitCfg {
  static constexpr int KC = D / 16, DB = D / 32, CPR = D / 8, ROWB = 2 * D;
  static constexpr int TB = 32 * ROWB;       // bytes of one 32-row tile
  static constexpr int E = TB / 1024;        // 1 KB copies per tile
  static constexpr int STAGEB = 2 * TB + 256;  // a tile pair, and the LSE and Delta of its rows (KV items)
  static constexpr int WAVEB = 2 * STAGEB;
  static constexpr int COMBB = NW * 2 * DB * 16 * 64 * 4;  // the waves' dK^T and dV^T for the combine
  static constexpr int LDSB = NW * WAVEB > COMBB ? NW * WAVEB : COMBB;
  static_assert(E >= 1 && E * 1024 == TB && LDSB <= 160 * 1024, "LDS layout");
};

// One layout for both reads of a tile (rows and columns).
template <int CPR>
__device__ __forceinline__ int bsplit_swz(int r, int c) {
  if constexpr (CPR == 4) return c ^ ((r >> 2) & 3);
  else return swz_dual<CPR>(r, c);
}

template <class T, int D, int NW, bool SOFTCAP, bool ALIBI>
__global__ __launch_bounds__(NW * 64) void bwd_split_kernel(BwdSplitArgs a) {
  using C = BSplitCfg<D, NW>;
  using M = Mfma<T>;
  using V8 = typename M::v8;
  constexpr bool RAW = !SOFTCAP && !ALIBI;
  constexpr bool SCALED = D == 32;  // dS is rounded with the scale in it
  __shared__ __attribute__((aligned(1024))) char smem[C::LDSB];

  const Shape& p = a.p;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int h = lane >> 5, l32 = lane & 31;
  const int R = p.G * p.Sq;
  char* const wlds = smem + wave * C::WAVEB;
  const unsigned wbase = lds_addr_of(smem) + wave * C::WAVEB;

  // Lane-constant byte offsets of the row reads and the transpose reads in a tile.
  int rowoff[C::KC], clo[C::DB], chi[C::DB];
#pragma unroll
  for (int kc = 0; kc < C::KC; ++kc) rowoff[kc] = l32 * C::ROWB + bsplit_swz<C::CPR>(l32, 2 * kc + h) * 16;
  {
    const int tr_row = 4 * h + ((lane & 15) >> 2);
    const int tr_col = 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
#pragma unroll
    for (int db = 0; db < C::DB; ++db) {
      const int c = 4 * db + (tr_col >> 3), e2 = (tr_col & 7) * 2;
      clo[db] = tr_row * C::ROWB + bsplit_swz<C::CPR>(tr_row, c) * 16 + e2;
      chi[db] = (tr_row + 8) * C::ROWB + bsplit_swz<C::CPR>(tr_row + 8, c) * 16 + e2;
    }
  }
  // Rows [n0, n0 + 32) of a tensor (clamped to its last row) into a tile.
  auto copy_tile = [&](const T* base, int64_t ss, int n0, int last, unsigned dst) {
#pragma unroll
    for (int e = 0; e < C::E; ++e) {
      const int q = e * 64 + lane, row = q / C::CPR, pc = q % C::CPR;
      load_lds16(base + (int64_t)min(n0 + row, last) * ss + bsplit_swz<C::CPR>(row, pc) * 8, dst + e * 1024);
    }
  };
  auto reads_done = [] { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); };
  auto load_rows = [&](V8(&x)[C::KC], const View& t, int bb, int hh, int row, bool negate) {
    const T* src = (const T*)t.data + bb * t.sb + hh * t.sh + (int64_t)row * t.ss + 8 * h;
    const int s = negate ? (int)0x80008000 : 0;
#pragma unroll
    for (int kc = 0; kc < C::KC; ++kc) x[kc] = as_v8<V8>(ld_global16(src + 16 * kc) ^ i32x4{s, s, s, s});
  };
  // acc += A B^T over the head dim, A the rows of a tile, B a lane's row.
  auto rows_mma = [&](const char* tile, const V8(&x)[C::KC], f32x16& acc) {
#pragma unroll
    for (int kc = 0; kc < C::KC; ++kc) acc = M::mma(as_v8<V8>(lds_read16(tile + rowoff[kc])), x[kc], acc);
  };
  // acc[db] += A^T B over a tile's 32 rows, A the tile's columns, B the packed values.
  auto cols_mma = [&](const char* tile, const V8(&x)[2], f32x16(&acc)[C::DB]) {
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int db = 0; db < C::DB; ++db) {
        const char* t = tile + 16 * c * C::ROWB;
        acc[db] = M::mma(cat_tr<V8>(lds_read_tr4(t + clo[db]), lds_read_tr4(t + chi[db])), x[c], acc[db]);
      }
  };
  // P and -dS of a tile from its scores, LSE (log2 units) and Delta - dP;
  // masked elements are outside [lo, lo + w) of the element offsets
  // 8 (e / 4) + e % 4.
  auto form = [&](f32x16& s, f32x16& dp, auto lse2, auto slope, float dij0, float sgn, bool masked, int lo, unsigned w) {
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const int off = 8 * (e >> 2) + (e & 3);
      float t = 0.f, y;
      if constexpr (RAW) y = __builtin_fmaf(s[e], p.scale_log2, -lse2(e));
      else y = score_log2_d<SOFTCAP, ALIBI>(s[e], p, slope, dij0 + sgn * (float)off, t) - lse2(e);
      float x = fast_exp2(y);
      if (masked) x = (unsigned)(off - lo) < w ? x : 0.f;
      float ds = -x * dp[e];
      if constexpr (SCALED) ds *= p.scale;
      if constexpr (SOFTCAP) ds *= 1.f - t * t;
      s[e] = x;
      dp[e] = ds;
    }
  };

  const int nkv = a.nkt * p.B * p.Hkv * a.nsplit;
  if ((int)blockIdx.x < nkv) {
    // ---- KV item: 32 KV rows, one share of the group's query tiles ---------
    // (the first KV rows, which have the longest causal stream, go first)
    const int split = blockIdx.x % a.nsplit;
    const int bh = blockIdx.x / a.nsplit % (p.B * p.Hkv), kt = blockIdx.x / a.nsplit / (p.B * p.Hkv);
    const int hk = bh % p.Hkv, b = bh / p.Hkv;
    const int n0 = 32 * kt, n1 = min(n0 + 31, p.Skv - 1);
    const int my_kv = n0 + l32, row = min(my_kv, p.Skv - 1);
    V8 kr[C::KC], vr[C::KC];
    load_rows(kr, a.k, b, hk, row, false);
    load_rows(vr, a.v, b, hk, row, true);  // -V: the dP MFMAs start from Delta and end at Delta - dP

    // Query rows this lane's key meets, those some key of the item meets, and
    // those every key meets (column bounds are non-decreasing in the key).
    int lo, hi, l0, h0, l1, h1;
    col_bounds(p, b, row, lo, hi);
    col_bounds(p, b, n0, l0, h0);
    col_bounds(p, b, n1, l1, h1);
    lo = max(lo, 0), hi = min(hi, p.Sq);
    int q_lo = max(l0, 0), q_hi = min(h1, p.Sq), f_lo = max(l1, 0), f_hi = min(h0, p.Sq);
    if (p.causal) lo = max(lo, my_kv), q_lo = max(q_lo, n0), f_lo = max(f_lo, n1);
    if (p.window > 0) {
      hi = min(hi, my_kv + p.window + 1);
      q_hi = min(q_hi, n1 + p.window + 1);
      f_hi = min(f_hi, n0 + p.window + 1);
    }
    if (my_kv >= p.Skv) hi = lo;
    if (n0 + 32 > p.Skv) f_hi = 0;  // a KV tail: mask every tile
    const unsigned w = (unsigned)max(hi - lo, 0);
    const int qt_lo = q_lo / 32;
    const int total = p.G * max((q_hi + 31) / 32 - qt_lo, 0);
    const int u_lo = (int)((int64_t)total * split / a.nsplit), u_hi = (int)((int64_t)total * (split + 1) / a.nsplit);
    const int u0 = __builtin_amdgcn_readfirstlane(u_lo + wave);
    const int nt = __builtin_amdgcn_readfirstlane(max((u_hi - u0 + NW - 1) / NW, 0));
    f_lo = __builtin_amdgcn_readfirstlane(f_lo);
    f_hi = __builtin_amdgcn_readfirstlane(f_hi);

    constexpr int CNT = 2 * C::E + 1;
    auto issue = [&](int u, int st) {
      const int hq = hk * p.G + u % p.G, m0 = 32 * (qt_lo + u / p.G);
      const unsigned dst = wbase + st * C::STAGEB;
      copy_tile((const T*)a.q.data + b * a.q.sb + hq * a.q.sh, a.q.ss, m0, p.Sq - 1, dst);
      copy_tile((const T*)a.dout.data + b * a.dout.sb + hq * a.dout.sh, a.dout.ss, m0, p.Sq - 1, dst + C::TB);
      load_lds4((h ? a.delta : a.lse) + (int64_t)(b * p.Hq + hq) * p.Sq + min(m0 + l32, p.Sq - 1), dst + 2 * C::TB);
    };
    if (nt > 0) issue(u0, 0);
    // K and V land with the first tile (a wait inside the loop would drain
    // the copies in flight on every tile)
#pragma unroll
    for (int kc = 0; kc < C::KC; ++kc) {
      pin(kr[kc]);
      pin(vr[kc]);
    }
    f32x16 acc[2][C::DB];  // dK^T, dV^T
#pragma unroll
    for (int db = 0; db < C::DB; ++db) acc[0][db] = acc[1][db] = f32x16{};
    for (int j = 0; j < nt; ++j) {
      const int u = u0 + NW * j;
      if (j + 1 < nt) {
        reads_done();  // of tile j - 1, whose stage is refilled
        issue(u + NW, (j + 1) & 1);
        wait_vmcnt<CNT>();
      } else {
        wait_vmcnt<0>();
      }
      const char* sQ = wlds + (j & 1) * C::STAGEB;
      const char* sO = sQ + C::TB;
      const char* sR = sO + C::TB;  // LSE then Delta
      const int m0 = 32 * (qt_lo + u / p.G);
      f32x16 s = f32x16{}, dp;
      f32x4 L[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        L[i] = __builtin_bit_cast(f32x4, lds_read16(sR + 4 * (8 * i + 4 * h)));
        const f32x4 d4 = __builtin_bit_cast(f32x4, lds_read16(sR + 128 + 4 * (8 * i + 4 * h)));
#pragma unroll
        for (int jj = 0; jj < 4; ++jj) {
          L[i][jj] *= kLog2e;
          dp[4 * i + jj] = d4[jj];
        }
      }
      rows_mma(sQ, kr, s);
      rows_mma(sO, vr, dp);
      const float slope = ALIBI ? p.alibi[hk * p.G + u % p.G] * kLog2e : 0.f;
      form(s, dp, [&](int e) { return L[e >> 2][e & 3]; }, slope, (float)(m0 + 4 * h - my_kv), 1.f,
           m0 < f_lo || m0 + 32 > f_hi, lo - m0 - 4 * h, w);
      const V8 P[2] = {pack8<T>(s, 0), pack8<T>(s, 8)};
      const V8 S[2] = {pack8<T>(dp, 0), pack8<T>(dp, 8)};
      cols_mma(sO, P, acc[1]);
      cols_mma(sQ, S, acc[0]);
    }
    const bool in = my_kv < p.Skv;
    const int64_t prow = ((int64_t)bh * p.Skv + row) * D + 4 * h;
    const int64_t pn = (int64_t)p.B * p.Hkv * p.Skv * D;
    T* out[2] = {(T*)a.dk.data + b * a.dk.sb + hk * a.dk.sh + (int64_t)row * a.dk.ss + 4 * h,
                 (T*)a.dv.data + b * a.dv.sb + hk * a.dv.sh + (int64_t)row * a.dv.ss + 4 * h};
    combine_waves<2, C::DB, NW>(smem, acc, wave, lane, [&](int i, int db, int qr, f32x4 v) {
      if (!SCALED && i == 0) v *= p.scale;
      if (!in) return;
      const int col = 32 * db + 8 * qr;
      if (a.nsplit > 1) *(f32x4*)(a.part + (2 * split + i) * pn + prow + col) = v;
      else st_global8((i ? out[1] : out[0]) + col, pack4<T>(v[0], v[1], v[2], v[3]));
    });
  } else {
    // ---- Q item: 32 packed query rows, every key tile they meet ------------
    const int item = blockIdx.x - nkv;
    const int bh = item % (p.B * p.Hkv), rt = a.nrt - 1 - item / (p.B * p.Hkv);
    const int hk = bh % p.Hkv, b = bh / p.Hkv;
    const int r = min(32 * rt + l32, R - 1);
    const int qi = r / p.G, hq = hk * p.G + r % p.G;
    V8 qr[C::KC], dr[C::KC];
    load_rows(qr, a.q, b, hq, qi, false);
    load_rows(dr, a.dout, b, hq, qi, true);  // -dO: dP^T starts from Delta and ends at Delta - dP
    const int64_t srow = (int64_t)(b * p.Hq + hq) * p.Sq + qi;
    float lse2 = a.lse[srow] * kLog2e, dlt = a.delta[srow];
    // a row with no allowed key: +inf makes its P zero (every pair is masked)
    if (!(lse2 > kNegInf)) lse2 = kPosInf;
    float slope = ALIBI ? p.alibi[hq] * kLog2e : 0.f;

    const int i0 = 32 * rt / p.G, i1 = min(32 * rt + 31, R - 1) / p.G;
    int lo, hi, l0, h0, l1, h1;
    doc_bounds(p, b, qi, lo, hi);
    doc_bounds(p, b, i0, l0, h0);
    doc_bounds(p, b, i1, l1, h1);
    lo = max(lo, 0), hi = min(hi, p.Skv);
    int k_lo = max(l0, 0), k_hi = min(h1, p.Skv), f_lo = max(l1, 0), f_hi = min(h0, p.Skv);
    if (p.causal) hi = min(hi, qi + 1), k_hi = min(k_hi, i1 + 1), f_hi = min(f_hi, i0 + 1);
    if (p.window > 0) {
      lo = max(lo, qi - p.window);
      k_lo = max(k_lo, i0 - p.window);
      f_lo = max(f_lo, i1 - p.window);
    }
    const unsigned w = (unsigned)max(hi - lo, 0);
    const int t0 = __builtin_amdgcn_readfirstlane(k_lo / 32 + wave);
    const int nt = __builtin_amdgcn_readfirstlane(max(((k_hi + 31) / 32 - t0 + NW - 1) / NW, 0));
    f_lo = __builtin_amdgcn_readfirstlane(f_lo);
    f_hi = __builtin_amdgcn_readfirstlane(f_hi);
    const T* kp = (const T*)a.k.data + b * a.k.sb + hk * a.k.sh;
    const T* vp = (const T*)a.v.data + b * a.v.sb + hk * a.v.sh;
    auto issue = [&](int t, int st) {
      copy_tile(kp, a.k.ss, 32 * t, p.Skv - 1, wbase + st * C::STAGEB);
      copy_tile(vp, a.v.ss, 32 * t, p.Skv - 1, wbase + st * C::STAGEB + C::TB);
    };
    if (nt > 0) issue(t0, 0);
#pragma unroll
    for (int kc = 0; kc < C::KC; ++kc) {
      pin(qr[kc]);
      pin(dr[kc]);
    }
    pin(lse2);
    pin(dlt);
    if constexpr (ALIBI) pin(slope);
    f32x16 acc[1][C::DB];
#pragma unroll
    for (int db = 0; db < C::DB; ++db) acc[0][db] = f32x16{};
    for (int j = 0; j < nt; ++j) {
      const int t = t0 + NW * j, n0 = 32 * t;
      if (j + 1 < nt) {
        reads_done();
        issue(t + NW, (j + 1) & 1);
        wait_vmcnt<2 * C::E>();
      } else {
        wait_vmcnt<0>();
      }
      const char* sK = wlds + (j & 1) * C::STAGEB;
      f32x16 s = f32x16{}, dp;
#pragma unroll
      for (int e = 0; e < 16; ++e) dp[e] = dlt;
      rows_mma(sK, qr, s);
      rows_mma(sK + C::TB, dr, dp);
      form(s, dp, [&](int) { return lse2; }, slope, (float)(qi - n0 - 4 * h), -1.f, n0 < f_lo || n0 + 32 > f_hi,
           lo - n0 - 4 * h, w);
      const V8 S[2] = {pack8<T>(dp, 0), pack8<T>(dp, 8)};
      cols_mma(sK, S, acc[0]);
    }
    const bool in = 32 * rt + l32 < R;
    T* out = (T*)a.dq.data + b * a.dq.sb + hq * a.dq.sh + (int64_t)qi * a.dq.ss + 4 * h;
    combine_waves<1, C::DB, NW>(smem, acc, wave, lane, [&](int, int db, int qr4, f32x4 v) {
      if (!SCALED) v *= p.scale;
      if (in) st_global8(out + 32 * db + 8 * qr4, pack4<T>(v[0], v[1], v[2], v[3]));
    });
  }
}

template <class T, int D, int NW>
hipError_t launch_bwd_split(const BwdSplitArgs& a, hipStream_t st) {
  const dim3 grid(a.p.B * a.p.Hkv * (a.nkt * a.nsplit + a.nrt)), block(NW * 64);
  const bool sc = a.p.cap > 0.f, al = a.p.alibi != nullptr;
  if (sc && al) hipLaunchKernelGGL((bwd_split_kernel<T, D, NW, true, true>), grid, block, 0, st, a);
  else if (sc) hipLaunchKernelGGL((bwd_split_kernel<T, D, NW, true, false>), grid, block, 0, st, a);
  else if (al) hipLaunchKernelGGL((bwd_split_kernel<T, D, NW, false, true>), grid, block, 0, st, a);
  else hipLaunchKernelGGL((bwd_split_kernel<T, D, NW, false, false>), grid, block, 0, st, a);
  const hipError_t e = hipGetLastError();
  return e != hipSuccess || a.nsplit == 1 ? e : launch_split_sum<T, D>(a, st);
}

template <class T, int D>
hipError_t launch_bwd_split(const BwdSplitArgs& a, hipStream_t st) {
  BwdSplitArgs x = a;
  x.nkt = (a.p.Skv + 31) / 32;
  x.nrt = (a.p.G * a.p.Sq + 31) / 32;
  if constexpr (D <= 64) {
    if (x.nw == 8) return launch_bwd_split<T, D, 8>(x, st);
  }
  return launch_bwd_split<T, D, 4>(x, st);
}

hipError_t FLEXATT_CAT(bwd_split_bf16_d, FLEXATT_D)(const BwdSplitArgs& a, hipStream_t st) {
  return launch_bwd_split<__bf16, FLEXATT_D>(a, st);
}
hipError_t FLEXATT_CAT(bwd_split_f16_d, FLEXATT_D)(const BwdSplitArgs& a, hipStream_t st) {
  return launch_bwd_split<_Float16, FLEXATT_D>(a, st);
}

#endif  // FLEXATT_D <= 128

}  // namespace flexatt
