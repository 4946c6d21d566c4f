// Forward with the KV range split over the waves of a workgroup, and over
// workgroups where one is not enough: KV-cache decoding, and any problem whose
// query rows fill too few of the regular forward's 256-row workgroups.
//
// Semantics: those of the forward, npu_flash_attention.py:17-166 (score order
// scale -> soft-cap -> ALiBi -> mask, online softmax in the log2 domain, LSE
// in natural log).  The reference sketches a split at :169-293
// (flash_attn_fwd_split_kv_kernel / flash_attn_fwd_reduce_kernel) but never
// calls it; this is a gfx950 design of its own.
//
// Decomposition
//  * The G * Sq query rows of one KV head (G = Hq / Hkv) are packed row-major
//    with the heads innermost (row r: query row r / G of head r % G) into tiles
//    of 32, the columns of one MFMA tile: heads that share K/V read it
//    once, and the rows of a tile have nearly one causal range.  (Unused
//    columns of the last tile repeat the last row and are not written.)
//  * One workgroup = NW waves for one row tile of one (b, hkv) and one
//    contiguous chunk of 32-row KV tiles; wave w takes tiles w, w + NW, ...
//    of the chunk on its own: its own LDS stages (K with the column-read
//    swizzle, V with the transpose-read swizzle, direct-to-LDS copies), its own
//    online softmax, no barriers.
//  * The waves' online-softmax states are combined through LDS.  With one
//    chunk per row tile the workgroup writes O and LSE itself.  Otherwise it
//    writes one partial result: O normalised by its row sums (fp32) and
//    its LSE in log2 units, in the caller's workspace, and a merge kernel (one
//    workgroup per row) combines the partials of a row in a fixed
//    order: M = max LSE_s, O = sum 2^(LSE_s - M) O_s / sum 2^(LSE_s - M),
//    LSE = (M + log2 sum 2^(LSE_s - M)) ln 2.  A partial without keys has LSE
//    -inf and is left out; one with a NaN score has LSE NaN, which makes the
//    row's O and LSE NaN.  Deterministic.
//  * What bounds it: long decodes stream K and V from HBM (two stages per
//    wave, 5.8 TB/s at bf16 B=8 Hkv=8 Skv=32768 D=128); everything smaller is
//    a chain of tiles, each one LDS round trip, one softmax and one more round
//    trip, which the split shortens by the number of waves.
#include "flexatt_device.h"
#include "flexatt_kernels.h"

#ifndef FLEXATT_D
#error "FLEXATT_D (head dim) must be defined"
#endif

namespace flexatt {

constexpr float kDecRescale = 8.0f;  // lazy rescale threshold, log2 units (as the forward)

// NW waves per workgroup.  ST = 2: two stages of a K and a V tile per wave, the
// next tile in flight during the whole of this one (four such waves beat two,
// or four with four stages and fewer waves per CU, 5.6 against 4.6 TB/s at
// D = 128).  ST = 1: one K and one V buffer, K refilled after the tile's S
// MFMAs and V after its PV MFMAs, at half the LDS: D = 256, and problems of
// many row tiles, where it lets a second workgroup onto the CU.
template <int D, int NW, int ST>
struct SplitCfg {
  static constexpr int BN = 32;          // KV rows per tile
  static constexpr int KC = D / 16;      // k steps of S^T = K Q^T
  static constexpr int DB = D / 32;      // 32-row blocks of O^T
  static constexpr int CPR = D / 8;      // 16-byte chunks per row
  static constexpr int ROWB = 2 * D;     // bytes per row
  static constexpr int TB = BN * ROWB;   // bytes of one K or V tile
  static constexpr int E = TB / 1024;    // 1 KB copies per tile per tensor
  static constexpr int WAVEB = ST * 2 * TB;  // LDS bytes per wave
  static constexpr int COMBB = NW * 64 * 4 * (2 + 16 * DB);  // the waves' m, l and O^T for the combine
  static constexpr int LDSB = NW * WAVEB > COMBB ? NW * WAVEB : COMBB;
  static_assert(E >= 1 && E * 1024 == TB, "tile must split into 1 KB copies");
  static_assert(LDSB <= 160 * 1024, "LDS");
};

template <class T, int D, int NW, int ST, bool SOFTCAP, bool ALIBI>
__global__ __launch_bounds__(NW * 64) __attribute__((amdgpu_waves_per_eu(D == 256 ? 1 : 2)))
void fwd_split_kernel(DecodeArgs a) {
  using C = SplitCfg<D, NW, ST>;
  using M = Mfma<T>;
  using V8 = typename M::v8;
  __shared__ __attribute__((aligned(1024))) char smem[C::LDSB];

  const Shape& p = a.p;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int h = lane >> 5, l32 = lane & 31;

  // Work item: (b, hkv, row tile, split); the splits of one row tile are
  // consecutive, and its last row tile (the longest causal range) goes first.
  // Row tiles of one (b, hkv) share an XCD; a single one (decoding) has nothing
  // to share, and contiguous ranges per XCD then only bunch the cache's
  // addresses: bf16 D=64 B=128 Hq=32 Hkv=8 Skv=8192 389 -> 367 us in plain order,
  // D=32 Skv=16384 384 -> 370, D=128 B=64 704 -> 700.
  const int s = blockIdx.x % a.nsplit;
  const int item = blockIdx.x / a.nsplit;
  int krt, bh;
  if (a.plain || !xcd_lpt_item(item, a.nrt, p.B * p.Hkv, krt, bh)) {
    krt = item % a.nrt;
    bh = item / a.nrt;
  }
  const int rt = a.nrt - 1 - krt;
  const int hk = bh % p.Hkv, b = bh / p.Hkv;

  // Packed query row of this lane.
  const int R = p.G * p.Sq;
  const int r = min(32 * rt + l32, R - 1);
  const int g = r % p.G, qi = r / p.G;
  const int hq = hk * p.G + g;

  // Q^T as MFMA B operands (k = 8 consecutive d of query row qi).
  V8 qf[C::KC];
  {
    const T* src = (const T*)a.q.data + b * a.q.sb + hq * a.q.sh + (int64_t)qi * a.q.ss + 8 * h;
#pragma unroll
    for (int kc = 0; kc < C::KC; ++kc) qf[kc] = as_v8<V8>(ld_global16(src + 16 * kc));
  }

  // The keys [row_lo, row_lo + row_w) this lane's row attends to, the tiles
  // [t_lo, t_hi) of the workgroup, and the keys [full_lo, full_hi) every row of
  // the tile attends to (all bounds are non-decreasing in the query row).
  const int i0 = 32 * rt / p.G, i1 = min(32 * rt + 31, R - 1) / p.G;
  int row_lo, row_hi, dl0, dh0, dl1, dh1;
  doc_bounds(p, b, qi, row_lo, row_hi);
  doc_bounds(p, b, i0, dl0, dh0);
  doc_bounds(p, b, i1, dl1, dh1);
  row_lo = max(row_lo, 0);
  row_hi = min(row_hi, p.Skv);
  int kv_lo = max(dl0, 0), kv_hi = min(dh1, p.Skv), full_lo = max(dl1, 0), full_hi = min(dh0, p.Skv);
  if (p.causal) {
    row_hi = min(row_hi, qi + 1);
    kv_hi = min(kv_hi, i1 + 1);
    full_hi = min(full_hi, i0 + 1);
  }
  if (p.window > 0) {
    row_lo = max(row_lo, qi - p.window);
    kv_lo = max(kv_lo, i0 - p.window);
    full_lo = max(full_lo, i1 - p.window);
  }
  const unsigned row_w = (unsigned)max(row_hi - row_lo, 0);
  full_lo = __builtin_amdgcn_readfirstlane(full_lo);
  full_hi = __builtin_amdgcn_readfirstlane(full_hi);

  // This wave's tiles: first + NW * j, j < nt.
  const int t_lo = max(kv_lo / C::BN, s * a.chunk);
  const int t_hi = min((kv_hi + C::BN - 1) / C::BN, a.nsplit > 1 ? (s + 1) * a.chunk : 0x7fffffff);
  const int first = __builtin_amdgcn_readfirstlane(t_lo + wave);
  const int nt = __builtin_amdgcn_readfirstlane(max((t_hi - first + NW - 1) / NW, 0));

  const T* kp = (const T*)a.k.data + b * a.k.sb + hk * a.k.sh;
  const T* vp = (const T*)a.v.data + b * a.v.sb + hk * a.v.sh;
  const unsigned wbase = lds_addr_of(smem) + wave * C::WAVEB;
  auto issue_k = [&](int t, int st) {
#pragma unroll
    for (int e = 0; e < C::E; ++e) {
      const int q = e * 64 + lane, row = q / C::CPR, pc = q % C::CPR;
      const int64_t n = min(t * C::BN + row, p.Skv - 1);
      load_lds16(kp + n * a.k.ss + swz_col<C::CPR>(row, pc) * 8, wbase + st * 2 * C::TB + e * 1024);
    }
  };
  auto issue_v = [&](int t, int st) {
#pragma unroll
    for (int e = 0; e < C::E; ++e) {
      const int q = e * 64 + lane, row = q / C::CPR, pc = q % C::CPR;
      const int64_t n = min(t * C::BN + row, p.Skv - 1);
      load_lds16(vp + n * a.v.ss + swz_tr_inv<C::CPR>(row, pc) * 8, wbase + st * 2 * C::TB + C::TB + e * 1024);
    }
  };
  // this wave's LDS reads have returned: the buffer they read may be refilled
  auto reads_done = [] { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); };
  if (nt > 0) {
    issue_k(first, 0);
    issue_v(first, 0);
  }

  constexpr bool RAW = !SOFTCAP && !ALIBI;
  float c2 = p.scale_log2;
  if constexpr (RAW) {  // as in the forward: a negative scale moves into Q
    if (c2 < 0.f) {
#pragma unroll
      for (int kc = 0; kc < C::KC; ++kc)
        qf[kc] = as_v8<V8>(__builtin_bit_cast(i32x4, qf[kc]) ^ i32x4{(int)0x80008000, (int)0x80008000,
                                                                     (int)0x80008000, (int)0x80008000});
      c2 = -c2;
    }
    if (c2 == 0.f) c2 = 1e-30f;
  }
  float slope_log2 = ALIBI ? p.alibi[hq] * kLog2e : 0.f;
  // Wait for Q here, once, together with the first tile: without the pins the
  // compiler waits at the first use, inside the tile loop, where its vmcnt(0)
  // drains the copies in flight on every tile.
#pragma unroll
  for (int kc = 0; kc < C::KC; ++kc) pin(qf[kc]);
  if constexpr (ALIBI) pin(slope_log2);

  int koff[C::KC], voff[C::DB];
  {
    const int tr_row = 4 * h + ((lane & 15) >> 2);
    const int tr_col = 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
#pragma unroll
    for (int kc = 0; kc < C::KC; ++kc) koff[kc] = l32 * C::ROWB + swz_col<C::CPR>(l32, 2 * kc + h) * 16;
#pragma unroll
    for (int db = 0; db < C::DB; ++db)
      voff[db] = tr_row * C::ROWB + swz_tr<C::CPR>(tr_row, 4 * db + (tr_col >> 3)) * 16 + (tr_col & 7) * 2;
  }

  f32x16 acc[C::DB];
#pragma unroll
  for (int db = 0; db < C::DB; ++db) acc[db] = f32x16{};
  float m_run = kNegInf, l_run = 0.f;

  for (int j = 0; j < nt; ++j) {
    const int t = first + NW * j;
    const bool more = j + 1 < nt;
    if constexpr (ST == 2) {
      if (more) {  // into the stage of tile j - 1, read in the previous iteration
        reads_done();
        issue_k(t + NW, (j + 1) & 1);
        issue_v(t + NW, (j + 1) & 1);
        wait_vmcnt<2 * C::E>();  // tile j landed, the next in flight
      } else {
        wait_vmcnt<0>();
      }
    } else {
      wait_vmcnt<C::E>();  // K of tile j landed (its V, issued later, may be in flight)
    }
    const char* sK = smem + wave * C::WAVEB + (ST == 2 ? (j & 1) * 2 * C::TB : 0);
    const char* sV = sK + C::TB;
    const int n0 = t * C::BN;

    f32x16 sc = f32x16{};
#pragma unroll
    for (int kc = 0; kc < C::KC; ++kc) sc = M::mma(as_v8<V8>(lds_read16(sK + koff[kc])), qf[kc], sc);
    if constexpr (ST == 1) {
      reads_done();
      if (more) issue_k(t + NW, 0);
    }

    // element e is KV row n0 + 8(e/4) + 4h + e%4, query row qi of head hq
    if constexpr (!RAW) {
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int jj = n0 + 8 * (e >> 2) + 4 * h + (e & 3);
        float tv;
        sc[e] = score_log2<SOFTCAP, ALIBI>(sc[e], p, slope_log2, qi, jj, tv);
      }
    }
    if (n0 < full_lo || n0 + C::BN > full_hi) {
      const int a0 = row_lo - n0 - 4 * h;
#pragma unroll
      for (int e = 0; e < 16; ++e)
        if ((unsigned)(8 * (e >> 2) + (e & 3) - a0) >= row_w) sc[e] = kNegInf;
    }
    float mx, mx2;
    max16_partial(sc, mx, mx2);
    mx = max2(mx, mx2);
    if constexpr (RAW) mx *= c2;
    mx = fmaxf(mx, swap_halves(mx));
    if (mx != mx) mx = kNegInf;
    const bool grow = mx > m_run + kDecRescale;
    if (__builtin_amdgcn_ballot_w64(grow)) {
      const float m_new = grow ? mx : m_run;
      const float alpha = grow ? fast_exp2(m_run - m_new) : 1.f;
      l_run *= alpha;
#pragma unroll
      for (int db = 0; db < C::DB; ++db) scale_inplace(acc[db], alpha);
      m_run = m_new;
    }
    const float m_use = (m_run == kNegInf) ? 0.f : m_run;
    f32x16 pe;
    float rs[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      if constexpr (RAW) pe[e] = fast_exp2(__builtin_fmaf(sc[e], c2, -m_use));
      else pe[e] = fast_exp2(sc[e] - m_use);
      rs[e & 3] += pe[e];
    }
    l_run += (rs[0] + rs[1]) + (rs[2] + rs[3]);
    if constexpr (ST == 1) {  // V of tile j landed (the next K may be in flight)
      if (more) wait_vmcnt<C::E>();
      else wait_vmcnt<0>();
    }
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const V8 pb = pack8<T>(pe, 8 * c);
      const char* vr = sV + 16 * c * C::ROWB;
#pragma unroll
      for (int db = 0; db < C::DB; ++db) {
        const i16x4 lo = lds_read_tr4(vr + voff[db]);
        const i16x4 hi = lds_read_tr4(vr + 8 * C::ROWB + voff[db]);
        acc[db] = M::mma(cat_tr<V8>(lo, hi), pb, acc[db]);
      }
    }
    if constexpr (ST == 1) {
      reads_done();
      if (more) issue_v(t + NW, 0);
    }
  }

  // The workgroup's result: the NW waves' (m, l, acc) combined in a fixed
  // order through LDS (every wave's copies have landed: its last tile waited
  // for vmcnt 0), then O / l and LSE.
  const float l_tot = l_run + swap_halves(l_run);  // this wave's row sum
  __syncthreads();
  float* xm = (float*)smem;         // [NW][64]
  float* xl = xm + NW * 64;         // [NW][64]
  float* xa = xl + NW * 64;         // [NW][DB][16][64]
  xm[wave * 64 + lane] = m_run;
  xl[wave * 64 + lane] = l_tot;
#pragma unroll
  for (int db = 0; db < C::DB; ++db)
#pragma unroll
    for (int e = 0; e < 16; ++e) xa[((wave * C::DB + db) * 16 + e) * 64 + lane] = acc[db][e];
  __syncthreads();
  float mw[NW], mall = kNegInf;
#pragma unroll
  for (int w = 0; w < NW; ++w) {
    mw[w] = xm[w * 64 + lane];
    mall = fmaxf(mall, mw[w]);
  }
  float al[NW], L = 0.f;
#pragma unroll
  for (int w = 0; w < NW; ++w) {
    al[w] = mw[w] == kNegInf ? 0.f : fast_exp2(mw[w] - mall);  // 0 for a wave without keys
    L = __builtin_fmaf(al[w], xl[w * 64 + lane], L);
  }
  const bool empty = L == 0.f;  // no key; NaN (a NaN query row or key) is not
  const float inv = empty ? 0.f : 1.0f / L;
  if (32 * rt + l32 < R) {
    const int64_t row = ((int64_t)b * p.Hq + hq) * p.Sq + qi;
    float* po = a.part_o + (row * a.nsplit + s) * D + 4 * h;
    T* out = (T*)a.o.data + b * a.o.sb + hq * a.o.sh + (int64_t)qi * a.o.ss + 4 * h;
    for (int x = wave; x < 4 * C::DB; x += NW) {  // 4 columns of this row per half wave
      f32x4 o = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int w = 0; w < NW; ++w)
#pragma unroll
        for (int j = 0; j < 4; ++j) o[j] = __builtin_fmaf(al[w], xa[(w * C::DB * 16 + 4 * x + j) * 64 + lane], o[j]);
      o *= inv;
      if (a.nsplit > 1) *(f32x4*)(po + 8 * x) = o;
      else st_global8(out + 8 * x, pack4<T>(o[0], o[1], o[2], o[3]));
    }
    if (wave == 0 && h == 0) {
      const float lse = empty ? kNegInf : mall + log2f(L);
      if (a.nsplit > 1) a.part_lse[row * a.nsplit + s] = lse;
      else a.lse[row] = lse * kLn2;
    }
  }
}

// Merge of the workgroups' partials: one workgroup per row, four columns per
// thread, D / 4 threads for every NG-th partial.  Latency-bound (a row is a few KB
// that the partials' launch left in cache): the LSEs are read by the lanes of a
// wave at once and the first partials are in flight meanwhile, where one thread
// per output element walked the row's LSEs twice, each a dependent load.
// The NG sums are added in order through LDS.  bf16 B=2 Hq=16 Hkv=8 Skv=4097 D=256,
// 15 partials of 32 rows: 5.4 -> 4.0 us.
template <class T, int D>
__global__ __launch_bounds__(256) void fwd_split_merge_kernel(DecodeArgs a) {
  constexpr int TPR = D / 4, NG = 256 / TPR, U = 4;
  __shared__ f32x4 sums[NG][TPR];
  const Shape& p = a.p;
  const int tid = threadIdx.x, lane = tid & 63;
  const int c = tid % TPR, g = tid / TPR;
  const int64_t row = blockIdx.x;
  const int ns = a.nsplit;  // at most 256
  const float* pl = a.part_lse + row * ns;
  const f32x4* po = (const f32x4*)(a.part_o + row * ns * D) + c;

  f32x4 v[U];
  float lw[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {  // (a partial past the last: the last again, without a weight)
    const int s = g + NG * u, t = min(s, ns - 1);
    v[u] = po[(int64_t)t * TPR];
    lw[u] = s < ns ? pl[t] : kNegInf;
  }
  float ll[4], mx = kNegInf;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int s = lane + 64 * k;
    ll[k] = s < ns ? pl[s] : kNegInf;
    mx = fmaxf(mx, ll[k]);
  }
#pragma unroll
  for (int x = 32; x; x >>= 1) mx = fmaxf(mx, __shfl_xor(mx, x));
  const float m0 = mx == kNegInf ? 0.f : mx;
  float ws = 0.f;
#pragma unroll
  for (int k = 0; k < 4; ++k) ws += fast_exp2(ll[k] - m0);  // 0 for an empty partial
#pragma unroll
  for (int x = 32; x; x >>= 1) ws += __shfl_xor(ws, x);
  const bool none = ws == 0.f;  // no allowed key for this row

  f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int s0 = g;;) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const float w = fast_exp2(lw[u] - m0);
      const bool keys = lw[u] != kNegInf;  // without keys the values do not count, not even an inf
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[j] = keys ? __builtin_fmaf(w, v[u][j], acc[j]) : acc[j];
    }
    s0 += NG * U;
    if (s0 >= ns) break;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int s = s0 + NG * u, t = min(s, ns - 1);
      v[u] = po[(int64_t)t * TPR];
      lw[u] = s < ns ? pl[t] : kNegInf;
    }
  }
  sums[g][c] = acc;
  __syncthreads();
  if (g != 0) return;
#pragma unroll
  for (int k = 1; k < NG; ++k) acc += sums[k][c];
  const int i = (int)(row % p.Sq);
  const int64_t bh = row / p.Sq;
  const int hq = (int)(bh % p.Hq), b = (int)(bh / p.Hq);
  T* out = (T*)a.o.data + b * a.o.sb + hq * a.o.sh + (int64_t)i * a.o.ss + 4 * c;
#pragma unroll
  for (int j = 0; j < 4; ++j) acc[j] = none ? 0.f : acc[j] / ws;
  st_global8(out, pack4<T>(acc[0], acc[1], acc[2], acc[3]));
  if (c == 0) a.lse[row] = none ? kNegInf : (mx + log2f(ws)) * kLn2;
}

template <class T, int D, int NW, int ST>
hipError_t launch_split(const DecodeArgs& a, hipStream_t st) {
  const dim3 grid(a.nsplit * a.nrt * a.p.B * a.p.Hkv), block(NW * 64);
  const bool sc = a.p.cap > 0.f, al = a.p.alibi != nullptr;
  if (sc && al) hipLaunchKernelGGL((fwd_split_kernel<T, D, NW, ST, true, true>), grid, block, 0, st, a);
  else if (sc) hipLaunchKernelGGL((fwd_split_kernel<T, D, NW, ST, true, false>), grid, block, 0, st, a);
  else if (al) hipLaunchKernelGGL((fwd_split_kernel<T, D, NW, ST, false, true>), grid, block, 0, st, a);
  else hipLaunchKernelGGL((fwd_split_kernel<T, D, NW, ST, false, false>), grid, block, 0, st, a);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || a.nsplit == 1) return e;
  const int64_t rows = (int64_t)a.p.B * a.p.Hq * a.p.Sq;
  hipLaunchKernelGGL((fwd_split_merge_kernel<T, D>), dim3((unsigned)rows), dim3(256), 0, st, a);
  return hipGetLastError();
}

template <class T, int D>
hipError_t launch_split(const DecodeArgs& a, hipStream_t st) {
  DecodeArgs x = a;
  x.nrt = (int)(((int64_t)a.p.G * a.p.Sq + 31) / 32);
  x.plain = x.nsplit > 1 || x.nrt == 1;
  if constexpr (D == 256) {
    return launch_split<T, D, 4, 1>(x, st);
  } else {
    // (one split of a long cache, a batch with a workgroup or more per slot: ST = 1
    // and 2 within 2% at 8192 and 16384 keys, ST = 1 ahead at 500, D = 128 42 against 48 us)
    if (x.nsplit > 1) return launch_split<T, D, 4, 2>(x, st);
    if (x.nw == 8) return launch_split<T, D, 8, 1>(x, st);
    return launch_split<T, D, 4, 1>(x, st);
  }
}

#define FLEXATT_CAT2(a, b) a##b
#define FLEXATT_CAT(a, b) FLEXATT_CAT2(a, b)
hipError_t FLEXATT_CAT(fwd_split_bf16_d, FLEXATT_D)(const DecodeArgs& a, hipStream_t st) {
  return launch_split<__bf16, FLEXATT_D>(a, st);
}
hipError_t FLEXATT_CAT(fwd_split_f16_d, FLEXATT_D)(const DecodeArgs& a, hipStream_t st) {
  return launch_split<_Float16, FLEXATT_D>(a, st);
}

}  // namespace flexatt
