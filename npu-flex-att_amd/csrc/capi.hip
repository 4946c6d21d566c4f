// extern "C" entry points of libflexatt (declared in include/flexatt.h):
// argument checks, then dispatch to the kernel launchers by dtype and head dim.
#include <math.h>
#include <stdint.h>

#include <atomic>
#include <mutex>

#include "../../include/flexatt.h"
#include "flexatt_kernels.h"

namespace {
using namespace flexatt;

size_t elt_size(int dt) {
  switch (dt) {
    case FLEXATT_F32: return 4;
    case FLEXATT_F16:
    case FLEXATT_BF16: return 2;
    default: return 0;
  }
}

int head_index(int d) {
  switch (d) {
    case 32: return 0;
    case 64: return 1;
    case 128: return 2;
    case 256: return 3;
    default: return -1;
  }
}

int check_problem(const flexatt_problem* p) {
  if (!p) return FLEXATT_EINVAL;
  if (elt_size(p->dtype) == 0) return FLEXATT_EDTYPE;
  if (p->batch <= 0 || p->heads_q <= 0 || p->heads_kv <= 0 || p->seqlen_q <= 0 || p->seqlen_kv <= 0)
    return FLEXATT_EINVAL;
  if (p->heads_q % p->heads_kv != 0) return FLEXATT_ESHAPE;
  if (p->doc_bounds && !p->col_bounds && p->seqlen_q != p->seqlen_kv) return FLEXATT_ESHAPE;
  if (p->col_bounds && !p->doc_bounds) return FLEXATT_EINVAL;
  if (p->reserved != 0) return FLEXATT_EINVAL;
  if (p->block_map) {
    if (p->block_heads != 1 && p->block_heads != p->heads_q) return FLEXATT_EINVAL;
    if ((p->seqlen_kv + kBlk - 1) / kBlk > kBlkRowMax) return FLEXATT_ERANGE;
  }
  if (head_index(p->head_dim) < 0) return FLEXATT_EHEADDIM;
  if (p->causal != 0 && p->causal != 1) return FLEXATT_EINVAL;
  if (p->sliding_window < 0) return FLEXATT_EINVAL;
  if (!(p->soft_cap >= 0.f) || !isfinite(p->soft_cap) || !isfinite(p->scale)) return FLEXATT_EINVAL;
  // Grid sizes: tiles * B * H must fit a 1-D grid; row counts fit int32.
  const int64_t rows_q = (int64_t)p->batch * p->heads_q * p->seqlen_q;
  const int64_t rows_k = (int64_t)p->batch * p->heads_kv * p->seqlen_kv;
  if (rows_q > INT32_MAX || rows_k > INT32_MAX) return FLEXATT_ESHAPE;
  return FLEXATT_OK;
}

#define FLEXATT_TRY_OK(x)               \
  do {                                  \
    const int rc_ = (x);                \
    if (rc_ != FLEXATT_OK) return rc_;  \
  } while (0)

int check_tensor(const flexatt_tensor* t, int dt) {
  if (!t || !t->data) return FLEXATT_EINVAL;
  const int64_t es = (int64_t)elt_size(dt);
  if (t->stride_d != 1) return FLEXATT_ELAYOUT;
  if (t->stride_b < 0 || t->stride_h < 0 || t->stride_s < 0) return FLEXATT_ELAYOUT;
  if (((uintptr_t)t->data) % 16 != 0) return FLEXATT_ELAYOUT;
  if ((t->stride_b * es) % 16 || (t->stride_h * es) % 16 || (t->stride_s * es) % 16) return FLEXATT_ELAYOUT;
  return FLEXATT_OK;
}

// Output tensors: the input rules, and no two elements of the [b, h, s, d]
// index space may share an address (several workgroups would store to it,
// and the results would depend on their order).  Sufficient test: over the
// dimensions of extent > 1 sorted by stride, each stride exceeds the span of
// the smaller ones.
int check_out_tensor(const flexatt_tensor* t, int dt, int64_t n_b, int64_t n_h, int64_t n_s, int64_t n_d) {
  FLEXATT_TRY_OK(check_tensor(t, dt));
  int64_t st[4] = {t->stride_b, t->stride_h, t->stride_s, 1};
  int64_t ext[4] = {n_b, n_h, n_s, n_d};
  int order[4], n = 0;
  for (int i = 0; i < 4; ++i)
    if (ext[i] > 1) order[n++] = i;
  for (int i = 1; i < n; ++i)  // insertion sort by stride
    for (int j = i; j > 0 && st[order[j]] < st[order[j - 1]]; --j) {
      const int x = order[j];
      order[j] = order[j - 1];
      order[j - 1] = x;
    }
  int64_t span = 0;  // largest offset reachable with the dims sorted so far
  for (int i = 0; i < n; ++i) {
    const int d = order[i];
    if (st[d] <= span) return FLEXATT_ELAYOUT;
    span += (ext[d] - 1) * st[d];
  }
  return FLEXATT_OK;
}

// The window the kernels and the staged-dS layout see, at most Sq: the same mask
// (i - j < Sq), and neither row + window nor the layout's sums over it leave 32
// bits, whatever W the caller gives.
int window_of(const flexatt_problem* p) {
  return p->sliding_window < p->seqlen_q ? p->sliding_window : p->seqlen_q;
}

Shape make_shape(const flexatt_problem* p) {
  Shape s;
  s.B = p->batch;
  s.Hq = p->heads_q;
  s.Hkv = p->heads_kv;
  s.G = p->heads_q / p->heads_kv;
  s.Sq = p->seqlen_q;
  s.Skv = p->seqlen_kv;
  s.scale = p->scale;
  s.scale_log2 = p->scale * kLog2e;
  s.causal = p->causal;
  s.window = window_of(p);
  s.cap = p->soft_cap;
  s.inv_cap = p->soft_cap > 0.f ? 1.0f / p->soft_cap : 0.f;
  s.tanh_k = p->soft_cap > 0.f ? 2.0f * kLog2e * p->scale / p->soft_cap : 0.f;
  s.cap_log2 = p->soft_cap * kLog2e;
  s.alibi = p->alibi_slopes;
  s.doc = p->doc_bounds;
  s.docc = p->col_bounds ? p->col_bounds : p->doc_bounds;
  s.blk = p->block_map;
  s.blk_h = p->block_map ? p->block_heads : 1;
  s.blk_nq = (p->seqlen_q + kBlk - 1) / kBlk;
  s.blk_nk = (p->seqlen_kv + kBlk - 1) / kBlk;
  return s;
}

View view(const flexatt_tensor* t) { return View{t->data, t->stride_b, t->stride_h, t->stride_s}; }
MutView mview(const flexatt_tensor* t) { return MutView{t->data, t->stride_b, t->stride_h, t->stride_s}; }

// [dtype][head index]
const FwdLauncher kFwd[3][4] = {
    {fwd_f32_d32, fwd_f32_d64, fwd_f32_d128, fwd_f32_d256},
    {fwd_mfma_f16_d32, fwd_mfma_f16_d64, fwd_mfma_f16_d128, fwd_mfma_f16_d256},
    {fwd_mfma_bf16_d32, fwd_mfma_bf16_d64, fwd_mfma_bf16_d128, fwd_mfma_bf16_d256},
};
const BwdLauncher kDq[3][4] = {
    {bwd_dq_f32_d32, bwd_dq_f32_d64, bwd_dq_f32_d128, bwd_dq_f32_d256},
    {bwd_dq_mfma_f16_d32, bwd_q_f16_d64, bwd_q_f16_d128, bwd_dq_mfma_f16_d256},
    {bwd_dq_mfma_bf16_d32, bwd_q_bf16_d64, bwd_q_bf16_d128, bwd_dq_mfma_bf16_d256},
};
const BwdLauncher kDkdv[3][4] = {
    {bwd_dkdv_f32_d32, bwd_dkdv_f32_d64, bwd_dkdv_f32_d128, bwd_dkdv_f32_d256},
    {bwd_dkdv_mfma_f16_d32, bwd_kv_f16_d64, bwd_kv_f16_d128, bwd_kv_f16_d256},
    {bwd_dkdv_mfma_bf16_d32, bwd_kv_bf16_d64, bwd_kv_bf16_d128, bwd_kv_bf16_d256},
};

// Split-KV decode: range, plan and workspace.
constexpr int kDecWaves = 4;  // waves per workgroup
constexpr int kDecTile = 32;   // KV rows per tile
bool is_16bit(const flexatt_problem* p) { return p->dtype == FLEXATT_F16 || p->dtype == FLEXATT_BF16; }
// flexatt_fwd_split: the query rows of a KV head fit one 32-row tile.
bool split_applies(const flexatt_problem* p) {
  return is_16bit(p) && !p->doc_bounds && !p->block_map &&
         (int64_t)(p->heads_q / p->heads_kv) * p->seqlen_q <= 32;
}
// flexatt_fwd_decode (and _noalloc): the same at head_dim <= 128.
bool decode_applies(const flexatt_problem* p) { return split_applies(p) && p->head_dim <= 128; }
struct DecodePlan {
  int nsplit, chunk, ntiles;
  size_t bytes;  // workspace: partial O then partial LSE
};
DecodePlan decode_plan(const flexatt_problem* p) {
  DecodePlan d;
  // attended KV range: with top-left causal alignment no query row sees past Sq - 1
  const int kv_hi = p->causal ? (p->seqlen_kv < p->seqlen_q ? p->seqlen_kv : p->seqlen_q) : p->seqlen_kv;
  d.ntiles = (kv_hi + kDecTile - 1) / kDecTile;
  // about two workgroups per CU (256 CUs), but at least two tiles per wave
  const int64_t groups = (int64_t)p->batch * p->heads_kv;
  int64_t ns = (512 + groups - 1) / groups;
  const int64_t most = d.ntiles / (2 * kDecWaves);
  if (ns > most) ns = most;
  if (ns > 256) ns = 256;
  if (ns < 1) ns = 1;
  d.chunk = (int)((d.ntiles + ns - 1) / ns);
  d.nsplit = (d.ntiles + d.chunk - 1) / d.chunk;  // no workgroup without tiles
  const int64_t rows = (int64_t)p->batch * p->heads_q * p->seqlen_q;
  const int64_t parts = d.nsplit;  // one partial per workgroup
  d.bytes = (size_t)(rows * parts * (p->head_dim + 1) * (int64_t)sizeof(float));
  return d;
}
const DecodeLauncher kSplit[3][4] = {
    {fwd_split_f32_d32, fwd_split_f32_d64, fwd_split_f32_d128, nullptr},  // one workgroup per row tile only
    {fwd_split_f16_d32, fwd_split_f16_d64, fwd_split_f16_d128, fwd_split_f16_d256},
    {fwd_split_bf16_d32, fwd_split_bf16_d64, fwd_split_bf16_d128, fwd_split_bf16_d256},
};

// Launch the decode kernels with their partials in `ws` (d.bytes, 16-byte
// aligned); the problem and tensors are already checked.
int decode_run(const flexatt_problem* p, const DecodePlan& d, const flexatt_tensor* q, const flexatt_tensor* k,
               const flexatt_tensor* v, const flexatt_tensor* o, float* lse, void* ws, hipStream_t stream,
               int nw = kDecWaves) {
  DecodeArgs a;
  a.q = view(q);
  a.k = view(k);
  a.v = view(v);
  a.o = mview(o);
  a.lse = lse;
  a.p = make_shape(p);
  a.nsplit = d.nsplit;
  a.chunk = d.chunk;
  a.nw = nw;
  a.nrt = a.plain = 0;
  const int64_t rows = (int64_t)p->batch * p->heads_q * p->seqlen_q;
  a.part_o = (float*)ws;
  a.part_lse = a.part_o + rows * d.nsplit * p->head_dim;
  return (int)kSplit[p->dtype][head_index(p->head_dim)](a, stream);
}

// Fixed partial-result buffer of flexatt_fwd_decode_noalloc: one copy per GPU,
// held until the process ends.  Host code never passes the name `scratch`
// itself to a kernel (on the host it is a stand-in, not a device address):
// the device address of each GPU's copy is looked up once, with that GPU
// current, and kept in scratch_ptr.
static __device__ __align__(256) unsigned char scratch[FLEXATT_NOALLOC_SCRATCH_BYTES];
constexpr int kMaxDevices = 64;
std::mutex scratch_mu;
void* scratch_ptr[kMaxDevices] = {};

// Device address of the scratch copy of the GPU that `stream` runs on, which
// must be the current device (the lookup needs it current).
int scratch_for_stream(hipStream_t stream, void** out) {
  int cur = -1;
  hipError_t e = hipGetDevice(&cur);
  if (e != hipSuccess) return (int)e;
  if (stream) {
    int sdev = -1;
    e = hipStreamGetDevice(stream, &sdev);
    if (e != hipSuccess) return (int)e;
    if (sdev != cur) return FLEXATT_EINVAL;
  }
  if (cur < 0 || cur >= kMaxDevices) return FLEXATT_EINVAL;
  std::lock_guard<std::mutex> lock(scratch_mu);
  if (!scratch_ptr[cur]) {
    void* ptr = nullptr;
    e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return (int)e;
    if (!ptr) return (int)hipErrorInvalidSymbol;
    scratch_ptr[cur] = ptr;
  }
  *out = scratch_ptr[cur];
  return FLEXATT_OK;
}

// Interval and block masks take the general dQ kernel (the recomputing
// D = 128 tile stream has neither); the D = 128 dK/dV tile stream has both.
bool has_masks(const flexatt_problem* p) { return p->doc_bounds || p->block_map; }
BwdLauncher pick_dq(const flexatt_problem* p) {
  // the query-stationary tile stream (bwd_q.hip) has no document, prefix or
  // block-map masks: with them the general kernel runs
  if (has_masks(p) && p->dtype != FLEXATT_F32) {
    const bool bf = p->dtype == FLEXATT_BF16;
    if (p->head_dim == 128) return bf ? bwd_dq_mfma_bf16_d128 : bwd_dq_mfma_f16_d128;
    if (p->head_dim == 64) return bf ? bwd_dq_mfma_bf16_d64 : bwd_dq_mfma_f16_d64;
  }
  return kDq[p->dtype][head_index(p->head_dim)];
}
// The dQ kernel that can also form Delta itself (the D = 64 and 128 tile stream).
bool dq_fuses_delta(const flexatt_problem* p) {
  const BwdLauncher f = pick_dq(p);
  return f == bwd_q_bf16_d128 || f == bwd_q_f16_d128 || f == bwd_q_bf16_d64 || f == bwd_q_f16_d64;
}
BwdLauncher pick_dkdv(const flexatt_problem* p) { return kDkdv[p->dtype][head_index(p->head_dim)]; }

#define FLEXATT_TRY(x)             \
  do {                             \
    const int rc_ = (x);           \
    if (rc_ != FLEXATT_OK) return rc_; \
  } while (0)

// CUs of the current device (cached per device), 0 if unknown.  Host threads
// may call the ABI concurrently: the cache is atomic (a racing first lookup
// stores the same value twice).
int cu_count() {
  static std::atomic<int> cache[kMaxDevices];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return 0;
  int n = cache[dev].load(std::memory_order_relaxed);
  if (n == 0) {
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return 0;
    cache[dev].store(n, std::memory_order_relaxed);
  }
  return n;
}

int cus() {  // 256 if unknown
  const int n = cu_count();
  return n > 0 ? n : 256;
}

// Attended (query row, key) pairs of one head under the causal and window
// masks (interval masks, whose bounds are on the device, not counted).
int64_t attended_pairs(const flexatt_problem* p) {
  const int64_t n = p->seqlen_q, m = p->seqlen_kv, w = p->sliding_window;
  auto tri = [](int64_t x) { return x > 0 ? x * (x + 1) / 2 : 0; };
  // sum over rows i of the row's end (i + 1 capped at m, or m) ...
  int64_t sum = !p->causal ? n * m : n <= m ? tri(n) : tri(m) + (n - m) * m;
  if (w > 0) {
    // ... less its start i - w, and less the whole row once the start reaches m
    const int64_t live = n < m + w ? n : m + w;  // rows that keep a key
    sum -= tri(live - 1 - w) + (n - live) * m;
  }
  return sum;
}

// Waves per workgroup of the forward that splits a 32-row tile's keys over
// the waves (fwd_split.hip, one workgroup per row tile), or 0 for the regular
// forward.  The regular workgroup covers 256 query rows and walks their keys as
// one chain, so its time is the longest chain until its grid fills the chip;
// the split workgroup covers 32 rows, shortens the chain by its wave count and
// costs about twice the regular kernel's time per pair.  Measured at the
// crossover, in tiles of 32 x 32 pairs per CU (U / CUs) against the longest
// chain L in 32-key tiles (bf16, regular -> split, us): D = 128: U = 2 CUs L
// B=1 Hq=32 Hkv=8 S=1024 causal 27.0 -> 23.4, non-causal (4 CUs L) 26.9 -> 34.1;
// D = 64: 4 CUs L, the same heads at S=2048 causal 39.8 -> 34.6, non-causal
// (8 CUs L) 42.8 -> 61.5; D = 256: one workgroup per CU, Hq=16 S=512 19.4 ->
// 15.6, S=1024 30.7 -> 31.3.  Far from it: B=1 H=2 D=64 S=2048 39.4 -> 10.7, S=128
// 6.7 -> 4.4.
// Eight waves instead of four where the chip has a CU per workgroup and the
// chain is long enough to pay for the larger combine: H=2 D=64 S=2048 14.0 ->
// 10.7, Hq=8 Hkv=2 D=128 S=2048 causal 27.2 -> 23.1 but non-causal 31.0 -> 34.4,
// S=512 8.1 -> 8.9.
// fp32 (f32_split.hip, four waves): an estimate in us of the split workgroups'
// chain, or of the chip's time per 1024 tile pairs when they fill it, against
// the regular kernel's chain (which eight waves of 256 rows walk together).
// Measured, regular -> split: D = 128 Hq=8 S=1024 273 -> 52, B=2 S=2048 551 -> 217,
// S=4096 non-causal 1126 -> 753; D = 64 H=2 S=2048 318 -> 55; D = 32 H=8 S=2048 204
// -> 43.  The estimate of a full chip (5.9 us per 1024 pairs at D = 128, the
// regular kernel 4.5) keeps large problems on the regular kernel.
// Many row tiles of few keys: each 32-row workgroup costs its launch, its Q rows and its combine
// besides its tile pairs (`wg` per 1024 of them, `pair` per 1024 pairs), against a regular
// workgroup whose chain spans all its rows' keys (with a window, the window and those rows).
// Estimates in us of both (FwdCost: split with four waves, regular), fitted to 1700 shapes, 33 ..
// 5000 positions, B = 1 .. 8, windowed, causal and not, where the line above alone left 5% of the
// calls more than 5% slower than the regular kernel: bf16 D = 128 B=8 Hq=32 Hkv=8 S=143 causal 11.9
// (regular) against 18.0, window 32 Hq=32 Hkv=8 Sq=2286 Skv=72 16.0 against 23.4; D = 64 B=4 Hq=128
// Hkv=16 S=144 causal 11.4 against 15.3; fp32 D = 128 B=4 Hq=56 Hkv=8 S=183 73 against 108.  Of 1184
// other shapes 2 are now, of 28.
// D = 256 loses its 1 us at one or two tiles of keys (S=42 8.7 against 10.1).
struct FwdCost {
  double base, tile, pair, wg, reg_base, reg_tile, reg_pair, reg_wg;
};
int split_waves(const flexatt_problem* p) {
  if (p->block_map || !kSplit[p->dtype][head_index(p->head_dim)]) return 0;
  const int64_t ncu = cus();
  const int64_t G = p->heads_q / p->heads_kv, groups = (int64_t)p->batch * p->heads_kv;
  const int64_t wgs = groups * ((G * p->seqlen_q + 31) / 32);
  int64_t keys = p->causal && p->seqlen_q < p->seqlen_kv ? p->seqlen_q : p->seqlen_kv;  // the longest row's
  if (p->sliding_window > 0) {
    const int64_t w = (int64_t)p->sliding_window + (p->causal ? 32 : p->seqlen_kv);
    if (w < keys) keys = w;
  }
  const int64_t chain = (keys + 31) / 32;
  const int64_t units = groups * G * attended_pairs(p) / (32 * 32);
  if (p->dtype == FLEXATT_F32) {
    constexpr double tile[3] = {1.9, 3.2, 5.85}, unit[3] = {1.7, 2.9, 5.9}, other[3] = {3.2, 5.0, 8.4};
    constexpr double wg[3] = {5, 15, 32};
    const int d = head_index(p->head_dim);
    const double c = tile[d] * chain / 4, w = (unit[d] * units + wg[d] * wgs) / 1024;
    const double rows = p->seqlen_q <= 128 ? 0.6 : 1.0;  // the regular workgroup then runs one wave a SIMD
    return 5 + (c > w ? c : w) < 6 + rows * other[d] * chain ? 4 : 0;
  }
  if (p->head_dim == 256) return wgs <= ncu && chain > 2 ? 4 : 0;
  // (an eighth above the measured points, whose causal pairs are just over half)
  const int64_t load = 8 * units / (ncu * chain);  // in eighths
  if (load > (p->head_dim == 128 ? 18 : 36)) return 0;
  if (wgs <= ncu && (p->head_dim == 128 ? chain >= 64 && load <= 9 : chain >= 32)) return 8;
  constexpr FwdCost cost[3] = {{4.3, 0.54, 0.30, 2.5, 6.6, 0.43, 0.32, 2.1},   // D = 32
                               {4.8, 0.72, 0.48, 3.7, 6.0, 0.60, 0.38, 2.5},   // 64
                               {5.6, 1.02, 0.85, 9.2, 7.8, 0.70, 0.54, 4.7}};  // 128
  const FwdCost& c = cost[head_index(p->head_dim)];
  // the regular workgroup's chain: 256 rows, shared by up to 8 heads of a group
  const int64_t low = G & -G, rows = 256 / (low < 8 ? low : 8);
  int64_t reg_keys = p->causal && p->seqlen_q < p->seqlen_kv ? p->seqlen_q : p->seqlen_kv;
  if (p->sliding_window > 0) {
    const int64_t w = p->sliding_window + (p->causal ? (rows < p->seqlen_q ? rows : p->seqlen_q) : (int64_t)p->seqlen_kv);
    if (w < reg_keys) reg_keys = w;
  }
  const double wait = c.tile * chain / 4, busy = (c.pair * units + c.wg * wgs) / 1024;
  const double reg_wait = c.reg_tile * ((reg_keys + 31) / 32), reg_busy = (c.reg_pair * units + c.reg_wg * wgs) / 1024;
  return c.base + (wait > busy ? wait : busy) < c.reg_base + (reg_wait > reg_busy ? reg_wait : reg_busy) ? 4 : 0;
}

int bwd_common(const flexatt_problem* p, const flexatt_tensor* q, const flexatt_tensor* k,
               const flexatt_tensor* v, const flexatt_tensor* dout, const float* lse, const float* delta,
               BwdArgs& a) {
  FLEXATT_TRY(check_problem(p));
  FLEXATT_TRY(check_tensor(q, p->dtype));
  FLEXATT_TRY(check_tensor(k, p->dtype));
  FLEXATT_TRY(check_tensor(v, p->dtype));
  FLEXATT_TRY(check_tensor(dout, p->dtype));
  if (!lse || !delta) return FLEXATT_EINVAL;
  a.q = view(q);
  a.k = view(k);
  a.v = view(v);
  a.dout = view(dout);
  a.lse = lse;
  a.delta = delta;
  a.p = make_shape(p);
  a.ntiles = 0;
  a.o = View{nullptr, 0, 0, 0};
  a.delta_out = nullptr;
  a.ds = nullptr;
  a.ds_head = 0;
  a.queue = nullptr;
  a.part = nullptr;
  a.nparts = 1;
  a.nstatic = cu_count() & ~7;  // the first round of workgroups (also sets the dK/dV walk direction)
  return FLEXATT_OK;
}

// Staged dS (fp16/bf16 at D = 64, 128 and 256; fp32 at every D;
// every mask primitive: the dK/dV kernel masks per element and stores every
// unit of the causal / window band, zero where masked): units per query head
// and workspace bytes; 0 when the problem takes the recomputing dQ kernel.
bool ds_applies(const flexatt_problem* p) {
  if (p->dtype == FLEXATT_F32) return true;
  return (p->dtype == FLEXATT_F16 || p->dtype == FLEXATT_BF16) &&
         (p->head_dim == 64 || p->head_dim == 128 || p->head_dim == 256);
}
int64_t ds_unit_bytes(const flexatt_problem* p) { return p->dtype == FLEXATT_F32 ? kDsUnitB32 : kDsUnitB; }
BwdLauncher pick_kv_ds(const flexatt_problem* p) {
  if (p->dtype == FLEXATT_F32)
    return p->head_dim == 32 ? bwd_kv_ds_f32_d32
           : p->head_dim == 64 ? bwd_kv_ds_f32_d64
           : p->head_dim == 128 ? bwd_kv_ds_f32_d128 : bwd_kv_ds_f32_d256;
  const bool bf = p->dtype == FLEXATT_BF16;
  if (p->head_dim == 64) return bf ? bwd_kv_ds_bf16_d64 : bwd_kv_ds_f16_d64;
  if (p->head_dim == 256) return bf ? bwd_kv_ds_bf16_d256 : bwd_kv_ds_f16_d256;
  return bf ? bwd_kv_ds_bf16_d128 : bwd_kv_ds_f16_d128;
}
BwdLauncher pick_dq_ds(const flexatt_problem* p) {
  if (p->dtype == FLEXATT_F32)
    return p->head_dim == 32 ? bwd_dq_ds_f32_d32
           : p->head_dim == 64 ? bwd_dq_ds_f32_d64
           : p->head_dim == 128 ? bwd_dq_ds_f32_d128 : bwd_dq_ds_f32_d256;
  const bool bf = p->dtype == FLEXATT_BF16;
  if (p->head_dim == 64) return bf ? bwd_dq_ds_bf16_d64 : bwd_dq_ds_f16_d64;
  if (p->head_dim == 256) return bf ? bwd_dq_ds_bf16_d256 : bwd_dq_ds_f16_d256;
  return bf ? bwd_dq_ds_bf16_d128 : bwd_dq_ds_f16_d128;
}
int64_t ds_units_per_head(const flexatt_problem* p) {
  const int nqt = (p->seqlen_q + kDsQT - 1) / kDsQT;
  const int nkb = (p->seqlen_kv + kDsKB - 1) / kDsKB;
  return ds_tile_offset(nqt, p->causal, window_of(p), nkb);
}
size_t ds_bytes(const flexatt_problem* p) {
  if (!ds_applies(p)) return 0;
  return (size_t)((int64_t)p->batch * p->heads_q * ds_units_per_head(p) * ds_unit_bytes(p));
}
int ds_workspace(const flexatt_problem* p, void* ws, size_t bytes, BwdArgs& a) {
  if (!ds_applies(p)) return FLEXATT_ERANGE;
  if (!ws) return FLEXATT_EINVAL;
  if (bytes < ds_bytes(p)) return FLEXATT_EINVAL;
  if (((uintptr_t)ws) % 16 != 0) return FLEXATT_ELAYOUT;
  a.ds = (char*)ws;
  a.ds_head = ds_units_per_head(p);
  return FLEXATT_OK;
}

// Bounded workspaces: the staged backward of a problem whose whole dS band
// exceeds the caller's workspace runs in passes over chunks of (batch, KV
// head) groups, each pass a problem of its own over the same buffers.  A
// group (one KV head and its G query heads) is the smallest chunk: its dK /
// dV sum and its dQ rows need only its own dS units.
int64_t ds_group_bytes(const flexatt_problem* p) {
  return (int64_t)(p->heads_q / p->heads_kv) * ds_units_per_head(p) * ds_unit_bytes(p);
}
// Groups per pass for a workspace of `bytes` (>= one group's band): whole
// batches when at least one batch fits, else KV heads of one batch.
int64_t chunk_groups(const flexatt_problem* p, size_t bytes) {
  int64_t k = (int64_t)(bytes / (size_t)ds_group_bytes(p));
  if (k >= p->heads_kv) k = k / p->heads_kv * p->heads_kv;
  return k;
}
// One pass: batches [b0, b0 + nb) with every KV head, or (nb = 1) the KV
// heads [h0, h0 + nh) of batch b0.
struct Chunk {
  int b0, nb, h0, nh;
};
flexatt_problem sub_problem(const flexatt_problem* p, const Chunk& c) {
  flexatt_problem s = *p;
  const int G = p->heads_q / p->heads_kv;
  s.batch = c.nb;
  s.heads_kv = c.nh;
  s.heads_q = c.nh * G;
  if (p->alibi_slopes) s.alibi_slopes = p->alibi_slopes + (int64_t)c.h0 * G;
  if (p->doc_bounds) s.doc_bounds = p->doc_bounds + (int64_t)c.b0 * p->seqlen_q * 2;
  if (p->col_bounds) s.col_bounds = p->col_bounds + (int64_t)c.b0 * p->seqlen_kv * 2;
  if (p->block_map) {
    const int64_t nq = (p->seqlen_q + kBlk - 1) / kBlk, nk = (p->seqlen_kv + kBlk - 1) / kBlk;
    const bool per_head = p->block_heads == p->heads_q && p->heads_q > 1;
    s.block_map = p->block_map + ((int64_t)c.b0 * p->block_heads + (per_head ? (int64_t)c.h0 * G : 0)) * nq * nk;
    s.block_heads = per_head ? s.heads_q : 1;
  }
  return s;
}
// The chunk's view of a [B, H, S, D] tensor whose head h0 is at `h0`.
flexatt_tensor sub_tensor(const flexatt_tensor* t, int dt, int64_t b0, int64_t h0) {
  flexatt_tensor s = *t;
  s.data = (char*)t->data + (b0 * t->stride_b + h0 * t->stride_h) * (int64_t)elt_size(dt);
  return s;
}

}  // namespace

extern "C" {

int flexatt_abi_version(void) { return FLEXATT_ABI_VERSION; }

const char* flexatt_status_string(int status) {
  switch (status) {
    case FLEXATT_OK: return "ok";
    case FLEXATT_EINVAL: return "invalid argument (null pointer, non-positive size or bad flag)";
    case FLEXATT_EDTYPE: return "unsupported dtype (expected fp32, fp16 or bf16)";
    case FLEXATT_EHEADDIM: return "unsupported head_dim (expected 32, 64, 128 or 256)";
    case FLEXATT_ESHAPE: return "inconsistent shape (heads_q % heads_kv != 0 or sizes overflow)";
    case FLEXATT_ELAYOUT: return "unsupported layout (innermost stride != 1 or rows not 16-byte aligned)";
    case FLEXATT_ERANGE: return "problem outside the entry point's range";
    case FLEXATT_ESCRATCH: return "problem needs more than the library's fixed scratch buffer (FLEXATT_NOALLOC_SCRATCH_BYTES)";
    default: return status > 0 ? hipGetErrorString((hipError_t)status) : "unknown flexatt status";
  }
}

namespace {
// `by_size`: the split kernels where split_waves says so, else the regular forward.
int run_fwd(const flexatt_problem* p, const flexatt_tensor* q, const flexatt_tensor* k, const flexatt_tensor* v,
            const flexatt_tensor* o, float* lse, void* stream, bool by_size) {
  FLEXATT_TRY(check_problem(p));
  FLEXATT_TRY(check_tensor(q, p->dtype));
  FLEXATT_TRY(check_tensor(k, p->dtype));
  FLEXATT_TRY(check_tensor(v, p->dtype));
  FLEXATT_TRY(check_out_tensor(o, p->dtype, p->batch, p->heads_q, p->seqlen_q, p->head_dim));
  if (!lse) return FLEXATT_EINVAL;
  const int nw = by_size ? split_waves(p) : 0;
  if (nw) {
    const DecodePlan d{1, 0, 0, 0};
    return decode_run(p, d, q, k, v, o, lse, nullptr, (hipStream_t)stream, nw);
  }
  FwdArgs a;
  a.q = view(q);
  a.k = view(k);
  a.v = view(v);
  a.o = mview(o);
  a.lse = lse;
  a.p = make_shape(p);
  a.nqt = 0;
  return (int)kFwd[p->dtype][head_index(p->head_dim)](a, (hipStream_t)stream);
}
}  // namespace

int flexatt_fwd(const flexatt_problem* p, const flexatt_tensor* q, const flexatt_tensor* k,
                const flexatt_tensor* v, const flexatt_tensor* o, float* lse, void* stream) {
  return run_fwd(p, q, k, v, o, lse, stream, true);
}

int flexatt_fwd_regular(const flexatt_problem* p, const flexatt_tensor* q, const flexatt_tensor* k,
                        const flexatt_tensor* v, const flexatt_tensor* o, float* lse, void* stream) {
  return run_fwd(p, q, k, v, o, lse, stream, false);
}

size_t flexatt_fwd_decode_workspace(const flexatt_problem* p) {
  if (check_problem(p) != FLEXATT_OK || !decode_applies(p)) return 0;
  return decode_plan(p).bytes;
}

int flexatt_fwd_decode(const flexatt_problem* p, const flexatt_tensor* q, const flexatt_tensor* k,
                       const flexatt_tensor* v, const flexatt_tensor* o, float* lse, void* workspace,
                       size_t workspace_bytes, void* stream) {
  FLEXATT_TRY(check_problem(p));
  FLEXATT_TRY(check_tensor(q, p->dtype));
  FLEXATT_TRY(check_tensor(k, p->dtype));
  FLEXATT_TRY(check_tensor(v, p->dtype));
  FLEXATT_TRY(check_out_tensor(o, p->dtype, p->batch, p->heads_q, p->seqlen_q, p->head_dim));
  if (!lse || !workspace) return FLEXATT_EINVAL;
  if (!decode_applies(p)) return FLEXATT_ERANGE;
  const DecodePlan d = decode_plan(p);
  if (workspace_bytes < d.bytes) return FLEXATT_EINVAL;
  if (((uintptr_t)workspace) % 16 != 0) return FLEXATT_ELAYOUT;
  if (d.ntiles == 0) return FLEXATT_EINVAL;
  return decode_run(p, d, q, k, v, o, lse, workspace, (hipStream_t)stream);
}

size_t flexatt_fwd_split_workspace(const flexatt_problem* p) {
  if (check_problem(p) != FLEXATT_OK || !split_applies(p)) return 0;
  return decode_plan(p).bytes;
}

int flexatt_fwd_split(const flexatt_problem* p, const flexatt_tensor* q, const flexatt_tensor* k,
                      const flexatt_tensor* v, const flexatt_tensor* o, float* lse, void* workspace,
                      size_t workspace_bytes, void* stream) {
  FLEXATT_TRY(check_problem(p));
  FLEXATT_TRY(check_tensor(q, p->dtype));
  FLEXATT_TRY(check_tensor(k, p->dtype));
  FLEXATT_TRY(check_tensor(v, p->dtype));
  FLEXATT_TRY(check_out_tensor(o, p->dtype, p->batch, p->heads_q, p->seqlen_q, p->head_dim));
  if (!lse || !workspace) return FLEXATT_EINVAL;
  if (!split_applies(p)) return FLEXATT_ERANGE;
  const DecodePlan d = decode_plan(p);
  if (workspace_bytes < d.bytes) return FLEXATT_EINVAL;
  if (((uintptr_t)workspace) % 16 != 0) return FLEXATT_ELAYOUT;
  if (d.ntiles == 0) return FLEXATT_EINVAL;
  return decode_run(p, d, q, k, v, o, lse, workspace, (hipStream_t)stream);
}

int flexatt_fwd_decode_noalloc(const flexatt_problem* p, const flexatt_tensor* q, const flexatt_tensor* k,
                               const flexatt_tensor* v, const flexatt_tensor* o, float* lse, void* stream) {
  FLEXATT_TRY(check_problem(p));
  FLEXATT_TRY(check_tensor(q, p->dtype));
  FLEXATT_TRY(check_tensor(k, p->dtype));
  FLEXATT_TRY(check_tensor(v, p->dtype));
  FLEXATT_TRY(check_out_tensor(o, p->dtype, p->batch, p->heads_q, p->seqlen_q, p->head_dim));
  if (!lse) return FLEXATT_EINVAL;
  if (!decode_applies(p)) return FLEXATT_ERANGE;
  const DecodePlan d = decode_plan(p);
  if (d.ntiles == 0) return FLEXATT_EINVAL;
  // sizes are checked before anything touches the GPU
  if (d.bytes > (size_t)FLEXATT_NOALLOC_SCRATCH_BYTES) return FLEXATT_ESCRATCH;
  void* ws = nullptr;
  FLEXATT_TRY(scratch_for_stream((hipStream_t)stream, &ws));
  return decode_run(p, d, q, k, v, o, lse, ws, (hipStream_t)stream);
}

int flexatt_document_bounds(const void* ids, int ids_bytes, int batch, int seqlen, int32_t* bounds, void* stream) {
  if (!ids || !bounds || batch <= 0 || seqlen <= 0) return FLEXATT_EINVAL;
  if (ids_bytes != 1 && ids_bytes != 2 && ids_bytes != 4 && ids_bytes != 8) return FLEXATT_EINVAL;
  if ((uintptr_t)ids % ids_bytes != 0 || (uintptr_t)bounds % sizeof(int32_t) != 0) return FLEXATT_ELAYOUT;
  if ((int64_t)batch * seqlen > INT32_MAX) return FLEXATT_ESHAPE;
  return (int)doc_bounds_run(ids, ids_bytes, batch, seqlen, bounds, (hipStream_t)stream);
}

namespace {
int run_delta(const flexatt_problem* p, const flexatt_tensor* o, const flexatt_tensor* dout, float* delta,
              int* zero, void* stream) {
  FLEXATT_TRY(check_problem(p));
  FLEXATT_TRY(check_tensor(o, p->dtype));
  FLEXATT_TRY(check_tensor(dout, p->dtype));
  if (!delta) return FLEXATT_EINVAL;
  DeltaArgs a;
  a.o = view(o);
  a.dout = view(dout);
  a.delta = delta;
  a.B = p->batch;
  a.H = p->heads_q;
  a.S = p->seqlen_q;
  a.D = p->head_dim;
  a.zero = zero;
  return (int)bwd_delta(p->dtype, a, (hipStream_t)stream);
}
}  // namespace

int flexatt_bwd_delta(const flexatt_problem* p, const flexatt_tensor* o, const flexatt_tensor* dout,
                      float* delta, void* stream) {
  return run_delta(p, o, dout, delta, nullptr, stream);
}

int flexatt_bwd_dq(const flexatt_problem* p, const flexatt_tensor* q, const flexatt_tensor* k,
                   const flexatt_tensor* v, const flexatt_tensor* dout, const float* lse,
                   const float* delta, const flexatt_tensor* dq, void* stream) {
  BwdArgs a;
  FLEXATT_TRY(bwd_common(p, q, k, v, dout, lse, delta, a));
  FLEXATT_TRY(check_out_tensor(dq, p->dtype, p->batch, p->heads_q, p->seqlen_q, p->head_dim));
  a.dq = mview(dq);
  return (int)pick_dq(p)(a, (hipStream_t)stream);
}

int flexatt_bwd_dq_delta(const flexatt_problem* p, const flexatt_tensor* q, const flexatt_tensor* k,
                         const flexatt_tensor* v, const flexatt_tensor* o, const flexatt_tensor* dout,
                         const float* lse, float* delta, const flexatt_tensor* dq, void* stream) {
  BwdArgs a;
  FLEXATT_TRY(bwd_common(p, q, k, v, dout, lse, delta, a));
  FLEXATT_TRY(check_tensor(o, p->dtype));
  FLEXATT_TRY(check_out_tensor(dq, p->dtype, p->batch, p->heads_q, p->seqlen_q, p->head_dim));
  if (!dq_fuses_delta(p)) {  // Delta pass, then dQ
    FLEXATT_TRY(flexatt_bwd_delta(p, o, dout, delta, stream));
    a.dq = mview(dq);
    return (int)pick_dq(p)(a, (hipStream_t)stream);
  }
  a.o = view(o);
  a.delta_out = delta;
  a.dq = mview(dq);
  return (int)pick_dq(p)(a, (hipStream_t)stream);
}

int flexatt_bwd_dkdv(const flexatt_problem* p, const flexatt_tensor* q, const flexatt_tensor* k,
                     const flexatt_tensor* v, const flexatt_tensor* dout, const float* lse,
                     const float* delta, const flexatt_tensor* dk, const flexatt_tensor* dv,
                     void* stream) {
  BwdArgs a;
  FLEXATT_TRY(bwd_common(p, q, k, v, dout, lse, delta, a));
  FLEXATT_TRY(check_out_tensor(dk, p->dtype, p->batch, p->heads_kv, p->seqlen_kv, p->head_dim));
  FLEXATT_TRY(check_out_tensor(dv, p->dtype, p->batch, p->heads_kv, p->seqlen_kv, p->head_dim));
  a.dk = mview(dk);
  a.dv = mview(dv);
  return (int)pick_dkdv(p)(a, (hipStream_t)stream);
}

int flexatt_bwd(const flexatt_problem* p, const flexatt_tensor* q, const flexatt_tensor* k,
                const flexatt_tensor* v, const flexatt_tensor* o, const flexatt_tensor* dout,
                const float* lse, float* delta, const flexatt_tensor* dq, const flexatt_tensor* dk,
                const flexatt_tensor* dv, void* stream) {
  BwdArgs a;
  FLEXATT_TRY(bwd_common(p, q, k, v, dout, lse, delta, a));
  FLEXATT_TRY(check_tensor(o, p->dtype));
  FLEXATT_TRY(check_out_tensor(dq, p->dtype, p->batch, p->heads_q, p->seqlen_q, p->head_dim));
  FLEXATT_TRY(check_out_tensor(dk, p->dtype, p->batch, p->heads_kv, p->seqlen_kv, p->head_dim));
  FLEXATT_TRY(check_out_tensor(dv, p->dtype, p->batch, p->heads_kv, p->seqlen_kv, p->head_dim));
  FLEXATT_TRY(flexatt_bwd_dq_delta(p, q, k, v, o, dout, lse, delta, dq, stream));
  a.dk = mview(dk);
  a.dv = mview(dv);
  return (int)pick_dkdv(p)(a, (hipStream_t)stream);
}

namespace {
size_t part_bytes(const flexatt_problem* p, int nparts) {
  return 2 * sizeof(float) * (size_t)nparts * p->batch * p->heads_kv * p->seqlen_kv * p->head_dim;
}
// Interval and block masks are device data: the longest walk and the work that
// the host counts for a problem, times this and its square, are what packed documents of
// 40 .. 8000 positions measured closest to (either way from 0.6 to 0.8).
double mask_share(const flexatt_problem* p) { return has_masks(p) ? 0.7 : 1.0; }

// 32-row query tiles that the longest KV block of the staged dK/dV walks for one head.
int64_t longest_walk(const flexatt_problem* p) {
  const int64_t nqt = (p->seqlen_q + kDsQT - 1) / kDsQT;
  if (p->sliding_window == 0) return nqt;
  const int64_t keys = p->causal ? kDsKB : (p->seqlen_kv + kDsKB - 1) / kDsKB * (int64_t)kDsKB;
  const int64_t w = (keys + window_of(p) + kDsQT - 1) / kDsQT;
  return w < nqt ? w : nqt;
}

// Workgroups that share the query tiles of one KV block in the staged dK/dV
// launch (fp16/bf16).  The launch lasts as long as its longest block, or as the
// work per CU where that is longer; parts divide the first (blocks of equal length
// run in whole rounds) and cost their fp32 sums, written and read at about 5.5 TB/s,
// and one more launch.  Estimates in us, fitted to 940 shapes (450 without documents: H = 1 ..
// 128, G = 1 .. 8, 64 .. 8000 positions, causal, windowed and not; 490 with them): `tile` per
// 32-row query tile of the longest block, `work` per tile and CU, `start` per 1024
// workgroups, `sums` for the launch.  Under interval and block masks, whose walks may be
// far shorter, parts have to gain a fifth of the walk besides: bf16 Hq=32 Hkv=8 S=7034 D=128,
// parts 1 / 2, documents of 125 on average 186 / 231, 700 331 / 332, 2000 618 / 595.  Of 905 shapes it
// was not fitted to, 19 are more than 5% slower than one part; a rule that counted blocks
// against CUs had 144.  Backward, parts 1 / 2 / 3 / 4, D = 128 causal: Hq=32 Hkv=8 S=4096
// 604 / 501 / 515 / 523, S=3000 429 / 333 / 318 / 331, S=2048 295 / 218 / 194 / 194; documents of
// 2000 S=3000 310 / - / 226; Hq=Hkv=16 S=2048 of 200 53 / 76 (G = 1: short walks, the same sums);
// D = 64 with half the blocks masked S=4096 416 / 311 / 285 / 272; D = 256 Hq=16 S=1000 141 / 102 / 97
// / 101, non-causal Hq=14 Hkv=2 S=3561 (112 items on 256 CUs) - / 661 / 809.
int staged_parts(const flexatt_problem* p) {
  if (!is_16bit(p) || p->head_dim == 32) return 1;
  const int d = head_index(p->head_dim);
  constexpr double tile[4] = {0, 0.91, 0.78, 0.94}, work[4] = {0, 0.92, 1.08, 1.0};
  constexpr double start[4] = {0, 0, 5.5, 5.0}, sums[4] = {0, 2.5, 0.7, 2.5};
  const double slots = p->head_dim == 64 ? 2 * cus() : cus();
  const int passes = p->head_dim == 256 ? 2 : 1;
  const int64_t nkb = (p->seqlen_kv + kDsKB - 1) / kDsKB, blocks = (int64_t)p->batch * p->heads_kv * nkb * passes;
  const int64_t units = ds_units_per_head(p), walk = longest_walk(p);
  const double share = mask_share(p), cap = p->soft_cap > 0.f ? 1.2 : 1.0;
  const double longest = tile[d] * cap * share * walk * (p->heads_q / p->heads_kv);
  const double even = work[d] * cap * share * share * passes * p->batch * p->heads_q * units / slots;
  const bool equal = !has_masks(p) && units > 0.8 * nkb * walk;
  const double margin = (has_masks(p) ? 0.2 : 0.01) * longest;
  const int64_t most = (p->seqlen_q + 4 * kDsQT - 1) / (4 * kDsQT);  // at least about four query tiles each
  double best = 1e30;
  int parts = 1;
  for (int n = 1; n <= 4 && n <= most; ++n) {
    const double one = longest / n * (equal ? ceil(n * blocks / slots) : 1.0);
    const double busy = even + start[d] * n * blocks / 1024;
    const double est = (one > busy ? one : busy) + (n > 1 ? sums[d] + margin + 0.36e-6 * part_bytes(p, n) : 0.0);
    if (est < best) {
      best = est;
      parts = n;
    }
  }
  return parts;
}

const BwdSplitLauncher kBwdSplit[3][4] = {
    {bwd_split_f32_d32, bwd_split_f32_d64, bwd_split_f32_d128, nullptr},
    {bwd_split_f16_d32, bwd_split_f16_d64, bwd_split_f16_d128, nullptr},
    {bwd_split_bf16_d32, bwd_split_bf16_d64, bwd_split_bf16_d128, nullptr},
};
bool bwd_split_applies(const flexatt_problem* p) {
  return kBwdSplit[p->dtype][head_index(p->head_dim)] && !p->block_map;
}
// The split backward's plan, and whether it beats the staged / recomputing
// backward, from estimates in us fitted to graph replays of 3100 shapes without documents
// (H = 1 .. 128, G = 1 .. 8, 64 .. 8000 positions, B = 1 .. 8, causal, windowed and not), rms 7 to
// 13% a side, 20% at D = 32.
// A split workgroup's time is its longest chain of 32 x 32 tiles until the chip is full; then the
// chip's time is `unit` per 1024 tile pairs and `wg` per 1024 workgroups.  The other backward's
// (BwdOtherCost) is its longest dK/dV walk, divided by staged_parts, or the work per CU, and its
// longest dQ chain or the work; interval masks count for mask_share on both sides.  Of 890 other
// shapes, a third of them with documents, 3 are more than 5% slower than the other backward
// without parts, the worst 1.15 times; constants fitted to 56 shapes, without the work on the
// other side, had 22.
// Measured, other -> split (waves x splits): D = 64 H=2 S=2048 causal 75 -> 20
// (8 x 1), Hq=8 Hkv=2 S=2048 193 -> 41 (8 x 2); D = 128 Hq=8 Hkv=2 S=1000 155
// -> 34 (4 x 4), S=2048 286 -> 74 (4 x 2); past the crossover: Hq=32 Hkv=8 B=2 S=2048 D=128
// 326 -> 472; D = 128 B=4 H=4 S=1099 73 -> 92, B=8 Hq=8 Hkv=8 S=347 causal 39 -> 51; D = 64 B=4
// Hq=64 Hkv=8 S=1522 documents of 1000 on average 425 -> 533.
// fp32 (four waves; 740 of the shapes): Hq=8 Hkv=2 S=1000 D=128 1264 -> 108 (4 x 4), H=2 S=2048
// D=64 480 -> 93 (4 x 1); past the crossover: D = 128 B=8 H=2 Sq=107 Skv=7443 causal 71 -> 112.
struct BwdSplitCost {
  double tile4, tile8, base4, base8, unit, wg4, wg8;
};
// Which waves and splits (fitted to 86 shapes' choices) ...
constexpr BwdSplitCost kBwdSplitPick[2][3] = {
    {{0.8, 1.0, 6.0, 7.0, 1.0, 5.0, 10.0},     // fp16/bf16, D = 32
     {1.2, 1.4, 7.0, 8.5, 1.4, 8.0, 14.0},     // 64
     {1.6, 0.0, 9.0, 0.0, 2.8, 20.0, 0.0}},    // 128 (four waves only)
    {{3.5, 0.0, 7.0, 0.0, 5.5, 8.0, 0.0},      // fp32, D = 32
     {5.7, 0.0, 8.0, 0.0, 9.0, 8.0, 0.0},      // 64
     {10.0, 0.0, 10.0, 0.0, 19.5, 10.0, 0.0}}, // 128
};
// ... and how long they take (fitted to the 3100 shapes' times; rows as above).
constexpr BwdSplitCost kBwdSplitTime[2][3] = {
    {{1.15, 1.34, 6.6, 6.5, 1.07, 4.7, 9.3},
     {1.45, 1.62, 7.5, 8.35, 1.52, 8.8, 15.3},
     {1.88, 0.0, 9.3, 0.0, 3.05, 21.7, 0.0}},
    {{4.4, 0.0, 7.0, 0.0, 4.8, 8.0, 0.0},
     {6.7, 0.0, 8.5, 0.0, 8.5, 19.0, 0.0},
     {10.7, 0.0, 13.0, 0.0, 18.8, 43.0, 0.0}},
};
// What both need of a problem.
struct BwdStreams {
  double G, groups, units, part;  // units: 1024 tile pairs; part: bytes of one split's sums
  int64_t lq, lk, nkt, nrt;       // longest streams: query tiles of a KV item, key tiles of a Q item; tiles of each
};
BwdStreams bwd_streams(const flexatt_problem* p) {
  BwdStreams s;
  s.G = p->heads_q / p->heads_kv;
  s.groups = (double)p->batch * p->heads_kv;
  s.lq = (p->seqlen_q + 31) / 32;
  s.nkt = s.lk = (p->seqlen_kv + 31) / 32;
  if (p->causal && s.lq < s.lk) s.lk = s.lq;
  if (p->sliding_window > 0 && p->causal) {
    const int64_t l = p->sliding_window / 32 + 2;
    if (l < s.lq) s.lq = l;
    if (l < s.lk) s.lk = l;
  }
  s.nrt = ((int64_t)(p->heads_q / p->heads_kv) * p->seqlen_q + 31) / 32;
  s.units = s.groups * s.G * (double)attended_pairs(p) / (32.0 * 32 * 1024);
  s.part = (double)part_bytes(p, 1);
  return s;
}
double bwd_split_us(const BwdSplitCost& c, const BwdStreams& s, bool cap, double share, int nw, int ns) {
  const double t = nw == 8 ? c.tile8 : c.tile4, base = nw == 8 ? c.base8 : c.base4;
  const double wgs = s.groups * (double)(s.nkt * ns + s.nrt) / 1024;
  const double chain = t * share * (s.G * s.lq / ns > s.lk ? s.G * s.lq / ns : s.lk) / nw;
  const double work = c.unit * (cap ? 1.25 : 1.0) * share * share * s.units + (nw == 8 ? c.wg8 : c.wg4) * wgs;
  // the sums written and read back at about 8 TB/s (they stay in cache), and one more launch
  return base + (chain > work ? chain : work) + (ns > 1 ? 4 + 0.25e-6 * ns * s.part : 0);
}
struct BwdSplitPlan {
  int nsplit, nw;
  size_t bytes;
};
BwdSplitPlan bwd_split_pick(const flexatt_problem* p, const BwdStreams& s) {
  const bool f32 = p->dtype == FLEXATT_F32, cap = p->soft_cap > 0.f;
  double best = 1e30;
  BwdSplitPlan r{1, 4, 0};
  for (int nw = 4; nw <= (p->head_dim < 128 && !f32 ? 8 : 4); nw += 4)
    for (int ns = 1; ns <= 8; ns *= 2) {
      const double est = bwd_split_us(kBwdSplitPick[f32][head_index(p->head_dim)], s, cap, 1.0, nw, ns);
      if (est < best) {
        best = est;
        r.nsplit = ns;
        r.nw = nw;
      }
    }
  if (r.nsplit > 1) r.bytes = part_bytes(p, r.nsplit);
  return r;
}
BwdSplitPlan bwd_split_plan(const flexatt_problem* p) { return bwd_split_pick(p, bwd_streams(p)); }

// The other backward: us around its kernels, per 32-row query tile of the longest dK/dV walk and
// per tile and CU of all, per 32-key tile of the longest dQ chain and per 1024 tile pairs, and
// per 1024 query tiles of 32 rows (Delta and the ends of the dQ workgroups).
struct BwdOtherCost {
  double base, kv, kv_work, q, q_work, rows;
};
BwdOtherCost bwd_other_cost(const flexatt_problem* p, bool staged) {
  const int d = head_index(p->head_dim);
  constexpr BwdOtherCost f32[3] = {{4.8, 3.2, 3.7, 2.0, 1.5, 3.4},      // D = 32
                                   {5.4, 4.85, 11.5, 2.55, 1.8, 5.9},   // 64
                                   {2.5, 8.1, 8.7, 5.0, 5.3, 9.3}};     // 128
  constexpr BwdOtherCost half[3] = {{18.5, 0.9, 0.72, 0.46, 0.12, 9.9},   // D = 32
                                    {14.0, 0.64, 1.23, 0.36, 0.5, 7.6},   // 64, recomputing
                                    {19.5, 0.85, 1.4, 0.48, 0.28, 7.8}};  // 128
  constexpr BwdOtherCost half64_staged = {13.9, 1.03, 0.96, 0.42, 0.99, 5.25};
  return p->dtype == FLEXATT_F32 ? f32[d] : d == 1 && staged ? half64_staged : half[d];
}
bool bwd_split_faster(const flexatt_problem* p) {
  const BwdStreams s = bwd_streams(p);
  const BwdSplitPlan plan = bwd_split_pick(p, s);
  const bool cap = p->soft_cap > 0.f;
  const double share = mask_share(p);
  const BwdSplitCost& c = kBwdSplitTime[p->dtype == FLEXATT_F32][head_index(p->head_dim)];
  const double split = bwd_split_us(c, s, cap, share, plan.nw, plan.nsplit);
  // the staged backward where it is preferred, its dK/dV streams shared by parts
  const bool staged = flexatt_bwd_prefers_staging(p);
  const int np = staged ? staged_parts(p) : 1;
  const BwdOtherCost o = bwd_other_cost(p, staged);
  const double walk = o.kv * share * s.G * longest_walk(p) / np;
  const double slots = p->head_dim == 64 ? 2 * cus() : cus();
  const double even = o.kv_work * share * share * p->batch * p->heads_q * ds_units_per_head(p) / slots;
  const double dq = o.q * share * s.lk, dq_even = o.q_work * share * share * s.units;
  const double rows = o.rows * p->batch * p->heads_q * ((p->seqlen_q + 31) / 32) / 1024;
  const double sums = np > 1 ? 3 + 0.38e-6 * part_bytes(p, np) : 0.0;
  const double other = o.base + (cap ? 1.2 : 1.0) * (walk > even ? walk : even) +
                       (dq > dq_even ? dq : dq_even) + rows + sums;
  return split < 0.97 * other;
}
}  // namespace

int flexatt_bwd_prefers_split(const flexatt_problem* p) {
  return check_problem(p) == FLEXATT_OK && bwd_split_applies(p) && bwd_split_faster(p);
}

size_t flexatt_bwd_split_workspace(const flexatt_problem* p) {
  return check_problem(p) == FLEXATT_OK && bwd_split_applies(p) ? bwd_split_plan(p).bytes : 0;
}

int flexatt_bwd_split(const flexatt_problem* p, const flexatt_tensor* q, const flexatt_tensor* k,
                      const flexatt_tensor* v, const flexatt_tensor* o, const flexatt_tensor* dout, const float* lse,
                      float* delta, const flexatt_tensor* dq, const flexatt_tensor* dk, const flexatt_tensor* dv,
                      void* workspace, size_t workspace_bytes, void* stream) {
  BwdArgs c;
  FLEXATT_TRY(bwd_common(p, q, k, v, dout, lse, delta, c));
  FLEXATT_TRY(check_tensor(o, p->dtype));
  FLEXATT_TRY(check_out_tensor(dq, p->dtype, p->batch, p->heads_q, p->seqlen_q, p->head_dim));
  FLEXATT_TRY(check_out_tensor(dk, p->dtype, p->batch, p->heads_kv, p->seqlen_kv, p->head_dim));
  FLEXATT_TRY(check_out_tensor(dv, p->dtype, p->batch, p->heads_kv, p->seqlen_kv, p->head_dim));
  if (!bwd_split_applies(p)) return FLEXATT_ERANGE;
  const BwdSplitPlan plan = bwd_split_plan(p);
  if (plan.bytes && !workspace) return FLEXATT_EINVAL;
  if (workspace_bytes < plan.bytes) return FLEXATT_EINVAL;
  if (((uintptr_t)workspace) % 16 != 0) return FLEXATT_ELAYOUT;
  FLEXATT_TRY(flexatt_bwd_delta(p, o, dout, delta, stream));
  BwdSplitArgs a;
  a.q = c.q;
  a.k = c.k;
  a.v = c.v;
  a.dout = c.dout;
  a.lse = lse;
  a.delta = delta;
  a.dq = mview(dq);
  a.dk = mview(dk);
  a.dv = mview(dv);
  a.p = c.p;
  a.part = (float*)workspace;
  a.nsplit = plan.nsplit;
  a.nw = plan.nw;
  a.nkt = a.nrt = 0;
  return (int)kBwdSplit[p->dtype][head_index(p->head_dim)](a, (hipStream_t)stream);
}

size_t flexatt_bwd_workspace(const flexatt_problem* p) {
  if (check_problem(p) != FLEXATT_OK) return 0;
  const size_t n = ds_bytes(p);
  return n ? n + FLEXATT_BWD_QUEUE_BYTES : 0;
}

int flexatt_bwd_prefers_staging(const flexatt_problem* p) {
  if (flexatt_bwd_workspace(p) == 0) return 0;  // outside the staged range (or an invalid problem)
  // fp16/bf16 at head_dim 64 without soft-cap and without document, prefix or
  // block-map masks: the recomputing backward (the query-stationary dQ kernel
  // forming Delta, dK/dV without dS stores) measured 2-15% faster than
  // staging; with soft-cap its tanh recompute in dQ makes it 0-8% slower
  if (p->dtype != FLEXATT_F32 && p->head_dim == 64 && !(p->soft_cap > 0.f) && !has_masks(p)) return 0;
  return 1;
}

size_t flexatt_bwd_workspace_limited(const flexatt_problem* p, size_t limit_bytes) {
  const size_t full = flexatt_bwd_workspace(p);
  if (full == 0 || full <= limit_bytes) return full;
  const size_t gb = (size_t)ds_group_bytes(p);
  if (limit_bytes < gb + FLEXATT_BWD_QUEUE_BYTES) return 0;  // not even one group: recompute
  return (size_t)chunk_groups(p, limit_bytes - FLEXATT_BWD_QUEUE_BYTES) * gb + FLEXATT_BWD_QUEUE_BYTES;
}

namespace {
const BwdSplitLauncher kPartSum[3][4] = {
    {nullptr, nullptr, nullptr, nullptr},
    {bwd_split_sum_f16_d32, bwd_split_sum_f16_d64, bwd_split_sum_f16_d128, bwd_split_sum_f16_d256},
    {bwd_split_sum_bf16_d32, bwd_split_sum_bf16_d64, bwd_split_sum_bf16_d128, bwd_split_sum_bf16_d256},
};
int run_dkdv_ds(const flexatt_problem* p, const flexatt_tensor* q, const flexatt_tensor* k, const flexatt_tensor* v,
                const flexatt_tensor* dout, const float* lse, const float* delta, const flexatt_tensor* dk,
                const flexatt_tensor* dv, void* workspace, size_t workspace_bytes, int* queue, float* part, int nparts,
                void* stream) {
  BwdArgs a;
  FLEXATT_TRY(bwd_common(p, q, k, v, dout, lse, delta, a));
  FLEXATT_TRY(check_out_tensor(dk, p->dtype, p->batch, p->heads_kv, p->seqlen_kv, p->head_dim));
  FLEXATT_TRY(check_out_tensor(dv, p->dtype, p->batch, p->heads_kv, p->seqlen_kv, p->head_dim));
  FLEXATT_TRY(ds_workspace(p, workspace, workspace_bytes, a));
  a.dk = mview(dk);
  a.dv = mview(dv);
  a.queue = queue;
  a.nstatic = cu_count() & ~7;
  a.part = part;
  a.nparts = nparts;
  FLEXATT_TRY((int)pick_kv_ds(p)(a, (hipStream_t)stream));
  if (nparts == 1) return FLEXATT_OK;
  BwdSplitArgs s;
  s.dk = a.dk;
  s.dv = a.dv;
  s.p = a.p;
  s.part = part;
  s.nsplit = nparts;
  return (int)kPartSum[p->dtype][head_index(p->head_dim)](s, (hipStream_t)stream);
}

int run_dq_ds(const flexatt_problem* p, const flexatt_tensor* k, const void* workspace, size_t workspace_bytes,
              const flexatt_tensor* dq, int* queue, void* stream) {
  FLEXATT_TRY(check_problem(p));
  FLEXATT_TRY(check_tensor(k, p->dtype));
  FLEXATT_TRY(check_out_tensor(dq, p->dtype, p->batch, p->heads_q, p->seqlen_q, p->head_dim));
  BwdArgs a;
  a.k = view(k);
  a.dq = mview(dq);
  a.p = make_shape(p);
  a.ntiles = 0;
  a.delta_out = nullptr;
  a.queue = queue;
  a.nstatic = cu_count() & ~7;
  FLEXATT_TRY(ds_workspace(p, (void*)workspace, workspace_bytes, a));
  return (int)pick_dq_ds(p)(a, (hipStream_t)stream);
}
}  // namespace

int flexatt_bwd_dkdv_ds(const flexatt_problem* p, const flexatt_tensor* q, const flexatt_tensor* k,
                        const flexatt_tensor* v, const flexatt_tensor* dout, const float* lse, const float* delta,
                        const flexatt_tensor* dk, const flexatt_tensor* dv, void* workspace,
                        size_t workspace_bytes, void* stream) {
  return run_dkdv_ds(p, q, k, v, dout, lse, delta, dk, dv, workspace, workspace_bytes, nullptr, nullptr, 1,
                     stream);
}

int flexatt_bwd_dq_ds(const flexatt_problem* p, const flexatt_tensor* k, const void* workspace,
                      size_t workspace_bytes, const flexatt_tensor* dq, void* stream) {
  return run_dq_ds(p, k, workspace, workspace_bytes, dq, nullptr, stream);
}

size_t flexatt_bwd_ws_parts_bytes(const flexatt_problem* p) {
  if (check_problem(p) != FLEXATT_OK || !ds_applies(p)) return 0;
  const int n = staged_parts(p);
  return n > 1 ? part_bytes(p, n) : 0;
}

namespace {
// One staged pass (the arguments are checked): Delta, dK/dV writing dS, dQ.
int run_staged(const flexatt_problem* p, const flexatt_tensor* q, const flexatt_tensor* k, const flexatt_tensor* v,
               const flexatt_tensor* o, const flexatt_tensor* dout, const float* lse, float* delta,
               const flexatt_tensor* dq, const flexatt_tensor* dk, const flexatt_tensor* dv, void* workspace,
               size_t workspace_bytes, void* stream) {
  // queue counters after the dS band: [0] the dK/dV launch, [2] dQ
  int* queue = nullptr;
  if (workspace_bytes >= ds_bytes(p) + FLEXATT_BWD_QUEUE_BYTES && (cu_count() & ~7) > 0)
    queue = (int*)((char*)workspace + ds_bytes(p));
  FLEXATT_TRY(run_delta(p, o, dout, delta, queue, stream));
  float* part = nullptr;
  int nparts = queue ? staged_parts(p) : 1;
  if (nparts > 1 && workspace_bytes >= ds_bytes(p) + FLEXATT_BWD_QUEUE_BYTES + part_bytes(p, nparts))
    part = (float*)((char*)workspace + ds_bytes(p) + FLEXATT_BWD_QUEUE_BYTES);
  else
    nparts = 1;
  FLEXATT_TRY(run_dkdv_ds(p, q, k, v, dout, lse, delta, dk, dv, workspace, workspace_bytes, queue, part, nparts, stream));
  return run_dq_ds(p, k, workspace, workspace_bytes, dq, queue ? queue + 2 : nullptr, stream);
}
}  // namespace

int flexatt_bwd_ws(const flexatt_problem* p, const flexatt_tensor* q, const flexatt_tensor* k,
                   const flexatt_tensor* v, const flexatt_tensor* o, const flexatt_tensor* dout, const float* lse,
                   float* delta, const flexatt_tensor* dq, const flexatt_tensor* dk, const flexatt_tensor* dv,
                   void* workspace, size_t workspace_bytes, void* stream) {
  FLEXATT_TRY(check_problem(p));
  // outside the range, or no workspace at all: the recomputing backward
  if (!ds_applies(p) || (!workspace && workspace_bytes == 0))
    return flexatt_bwd(p, q, k, v, o, dout, lse, delta, dq, dk, dv, stream);
  BwdArgs a;
  FLEXATT_TRY(bwd_common(p, q, k, v, dout, lse, delta, a));
  FLEXATT_TRY(check_tensor(o, p->dtype));
  FLEXATT_TRY(check_out_tensor(dq, p->dtype, p->batch, p->heads_q, p->seqlen_q, p->head_dim));
  FLEXATT_TRY(check_out_tensor(dk, p->dtype, p->batch, p->heads_kv, p->seqlen_kv, p->head_dim));
  FLEXATT_TRY(check_out_tensor(dv, p->dtype, p->batch, p->heads_kv, p->seqlen_kv, p->head_dim));
  if (!workspace) return FLEXATT_EINVAL;
  if (((uintptr_t)workspace) % 16 != 0) return FLEXATT_ELAYOUT;
  if (workspace_bytes >= ds_bytes(p))
    return run_staged(p, q, k, v, o, dout, lse, delta, dq, dk, dv, workspace, workspace_bytes, stream);
  // A smaller workspace: passes over chunks of whole (batch, KV head) groups.
  if (workspace_bytes < (size_t)ds_group_bytes(p)) return FLEXATT_EINVAL;
  const int64_t kg = chunk_groups(p, workspace_bytes);
  const int G = p->heads_q / p->heads_kv;
  const int nbc = kg >= p->heads_kv ? (int)(kg / p->heads_kv) : 1;  // batches per pass
  const int nhc = kg >= p->heads_kv ? p->heads_kv : (int)kg;        // KV heads per pass
  for (int b0 = 0; b0 < p->batch; b0 += nbc)
    for (int h0 = 0; h0 < p->heads_kv; h0 += nhc) {
      const Chunk c{b0, nbc < p->batch - b0 ? nbc : p->batch - b0, h0, nhc < p->heads_kv - h0 ? nhc : p->heads_kv - h0};
      const flexatt_problem sp = sub_problem(p, c);
      const int64_t hq0 = (int64_t)h0 * G;
      const flexatt_tensor sq = sub_tensor(q, p->dtype, b0, hq0), sk = sub_tensor(k, p->dtype, b0, h0),
                           sv = sub_tensor(v, p->dtype, b0, h0), so = sub_tensor(o, p->dtype, b0, hq0),
                           sdo = sub_tensor(dout, p->dtype, b0, hq0), sdq = sub_tensor(dq, p->dtype, b0, hq0),
                           sdk = sub_tensor(dk, p->dtype, b0, h0), sdv = sub_tensor(dv, p->dtype, b0, h0);
      const int64_t r0 = ((int64_t)b0 * p->heads_q + hq0) * p->seqlen_q;  // first LSE / Delta row
      FLEXATT_TRY(run_staged(&sp, &sq, &sk, &sv, &so, &sdo, lse + r0, delta + r0, &sdq, &sdk, &sdv, workspace,
                             workspace_bytes, stream));
    }
  return FLEXATT_OK;
}

}  // extern "C"
