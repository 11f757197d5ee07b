// Paged causal prefill (ragged, prefix-cache aware) on gfx950 matrix cores.
//
// Reference semantics: FlashInferBackend::forward, prefill branch
// (src/attention/flashinfer_backend.cu:596-679) with MaskMode::kCausal:
// query i of request r (qo_len q_r, kv_len k_r) attends kv token j iff
// j <= i + (k_r - q_r) (bottom-right alignment, so cached prefix tokens are
// visible to every new token), kv slots taken from the token-granular
// indices[kv_indptr[r] + j].
//
// Work decomposition: one workgroup (4 or 8 waves, 32 query rows each) per
// (request, kv head, query tile), or per pair of tiles from both ends of the
// causal range (see paged_prefill_kernel). The G query heads that share a kv
// head are packed row-wise (packed row p -> token p / G, head h G + p % G),
// so each K/V tile staged in LDS feeds G heads. K/V tiles of 64 tokens are
// gathered from the pool (one 16-byte chunk per lane, slots from the index
// list) into a double-buffered LDS ring; the gathers of the next tiles are
// in flight while the current one is on the matrix cores.
//
// Matrix formulation (v_mfma_f32_32x32x16_bf16, lane l, c = l % 32, hl = l / 32):
//   S^T[tok, row] = K[tok, :] . Q[row, :]      (A = K from LDS, B = Q^T in VGPRs)
//   O^T[d, row]  += V^T[d, tok] . P^T[tok, row] (A = V^T by LDS transpose reads)
// The query row sits on the lane's column c in both products, so the online
// softmax (max, sum, rescale of O) is lane-local apart from one exchange with
// lane l ^ 32. V^T comes straight from the row-major V tile through
// ds_read_b64_tr_b16.
#include <algorithm>

#include "prefill_impl.h"

namespace sgl {
namespace pf {
namespace {

// The plan's model of a launch, in 0.1 us, from 32q/8kv launches that fill
// the device: a step of a planned item by its waves of rows (33 us of 18
// steps at one to four waves, 44, 48, 52 and 57 us at five to eight, of which
// 8 are the launch and the states), the states a share writes (17 KiB a wave),
// the shortest share worth its prologue, and the fold's launch; the fold reads
// the states at about 7 TB/s, mostly from the last-level cache. The last three
// were set where both routes were timed: 500 new tokens on 3000 cached 63 -> 50
// us a layer, 100 on 1500 34 -> 23, 512 on 1000 (16q/8kv) 35 -> 30, while
// 1000 tokens without a prefix (34 us, planned 40) and 100 on 500 (20 and 20)
// stay unplanned. Over 111 batches that are planned (2 to 600 new tokens on 64 to
// 16,000, up to 16 requests, twelve head layouts) the planned route takes 0.45 of
// the other's time on average and was the slower one once, by 4%.
constexpr int32_t kStepCost[9] = {0, 14, 14, 15, 15, 20, 22, 24, 27};
constexpr int64_t kStateCost = 2;
constexpr int64_t kMinShare = 60;
constexpr int64_t kFoldCost = 35;
constexpr int64_t kMaxListed = 512;  // query tiles, and shares, of a plan
static_assert(4 * (kMaxListed + kMaxListed / 2) <= SGL_PREFILL_PLAN_INTS,
              "a folded tile has at least two shares");

// Two workgroups per CU at 4 waves, one at 8; the split-kv variant (KS = 2)
// holds the whole LDS, so one.
template <int W, bool kPair, int KS>
__global__ void __launch_bounds__(64 * W, KS == 2 ? 1 : 8 / W) paged_prefill_kernel(PrefillArgs a) {
  __shared__ __attribute__((aligned(16))) char lds_raw[prefill_lds_bytes<W, KS>()];
  prefill_item<W, kPair, KS>(a, lds_raw, blockIdx.x, gridDim.x);
}

// Items of a host plan (sgl_prefill_plan): query tiles of up to 256 rows, long
// kv ranges cut into shares.
__global__ void __launch_bounds__(2 * kListRows, 1) paged_prefill_list_kernel(PrefillArgs a) {
  __shared__ __attribute__((aligned(16))) char lds_raw[prefill_lds_bytes<kListRows / 32, 1>()];
  prefill_item<kListRows / 32, false, 1, true>(a, lds_raw, blockIdx.x, gridDim.x);
}

// Folds the shares of one query tile: workgroup (merge m, kv head; db; row
// group w) takes d = [32 db, 32 db + 32) of the tile's rows [32 w, 32 w + 32),
// lane for lane as wave w of the items holds them. Bound by the latency of
// the loads: the four waves each fold a quarter of the shares, four shares'
// loads in flight at a time, and are folded in wave order through LDS.
constexpr int kFoldWaves = 4;

__global__ void __launch_bounds__(64 * kFoldWaves) prefill_merge_kernel(PrefillArgs a,
                                                                        const int32_t* merges) {
  __shared__ float xch[18][kFoldWaves][64];
  const int m = blockIdx.x / a.num_kv_heads;
  const int h = blockIdx.x - m * a.num_kv_heads;
  const int db = blockIdx.y, w = blockIdx.z;
  const int r = merges[4 * m], tile = merges[4 * m + 1];
  const int e0 = merges[4 * m + 2], n = merges[4 * m + 3];
  const int rows = (a.qo_indptr[r + 1] - a.qo_indptr[r]) * a.group;
  const int row0 = (tile >> 4) + 32 * w;
  if (w >= (tile & 15) || row0 >= rows) return;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const float* p0 = a.part + (static_cast<int64_t>(e0) * a.num_kv_heads + h) * kPartFloats +
                    64 * w + lane;
  const int64_t step = static_cast<int64_t>(a.num_kv_heads) * kPartFloats;
  float mx = -INFINITY, den = 0.f, acc[16];
#pragma unroll
  for (int v = 0; v < 16; ++v) acc[v] = 0.f;
  const int per = (n + kFoldWaves - 1) / kFoldWaves;
  const int k1 = min(n, (wave + 1) * per);
  for (int k = wave * per; k < k1; k += 4) {
    float x[4][18];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float* p = p0 + min(k + i, k1 - 1) * step;
#pragma unroll
      for (int v = 0; v < 16; ++v) x[i][v] = p[(16 * db + v) * 2 * kListRows];
      x[i][16] = k + i < k1 ? p[64 * 2 * kListRows] : -INFINITY;
      x[i][17] = p[65 * 2 * kListRows];
    }
    float mc = mx;
#pragma unroll
    for (int i = 0; i < 4; ++i) mc = fmaxf(mc, x[i][16]);
    const float keep = mx == -INFINITY ? 0.f : exp2f(mx - mc);
    den *= keep;
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[v] *= keep;
    mx = mc;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (k + i >= k1) break;  // the last share again: not added, it may hold infinities
      const float wgt = x[i][16] == -INFINITY ? 0.f : exp2f(x[i][16] - mc);
      den += x[i][17] * wgt;
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[v] += x[i][v] * wgt;
    }
  }
#pragma unroll
  for (int v = 0; v < 16; ++v) xch[v][wave][lane] = acc[v];
  xch[16][wave][lane] = mx;
  xch[17][wave][lane] = den;
  __syncthreads();
  // Wave g writes the values [4 g, 4 g + 4): d = 32 db + 8 g + 4 (lane / 32) + i.
  const int g = wave;
  float all = -INFINITY;
#pragma unroll
  for (int f = 0; f < kFoldWaves; ++f) all = fmaxf(all, xch[16][f][lane]);
  float sum = 0.f, o4[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int f = 0; f < kFoldWaves; ++f) {
    const float mf = xch[16][f][lane];
    const float wgt = mf == -INFINITY ? 0.f : exp2f(mf - all);
    sum += xch[17][f][lane] * wgt;
#pragma unroll
    for (int i = 0; i < 4; ++i) o4[i] += xch[4 * g + i][f][lane] * wgt;
  }
  const int prow = row0 + (lane & 31);
  if (prow >= rows) return;
  const float inv = sum > 0.f ? 1.0f / sum : 0.f;
  const int tok = prow / a.group;
  const int qo_beg = a.q_start ? a.q_start[r] : a.qo_indptr[r];
  uint16_t* op = a.o + static_cast<int64_t>(qo_beg + tok) * a.o_st +
                 static_cast<int64_t>(h * a.group + (prow - tok * a.group)) * a.o_sh + 32 * db +
                 8 * g + 4 * (lane >> 5);
  *reinterpret_cast<u32x2_t*>(op) =
      u32x2_t{pack_bf16x2(o4[0] * inv, o4[1] * inv), pack_bf16x2(o4[2] * inv, o4[3] * inv)};
}

}  // namespace
}  // namespace pf
}  // namespace sgl

using namespace sgl;
using namespace sgl::pf;

// Compute units of the current device (256 on MI355X; 256 when none is visible).
static int device_cus() {
  int dev = 0, cus = 0;
  if (hipGetDevice(&dev) == hipSuccess &&
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess &&
      cus > 0)
    return cus;
  return 256;
}

extern "C" int sgl_paged_prefill(const void* q, int64_t q_stride_token, int64_t q_stride_head,
                                 const void* k_cache, const void* v_cache, int64_t kv_stride_slot,
                                 int64_t kv_stride_head, const int32_t* indices,
                                 const int32_t* qo_indptr, const int32_t* kv_indptr,
                                 const int32_t* q_start, int batch_size, int max_qo_len,
                                 int num_qo_heads,
                                 int num_kv_heads, int head_dim, float sm_scale, void* o,
                                 int64_t o_stride_token, int64_t o_stride_head, void* stream) {
  if (batch_size < 0 || max_qo_len < 0 || num_qo_heads <= 0 || num_kv_heads <= 0)
    return SGL_ERR_INVALID_ARG;
  if (batch_size == 0 || max_qo_len == 0) return SGL_OK;
  PrefillArgs a{};
  const int st = prefill_args(q, q_stride_token, q_stride_head, k_cache, v_cache, kv_stride_slot,
                              kv_stride_head, indices, qo_indptr, kv_indptr, q_start,
                              num_qo_heads, num_kv_heads, head_dim, sm_scale, o,
                              o_stride_token, o_stride_head, a);
  if (st != SGL_OK) return st;
  const int group = a.group;
  // 8-wave workgroups pay off on long chunks that still fill every CU once
  // (measured: 2048-token chunks at G = 8, 4096 at G = 4); short or few
  // chunks keep 4-wave workgroups, two per CU.
  const int64_t rows_max = static_cast<int64_t>(max_qo_len) * group;
  const int64_t tiles8 = (rows_max + 255) / 256;
  const bool wide = rows_max >= 8192 &&
                    tiles8 * num_kv_heads * batch_size >= static_cast<int64_t>(device_cus());
  // Pairing (one tile from each end of the causal range per workgroup) when
  // the launch is at most one workgroup per CU: the dispatcher cannot then
  // even out unequal tiles, and measured it is 3-6% faster; with several
  // workgroups per CU, heavy-first dispatch balances better.
  const int64_t pairs = ((rows_max + 127) / 128 + 1) / 2;
  const bool pair = wide && pairs * num_kv_heads * batch_size <= static_cast<int64_t>(device_cus());
  // Launches that would leave CUs idle even with 64-row items split each
  // item's kv tiles between two 2-wave groups (KS = 2): 64-row items reach
  // twice the CUs, each group streaming half the kv tiles.
  const bool split_kv = !wide && ((rows_max + 63) / 64) * num_kv_heads * batch_size <=
                                     static_cast<int64_t>(device_cus());
  const int bm = wide ? 256 : split_kv ? 64 : 128;
  const int64_t items = pair ? pairs * num_kv_heads * batch_size
                             : unpaired_items(a, max_qo_len, bm, batch_size);
  if (items > 0x7fffffff) return SGL_ERR_INVALID_ARG;
  if (pair) a.tiles_per_req = static_cast<int>(pairs);
  const dim3 grid(static_cast<uint32_t>(items));
  const hipStream_t s = static_cast<hipStream_t>(stream);
  if (pair)
    hipLaunchKernelGGL((paged_prefill_kernel<8, true, 1>), grid, dim3(512), 0, s, a);
  else if (wide)
    hipLaunchKernelGGL((paged_prefill_kernel<8, false, 1>), grid, dim3(512), 0, s, a);
  else if (split_kv)
    hipLaunchKernelGGL((paged_prefill_kernel<4, false, 2>), grid, dim3(256), 0, s, a);
  else
    hipLaunchKernelGGL((paged_prefill_kernel<4, false, 1>), grid, dim3(256), 0, s, a);
  return launch_status();
}

// ------------------------------------------------------------------ planned prefill
//
// Query tiles are the only parallelism of the launches above: a few new
// tokens behind a long cached prefix (the next turn of a chat) are a handful
// of tiles, each walking thousands of kv tokens on its own CU while the rest
// idle. With the lengths on the host, the plan cuts the kv ranges of 256-row
// query tiles into shares of about equal length that fill the device's
// workgroup slots (one per CU) and lists the shares, longest first; a second
// launch folds them.

extern "C" int sgl_prefill_plan(const int32_t* qo_indptr_host, const int32_t* kv_indptr_host,
                                int batch_size, int num_qo_heads, int num_kv_heads, int head_dim,
                                sgl_prefill_plan_t* plan, int32_t* items, int64_t capacity) {
  if (!qo_indptr_host || !kv_indptr_host || !plan || !items || batch_size < 0 || capacity < 0 ||
      num_qo_heads <= 0 || num_kv_heads <= 0 || num_qo_heads % num_kv_heads != 0)
    return SGL_ERR_INVALID_ARG;
  if (head_dim != kD) return SGL_ERR_UNSUPPORTED;
  *plan = sgl_prefill_plan_t{};
  plan->num_qo_heads = num_qo_heads;
  plan->num_kv_heads = num_kv_heads;
  plan->head_dim = head_dim;
  const int group = num_qo_heads / num_kv_heads;
  // Workgroup slots per kv head: one per CU.
  const int64_t cus = device_cus();
  const int64_t slots = std::min<int64_t>(kMaxListed, cus / num_kv_heads);
  // Query tiles, the kv tiles each one walks (as the kernel counts them) and
  // what a step costs, in 0.1 us.
  struct Tile { int32_t r, row0, waves, n, cost, share; } list[kMaxListed];
  int64_t tiles = 0, total = 0, longest = 0, longest_n = 0, items64 = 0, items128 = 0;
  for (int r = 0; r < batch_size; ++r) {
    const int64_t qo = qo_indptr_host[r + 1] - static_cast<int64_t>(qo_indptr_host[r]);
    const int64_t kv = kv_indptr_host[r + 1] - static_cast<int64_t>(kv_indptr_host[r]);
    if (qo < 0 || kv < 0) return SGL_ERR_INVALID_ARG;
    // The waves of the request's rows, spread evenly over its tiles.
    const int64_t rows = qo * group, nw = (rows + 31) / 32, nt = (nw + kListRows / 32 - 1) / (kListRows / 32);
    // Enough query tiles for the device, or rows that see no token (written
    // by the unplanned launch): nothing to plan.
    if (tiles + nt > slots || kv < qo) return SGL_OK;
    items64 = std::max(items64, (rows + 63) / 64);
    items128 += (rows + 127) / 128;
    int64_t row0 = 0;
    for (int64_t i = 0; i < nt; ++i) {
      const int64_t waves = nw / nt + (i < nw % nt);
      const int64_t last = std::min(rows, row0 + 32 * waves) - 1;
      const int64_t n = (std::min(kv, last / group + kv - qo + 1) + kBN - 1) / kBN;
      list[tiles++] = {r, static_cast<int32_t>(row0), static_cast<int32_t>(waves),
                       static_cast<int32_t>(n), kStepCost[waves], 0};
      total += n * kStepCost[waves];
      longest = std::max<int64_t>(longest, n * kStepCost[waves]);
      longest_n = std::max(longest_n, n);
      row0 += 32 * waves;
    }
  }
  if (tiles == 0) return SGL_OK;
  // The shortest time in which every tile's shares, all running at once, can
  // be done; a tile that is cut also writes its states.
  auto tile_shares = [](const Tile& t, int64_t c) {
    const int64_t walk = static_cast<int64_t>(t.n) * t.cost, room = c - kStateCost * t.waves;
    return walk <= c ? int64_t{1} : std::min<int64_t>(t.n, (walk + room - 1) / room);
  };
  auto shares = [&](int64_t c) {
    int64_t k = 0;
    for (int64_t t = 0; t < tiles; ++t) k += tile_shares(list[t], c);
    return k;
  };
  int64_t c = std::max(kMinShare, (total + slots - 1) / slots), hi = std::max(c, longest);
  while (c < hi) {
    const int64_t mid = (c + hi) / 2;
    if (shares(mid) > slots) c = mid + 1; else hi = mid;
  }
  int64_t states = 0;  // waves of rows whose states are written
  for (int64_t t = 0; t < tiles; ++t) {
    const int64_t k = tile_shares(list[t], c);
    if (k > 1) states += k * list[t].waves;
  }
  // Against the unplanned launch: two 64-row groups a workgroup, each on half
  // of the kv tiles, or 128-row tiles, where a second workgroup on some CUs
  // slows the first.
  const int64_t wgs = items128 * num_kv_heads;
  const int64_t unplanned = items64 * batch_size * num_kv_heads <= cus
                                ? longest_n * 9
                                : longest_n * 13 * std::max(wgs, cus) / cus;
  if (c + kFoldCost + states * num_kv_heads / 40 >= unplanned) return SGL_OK;
  for (int64_t t = 0; t < tiles; ++t) {
    const int64_t k = tile_shares(list[t], c);
    list[t].share = static_cast<int32_t>((list[t].n + k - 1) / k);
  }
  // Longest shares first; a tile's shares stay together for the fold.
  std::sort(list, list + tiles, [](const Tile& x, const Tile& y) {
    const int64_t a = static_cast<int64_t>(x.share) * x.cost;
    const int64_t b = static_cast<int64_t>(y.share) * y.cost;
    return a != b ? a > b : x.r != y.r ? x.r < y.r : x.row0 < y.row0;
  });
  int64_t n_items = 0, n_merges = 0;
  for (int64_t t = 0; t < tiles; ++t) {
    n_items += (list[t].n + list[t].share - 1) / list[t].share;
    n_merges += list[t].n > list[t].share;
  }
  if (4 * (n_items + n_merges) > capacity) return SGL_ERR_CAPACITY;
  int32_t* it = items;
  int32_t* mg = items + 4 * n_items;
  for (int64_t t = 0; t < tiles; ++t) {
    const Tile& x = list[t];
    const bool part = x.n > x.share;
    const int32_t first = static_cast<int32_t>((it - items) / 4);
    const int32_t tile = x.row0 << 4 | x.waves;
    for (int32_t t0 = 0; t0 < x.n; t0 += x.share, it += 4) {
      const int32_t end = std::min(x.n, t0 + x.share);
      it[0] = x.r, it[1] = tile, it[2] = t0, it[3] = part ? end | kPartial : end;
    }
    if (part) {
      mg[0] = x.r, mg[1] = tile, mg[2] = first;
      mg[3] = static_cast<int32_t>((it - items) / 4) - first;
      mg += 4;
    }
  }
  plan->num_items = static_cast<int32_t>((it - items) / 4);
  plan->num_merges = static_cast<int32_t>(n_merges);
  plan->workspace_bytes = static_cast<int64_t>(plan->num_items) * num_kv_heads * kPartFloats * 4;
  return SGL_OK;
}

extern "C" int sgl_paged_prefill_planned(
    const sgl_prefill_plan_t* plan, const int32_t* items, const void* q, int64_t q_stride_token,
    int64_t q_stride_head, const void* k_cache, const void* v_cache, int64_t kv_stride_slot,
    int64_t kv_stride_head, const int32_t* indices, const int32_t* qo_indptr,
    const int32_t* kv_indptr, const int32_t* q_start, int num_qo_heads, int num_kv_heads,
    int head_dim, float sm_scale, void* o, int64_t o_stride_token, int64_t o_stride_head,
    void* workspace, int64_t workspace_bytes, void* stream) {
  if (!plan || !items || plan->num_items <= 0 || plan->num_merges < 0) return SGL_ERR_INVALID_ARG;
  if (num_qo_heads != plan->num_qo_heads || num_kv_heads != plan->num_kv_heads)
    return SGL_ERR_INVALID_ARG;
  PrefillArgs a{};
  int st = prefill_args(q, q_stride_token, q_stride_head, k_cache, v_cache, kv_stride_slot,
                        kv_stride_head, indices, qo_indptr, kv_indptr, q_start, num_qo_heads,
                        num_kv_heads, head_dim, sm_scale, o, o_stride_token, o_stride_head, a);
  if (st != SGL_OK) return st;
  const int64_t grid = static_cast<int64_t>(plan->num_items) * num_kv_heads;
  if (grid > 0x7fffffff) return SGL_ERR_INVALID_ARG;
  if (!workspace || workspace_bytes < grid * kPartFloats * 4) return SGL_ERR_CAPACITY;
  if (!aligned16(workspace)) return SGL_ERR_ALIGNMENT;
  a.items = items;
  a.part = static_cast<float*>(workspace);
  const hipStream_t s = static_cast<hipStream_t>(stream);
  hipLaunchKernelGGL(paged_prefill_list_kernel, dim3(static_cast<uint32_t>(grid)),
                     dim3(2 * kListRows), 0, s, a);
  st = launch_status();
  if (st != SGL_OK || plan->num_merges == 0) return st;
  hipLaunchKernelGGL(prefill_merge_kernel, dim3(plan->num_merges * num_kv_heads, 4, kListRows / 32),
                     dim3(64 * kFoldWaves), 0, s, a, items + 4 * static_cast<int64_t>(plan->num_items));
  return launch_status();
}
