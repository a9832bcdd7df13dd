// extern "C" entry points of libpallas_flash_amd.so (declared in
// include/pallas_flash_amd.h). Each one validates its arguments on the host
// (no HIP call before validation passes), fills a kernel parameter block and
// enqueues on the caller's stream. Nothing here allocates or synchronises.
#include <math.h>
#include <stdint.h>
#include <stdlib.h>

#include <algorithm>
#include <atomic>
#include <mutex>

#include "../../include/pallas_flash_amd.h"
#include "pf_kernels.hpp"

namespace {

// Process-wide tuning (pf_get_tuning / pf_set_tuning). The environment is read
// once, at the first call that needs a value; afterwards every launch reads
// three atomics and makes no environment or device query of its own.
// Share of a prefill launch's work items handed out by tickets (plan_tail).
constexpr int kDefaultTailDynamicPct = 30;

struct Tuning {
  std::atomic<int> tail_dynamic_pct{kDefaultTailDynamicPct};
  std::atomic<int> decode_stages{2};
  std::atomic<int> decode_waves{0};
};

bool tuning_valid(int dyn, int stages, int waves) {
  return dyn >= 0 && dyn <= 100 && stages >= 2 && stages <= 4 && waves >= 0;
}

Tuning& tuning() {
  static Tuning t;
  static std::once_flag once;
  std::call_once(once, [] {
    const char* f = getenv("PF_TAIL_DYNAMIC_PCT");
    const char* s = getenv("PF_DECODE_STAGES");
    const char* w = getenv("PF_DECODE_WAVES");
    if (f != nullptr && atoi(f) >= 0 && atoi(f) <= 100) t.tail_dynamic_pct = atoi(f);
    if (s != nullptr && atoi(s) >= 2 && atoi(s) <= 4) t.decode_stages = atoi(s);
    if (w != nullptr && atoi(w) > 0) t.decode_waves = atoi(w);
  });
  return t;
}

bool dtype_ok(int32_t d) { return d == PF_DTYPE_F32 || d == PF_DTYPE_BF16 || d == PF_DTYPE_F16; }
// Kernel head dims: 64 and 128 for every dtype, 256 for bf16/f16 (a float32
// tile of 256 columns would not fit the LDS double buffers). dtype must
// already be valid.
int32_t max_head_dim(int32_t dtype) { return dtype == PF_DTYPE_F32 ? 128 : 256; }
bool head_dim_ok(int32_t d, int32_t dtype) { return d == 64 || d == 128 || (d == 256 && d <= max_head_dim(dtype)); }

// Decode and paged decode also read rows of any head_dim up to the dtype's
// maximum that are whole 16-byte chunks (a multiple of 8 elements for
// bf16/f16, 4 for float32) in place: the generic kernel computes at the next
// kernel head dim with the missing columns as zeros.
bool decode_head_dim_ok(int32_t d, int32_t dtype) {
  const int32_t es = dtype == PF_DTYPE_F32 ? 4 : 2;
  return d >= 1 && d <= max_head_dim(dtype) && (d * es) % 16 == 0;
}
int32_t decode_compute_dim(int32_t d) { return d <= 64 ? 64 : d <= 128 ? 128 : 256; }

constexpr int64_t kMaxGrid = 0x7fffffff;
constexpr int kCus = 256;  // of an MI355X

int check_attn_dims(int32_t B, int32_t Hq, int32_t Hkv, int32_t Sq, int32_t Sk, int32_t D,
                    int32_t kv_len, float scale, int32_t dtype) {
  // flash_attention.py:527-545: ranks/shape agreement, Hq % Hkv, kv_len in (0, Sk].
  if (B < 0 || Hq < 1 || Hkv < 1 || Sq < 0 || Sk < 1 || D < 1) return PF_ERR_INVALID;
  if (Hq % Hkv != 0) return PF_ERR_INVALID;
  if (kv_len < 1 || kv_len > Sk) return PF_ERR_INVALID;
  if (!isfinite(scale)) return PF_ERR_INVALID;
  if (!dtype_ok(dtype)) return PF_ERR_UNSUPPORTED;
  if (!head_dim_ok(D, dtype)) return PF_ERR_UNSUPPORTED;
  return PF_OK;
}

int finish(hipError_t e) { return e == hipSuccess ? PF_OK : PF_ERR_LAUNCH; }

// (batch, kv head) pairs each XCD streams at a time in the forward
// (fwd_work_item): with more than one pair per XCD, the largest divisor of
// the per-XCD pair count whose pairs' live K/V (kv_len rows each) fits an
// XCD's 4 MB L2, at least 1; 0 (the default item order) when the pairs are
// not a multiple of the 8 XCDs or one pair per XCD. (Config 2's shape, four
// 2 MiB pairs per XCD: two at a time measured 1.5% faster than one and as
// fast as all four, with half of their HBM traffic.)
int fwd_pair_group(const pf_attn_fwd_args* a) {
  const int64_t npairs = (int64_t)a->batch * a->num_kv_heads;
  if (npairs % 8 != 0 || npairs == 8) return 0;
  const int per_xcd = (int)(npairs / 8);
  const int64_t es = a->dtype == PF_DTYPE_F32 ? 4 : 2;
  const int64_t pair_bytes = (int64_t)a->kv_len * a->head_dim * es * 2;
  int best = 1;
  for (int P = 1; P <= per_xcd; ++P)
    if (per_xcd % P == 0 && P * pair_bytes <= (int64_t)(4 << 20)) best = P;
  return best;
}

int fill_fwd(const pf_attn_fwd_args* a, pf::FwdParams* p) {
  int st = check_attn_dims(a->batch, a->num_heads, a->num_kv_heads, a->seq_len_q, a->seq_len_k,
                           a->head_dim, a->kv_len, a->sm_scale, a->dtype);
  if (st != PF_OK) return st;
  if (!a->q || !a->k || !a->v || !a->o) return PF_ERR_INVALID;
  p->q = a->q;
  p->k = a->k;
  p->v = a->v;
  p->o = a->o;
  p->lse = a->lse;
  p->q_cos = p->q_sin = nullptr;
  p->B = a->batch;
  p->Hq = a->num_heads;
  p->Hkv = a->num_kv_heads;
  p->Sq = a->seq_len_q;
  p->Sk = a->seq_len_k;
  p->kv_len = a->kv_len;
  p->g = a->num_heads / a->num_kv_heads;
  p->scale_log2 = a->sm_scale * 1.4426950408889634f;
  // A workgroup's 4 waves cover hpw query heads of one GQA group x rpw rows:
  // the K/V tiles it stages serve all of them.
  p->hpw = (p->g % 4 == 0) ? 4 : (p->g % 2 == 0) ? 2 : 1;
  p->rpw = 128 / p->hpw;
  p->n_qblk = (a->seq_len_q + p->rpw - 1) / p->rpw;
  const int64_t n_work = (int64_t)a->batch * (a->num_heads / p->hpw) * p->n_qblk;
  if (n_work > kMaxGrid) return PF_ERR_UNSUPPORTED;
  // per-(batch, kv head) byte offsets are 32-bit inside the kernels
  if ((int64_t)(a->seq_len_k + 256) * a->head_dim * 4 > 0x7fffffff) return PF_ERR_UNSUPPORTED;
  p->n_work = (int)n_work;
  p->pair_group = fwd_pair_group(a);
  // Causal items that are all resident at once (no slot takes a second one)
  // gain nothing from heavy first alone: a CU's items then add up unevenly.
  // With every other round of 256 reversed they add up alike. 16-bit head_dim
  // 64, three workgroups a CU: B=4, 4 heads, S=5905 94.7 -> 89.7 us; up to 2%
  // elsewhere, and nothing at two a CU.
  p->snake = a->causal && a->head_dim == 64 && a->dtype != PF_DTYPE_F32 && n_work <= 3 * kCus;
  p->tail = pf::WorkTail{nullptr, p->n_work, 0};
  p->n_split = 1;
  p->chunk = p->split_grid = 0;
  p->part_o = p->part_ml = nullptr;
  return PF_OK;
}

// Dynamic tail of a prefill launch (pf::WorkTail): the last tail_dynamic_pct
// percent of the work items (the lightest under the heavy-first orders) go to
// ticket-drawing workgroups, kTailSlack times as many as those items so an
// XCD that runs ahead can take up to that multiple of its share. The static
// part is a multiple of the 8 XCDs so each gets the same number of its own
// items. Launches of fewer than min_items items (two per resident workgroup
// slot of the kernel) keep every item static, as do launches whose stream
// gets no ticket counter. The dK/dV kernel, one workgroup per CU and two
// items per CU, gains nothing from a tail (measured) and runs without one:
// its items drawn by other XCDs only add HBM traffic (889 against 578 MB at
// config 3).
constexpr double kTailSlack = 2.0;

pf::WorkTail plan_tail(int n_work, int min_items, hipStream_t stream) {
  pf::WorkTail w{nullptr, n_work, 0};
  const int pct = tuning().tail_dynamic_pct.load(std::memory_order_relaxed);
  if (pct <= 0 || n_work < min_items) return w;
  const int n_static = 8 * (int)(((int64_t)n_work * (100 - pct) / 100) / 8);
  const int pool = n_work - n_static;
  if (pool <= 0) return w;
  unsigned int* t = pf::work_tickets(stream);
  if (t == nullptr) return w;
  w.tickets = t;
  w.n_static = n_static;
  w.n_tickets = (int)(pool * kTailSlack) + 1;
  return w;
}

// ---------------------------------------------------------------------------
// Split plans. A prefill launch with fewer work items than CUs leaves CUs idle
// while each item walks its whole key range (forward, dQ) or all its query
// blocks (dK/dV) alone: 32 items of 64 steps took 1020 us in float32 dK/dV,
// where 1152 steps on 256 CUs are 72 us of work. Such launches cut every item
// into chunks of `per` steps, one workgroup each, with float32 partials that a
// second kernel sums.
//
// plan_split returns the steps per chunk, or 0 to leave the items whole: the
// chunk that minimises a model of the launch time,
//   rounds of 256 workgroups x (start + per x step) + (kSplitLaunch + partial
//   bytes written and read back),
// against the whole items' start + step x (the longest item's steps, or a CU's
// share of all steps where that is more). Step times are measured, one
// workgroup per CU (two resident ones take about twice as long per step, so
// counting 256 at a time prices them alike). wgs(per): the workgroups of that
// chunk; min_per: the chunk's granularity.
// ---------------------------------------------------------------------------
struct StepCost {
  double fwd, dq, dkv;  // us per step (64 keys, 64 keys, 128 or 64 query rows)
};
StepCost step_cost(int32_t dtype, int32_t head_dim) {
  if (dtype == PF_DTYPE_F32) return head_dim == 64 ? StepCost{4.6, 6.6, 8.0} : StepCost{9.0, 13.0, 16.0};
  if (head_dim == 64) return {0.6, 0.9, 2.0};
  if (head_dim == 256) return {2.0, 3.2, 3.9};
  return {1.0, 1.5, 3.8};
}
constexpr double kStartUs = 5.0;        // a workgroup's prologue and epilogue
constexpr double kSplitLaunchUs = 5.0;  // the second kernel
constexpr double kPartialBytesPerUs = 4.0e6;
constexpr int kMaxSplit = 64;
// The partials of one kernel at most: a call must not need memory out of
// proportion to its own. Without a bound the model alone asked up to 2 GiB (float32
// dK/dV, 32/1 heads, 32768 keys, whose gradients are 544 MiB). At 192 MiB 1 in 100
// causal training shapes of up to 8192 rows loses over 2% of its modelled time, the
// worst 10%; at 128 MiB 2 in 100, the worst 37%; at 64 MiB 8 in 100, the worst 103%.
constexpr int64_t kMaxPartialBytes = (int64_t)192 << 20;

template <typename F>
int plan_split(int64_t items, int max_steps, double total_steps, int min_per, double step_us, int64_t partial_bytes,
               F wgs) {  // partial_bytes: of one chunk of every item
  if (items <= 0 || items >= 2 * kCus) return 0;
  double best = kStartUs + step_us * fmax((double)max_steps, total_steps / kCus);
  int best_per = 0, last = 0;
  for (int n = 2; n <= kMaxSplit; n += 1 + n / 8) {
    int per = (max_steps + n - 1) / n;
    per = (per + min_per - 1) / min_per * min_per;
    if (per >= max_steps || per == last) continue;
    last = per;
    if ((max_steps + per - 1) / per * partial_bytes > kMaxPartialBytes) break;
    const double n_wgs = wgs(per);
    const double us = ceil(n_wgs / kCus) * (kStartUs + per * step_us) + kSplitLaunchUs +
                      2.0 * n_wgs / (double)items * (double)partial_bytes / kPartialBytesPerUs;
    if (us < 0.95 * best) {
      best = us;
      best_per = per;
    }
  }
  return best_per;
}

size_t align_ws(size_t x) { return (x + 255) & ~(size_t)255; }

// Workgroups of the key split into chunks of 64 per keys, for one head of one
// batch: chunks summed over the query blocks of `rows` (32, 64 or 128) rows, which
// need all of kv_len, or up to their diagonal. (per = 1: the steps.) Chunk c is
// needed by all blocks but the first floor(64 per c / rows). In closed form: the
// planner asks for some 20 values of per, where a loop over the blocks took 23 us
// at 16000 rows.
double key_split_grid(int Sq, int rows, int kv_len, int per, bool causal) {
  const double nq = (Sq + rows - 1) / rows;
  const int keys = causal && Sq < kv_len ? Sq : kv_len;
  const int n = (int)((keys + (int64_t)64 * per - 1) / ((int64_t)64 * per));
  if (!causal) return nq * n;
  const double sum_c = 0.5 * n * (n - 1.0);
  const double skipped = rows == 128 ? 0.5 * (per * sum_c - (per % 2 != 0 ? n / 2 : 0)) : 64 / rows * (per * sum_c);
  return nq * n - skipped;
}

int chunks_of(int q0, int rows, int Sq, int kv_len, int chunk, bool causal) {
  return causal ? pf::key_chunks<true>(q0, rows, Sq, kv_len, chunk) : pf::key_chunks<false>(q0, rows, Sq, kv_len, chunk);
}

// The forward's key split: chunk and n_split of `p`, and its workspace bytes
// (0: whole items).
size_t plan_fwd_split(const pf_attn_fwd_args* a, pf::FwdParams* p) {
  p->n_split = 1;
  p->chunk = 0;
  if (p->n_work == 0 || p->n_work >= 2 * kCus) return 0;
  const int max_keys = a->causal && a->seq_len_q < a->kv_len ? a->seq_len_q : a->kv_len;
  const int max_steps = (max_keys + 63) / 64;
  if (max_steps <= 1) return 0;
  const int64_t rows = (int64_t)a->batch * a->num_heads * a->seq_len_q;
  const int members = p->n_work / p->n_qblk;
  const auto wgs = [&](int per) { return members * key_split_grid(a->seq_len_q, p->rpw, a->kv_len, per, a->causal); };
  const int min_per = a->causal && p->rpw > 64 ? 2 : 1;  // whole multiples of rpw
  const int per = plan_split(p->n_work, max_steps, wgs(1), min_per, step_cost(a->dtype, a->head_dim).fwd,
                             rows * a->head_dim * 4, wgs);
  if (per == 0) return 0;
  p->chunk = per * 64;
  p->split_grid = 0;
  for (int i = 0; i < p->n_qblk; ++i)
    p->split_grid += chunks_of(i * p->rpw, p->rpw, a->seq_len_q, a->kv_len, p->chunk, a->causal) * members;
  p->n_split = (max_steps + per - 1) / per;
  const size_t prow = (size_t)p->n_split * rows;
  return align_ws(prow * a->head_dim * 4) + align_ws(prow * 8);
}

void bind_fwd_split(const pf_attn_fwd_args* a, pf::FwdParams* p, void* ws) {
  const size_t prow = (size_t)p->n_split * a->batch * a->num_heads * a->seq_len_q;
  p->part_o = static_cast<float*>(ws);
  p->part_ml = reinterpret_cast<float*>(static_cast<char*>(ws) + align_ws(prow * a->head_dim * 4));
}

// Minimum items for a dynamic tail: four per CU of a 256-CU MI355X, two per
// resident workgroup where two are resident (the 16-bit forward and dQ; at
// head_dim 64 the forward has three, so 1.33).
constexpr int kTwoPerCu = 2 * 2 * 256;

}  // namespace

extern "C" {

const char* pf_version(void) { return "pallas_flash_amd 0.1.0 (gfx950)"; }

int pf_get_tuning(pf_tuning* out) {
  if (!out) return PF_ERR_INVALID;
  Tuning& t = tuning();
  out->tail_dynamic_pct = t.tail_dynamic_pct.load();
  out->decode_stages = t.decode_stages.load();
  out->decode_waves = t.decode_waves.load();
  return PF_OK;
}

int pf_set_tuning(const pf_tuning* in) {
  if (!in || !tuning_valid(in->tail_dynamic_pct, in->decode_stages, in->decode_waves))
    return PF_ERR_INVALID;
  Tuning& t = tuning();
  t.tail_dynamic_pct = in->tail_dynamic_pct;
  t.decode_stages = in->decode_stages;
  t.decode_waves = in->decode_waves;
  return PF_OK;
}

int pf_attn_fwd(const pf_attn_fwd_args* a, void* stream) {
  if (!a) return PF_ERR_INVALID;
  pf::FwdParams p;
  int st = fill_fwd(a, &p);
  if (st != PF_OK) return st;
  if (p.n_work == 0) return PF_OK;
  p.tail = plan_tail(p.n_work, kTwoPerCu, (hipStream_t)stream);
  return finish(pf::launch_attn_fwd(p, a->dtype, a->head_dim, a->causal != 0, false,
                                    (hipStream_t)stream));
}

size_t pf_attn_fwd_workspace_size(const pf_attn_fwd_args* a) {
  pf::FwdParams p;
  if (!a || fill_fwd(a, &p) != PF_OK) return 0;
  return plan_fwd_split(a, &p);
}

int pf_attn_fwd_ws(const pf_attn_fwd_args* a, void* workspace, size_t workspace_bytes, void* stream) {
  if (!a) return PF_ERR_INVALID;
  pf::FwdParams p;
  int st = fill_fwd(a, &p);
  if (st != PF_OK) return st;
  if (p.n_work == 0) return PF_OK;
  const size_t need = plan_fwd_split(a, &p);
  if (need == 0) return pf_attn_fwd(a, stream);
  if (!workspace || workspace_bytes < need || ((uintptr_t)workspace & 255) != 0) return PF_ERR_WORKSPACE;
  bind_fwd_split(a, &p, workspace);
  return finish(pf::launch_attn_fwd(p, a->dtype, a->head_dim, a->causal != 0, false, (hipStream_t)stream));
}

static size_t rope_ws_bytes(const pf_attn_fwd_args& b) {
  const size_t es = b.dtype == PF_DTYPE_F32 ? 4 : 2;
  return (((size_t)b.batch * b.num_kv_heads * b.seq_len_k * b.head_dim * es) + 255) & ~(size_t)255;
}

size_t pf_attn_fwd_rope_workspace_size(const pf_attn_fwd_rope_args* a) {
  if (!a) return 0;
  pf::FwdParams p;
  if (fill_fwd(&a->base, &p) != PF_OK) return 0;
  return rope_ws_bytes(a->base) + plan_fwd_split(&a->base, &p);
}

int pf_attn_fwd_rope(const pf_attn_fwd_rope_args* a, void* stream) {
  if (!a) return PF_ERR_INVALID;
  pf::FwdParams p;
  int st = fill_fwd(&a->base, &p);
  if (st != PF_OK) return st;
  if (!a->q_cos || !a->q_sin || !a->k_cos || !a->k_sin) return PF_ERR_INVALID;
  if (a->base.head_dim % 2 != 0) return PF_ERR_INVALID;  // fused_rope.py:168-169
  if (p.n_work == 0) return PF_OK;
  const size_t need = rope_ws_bytes(a->base);
  if (!a->workspace || a->workspace_bytes < need || ((uintptr_t)a->workspace & 255) != 0)
    return PF_ERR_WORKSPACE;
  hipStream_t s = (hipStream_t)stream;
  st = finish(pf::launch_rope_rotate_k(a->base.k, a->workspace, a->k_cos, a->k_sin, a->base.batch,
                                       a->base.num_kv_heads, a->base.seq_len_k, a->base.kv_len,
                                       a->base.dtype, a->base.head_dim, s));
  if (st != PF_OK) return st;
  p.k = a->workspace;  // rotated K
  p.q_cos = a->q_cos;
  p.q_sin = a->q_sin;
  p.lse = nullptr;  // the reference's fused kernel has no LSE output
  // A workspace of the rotated K alone (a caller that sized it itself) runs
  // whole items.
  if (plan_fwd_split(&a->base, &p) > a->workspace_bytes - need) p.n_split = 1;
  if (p.n_split > 1) bind_fwd_split(&a->base, &p, static_cast<char*>(a->workspace) + need);
  else p.tail = plan_tail(p.n_work, kTwoPerCu, s);
  return finish(pf::launch_attn_fwd(p, a->base.dtype, a->base.head_dim, a->base.causal != 0, true, s));
}

// ---------------------------------------------------------------------------
// Backward
// ---------------------------------------------------------------------------
static int fill_bwd(const pf_attn_bwd_args* a, pf::BwdParams* p, bool need_grads) {
  if (!a) return PF_ERR_INVALID;
  int st = check_attn_dims(a->batch, a->num_heads, a->num_kv_heads, a->seq_len_q, a->seq_len_k,
                           a->head_dim, a->kv_len, a->sm_scale, a->dtype);
  if (st != PF_OK) return st;
  if (!a->o || !a->do_ || !a->delta) return PF_ERR_INVALID;
  if (need_grads && (!a->q || !a->k || !a->v || !a->lse || !a->dq || !a->dk || !a->dv))
    return PF_ERR_INVALID;
  p->q = a->q;
  p->k = a->k;
  p->v = a->v;
  p->o = a->o;
  p->dout = a->do_;
  p->lse = a->lse;
  p->delta = a->delta;
  p->dq = a->dq;
  p->dk = a->dk;
  p->dv = a->dv;
  p->B = a->batch;
  p->Hq = a->num_heads;
  p->Hkv = a->num_kv_heads;
  p->Sq = a->seq_len_q;
  p->Sk = a->seq_len_k;
  p->kv_len = a->kv_len;
  p->g = a->num_heads / a->num_kv_heads;
  p->sm_scale = a->sm_scale;
  p->scale_log2 = a->sm_scale * 1.4426950408889634f;
  p->tail = pf::WorkTail{nullptr, 0, 0};
  p->n_split_q = p->n_split_k = 1;
  p->chunk_q = p->grid_q = p->steps_k = p->grid_k = 0;
  p->part_dq = p->part_dk = p->part_dv = nullptr;
  const int64_t rows = (int64_t)a->batch * a->num_heads * a->seq_len_q;
  if (rows > kMaxGrid) return PF_ERR_UNSUPPORTED;
  // Per-(batch, head) byte offsets and buffer sizes are 32-bit inside the
  // kernels (Q/dO rows of one query head, K/V rows of one kv head), as in
  // the forward.
  const int64_t max_rows = a->seq_len_q > a->seq_len_k ? a->seq_len_q : a->seq_len_k;
  if ((max_rows + 256) * a->head_dim * 4 > 0x7fffffff) return PF_ERR_UNSUPPORTED;
  return PF_OK;
}

int pf_attn_bwd_delta(const pf_attn_bwd_args* a, void* stream) {
  pf::BwdParams p;
  int st = fill_bwd(a, &p, false);
  if (st != PF_OK) return st;
  if ((int64_t)p.B * p.Hq * p.Sq == 0) return PF_OK;
  return finish(pf::launch_attn_bwd_delta(p, a->dtype, a->head_dim, (hipStream_t)stream));
}

int pf_attn_bwd_dq(const pf_attn_bwd_args* a, void* stream) {
  pf::BwdParams p;
  int st = fill_bwd(a, &p, true);
  if (st != PF_OK) return st;
  if ((int64_t)p.B * p.Hq * p.Sq == 0) return PF_OK;
  p.tail = plan_tail(pf::bwd_dq_items(p), kTwoPerCu, (hipStream_t)stream);
  return finish(pf::launch_attn_bwd_dq(p, a->dtype, a->head_dim, a->causal != 0, (hipStream_t)stream));
}

int pf_attn_bwd_dkv(const pf_attn_bwd_args* a, void* stream) {
  pf::BwdParams p;
  int st = fill_bwd(a, &p, true);
  if (st != PF_OK) return st;
  if ((int64_t)p.B * p.Hkv * p.Sk == 0) return PF_OK;
  return finish(pf::launch_attn_bwd_dkv(p, a->dtype, a->head_dim, a->causal != 0, (hipStream_t)stream));
}

// The backward's splits and their workspace: part_dq, part_dk, part_dv.
static size_t plan_bwd_split(const pf_attn_bwd_args* a, pf::BwdParams* p, size_t* dq_bytes, size_t* dkv_bytes) {
  *dq_bytes = *dkv_bytes = 0;
  const StepCost cost = step_cost(a->dtype, a->head_dim);
  const int64_t rows_q = (int64_t)p->B * p->Hq * p->Sq, rows_k = (int64_t)p->B * p->Hkv * p->Sk;
  if (rows_q == 0 || rows_k == 0) return 0;
  const bool causal = a->causal != 0;
  const int max_keys = causal && p->Sq < p->kv_len ? p->Sq : p->kv_len;
  const int kb = (max_keys + 63) / 64;
  const int64_t dq_items = (int64_t)p->B * p->Hq * ((p->Sq + 127) / 128);
  if (kb > 1 && dq_items < 2 * kCus) {
    const auto wgs = [&](int per) { return (double)p->B * p->Hq * key_split_grid(p->Sq, 128, p->kv_len, per, causal); };
    const int per = plan_split(dq_items, kb, wgs(1), 1, cost.dq, rows_q * a->head_dim * 4, wgs);
    if (per > 0) {
      p->chunk_q = per * 64;
      p->grid_q = 0;
      for (int q0 = 0; q0 < p->Sq; q0 += 128)
        p->grid_q += chunks_of(q0, 128, p->Sq, p->kv_len, p->chunk_q, causal) * p->B * p->Hq;
      p->n_split_q = (kb + per - 1) / per;
      *dq_bytes = align_ws((size_t)p->n_split_q * rows_q * a->head_dim * 4);
    }
  }
  const int bmq = a->dtype != PF_DTYPE_F32 && a->head_dim <= 128 ? 128 : 64;
  const int halves = a->head_dim > 128 ? 2 : 1;
  const int64_t nk = (p->Sk + 127) / 128, items = (int64_t)p->B * p->Hkv * nk;
  if (items * halves < 2 * kCus) {
    const int64_t max_steps = (int64_t)((p->Sq + bmq - 1) / bmq) * p->g;
    if (max_steps <= 0x7fffffff) {
      // As key_split_grid, over key blocks: block i < busy has (nqb - r i) g steps
      // (not causal: nqb g), the others none, and every block at least one run.
      const int64_t nqb = (p->Sq + bmq - 1) / bmq, r = 128 / bmq, members = (int64_t)p->B * p->Hkv * halves;
      const int64_t busy = ((causal && p->Sq < p->kv_len ? p->Sq : p->kv_len) + 127) / 128;
      const double total = (double)p->g * (busy * nqb - (causal ? r * (busy * (busy - 1) / 2) : 0));
      const auto wgs = [&](int per) {
        int64_t n = nk - busy;
        if (!causal) n += busy * ((max_steps + per - 1) / per);
        for (int64_t c = 0; causal && c < max_steps; c += per)  // run c / per: the blocks with more than c steps
          n += std::min(busy, (nqb - 1 - c / p->g) / r + 1);
        return (double)(n * members);
      };
      const int per = plan_split(items * halves, (int)max_steps, total * members, 1, cost.dkv,
                                 2 * rows_k * a->head_dim * 4, wgs);
      p->steps_k = per;
      if (per > 0) {
        p->grid_k = 0;
        for (int64_t i = 0; i < nk; ++i) p->grid_k += pf::dkv_runs(*p, (int)(128 * i), bmq, causal) * p->B * p->Hkv;
        p->n_split_k = (int)((max_steps + per - 1) / per);
        *dkv_bytes = align_ws((size_t)p->n_split_k * rows_k * a->head_dim * 4);
      }
    }
  }
  return *dq_bytes + 2 * *dkv_bytes;
}

size_t pf_attn_bwd_workspace_size(const pf_attn_bwd_args* a) {
  pf::BwdParams p;
  if (fill_bwd(a, &p, true) != PF_OK) return 0;
  size_t dq, dkv;
  return plan_bwd_split(a, &p, &dq, &dkv);
}

int pf_attn_bwd_ws(const pf_attn_bwd_args* a, void* workspace, size_t workspace_bytes, void* stream) {
  pf::BwdParams p;
  int st = fill_bwd(a, &p, true);
  if (st != PF_OK) return st;
  size_t dq, dkv;
  const size_t need = plan_bwd_split(a, &p, &dq, &dkv);
  if (need == 0) return pf_attn_bwd(a, stream);
  if (!workspace || workspace_bytes < need || ((uintptr_t)workspace & 255) != 0) return PF_ERR_WORKSPACE;
  char* ws = static_cast<char*>(workspace);
  p.part_dq = reinterpret_cast<float*>(ws);
  p.part_dk = reinterpret_cast<float*>(ws + dq);
  p.part_dv = reinterpret_cast<float*>(ws + dq + dkv);
  hipStream_t s = (hipStream_t)stream;
  if (p.n_split_q <= 1) p.tail = plan_tail(pf::bwd_dq_items(p), kTwoPerCu, s);
  st = finish(pf::launch_attn_bwd_dq(p, a->dtype, a->head_dim, a->causal != 0, s));
  if (st != PF_OK) return st;
  p.tail = pf::WorkTail{nullptr, 0, 0};
  st = finish(pf::launch_attn_bwd_dkv(p, a->dtype, a->head_dim, a->causal != 0, s));
  if (st != PF_OK) return st;
  return finish(pf::launch_attn_bwd_reduce(p, a->dtype, a->head_dim, a->causal != 0, s));
}

int pf_attn_bwd(const pf_attn_bwd_args* a, void* stream) {
  pf::BwdParams p;
  int st = fill_bwd(a, &p, true);
  if (st != PF_OK) return st;
  hipStream_t s = (hipStream_t)stream;
  if ((int64_t)p.B * p.Hq * p.Sq > 0) {
    // the dQ kernel computes delta itself and stores it for dK/dV
    p.tail = plan_tail(pf::bwd_dq_items(p), kTwoPerCu, s);
    st = finish(pf::launch_attn_bwd_dq(p, a->dtype, a->head_dim, a->causal != 0, s));
    if (st != PF_OK) return st;
  }
  if ((int64_t)p.B * p.Hkv * p.Sk > 0) {
    p.tail = pf::WorkTail{nullptr, 0, 0};  // dK/dV runs without a tail (plan_tail)
    st = finish(pf::launch_attn_bwd_dkv(p, a->dtype, a->head_dim, a->causal != 0, s));
  }
  return st;
}

// ---------------------------------------------------------------------------
// Decode (contiguous cache) and paged decode
// ---------------------------------------------------------------------------
static size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

// Key-chunk size for split-KV: enough (b, kv head, chunk) waves to fill the
// chip several times over (256 CUs x 8 resident waves), chunks a multiple of
// the 64-key block and at least 256 keys so each wave streams a useful run.
constexpr int kMinChunk = 256;
static int64_t decode_splits(int64_t units) {  // the chunks aimed at
  const int64_t target_waves = 4096;
  const int64_t n = (target_waves + units - 1) / (units > 0 ? units : 1);
  return n > 1 ? n : 1;
}
static int decode_chunk(int64_t units, int max_len) {
  const int64_t n_split = decode_splits(units);
  int64_t chunk = (max_len + n_split - 1) / n_split;
  chunk = ((chunk + 63) / 64) * 64;
  if (chunk < kMinChunk) chunk = kMinChunk;
  return (int)chunk;
}

// Streaming kernel (decode_stream.hpp): a persistent grid of one-wave
// workgroups, as many as are resident at once (queried once per device),
// with an LDS ring of 2 stages (measured on MI355X: 2 stages x 4 waves per
// CU beat 3 x 3 and 4 x 2). Tuning and test overrides: decode_stages (2..4,
// of the 16-bit head_dim 128 kernels) and decode_waves (grid size; any value
// >= 1 is correct, only the resident count is fast).
// A short problem starts only as many waves as it has stages (32 keys; 16 in
// float32 at head_dim 128 and with fine stages); at 16-bit head_dim 256 a wave
// takes at least two 16-key stages, which halves the pieces to merge for 0.6 us.
// One stage a wave also cuts equal sequences alike, whatever their place in the
// list. max_len: the most keys a sequence can have.
static int stream_grid(int dtype, int32_t head_dim, int group, bool fine) {
  const int wv = tuning().decode_waves.load(std::memory_order_relaxed);
  if (wv > 0) return wv;
  return pf::decode_stream_waves(dtype, head_dim, tuning().decode_stages.load(std::memory_order_relaxed), group, fine);
}
static int stream_setup(pf::DecodeParams* p, int dtype, int64_t max_len) {
  const int group = p->Hq / p->Hkv;
  p->stages = tuning().decode_stages.load(std::memory_order_relaxed);
  p->fixed_grid = tuning().decode_waves.load(std::memory_order_relaxed) > 0;
  // Float32 at head_dim 64: a stage is 0.9 us of float32 MFMAs, so with a few
  // stages a wave half as long ones, on twice as many waves (8 a CU), divide
  // more evenly and hide each other's loads: 16 x 4 sequences of 64-2048 keys
  // 16.0 -> 14.8 us, 8 x 8 of 1672 17.1 -> 14.7; past 32 stages a wave (by the
  // longest lengths) nothing is left to gain and 190 a wave lose 2%. Where each
  // 32-key stage has a wave of its own they only double the pieces to merge
  // (8 sequences of 2447 keys 10.4 -> 11.5 us). Sequences of up to 12 stages
  // have a form of their own.
  const int64_t seqs = (int64_t)p->B * p->Hkv * ((group + 15) / 16);
  const int64_t stages32 = seqs * ((max_len + 31) / 32);
  const bool f32 = dtype == PF_DTYPE_F32, can_fine = f32 && p->D == 64;
  p->fine = can_fine && max_len > 12 * 32 && stages32 > 4 * kCus && stages32 <= 32 * 4 * kCus;
  const int sk = p->D * (f32 ? 4 : 2) == 512 || p->fine ? 16 : 32;  // keys per stage
  const int unit = f32 ? sk : 32;
  const int64_t runs = seqs * ((max_len + unit - 1) / unit);
  const int grid = p->full_waves = stream_grid(dtype, p->D, group, p->fine != 0);
  p->n_waves = grid > runs ? (int)(runs > 1 ? runs : 1) : grid;
  p->n_split = 0;
  p->chunk = 0;
  p->g = group;
  if (p->block_tables == nullptr && p->positions == nullptr && p->context_lens == nullptr) {
    const int64_t stages = seqs * ((max_len + sk - 1) / sk);
    p->part_q = stages / p->n_waves;
    p->part_rem = stages % p->n_waves;
  }
  return p->n_waves;
}

// Whether the streaming kernel's 32-bit byte offsets reach every row of a run
// of `rows` rows (a cache slot range or a page).
static bool stream_range_ok(int64_t rows, int32_t head_dim, int32_t dtype) {
  return rows * head_dim * (dtype == PF_DTYPE_F32 ? 4 : 2) < ((int64_t)1 << 31);
}
// Its LDS loads want 16-byte aligned rows; the generic kernel reads any.
static bool stream_aligned(const void* q, const void* k, const void* v) {
  return (((uintptr_t)q | (uintptr_t)k | (uintptr_t)v) & 15) == 0;
}
// Forms with one workspace size, whatever the batch and the cache; past the
// streaming kernel's range they are refused, where the others run the generic
// kernel. Unaligned operands run it in either case.
static bool stream_only(int32_t head_dim, int32_t dtype) { return head_dim == 128 && dtype != PF_DTYPE_F32; }
// Partial slots of that one size: two pieces for every wave of a full grid, and
// at least a batch's heads, for the generic kernel.
static int64_t stream_room(const pf::DecodeParams& p, int dtype) {
  const int group = p.Hq / p.Hkv;
  const int grid = p.full_waves > 0 ? p.full_waves : stream_grid(dtype, p.D, group, false);
  return std::max((int64_t)2 * grid * pf::decode_stream_qrows(group), (int64_t)p.Hq);
}

// The generic kernel's chunks of up to max_len keys. room > 0: no more partials
// than that, by fewer chunks and, past one chunk, by batches (p->slice) whose
// launches follow each other on the stream.
static int generic_setup(pf::DecodeParams* p, int64_t max_len, int64_t room) {
  const int64_t per_batch = (int64_t)p->Hkv * ((p->Hq / p->Hkv + 31) / 32);
  p->n_waves = 0;
  p->slice = p->B;
  if (room > 0) p->slice = (int)std::min((int64_t)p->B, room / p->Hq);
  p->chunk = decode_chunk(per_batch * p->slice, (int)max_len);
  if (room > 0 && p->slice > 0) {
    const int64_t n = room / ((int64_t)p->slice * p->Hq);
    p->chunk = (int)std::max((int64_t)p->chunk, ((max_len + n - 1) / n + 63) / 64 * 64);
  }
  p->n_split = (int)((max_len + p->chunk - 1) / p->chunk);
  return per_batch * p->slice * p->n_split > kMaxGrid ? PF_ERR_UNSUPPORTED : PF_OK;
}

// *streams: whether the call's shape is one of the streaming kernel's.
static int fill_decode(const pf_attn_decode_args* a, pf::DecodeParams* p, bool* streams) {
  if (!a) return PF_ERR_INVALID;
  if (a->batch < 0 || a->num_heads < 1 || a->num_kv_heads < 1 || a->cache_size < 1)
    return PF_ERR_INVALID;
  if (a->num_heads % a->num_kv_heads != 0) return PF_ERR_INVALID;
  if (a->cache_len < 1 || a->cache_len > a->cache_size) return PF_ERR_INVALID;
  if (!isfinite(a->sm_scale)) return PF_ERR_INVALID;
  if (!dtype_ok(a->dtype)) return PF_ERR_UNSUPPORTED;
  if (!decode_head_dim_ok(a->head_dim, a->dtype)) return PF_ERR_UNSUPPORTED;
  const int g = a->num_heads / a->num_kv_heads;
  *p = pf::DecodeParams{};
  p->q = a->q;
  p->k = a->k_cache;
  p->v = a->v_cache;
  p->o = a->o;
  p->B = a->batch;
  p->Hq = a->num_heads;
  p->Hkv = a->num_kv_heads;
  p->D = decode_compute_dim(a->head_dim);
  p->dr = a->head_dim;
  p->cache_size = a->cache_size;
  p->cache_len = a->cache_len;
  p->scale_log2 = a->sm_scale * 1.4426950408889634f;
  *streams = false;
  const bool only = stream_only(a->head_dim, a->dtype);
  if (pf::decode_stream_supported(a->dtype, a->head_dim, g, false, 0)) {
    // buffer offsets within one (b, kv head) run are 32-bit
    *streams = stream_range_ok(a->cache_size, a->head_dim, a->dtype);
    if (*streams && stream_aligned(a->q, a->k_cache, a->v_cache))
      return stream_setup(p, a->dtype, a->cache_len) > 0 ? PF_OK : PF_ERR_LAUNCH;
    if (!*streams && only) return PF_ERR_UNSUPPORTED;
  }
  return generic_setup(p, a->cache_len, *streams && only ? stream_room(*p, a->dtype) : 0);
}

// The bytes of `slots` partials (max, sum and D accumulators each).
static size_t partial_bytes(size_t slots, int D) {
  return align256(slots * D * sizeof(float)) + align256(slots * 2 * sizeof(float));
}

// Partial slots of a launch: streaming kernel one per piece (piece_slot) x
// query rows -- at most one piece that a wave opens with and one that it ends
// with --, generic kernel one per (b, query head, chunk).
static size_t decode_slots(const pf::DecodeParams& p) {
  if (p.n_waves == 0) return (size_t)p.slice * p.Hq * p.n_split;
  const int group = p.Hq / p.Hkv;
  const int64_t seqs = (int64_t)p.B * p.Hkv * ((group + 15) / 16);
  return (size_t)(p.n_waves + (seqs < p.n_waves ? seqs : p.n_waves)) * pf::decode_stream_qrows(group);
}

// What the size queries answer: enough for the same call with any cache length
// up to `cap` keys and wherever its operands lie, and for the streaming forms
// whatever the batch -- a program asks once and keeps the workspace while its
// sequences grow. So it counts two pieces for every wave of a full streaming
// grid, and the chunks that generic_setup makes without a bound.
static size_t decode_ws_most(const pf::DecodeParams& p, int dtype, bool streams, int64_t cap) {
  const int group = p.Hq / p.Hkv;
  size_t most = 0;
  if (streams && stream_only(p.dr, dtype)) return partial_bytes(stream_room(p, dtype), p.D);
  if (streams) {
    int waves = stream_grid(dtype, p.D, group, false);
    if (dtype == PF_DTYPE_F32 && p.D == 64) waves = std::max(waves, stream_grid(dtype, p.D, group, true));
    most = partial_bytes((size_t)2 * waves * pf::decode_stream_qrows(group), p.D);
  }
  // decode_chunk's chunks have at least kMinChunk keys and at least cap / splits.
  const int64_t units = (int64_t)p.B * p.Hkv * ((group + 31) / 32);
  int64_t n = std::min(decode_splits(units), (cap + kMinChunk - 1) / kMinChunk);
  if (n < 1) n = 1;
  return std::max(most, partial_bytes((size_t)p.B * p.Hq * n, p.D));
}

// The bytes that a launch insists on: what it uses; the 16-bit head_dim 128
// forms the full size that their query answers.
static size_t decode_ws_bytes(const pf::DecodeParams& p, int dtype, bool streams) {
  if (streams && stream_only(p.dr, dtype)) return decode_ws_most(p, dtype, true, 0);
  return partial_bytes(decode_slots(p), p.D);
}

static int bind_workspace(pf::DecodeParams* p, int dtype, bool streams, void* ws, size_t bytes) {
  const size_t need = decode_ws_bytes(*p, dtype, streams);
  if (need == 0) return PF_OK;
  if (!ws || bytes < need || ((uintptr_t)ws & 255) != 0) return PF_ERR_WORKSPACE;
  const size_t slots = decode_slots(*p);
  p->part_o = static_cast<float*>(ws);
  p->part_ml = reinterpret_cast<float*>(static_cast<char*>(ws) + align256(slots * p->D * sizeof(float)));
  return PF_OK;
}

// The launch: all of it, or the generic kernel slice after slice.
static int run_decode(const pf::DecodeParams& p, int dtype, bool paged, hipStream_t stream) {
  if (p.n_waves > 0 || p.slice >= p.B) return finish(pf::launch_decode(p, dtype, paged, stream));
  const int64_t es = dtype == PF_DTYPE_F32 ? 4 : 2;
  const int64_t q_bytes = (int64_t)p.Hq * p.dr * es, kv_bytes = paged ? 0 : (int64_t)p.Hkv * p.cache_size * p.dr * es;
  int st = PF_OK;
  for (int b = 0; b < p.B && st == PF_OK; b += p.slice) {
    pf::DecodeParams s = p;
    s.B = std::min(p.slice, p.B - b);
    s.q = static_cast<const char*>(p.q) + b * q_bytes;
    s.o = static_cast<char*>(p.o) + b * q_bytes;
    s.k = static_cast<const char*>(p.k) + b * kv_bytes;
    s.v = static_cast<const char*>(p.v) + b * kv_bytes;
    if (paged) {
      s.context_lens = p.context_lens + b;
      if (p.block_tables != nullptr) s.block_tables = p.block_tables + (int64_t)b * p.pages_per_seq;
    }
    st = finish(pf::launch_decode(s, dtype, paged, stream));
  }
  return st;
}

size_t pf_attn_decode_workspace_size(const pf_attn_decode_args* a) {
  pf::DecodeParams p;
  bool streams;
  if (fill_decode(a, &p, &streams) != PF_OK) return 0;
  return decode_ws_most(p, a->dtype, streams, a->cache_size);
}

size_t pf_attn_decode_workspace_min(const pf_attn_decode_args* a) {
  pf::DecodeParams p;
  bool streams;
  if (fill_decode(a, &p, &streams) != PF_OK) return 0;
  return decode_ws_bytes(p, a->dtype, streams);
}

int pf_attn_decode(const pf_attn_decode_args* a, void* stream) {
  pf::DecodeParams p;
  bool streams;
  int st = fill_decode(a, &p, &streams);
  if (st != PF_OK) return st;
  if (!a->q || !a->k_cache || !a->v_cache || !a->o) return PF_ERR_INVALID;
  if (a->batch == 0) return PF_OK;
  st = bind_workspace(&p, a->dtype, streams, a->workspace, a->workspace_bytes);
  if (st != PF_OK) return st;
  return run_decode(p, a->dtype, false, (hipStream_t)stream);
}

// most_ws: the partials' room, where it cannot grow (the streaming grid can be
// set by hand to more waves than fit; the generic kernel then runs).
static int fill_paged(const pf_paged_attn_args* a, pf::DecodeParams* p, bool* streams, size_t most_ws) {
  if (!a) return PF_ERR_INVALID;
  // paged.py:129-149: Sq == 1 (implied by the struct), heads divisible, table [B, P], lens [B].
  if (a->batch < 0 || a->num_heads < 1 || a->num_kv_heads < 1 || a->num_pages < 1 ||
      a->page_size < 1 || a->pages_per_seq < 0)
    return PF_ERR_INVALID;
  if (a->num_heads % a->num_kv_heads != 0) return PF_ERR_INVALID;
  if (!isfinite(a->sm_scale)) return PF_ERR_INVALID;
  if (!dtype_ok(a->dtype)) return PF_ERR_UNSUPPORTED;
  if (!decode_head_dim_ok(a->head_dim, a->dtype)) return PF_ERR_UNSUPPORTED;
  const int64_t max_len = (int64_t)a->pages_per_seq * a->page_size;
  if (max_len > 0x7fffffff) return PF_ERR_UNSUPPORTED;
  const int g = a->num_heads / a->num_kv_heads;
  *p = pf::DecodeParams{};
  p->q = a->q;
  p->k = a->k_pages;
  p->v = a->v_pages;
  p->o = a->o;
  p->block_tables = a->block_tables;
  p->context_lens = a->context_lens;
  p->B = a->batch;
  p->Hq = a->num_heads;
  p->Hkv = a->num_kv_heads;
  p->D = decode_compute_dim(a->head_dim);
  p->dr = a->head_dim;
  p->num_pages = a->num_pages;
  p->page_size = a->page_size;
  p->pages_per_seq = a->pages_per_seq;
  p->scale_log2 = a->sm_scale * 1.4426950408889634f;
  *streams = false;
  const bool only = stream_only(a->head_dim, a->dtype);
  if (pf::decode_stream_supported(a->dtype, a->head_dim, g, true, a->page_size)) {
    *streams = stream_range_ok(a->page_size, a->head_dim, a->dtype);
    if (*streams && stream_aligned(a->q, a->k_pages, a->v_pages)) {
      if (stream_setup(p, a->dtype, max_len) <= 0) return PF_ERR_LAUNCH;
      if (only || decode_ws_bytes(*p, a->dtype, *streams) <= most_ws) return PF_OK;
    }
    if (!*streams && only) return PF_ERR_UNSUPPORTED;
  }
  return generic_setup(p, max_len > 0 ? max_len : 1, *streams && only ? stream_room(*p, a->dtype) : 0);
}

size_t pf_paged_attn_workspace_size(const pf_paged_attn_args* a) {
  pf::DecodeParams p;
  bool streams;
  if (fill_paged(a, &p, &streams, SIZE_MAX) != PF_OK) return 0;
  return decode_ws_most(p, a->dtype, streams, (int64_t)a->pages_per_seq * a->page_size);
}

size_t pf_paged_attn_workspace_min(const pf_paged_attn_args* a) {
  pf::DecodeParams p;
  bool streams;
  if (fill_paged(a, &p, &streams, SIZE_MAX) != PF_OK) return 0;
  return decode_ws_bytes(p, a->dtype, streams);
}

int pf_paged_attn(const pf_paged_attn_args* a, void* stream) {
  pf::DecodeParams p;
  bool streams;
  int st = fill_paged(a, &p, &streams, SIZE_MAX);
  if (st != PF_OK) return st;
  if (!a->q || !a->k_pages || !a->v_pages || !a->o || !a->context_lens) return PF_ERR_INVALID;
  if (a->pages_per_seq > 0 && !a->block_tables) return PF_ERR_INVALID;
  if (a->batch == 0) return PF_OK;
  st = bind_workspace(&p, a->dtype, streams, a->workspace, a->workspace_bytes);
  if (st != PF_OK) return st;
  return run_decode(p, a->dtype, true, (hipStream_t)stream);
}

}  // extern "C"

// ---------------------------------------------------------------------------
// Paged decode with no caller workspace (pf_paged_attn_noalloc): the split-KV
// partials live in `scratch`, a file-scope device array that every GPU holds
// once, for the life of the process. On the host `scratch` names a host-side
// stand-in, not device memory: its device address is looked up once per
// device (hipGetSymbolAddress, with that device current) and only that
// address is handed to the kernels. Every call on one GPU shares the array;
// nothing in it needs clearing between calls (each launch writes every
// partial slot its combine step reads), and calls that overlap on one GPU
// (concurrent streams) race on it.
// ---------------------------------------------------------------------------
namespace {

static_assert(PF_NOALLOC_SCRATCH_BYTES % 256 == 0, "scratch keeps the workspace alignment");
static __device__ __align__(256) char scratch[PF_NOALLOC_SCRATCH_BYTES];

constexpr int kMaxScratchDevices = 64;

struct ScratchAddr {
  std::once_flag once;
  void* ptr = nullptr;
  hipError_t err = hipErrorNotInitialized;
};
ScratchAddr g_scratch[kMaxScratchDevices];

// Device address of `scratch` on the device that `stream` belongs to (the
// null stream's: the current device), resolved on the first call on each
// device (symbol_address, with that device current, also under graph
// capture).
int scratch_address(hipStream_t stream, void** out) {
  int dev = -1;
  if (hipStreamGetDevice(stream, &dev) != hipSuccess || dev < 0 || dev >= kMaxScratchDevices)
    return PF_ERR_LAUNCH;
  ScratchAddr& s = g_scratch[dev];
  std::call_once(s.once, [&s, dev] { s.err = pf::symbol_address(dev, HIP_SYMBOL(scratch), &s.ptr); });
  if (s.err != hipSuccess || s.ptr == nullptr) return PF_ERR_LAUNCH;
  *out = s.ptr;
  return PF_OK;
}

}  // namespace

extern "C" {

int pf_paged_attn_noalloc(const pf_paged_attn_args* a, void* stream) {
  pf::DecodeParams p;
  bool streams;
  int st = fill_paged(a, &p, &streams, PF_NOALLOC_SCRATCH_BYTES);
  if (st != PF_OK) return st;
  if (!a->q || !a->k_pages || !a->v_pages || !a->o || !a->context_lens) return PF_ERR_INVALID;
  if (a->pages_per_seq > 0 && !a->block_tables) return PF_ERR_INVALID;
  if (a->batch == 0) return PF_OK;
  if (decode_ws_bytes(p, a->dtype, streams) > (size_t)PF_NOALLOC_SCRATCH_BYTES) return PF_ERR_WORKSPACE;
  void* ws = nullptr;
  st = scratch_address((hipStream_t)stream, &ws);
  if (st != PF_OK) return st;
  st = bind_workspace(&p, a->dtype, streams, ws, PF_NOALLOC_SCRATCH_BYTES);
  if (st != PF_OK) return st;
  return run_decode(p, a->dtype, true, (hipStream_t)stream);
}

int pf_rope(const pf_rope_args* a, void* stream) {
  if (!a) return PF_ERR_INVALID;
  if (a->batch < 0 || a->heads < 0 || a->seq_len < 0 || a->head_dim < 2 || a->head_dim % 2 != 0)
    return PF_ERR_INVALID;
  if (a->inverse != 0 && a->inverse != 1) return PF_ERR_INVALID;
  if (!dtype_ok(a->dtype)) return PF_ERR_UNSUPPORTED;
  if (!head_dim_ok(a->head_dim, a->dtype)) return PF_ERR_UNSUPPORTED;
  if ((int64_t)a->batch * a->heads * a->seq_len == 0) return PF_OK;
  if (!a->x || !a->out || !a->cos || !a->sin || a->rope_len < a->seq_len) return PF_ERR_INVALID;
  return finish(pf::launch_rope_rotate_k(a->x, a->out, a->cos, a->sin, a->batch, a->heads, a->seq_len,
                                         a->seq_len, a->dtype, a->head_dim, (hipStream_t)stream,
                                         a->inverse != 0));
}

// ---------------------------------------------------------------------------
// Cache writes and the fused decode step
// ---------------------------------------------------------------------------
int pf_kv_cache_write(const pf_kv_cache_write_args* a, void* stream) {
  if (!a) return PF_ERR_INVALID;
  if (a->batch < 0 || a->num_kv_heads < 1 || a->seq_len < 0 || a->cache_size < 1) return PF_ERR_INVALID;
  if (a->positions_stride != 0 && a->positions_stride != 1) return PF_ERR_INVALID;
  if (a->ring != 0 && a->ring != 1) return PF_ERR_INVALID;
  if (!dtype_ok(a->dtype)) return PF_ERR_UNSUPPORTED;
  if (!decode_head_dim_ok(a->head_dim, a->dtype)) return PF_ERR_UNSUPPORTED;
  if ((int64_t)a->batch * a->num_kv_heads * a->seq_len == 0) return PF_OK;
  if (!a->k || !a->v || !a->k_cache || !a->v_cache || !a->positions) return PF_ERR_INVALID;
  pf::KvWriteParams p{a->k, a->v, a->k_cache, a->v_cache, a->positions, a->positions_stride,
                      a->batch, a->num_kv_heads, a->seq_len, a->cache_size, a->ring, a->head_dim};
  return finish(pf::launch_kv_cache_write(p, a->dtype, a->head_dim, (hipStream_t)stream));
}

int pf_paged_cache_write(const pf_paged_cache_write_args* a, void* stream) {
  if (!a) return PF_ERR_INVALID;
  if (a->batch < 0 || a->num_kv_heads < 1 || a->seq_len < 0 || a->num_pages < 1 || a->page_size < 1 ||
      a->pages_per_seq < 0)
    return PF_ERR_INVALID;
  if (a->positions_stride != 0 && a->positions_stride != 1) return PF_ERR_INVALID;
  if (!dtype_ok(a->dtype)) return PF_ERR_UNSUPPORTED;
  if (!decode_head_dim_ok(a->head_dim, a->dtype)) return PF_ERR_UNSUPPORTED;
  if ((int64_t)a->batch * a->num_kv_heads * a->seq_len == 0 || a->pages_per_seq == 0) return PF_OK;
  if (!a->k || !a->v || !a->k_pages || !a->v_pages || !a->positions || !a->block_tables) return PF_ERR_INVALID;
  pf::PagedWriteParams p{a->k, a->v, a->k_pages, a->v_pages, a->block_tables, a->positions,
                         a->positions_stride, a->batch, a->num_kv_heads, a->seq_len, a->num_pages,
                         a->page_size, a->pages_per_seq, a->head_dim};
  return finish(pf::launch_paged_cache_write(p, a->dtype, a->head_dim, (hipStream_t)stream));
}

// The fused decode step is one streaming-decode launch in its step mode
// (decode_stream.hip, PG == 1) plus the combine; its workspace is the split
// partials only.
static int fill_decode_step(const pf_attn_decode_step_args* a, pf::DecodeParams* p) {
  if (!a) return PF_ERR_INVALID;
  if (a->batch < 0 || a->num_heads < 1 || a->num_kv_heads < 1 || a->cache_size < 1) return PF_ERR_INVALID;
  if (a->num_heads % a->num_kv_heads != 0) return PF_ERR_INVALID;
  if (a->positions_stride != 0 && a->positions_stride != 1) return PF_ERR_INVALID;
  if (a->ring != 0 && a->ring != 1) return PF_ERR_INVALID;
  if ((a->cos == nullptr) != (a->sin == nullptr)) return PF_ERR_INVALID;
  if (a->cos != nullptr && a->rope_len < 1) return PF_ERR_INVALID;
  if (!isfinite(a->sm_scale)) return PF_ERR_INVALID;
  if (!dtype_ok(a->dtype)) return PF_ERR_UNSUPPORTED;
  if (!stream_only(a->head_dim, a->dtype)) return PF_ERR_UNSUPPORTED;  // 16-bit head_dim 128
  if (!stream_range_ok(a->cache_size, a->head_dim, a->dtype)) return PF_ERR_UNSUPPORTED;
  *p = pf::DecodeParams{};
  p->q = a->q;
  p->k = a->k_cache;
  p->v = a->v_cache;
  p->o = a->o;
  p->B = a->batch;
  p->Hq = a->num_heads;
  p->Hkv = a->num_kv_heads;
  p->D = decode_compute_dim(a->head_dim);
  p->dr = a->head_dim;
  p->cache_size = a->cache_size;
  p->cache_len = a->cache_size;
  p->scale_log2 = a->sm_scale * 1.4426950408889634f;
  p->positions = a->positions;
  p->pos_stride = a->positions_stride;
  p->ring = a->ring;
  p->rope_cos = a->cos;
  p->rope_sin = a->sin;
  p->rope_len = a->rope_len;
  p->k_new = a->k_new;
  p->v_new = a->v_new;
  p->k_out = a->k_cache;
  p->v_out = a->v_cache;
  if (stream_setup(p, a->dtype, a->cache_size) <= 0) return PF_ERR_LAUNCH;
  return PF_OK;
}

size_t pf_attn_decode_step_workspace_size(const pf_attn_decode_step_args* a) {
  pf::DecodeParams p;
  if (fill_decode_step(a, &p) != PF_OK) return 0;
  return decode_ws_bytes(p, a->dtype, true);
}

int pf_attn_decode_step(const pf_attn_decode_step_args* a, void* stream) {
  pf::DecodeParams p;
  int st = fill_decode_step(a, &p);
  if (st != PF_OK) return st;
  if (a->batch == 0) return PF_OK;
  if (!a->q || !a->k_new || !a->v_new || !a->k_cache || !a->v_cache || !a->o || !a->positions)
    return PF_ERR_INVALID;
  st = bind_workspace(&p, a->dtype, true, a->workspace, a->workspace_bytes);
  if (st != PF_OK) return st;
  if (!stream_aligned(a->q, a->k_cache, a->v_cache)) return PF_ERR_INVALID;
  return finish(pf::launch_decode(p, a->dtype, false, (hipStream_t)stream));
}

}  // extern "C"
