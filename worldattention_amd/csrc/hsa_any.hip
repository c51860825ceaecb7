// One call for the inference forward of any head plan (host code, and the cast kernel of its bf16
// operands): heads in one branch or both, Gini or top-k routing, the low-rank branch (compressing in
// the call or over given coarse keys) or the elu(x)+1 branch, fp32 or bf16 activations, keys pooled
// in the call or held as block sums / means. It runs the entry points that hsa_forward's Python
// orchestration runs, with the same arguments on the same two streams, from one workspace:
//  * linear branch on the caller's side stream when there is a sparse branch to run beside it:
//    compression and dense attention over the compressed keys, or elu1 state and readout;
//  * pooling and routing on the caller's stream, then the block-sparse launches; heads in both
//    branches wait for the side stream first (their epilogue fuses the linear branch's output).
// What it saves is the host's time per call: ~20 allocations, argument structs, stream switches and
// launches from Python took 200-240 us a call, which is what a small call or a cached denoising step
// (whose host work starts after a synchronization) waits for; one crossing 80-100 us. Heads that take
// one branch each in bf16 keep wa_hsa_fwd, which also serves training. The call keeps no state and
// takes no lock.
//
// Reference semantics: wan/modules/hsa/attention.py:153-259 (hsa_attention) with the head modes.
#include <algorithm>

#include "common.h"

namespace {

int64_t align256(int64_t x) { return (x + 255) / 256 * 256; }

// ---------------------------------------------------------------------------------------------
// Contiguous bf16 copies of [B, L, H, D] tensors the attention kernels cannot read in place (fp32, or
// rows that are not 16-byte aligned): up to five tensors (q, k, v, coarse k, coarse v) in one launch,
// 8 channels a thread. Bound by memory: each tensor is read once and half of it written.
// ---------------------------------------------------------------------------------------------
struct CastJob {
  const void* src; int64_t s_sb, s_st, s_sh; int dtype, vec;  // vec: 16-byte aligned rows
  bf16_t* dst;
  int64_t L, first;  // first 8-channel run of the job in the launch
};
struct CastJobs {
  CastJob j[5];
  int n, H, D;
  int64_t total;
};

__global__ void __launch_bounds__(256) cast_blhd_kernel(CastJobs c) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= c.total) return;
  int w = 0;
#pragma unroll
  for (int k = 1; k < 5; ++k)
    if (k < c.n && i >= c.j[k].first) w = k;
  const CastJob& job = c.j[w];
  const int64_t u = i - job.first;
  const int per_row = c.D / 8, c8 = (int)(u % per_row);
  const int64_t r = u / per_row;
  const int h = (int)(r % c.H);
  const int64_t bt = r / c.H, b = bt / job.L, t = bt % job.L;
  const int64_t off = b * job.s_sb + t * job.s_st + (int64_t)h * job.s_sh + 8 * c8;
  bf16x8 y;
  if (job.dtype == WA_F32 && job.vec) {
    const f32x4 a = *(const f32x4*)((const float*)job.src + off), d = *(const f32x4*)((const float*)job.src + off + 4);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      y[e] = (bf16_t)a[e];
      y[e + 4] = (bf16_t)d[e];
    }
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) y[e] = (bf16_t)wa_load_f(job.src, off + e, job.dtype);
  }
  *(bf16x8*)(job.dst + u * 8) = y;
}

// A bf16 tensor as the attention kernels read it.
struct View {
  const void* p;
  int64_t sb, st, sh;
};

struct Plan {
  int64_t nq, nkv, lc, dense_block, rows_only, rows_both, split_only, split_both;
  bool linear_side;  // the linear branch runs beside a sparse branch
  // workspace offsets
  int64_t q, k, v, kc, vc, qp, kp, index, num, thresholds, route, arrivals, lin, bsa_only, bsa_both, dense_only,
      dense_both, elu1, state, zsum, total;
};

bool kernel_ready(const void* p, int64_t sb, int64_t st, int64_t sh, int dtype) {
  return dtype == WA_BF16 && wa_aligned16(p) && sb % 8 == 0 && st % 8 == 0 && sh % 8 == 0;
}

bool lowrank(const wa_hsa_any_args* a) { return a->linear_mode == WA_LINEAR_LOWRANK; }

int64_t coarse_rows(const wa_hsa_any_args* a) {
  if (a->kc) return a->lc;
  const int64_t seg = a->segment_len > 0 ? a->segment_len : a->Lkv;
  int64_t total = 0;
  for (int64_t s = 0; s < a->Lkv; s += seg)
    total += std::min(a->proj_rank, (std::min(seg, a->Lkv - s) + a->block_size - 1) / a->block_size);
  return total;
}

Plan make_plan(const wa_hsa_any_args* a) {
  Plan p{};
  const int64_t bs = a->block_size, D = a->D, es = a->o_dtype == WA_BF16 ? 2 : 4;
  const int64_t n_sparse = a->n_both + a->n_sparse_only, n_linear = a->n_both + a->n_linear_only;
  p.nq = (a->Lq + bs - 1) / bs;
  p.nkv = (a->Lkv + bs - 1) / bs;
  p.rows_only = a->B * a->n_sparse_only * p.nq;
  p.rows_both = a->B * a->n_both * p.nq;
  p.split_only = a->split_visits;
  p.split_both = a->split_both > 0 ? a->split_both : a->split_visits;
  p.linear_side = n_sparse > 0 && n_linear > 0;
  const bool attends = n_sparse > 0 || (n_linear > 0 && lowrank(a));  // some launch reads bf16 q
  int64_t o = 0;
  auto take = [&](int64_t bytes) {
    const int64_t at = o;
    o += align256(bytes);
    return at;
  };
  if (attends && !kernel_ready(a->q, a->q_sb, a->q_st, a->q_sh, a->dtype)) p.q = take(a->B * a->Lq * a->H * D * 2);
  if (n_sparse > 0) {
    if (!kernel_ready(a->k, a->k_sb, a->k_st, a->k_sh, a->dtype)) p.k = take(a->B * a->Lkv * a->H * D * 2);
    if (!kernel_ready(a->v, a->v_sb, a->v_st, a->v_sh, a->dtype)) p.v = take(a->B * a->Lkv * a->H * D * 2);
    p.qp = take(a->B * a->H * p.nq * D * 4);
    p.kp = a->held ? 0 : take(a->B * a->H * p.nkv * D * 4);
    p.index = take(a->B * a->H * p.nq * p.nkv * 4);
    p.num = take(a->B * a->H * p.nq * 4);
    p.thresholds = take(a->H * 4);
    p.route = a->routing == WA_ROUTE_GINI ? take(wa_route_workspace_bytes(a->B, a->H, p.nq, p.nkv)) : 0;
    p.arrivals = take((p.rows_only + p.rows_both) * 4);
    const int64_t mv_only = a->units_only ? a->max_visits_only : p.nkv, mv_both = a->units_both ? a->max_visits_both : p.nkv;
    if (a->n_sparse_only > 0) p.bsa_only = take(wa_bsa_fwd_workspace_bytes(p.rows_only, mv_only, p.split_only, bs, D));
    if (a->n_both > 0) p.bsa_both = take(wa_bsa_fwd_workspace_bytes(p.rows_both, mv_both, p.split_both, bs, D));
  }
  if (n_linear > 0) {
    if (a->n_both > 0) p.lin = take(a->B * a->Lq * a->H * D * es);
    if (lowrank(a)) {
      p.lc = coarse_rows(a);
      // 128-query units at D = 128 walk the same 64-key steps in half the units
      p.dense_block = D == 128 ? 128 : bs;
      if (!a->kc || !kernel_ready(a->kc, a->kc_sb, a->kc_st, a->kc_sh, a->kc_dtype)) p.kc = take(a->B * p.lc * a->H * D * 2);
      if (!a->vc || !kernel_ready(a->vc, a->vc_sb, a->vc_st, a->vc_sh, a->vc_dtype)) p.vc = take(a->B * p.lc * a->H * D * 2);
      const int64_t dq = (a->Lq + p.dense_block - 1) / p.dense_block, dkv = (p.lc + p.dense_block - 1) / p.dense_block;
      if (a->n_both > 0) p.dense_both = take(wa_bsa_fwd_workspace_bytes(a->B * a->n_both * dq, dkv, 0, p.dense_block, D));
      if (a->n_linear_only > 0)
        p.dense_only = take(wa_bsa_fwd_workspace_bytes(a->B * a->n_linear_only * dq, dkv, 0, p.dense_block, D));
    } else {
      const int64_t n_max = std::max(a->n_both, a->n_linear_only);  // the two lists run one after the other
      p.elu1 = take(wa_elu1_state_workspace_bytes(a->B, n_max, a->Lkv, D));
      p.state = take(a->B * n_max * D * D * 4);
      p.zsum = take(a->B * n_max * D * 4);
    }
  }
  p.total = o;
  return p;
}

// Linear branch of the heads in both branches (into lin) and of the linear-only heads (into the output).
int run_linear(const wa_hsa_any_args* a, const Plan& p, char* ws, const View& q, const View& kc, const View& vc, void* s) {
  const int64_t D = a->D;
  int rc = WA_OK;
  for (int which = 0; which < 2; ++which) {
    const bool both = which == 0;
    const int32_t* heads = both ? a->both_heads : a->linear_only_heads;
    const int64_t n = both ? a->n_both : a->n_linear_only;
    if (n == 0) continue;
    void* out = both ? (void*)(ws + p.lin) : a->o;
    const int64_t o_sb = both ? a->Lq * a->H * D : a->o_sb, o_st = both ? a->H * D : a->o_st, o_sh = both ? D : a->o_sh;
    if (lowrank(a)) {
      wa_bsa_fwd_args f{};
      f.q = q.p; f.q_sb = q.sb; f.q_st = q.st; f.q_sh = q.sh;
      f.k = kc.p; f.k_sb = kc.sb; f.k_st = kc.st; f.k_sh = kc.sh;
      f.v = vc.p; f.v_sb = vc.sb; f.v_st = vc.st; f.v_sh = vc.sh;
      f.o = out; f.o_sb = o_sb; f.o_st = o_st; f.o_sh = o_sh; f.o_dtype = a->o_dtype;
      f.heads = heads; f.n_heads = n;
      f.B = a->B; f.H = a->H; f.Lq = a->Lq; f.Lkv = p.lc; f.D = D; f.block_size = p.dense_block;
      f.scale = a->scale;
      f.workspace = ws + (both ? p.dense_both : p.dense_only);
      if (!both) {
        f.epilogue = WA_EPI_GATED; f.attn_round_bf16 = a->lin_round_bf16;
        f.gate_w = a->gate_w; f.gate_b = a->gate_b;
        f.gate_pre_bf16 = a->gate_pre_bf16; f.gate_out_bf16 = a->gate_out_bf16;
      }
      if ((rc = wa_bsa_fwd(&f, s)) != WA_OK) return rc;
      continue;
    }
    wa_elu1_state_args e{};
    e.k = a->k; e.k_sb = a->k_sb; e.k_st = a->k_st; e.k_sh = a->k_sh;
    e.v = a->v; e.v_sb = a->v_sb; e.v_st = a->v_st; e.v_sh = a->v_sh; e.dtype = a->dtype;
    e.B = a->B; e.H = a->H; e.L = a->Lkv; e.D = D; e.heads = heads; e.n_heads = n;
    e.state = (float*)(ws + p.state); e.zsum = (float*)(ws + p.zsum); e.workspace = ws + p.elu1;
    if ((rc = wa_elu1_state(&e, s)) != WA_OK) return rc;
    wa_elu1_readout_args r{};
    r.q = a->q; r.q_sb = a->q_sb; r.q_st = a->q_st; r.q_sh = a->q_sh; r.q_dtype = a->dtype;
    r.state = e.state; r.zsum = e.zsum;
    r.o = out; r.o_sb = o_sb; r.o_st = o_st; r.o_sh = o_sh; r.o_dtype = a->o_dtype;
    r.B = a->B; r.H = a->H; r.L = a->Lq; r.D = D; r.heads = heads; r.n_heads = n;
    if (!both) {
      r.epilogue = WA_EPI_GATED; r.gate_w = a->gate_w; r.gate_b = a->gate_b;
      r.gate_pre_bf16 = a->gate_pre_bf16; r.gate_out_bf16 = a->gate_out_bf16; r.lin_round_bf16 = a->lin_round_bf16;
    }
    if ((rc = wa_elu1_readout(&r, s)) != WA_OK) return rc;
  }
  return rc;
}

int run_routing(const wa_hsa_any_args* a, const Plan& p, char* ws, void* s) {
  wa_pool_args pj[2] = {};
  const void* xs[2] = {a->q, a->k};
  const int64_t sb[2] = {a->q_sb, a->k_sb}, st[2] = {a->q_st, a->k_st}, sh[2] = {a->q_sh, a->k_sh};
  const int64_t len[2] = {a->Lq, a->Lkv}, nb[2] = {p.nq, p.nkv}, at[2] = {p.qp, p.kp};
  for (int i = 0; i < 2; ++i) {
    pj[i].x = xs[i]; pj[i].x_sb = sb[i]; pj[i].x_st = st[i]; pj[i].x_sh = sh[i]; pj[i].x_dtype = a->dtype;
    pj[i].B = a->B; pj[i].L = len[i]; pj[i].H = a->H; pj[i].D = a->D; pj[i].block_size = a->block_size;
    pj[i].num_blocks = nb[i];
    pj[i].heads = a->sparse_heads; pj[i].n_heads = a->n_both + a->n_sparse_only;
    pj[i].out = (float*)(ws + at[i]); pj[i].emulate_rounding = 1;
  }
  int rc = wa_block_mean_pool_n(pj, a->held ? 1 : 2, s);
  if (rc != WA_OK) return rc;
  wa_route_args r{};
  r.q_pooled = (const float*)(ws + p.qp);
  r.k_pooled = a->held ? a->held : (const float*)(ws + p.kp);
  r.B = a->B; r.H = a->H; r.Nq = p.nq; r.Nkv = p.nkv; r.D = a->D; r.mode = a->routing;
  r.tau_min = a->tau_min; r.tau_span = a->tau_span; r.head_k = a->head_k;
  r.heads = a->sparse_heads; r.n_heads = a->n_both + a->n_sparse_only;
  r.index = (int32_t*)(ws + p.index); r.num = (int32_t*)(ws + p.num); r.thresholds = (float*)(ws + p.thresholds);
  r.workspace = a->routing == WA_ROUTE_GINI ? ws + p.route : nullptr;
  r.clear = (int32_t*)(ws + p.arrivals); r.n_clear = p.rows_only + p.rows_both;
  if (a->held) {
    r.k_pooled_blocks = a->held_blocks;
    if (a->held_sums) {
      r.k_sum_len = a->Lkv; r.block_size = a->block_size; r.k_sum_bf16 = a->dtype == WA_BF16;
    }
  }
  r.scale = a->scale;
  return wa_route(&r, s);
}

int run_sparse(const wa_hsa_any_args* a, const Plan& p, char* ws, const View& q, const View& k, const View& v, bool both,
               void* s) {
  wa_bsa_fwd_args f{};
  f.q = q.p; f.q_sb = q.sb; f.q_st = q.st; f.q_sh = q.sh;
  f.k = k.p; f.k_sb = k.sb; f.k_st = k.st; f.k_sh = k.sh;
  f.v = v.p; f.v_sb = v.sb; f.v_st = v.st; f.v_sh = v.sh;
  f.o = a->o; f.o_sb = a->o_sb; f.o_st = a->o_st; f.o_sh = a->o_sh; f.o_dtype = a->o_dtype;
  f.index = (const int32_t*)(ws + p.index); f.num = (const int32_t*)(ws + p.num); f.index_width = p.nkv;
  f.heads = both ? a->both_heads : a->sparse_only_heads; f.n_heads = both ? a->n_both : a->n_sparse_only;
  f.B = a->B; f.H = a->H; f.Lq = a->Lq; f.Lkv = a->Lkv; f.D = a->D; f.block_size = a->block_size;
  f.scale = a->scale; f.attn_round_bf16 = 1;
  if (both) {
    f.epilogue = WA_EPI_FUSE;
    f.x = ws + p.lin; f.x_sb = a->Lq * a->H * a->D; f.x_st = a->H * a->D; f.x_sh = a->D; f.x_dtype = a->o_dtype;
    f.gate_w = a->gate_w; f.gate_b = a->gate_b;
    f.gate_pre_bf16 = a->gate_pre_bf16; f.gate_out_bf16 = a->gate_out_bf16;
  }
  f.workspace = ws + (both ? p.bsa_both : p.bsa_only);
  f.units = both ? a->units_both : a->units_only; f.n_units = both ? a->n_units_both : a->n_units_only;
  f.max_visits = f.units ? (both ? a->max_visits_both : a->max_visits_only) : p.nkv;
  f.split_visits = (int32_t)(both ? p.split_both : p.split_only);
  f.arrivals = (int32_t*)(ws + p.arrivals) + (both ? p.rows_only : 0);
  return wa_bsa_fwd(&f, s);
}

int check_args(const wa_hsa_any_args* a) {
  WA_CHECK_ARG(a && a->q && a->k && a->v && a->o, "wa_hsa_fwd_any: null argument");
  WA_CHECK_ARG(a->dtype == WA_F32 || a->dtype == WA_BF16, "wa_hsa_fwd_any: q / k / v must be fp32 or bf16");
  WA_CHECK_ARG(a->o_dtype == WA_F32 || a->o_dtype == WA_BF16, "wa_hsa_fwd_any: bad output dtype");
  WA_CHECK_ARG(a->D == 64 || a->D == 128, "wa_hsa_fwd_any: head dim %lld not in {64, 128}", (long long)a->D);
  WA_CHECK_ARG(a->block_size == 64 || a->block_size == 128, "wa_hsa_fwd_any: block size %lld not in {64, 128}",
               (long long)a->block_size);
  WA_CHECK_ARG(a->B > 0 && a->H > 0 && a->Lq > 0 && a->Lkv > 0 && a->B < (1 << 20) && a->Lq < (1 << 30) && a->Lkv < (1 << 30) &&
                   a->H < (1 << 20),
               "wa_hsa_fwd_any: bad sizes");
  WA_CHECK_ARG(a->n_both >= 0 && a->n_sparse_only >= 0 && a->n_linear_only >= 0 &&
                   a->n_both + a->n_sparse_only + a->n_linear_only <= a->H,
               "wa_hsa_fwd_any: bad head counts");
  WA_CHECK_ARG((a->n_both == 0 || a->both_heads) && (a->n_sparse_only == 0 || a->sparse_only_heads) &&
                   (a->n_linear_only == 0 || a->linear_only_heads) &&
                   (a->n_both + a->n_sparse_only == 0 || a->sparse_heads),
               "wa_hsa_fwd_any: head lists are missing");
  WA_CHECK_ARG(a->routing == WA_ROUTE_GINI || (a->routing == WA_ROUTE_TOPK && (a->head_k || a->n_both + a->n_sparse_only == 0)),
               "wa_hsa_fwd_any: bad routing");
  WA_CHECK_ARG(a->linear_mode == WA_LINEAR_LOWRANK || a->linear_mode == WA_LINEAR_ELU1, "wa_hsa_fwd_any: bad linear mode");
  WA_CHECK_ARG((a->kc == nullptr) == (a->vc == nullptr), "wa_hsa_fwd_any: kc and vc go together");
  WA_CHECK_ARG(!lowrank(a) || a->n_both + a->n_linear_only == 0 ||
                   (a->kc ? a->lc > 0 && a->lc < (1 << 30) : a->k_proj && a->v_proj && a->proj_rank > 0 && a->proj_len > 0),
               "wa_hsa_fwd_any: the low-rank branch needs coarse keys and values or their projections");
  WA_CHECK_ARG(a->split_visits >= 0 && a->split_visits <= 64 && a->split_both >= 0 && a->split_both <= 64,
               "wa_hsa_fwd_any: bad split");
  WA_CHECK_ARG((a->units_only == nullptr || a->max_visits_only > 0) && (a->units_both == nullptr || a->max_visits_both > 0),
               "wa_hsa_fwd_any: a unit table needs its largest visit count");
  WA_CHECK_ARG(a->held == nullptr || a->held_blocks >= (a->Lkv + a->block_size - 1) / a->block_size,
               "wa_hsa_fwd_any: too few held key blocks");
  WA_CHECK_ARG(a->side_stream == nullptr || (a->fork_event && a->join_event),
               "wa_hsa_fwd_any: a side stream needs its fork and join events");
  return WA_OK;
}

}  // namespace

extern "C" int64_t wa_hsa_fwd_any_workspace_bytes(const wa_hsa_any_args* a) {
  return check_args(a) == WA_OK ? make_plan(a).total : 0;
}

extern "C" int wa_hsa_fwd_any(const wa_hsa_any_args* a, void* stream) {
  int rc = check_args(a);
  if (rc != WA_OK) return rc;
  WA_CHECK_ARG(a->workspace && wa_aligned16(a->workspace), "wa_hsa_fwd_any: workspace must be 16-byte aligned");
  const Plan p = make_plan(a);
  char* ws = (char*)a->workspace;
  const bool sparse = a->n_both + a->n_sparse_only > 0, linear = a->n_both + a->n_linear_only > 0;
  const bool dense = linear && lowrank(a);
  const int64_t D = a->D;

  // bf16 views; the copies that some need are made by one launch ahead of both branches
  CastJobs c{};
  c.H = (int)a->H; c.D = (int)D;
  auto view = [&](bool used, const void* t, int64_t sb, int64_t st, int64_t sh, int dtype, int64_t L, int64_t at) -> View {
    if (!used || kernel_ready(t, sb, st, sh, dtype)) return {t, sb, st, sh};
    const int64_t vec = dtype == WA_F32 ? 4 : 8;
    c.j[c.n++] = CastJob{t, sb, st, sh, dtype, wa_aligned16(t) && sb % vec == 0 && st % vec == 0 && sh % vec == 0,
                         (bf16_t*)(ws + at), L, c.total};
    c.total += a->B * L * a->H * (D / 8);
    return {ws + at, L * a->H * D, a->H * D, D};
  };
  const View q = view(sparse || dense, a->q, a->q_sb, a->q_st, a->q_sh, a->dtype, a->Lq, p.q);
  const View k = view(sparse, a->k, a->k_sb, a->k_st, a->k_sh, a->dtype, a->Lkv, p.k);
  const View v = view(sparse, a->v, a->v_sb, a->v_st, a->v_sh, a->dtype, a->Lkv, p.v);
  View kc{ws + p.kc, p.lc * a->H * D, a->H * D, D}, vc{ws + p.vc, p.lc * a->H * D, a->H * D, D};
  if (dense && a->kc) {
    kc = view(true, a->kc, a->kc_sb, a->kc_st, a->kc_sh, a->kc_dtype, p.lc, p.kc);
    vc = view(true, a->vc, a->vc_sb, a->vc_st, a->vc_sh, a->vc_dtype, p.lc, p.vc);
  }
  if (c.n > 0) {
    WA_CHECK_ARG((c.total + 255) / 256 < ((int64_t)1 << 31), "wa_hsa_fwd_any: sizes too large");
    hipLaunchKernelGGL(cast_blhd_kernel, dim3((unsigned)((c.total + 255) / 256)), dim3(256), 0, (hipStream_t)stream, c);
    if ((rc = wa_launch_status("hsa_cast")) != WA_OK) return rc;
  }

  const bool two = p.linear_side && a->side_stream != nullptr && a->side_stream != stream;
  hipStream_t main = (hipStream_t)stream, side = two ? (hipStream_t)a->side_stream : main;
  hipEvent_t fork = (hipEvent_t)a->fork_event, join = (hipEvent_t)a->join_event;
  hipError_t e;
  if (two) {
    if ((e = hipEventRecord(fork, main)) != hipSuccess || (e = hipStreamWaitEvent(side, fork, 0)) != hipSuccess)
      return wa_fail((int)e, "wa_hsa_fwd_any: fork: %s", hipGetErrorString(e));
  }
  if (dense && !a->kc) {
    wa_compress_args cj[2] = {};
    for (int i = 0; i < 2; ++i) {
      wa_compress_args& j = cj[i];
      j.x = i ? a->v : a->k; j.x_sb = i ? a->v_sb : a->k_sb; j.x_st = i ? a->v_st : a->k_st; j.x_sh = i ? a->v_sh : a->k_sh;
      j.x_dtype = a->dtype;
      j.proj = i ? a->v_proj : a->k_proj; j.proj_dtype = a->proj_dtype; j.proj_rank = a->proj_rank; j.proj_len = a->proj_len;
      j.B = a->B; j.L = a->Lkv; j.H = a->H; j.D = D;
      j.segment_len = a->segment_len > 0 ? a->segment_len : a->Lkv; j.block_size = a->block_size;
      j.out = ws + (i ? p.vc : p.kc); j.o_sb = p.lc * a->H * D; j.o_st = a->H * D; j.o_sh = D; j.o_dtype = WA_BF16;
    }
    rc = wa_compress_kv_n(cj, 2, side);
  }
  if (rc == WA_OK && linear) rc = run_linear(a, p, ws, q, kc, vc, side);
  if (rc == WA_OK && sparse) rc = run_routing(a, p, ws, main);
  if (rc == WA_OK && a->n_sparse_only > 0) rc = run_sparse(a, p, ws, q, k, v, false, main);
  if (two) {  // the side stream is joined on every path (a capture must end joined)
    if ((e = hipEventRecord(join, side)) != hipSuccess || (e = hipStreamWaitEvent(main, join, 0)) != hipSuccess)
      return rc != WA_OK ? rc : wa_fail((int)e, "wa_hsa_fwd_any: join: %s", hipGetErrorString(e));
  }
  if (rc == WA_OK && a->n_both > 0) rc = run_sparse(a, p, ws, q, k, v, true, main);
  return rc;
}
