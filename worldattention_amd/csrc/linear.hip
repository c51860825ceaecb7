// Low-rank linear branch of the reference (wan/modules/hsa/attention.py:64-118) for gfx950:
//  * compress_kv — low-rank sequence projection per segment (attention.py:64-110); the softmax
//    over the compressed keys then runs in the block-sparse kernel as dense attention;
//  * its backward (dx and the projection's gradient) for training in the reference's head mode.
// The contraction runs on v_mfma_f32_32x32x16_bf16 with fp32 accumulation; the token-axis
// operand is staged through LDS transposed ([channel][token]).
// The north-star elu(x)+1 linear branch lives in elu1.hip.
#include <algorithm>
#include <type_traits>

#include "common.h"
#include "split3.h"
#include "tile.h"

namespace {

struct CompressParams {
  const void* x; int64_t x_sb, x_st, x_sh; int x_dtype;
  const void* proj; int proj_dtype; int proj_rank, proj_len;
  int L, H, D, seg, block;
  void* out; int64_t o_sb, o_st, o_sh; int o_dtype;
  int64_t x_slab;   // bytes of one (batch, head) x slab: first row to the last row's end
  int proj_vec;     // rows of E 16-byte aligned, a multiple of 8 elements long
};

// One launch takes up to two jobs of one grid (a call's keys and values): grid.z = jobs x batch.
struct CompressJobs {
  CompressParams j[2];
  int batch;
};

// =============================================================================================
// compress_kv: out[row0 + r, d] = sum_t E[r, t] x[start + t, d], one workgroup per
// (segment, head, batch, job), as out^T = x^T E^T on the matrix cores (operands rounded to bf16,
// fp32 sums). General kernel (any x type and alignment, D 32 / 64 / 128, rank up to 128); bf16 x
// with 16-byte aligned rows takes compress_stream_kernel instead.
//
// Bound by reading x once. 4 token groups x D / 32 channel tiles of waves: a wave loads its operand
// straight from global memory (lane = channel, 8 consecutive tokens: every load instruction covers
// two 32-channel rows) for 32 tokens at a time, chunks dealt to the groups in turn, and the groups'
// sums meet in LDS in group order. 16 waves x 16 loads in flight cover a memory round trip; the
// kernel before it staged x through LDS with 4 waves and one barrier pair per 64 tokens, one
// element per load: keys and values of H 12, L 32,760, D 128 fp32 at segment 1,560,
// rank 25 took 379 us (two launches) against 84 us here, and B 2, H 6, L 5,003 335 us against 20 (27-30
// beside a call's other kernels).
// =============================================================================================
constexpr int kTokenGroups = 4;

__device__ __forceinline__ bf16x8 compress_e8(const CompressParams& p, int r, int t, int seg_len) {
  bf16x8 f;
  const int64_t off = (int64_t)r * p.proj_len + t;
  if (p.proj_vec && t + 8 <= seg_len) {
    if (p.proj_dtype == WA_BF16) return *(const bf16x8*)((const bf16_t*)p.proj + off);
    const f32x4 a = *(const f32x4*)((const float*)p.proj + off), c = *(const f32x4*)((const float*)p.proj + off + 4);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      f[e] = (bf16_t)a[e];
      f[e + 4] = (bf16_t)c[e];
    }
    return f;
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) f[e] = t + e < seg_len ? (bf16_t)wa_load_f(p.proj, off + e, p.proj_dtype) : (bf16_t)0.f;
  return f;
}

template <typename T, int D, int MT>
__global__ void __launch_bounds__(kTokenGroups * 2 * D) compress_direct_kernel(CompressJobs jobs) {
  constexpr int DT = D / 32;
  __shared__ float red[kTokenGroups - 1][DT][16][64];
  const CompressParams p = jobs.j[blockIdx.z / jobs.batch];
  const int sidx = blockIdx.x, h = blockIdx.y, b = blockIdx.z % jobs.batch;
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ct = w % DT, tg = w / DT, g = lane >> 5, l32 = lane & 31;
  const int start = sidx * p.seg;
  const int seg_len = min(p.seg, p.L - start);
  const int rank = min(p.proj_rank, (seg_len + p.block - 1) / p.block);
  const int row0 = sidx * min(p.proj_rank, (p.seg + p.block - 1) / p.block);
  const T* xcol = (const T*)p.x + (int64_t)b * p.x_sb + (int64_t)h * p.x_sh + (int64_t)start * p.x_st + 32 * ct + l32;
  f32x16 acc[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) acc[m] = f32x16{};
  for (int t0 = 32 * tg; t0 < seg_len; t0 += 32 * kTokenGroups) {
    T xv[2][8];  // tokens t0 + 16 ks + 8 g + e
    if (t0 + 32 <= seg_len) {
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
#pragma unroll
        for (int e = 0; e < 8; ++e) xv[ks][e] = xcol[(int64_t)(t0 + 16 * ks + 8 * g + e) * p.x_st];
      }
    } else {
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const int t = t0 + 16 * ks + 8 * g + e;
          xv[ks][e] = xcol[(int64_t)min(t, seg_len - 1) * p.x_st];
          if (t >= seg_len) xv[ks][e] = (T)0.f;
        }
      }
    }
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      bf16x8 xf;
#pragma unroll
      for (int e = 0; e < 8; ++e) xf[e] = (bf16_t)xv[ks][e];
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        if (32 * m >= rank) break;  // uniform
        // rows of E past the rank repeat its last one (their results are not stored)
        acc[m] = wa_mfma32(xf, compress_e8(p, min(32 * m + l32, rank - 1), t0 + 16 * ks + 8 * g, seg_len), acc[m]);
      }
    }
  }
  // lane l32 holds rank row r = 32 m + l32, channels 32 ct + 8 (i / 4) + 4 g + i % 4
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    if (32 * m >= rank) break;  // uniform over the workgroup
    if (m) __syncthreads();
    if (tg > 0) {
#pragma unroll
      for (int i = 0; i < 16; ++i) red[tg - 1][ct][i][lane] = acc[m][i];
    }
    __syncthreads();
    const int r = 32 * m + l32;
    if (tg == 0 && r < rank) {
      const int64_t o0 = (int64_t)b * p.o_sb + (int64_t)(row0 + r) * p.o_st + (int64_t)h * p.o_sh + 32 * ct + 4 * g;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        float v = acc[m][i];
#pragma unroll
        for (int q = 0; q < kTokenGroups - 1; ++q) v += red[q][ct][i][lane];
        wa_store_f(p.out, o0 + 8 * (i >> 2) + (i & 3), v, p.o_dtype);
      }
    }
  }
}

// =============================================================================================
// compress_kv for bf16 x with 16-byte aligned rows, as out^T[d, r] = sum_t x^T[d, t] E^T[t, r]:
// the segment's x rows stream global -> LDS in 64-token tiles (direct-to-LDS loads, a 4-stage
// ring, three tiles in flight; inline-assembly loads that the kernel orders itself, so the
// compiler adds no waits of its own), each with the 32 x 64 slice of E it needs; wave w takes the A
// operand of its 32 channels by transpose reads of the row-major x tile and the B operand (lane =
// row r of E, 8 consecutive tokens) by one 16-byte read of the E slice. Rows of E past this
// segment's rank and rows of x past the tensor's end read zeros (buffer range); tokens past the
// segment's end get zero weights in its last tile. One workgroup per (segment, head, batch,
// job); a call's keys and values share a launch, so that two workgroups run on a CU: at H 12, D 128,
// L 32,760, segment 1,560 39.5 us in two
// launches, 36 us in one.
// =============================================================================================
template <int D>
__global__ void __launch_bounds__(2 * D) compress_stream_kernel(CompressJobs jobs) {
  constexpr int NW = D / 32, TILE = 64 * D, SS = TILE + 32 * 64;  // stage: x tile, then E slice
  constexpr int CPR = D / 8, RPI = 64 / CPR, NI = 64 / (RPI * NW);  // x tile: NI loads per wave
  constexpr int EI = 4 / NW;                                         // E slice: EI loads per wave
  __shared__ __attribute__((aligned(1024))) bf16_t st0[SS];
  __shared__ __attribute__((aligned(1024))) bf16_t st1[SS];
  __shared__ __attribute__((aligned(1024))) bf16_t st2[SS];
  __shared__ __attribute__((aligned(1024))) bf16_t st3[SS];
  const CompressParams p = jobs.j[blockIdx.z / jobs.batch];
  const int sidx = blockIdx.x, h = blockIdx.y, b = blockIdx.z % jobs.batch;
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 5, l32 = lane & 31;
  const int start = sidx * p.seg;
  const int seg_len = min(p.seg, p.L - start);
  const int rank = min(p.proj_rank, (seg_len + p.block - 1) / p.block);
  const int row0 = sidx * min(p.proj_rank, (p.seg + p.block - 1) / p.block);
  const int nt = (seg_len + 63) / 64;

  // x tile i = segment tokens 64 i .. 64 i + 63: lane L of wave instruction k writes row
  // (k NW + w) RPI + L / CPR, chunk slot L % CPR (dual swizzle)
  const char* xbase = (const char*)p.x + ((int64_t)b * p.x_sb + (int64_t)h * p.x_sh) * 2;
  int xoff[NI];
#pragma unroll
  for (int k = 0; k < NI; ++k) {
    const int row = (k * NW + w) * RPI + lane / CPR, pos = lane % CPR;
    xoff[k] = (int)(row * p.x_st * 2) + (pos ^ dual_swizzle<D>(row)) * 16;
  }
  // E slice of tile i: rank rows 0..31 x tokens 64 i .. +63 (128 bytes a row); lane L of wave
  // instruction k writes row (k NW + w) 8 + L / 8, chunk slot L % 8 holding chunk slot ^ (row & 7)
  int eoff[EI];
#pragma unroll
  for (int k = 0; k < EI; ++k) {
    const int row = (k * NW + w) * 8 + lane / 8, pos = lane % 8;
    eoff[k] = row < rank ? row * p.proj_len * 2 + ((pos ^ (row & 7)) * 16) : 0x7fff0000;  // past the range: 0
  }
  auto issue = [&](bf16_t* stage, int i) {
    if (i >= nt) return;  // uniform
    const int64_t o = (int64_t)(start + 64 * i) * p.x_st * 2;
    const __amdgpu_buffer_rsrc_t xrs =
        __builtin_amdgcn_make_buffer_rsrc((void*)(xbase + o), (short)0, (int)(p.x_slab - o), WA_BUF_DWORD3);
#pragma unroll
    for (int k = 0; k < NI; ++k) lds_dma16(xrs, stage + (k * NW + w) * RPI * D, xoff[k]);
    const __amdgpu_buffer_rsrc_t ers = __builtin_amdgcn_make_buffer_rsrc((void*)((const char*)p.proj + 128 * i), (short)0,
                                                                         p.proj_rank * p.proj_len * 2 - 128 * i, WA_BUF_DWORD3);
#pragma unroll
    for (int k = 0; k < EI; ++k) lds_dma16(ers, stage + TILE + (k * NW + w) * 512, eoff[k]);
  };
  issue(st0, 0);
  issue(st1, 1);
  issue(st2, 2);
  f32x16 acc = f32x16{};
  // tile i computes on stage i % 4; every tile issues the same NI + EI loads per wave, so tile i has
  // landed once at most that many per later tile remain in flight
  auto step = [&](bf16_t* stage, bf16_t* refill, int i) {
    const int ahead = min(2, nt - 1 - i);
    if (ahead >= 2) asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(2 * (NI + EI)) : "memory");
    else if (ahead == 1) asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(NI + EI) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
    bf16x8 ef[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) ef[c] = *(const bf16x8*)(stage + TILE + l32 * 64 + (((2 * c + g) ^ (l32 & 7)) * 8));
    if (64 * i + 64 > seg_len) {  // uniform: the segment's partial last tile
#pragma unroll
      for (int c = 0; c < 4; ++c) {
#pragma unroll
        for (int e = 0; e < 8; ++e) ef[c][e] = 64 * i + 16 * c + 8 * g + e < seg_len ? ef[c][e] : (bf16_t)0.f;
      }
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) acc = wa_mfma32(tile_tr8n<D>(stage, c, 32 * w, lane), ef[c], acc);
    // the stage of tile i - 1, which every wave had read before the barrier above (issued after
    // this tile's reads, so that no read of this stage waits for it)
    issue(refill, i + 3);
  };
  for (int i = 0; i < nt; i += 4) {
    step(st0, st3, i);
    if (i + 1 < nt) step(st1, st0, i + 1);
    if (i + 2 < nt) step(st2, st1, i + 2);
    if (i + 3 < nt) step(st3, st2, i + 3);
  }
  // lane l32 holds rank row r = l32, channels d = 32 w + 8 (i / 4) + 4 g + i % 4
  if (l32 >= rank) return;
  const int64_t o0 = (int64_t)b * p.o_sb + (int64_t)(row0 + l32) * p.o_st + (int64_t)h * p.o_sh + 32 * w + 4 * g;
#pragma unroll
  for (int rq = 0; rq < 4; ++rq) {
#pragma unroll
    for (int i = 0; i < 4; ++i) wa_store_f(p.out, o0 + 8 * rq + i, acc[rq * 4 + i], p.o_dtype);
  }
}

// =============================================================================================
// compress_kv backward. For segment s (tokens start .. start + n, rows row0 .. row0 + r of the
// compressed output, row0 = s * r_full): dx[start + t] = sum_j E[j, t] dout[row0 + j] and the
// segment's share of dE[j, t] = sum_{b, h, d} dout[b, row0 + j, h, d] x[b, start + t, h, d].
// fp32 arithmetic throughout; E is the projection's stored value (bf16 widened exactly).
// =============================================================================================
struct CompressBwdParams {
  const float* dout; int64_t d_sb, d_st, d_sh;
  const void* x; int64_t x_sb, x_st, x_sh; int x_dtype;
  const void* proj; int proj_dtype; int R, P;
  int B, L, H, D, seg, block, n_first, r_full, n_seg;
  float* dx; int64_t dx_sb, dx_st, dx_sh; int dx_acc;
  void* dx_out; int64_t dxo_sb, dxo_st, dxo_sh;  // bf16 result instead of writing dx back
  float* dproj; int dproj_acc;
  float* part;  // [n_seg][r_full][n_first]
};

// dx: one workgroup per (64-token tile of a segment, four 32-channel columns of (head, channel),
// batch); wave w owns column 4 blockIdx.x + w. dx^T = dout^T E with E from LDS by transpose reads
// (32 rank rows x 64 tokens at a time) and dout split in registers; lane = token, registers = four
// consecutive channels, so the fp32 gradient it adds to is read by 16 bytes per lane and the result
// stored by 16 (bf16: 8). Bound by that traffic: the products are 6 (bf16 E) or 12 per 32 x 32 tile.
// H 12, D 128, L 32,760, rank 25: adding to an fp32 gradient and writing it back took 142 us as fp32
// VALU products, and a separate pass to bf16 51 us more; here adding and writing bf16 takes
// 118 us (with lane = channel, 4-byte reads and 2-byte stores: 129 us).
constexpr int kDxTokens = 64;

template <typename PT>
__global__ void __launch_bounds__(256) compress_bwd_dx_kernel(CompressBwdParams p) {
  constexpr bool SPLIT_E = sizeof(PT) == 4;
  constexpr int ET = 32 * kDxTokens;
  __shared__ __attribute__((aligned(1024))) bf16_t es[(SPLIT_E ? 3 : 1) * ET];
  const int tps = (p.n_first + kDxTokens - 1) / kDxTokens;
  const int s = blockIdx.y / tps, t0 = (blockIdx.y % tps) * kDxTokens, b = blockIdx.z;
  const int start = s * p.seg, n = min(p.seg, p.L - start);
  if (t0 >= n) return;  // uniform
  const int r = min(p.R, (n + p.block - 1) / p.block), row0 = s * p.r_full;
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 5, l32 = lane & 31;
  const int ct = blockIdx.x * 4 + w;
  const bool active = ct < p.H * p.D / 32;  // uniform over the wave
  const int h = active ? ct * 32 / p.D : 0, d = active ? ct * 32 % p.D : 0;
  const float* gcol = p.dout + (int64_t)b * p.d_sb + (int64_t)row0 * p.d_st + (int64_t)h * p.d_sh + d + l32;
  // this lane's tokens t0 + 32 tt + l32, channels d + 8 rq + 4 g + i
  const int64_t dx0 = (int64_t)b * p.dx_sb + (int64_t)start * p.dx_st + (int64_t)h * p.dx_sh + d + 4 * g;
  f32x4 prev[2][4];
#pragma unroll
  for (int tt = 0; tt < 2; ++tt) {
#pragma unroll
    for (int rq = 0; rq < 4; ++rq)
      prev[tt][rq] = p.dx_acc && active
                         ? *(const f32x4*)(p.dx + dx0 + (int64_t)min(t0 + 32 * tt + l32, n - 1) * p.dx_st + 8 * rq)
                         : f32x4{};
  }
  f32x16 acc[2] = {f32x16{}, f32x16{}}, low[2] = {f32x16{}, f32x16{}};
  for (int j0 = 0; j0 < r; j0 += 32) {
    if (j0) __syncthreads();  // the previous rows have been read
    {
      const int jj = tid / 8, c = tid % 8, j = j0 + jj, t = t0 + 8 * c;  // 8 tokens of one row per thread
      float e8[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) e8[e] = j < r && t + e < n ? (float)((const PT*)p.proj)[(int64_t)j * p.P + t + e] : 0.f;
      const Split3 sp = split3(e8);  // a bf16 value is its own hi part
      tile_put8<kDxTokens>(es, jj, c, sp.hi);
      if constexpr (SPLIT_E) {
        tile_put8<kDxTokens>(es + ET, jj, c, sp.mid);
        tile_put8<kDxTokens>(es + 2 * ET, jj, c, sp.lo);
      }
    }
    Split3 gs[2];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      float v[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int j = j0 + 16 * ks + 8 * g + e;
        v[e] = gcol[(int64_t)min(j, r - 1) * p.d_st];
        if (j >= r) v[e] = 0.f;
      }
      gs[ks] = split3(v);
    }
    __syncthreads();
#pragma unroll
    for (int tt = 0; tt < 2; ++tt) {
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        const bf16x8 eh = tile_tr8n<kDxTokens>(es, ks, 32 * tt, lane);
        if constexpr (SPLIT_E) {
          const Split3 ea = {eh, tile_tr8n<kDxTokens>(es + ET, ks, 32 * tt, lane),
                             tile_tr8n<kDxTokens>(es + 2 * ET, ks, 32 * tt, lane), finite8(eh)};
          mfma_split(gs[ks], ea, acc[tt], low[tt]);
        } else {
          mfma_split(gs[ks], Plain{eh, finite8(eh)}, acc[tt], low[tt]);
        }
      }
    }
  }
  if (!active) return;
#pragma unroll
  for (int tt = 0; tt < 2; ++tt) {
    const int t = t0 + 32 * tt + l32;
    if (t >= n) continue;
    bf16_t* o16 = (bf16_t*)p.dx_out + ((int64_t)b * p.dxo_sb + (int64_t)(start + t) * p.dxo_st + (int64_t)h * p.dxo_sh + d + 4 * g);
    float* o32 = p.dx + dx0 + (int64_t)t * p.dx_st;
#pragma unroll
    for (int rq = 0; rq < 4; ++rq) {
      f32x4 v;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float a = SPLIT_E ? acc[tt][4 * rq + i] + low[tt][4 * rq + i] : acc[tt][4 * rq + i];
        v[i] = prev[tt][rq][i] + a;
      }
      if (p.dx_out) *(bf16x4*)(o16 + 8 * rq) = bf16x4{(bf16_t)v[0], (bf16_t)v[1], (bf16_t)v[2], (bf16_t)v[3]};
      else *(f32x4*)(o32 + 8 * rq) = v;
    }
  }
}

// dE share of one segment, as dout (rows) times x^T over (batch, head, channel): one workgroup of 8
// waves per (64-token tile, segment); wave w sums the 32-channel runs w, w + 8, ... on the matrix
// cores (A: dout rows split in three, B: x rows, lane = token), then the waves' sums are added in
// wave order through LDS into the segment's partial. Bound by reading x once (each token tile
// re-reads the segment's dout rows from L2). H 12, D 128, L 32,760, rank 25, bf16 x: 251 us as fp32
// VALU products, 60 us with four waves a workgroup, 50 us here.
constexpr int kDprojWaves = 8;

template <typename T, int MT>
__global__ void __launch_bounds__(64 * kDprojWaves) compress_bwd_dproj_kernel(CompressBwdParams p) {
  __shared__ float red[kDprojWaves][16][64];
  constexpr bool SPLIT_X = sizeof(T) == 4, LOW = SPLIT_X && MT < 4;  // (registers)
  const int s = blockIdx.y, t0 = blockIdx.x * 64;
  const int start = s * p.seg, n = min(p.seg, p.L - start);
  if (t0 >= n) return;  // uniform
  const int r = min(p.R, (n + p.block - 1) / p.block), row0 = s * p.r_full;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = lane >> 5, l32 = lane & 31;
  f32x16 acc[MT][2], low[MT][2];
#pragma unroll
  for (int m = 0; m < MT; ++m) acc[m][0] = acc[m][1] = low[m][0] = low[m][1] = f32x16{};
  // rows past the rank and tokens past the segment repeat the last one (their results are dropped)
  int64_t xo[2], go[MT];
#pragma unroll
  for (int tt = 0; tt < 2; ++tt) xo[tt] = (int64_t)(start + min(t0 + 32 * tt + l32, n - 1)) * p.x_st + 8 * g;
#pragma unroll
  for (int m = 0; m < MT; ++m) go[m] = (int64_t)(row0 + min(32 * m + l32, r - 1)) * p.d_st + 8 * g;
  const int runs = p.D / 32, total = p.B * p.H * runs;
#pragma unroll 2
  for (int u = w; u < total; u += kDprojWaves) {
    const int bh = u / runs, c0 = (u % runs) * 32, b = bh / p.H, h = bh % p.H;
    const T* xb = (const T*)p.x + (int64_t)b * p.x_sb + (int64_t)h * p.x_sh + c0;
    const float* gb = p.dout + (int64_t)b * p.d_sb + (int64_t)h * p.d_sh + c0;
#pragma unroll
    for (int d0 = 0; d0 < 32; d0 += 16) {
      std::conditional_t<SPLIT_X, Split3, Plain> xf[2];
#pragma unroll
      for (int tt = 0; tt < 2; ++tt) {
        if constexpr (SPLIT_X) {
          const f32x4 v0 = *(const f32x4*)(xb + xo[tt] + d0), v1 = *(const f32x4*)(xb + xo[tt] + d0 + 4);
          const float v[8] = {v0[0], v0[1], v0[2], v0[3], v1[0], v1[1], v1[2], v1[3]};
          xf[tt] = split3(v);
        } else {
          const bf16x8 v = *(const bf16x8*)(xb + xo[tt] + d0);
          xf[tt] = {v, finite8(v)};
        }
      }
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        if (32 * m >= r) break;  // uniform
        const f32x4 v0 = *(const f32x4*)(gb + go[m] + d0), v1 = *(const f32x4*)(gb + go[m] + d0 + 4);
        const float v[8] = {v0[0], v0[1], v0[2], v0[3], v1[0], v1[1], v1[2], v1[3]};
        const Split3 gs = split3(v);
#pragma unroll
        for (int tt = 0; tt < 2; ++tt) mfma_split(gs, xf[tt], acc[m][tt], LOW ? low[m][tt] : acc[m][tt]);
      }
    }
  }
  float* part = p.part + (int64_t)s * p.r_full * p.n_first;
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    if (32 * m >= r) break;
#pragma unroll
    for (int tt = 0; tt < 2; ++tt) {
      __syncthreads();
#pragma unroll
      for (int i = 0; i < 16; ++i) red[w][i][lane] = LOW ? acc[m][tt][i] + low[m][tt][i] : acc[m][tt][i];
      __syncthreads();
      // wave q adds registers q, q + 8: lane (l32, g) of register i is row 32 m + 8 (i / 4) + 4 g + i % 4
      const int t = t0 + 32 * tt + l32;
      for (int i = w; i < 16; i += kDprojWaves) {
        const int j = 32 * m + 8 * (i >> 2) + 4 * g + (i & 3);
        float v = red[0][i][lane];
#pragma unroll
        for (int q = 1; q < kDprojWaves; ++q) v += red[q][i][lane];
        if (j < r && t < n) part[(int64_t)j * p.n_first + t] = v;
      }
    }
  }
}

// dproj[j, t] (+)= sum over segments, in segment order, of the partials that cover (j, t); every
// entry of the [R, P] matrix is visited, so in write mode untouched entries become zero.
__global__ void __launch_bounds__(256) compress_bwd_reduce_kernel(CompressBwdParams p) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= (int64_t)p.R * p.P) return;
  const int j = (int)(i / p.P), t = (int)(i % p.P);
  float sum = 0.f;
  if (j < p.r_full && t < p.n_first) {
    // every segment but the last is full: it covers (j, t)
    const float* pp = p.part + (int64_t)j * p.n_first + t;
    const int64_t stride = (int64_t)p.r_full * p.n_first;
    int s = 0;
    for (; s + 8 < p.n_seg; s += 8) {  // eight loads in flight
      float v[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) v[q] = pp[(s + q) * stride];
#pragma unroll
      for (int q = 0; q < 8; ++q) sum += v[q];
    }
    for (; s < p.n_seg; ++s) {
      const int n = min(p.seg, p.L - s * p.seg);
      const int r = min(p.R, (n + p.block - 1) / p.block);
      if (j < r && t < n) sum += pp[s * stride];
    }
  }
  p.dproj[i] = p.dproj_acc ? p.dproj[i] + sum : sum;
}

}  // namespace

extern "C" int64_t wa_compress_kv_bwd_workspace_bytes(int64_t L, int64_t proj_rank, int64_t segment_len,
                                                      int64_t block_size) {
  if (L <= 0 || proj_rank <= 0 || segment_len <= 0 || block_size <= 0) return 0;
  const int64_t n_first = segment_len < L ? segment_len : L;
  const int64_t r_full = std::min(proj_rank, (n_first + block_size - 1) / block_size);
  const int64_t n_seg = (L + segment_len - 1) / segment_len;
  return n_seg * r_full * n_first * 4;
}

extern "C" int wa_compress_kv_bwd(const wa_compress_bwd_args* a, void* stream) {
  WA_CHECK_ARG(a && a->dout && a->x && a->proj, "wa_compress_kv_bwd: null argument");
  WA_CHECK_ARG(a->dproj == nullptr || a->workspace != nullptr, "wa_compress_kv_bwd: dproj needs the workspace");
  WA_CHECK_ARG(a->D == 32 || a->D == 64 || a->D == 128, "wa_compress_kv_bwd: head dim %lld not in {32, 64, 128}",
               (long long)a->D);
  WA_CHECK_ARG(a->x_dtype == WA_F32 || a->x_dtype == WA_BF16, "wa_compress_kv_bwd: bad dtype");
  WA_CHECK_ARG(a->proj_dtype == WA_F32 || a->proj_dtype == WA_BF16, "wa_compress_kv_bwd: bad proj dtype");
  WA_CHECK_ARG(a->segment_len > 0 && a->block_size > 0 && a->L > 0 && a->B >= 0 && a->H > 0,
               "wa_compress_kv_bwd: bad sizes");
  WA_CHECK_ARG(a->proj_rank > 0 && a->proj_rank <= 128, "wa_compress_kv_bwd: projection rank must be in [1, 128]");
  const int64_t n_first = a->segment_len < a->L ? a->segment_len : a->L;
  WA_CHECK_ARG(n_first <= a->proj_len, "wa_compress_kv_bwd: segment length %lld exceeds projection length %lld",
               (long long)n_first, (long long)a->proj_len);
  // vector accesses: dout by float4, x by 16 bytes (8 bf16 or 2 x 4 fp32)
  const int64_t xv = a->x_dtype == WA_BF16 ? 8 : 4;
  WA_CHECK_ARG(wa_aligned16(a->dout) && a->d_sb % 4 == 0 && a->d_st % 4 == 0 && a->d_sh % 4 == 0,
               "wa_compress_kv_bwd: dout must be 16-byte aligned with strides that are multiples of 4");
  WA_CHECK_ARG(wa_aligned16(a->x) && a->x_sb % xv == 0 && a->x_st % xv == 0 && a->x_sh % xv == 0,
               "wa_compress_kv_bwd: x must be 16-byte aligned with strides that are multiples of 16 bytes");
  WA_CHECK_ARG(a->dx == nullptr || (wa_aligned16(a->dx) && a->dx_sb % 4 == 0 && a->dx_st % 4 == 0 && a->dx_sh % 4 == 0),
               "wa_compress_kv_bwd: dx must be 16-byte aligned with strides that are multiples of 4");
  WA_CHECK_ARG(a->dx_bf16 == nullptr || (((uintptr_t)a->dx_bf16 & 7u) == 0 && a->dxo_sb % 4 == 0 && a->dxo_st % 4 == 0 &&
                                         a->dxo_sh % 4 == 0),
               "wa_compress_kv_bwd: dx_bf16 must be 8-byte aligned with strides that are multiples of 4");
  WA_CHECK_ARG(a->L <= INT32_MAX && a->proj_rank * a->proj_len <= INT32_MAX, "wa_compress_kv_bwd: sizes too large");
  const int64_t r_full = std::min(a->proj_rank, (n_first + a->block_size - 1) / a->block_size);
  const int64_t n_seg = (a->L + a->segment_len - 1) / a->segment_len;
  CompressBwdParams cp{a->dout, a->d_sb, a->d_st, a->d_sh, a->x, a->x_sb, a->x_st, a->x_sh, a->x_dtype,
                       a->proj, a->proj_dtype, (int)a->proj_rank, (int)a->proj_len,
                       (int)a->B, (int)a->L, (int)a->H, (int)a->D, (int)a->segment_len, (int)a->block_size,
                       (int)n_first, (int)r_full, (int)n_seg,
                       a->dx, a->dx_sb, a->dx_st, a->dx_sh, a->dx ? a->dx_accumulate : 0,
                       a->dx_bf16, a->dxo_sb, a->dxo_st, a->dxo_sh,
                       a->dproj, a->dproj_accumulate, (float*)a->workspace};
  hipStream_t s = (hipStream_t)stream;
  if (a->B > 0 && (a->dx || a->dx_bf16)) {
    const int64_t tps = (n_first + kDxTokens - 1) / kDxTokens;
    // the columns of a token tile are neighbours in launch order: whole rows of memory at a time
    dim3 grid((unsigned)((a->H * a->D / 32 + 3) / 4), (unsigned)(n_seg * tps), (unsigned)a->B);
    if (a->proj_dtype == WA_BF16) hipLaunchKernelGGL(compress_bwd_dx_kernel<bf16_t>, grid, dim3(256), 0, s, cp);
    else hipLaunchKernelGGL(compress_bwd_dx_kernel<float>, grid, dim3(256), 0, s, cp);
    const int rc = wa_launch_status("compress_kv_bwd (dx)");
    if (rc != WA_OK) return rc;
  }
  if (a->dproj) {
    if (a->B > 0) {
      dim3 grid((unsigned)((n_first + 63) / 64), (unsigned)n_seg);
      auto go = [&](auto bf, auto fp) {
        if (a->x_dtype == WA_BF16) hipLaunchKernelGGL(bf, grid, dim3(64 * kDprojWaves), 0, s, cp);
        else hipLaunchKernelGGL(fp, grid, dim3(64 * kDprojWaves), 0, s, cp);
      };
      if (r_full <= 32) go(compress_bwd_dproj_kernel<bf16_t, 1>, compress_bwd_dproj_kernel<float, 1>);
      else if (r_full <= 64) go(compress_bwd_dproj_kernel<bf16_t, 2>, compress_bwd_dproj_kernel<float, 2>);
      else go(compress_bwd_dproj_kernel<bf16_t, 4>, compress_bwd_dproj_kernel<float, 4>);
      const int rc = wa_launch_status("compress_kv_bwd (dproj)");
      if (rc != WA_OK) return rc;
    } else {
      cp.n_seg = 0;  // no batches: every partial is zero
    }
    const int64_t total = a->proj_rank * a->proj_len;
    hipLaunchKernelGGL(compress_bwd_reduce_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s, cp);
    return wa_launch_status("compress_kv_bwd (reduce)");
  }
  return WA_OK;
}

namespace {

// Kernel of a job: the streaming one for bf16 x with 16-byte aligned rows and a rank of at most 32.
enum CompressKernel { kStream, kDirect };

int plan_compress(const wa_compress_args* a, CompressParams& cp, CompressKernel& kernel) {
  WA_CHECK_ARG(a && a->x && a->proj && a->out, "wa_compress_kv: null argument");
  WA_CHECK_ARG(a->D == 64 || a->D == 128 || a->D == 32, "wa_compress_kv: head dim %lld not in {32, 64, 128}",
               (long long)a->D);
  WA_CHECK_ARG(a->x_dtype == WA_F32 || a->x_dtype == WA_BF16, "wa_compress_kv: bad dtype");
  WA_CHECK_ARG(a->proj_dtype == WA_F32 || a->proj_dtype == WA_BF16, "wa_compress_kv: bad proj dtype");
  WA_CHECK_ARG(a->segment_len > 0 && a->block_size > 0 && a->L > 0, "wa_compress_kv: bad sizes");
  WA_CHECK_ARG(a->proj_rank > 0 && a->proj_rank <= 128, "wa_compress_kv: projection rank must be in [1, 128]");
  const int64_t first_seg = a->segment_len < a->L ? a->segment_len : a->L;
  WA_CHECK_ARG(first_seg <= a->proj_len, "wa_compress_kv: segment length %lld exceeds projection length %lld",
               (long long)first_seg, (long long)a->proj_len);
  cp = CompressParams{a->x, a->x_sb, a->x_st, a->x_sh, a->x_dtype, a->proj, a->proj_dtype, (int)a->proj_rank,
                      (int)a->proj_len, (int)a->L, (int)a->H, (int)a->D, (int)a->segment_len, (int)a->block_size,
                      a->out, a->o_sb, a->o_st, a->o_sh, a->o_dtype};
  cp.proj_vec = wa_aligned16(a->proj) && a->proj_len % 8 == 0;
  const int64_t slab = ((a->L - 1) * a->x_st + a->D) * 2;
  const int64_t rank_used = std::min<int64_t>(a->proj_rank, (first_seg + a->block_size - 1) / a->block_size);
  kernel = kDirect;
  if ((a->D == 128 || a->D == 64) && a->x_dtype == WA_BF16 && wa_aligned16(a->x) && a->x_sb % 8 == 0 &&
      a->x_st % 8 == 0 && a->x_sh % 8 == 0 && slab < ((int64_t)1 << 31) && rank_used <= 32 &&
      a->proj_dtype == WA_BF16 && (((uintptr_t)a->proj) & 3) == 0 && a->proj_len % 2 == 0 &&
      a->proj_rank * a->proj_len * 2 < ((int64_t)1 << 31)) {
    kernel = kStream;
    cp.x_slab = slab;
  }
  return WA_OK;
}

template <typename T, int MT>
void launch_direct(const CompressJobs& jobs, int D, dim3 grid, hipStream_t s) {
  if (D == 128) hipLaunchKernelGGL((compress_direct_kernel<T, 128, MT>), grid, dim3(kTokenGroups * 256), 0, s, jobs);
  else if (D == 64) hipLaunchKernelGGL((compress_direct_kernel<T, 64, MT>), grid, dim3(kTokenGroups * 128), 0, s, jobs);
  else hipLaunchKernelGGL((compress_direct_kernel<T, 32, MT>), grid, dim3(kTokenGroups * 64), 0, s, jobs);
}

}  // namespace

extern "C" int wa_compress_kv_n(const wa_compress_args* a, int32_t n, void* stream) {
  WA_CHECK_ARG(a && n >= 1 && n <= 64, "wa_compress_kv_n: between 1 and 64 jobs");
  CompressParams cp[64];
  CompressKernel kernel[64];
  for (int i = 0; i < n; ++i) {  // every job is checked before the first launch
    const int rc = plan_compress(a + i, cp[i], kernel[i]);
    if (rc != WA_OK) return rc;
  }
  hipStream_t s = (hipStream_t)stream;
  for (int i = 0; i < n;) {
    const wa_compress_args& j = a[i];
    const bool pair = i + 1 < n && kernel[i + 1] == kernel[i] && a[i + 1].x_dtype == j.x_dtype && a[i + 1].B == j.B &&
                      a[i + 1].L == j.L && a[i + 1].H == j.H && a[i + 1].D == j.D &&
                      a[i + 1].segment_len == j.segment_len && a[i + 1].block_size == j.block_size &&
                      a[i + 1].proj_rank == j.proj_rank && 2 * j.B <= 65535;
    CompressJobs jobs{{cp[i], cp[pair ? i + 1 : i]}, (int)j.B};
    i += pair ? 2 : 1;
    if (j.B == 0) continue;
    const int64_t nseg = (j.L + j.segment_len - 1) / j.segment_len;
    const dim3 grid((unsigned)nseg, (unsigned)j.H, (unsigned)(pair ? 2 * j.B : j.B));
    if (kernel[i - 1] == kStream) {
      if (j.D == 128) hipLaunchKernelGGL(compress_stream_kernel<128>, grid, dim3(256), 0, s, jobs);
      else hipLaunchKernelGGL(compress_stream_kernel<64>, grid, dim3(128), 0, s, jobs);
    } else {
      const int64_t rank = std::min<int64_t>(j.proj_rank, (std::min(j.segment_len, j.L) + j.block_size - 1) / j.block_size);
      if (j.x_dtype == WA_F32) {
        if (rank <= 32) launch_direct<float, 1>(jobs, (int)j.D, grid, s);
        else launch_direct<float, 4>(jobs, (int)j.D, grid, s);
      } else {
        if (rank <= 32) launch_direct<bf16_t, 1>(jobs, (int)j.D, grid, s);
        else launch_direct<bf16_t, 4>(jobs, (int)j.D, grid, s);
      }
    }
    const int rc = wa_launch_status("compress_kv");
    if (rc != WA_OK) return rc;
  }
  return WA_OK;
}

extern "C" int wa_compress_kv(const wa_compress_args* a, void* stream) { return wa_compress_kv_n(a, 1, stream); }
