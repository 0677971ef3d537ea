// The router of a prompt's tokens (k_route's work for batches of hundreds of tokens and more): the
// logits on the f32 MFMA, then top-k, the grouped GEMM's records and the grouping by expert.
//
// v_mfma_f32_16x16x1_4b_f32 is four 16 x 16 outer products with one fused multiply-add per output
// and instruction, so a chain of them keeps router_dot's canonical order: block b of the MFMA holds
// one residue k mod 64 of the chains of 16 experts x 16 tokens, step i multiplies in k = residue +
// 64 i, and the 64 partial sums of a logit meet in the xor butterfly's tree (32 first, 1 last). The
// same bits as the VALU chains, at 2 x their FMA rate and without their conversion per product (the
// bf16 weights are widened once per 16 tokens).
//
// A workgroup is 16 tokens x up to 32 experts. Eight wavefronts take the logits: 4 residue sets (16
// residues: a float4 of x per lane and step, 4 MFMA blocks x 4 components) x 2 groups of 16 experts.
// 8 steps at a time x and the weights go through LDS: the MFMA's operands have a token or expert
// per lane, and loads of that layout straight from memory touch 64 lines an instruction (measured:
// they alone took 20 of 35 us at 1000 tokens). Four more wavefronts write the records of each staged
// tile meanwhile, so x is read from memory once.
// 4096 tokens of 2880, 32 experts: k_route 80 us -> 35 + k_group 7 (traced); 1000 tokens, one-term
// records: 39 -> 24 + 6. What is left is serial: the staging's barriers, top-k, the MFMA (a fifth).
#include <algorithm>

#include "device.hpp"
#include "kernels.hpp"

namespace moe {

constexpr int kRwTokens = 16, kRwThreads = 768, kRwMaxE = 32, kRwMaxK = 4;
constexpr int kRwMain = 512;  // the wavefronts of the logits; the others write the records

constexpr int kRwXRow = 516;  // floats of a token's row of the staged x tile (512 values), rows on distinct banks
constexpr int kRwWRow = 65;   // uint4 of an expert's row of the staged weights (64 residues x 8 steps)
constexpr size_t kRwLds = kRwTokens * kRwXRow * sizeof(float) + 32 * kRwWRow * 16;

template <int NT, bool NORM>
__global__ __launch_bounds__(kRwThreads) __attribute__((amdgpu_waves_per_eu(3, 3))) void k_route_wide(RouteArgs a) {
  extern __shared__ __attribute__((aligned(16))) float s_x[];  // [16][kRwXRow], then the weights [32][kRwWRow] uint4
  uint4 *const s_wt = reinterpret_cast<uint4 *>(s_x + kRwTokens * kRwXRow);
  // partial sums on their way across the residue sets (two components), in the staged tiles' place
  f32x4 (*const s_ex)[2][8][64] = reinterpret_cast<f32x4 (*)[2][8][64]>(s_x);
  static_assert(2 * 2 * 8 * 64 * sizeof(f32x4) <= kRwLds, "the exchange fits the tiles");
  __shared__ float s_logit[kRwTokens][kRwMaxE];
  __shared__ int s_order[kRwTokens][kMaxTopK];
  __shared__ float s_w[kRwTokens][kMaxTopK];
  __shared__ int s_sel[kRwTokens];
  __shared__ float s_r[kRwTokens];
  __shared__ int s_cnt[kRwMaxE];
  const int t0 = blockIdx.x * kRwTokens, nt = min(kRwTokens, a.T - t0);
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int H = a.H, E = a.E, nq = ((H + 63) / 64 + 7) / 8, Hp = nq * 512;
  if constexpr (NORM) {
    // rms_inv_wave's order; a wavefront's two tokens at once, 2 x 24 loads in flight
    const float *xr[2];
#pragma unroll
    for (int u = 0; u < 2; u++) xr[u] = a.x + (size_t)(t0 + min(wv + 8 * u, nt - 1)) * H;
    float p[2] = {0.0f, 0.0f};
    for (int k0 = lane; k0 < (wv < 8 ? Hp : 0); k0 += 64 * 24) {
      float v[2][24];
#pragma unroll
      for (int i = 0; i < 24; i++)
#pragma unroll
        for (int u = 0; u < 2; u++) v[u][i] = xr[u][min(k0 + 64 * i, H - 1)];
#pragma unroll
      for (int i = 0; i < 24; i++)
#pragma unroll
        for (int u = 0; u < 2; u++) {
          const float sq = v[u][i] * v[u][i];
          p[u] = p[u] + (k0 + 64 * i < H ? sq : 0.0f);  // (a zero past H adds nothing)
        }
    }
#pragma unroll
    for (int u = 0; u < 2; u++) {
      const float r = 1.0f / sqrtf(wave_sum_xor(p[u]) / (float)H + a.eps);
      if (lane == 0 && wv < 8 && wv + 8 * u < nt) s_r[wv + 8 * u] = r;
    }
    __syncthreads();
  }

  // ---- logits, and the grouped GEMM's records
  const bool main = wv < kRwMain / 64;
  const int rs = wv & 3, es = wv >> 2, col = lane & 15, blk = lane >> 4;  // es: the group of 16 experts
  const int res0 = 16 * rs + 4 * blk;  // the lane's residues res0 .. res0 + 3
  const bool mine = main && 16 * es < E;
  // staging: the thread's float4 of 4 tokens' rows, and a residue of 4 experts
  const int sk = 4 * ((int)threadIdx.x & 127), sr = (int)threadIdx.x >> 7;
  f32x16v acc[4];
  if (main) {
    f32x4 lx[4], lg;
    u32x4 lw[4];
    auto load = [&](int q) {
      const int k = min(512 * q + sk, H - 4);  // (past H: a repeat, cleared when staged)
#pragma unroll
      for (int i = 0; i < 4; i++)
        lx[i] = *reinterpret_cast<const f32x4 *>(a.x + (size_t)(t0 + min(4 * i + sr, nt - 1)) * H + k);
      if (NORM) lg = *reinterpret_cast<const f32x4 *>(a.gamma + k);
#pragma unroll
      for (int i = 0; i < 4; i++)
        lw[i] = reinterpret_cast<const u32x4 *>(a.w)[((size_t)min(8 * i + wv, E - 1) * nq + q) * 64 + lane];
    };
#pragma unroll
    for (int c = 0; c < 4; c++) acc[c] = f32x16v{};
    load(0);
    for (int q = 0; q < nq; q++) {
      __syncthreads();  // the tiles are free
      const bool in = 512 * q + sk < H;
#pragma unroll
      for (int i = 0; i < 4; i++) {
        f32x4 v = lx[i];
        if constexpr (NORM) {
          const float r = s_r[min(4 * i + sr, nt - 1)];
#pragma unroll
          for (int c = 0; c < 4; c++) {
            const float vr = v[c] * r;
            v[c] = vr * lg[c];
          }
        }
        *reinterpret_cast<f32x4 *>(s_x + (4 * i + sr) * kRwXRow + sk) = in ? v : f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        reinterpret_cast<u32x4 *>(s_wt)[(8 * i + wv) * kRwWRow + lane] = lw[i];
      }
      __syncthreads();
      if (q + 1 < nq) load(q + 1);
      if (mine) {
        uint4 w[4];
#pragma unroll
        for (int c = 0; c < 4; c++) w[c] = s_wt[(16 * es + col) * kRwWRow + res0 + c];
#pragma unroll
        for (int h = 0; h < 8; h++) {
          const float4 x4 = *reinterpret_cast<const float4 *>(s_x + col * kRwXRow + 64 * h + res0);
          const float xv[4] = {x4.x, x4.y, x4.z, x4.w};
#pragma unroll
          for (int c = 0; c < 4; c++) {
            const uint32_t u = h < 2 ? w[c].x : (h < 4 ? w[c].y : (h < 6 ? w[c].z : w[c].w));
            const float wf = bf16_to_f32((uint16_t)(u >> (16 * (h & 1))));
            acc[c] = __builtin_amdgcn_mfma_f32_16x16x1f32(wf, xv[c], acc[c], 0, 0, 0);
          }
        }
      }
    }
  } else {
    for (int q = 0; q < nq; q++) {
      __syncthreads();
      __syncthreads();  // tile q is staged
      // its 16 x 16 record blocks, a lane each (four lanes a step of a record)
      const int u = (int)threadIdx.x - kRwMain, tb = (u >> 2) & 15, b = (u & 3) + 4 * (u >> 6);
      if (a.xrec && tb < nt && 16 * q + b < 4 * kGemmNs) {
        float xv[32];
#pragma unroll
        for (int i = 0; i < 8; i++) {
          const float4 x4 = *reinterpret_cast<const float4 *>(s_x + tb * kRwXRow + 32 * b + 4 * i);
          xv[4 * i] = x4.x;
          xv[4 * i + 1] = x4.y;
          xv[4 * i + 2] = x4.z;
          xv[4 * i + 3] = x4.w;
        }
        rec_split_block<NT>(xv, 16 * q + b, a.xrec + (size_t)(t0 + tb) * GemmRecT<NT>::kBytes);
      }
    }
  }
  // the butterfly: residue bits 5 and 4 across the residue sets, 3 and 2 across the MFMA's
  // blocks (registers 4 b + row), 1 and 0 across the components
  auto put = [&](int slot, const f32x16v (&p)[4], int c0) {
#pragma unroll
    for (int c = 0; c < 2; c++)
#pragma unroll
      for (int b = 0; b < 4; b++) {
        const f32x16v &v = p[c0 + c];
        s_ex[es][slot][4 * c + b][lane] = f32x4{v[4 * b], v[4 * b + 1], v[4 * b + 2], v[4 * b + 3]};
      }
  };
  auto add = [&](int slot, f32x16v (&p)[4], int c0) {
#pragma unroll
    for (int c = 0; c < 2; c++)
#pragma unroll
      for (int b = 0; b < 4; b++) {
        const f32x4 v = s_ex[es][slot][4 * c + b][lane];
#pragma unroll
        for (int r = 0; r < 4; r++) p[c0 + c][4 * b + r] = p[c0 + c][4 * b + r] + v[r];
      }
  };
#pragma unroll
  for (int c0 = 0; c0 < 4; c0 += 2) {
    __syncthreads();  // s_ex is free
    if (mine && rs >= 2) put(rs - 2, acc, c0);
    __syncthreads();
    if (mine && rs < 2) add(rs, acc, c0);
    __syncthreads();
    if (mine && rs == 1) put(0, acc, c0);
    __syncthreads();
    if (mine && rs == 0) add(0, acc, c0);
  }
  if (mine && rs == 0) {
#pragma unroll
    for (int r = 0; r < 4; r++) {
      float v[4];
#pragma unroll
      for (int c = 0; c < 4; c++) v[c] = (acc[c][r] + acc[c][8 + r]) + (acc[c][4 + r] + acc[c][12 + r]);
      const int e = 16 * es + 4 * blk + r;
      if (e < E) s_logit[col][e] = canon_nan(((v[0] + v[2]) + (v[1] + v[3])) + a.bias[e]);
    }
  }
  __syncthreads();

  // ---- top-k, a wavefront per token
  const TopkCfg c{E, a.k, a.adaptive, a.min_k, a.top1_min, a.margin_min, a.top2_mass};
  for (int tb = wv; tb < nt; tb += kRwThreads / 64) {
    const int t = t0 + tb;
    const float l[1] = {lane < E ? s_logit[tb][lane] : 0.0f};
    if (lane < E) a.logits[(size_t)t * E + lane] = l[0];
    int ord[4];
    wave_topk_order<1>(c, l, lane, ord);
    wave_topk_weights<1>(c, l, lane, ord, true, s_order[tb], s_w[tb], &s_sel[tb]);
    if (lane < a.k) {
      const size_t o = (size_t)t * a.k + lane;
      a.idx[o] = s_order[tb][lane];
      a.wts[o] = s_w[tb][lane];
    }
  }
  if (a.xrec) {  // the records' blocks past the router's chain are zero
    const int b0 = 16 * nq, nb = max(4 * kGemmNs - b0, 0);
    const float zero[32] = {};
    for (int u = threadIdx.x; u < nt * nb; u += kRwThreads) {
      const int tb = u / nb;
      rec_split_block<NT>(zero, b0 + u - tb * nb, a.xrec + (size_t)(t0 + tb) * GemmRecT<NT>::kBytes);
    }
  }
  // ---- the block's entries per expert, and each entry's rank among them, for k_group
  if (!a.blk_count) return;
  __syncthreads();  // s_order
  if (wv == 0) {
    for (int e = lane; e < E; e += 64) s_cnt[e] = 0;
    const int tb = lane / a.k, slot = lane - tb * a.k;  // at most 64 entries
    const int e = lane < nt * a.k ? s_order[tb][slot] : -1;
    const uint32_t v = (uint32_t)(e + 1);
    uint64_t same = ~0ull;
#pragma unroll
    for (int bit = 0; bit < 8; bit++) {
      const uint64_t bb = __ballot((v >> bit) & 1u);
      same &= ((v >> bit) & 1u) ? bb : ~bb;
    }
    const uint64_t below = same & ((1ull << lane) - 1ull);
    if (e >= 0) {
      a.rank[(size_t)t0 * a.k + lane] = __popcll(below);
      if (below == 0) s_cnt[e] = __popcll(same);
    }
    for (int e2 = lane; e2 < E; e2 += 64) a.blk_count[(size_t)blockIdx.x * E + e2] = s_cnt[e2];
  }
}

// The grouping by expert, in entry order t k + slot: a workgroup scatters the entries of kGrpBlocks
// router workgroups to base + rank, every workgroup summing the count table (nblk x E, in the L2)
// itself. A launch of its own (about 4 us) instead of the last router workgroup's pass over all
// entries, whose scattered stores one CU issued.
constexpr int kGrpThreads = 1024, kGrpBlocks = 8;

__global__ __launch_bounds__(kGrpThreads) void k_group(RouteArgs a, int nblk) {
  __shared__ int s_all[kGrpThreads], s_bef[kGrpThreads];
  __shared__ int s_tot[kRwMaxE], s_base[kRwMaxE];
  __shared__ int s_pre[kGrpBlocks][kRwMaxE];
  const int E = a.E, b0 = blockIdx.x * kGrpBlocks, tid = threadIdx.x;
  const int P = kGrpThreads / E;  // parts of the table's rows
  const int part = tid / E, e = tid - part * E;
  int all = 0, bef = 0;
  if (part < P) {
    constexpr int kB = 8;
    for (int r0 = part; r0 < nblk; r0 += kB * P) {
      int v[kB];
#pragma unroll
      for (int i = 0; i < kB; i++) v[i] = r0 + i * P < nblk ? a.blk_count[(size_t)(r0 + i * P) * E + e] : 0;
#pragma unroll
      for (int i = 0; i < kB; i++) {
        all += v[i];
        bef += r0 + i * P < b0 ? v[i] : 0;
      }
    }
  }
  s_all[tid] = all;
  s_bef[tid] = bef;
  __syncthreads();
  if (tid < E) {
    int s = 0, p = 0;
    for (int q = 0; q < P; q++) {
      s += s_all[q * E + tid];
      p += s_bef[q * E + tid];
    }
    s_tot[tid] = s;
#pragma unroll
    for (int i = 0; i < kGrpBlocks; i++) {
      s_pre[i][tid] = p;
      if (b0 + i < nblk) p += a.blk_count[(size_t)(b0 + i) * E + tid];
    }
  }
  __syncthreads();
  // every workgroup derives the bases; the lists are the first one's to write
  if (tid < 64) {
    int run = 0;
    for (int q = 0; q < (E + 63) / 64; q++) {
      const int ee = 64 * q + tid, c = ee < E ? s_tot[ee] : 0;
      int incl = c;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const int u = __shfl_up(incl, o);
        if (tid >= o) incl += u;
      }
      if (ee < E) s_base[ee] = run + incl - c;
      run += __shfl(incl, 63);
    }
    if (blockIdx.x == 0) expert_list_wave(s_tot, E, tid, s_base, a.active_ids, a.active_off, a.n_active);
  }
  __syncthreads();
  const int n0 = b0 * kRwTokens * a.k, n = n0 + tid;  // kGrpBlocks * 16 tokens * k <= 512 entries
  if (tid < kGrpBlocks * kRwTokens * a.k && n < a.T * a.k) {
    const int ee = a.idx[n];
    if (ee < 0) {
      a.pos[n] = -1;
    } else {
      const int ge = s_base[ee] + s_pre[tid / (kRwTokens * a.k)][ee] + a.rank[n];
      a.entry_src[ge] = n / a.k;
      a.pos[n] = ge;
    }
  }
}

// Where it is ahead of k_route: its 16-token workgroups need the tokens to fill the CUs, and k_group
// is a launch that few entries over few experts hardly repay (a whole layer of H x I, E experts, k
// chosen, us, k_route against this):
//   768 tokens   3072 x 96, E 4, k 1  69.6 / 76.4;  2880 x 2880, E 8, k 1  96.9 / 101.1;  512 x 3072, E 2,
//                k 1  68.9 / 73.3;  1024 x 512, E 16, k 2  58.1 / 54.5: behind for more shapes than not
//   896 tokens   E k >= 8: 1024 x 512, E 8, k 4  66.6 / 59.6;  3072 x 96, E 8, k 1  75.0 / 75.4.  E k < 8:
//                level to 4 % behind, as at 1024 tokens (3072 x 96, E 2, k 1  79.0 / 79.6, E 4 3 % behind)
//   1100 tokens  k_route's token per workgroup, two to a CU, is in its third round: 0 to 22 % ahead
//   2048 tokens  k_route's 8-token workgroups fill the CUs exactly once. E k < 8: 3072 x 96, E 2, k 1
//                78.8 / 84.3, 2880 x 2880 141.6 / 147.2 (2200 tokens of 3072 x 96: 92.9 / 85.3); level from E k = 8 on
// More than 32 experts would need a pass over x for each 32, at which it was no faster (2048 tokens,
// 128 experts: 79 / 82 + 8).
static bool route_wide_ahead(int T, int E, int k) {
  return E * k < 8 ? T > 1024 && T != 2048 : T >= 896;
}

bool route_wide_fits(const RouteArgs &a) {
  return route_wide_ahead(a.T, a.E, a.k) && a.E <= kRwMaxE && a.k <= kRwMaxK && a.H % 32 == 0 && a.H <= 128 * kGemmNs && !a.xsplit &&
         !a.fuse_bucket && (reinterpret_cast<uintptr_t>(a.x) & 15) == 0;
}

template <int NT, bool NORM>
static hipError_t launch_wide(const RouteArgs &a, hipStream_t s) {
  static DynLdsOnce once;
  const hipError_t e = ensure_dyn_lds(once, reinterpret_cast<const void *>(&k_route_wide<NT, NORM>), kRwLds);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((k_route_wide<NT, NORM>), dim3((a.T + kRwTokens - 1) / kRwTokens), dim3(kRwThreads), kRwLds, s, a);
  return hipGetLastError();
}

hipError_t launch_route_wide(RouteArgs a, bool group, hipStream_t s) {
  if (!route_wide_fits(a) || a.E < 1 || a.k < 1 || a.k > a.E || (group && (!a.blk_count || !a.rank)))
    return hipErrorInvalidValue;
  if (!group) a.blk_count = nullptr;
  hipError_t e = hipErrorInvalidValue;
  switch (a.xrec ? a.rec_terms : kGemmTerms) {
    case 1: e = a.gamma ? launch_wide<1, true>(a, s) : launch_wide<1, false>(a, s); break;
    case kGemmTerms: e = a.gamma ? launch_wide<kGemmTerms, true>(a, s) : launch_wide<kGemmTerms, false>(a, s); break;
  }
  if (e != hipSuccess) return e;
  if (group) {
    const int nblk = (a.T + kRwTokens - 1) / kRwTokens;
    hipLaunchKernelGGL(k_group, dim3((nblk + kGrpBlocks - 1) / kGrpBlocks), dim3(kGrpThreads), 0, s, a, nblk);
  }
  return hipGetLastError();
}

}  // namespace moe
