// Grouped W4A16 MoE GEMM for few routed rows per expert (decode batches):
// one workgroup per (16-row block of an expert, column-tile group), K split
// over its waves (awq_kwave.h).
//
// The pipelined grouped kernel (awq_moe.hip) runs several column slices of an
// expert per workgroup and sizes that for every expert being busy.  With few
// tokens only min(E, T * k) experts have rows, each a handful, and the work is
// reading their weights once: this form starts one workgroup per block of the
// sorted rows, so its grid is as large as the work, and every wave has its
// k-tiles' loads in flight as soon as it knows its expert.
#include <math.h>

#include <algorithm>

#include "awq_epilogue.h"
#include "awq_kwave.h"
#include "awq_launch.h"

namespace sgl_awq {

namespace {

struct RowsArgs {
  const void* x;
  uint32_t x_bytes;        // activation bytes the routed rows span (below 2^31: the host checks)
  const u32x4* wt;
  const uint16_t* s_r;
  const uint64_t* z_r;
  const int32_t* sorted;
  const int32_t* offsets;  // padded bucket offsets [E + 1]
  const float* topk_w;
  void* out;
  int a_div, num_routed, sorted_cap, E;
  int N, K, NT, KT, NG, gshift;
  int64_t w_stride, s_stride, z_stride;
  int mul_rw;
};

typedef int i32x4u __attribute__((ext_vector_type(4), aligned(4)));  // four offsets, aligned as one

// The 16-row blocks of the experts' buckets, counted over the experts in
// order.  One lane per EPL (2 or 8) experts; every wave of a workgroup finds
// its blocks by itself.
template <int EPL>
struct Blocks {
  int r0[EPL], nb[EPL];  // first sorted row and blocks of the lane's experts
  int excl, incl;        // blocks before the lane's first expert and past its last one

  __device__ __forceinline__ void scan(const RowsArgs& a, int lane) {
    int o[EPL + 1];
    if (EPL % 4 == 0 && a.E % EPL == 0) {
      // Vectors of the lanes' own experts (lanes past the last expert reload
      // the last ones'): nine loads of 32-byte stride a lane cost a CU whose 16
      // waves all look for their blocks about 1 us (E = 512, K = 1024, N = 512
      // gated at 256 rows 30.6 -> 22.8 us).
      const int e0 = min(lane * EPL, a.E - EPL);
#pragma unroll
      for (int i = 0; i < EPL / 4; ++i) {
        const i32x4u v = *(const i32x4u*)(a.offsets + e0 + 4 * i);
#pragma unroll
        for (int k = 0; k < 4; ++k) o[4 * i + k] = v[k];
      }
      o[EPL] = a.offsets[e0 + EPL];
    } else {
#pragma unroll
      for (int i = 0; i <= EPL; ++i) o[i] = a.offsets[min(lane * EPL + i, a.E)];
    }
    int sum = 0;
#pragma unroll
    for (int i = 0; i < EPL; ++i) {
      r0[i] = min(max(o[i], 0), a.sorted_cap);
      const int r1 = min(max(o[i + 1], r0[i]), a.sorted_cap);
      nb[i] = lane * EPL + i < a.E ? (r1 - r0[i]) >> 4 : 0;
      sum += nb[i];
    }
    incl = sum;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int u = __shfl_up(incl, d);
      if (lane >= d) incl += u;
    }
    excl = incl - sum;
  }

  // Block b's expert and first sorted row; e = -1 past the last block.
  __device__ __forceinline__ void find(int b, int lane, int& e, int& rb) const {
    const uint64_t hit = __ballot(b >= excl && b < incl);
    if (hit == 0) {
      e = -1;
      return;
    }
    int fe = 0, fr = 0, pos = excl;
#pragma unroll
    for (int i = 0; i < EPL; ++i) {
      if (b >= pos && b < pos + nb[i]) {
        fe = lane * EPL + i;
        fr = r0[i] + (b - pos) * 16;
      }
      pos += nb[i];
    }
    const int src = __builtin_ctzll(hit);
    e = __builtin_amdgcn_readlane(fe, src);
    rb = __builtin_amdgcn_readlane(fr, src);
  }
};

// Two column tiles per workgroup (with a gate/up activation one gate tile and
// its up tile), kMaxWaves waves at most, which split K.  What bounds it is the
// chain of a short workgroup -- offsets, then weights and rows, then the sum --
// against the few workgroups that few rows give, so tiles and waves are few and
// workgroups many: four waves while the blocks are fewer than half the experts,
// two beyond, where more resident workgroups hide the chain better (E = 128,
// H = 2048, I = 768 top-8 fp16, a block's whole forward at T = 1 / 4 / 8 / 16:
// four waves 25.6 / 39.7 / 55.1 / 76.6 us, two 27.6 / 37.1 / 50.5 / 65.6, and
// 55.0 / 55.2 / 67.3 / 74.4 in the pipelined kernel: the two cross between 8 and
// 32 rows here, below the line).  Four tiles at four waves cost 3% at T = 1, and
// 5% at T = 16 against two at two.
constexpr int kTiles = 2;
constexpr int kMaxWaves = 4;

template <int EPL, int GPT, int ACT, typename DT>
__global__ __launch_bounds__(64 * kMaxWaves, GPT < 4 && EPL <= 2 ? 4 : 3) void moe_rows_kernel(RowsArgs a) {
  using E = typename DT::elem;
  using V4 = typename DT::vec4;
  constexpr int NTW = kTiles;
  constexpr int HT = ACT == kActNone ? NTW : NTW / 2;  // tiles in each half
  constexpr int NQ = NTW * 64;                         // 4-column quads of a block
  __shared__ f32x4 red[kMaxWaves * NQ];
  const int WK = blockDim.x >> 6;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int c = lane & 15;
  const int tile0 = blockIdx.x * HT;
  const int kt0 = wave * a.KT / WK, kt1 = (wave + 1) * a.KT / WK;

  // The first block's rows are fetched along with the offsets: blocks of a
  // table that starts at 0 without gaps start at 16 b.
  const int c0 = blockIdx.y * 16 + c;
  const int sid0 = c0 < a.sorted_cap ? a.sorted[c0] : -1;
  Blocks<EPL> blocks;
  blocks.scan(a, lane);
  for (int b = blockIdx.y;; b += gridDim.y) {
    int e, rb;
    blocks.find(b, lane, e, rb);
    if (e < 0) break;  // the same in every wave
    const int sid = rb + c == c0 ? sid0 : a.sorted[rb + c];  // rb + 16 <= sorted_cap
    const bool valid = sid >= 0 && sid < a.num_routed;
    // Padding alone (a table padded to more than 16 rows): the same in every
    // wave.  Multiplying it by zeros cost a pass over the weights a block, more
    // than the pipelined kernel's 64-row passes over it (E = 128, K = 2048, N =
    // 1536 top-8 silu fp16, tables of 64 rows: T = 8 66.8 -> 37.3 us, 52.9
    // there; T = 16 94.2 -> 45.5, 53.9; of 256 rows at T = 8 272 -> 88, 193).
    if (__ballot(valid) == 0) continue;
    const float rw = a.mul_rw && valid ? a.topk_w[sid] : 1.f;

    KWave<NTW, GPT, DT> kw;
    kw.w.KT = a.KT;
    kw.w.NG = a.NG;
    kw.w.gshift = a.gshift;
    kw.w.set_matrix(a.wt + e * a.w_stride, a.s_r + e * a.s_stride, a.z_r + e * a.z_stride, a.NT);
    const int half = ACT == kActNone ? a.NT : a.NT >> 1;
#pragma unroll
    for (int j = 0; j < NTW; ++j) {
      const int t = tile0 + j % HT;
      kw.w.set_tile(j, t + j / HT * half, t < half);
    }
    kw.K = a.K;
    kw.lane = lane;
    kw.dk = dq_consts();
    kw.xr = make_rsrc(a.x, a.x_bytes);
    kw.xoff = valid ? (uint32_t)(sid / a.a_div) * (uint32_t)a.K * 2u + (uint32_t)(lane >> 4) * 16u : kPastEnd;
    f32x4 acc[NTW];
#pragma unroll
    for (int j = 0; j < NTW; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
    kw.template run<2>(kt0, kt1, acc);

#pragma unroll
    for (int j = 0; j < NTW; ++j) red[wave * NQ + j * 64 + lane] = acc[j];
    __syncthreads();
    // Wave w sums and stores tiles w, w + WK, ... of the group: lane (c, lg)
    // holds row c of the block and columns 4 lg .. 4 lg + 3.
    auto sum = [&](int j) {
      f32x4 v = red[j * 64 + lane];
      for (int o = 1; o < WK; ++o) v += red[o * NQ + j * 64 + lane];
      return v;
    };
    E* out = (E*)a.out;
    for (int j = wave; j < HT; j += WK) {
      const int t = tile0 + j, n0 = t * 16 + 4 * (lane >> 4);
      const f32x4 g = sum(j);
      V4 r;
      if constexpr (ACT == kActNone) {
        if (valid && n0 < a.N) {  // N % 16 == 8: half of the last tile
#pragma unroll
          for (int i = 0; i < 4; ++i) r[i] = (E)(g[i] * rw);
          *(V4*)(out + (int64_t)sid * a.N + n0) = r;
        }
      } else {
        // Gate and up are rounded before the activation (fused.py:175-177).
        const f32x4 u = sum(j + HT);
        if (valid && t < half) {
#pragma unroll
          for (int i = 0; i < 4; ++i)
            r[i] = (E)(gated_act(ACT, (float)(E)(g[i] * rw)) * (float)(E)(u[i] * rw));
          *(V4*)(out + (int64_t)sid * (a.N >> 1) + n0) = r;
        }
      }
    }
    __syncthreads();  // before the next block's partial sums
  }
}

template <int EPL, typename DT>
hipError_t launch_rows(const RowsArgs& a, int gpt, int act, dim3 grid, int waves, hipStream_t s) {
#define SGL_ROWS(GPT_, ACT_)                                                                                  \
  if (gpt == GPT_ && act == ACT_) {                                                                           \
    hipLaunchKernelGGL((moe_rows_kernel<EPL, GPT_, ACT_, DT>), grid, dim3(64 * waves), 0, s, a);              \
    return hipGetLastError();                                                                                 \
  }
#define SGL_ROWS_G(GPT_) SGL_ROWS(GPT_, kActNone) SGL_ROWS(GPT_, kActSilu) SGL_ROWS(GPT_, kActGelu)
  SGL_ROWS_G(1)
  SGL_ROWS_G(2)
  SGL_ROWS_G(4)
#undef SGL_ROWS_G
#undef SGL_ROWS
  return hipErrorInvalidValue;
}

}  // namespace

int moe_rows_waves(const MoeGemmParams& p) { return 2 * p.num_routed > p.E ? 2 : kMaxWaves; }

int64_t moe_rows_groups(const MoeGemmParams& p) {
  const int64_t ht = p.epi ? kTiles / 2 : kTiles, cols = p.epi ? p.g.NT / 2 : p.g.NT;
  return (cols + ht - 1) / ht;
}

hipError_t launch_moe_rows(const MoeGemmParams& p, hipStream_t s) {
  RowsArgs a{};
  a.x = p.x;
  a.x_bytes = (uint32_t)((p.num_routed + p.a_div - 1) / p.a_div * p.g.K * 2);
  a.wt = (const u32x4*)p.w;
  a.s_r = (const uint16_t*)p.s;
  a.z_r = (const uint64_t*)p.z;
  a.sorted = p.sorted;
  a.offsets = p.offsets;
  a.topk_w = p.topk_w;
  a.out = p.out;
  a.a_div = (int)p.a_div;
  a.num_routed = (int)p.num_routed;
  a.sorted_cap = (int)p.sorted_cap;
  a.E = (int)p.E;
  a.N = (int)p.g.N;
  a.K = (int)p.g.K;
  a.NT = (int)p.g.NT;
  a.KT = (int)p.g.KT;
  a.NG = (int)p.g.NG;
  a.gshift = p.g.gshift;
  const MoeStrides st = moe_expert_strides(p.g);
  a.w_stride = st.w / 16;
  a.s_stride = st.s / 2;
  a.z_stride = st.z / 8;
  a.mul_rw = p.mul_rw;
  const int gpt = (p.g.NG > 1 && p.g.G < 128) ? (int)(128 / p.g.G) : 1;
  const int waves = moe_rows_waves(p);
  // At most one block with rows per routed row; each block of a table padded to 16 rows has one.
  const dim3 grid((unsigned)moe_rows_groups(p), (unsigned)p.num_routed);
#define SGL_EPL(N_)                                                               \
  (p.dtype == 0 ? launch_rows<N_, F16>(a, gpt, p.epi, grid, waves, s)             \
                : launch_rows<N_, BF16>(a, gpt, p.epi, grid, waves, s))
  return p.E <= 128 ? SGL_EPL(2) : SGL_EPL(8);
#undef SGL_EPL
}

}  // namespace sgl_awq
