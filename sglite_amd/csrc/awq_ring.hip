// W4A16 GEMM for 17-64 rows: many waves per workgroup, the activations through
// a two-slot ring of k-steps in LDS.
//
// A workgroup owns NTW * WN column tiles (with a gated activation half of them
// gate tiles, the others their up tiles) and all M rows; WN * WK waves.  Wave
// (wn, kw) owns NTW of the tiles and every WK-th k-tile, so a step is WK
// k-tiles and the WN waves of a k-tile share its activations.  A step's
// weights, zero points and scales (registers) and activations (LDS-DMA into
// the ring) are in flight during the step before it.  The WK partial sums meet
// in LDS at the end.  K stays unsplit where the column tiles give enough
// workgroups (qkv and gate_up of Qwen3-4B and Llama-3-8B); their o and down
// leave K in 3 to 6 slices, summed by a second launch (3-5 us) as the tiled
// plans' 4 to 16 are.
//
// What bounds these shapes is not the weight stream but the dequantisation,
// LDS reads and MFMAs of a k-tile following one another: the tiled kernels put
// four waves on a CU here, one per SIMD.  With 8 to 16 waves on a CU the units
// overlap.  Measured against them (graph replay, us; floor at the copy rate of
// 4.8 TB/s in brackets): Qwen3-4B at M = 32, fp16, qkv 11.5 -> 8.2 (1.7), o
// 10.9 -> 8.2 (1.1), gate_up 16.7 -> 13.4 (5.4), down 12.7 -> 11.3 (2.7);
// Llama-3-8B at M = 64 qkv 15.7 -> 13.1 (2.7), o 14.1 -> 11.9 (1.8), gate_up
// 34.8 -> 27.0 (12.5), down 20.7 -> 20.0 (6.3: alone on the device its GEMM is
// a little longer than the tiled one, 17.9 against 16.6).  Tried: four slots,
// three steps ahead, with half the waves (gate_up at M = 64 27.6 against 25.2);
// four tiles per wave and half the waves, which halves the LDS reads (26.0
// against 25.2); one m-tile at M = 8, where the GEMV and decode kernels stay
// ahead (qkv 5.9 against 5.7).
#include <algorithm>

#include "awq_buffer.h"
#include "awq_epilogue.h"
#include "awq_launch.h"

namespace sgl_awq {

namespace {

constexpr int kRingLds = 160 * 1024;

struct RingArgs {
  const void* x;
  const void* w;
  const void* s;
  const void* z;
  const void* bias;
  void* out;
  float* part;
  int M, N, K, NT, KT, NG, gshift;
  int ktc, ks;  // k-tiles per slice, slices
  int WN, WK, act;
};

// x slots: [k-tile of the step][row][16 chunks of 16 bytes], chunk q of row r
// at position q ^ (r & 15): a DMA instruction brings four rows of 256
// contiguous bytes, and the 16 rows that a fragment read touches at one chunk
// lie in 16 different positions.
template <int MT, int NTW, int NX, int GPT, typename DT>
__global__ __launch_bounds__(1024, 4) void ring_kernel(RingArgs a) {
  using E = typename DT::elem;
  using V8 = typename DT::vec8;
  constexpr int XT = MT * 256;  // 16-byte vectors of one k-tile's activations
  extern __shared__ u32x4 ring[];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int WN = a.WN, WK = a.WK;
  const int wn = wave % WN, kw = wave / WN;
  const int c = lane & 15, lg = lane >> 4;
  const bool paired = a.act != kActNone;
  const int half = a.NT >> 1;
  constexpr int HT = NTW > 1 ? NTW / 2 : 1;  // gate tiles of a wave with a gated activation
  WTiles<NTW, GPT> wt;
  wt.KT = a.KT;
  wt.NG = a.NG;
  wt.gshift = a.gshift;
  wt.set_matrix(a.w, a.s, a.z, a.NT);
#pragma unroll
  for (int j = 0; j < NTW; ++j) {
    const int t = paired ? (blockIdx.x * WN + wn) * HT + j % HT + j / HT * half : (blockIdx.x * WN + wn) * NTW + j;
    wt.set_tile(j, t, t < (paired ? half + j / HT * half : a.NT));
  }
  const int kt_begin = blockIdx.y * a.ktc, kt_end = min(kt_begin + a.ktc, a.KT);
  const int steps = (kt_end - kt_begin + WK - 1) / WK;
  const DqK dk = dq_consts();

  const __amdgpu_buffer_rsrc_t xr = make_rsrc(a.x, (uint32_t)a.M * (uint32_t)a.K * 2u);

  // The wave's share of its k-tile's activations: NX groups of four rows (a
  // group past the last repeats it, so that every wave counts NX loads).
  uint32_t xoff[NX];
  int xdst[NX], xk[NX];
#pragma unroll
  for (int i = 0; i < NX; ++i) {
    const int rg = min(wn + i * WN, MT * 4 - 1);
    const int row = rg * 4 + (lane >> 4);
    const int q = (lane & 15) ^ (row & 15);
    xoff[i] = row < a.M ? ((uint32_t)row * (uint32_t)a.K + (uint32_t)q * 8u) * 2u : kPastEnd;
    xk[i] = q * 8;
    xdst[i] = rg * 64;
  }

  using Stage = WStage16<NTW, GPT>;
  // Step i's loads in the order the wait counts rely on: activations, weights.
  auto issue = [&](Stage& st, int i, int slot) {
    const int kt = kt_begin + i * WK + kw;
    const uint32_t dead = kt < kt_end ? 0u : kPastEnd;
    u32x4* dst = ring + (slot * WK + kw) * XT;
#pragma unroll
    for (int n = 0; n < NX; ++n) {
      const uint32_t off = kt * 128 + xk[n] < a.K ? xoff[n] | dead : kPastEnd;
      load_lds16(xr, dst + xdst[n], off, kt * 256);
    }
    __builtin_amdgcn_sched_barrier(0);
    wt.load(st, kt, dead, lane);
    __builtin_amdgcn_sched_barrier(0);
  };

  f32x4 acc[MT][NTW];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int j = 0; j < NTW; ++j) acc[mt][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  auto mul = [&](const Stage& st, const u32x4* xs) {
    typename Dq<DT>::ZS zs[NTW][GPT];
    st.template zero_scale<DT>(lane, zs);
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      V8 b[MT];
      const int at = c * 16 + ((w * 4 + lg) ^ c);
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) b[mt] = __builtin_bit_cast(V8, xs[mt * 256 + at]);
#pragma unroll
      for (int j = 0; j < NTW; ++j) {
        const V8 v = Dq<DT>::word(st.q[j][w], zs[j][w / wt.BPG], dk);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) acc[mt][j] = mfma16x16x32(v, b[mt], acc[mt][j]);
      }
    }
  };

  // Step i: wait until its loads have landed, meet the other waves at a bare
  // barrier -- every wave's share of the step is in LDS then, and every wave is
  // done with step i - 1, whose slot step i + 1 takes -- and issue step i + 1.
  // The step past the last loads zeros and is never multiplied.  The loop
  // leaves by a branch past no load, so each stage keeps its registers.
  Stage st[2];
  issue(st[0], 0, 0);
  [&] {
    for (int i = 0;;) {
#pragma unroll
      for (int d = 0; d < 2; ++d) {
        __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        issue(st[1 - d], i + 1, 1 - d);
        mul(st[d], ring + (d * WK + kw) * XT);
        if (++i >= steps) return;
      }
    }
  }();

  // The k-waves' partial sums, in the ring's space once its last loads landed
  // and every wave is done with it.
  __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
  __syncthreads();
  f32x4* red = (f32x4*)ring;
  const int NQ = WN * NTW * MT * 64;
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int j = 0; j < NTW; ++j) red[kw * NQ + ((wn * NTW + j) * MT + mt) * 64 + lane] = acc[mt][j];
  __syncthreads();
  auto sum = [&](int q) {
    f32x4 v = red[q];
    for (int o = 1; o < WK; ++o) v += red[o * NQ + q];
    return v;
  };
  const int64_t Np = (int64_t)a.NT * 16;
  float* part = a.part + (int64_t)blockIdx.y * a.M * Np;
  // Quad q: lane l = q % 64 of fragment (wn', j, mt) holds row 16 mt + l % 16
  // and columns 4 (l / 16) .. + 3.
  const bool gate = paired && a.ks == 1;
  const int per = gate ? WN * HT * MT * 64 : NQ;
  for (int q = threadIdx.x; q < per; q += blockDim.x) {
    const int l = q & 63, f = q >> 6;
    const int mt = f % MT, m = mt * 16 + (l & 15), c4 = 4 * (l >> 4);
    if (m >= a.M) continue;
    if (gate) {
      const int w = f / MT / HT, j = f / MT % HT;
      const int t = (blockIdx.x * WN + w) * HT + j;
      if (t >= half) continue;
      const int q0 = ((w * NTW + j) * MT + mt) * 64 + l;
      store4_act<DT>((E*)a.out, (const E*)a.bias, m, a.N >> 1, t * 16 + c4, a.N >> 1, sum(q0),
                     sum(q0 + HT * MT * 64), a.act);
    } else {
      const int w = f / MT / NTW, j = f / MT % NTW;
      const int t = paired ? (blockIdx.x * WN + w) * HT + j % HT : (blockIdx.x * WN + w) * NTW + j;
      if (t >= (paired ? half : a.NT)) continue;
      const int n0 = (paired ? t + j / HT * half : t) * 16 + c4;
      const f32x4 v = sum(q);
      if (a.ks > 1) *(f32x4*)(part + m * Np + n0) = v;
      else if (n0 < a.N) store4<DT>((E*)a.out, (const E*)a.bias, m, a.N, n0, v);  // N % 16 == 8: half a tile
    }
  }
}

template <int MT, int NTW, int NX, int GPT, typename DT>
hipError_t launch_form(const RingArgs& a, dim3 grid, hipStream_t s) {
  const int lds = std::max(2 * a.WK * MT * 4096, a.WK * a.WN * NTW * MT * 1024);
  hipLaunchKernelGGL((ring_kernel<MT, NTW, NX, GPT, DT>), grid, dim3(64 * a.WN * a.WK), lds, s, a);
  return hipGetLastError();
}

template <int MT, int NTW, typename DT>
hipError_t launch_ring_f(const RingArgs& a, int gpt, dim3 grid, hipStream_t s) {
  const int nx = (MT * 4 + a.WN - 1) / a.WN;
#define SGL_RING(NX_)                                                           \
  if (nx <= NX_) {                                                              \
    if (gpt == 1) return launch_form<MT, NTW, NX_, 1, DT>(a, grid, s);          \
    if (gpt == 2) return launch_form<MT, NTW, NX_, 2, DT>(a, grid, s);          \
    return launch_form<MT, NTW, NX_, 4, DT>(a, grid, s);                        \
  }
  if constexpr (NTW > 1) {
    SGL_RING(MT)
  }
  SGL_RING(MT * 2)
  SGL_RING(MT * 4)
#undef SGL_RING
  return hipErrorInvalidValue;
}

}  // namespace

// Shapes that are instantiated: at most 16 waves, both ring slots within LDS;
// one tile a wave in at most three column waves (the planner takes more than
// two tiles as two a wave).
bool ring_variant_ok(int code, int act) {
  const int mt = code / 100000, ntw = code / 10000 % 10, wn = code / 100 % 10, wk = code % 100;
  return code > 0 && (ntw == 2 || wn <= 3) && code % 10000 < 1000 && mt >= 2 && mt <= 4 && (ntw == 2 || (ntw == 1 && !act)) && wn >= 1 && wk >= 1 &&
         wn * wk <= 16 && 2 * wk * mt * 4096 <= kRingLds;
}

// Workgroups of a launch: column-tile groups times k-slices.
dim3 ring_grid(const GemmPlan& p, const Geom& g, int act) {
  const int ntw = p.ring / 10000 % 10, wn = p.ring / 100 % 10;
  const int64_t tiles = act ? g.NT / 2 : g.NT, per = (int64_t)wn * (act ? ntw / 2 : ntw);
  return dim3((unsigned)((tiles + per - 1) / per), (unsigned)p.ring_ks);
}

hipError_t launch_ring(const GemmPlan& p, const void* x, const void* w, const void* sr, const void* zr,
                       const void* bias, void* out, int dtype, const Geom& g, void* ws, int act, hipStream_t s) {
  RingArgs a{};
  a.x = x;
  a.w = w;
  a.s = sr;
  a.z = zr;
  a.bias = bias;
  a.out = out;
  a.part = (float*)ws;
  a.M = (int)g.M;
  a.N = (int)g.N;
  a.K = (int)g.K;
  a.NT = (int)g.NT;
  a.KT = (int)g.KT;
  a.NG = (int)g.NG;
  a.gshift = g.gshift;
  a.ktc = p.ring_ktc;
  a.ks = p.ring_ks;
  a.WN = p.ring / 100 % 10;
  a.WK = p.ring % 100;
  a.act = act;
  const int mt = p.ring / 100000, ntw = p.ring / 10000 % 10;
  if (g.M > mt * 16 || !ring_variant_ok(p.ring, act)) return hipErrorInvalidValue;
  const int gpt = (g.NG > 1 && g.G < 128) ? (int)(128 / g.G) : 1;
  const dim3 grid = ring_grid(p, g, act);
  hipError_t e = hipErrorInvalidValue;
#define SGL_F(MT_, NTW_)                                                                          \
  if (mt == MT_ && ntw == NTW_)                                                                   \
    e = dtype == 0 ? launch_ring_f<MT_, NTW_, F16>(a, gpt, grid, s) : launch_ring_f<MT_, NTW_, BF16>(a, gpt, grid, s);
  SGL_F(2, 1)
  SGL_F(2, 2)
  SGL_F(3, 1)
  SGL_F(3, 2)
  SGL_F(4, 1)
  SGL_F(4, 2)
#undef SGL_F
  if (e != hipSuccess || p.ring_ks == 1) return e;
  return launch_splitk_reduce((const float*)ws, bias, out, g, p.ring_ks, act, dtype, s);
}

}  // namespace sgl_awq
