// K split over the waves of a workgroup, activations straight from global
// memory into MFMA operands: the inner loop of the decode forms that stage
// nothing (awq_moe_rows.hip).
//
// A wave owns NTW column tiles, MT m-tiles of 16 activation rows and its own
// k-tiles [kt0, kt1).  No other wave of the workgroup reads those activations
// at those k, so staging them in LDS would share nothing: it would only put a
// copy and a barrier between the loads and the MFMAs.  Each lane loads its B
// fragment (row lane % 16, 8 consecutive k of lane / 16) as one 16-byte vector
// per k-block; lanes of padding rows read past the buffer range, which returns
// zeros without a memory access.  Waves run without any barrier until the
// partial sums meet in LDS.
#pragma once

#include "awq_buffer.h"
#include "awq_device.h"

namespace sgl_awq {

// Offset past every buffer range (ranges stay below 2^31): such a load returns zeros.
constexpr uint32_t kPastEnd = 0x80000000u;

// One k-tile of a wave in registers.
template <int MT, int NTW, int GPT>
struct KwStage {
  u32x4 q[NTW];          // weight words
  uint32_t z[NTW][GPT];  // zero-point word holding the lane's nibble
  uint16_t s[NTW][GPT];  // scale bits
  u32x4 x[MT][4];        // B fragments of the four k-blocks
};

template <int MT, int NTW, int GPT, typename DT>
struct KWave {
  using V8 = typename DT::vec8;
  using Stage = KwStage<MT, NTW, GPT>;
  static constexpr int BPG = 4 / GPT;  // k-blocks per quantisation group

  __amdgpu_buffer_rsrc_t xr, wr, zr, sr;  // activation rows; the matrix's weights, zeros, scales
  uint32_t xoff[MT];                      // byte offset of the lane's row and k, or kPastEnd
  uint32_t tile[NTW];                     // column tiles of the wave
  uint32_t past[NTW];                     // kPastEnd for a tile the matrix does not have, else 0
  int K, KT, NG, gshift, lane;
  DqK dk;

  __device__ __forceinline__ void set_matrix(const void* w, const void* s, const void* z, int NT) {
    wr = make_rsrc(w, (uint32_t)NT * (uint32_t)KT * 1024u);
    zr = make_rsrc(z, (uint32_t)NT * (uint32_t)NG * 8u);
    sr = make_rsrc(s, (uint32_t)NT * (uint32_t)NG * 32u);
  }
  __device__ __forceinline__ void set_tile(int j, int nt, bool in) {
    tile[j] = in ? nt : 0;
    past[j] = in ? 0u : kPastEnd;
  }

  // k-tile kt; `live` false (past the wave's range) loads zeros without memory traffic.
  __device__ __forceinline__ void load(Stage& st, int kt, bool live) const {
    const uint32_t dead = live ? 0u : kPastEnd;
    const uint32_t wo = (uint32_t)lane * 16u | dead;
    const uint32_t zo = (uint32_t)((lane & 15) >> 3) * 4u | dead;
    const uint32_t so = (uint32_t)(lane & 15) * 2u | dead;
#pragma unroll
    for (int j = 0; j < NTW; ++j)
      st.q[j] = __builtin_amdgcn_raw_buffer_load_b128(wr, wo | past[j], (tile[j] * KT + kt) * 1024, kCacheStream);
#pragma unroll
    for (int gg = 0; gg < GPT; ++gg) {
      const int g = min((kt * 128 + 32 * BPG * gg) >> gshift, NG - 1);
#pragma unroll
      for (int j = 0; j < NTW; ++j) {
        st.z[j][gg] = __builtin_amdgcn_raw_buffer_load_b32(zr, zo | past[j], (tile[j] * NG + g) * 8, 0);
        st.s[j][gg] = __builtin_amdgcn_raw_buffer_load_b16(sr, so | past[j], (tile[j] * NG + g) * 32, 0);
      }
    }
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      // k-blocks past K (K is a multiple of 32) read zeros.
      const uint32_t off = kt * 128 + w * 32 < K ? dead : kPastEnd;
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
        st.x[mt][w] = __builtin_amdgcn_raw_buffer_load_b128(xr, xoff[mt] | off, kt * 256 + w * 64, 0);
    }
  }

  __device__ __forceinline__ void mul(const Stage& st, f32x4 (&acc)[MT][NTW]) const {
    typename Dq<DT>::ZS zs[NTW][GPT];
#pragma unroll
    for (int gg = 0; gg < GPT; ++gg)
#pragma unroll
      for (int j = 0; j < NTW; ++j) zs[j][gg] = Dq<DT>::make((st.z[j][gg] >> (4 * (lane & 7))) & 0xFu, st.s[j][gg]);
#pragma unroll
    for (int w = 0; w < 4; ++w)
#pragma unroll
      for (int j = 0; j < NTW; ++j) {
        const V8 a = Dq<DT>::word(st.q[j][w], zs[j][w / BPG], dk);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) acc[mt][j] = mfma16x16x32(a, __builtin_bit_cast(V8, st.x[mt][w]), acc[mt][j]);
      }
  }

  // acc += k-tiles [kt0, kt1), D - 1 of them in flight ahead of the multiply.
  // The loop leaves by a branch between steps, past no load, so every stage
  // keeps its registers.
  template <int D>
  __device__ __forceinline__ void run(int kt0, int kt1, f32x4 (&acc)[MT][NTW]) const {
    Stage st[D];
#pragma unroll
    for (int p = 0; p + 1 < D; ++p) load(st[p], kt0 + p, kt0 + p < kt1);
    for (int kt = kt0; kt < kt1;) {
#pragma unroll
      for (int i = 0; i < D; ++i) {
        load(st[(i + D - 1) % D], kt + D - 1, kt + D - 1 < kt1);
        __builtin_amdgcn_sched_barrier(0);  // the prefetch stays ahead of this k-tile's math
        mul(st[i], acc);
        if (++kt >= kt1) break;
      }
    }
  }
};

}  // namespace sgl_awq
