// K split over the waves of a workgroup, activations straight from global
// memory into MFMA operands: the inner loop of the decode forms that stage
// nothing (awq_moe_rows.hip).
//
// A wave owns NTW column tiles, one m-tile of 16 activation rows and its own
// k-tiles [kt0, kt1).  No other wave of the workgroup reads those activations
// at those k, so staging them in LDS would share nothing: it would only put a
// copy and a barrier between the loads and the MFMAs.  Each lane loads its B
// fragment (row lane % 16, 8 consecutive k of lane / 16) as one 16-byte vector
// per k-block; lanes of padding rows read past the buffer range.  Waves run
// without any barrier until the partial sums meet in LDS.
#pragma once

#include "awq_buffer.h"
#include "awq_device.h"

namespace sgl_awq {

template <int NTW, int GPT, typename DT>
struct KWave {
  using V8 = typename DT::vec8;
  // One k-tile of a wave in registers.
  struct Stage {
    WStage16<NTW, GPT> w;
    u32x4 x[4];  // B fragments of the four k-blocks
  };

  WTiles<NTW, GPT> w;
  __amdgpu_buffer_rsrc_t xr;  // activation rows
  uint32_t xoff;              // byte offset of the lane's row and k, or kPastEnd
  int K, lane;
  DqK dk;

  // k-tile kt; `live` false (past the wave's range) loads zeros.
  __device__ __forceinline__ void load(Stage& st, int kt, bool live) const {
    const uint32_t dead = live ? 0u : kPastEnd;
    w.load(st.w, kt, dead, lane);
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      // k-blocks past K (K is a multiple of 32) read zeros.
      const uint32_t off = kt * 128 + b * 32 < K ? dead : kPastEnd;
      st.x[b] = __builtin_amdgcn_raw_buffer_load_b128(xr, xoff | off, kt * 256 + b * 64, 0);
    }
  }

  __device__ __forceinline__ void mul(const Stage& st, f32x4 (&acc)[NTW]) const {
    typename Dq<DT>::ZS zs[NTW][GPT];
    st.w.template zero_scale<DT>(lane, zs);
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
      for (int j = 0; j < NTW; ++j) {
        const V8 a = Dq<DT>::word(st.w.q[j][b], zs[j][b / w.BPG], dk);
        acc[j] = mfma16x16x32(a, __builtin_bit_cast(V8, st.x[b]), acc[j]);
      }
  }

  // acc += k-tiles [kt0, kt1), D - 1 of them in flight ahead of the multiply.
  // The loop leaves by a branch between steps, past no load, so every stage
  // keeps its registers.
  template <int D>
  __device__ __forceinline__ void run(int kt0, int kt1, f32x4 (&acc)[NTW]) const {
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
