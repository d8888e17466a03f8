// Building blocks of the tile-parallel attention kernels (fwd_pp.hip, fwd_sk.hip): the 32x32
// MFMAs, global -> LDS transfers and their waits, LDS fragment reads, and the Q producer on Q
// fragments.
#pragma once
#include "common.h"
#include "kernels.h"

namespace orin {

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
typedef __attribute__((address_space(3))) const char* lds_ptr;

template <typename T>
__device__ __forceinline__ f32x16 mfma32(const u32x4& a, const u32x4& b, const f32x16& c);
template <>
__device__ __forceinline__ f32x16 mfma32<f16>(const u32x4& a, const u32x4& b, const f32x16& c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a),
                                                __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}
template <>
__device__ __forceinline__ f32x16 mfma32<bf16>(const u32x4& a, const u32x4& b, const f32x16& c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                 __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

template <typename T>
__device__ __forceinline__ uint32_t pack2(float x, float y) {
  typedef T T2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, T2{(T)x, (T)y});
}

template <typename T>
__device__ __forceinline__ float sum_pair(uint32_t p, float acc);
template <>
__device__ __forceinline__ float sum_pair<f16>(uint32_t p, float acc) {
  return __builtin_amdgcn_fdot2(__builtin_bit_cast(f16x2, p), f16x2{(f16)1.0f, (f16)1.0f}, acc,
                                false);
}
template <>
__device__ __forceinline__ float sum_pair<bf16>(uint32_t p, float acc) {
  return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, p),
                                         bf16x2{(bf16)1.0f, (bf16)1.0f}, acc, false);
}


// s_waitcnt vmcnt(N) leaving expcnt and lgkmcnt unconstrained (gfx9 encoding).
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | (15 << 8) | ((N >> 4) << 14));
}

// One 16-byte global -> LDS transfer per lane (global_load_lds_dwordx4): lane l's data
// lands at LDS byte lds_addr + 16 l.  Issued from inline asm so that the compiler does
// not treat it as an LDS store to wait for before every later LDS read: the kernel
// orders these transfers itself (vmcnt wait + barrier before the stage is read).  An LDS
// DMA that reads M0 right after an SALU write of M0 needs one wait state on gfx9-family
// parts, which the compiler cannot insert inside the asm: hence the s_nop.
// The address is a wave-uniform base (SGPR pair) plus a 32-bit per-lane byte offset: the per-tile
// address arithmetic stays on the scalar unit.
__device__ __forceinline__ void dma16_s(const void* sbase, uint32_t voff, uint32_t lds_addr) {
  __asm__ volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
                   :
                   : "v"(voff), "s"(sbase), "s"(lds_addr)
                   : "memory", "m0");
}

__device__ __forceinline__ uint32_t lds_addr(const char* p) {
  return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) char*)p;
}

// LDS reads at a per-lane address plus a compile-time offset (folded into the
// instruction's offset field).
__device__ __forceinline__ u32x4 lds_read128(lds_ptr p, int byte_off) {
  return *reinterpret_cast<const __attribute__((address_space(3))) u32x4*>(p + byte_off);
}

__device__ __forceinline__ u32x2 lds_read_tr(lds_ptr p, int byte_off) {
  const s16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(p + byte_off));
  return __builtin_bit_cast(u32x2, v);
}

// Fused Q producer on the Q fragments of one lane: qf[s] holds elements 16s + 8hf .. +7 of
// the lane's query row, so chunk c = 2s + hf (elements 8c .. 8c+7) of the first half of the
// head and its rotation partner (elements d/2 + 8c ..) are in qf[s] and qf[s + QS/2]; the
// partner lane (lane ^ 32) holds the other chunks.  Same arithmetic as qk_norm_rope_kernel
// (producers.hip), so the rounded row equals the one that producer writes.  The weight and
// table loads do not depend on the row and are issued first (rows past the end read the
// tables at position pos_ok and are left unchanged).
template <typename T, int D>
__device__ __forceinline__ void fuse_q_producer(const FwdArgs& a, u32x4 (&qf)[(D + 15) / 16],
                                                bool live, int pos, int pos_ok, int hf) {
  constexpr int QS = D / 16, H2 = QS / 2;  // chunks per lane in each half
  const int p = live ? pos : pos_ok;
  // table entries [p][2j], j = 16s + 8hf + i: four 16-byte loads per table and chunk
  const float* sn = a.rope_sin + (long)p * D + 16 * hf;
  const float* cn = a.rope_cos + (long)p * D + 16 * hf;
  f32x4 s4[H2][4], k4[H2][4];
#pragma unroll
  for (int s = 0; s < H2; ++s)
#pragma unroll
    for (int c4 = 0; c4 < 4; ++c4) {
      s4[s][c4] = *reinterpret_cast<const f32x4*>(sn + 32 * s + 4 * c4);
      k4[s][c4] = *reinterpret_cast<const f32x4*>(cn + 32 * s + 4 * c4);
    }
  const T* w = reinterpret_cast<const T*>(a.q_norm_weight);
  u32x4 wl_raw[H2], wh_raw[H2];
  if (w) {
#pragma unroll
    for (int s = 0; s < H2; ++s) {
      wl_raw[s] = load_chunk(w + 16 * s + 8 * hf).raw;
      wh_raw[s] = load_chunk(w + D / 2 + 16 * s + 8 * hf).raw;
    }
  }
  float lo[H2][8], hi[H2][8], cs[2 * H2];
  float own[H2];
#pragma unroll
  for (int s = 0; s < H2; ++s) {
    chunk_unpack(Chunk<T>{qf[s]}, lo[s]);
    chunk_unpack(Chunk<T>{qf[s + H2]}, hi[s]);
    own[s] = qk_chunk_sumsq(lo[s], hi[s]);
  }
#pragma unroll
  for (int s = 0; s < H2; ++s) {
    const float other = partner32(own[s]);
    cs[2 * s + hf] = own[s];
    cs[2 * s + (hf ^ 1)] = other;
  }
  if (w) {
    const float inv = qk_rms_inv(qk_butterfly_sum(cs), D, a.eps);
#pragma unroll
    for (int s = 0; s < H2; ++s) {
      float wl[8], wh[8];
      chunk_unpack(Chunk<T>{wl_raw[s]}, wl);
      chunk_unpack(Chunk<T>{wh_raw[s]}, wh);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        lo[s][i] = lo[s][i] * inv * wl[i];
        hi[s][i] = hi[s][i] * inv * wh[i];
      }
    }
  }
  if (!live) return;  // rows past the end stay zero
  typedef T T8 __attribute__((ext_vector_type(8)));
#pragma unroll
  for (int s = 0; s < H2; ++s) {
    T8 rl, rh;
#pragma unroll
    for (int c4 = 0; c4 < 4; ++c4)
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const int i = 2 * c4 + e;
        float ro, rv;
        qk_rope(lo[s][i], hi[s][i], k4[s][c4][2 * e], s4[s][c4][2 * e], ro, rv);
        rl[i] = from_f32<T>(ro);
        rh[i] = from_f32<T>(rv);
      }
    qf[s] = __builtin_bit_cast(u32x4, rl);
    qf[s + H2] = __builtin_bit_cast(u32x4, rh);
  }
}

}  // namespace orin
