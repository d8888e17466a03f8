// Matrix-core decode attention for 16-bit KV caches on gfx950.
//
// Serves the same launches as decode.hip (the reference's single-query attention,
// kuiper/source/op/kernels/cuda/flash_attention_kernel.cu:966-1175 and mha_kernel.cu:162-338,
// plus the batched / paged decode) for fp16 / bf16 K and V, head sizes 64 and 128, and up
// to 16 query heads per kv head.
//
// Two kernels: whole rows (first below) and split rows (further down).
//
// Whole rows.  Launches with a (row, kv head) per CU or more and one split per row, where a
// single CU must stream a whole row: the two contractions run on the matrix cores, the VALU
// work per 32-token tile is the softmax of 8 scores per lane, and the loads are whole coalesced
// rows.  Measured on the batch-32 paged decode (fp16, d 128, lengths U[512, 4096]): 0.64 of
// HBM, the dot-product kernel's 16-wave workgroups 0.59; a copy of this kernel with the
// arithmetic removed 0.67, so what remains is the rate at which one CU streams a row
// (~36 GB/s), not its arithmetic.
//
// Work decomposition.  A workgroup of 4 waves owns one (row, kv head) and all G query heads of
// that kv head (G <= 16, padded to 16 columns).  Wave w takes the 32-token tiles w, w + 4, ...
// of the row, with its own online-softmax state; the waves are merged once through LDS at the
// end.  Per tile:
//   S^T[32 x 16] = K[32 x D] . Q^T[D x 16]        2 x D/32  v_mfma_f32_16x16x32
//   O^T[D x 16] += V^T[D x 32] . P^T[32 x 16]     D/16      v_mfma_f32_16x16x32 (fp16)
//                                                 2 x D/16  (bf16: P = hi + lo, both bf16)
//   K and V arrive as whole rows (one load instruction covers 1 KB of consecutive rows) and
//   are written to per-wave LDS tiles.  Lane (n, g) = (lane % 16, lane / 16) reads K row n
//   (and n + 16), 16-byte chunk 4 j + g, which is the A layout of QK^T MFMA j with the
//   contraction index permuted identically in Q^T.  The S^T accumulator leaves lane (n, g)
//   the scores of head n for tokens 4g .. 4g+3 and 16 + 4g .. +3, which is the B layout of
//   P^T in the PV MFMAs.  V^T fragments come from ds_read_b64_tr_b16, which hands lane
//   (n, g) the four tokens 4g .. 4g+3 of dimension n from the row-major tile.  K rows are
//   stored with chunk c of row r at c ^ r (d 64: c ^ (r / 2)), V rows at c ^ (2r & 14):
//   both fragment reads are then free of bank conflicts.  Each wave keeps the next tile's
//   loads in flight while it computes the current one.
//
// Numerics match decode.hip: scores and the normaliser l in fp32, weights P rounded to
// fp16 for fp16 caches.  For bf16 caches P is split into bf16 hi + lo (hi + lo carries 16
// significant bits) and V stays bf16, so V keeps bf16's full range.  Paged and contiguous
// launches of the same KV run the same arithmetic and give identical bits.
#include <type_traits>

#include "common.h"
#include "kernels.h"
#include "decode_rows.h"

namespace orin {

namespace {

constexpr int kMWaves = 4;
constexpr int kMThreads = kMWaves * kWave;
constexpr int kMTile = 32;  // tokens per wave tile
// A wave keeps its running maximum while every weight stays at most 2^kMLazyLog2.
constexpr float kMLazyLog2 = 8.0f;

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;

template <typename T>
__device__ __forceinline__ f32x4 mfma16(const u32x4& a, const u32x4& b, const f32x4& c);
template <>
__device__ __forceinline__ f32x4 mfma16<f16>(const u32x4& a, const u32x4& b, const f32x4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a),
                                                __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}
template <>
__device__ __forceinline__ f32x4 mfma16<bf16>(const u32x4& a, const u32x4& b, const f32x4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                 __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// Packs two fp32 values into a 16-bit pair (round to nearest even).
template <typename T>
__device__ __forceinline__ uint32_t pack2m(float x, float y) {
  typedef T T2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, T2{(T)x, (T)y});
}

__device__ __forceinline__ float xor16(float x) { return shfl_xor_f(x, 16); }
__device__ __forceinline__ float xor32(float x) { return shfl_xor_f(x, 32); }

template <typename T, int D, bool PAGED>
__global__ void __launch_bounds__(kMThreads) decode_mfma_kernel(DecodeArgs a) {
  constexpr int NQK = D / 32;  // QK^T MFMAs per 16-token half (16-byte K pieces per token)
  constexpr int NDT = D / 16;  // 16-wide output tiles of O^T
  constexpr bool kBf16 = std::is_same<T, bf16>::value;
  static_assert(D == 64 || D == 128, "head size 64 or 128");
  // Per-wave K and V tiles (32 rows of D elements each) while the loop runs; the merge
  // reuses the space.
  extern __shared__ __attribute__((aligned(16))) char smem[];

  const int kvh = (int)blockIdx.x % a.Hkv;
  const int row = (int)blockIdx.x / a.Hkv;
  const int G = a.kv_mul;
  const int h0 = kvh * G;

  const int len = row_len(a, row);
  T* out = reinterpret_cast<T*>(a.o) + (long)row * a.o_row_stride;
  if (len > a.len_cap || len <= 0) {  // past the launch bound: NaN; empty row: zeros
    const float fill = len > 0 ? __builtin_nanf("") : 0.f;
    for (int i = threadIdx.x; i < G * D; i += kMThreads)
      out[(long)(h0 + i / D) * a.o_head_stride + i % D] = from_f32<T>(fill);
    return;
  }
  const int s1 = len;

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n = lane & 15;  // head column / token within a 16-token half / V^T dimension
  const int g = lane >> 4;  // 16-byte piece group

  // ---------------------------------------------------------------- address map
  const long tok_bytes = a.kv_tok_stride * (long)sizeof(T);
  const char* kbase = reinterpret_cast<const char*>(a.k) + a.kv_head_stride * (long)sizeof(T) * kvh;
  const char* vbase = reinterpret_cast<const char*>(a.v) + a.kv_head_stride * (long)sizeof(T) * kvh;
  const __attribute__((address_space(4))) int* bt = nullptr;
  long blk_bytes = 0;
  int bmask = 0;
  if constexpr (PAGED) {
    bt = (const __attribute__((address_space(4))) int*)(a.block_table + (long)row * a.bt_row_stride);
    blk_bytes = a.block_stride * (long)sizeof(T);
    bmask = (1 << a.bs_log2) - 1;
  } else {
    // contiguous: token t of the row is at element base + t * kv_tok_stride
    const long base = (long)row * a.kv_row_stride;
    kbase += base * (long)sizeof(T);
    vbase += base * (long)sizeof(T);
  }
  // Block ids of the four 8-token groups of the tile at t0 (paged): scalar loads.
  struct Blocks {
    int b[4];
  };
  auto tile_blocks = [&](int t0) __attribute__((always_inline)) {
    Blocks r;
#pragma unroll
    for (int q = 0; q < 4; ++q) r.b[q] = PAGED ? bt[min(t0 + 8 * q, s1 - 1) >> a.bs_log2] : 0;
    return r;
  };
  // Coalesced loads: instruction i of a tile covers rows RPI*i .. RPI*i + RPI-1 (whole rows,
  // RPI = 1 KB / row bytes), lane l row RPI*i + l / CPR, 16-byte chunk l % CPR.  Those rows
  // lie in one aligned 8-token group, so their block id is wave-uniform.
  constexpr int CPR = D / 8;        // 16-byte chunks per row
  constexpr int RPI = kWave / CPR;  // rows per load instruction
  constexpr int NLI = kMTile / RPI; // load instructions per tile (each of K and V)
  const int lrow = lane / CPR, lchunk = lane % CPR;
  // Row base (wave-uniform byte offset) and lane offset of load instruction i; rows past
  // the split read row s1 - 1.
  const uint32_t tok_b32 = (uint32_t)tok_bytes;
  auto row_base = [&](int t0, int i, const Blocks& bl) __attribute__((always_inline)) {
    const int rt = min(t0 + RPI * i, s1 - 1);
    if constexpr (PAGED) return (long)bl.b[(RPI * i) / 8] * blk_bytes + (long)(rt & bmask) * tok_bytes;
    return (long)rt * tok_bytes;
  };
  auto lane_off = [&](int t0, int i) __attribute__((always_inline)) {
    const int rt = min(t0 + RPI * i, s1 - 1);
    return (uint32_t)(min(t0 + RPI * i + lrow, s1 - 1) - rt) * tok_b32 + (uint32_t)(lchunk * 16);
  };

  // ---------------------------------------------------------------- Q^T operand
  // B operand of QK^T MFMA (h, j): lane (n, g) holds q[head h0 + n][32 j + 8 g .. +7]
  // (zero for columns n >= G).
  u32x4 qf[NQK];
  {
    const T* qp = reinterpret_cast<const T*>(a.q) + (long)row * a.q_row_stride +
                  (long)(h0 + n) * a.q_head_stride + 8 * g;
#pragma unroll
    for (int j = 0; j < NQK; ++j)
      qf[j] = n < G ? *reinterpret_cast<const u32x4*>(qp + 32 * j) : u32x4{0u, 0u, 0u, 0u};
  }

  // ---------------------------------------------------------------- LDS K / V tiles
  // Per wave: K tile then V tile, 32 rows of D elements each.
  char* const kt = smem + wave * (2 * kMTile * D * 2);
  char* const vt = kt + kMTile * D * 2;
  // K: row r, chunk c at chunk c ^ fk(r); the fragment reads (16 rows, one chunk) are then
  // conflict-free.  V: chunk c ^ (2r & 14), conflict-free for the transposing reads.
  auto kt_chunk = [&](int r, int c) __attribute__((always_inline)) {
    const int f = (D == 128 ? r : (r >> 1)) & (CPR - 1);
    return r * (D * 2) + ((c ^ f) * 16);
  };
  auto vt_chunk = [&](int r, int c) __attribute__((always_inline)) {
    return r * (D * 2) + ((c ^ ((2 * r) & (CPR - 1) & 14)) * 16);
  };
  // ds_read_b64_tr_b16 address of lane (n, g) = (4e + q4 within the 16-lane group g):
  // row 16 hh + 4 g + e, dimensions 16 t + 4 q4 .. +3 (one half of a 16-byte chunk).
  const int tr_e = n >> 2, tr_q = n & 3;

  f32x4 oacc[NDT];
#pragma unroll
  for (int t = 0; t < NDT; ++t) oacc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, lsum = 0.f;  // head n: running maximum (log2 units), lane's weight sum
  const float c = a.scale_log2;

  // Loads of one tile: whole K and V rows, NLI 16-byte pieces per lane each.
  struct Regs {
    u32x4 k[NLI];
    u32x4 v[NLI];
  };
  auto load_tile = [&](Regs& r, int t0, const Blocks& bl) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NLI; ++i) {
      const long rb = row_base(t0, i, bl);
      const uint32_t lo = lane_off(t0, i);
      r.k[i] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(kbase + rb + lo));
      r.v[i] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(vbase + rb + lo));
    }
  };

  typedef __attribute__((address_space(3))) u32x4 lds_u32x4;
  typedef __attribute__((address_space(3))) char lds_char;
  auto compute_tile = [&](const Regs& r, int t0) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NLI; ++i) {
      *reinterpret_cast<lds_u32x4*>((lds_char*)(kt + kt_chunk(RPI * i + lrow, lchunk))) = r.k[i];
      *reinterpret_cast<lds_u32x4*>((lds_char*)(vt + vt_chunk(RPI * i + lrow, lchunk))) = r.v[i];
    }
    // K fragments: lane (n, g) reads row 16 h + n, chunk 4 j + g.
    u32x4 kf[2][NQK];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int j = 0; j < NQK; ++j)
        kf[h][j] = *reinterpret_cast<const lds_u32x4*>((lds_char*)(kt + kt_chunk(16 * h + n, 4 * j + g)));
    // S^T halves: tokens 4g + i (h = 0) and 16 + 4g + i of head n.
    f32x4 s[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      s[h] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < NQK; ++j) s[h] = mfma16<T>(kf[h][j], qf[j], s[h]);
    }
    float x[8];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int tok = t0 + 16 * h + 4 * g + i;
        x[4 * h + i] = tok < s1 ? s[h][i] * c : -INFINITY;
      }
    // Lazy running maximum: raised only when a weight would exceed 2^8 (and on the first
    // tile, m = -inf); the four lanes of a head column agree on m.
    bool raise = false;
#pragma unroll
    for (int i = 0; i < 8; ++i) raise |= x[i] - m > kMLazyLog2;
    if (__builtin_amdgcn_ballot_w64(raise)) {
      float tm = x[0];
#pragma unroll
      for (int i = 1; i < 8; ++i) tm = fmaxf(tm, x[i]);
      tm = fmaxf(tm, xor16(tm));
      tm = fmaxf(tm, xor32(tm));
      const float mn = fmaxf(m, tm);
      const float alpha = fast_exp2(m - mn);
      m = mn;
      lsum *= alpha;
#pragma unroll
      for (int t = 0; t < NDT; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) oacc[t][i] *= alpha;
    }
    float p[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      p[i] = fast_exp2(x[i] - m);
      lsum += p[i];
    }
    // B operand P^T: items 0-3 = tokens 4g + i, items 4-7 = tokens 16 + 4g + i.
    u32x4 pb, pl;
    if constexpr (!kBf16) {
      pb = u32x4{pack2m<f16>(p[0], p[1]), pack2m<f16>(p[2], p[3]), pack2m<f16>(p[4], p[5]),
                 pack2m<f16>(p[6], p[7])};
    } else {
      float lo[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) lo[i] = p[i] - (float)(bf16)p[i];
      pb = u32x4{pack2m<bf16>(p[0], p[1]), pack2m<bf16>(p[2], p[3]), pack2m<bf16>(p[4], p[5]),
                 pack2m<bf16>(p[6], p[7])};
      pl = u32x4{pack2m<bf16>(lo[0], lo[1]), pack2m<bf16>(lo[2], lo[3]),
                 pack2m<bf16>(lo[4], lo[5]), pack2m<bf16>(lo[6], lo[7])};
    }
    // V^T tiles from LDS.  The writes above come first in this wave's LDS queue.
#pragma unroll
    for (int t = 0; t < NDT; ++t) {
      u32x2 part[2];
#pragma unroll
      for (int hh = 0; hh < 2; ++hh) {
        const int rr = 16 * hh + 4 * g + tr_e;
        const int col = 16 * t + 4 * tr_q;  // element column
        const int off = vt_chunk(rr, col >> 3) + (col & 7) * 2;
        const s16x4 v4 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (lds_s16x4*)((__attribute__((address_space(3))) char*)(vt + off)));
        part[hh] = __builtin_bit_cast(u32x2, v4);
      }
      const u32x4 va = u32x4{part[0][0], part[0][1], part[1][0], part[1][1]};
      if constexpr (!kBf16) {
        oacc[t] = mfma16<f16>(va, pb, oacc[t]);
      } else {
        oacc[t] = mfma16<bf16>(va, pb, oacc[t]);
        oacc[t] = mfma16<bf16>(va, pl, oacc[t]);
      }
    }
  };

  // ---------------------------------------------------------------- tile loop
  constexpr int step = kMWaves * kMTile;
  // Wave w runs tiles t = w, w + 8, ... (n_w of them).  Block ids are requested one tile
  // ahead of the loads that use them.  Loads are issued unconditionally, two buffers deep,
  // so that every wait before a tile's use is the same vmcnt: past the end of the split
  // every lane's token clamps to s1 - 1 and the tile reads one 256-byte row.
  const int tw0 = wave * kMTile;
  const int n_w = tw0 < s1 ? (s1 - tw0 + step - 1) / step : 0;
  if (n_w > 0) {
    Regs ra, rb;
    load_tile(ra, tw0, tile_blocks(tw0));
    Blocks bn = tile_blocks(tw0 + step);
    for (int i = 0;; i += 2) {
      const int t0 = tw0 + i * step;
      load_tile(rb, t0 + step, bn);
      bn = tile_blocks(t0 + 2 * step);
      __builtin_amdgcn_sched_barrier(0);  // the next tile's loads go out before this tile's work
      compute_tile(ra, t0);
      if (i + 1 >= n_w) break;
      load_tile(ra, t0 + 2 * step, bn);
      bn = tile_blocks(t0 + 3 * step);
      __builtin_amdgcn_sched_barrier(0);
      compute_tile(rb, t0 + step);
      if (i + 2 >= n_w) break;
    }
  }

  // ---------------------------------------------------------------- merge the waves
  lsum += xor16(lsum);
  lsum += xor32(lsum);
  __syncthreads();  // every wave is done with its V tile
  float* s_m = reinterpret_cast<float*>(smem);      // [waves][16]
  float* s_l = s_m + kMWaves * 16;                  // [waves][16]
  float* s_o = s_l + kMWaves * 16;                  // [waves][G][D]
  if (g == 0) {
    s_m[wave * 16 + n] = m;
    s_l[wave * 16 + n] = lsum;
  }
  __syncthreads();
  float M = -INFINITY;
#pragma unroll
  for (int w = 0; w < kMWaves; ++w) M = fmaxf(M, s_m[w * 16 + n]);
  const float f = m == -INFINITY ? 0.f : fast_exp2(m - M);
  if (n < G) {
#pragma unroll
    for (int t = 0; t < NDT; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) s_o[(wave * G + n) * D + 16 * t + 4 * g + i] = oacc[t][i] * f;
  }
  __syncthreads();
  for (int i = threadIdx.x; i < G * D; i += kMThreads) {
    const int hn = i / D, dd = i % D;
    float Mh = -INFINITY;
#pragma unroll
    for (int w = 0; w < kMWaves; ++w) Mh = fmaxf(Mh, s_m[w * 16 + hn]);
    float L = 0.f, o = 0.f;
#pragma unroll
    for (int w = 0; w < kMWaves; ++w) {
      const float mw = s_m[w * 16 + hn];
      L += mw == -INFINITY ? 0.f : fast_exp2(mw - Mh) * s_l[w * 16 + hn];
      o += s_o[(w * G + hn) * D + dd];
    }
    out[(long)(h0 + hn) * a.o_head_stride + dd] = from_f32<T>(o / L);
  }
}

constexpr size_t decode_mfma_lds_bytes(int head_size) {
  const size_t tiles = (size_t)kMWaves * 2 * kMTile * head_size * 2;
  const size_t merge = (size_t)kMWaves * 16 * (2 + head_size) * sizeof(float);  // G <= 16
  return tiles > merge ? tiles : merge;
}

// More than 64 KB of dynamic LDS must be granted per kernel (once per device).
template <auto kKernel>
hipError_t grant_lds(size_t bytes) {
  static unsigned long long configured = 0;
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if (dev >= 64 || !(__atomic_load_n(&configured, __ATOMIC_ACQUIRE) & (1ull << dev))) {
    e = hipFuncSetAttribute((const void*)kKernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                            (int)bytes);
    if (e != hipSuccess) return e;
    if (dev < 64) __atomic_fetch_or(&configured, 1ull << dev, __ATOMIC_RELEASE);
  }
  return hipSuccess;
}

template <typename T, int D, bool PAGED>
hipError_t launch_whole(const DecodeArgs& a, hipStream_t stream) {
  const long blocks = (long)a.n_rows * a.Hkv;
  constexpr size_t lds = decode_mfma_lds_bytes(D);
  hipError_t e = grant_lds<decode_mfma_kernel<T, D, PAGED>>(lds);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((decode_mfma_kernel<T, D, PAGED>), dim3((unsigned)blocks), dim3(kMThreads),
                     lds, stream, a);
  return hipGetLastError();
}

// ---------------------------------------------------------------- split rows
// Every launch that is not one whole row per CU: split rows, and rows fewer than the CUs.
// A workgroup of NW waves owns one (row, kv head, split); wave w takes the 16-token tiles w,
// w + NW, ... of the split.  Per tile and wave:
//   S^T[16 x 16] = K . Q^T        D/32 v_mfma_f32_16x16x32
//   O^T[D x 16] += V^T . P^T      D/16 v_mfma_f32_16x16x16 (bf16: two, P = hi + lo); the S^T
//                                 accumulator (tokens 4 g + i) is the B layout of P^T
// V goes through an LDS tile per wave for the transposing reads.  The next tile's K is
// requested once the current one is used, its V once the current rows are in LDS.
// Two shapes:
//  * NW = 8, few workgroups: bound by latency, the chain of round trips (length, K and V,
//    merge) and a CU's ~36 GB/s.  K pieces go from global memory straight to the MFMA operand
//    layout (lane (n, g): row n, chunk 4 j + g), and one barrier suffices: the waves' (m, l)
//    and unscaled O go to LDS together.
//  * NW = 4, many workgroups: bound by HBM.  K rows are loaded whole (1 KB of consecutive rows
//    per instruction, nontemporal) and turned in LDS like the whole-row kernel's: with KV
//    that the last-level cache does not hold, batch 31, 32/8 heads, bf16, lengths U[512, 4096]
//    61.2 -> 56.5 us against the K pieces' 64-byte segments (59.8); the waves' results then
//    share the tiles' space (four workgroups fit a CU).
// Against the dot-product kernel (decode.hip), split + merge, us: one row of 4096, 32/8 heads,
// fp16 11.5 -> 9.1; 28/4 heads, bf16, batch 5, lengths U[2048, 16000] 45.8 -> 30.5; 12/2 heads,
// bf16, batch 64, lengths U[300, 4000] 57.9 -> 39.9.
constexpr int kSTile = 16;

// LDS of a split workgroup: the waves' V (and K) tiles, then (m, l) [NW][16][2] and O [NW][G][D],
// which share the tiles' space for NW = 4.
template <int D, int NW>
constexpr size_t split_lds(int G) {
  const size_t tiles = (size_t)NW * (NW == 4 ? 2 : 1) * kSTile * D * 2;
  const size_t merge = (size_t)NW * (16 * 2 + G * D) * sizeof(float);
  return NW == 4 ? (tiles > merge ? tiles : merge) : tiles + merge;
}

template <typename T>
__device__ __forceinline__ f32x4 mfma16k16(const u32x2& a, const u32x2& b, const f32x4& c);
template <>
__device__ __forceinline__ f32x4 mfma16k16<f16>(const u32x2& a, const u32x2& b, const f32x4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x16f16(__builtin_bit_cast(f16x4, a),
                                               __builtin_bit_cast(f16x4, b), c, 0, 0, 0);
}
template <>
__device__ __forceinline__ f32x4 mfma16k16<bf16>(const u32x2& a, const u32x2& b, const f32x4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(s16x4, a),
                                                   __builtin_bit_cast(s16x4, b), c, 0, 0, 0);
}

template <typename T, int D, bool PAGED, int NW>
__global__ void __launch_bounds__(NW * kWave, 4) decode_split_mfma_kernel(DecodeArgs a) {
  constexpr int kThreads = NW * kWave;
  constexpr int NQK = D / 32;  // QK^T MFMAs (16-byte K pieces per token)
  constexpr int NDT = D / 16;  // 16-wide output tiles of O^T
  constexpr bool kKLds = NW == 4;  // K through LDS (above)
  constexpr bool kBf16 = std::is_same<T, bf16>::value;
  static_assert(D == 64 || D == 128, "head size 64 or 128");
  extern __shared__ __attribute__((aligned(16))) char smem[];

  int bid = blockIdx.x;
  const int kvh = bid % a.Hkv;
  bid /= a.Hkv;
  const int split = bid % a.max_splits;
  const int row = bid / a.max_splits;
  const int G = a.kv_mul;
  const int h0 = kvh * G;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n = lane & 15;  // head column / token of the tile / V^T dimension
  const int g = lane >> 4;  // 16-byte piece group

  // B operand of QK^T MFMA j: lane (n, g) holds q[head h0 + n][32 j + 8 g .. +7] (zero for
  // columns n >= G).  Requested before the row's length is known.
  u32x4 qf[NQK];
  {
    const T* qp = reinterpret_cast<const T*>(a.q) + (long)row * a.q_row_stride +
                  (long)(h0 + min(n, G - 1)) * a.q_head_stride + 8 * g;
#pragma unroll
    for (int j = 0; j < NQK; ++j) qf[j] = *reinterpret_cast<const u32x4*>(qp + 32 * j);
  }

  const int len = row_len(a, row);
  const int st = row_split_tokens(a, len);
  T* out = reinterpret_cast<T*>(a.o) + (long)row * a.o_row_stride;
  if (len > a.len_cap || len <= 0) {  // past the launch bound: NaN; empty row: zeros
    if (split == 0) {
      const float fill = len > 0 ? __builtin_nanf("") : 0.f;
      for (int i = threadIdx.x; i < G * D; i += kThreads)
        out[(long)(h0 + i / D) * a.o_head_stride + i % D] = from_f32<T>(fill);
    }
    return;
  }
  if ((long)split * st >= len) return;
  const int s0 = split * st;
  const int s1 = min(s0 + st, len);

  // ---------------------------------------------------------------- address map
  const long tok_bytes = a.kv_tok_stride * (long)sizeof(T);
  const char* kbase = reinterpret_cast<const char*>(a.k) + a.kv_head_stride * (long)sizeof(T) * kvh;
  const char* vbase = reinterpret_cast<const char*>(a.v) + a.kv_head_stride * (long)sizeof(T) * kvh;
  const __attribute__((address_space(4))) int* bt = nullptr;
  long blk_bytes = 0;
  int bmask = 0;
  if constexpr (PAGED) {
    bt = (const __attribute__((address_space(4))) int*)(a.block_table + (long)row * a.bt_row_stride);
    blk_bytes = a.block_stride * (long)sizeof(T);
    bmask = (1 << a.bs_log2) - 1;
  } else {
    const long base = (long)row * a.kv_row_stride;
    kbase += base * (long)sizeof(T);
    vbase += base * (long)sizeof(T);
  }
  // Byte offset of token t's row (t in the tile at t0, clamped to the split by the caller); the
  // two 8-token halves of a tile each lie in one block.
  struct Blocks { int b[2]; };
  auto tile_blocks = [&](int t0) __attribute__((always_inline)) {
    Blocks r;
#pragma unroll
    for (int q = 0; q < 2; ++q) r.b[q] = PAGED ? bt[min(t0 + 8 * q, s1 - 1) >> a.bs_log2] : 0;
    return r;
  };
  auto row_off = [&](int t, int t0, const Blocks& bl) __attribute__((always_inline)) {
    const int tc = min(t, s1 - 1);
    if constexpr (PAGED)
      return (long)(tc >= t0 + 8 ? bl.b[1] : bl.b[0]) * blk_bytes + (long)(tc & bmask) * tok_bytes;
    return (long)tc * tok_bytes;
  };

  // Per-wave V tile: 16 rows of D elements, chunk c of row r at c ^ (2r & 14); K tile the same
  // with chunk c at c ^ r (D 64: c ^ (r / 2)).
  constexpr int CPR = D / 8;        // 16-byte chunks per row
  constexpr int RPI = kWave / CPR;  // rows per load instruction
  constexpr int NLV = kSTile / RPI; // whole-row load instructions per tile
  char* const vt = smem + wave * ((kKLds ? 2 : 1) * kSTile * D * 2);
  char* const kt = vt + kSTile * D * 2;
  const int lrow = lane / CPR, lchunk = lane % CPR;
  auto vt_chunk = [&](int r, int c) __attribute__((always_inline)) {
    return r * (D * 2) + ((c ^ ((2 * r) & (CPR - 1) & 14)) * 16);
  };
  auto kt_chunk = [&](int r, int c) __attribute__((always_inline)) {
    return r * (D * 2) + ((c ^ ((D == 128 ? r : (r >> 1)) & (CPR - 1))) * 16);
  };
  const int tr_e = n >> 2, tr_q = n & 3;

  constexpr int NLK = kKLds ? NLV : NQK;  // (equal)
  u32x4 kr[NLK], vr[NLV];
  auto load_k = [&](int t0, const Blocks& bl) __attribute__((always_inline)) {
    if constexpr (kKLds) {
#pragma unroll
      for (int i = 0; i < NLK; ++i)
        kr[i] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(
            kbase + row_off(t0 + RPI * i + lrow, t0, bl) + 16 * lchunk));
    } else {
      const char* p = kbase + row_off(t0 + n, t0, bl) + 16 * g;
#pragma unroll
      for (int j = 0; j < NLK; ++j)
        kr[j] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p + 64 * j));
    }
  };
  auto load_v = [&](int t0, const Blocks& bl) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NLV; ++i)
      vr[i] = __builtin_nontemporal_load(
          reinterpret_cast<const u32x4*>(vbase + row_off(t0 + RPI * i + lrow, t0, bl) + 16 * lchunk));
  };

  f32x4 oacc[NDT];
#pragma unroll
  for (int t = 0; t < NDT; ++t) oacc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, lsum = 0.f;
  const float c = a.scale_log2;
  typedef __attribute__((address_space(3))) u32x4 lds_u32x4;
  typedef __attribute__((address_space(3))) char lds_char;

  int t0 = s0 + wave * kSTile;
  if (t0 < s1) {
    Blocks bl = tile_blocks(t0);
    load_k(t0, bl);
    load_v(t0, bl);
    while (true) {
      const int tn = t0 + NW * kSTile;
      const bool more = tn < s1;
      if (more) bl = tile_blocks(tn);
      if constexpr (kKLds) {
#pragma unroll
        for (int i = 0; i < NLK; ++i)
          *reinterpret_cast<lds_u32x4*>((lds_char*)(kt + kt_chunk(RPI * i + lrow, lchunk))) = kr[i];
      }
      f32x4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < NQK; ++j) {
        u32x4 kf;
        if constexpr (kKLds)
          kf = *reinterpret_cast<const lds_u32x4*>((lds_char*)(kt + kt_chunk(n, 4 * j + g)));
        else
          kf = kr[j];
        s = mfma16<T>(kf, qf[j], s);
      }
      if (more) load_k(tn, bl);
      float x[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) x[i] = t0 + 4 * g + i < s1 ? s[i] * c : -INFINITY;
#pragma unroll
      for (int i = 0; i < NLV; ++i)
        *reinterpret_cast<lds_u32x4*>((lds_char*)(vt + vt_chunk(RPI * i + lrow, lchunk))) = vr[i];
      if (more) load_v(tn, bl);
      bool raise = false;
#pragma unroll
      for (int i = 0; i < 4; ++i) raise |= x[i] - m > kMLazyLog2;
      if (__builtin_amdgcn_ballot_w64(raise)) {
        float tm = fmaxf(fmaxf(x[0], x[1]), fmaxf(x[2], x[3]));
        tm = fmaxf(tm, xor16(tm));
        tm = fmaxf(tm, partner32(tm));
        const float mn = fmaxf(m, tm);
        const float alpha = fast_exp2(m - mn);
        m = mn;
        lsum *= alpha;
#pragma unroll
        for (int t = 0; t < NDT; ++t)
#pragma unroll
          for (int i = 0; i < 4; ++i) oacc[t][i] *= alpha;
      }
      float p[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        p[i] = fast_exp2(x[i] - m);
        lsum += p[i];
      }
      u32x2 pb, pl;
      if constexpr (!kBf16) {
        pb = u32x2{pack2m<f16>(p[0], p[1]), pack2m<f16>(p[2], p[3])};
      } else {
        float lo[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) lo[i] = p[i] - (float)(bf16)p[i];
        pb = u32x2{pack2m<bf16>(p[0], p[1]), pack2m<bf16>(p[2], p[3])};
        pl = u32x2{pack2m<bf16>(lo[0], lo[1]), pack2m<bf16>(lo[2], lo[3])};
      }
#pragma unroll
      for (int t = 0; t < NDT; ++t) {
        const int rr = 4 * g + tr_e;
        const int col = 16 * t + 4 * tr_q;
        const int off = vt_chunk(rr, col >> 3) + (col & 7) * 2;
        const s16x4 v4 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (lds_s16x4*)((__attribute__((address_space(3))) char*)(vt + off)));
        const u32x2 va = __builtin_bit_cast(u32x2, v4);
        oacc[t] = mfma16k16<T>(va, pb, oacc[t]);
        if constexpr (kBf16) oacc[t] = mfma16k16<T>(va, pl, oacc[t]);
      }
      if (!more) break;
      t0 = tn;
    }
  }

  // ---------------------------------------------------------------- merge the waves
  lsum += xor16(lsum);
  lsum += partner32(lsum);
  if constexpr (kKLds) __syncthreads();  // every wave is done with its tiles
  float* s_m = reinterpret_cast<float*>(smem + (kKLds ? 0 : NW * kSTile * D * 2));  // [waves][16]
  float* s_l = s_m + NW * 16;
  float* s_o = s_l + NW * 16;  // [waves][G][D]
  if (g == 0) {
    s_m[wave * 16 + n] = m;
    s_l[wave * 16 + n] = lsum;
  }
  if (n < G) {
#pragma unroll
    for (int t = 0; t < NDT; ++t)
      *reinterpret_cast<f32x4*>(s_o + (wave * G + n) * D + 16 * t + 4 * g) = oacc[t];
  }
  __syncthreads();
  const bool direct = st >= len;
  for (int i = threadIdx.x; i < G * D; i += kThreads) {
    const int hn = i / D, dd = i % D;
    float mw[NW], M = -INFINITY;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      mw[w] = s_m[w * 16 + hn];
      M = fmaxf(M, mw[w]);
    }
    float L = 0.f, o = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float f = fast_exp2(mw[w] - M);
      L = __builtin_fmaf(f, s_l[w * 16 + hn], L);
      o = __builtin_fmaf(f, s_o[(w * G + hn) * D + dd], o);
    }
    if (direct) {
      out[(long)(h0 + hn) * a.o_head_stride + dd] = from_f32<T>(o / L);
    } else {
      const long pi = ((long)row * a.Hq + h0 + hn) * a.max_splits + split;
      a.ws[pi * D + dd] = o;
      if (dd == 0) {
        float* ml = a.ws + (long)a.n_rows * a.Hq * a.max_splits * D + pi * 2;
        ml[0] = M;
        ml[1] = L;
      }
    }
  }
}

template <typename T, int D, bool PAGED, int NW>
hipError_t launch_split(const DecodeArgs& a, hipStream_t stream) {
  const long blocks = (long)a.n_rows * a.Hkv * a.max_splits;
  const size_t lds = split_lds<D, NW>(a.kv_mul);
  hipError_t e = grant_lds<decode_split_mfma_kernel<T, D, PAGED, NW>>(split_lds<D, NW>(16));
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((decode_split_mfma_kernel<T, D, PAGED, NW>), dim3((unsigned)blocks),
                     dim3(NW * kWave), lds, stream, a);
  return hipGetLastError();
}

template <typename T, int D, bool PAGED>
hipError_t launch_p(const DecodeArgs& a, int n_cu, hipStream_t stream) {
  const long units = (long)a.n_rows * a.Hkv;
  // Whole rows with a unit per CU or more: the 4-wave kernel that keeps two 32-token tiles of
  // every wave in flight streams a row fastest.  The single-sequence decode never gets there.
  if (a.max_splits == 1 && units >= n_cu && a.dyn_splits_log2 < 0)
    return launch_whole<T, D, PAGED>(a, stream);
  // Up to two workgroups per CU: the latency shape.  28/4 heads, batch 16, lengths up to 4096,
  // bf16: 512 workgroups 24.0 us with 8 waves, 23.7 with 4; 1024 workgroups 25.1 and 23.2.
  return units * a.max_splits <= 2l * n_cu ? launch_split<T, D, PAGED, 8>(a, stream)
                                           : launch_split<T, D, PAGED, 4>(a, stream);
}

template <typename T, int D>
hipError_t launch_t(const DecodeArgs& a, int n_cu, hipStream_t stream) {
  return a.block_table ? launch_p<T, D, true>(a, n_cu, stream)
                       : launch_p<T, D, false>(a, n_cu, stream);
}

}  // namespace

bool decode_mfma_supports(int dtype, int head_size, int kv_mul) {
  return (dtype == kF16 || dtype == kBF16) && (head_size == 64 || head_size == 128) &&
         kv_mul >= 1 && kv_mul <= 16;
}

hipError_t launch_decode_mfma(const DecodeArgs& a, int n_cu, int dtype, hipStream_t stream) {
  if (dtype == kF16)
    return a.head_size == 64 ? launch_t<f16, 64>(a, n_cu, stream)
                             : launch_t<f16, 128>(a, n_cu, stream);
  return a.head_size == 64 ? launch_t<bf16, 64>(a, n_cu, stream)
                           : launch_t<bf16, 128>(a, n_cu, stream);
}

}  // namespace orin
