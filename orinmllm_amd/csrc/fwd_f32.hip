// fp32 attention over many query rows on the fp32 matrix cores (gfx950).
//
// Serves the fp32 prefill (kernel::batched_mha_kernel_cu, mha_kernel.cu:347-444, and the fp32
// flash_attention_prefill_cu, flash_attention_kernel.cu:777-818) and the fp32 bidirectional
// attention (vision_attention_pretransposed_cu, vision_encoder_kernel.cu:954-1021).
//
// What bounds it: v_mfma_f32_16x16x4_f32 (32 clocks, 64 FLOP/clk and SIMD), which takes 4096
// clocks for 32 rows x 16 keys at head size 128; everything else is arranged to stay under
// that (4096 rows x 28 heads: 1046 us, 884 at the rate of a large fp32 matrix product).
//
// Work decomposition.  The query heads that share a kv head are packed: row R of a kv head is
// query R / kv_mul, head R % kv_mul of its group, so a tile of rows spans few positions (little
// of a causal diagonal tile is masked), K and V are read once for the whole group and short
// prompts fill the tile.  A workgroup of 4 waves owns a tile of RS sets of 16 rows; wave w takes
// the 16-key tiles w, w + 4, ... with its own online softmax, and the waves are merged once
// through LDS.  The key split inside the workgroup is what fills the chip: 523 rows x 28 heads
// are 460 tiles of 32 rows for 1024 SIMDs.
//
// Per 16-key tile and wave, lane (i, g) = (lane % 16, lane / 16):
//   S^T[key][row] = K . Q^T     A = K (key i), B = Q (row i).  A 16-byte piece s holds dims
//                               16 s + 4 g .. +3; MFMA j of the piece contracts dims 16 s + 4 g'
//                               + j, g' = 0..3.
//   O^T[dim][row] += V^T . P^T  accumulator register r of S^T holds key 4 g + r, the B layout of
//                               an MFMA that contracts keys r, 4 + r, 8 + r, 12 + r, so P never
//                               moves.  Lane i's piece of a V row is dims EP i .. EP i + EP - 1
//                               (EP = D / 16): element t is the A operand of output tile t,
//                               whose row i is dim EP i + t.
// K and V go straight from global memory (L2) to registers: a wave reads 16 KB per tile, 4
// bytes a clock, and no other wave of the workgroup wants the same keys.  The loads form one
// stream (the K pieces of a tile, then its V rows) that runs kRing loads ahead of the MFMAs
// that use them.
#include "common.h"
#include "decode_rows.h"
#include "kernels.h"

namespace orin {

namespace {

constexpr int kFKeys = 16;          // keys per wave tile
constexpr float kFLazyLog2 = 8.0f;  // the running maximum is raised when a weight would pass 2^8
constexpr int kFWaves = 4;          // 8 (half the keys each): no faster, slower from 224 tiles on

template <int N>
struct FVec { typedef float type __attribute__((ext_vector_type(N))); };

template <int D, int RS>
constexpr size_t f32_lds_bytes() {
  return (size_t)kFWaves * 16 * RS * (D + 2) * sizeof(float);
}

template <int D, int RS>
__global__ void __launch_bounds__(kFWaves * kWave, 2) fwd_f32_kernel(FwdArgs a) {
  static_assert(D == 64 || D == 128, "head size 64 or 128");
  constexpr int kRows = 16 * RS;
  constexpr int KP = D / 16;  // K pieces of a tile
  constexpr int EP = D / 16;  // output tiles; elements of a V row per lane
  constexpr int VL = EP / 4;  // 16-byte loads of a V row per lane
  constexpr int CL = D / 32;  // MFMAs per chain of a score: a score is the sum of 8 chains
  // O accumulators: at head size 64 one per accumulator register of P, so that with the waves'
  // key split an output is the sum of 16 chains over the keys, as many as the 16 waves of the
  // dot-product kernel's workgroup form at that head size (128: its four waves form 4).
  constexpr int OS = D == 64 ? 4 : 1;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int i = lane & 15, g = lane >> 4;
  const int G = a.kv_mul;
  const int rows = a.n_q * G;  // packed rows of a kv head
  const int n_rt = (rows + kRows - 1) / kRows;
  // Causal: longest rows first, except that the second block a CU receives at the start (two fit)
  // is taken from the other end of the first 2 n_cu: a long one runs beside a short one.
  int rank = (int)blockIdx.x;
  const int n_cu = a.n_cu;
  if (a.causal && rank >= n_cu && rank < 2 * n_cu)
    rank = n_cu + min(2 * n_cu, (int)gridDim.x) - 1 - rank;
  const int kvh = rank % a.Hkv;
  const int rt = n_rt - 1 - rank / a.Hkv;
  const int r_first = rt * kRows, r_last = min(r_first + kRows, rows) - 1;

  // This lane's row of each set (rows past the end repeat the last one and are not stored), the
  // keys [lo, hi) it attends to, the key range of the tile and the part that every row sees.
  int tok[RS], head[RS], lo[RS], hi[RS];
#pragma unroll
  for (int u = 0; u < RS; ++u) {
    const int R = min(r_first + 16 * u + i, r_last);
    tok[u] = R / G;
    head[u] = kvh * G + R % G;
  }
  int k_lo = 0, k_hi, all_lo = 0, all_hi;
  if (a.cu_seqlens) {
#pragma unroll
    for (int u = 0; u < RS; ++u) {
      const int s = find_segment(a.cu_seqlens, a.n_seg, tok[u]);
      lo[u] = a.cu_seqlens[s];
      hi[u] = a.cu_seqlens[s + 1];
    }
    k_lo = min(lo[0], lo[RS - 1]), k_hi = max(hi[0], hi[RS - 1]);
    all_lo = max(lo[0], lo[RS - 1]), all_hi = min(hi[0], hi[RS - 1]);
#pragma unroll
    for (int m = 8; m >= 1; m >>= 1) {
      k_lo = min(k_lo, __shfl_xor(k_lo, m));
      k_hi = max(k_hi, __shfl_xor(k_hi, m));
      all_lo = max(all_lo, __shfl_xor(all_lo, m));
      all_hi = min(all_hi, __shfl_xor(all_hi, m));
    }
    k_lo = __builtin_amdgcn_readfirstlane(k_lo);
    k_hi = __builtin_amdgcn_readfirstlane(k_hi);
    all_lo = __builtin_amdgcn_readfirstlane(all_lo);
    all_hi = __builtin_amdgcn_readfirstlane(all_hi);
  } else {
#pragma unroll
    for (int u = 0; u < RS; ++u) {
      lo[u] = 0;
      hi[u] = a.causal ? a.start_pos + tok[u] + 1 : a.n_q;
    }
    k_hi = a.causal ? a.start_pos + r_last / G + 1 : a.n_q;
    all_hi = a.causal ? a.start_pos + r_first / G + 1 : a.n_q;
  }

  const long tstr = a.kv_tok_stride;
  const float* kb = reinterpret_cast<const float*>(a.k) + (long)kvh * a.kv_head_stride + 4 * g;
  const float* vb = reinterpret_cast<const float*>(a.v) + (long)kvh * a.kv_head_stride + EP * i;

  f32x4 qf[RS][KP];
#pragma unroll
  for (int u = 0; u < RS; ++u) {
    const float* qp = reinterpret_cast<const float*>(a.q) + (long)tok[u] * a.q_tok_stride +
                      (long)head[u] * a.q_head_stride + 4 * g;
#pragma unroll
    for (int s = 0; s < KP; ++s) qf[u][s] = *reinterpret_cast<const f32x4*>(qp + 16 * s);
  }

  f32x4 oacc[OS][RS][EP];
#pragma unroll
  for (int o = 0; o < OS; ++o)
#pragma unroll
    for (int u = 0; u < RS; ++u)
#pragma unroll
      for (int t = 0; t < EP; ++t) oacc[o][u][t] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m[RS], l[RS];  // log2 units; l: this lane's weights
#pragma unroll
  for (int u = 0; u < RS; ++u) {
    m[u] = -INFINITY;
    l[u] = 0.f;
  }
  const float c = a.scale_log2;

  const int n_tiles = k_hi > k_lo ? (k_hi - k_lo + kFKeys - 1) / kFKeys : 0;
  // The stream of a tile: loads 0 .. KP-1 are K pieces, then VL pieces of the V rows of each
  // accumulator register.  Rows past the range read its last row (their weights are 0).
  constexpr int NS = KP + 4 * VL;
  constexpr int kRing = 8;
  static_assert(NS % kRing == 0, "a tile's loads start at ring slot 0");
  f32x4 ring[kRing];
  const int last = k_hi - 1;
  auto load = [&](int n, int t0) __attribute__((always_inline)) {
    const float* p;
    if (n < KP) {
      p = kb + (long)min(t0 + i, last) * tstr + 16 * n;
    } else {
      const int r = (n - KP) / VL, q = (n - KP) % VL;
      p = vb + (long)min(t0 + 4 * g + r, last) * tstr + 4 * q;
    }
    ring[n % kRing] = *reinterpret_cast<const f32x4*>(p);
  };

  // A masked key's weight is 0, but 0 times a non-finite V element is NaN, and the MFMA
  // multiplies every key of the tile for every row.  In masked tiles non-finite elements are
  // replaced by 0 on the way in, and this adds them back for the rows that see their keys.
  auto add_nonfinite = [&](const f32x4 (&p)[RS], int t0) __attribute__((always_inline)) {
    for (int kk = 0; kk < kFKeys; ++kk) {
      const int key = t0 + kk;
      if (key > last) break;
      const float* row =
          reinterpret_cast<const float*>(a.v) + (long)kvh * a.kv_head_stride + (long)key * tstr;
#pragma unroll
      for (int u = 0; u < RS; ++u) {
        float mine = 0.f;
#pragma unroll
        for (int x = 0; x < 4; ++x) mine = x == (kk & 3) ? p[u][x] : mine;
        const float pk = __shfl(mine, i + 16 * (kk >> 2));
        if (key < lo[u] || key >= hi[u]) continue;
#pragma unroll
        for (int x = 0; x < 4; ++x)
#pragma unroll
          for (int e = 0; e < EP; ++e) {
            const float v = row[EP * (4 * g + x) + e];
            const float acc = oacc[0][u][e][x];
            oacc[0][u][e][x] = __builtin_isfinite(v) ? acc : __builtin_fmaf(pk, v, acc);
            __builtin_amdgcn_sched_barrier(0);  // a rare path: one element's registers at a time
          }
      }
    }
  };

  if (wave < n_tiles) {
    int t0 = k_lo + wave * kFKeys;
#pragma unroll
    for (int n = 0; n < kRing; ++n) {
      load(n, t0);
      __builtin_amdgcn_sched_barrier(0);  // in order: the waits count the younger ones
    }
    for (int t = wave; t < n_tiles; t += kFWaves) {
      const int tn = t + kFWaves < n_tiles ? t0 + kFWaves * kFKeys : t0;
      // ---- S^T: eight MFMA chains of D / 8 products, summed in a binary tree on the VALU, so a
      // score rounds no worse than the dot-product kernel's eight lane sums.
      f32x4 s[RS], part[3][RS];  // part[k]: the sum of 2^k chains, waiting for its partner
#pragma unroll
      for (int n = 0; n < KP; ++n) {
        const f32x4 kx = ring[n];
        if (n + kRing < NS) load(n + kRing, t0);
        else load(n + kRing - NS, tn);
#pragma unroll
        for (int jj = 0; jj < 4 / CL; ++jj) {
#pragma unroll
          for (int u = 0; u < RS; ++u) s[u] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int j = CL * jj; j < CL * jj + CL; ++j)
#pragma unroll
            for (int u = 0; u < RS; ++u)
              s[u] = __builtin_amdgcn_mfma_f32_16x16x4f32(kx[j], qf[u][n][j], s[u], 0, 0, 0);
#pragma unroll
          for (int k = 0; k < 3; ++k) {
            if (!(((n * (4 / CL) + jj) >> k) & 1)) {
              
#pragma unroll
              for (int u = 0; u < RS; ++u) part[k][u] = s[u];
              break;
            }
#pragma unroll
            for (int u = 0; u < RS; ++u)
#pragma unroll
              for (int r = 0; r < 4; ++r) s[u][r] += part[k][u][r];
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      // ---- softmax
      const bool masked = t0 < all_lo || t0 + kFKeys > all_hi;
      if (masked) {
#pragma unroll
        for (int u = 0; u < RS; ++u)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int key = t0 + 4 * g + r;
            s[u][r] = key >= lo[u] && key < hi[u] ? s[u][r] : -INFINITY;
          }
      }
      bool raise = false;
      float mx[RS];
#pragma unroll
      for (int u = 0; u < RS; ++u) {
        mx[u] = fmaxf(fmaxf(s[u][0], s[u][1]), fmaxf(s[u][2], s[u][3])) * c;
        raise |= mx[u] > m[u] + kFLazyLog2;
      }
      // m is raised only when a weight would pass 2^8 (a row's first keys: m = -inf).
      if (__builtin_amdgcn_ballot_w64(raise)) {
#pragma unroll
        for (int u = 0; u < RS; ++u) {
          float x = fmaxf(mx[u], shfl_xor_f(mx[u], 16));
          x = fmaxf(x, partner32(x));
          const float mn = fmaxf(m[u], x);
          const float alpha = mn == m[u] ? 1.f : fast_exp2(m[u] - mn);
          m[u] = mn;
          l[u] *= alpha;
#pragma unroll
          for (int o = 0; o < OS; ++o)
#pragma unroll
            for (int e = 0; e < EP; ++e)
#pragma unroll
              for (int r = 0; r < 4; ++r) oacc[o][u][e][r] *= alpha;
        }
      }
#pragma unroll
      for (int u = 0; u < RS; ++u) {
        const float mu = m[u] == -INFINITY ? 0.f : m[u];  // every key so far masked: weights 0
#pragma unroll
        for (int r = 0; r < 4; ++r) s[u][r] = fast_exp2(__builtin_fmaf(s[u][r], c, -mu));
        l[u] += (s[u][0] + s[u][1]) + (s[u][2] + s[u][3]);
      }
      // ---- O^T
      bool bad = false;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float vx[EP];
#pragma unroll
        for (int q = 0; q < VL; ++q) {
          const int n = KP + VL * r + q;
#pragma unroll
          for (int e = 0; e < 4; ++e) vx[4 * q + e] = ring[n % kRing][e];
          if (n + kRing < NS) load(n + kRing, t0);
          else load(n + kRing - NS, tn);
        }
        if (masked) {
#pragma unroll
          for (int e = 0; e < EP; ++e) {
            const bool ok = __builtin_isfinite(vx[e]);
            bad |= !ok;
            vx[e] = ok ? vx[e] : 0.f;
          }
        }
#pragma unroll
        for (int e = 0; e < EP; ++e)
#pragma unroll
          for (int u = 0; u < RS; ++u)
            oacc[r % OS][u][e] =
                __builtin_amdgcn_mfma_f32_16x16x4f32(vx[e], s[u][r], oacc[r % OS][u][e], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
      if (masked && __builtin_amdgcn_ballot_w64(bad)) add_nonfinite(s, t0);
      t0 = tn;
    }
  }

#pragma unroll
  for (int o = OS / 2; o >= 1; o >>= 1)
#pragma unroll
    for (int x = 0; x < o; ++x)
#pragma unroll
      for (int u = 0; u < RS; ++u)
#pragma unroll
        for (int e = 0; e < EP; ++e)
#pragma unroll
          for (int r = 0; r < 4; ++r) oacc[x][u][e][r] += oacc[x + o][u][e][r];

  // ---------------------------------------------------------------- merge the waves
  // s_o: [wave][row][D], 4-float chunk ch of a row at ch ^ (row & (chunks - 1)).
  float* s_o = reinterpret_cast<float*>(smem);
  float* s_ml = s_o + kFWaves * kRows * D;
  constexpr int CH = D / 4;
#pragma unroll
  for (int u = 0; u < RS; ++u) {
    l[u] += shfl_xor_f(l[u], 16);
    l[u] += partner32(l[u]);
    const int wr = wave * kRows + 16 * u + i;
    if (g == 0) {
      s_ml[wr * 2] = m[u];
      s_ml[wr * 2 + 1] = l[u];
    }
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int q = 0; q < VL; ++q)
        *reinterpret_cast<f32x4*>(
            s_o + wr * D + (((VL * (4 * g + r) + q) ^ ((16 * u + i) & (CH - 1))) * 4)) =
            f32x4{oacc[0][u][4 * q][r], oacc[0][u][4 * q + 1][r], oacc[0][u][4 * q + 2][r],
                  oacc[0][u][4 * q + 3][r]};
  }
  __syncthreads();
  for (int x = threadIdx.x; x < kRows * CH; x += kFWaves * kWave) {
    const int row = x / CH, ch = x % CH;
    const int Ro = r_first + row;
    if (Ro > r_last) break;
    float M = -INFINITY;
#pragma unroll
    for (int w = 0; w < kFWaves; ++w) M = fmaxf(M, s_ml[(w * kRows + row) * 2]);
    const float Mu = M == -INFINITY ? 0.f : M;
    float L = 0.f;
    f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < kFWaves; ++w) {
      const float f = fast_exp2(s_ml[(w * kRows + row) * 2] - Mu);
      L = __builtin_fmaf(f, s_ml[(w * kRows + row) * 2 + 1], L);
      const f32x4 y = *reinterpret_cast<const f32x4*>(s_o + (w * kRows + row) * D +
                                                      ((ch ^ (row & (CH - 1))) * 4));
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = __builtin_fmaf(f, y[e], o[e]);
    }
    const int to = Ro / G;
    bool empty = false;  // a row of an empty segment gives zeros
    if (a.cu_seqlens) {
      const int sg = find_segment(a.cu_seqlens, a.n_seg, to);
      empty = a.cu_seqlens[sg + 1] <= a.cu_seqlens[sg];
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = empty ? 0.f : o[e] / L;
    float* op = reinterpret_cast<float*>(a.o) + (long)to * a.o_tok_stride +
                (long)(kvh * G + Ro % G) * a.o_head_stride + 4 * ch;
    *reinterpret_cast<f32x4*>(op) = o;
  }
}

template <int D, int RS>
hipError_t launch_f32_t(const FwdArgs& a, hipStream_t stream) {
  const int rows = a.n_q * a.kv_mul;
  const long blocks = (long)((rows + 16 * RS - 1) / (16 * RS)) * a.Hkv;
  if (blocks <= 0) return hipSuccess;
  constexpr size_t lds = f32_lds_bytes<D, RS>();
  // More than 64 KB of dynamic LDS must be granted per kernel (once per device).
  static unsigned long long configured = 0;
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if (dev >= 64 || !(__atomic_load_n(&configured, __ATOMIC_ACQUIRE) & (1ull << dev))) {
    e = hipFuncSetAttribute((const void*)fwd_f32_kernel<D, RS>,
                            hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
    if (dev < 64) __atomic_fetch_or(&configured, 1ull << dev, __ATOMIC_RELEASE);
  }
  hipLaunchKernelGGL((fwd_f32_kernel<D, RS>), dim3((unsigned)blocks), dim3(kFWaves * kWave), lds,
                     stream, a);
  return hipGetLastError();
}

}  // namespace

// Measured against the dot-product kernel (decode.hip, one workgroup per query row and kv head,
// every row reading its keys again), us per call, start 0:
//   28/4 heads, d 128: 128 rows 16.3 -> 8.2, 523 rows 135 -> 30.8, 1024 rows 361 -> 92, 2048
//   rows 1273 -> 286 (the MFMAs alone: 221); 12/12, d 64: 523 rows 76 -> 12, 2048 rows 710 -> 78.
// The dot-product kernel stays
//  * below a tile of keys (8 rows, 28/4 heads: 6.6 against 5.3 us, but this kernel's error
//    against float64 is 7.4e-8 there, the other's 7.1e-8; from 17 keys on it is not larger);
//  * with at most 4 heads to pack, while a workgroup per row and kv head still finds a CU of its
//    own (32/8 heads, 32 rows: 5.0 against 5.8; 8 rows behind 400 keys 14.7 against 14.3), or
//    half a CU and few keys (8/8 heads: 64 rows 4.4 against 6.5, behind 400 keys 17.2 against
//    15.6, 128 rows 8.8 against 7.9).  With 6 or 7 heads this kernel is ahead from one row on
//    (behind 400 keys: 20.5 against 13.1);
//  * at head size 256 (the tile does not fit the registers).
bool fwd_f32_supports(const FwdArgs& a) {
  if (a.head_size != 64 && a.head_size != 128) return false;
  if ((long)a.n_q * a.kv_mul >= (1l << 30)) return false;  // packed rows are ints
  const long keys = a.start_pos + (long)(a.cu_seqlens ? a.max_seqlen : a.n_q);
  if (keys <= kFKeys) return false;
  if (a.kv_mul > 4) return true;
  const long per_cu = a.head_size == 64 || keys >= 128 ? 1 : 2;
  return (long)a.n_q * a.Hkv > per_cu * a.n_cu;
}

hipError_t launch_fwd_f32(const FwdArgs& a, hipStream_t stream) {
  if (a.head_size == 64) return launch_f32_t<64, 1>(a, stream);
  // 32-row tiles halve the K / V reads per MFMA, 16-row tiles give twice the workgroups: the
  // large tile wins once its grid has 7/4 workgroups per CU (28/4 heads: 352 workgroups of 32
  // rows 26.5 us against 23.1, 460 30.7 against 31.8, 1792 282 against 314).
  const long tiles = ((long)a.n_q * a.kv_mul + 31) / 32 * a.Hkv;
  return tiles * 4 >= (long)a.n_cu * 7 ? launch_f32_t<128, 2>(a, stream)
                                       : launch_f32_t<128, 1>(a, stream);
}

}  // namespace orin
