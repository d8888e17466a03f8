// Attention forward with the keys split inside the workgroup (fp16 / bf16 in, fp32 accumulate),
// for launches whose 256-query blocks do not fill the chip.
//
// Serves the same paths as fwd_pp.hip (causal GQA prefill over a kuiper KV cache,
// flash_attention_kernel.cu:554-905; bidirectional varlen attention,
// vision_encoder_kernel.cu:954-1021).
//
// What bounds small and mid-sized launches is not the MFMA rate but a block's serial chain: one
// workgroup per (head, 256 queries) walks every key tile by itself, ~1.5 us per 64 keys, while
// most CUs idle.  Here a workgroup of 4 waves owns 32 rows and wave w takes the 32-key tiles w,
// w + 4, ... with its own online softmax; the waves are merged once through LDS.  The chain is a
// quarter as long and the blocks are an eighth as large, so the grid fills the chip without a
// second launch that merges partials.  Rows of the query heads that share a kv head are packed
// (row R of a kv head = query R / kv_mul, head R % kv_mul of its group): short prompts fill the
// 32 rows, and little of a causal diagonal tile is masked.
//
// The price: K and V are read from L2 once per 32 rows (a CU streams ~110 GB/s from L2), with no
// wave sharing another's tile, so large launches stay on fwd_pp.hip.
//
// Per 32-key tile and wave, lane (lq, hf) = (lane % 32, lane / 32):
//   S^T[key][row] = K . Q^T      D/16 v_mfma_f32_32x32x16; lane: row lq, 16 keys
//   O^T[dim][row] += V^T . P^T   2 x D/32 v_mfma_f32_32x32x16 (fp16); P^T is taken from the S^T
//                                accumulator registers, V^T from two transposing LDS reads
// K and V tiles are per wave (8 KB each at head size 128) and reach LDS
// by global_load_lds_dwordx4: the next K tile is requested once the scores exist, the next V tile
// once the products with V do, so each has the other half of the tile's work, and the second
// wave of the SIMD, to arrive.  No barrier runs inside the loop.  bf16 V fragments are converted to
// fp16 after the LDS read (the softmax weights are fp16, see common.h).
// Head sizes below 128 pad the QK contraction to a multiple of 16 (zero Q elements) and O^T to a
// multiple of 32 (rows never stored).
#include <type_traits>

#include "common.h"
#include "fwd_tile.h"
#include "kernels.h"

namespace orin {

namespace {

constexpr int kSkRows = 32;                   // rows per workgroup
constexpr int kSkKeys = 32;                   // keys per wave tile

// LDS rows of a K or V tile, in 16-byte chunks.  Head size 128: 16, chunk c of row r at c ^ (r & 15)
// (K) or c ^ 4(r & 3) (V).  Smaller heads: the chunks the QK contraction reads plus what makes the
// row stride free of bank conflicts without a swizzle, so that no transfer is spent on padding
// 256-byte rows (5 transfers per tile instead of 8 at head sizes 64 to 80, where the loads bound
// the kernel).
template <int D>
constexpr int sk_row_chunks() { return D == 128 ? 16 : D == 96 ? 13 : D == 64 ? 9 : 10; }
template <int D>
constexpr int sk_transfers() { return (kSkKeys * sk_row_chunks<D>() + kWave - 1) / kWave; }
// K and V tiles of the waves (1 KB per transfer), or O [wave][row][DT * 32] in the merge; then the
// waves' (m, l).
template <int D, int NW>
constexpr int sk_ml_offset() {
  const int tiles = NW * 2 * sk_transfers<D>() * 1024;
  const int merge = NW * kSkRows * ((D + 31) / 32 * 32) * 4;
  return tiles > merge ? tiles : merge;
}
template <int D, int NW>
constexpr int sk_lds() { return sk_ml_offset<D, NW>() + NW * kSkRows * 2 * 4; }
// A lane's 16 weights of one tile may sum to at most this before the row maximum is raised.
constexpr float kSkSumMax = 256.0f;

// FQ: the query rows are raw and the Q producer runs on the fragments (a.rope_sin set).
template <typename T, bool CAUSAL, int D, bool FQ, int NW>
__global__ void __launch_bounds__(NW * kWave, 2) fwd_sk_kernel(FwdArgs a) {
  constexpr int QS = (D + 15) / 16;  // 16-wide slices of the QK contraction
  constexpr int DT = (D + 31) / 32;  // 32-wide output tiles of O^T
  constexpr int NCH = D / 8;         // valid 16-byte chunks of a K / V row
  constexpr bool kConvV = !std::is_same<T, f16>::value;
  constexpr int RC = sk_row_chunks<D>(), NI = sk_transfers<D>();
  constexpr int kTile = NI * 1024;  // bytes of a K or V tile
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lq = lane & 31, hf = lane >> 5;
  const int G = a.kv_mul;

  // ------------------------------------------------------------ block -> rows
  // Packed rows r_first .. r_last of kv head kvh, in the segment that starts at seg_start.
  int kvh, r_first, rows, seg_start = 0, kv_len;
  if (CAUSAL) {
    // Longest rows first, except that the second block a CU receives at the start (two fit) is
    // taken from the other end of the first 2 n_cu: a long one runs beside a short one.
    rows = a.n_q * G;
    const int n_rt = (rows + kSkRows - 1) / kSkRows;
    int rank = (int)blockIdx.x;
    if (rank >= a.n_cu && rank < 2 * a.n_cu)
      rank = a.n_cu + min(2 * a.n_cu, (int)gridDim.x) - 1 - rank;
    kvh = rank % a.Hkv;
    r_first = (n_rt - 1 - rank / a.Hkv) * kSkRows;
  } else {
    const int n_rt = (a.max_seqlen * G + kSkRows - 1) / kSkRows;
    kvh = (int)blockIdx.x % a.Hkv;
    const int rest = (int)blockIdx.x / a.Hkv;
    const int seg = rest / n_rt;
    r_first = rest % n_rt * kSkRows;
    seg_start = a.cu_seqlens ? a.cu_seqlens[seg] : 0;
    const int seg_n = a.cu_seqlens ? a.cu_seqlens[seg + 1] - seg_start : a.n_q;
    rows = seg_n * G;
    if (r_first >= rows) return;
  }
  const int r_last = min(r_first + kSkRows, rows) - 1;
  kv_len = CAUSAL ? a.start_pos + r_last / G + 1 : rows / G;
  const int n_tiles = (kv_len + kSkKeys - 1) / kSkKeys;
  // This lane's row (rows past the end repeat the last one and are not stored).
  const int R = min(r_first + lq, r_last);
  const int tok = R / G;
  const int head = kvh * G + R % G;
  const int pos = CAUSAL ? a.start_pos + tok : kv_len - 1;          // last key of the row
  const int pos_min = CAUSAL ? a.start_pos + r_first / G : kv_len - 1;

  const long tstr = a.kv_tok_stride;
  const T* kb = reinterpret_cast<const T*>(a.k) + (long)seg_start * tstr + (long)kvh * a.kv_head_stride;
  const T* vb = reinterpret_cast<const T*>(a.v) + (long)seg_start * tstr + (long)kvh * a.kv_head_stride;
  const uint32_t row_bytes = (uint32_t)tstr * sizeof(T);

  // ------------------------------------------------------------ K / V tiles
  // Transfer b of a tile fills its chunks 64 b .. 64 b + 63, lane l chunk 64 b + l = chunk
  // idx % RC of row idx / RC.  Chunks past the head (and rows past the tile) load chunk 0 of a
  // row: finite values that meet zero Q elements (K) or O^T rows never stored (V).
  auto chunk_row = [&](int b) __attribute__((always_inline)) {
    return min((64 * b + lane) / RC, kSkKeys - 1);
  };
  auto chunk_col = [&](int b, bool v) __attribute__((always_inline)) {  // byte column
    int cc = (64 * b + lane) % RC;
    if (D == 128) {
      const int r = (64 * b + lane) / RC;
      cc ^= v ? 4 * (r & 3) : r & 15;
    }
    return (uint32_t)(16 * (cc < NCH ? cc : 0));
  };
  // Offsets of whole tiles.  Head size 128: rows 4b + l / 16, so the lane parts repeat (K: every 4
  // transfers, V: each) and a scalar 4 b rows is added; else K and V share them.
  constexpr int NOK = D == 128 ? 4 : NI;
  uint32_t k_off[NOK];
#pragma unroll
  for (int b = 0; b < NOK; ++b)
    k_off[b] = __umul24(D == 128 ? lane >> 4 : chunk_row(b), row_bytes) + chunk_col(b, false);
  const uint32_t v_off = D == 128 ? __umul24(lane >> 4, row_bytes) + chunk_col(0, true) : 0u;
  char* const my = smem + wave * 2 * kTile;
  const lds_ptr k_lds = (lds_ptr)my, v_lds = k_lds + kTile;
  const uint32_t k_addr = __builtin_amdgcn_readfirstlane(lds_addr(my));
  auto issue = [&](const T* x, int t0, auto is_v) __attribute__((always_inline)) {
    constexpr bool V = decltype(is_v)::value;
    const uint32_t dst = k_addr + (V ? kTile : 0);
    const char* base = reinterpret_cast<const char*>(x + (long)t0 * tstr);
    if (t0 + kSkKeys <= kv_len) {
#pragma unroll
      for (int b = 0; b < NI; ++b) {
        const uint32_t off =
            D == 128 ? (V ? v_off : k_off[b & 3]) + 4 * b * row_bytes : k_off[b % NOK];
        dma16_s(base, off, dst + b * 1024);
      }
    } else {  // the last tile: rows past the sequence read its last row
#pragma unroll
      for (int b = 0; b < NI; ++b)
        dma16_s(base, __umul24(min(chunk_row(b), kv_len - 1 - t0), row_bytes) + chunk_col(b, V),
                dst + b * 1024);
    }
  };
  auto issue_k = [&](int t0) __attribute__((always_inline)) { issue(kb, t0, std::false_type{}); };
  auto issue_v = [&](int t0) __attribute__((always_inline)) { issue(vb, t0, std::true_type{}); };

  int t = wave;
  const bool any = wave < n_tiles;
  if (any) issue_k(t * kSkKeys);

  // ------------------------------------------------------------ Q fragments
  u32x4 qf[QS];
  {
    const T* qp = reinterpret_cast<const T*>(a.q) + (long)(seg_start + tok) * a.q_tok_stride +
                  (long)head * a.q_head_stride;
#pragma unroll
    for (int s = 0; s < QS; ++s) {
      u32x4 val = {0u, 0u, 0u, 0u};
      if (16 * s + 8 * hf < D) val = *reinterpret_cast<const u32x4*>(qp + 16 * s + 8 * hf);
      qf[s] = val;
    }
  }
  if constexpr (FQ && CAUSAL && (D == 64 || D == 128))
    fuse_q_producer<T, D>(a, qf, true, pos, pos, hf);
#pragma unroll
  for (int s = 0; s < QS; ++s) __asm__ volatile("" : "+v"(qf[s]));  // Q has arrived
  if (any) issue_v(t * kSkKeys);

  // Fragment addresses.  K fragment s: row lq, chunk 2s + hf.  V^T fragment (chunk ck of 16
  // keys, tile dt): lane L = 16g + 4e + q reads row 16 ck + 4(g/2) + e (+8 for the second half)
  // and columns dt*32 + 16(g&1) + 4q .. +3.
  lds_ptr k_p[QS], v_p[DT];
#pragma unroll
  for (int s = 0; s < QS; ++s)
    k_p[s] = k_lds + lq * RC * 16 + (D == 128 ? (2 * s + hf) ^ (lq & 15) : 2 * s + hf) * 16;
  {
    const int g = lane >> 4, e = (lane >> 2) & 3, q = lane & 3;
    const int row = 4 * (g >> 1) + e;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
      v_p[dt] = v_lds + row * RC * 16 + (D == 128 ? dt ^ e : dt) * 64 + (g & 1) * 32 + q * 8;
  }

  f32x16 oacc[DT];
#pragma unroll
  for (int d = 0; d < DT; ++d)
#pragma unroll
    for (int r = 0; r < 16; ++r) oacc[d][r] = 0.f;
  float mc = 0.f, l = 0.f;  // running row maximum times the scale (log2 units), this half's weights
  const float c = a.scale_log2;
  bool first = true;

  if (any)
    for (;;) {
      const int t0 = t * kSkKeys;
      const bool more = t + NW < n_tiles;
      // ---- S^T (K landed; the younger V transfers may be in flight)
      __builtin_amdgcn_sched_barrier(0);
      wait_vmcnt<NI>();
      __builtin_amdgcn_sched_barrier(0);
      f32x16 s;
#pragma unroll
      for (int r = 0; r < 16; ++r) s[r] = 0.f;
#pragma unroll
      for (int i = 0; i < QS; ++i) s = mfma32<T>(lds_read128(k_p[i], 0), qf[i], s);
      __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): the K tile has been read
      if (more) issue_k(t0 + NW * kSkKeys);

      // ---- softmax: P = 2^(c s - mc) with the running maximum left as it is while no weight
      // sum of a lane passes 2^8; else, and on the first tile, the row maximum is taken.
      if (t0 + kSkKeys - 1 > pos_min) {
        const int rel = pos - t0 - 4 * hf;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int cr = 8 * (r >> 2) + (r & 3);
          s[r] = cr > rel ? -INFINITY : s[r];
        }
      }
      u32x4 pf[2];
      float ls;
      auto weights = [&]() __attribute__((always_inline)) {
        float lsp[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int r = 0; r < 16; r += 2) {
          const uint32_t pk = pack2<f16>(fast_exp2(__builtin_fmaf(s[r], c, -mc)),
                                         fast_exp2(__builtin_fmaf(s[r + 1], c, -mc)));
          pf[r >> 3][(r & 7) >> 1] = pk;
          lsp[(r >> 1) & 3] = sum_pair<f16>(pk, lsp[(r >> 1) & 3]);
        }
        ls = (lsp[0] + lsp[1]) + (lsp[2] + lsp[3]);
      };
      if (!first) weights();
      if (first || __builtin_amdgcn_ballot_w64(!(ls <= kSkSumMax))) {
        float mx = s[0];
#pragma unroll
        for (int r = 1; r < 16; ++r) mx = fmaxf(mx, s[r]);
        mx = fmaxf(mx, partner32(mx)) * c;
        if (first) {
          mc = mx > -INFINITY ? mx : 0.f;  // no visible key yet: none later either
        } else {
          const float mn = fmaxf(mc, mx);
          const float alpha = fast_exp2(mc - mn);
          mc = mn;
          l *= alpha;
#pragma unroll
          for (int d = 0; d < DT; ++d)
#pragma unroll
            for (int r = 0; r < 16; ++r) oacc[d][r] *= alpha;
        }
        weights();
      }
      first = false;
      l += ls;

      // ---- O^T (V landed; the younger K transfers may be in flight)
      if (more) wait_vmcnt<NI>();
      else wait_vmcnt<0>();
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int ck = 0; ck < 2; ++ck)
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
          const u32x2 lo = lds_read_tr(v_p[dt], ck * 16 * RC * 16);
          const u32x2 hi = lds_read_tr(v_p[dt], (ck * 16 + 8) * RC * 16);
          u32x4 vf = {lo[0], lo[1], hi[0], hi[1]};
          if constexpr (kConvV) vf = bf16x8_to_f16x8(vf);
          oacc[dt] = mfma32<f16>(vf, pf[ck], oacc[dt]);
        }
      if (!more) break;
      __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): the V tile has been read
      t += NW;
      issue_v(t * kSkKeys);
    }

  // ------------------------------------------------------------ merge the waves and store
  // O [wave][row][DT * 32], 4-float chunk ch of a row at ch ^ row within its group of 8.
  const float l_row = l + partner32(l);
  const float m_row = l_row > 0.f ? mc : -INFINITY;  // a wave whose keys are all masked
  __syncthreads();  // every wave is done with its tiles
  constexpr int OW = DT * 32;
  float* s_o = reinterpret_cast<float*>(smem);
  float* s_ml = reinterpret_cast<float*>(smem + sk_ml_offset<D, NW>());
  if (hf == 0) {
    s_ml[(wave * kSkRows + lq) * 2] = m_row;
    s_ml[(wave * kSkRows + lq) * 2 + 1] = l_row;
  }
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int rg = 0; rg < 4; ++rg) {
      const int ch = dt * 8 + ((2 * rg + hf) ^ (lq & 7));
      *reinterpret_cast<f32x4*>(s_o + (wave * kSkRows + lq) * OW + ch * 4) =
          f32x4{oacc[dt][4 * rg], oacc[dt][4 * rg + 1], oacc[dt][4 * rg + 2], oacc[dt][4 * rg + 3]};
    }
  __syncthreads();
  for (int x = threadIdx.x; x < kSkRows * NCH; x += NW * kWave) {
    const int row = x / NCH, c8 = x % NCH;  // 8 dimensions of a row
    const int Ro = r_first + row;
    if (Ro > r_last) break;
    float M = -INFINITY, mw[NW];
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      mw[w] = s_ml[(w * kSkRows + row) * 2];
      M = fmaxf(M, mw[w]);
    }
    const float Mu = M > -INFINITY ? M : 0.f;
    float L = 0.f, o[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float f = fast_exp2(mw[w] - Mu);
      L = __builtin_fmaf(f, s_ml[(w * kSkRows + row) * 2 + 1], L);
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const int lc = 2 * c8 + q, ch = (lc & ~7) + ((lc & 7) ^ (row & 7));
        const f32x4 y = *reinterpret_cast<const f32x4*>(s_o + (w * kSkRows + row) * OW + ch * 4);
#pragma unroll
        for (int e = 0; e < 4; ++e) o[4 * q + e] = __builtin_fmaf(f, y[e], o[4 * q + e]);
      }
    }
    const float inv = 1.f / L;
    const int to = Ro / G;
    T* op = reinterpret_cast<T*>(a.o) + (long)(seg_start + to) * a.o_tok_stride +
            (long)(kvh * G + Ro % G) * a.o_head_stride + 8 * c8;
    *reinterpret_cast<u32x4*>(op) =
        u32x4{pack2<T>(o[0] * inv, o[1] * inv), pack2<T>(o[2] * inv, o[3] * inv),
              pack2<T>(o[4] * inv, o[5] * inv), pack2<T>(o[6] * inv, o[7] * inv)};
  }
}

template <bool CAUSAL>
long sk_blocks(const FwdArgs& a) {
  const long tiles = ((long)(CAUSAL ? a.n_q : a.max_seqlen) * a.kv_mul + kSkRows - 1) / kSkRows;
  return tiles * a.Hkv * (CAUSAL ? 1 : a.n_seg);
}

template <typename T, bool CAUSAL, int D, bool FQ, int NW>
hipError_t launch_sk_t(const FwdArgs& a, hipStream_t stream) {
  const long blocks = sk_blocks<CAUSAL>(a);
  if (blocks <= 0) return hipSuccess;
  constexpr int lds = sk_lds<D, NW>();
  const void* fn = (const void*)fwd_sk_kernel<T, CAUSAL, D, FQ, NW>;
  // More than 64 KB of dynamic LDS must be granted per kernel (once per device).
  static unsigned long long configured = 0;
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if (dev >= 64 || !(__atomic_load_n(&configured, __ATOMIC_ACQUIRE) & (1ull << dev))) {
    e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (e != hipSuccess) return e;
    if (dev < 64) __atomic_fetch_or(&configured, 1ull << dev, __ATOMIC_RELEASE);
  }
  hipLaunchKernelGGL((fwd_sk_kernel<T, CAUSAL, D, FQ, NW>), dim3((unsigned)blocks), dim3(NW * kWave),
                     lds, stream, a);
  return hipGetLastError();
}

template <typename T, bool CAUSAL, int D, bool FQ>
hipError_t launch_sk_w(const FwdArgs& a, hipStream_t stream) {
  // 8 waves where a workgroup has a CU of its own anyway and keys enough for them.
  const int keys = CAUSAL ? a.start_pos + a.n_q : a.max_seqlen;
  // 32/8 heads, 256 rows behind 4000 keys: 32.2 us with 4 waves, 28.6 with 8; 137 rows 5.9 and 6.8.
  return sk_blocks<CAUSAL>(a) <= a.n_cu && keys >= 512 ? launch_sk_t<T, CAUSAL, D, FQ, 8>(a, stream)
                                                       : launch_sk_t<T, CAUSAL, D, FQ, 4>(a, stream);
}

template <typename T, bool CAUSAL, int D>
hipError_t launch_sk_d(const FwdArgs& a, hipStream_t stream) {
  if constexpr (CAUSAL && (D == 64 || D == 128))
    if (a.rope_sin) return launch_sk_w<T, CAUSAL, D, true>(a, stream);
  return launch_sk_w<T, CAUSAL, D, false>(a, stream);
}

template <typename T, bool CAUSAL>
hipError_t launch_sk(const FwdArgs& a, hipStream_t stream) {
  switch (a.head_size) {
    case 64: return launch_sk_d<T, CAUSAL, 64>(a, stream);
    case 72: return launch_sk_d<T, CAUSAL, 72>(a, stream);
    case 80: return launch_sk_d<T, CAUSAL, 80>(a, stream);
    case 96: return launch_sk_d<T, CAUSAL, 96>(a, stream);
    case 128: return launch_sk_d<T, CAUSAL, 128>(a, stream);
  }
  return hipErrorInvalidValue;
}

}  // namespace

// Which launches run here, against what they ran on before: the ping-pong kernel (256-query
// workgroups fill the device, or a key split and its merge), else the tile kernel of fwd.hip.
// us, fp16, d 128 unless noted:
//   causal 32/8 heads: 137 rows 8.2 -> 5.9, 512 rows 22.9 -> 9.7, 1536 rows 41.3 -> 38.4, 2048 rows
//   57.7 against 60.1; 12/2: 2048 rows 32.6 -> 25.7, 3072 rows 53.2 -> 49.3, 1024 rows behind 3000
//   36.4 against 36.9; 28/4 (tile kernel before): 2048 rows 68.6 -> 55.0
//   vision, 16 heads, d 72: one image of 1024 26.7 -> 13.3, of 2300 (tile kernel) 67.8 -> 48.2;
//   four of 1024 (fill the device) 30.3 against 40.3
bool fwd_sk_prefers(const FwdArgs& a, int dtype, bool causal) {
  if (!fwd_pp_supports(a, dtype)) return false;
  const long n_q = causal ? a.n_q : a.max_seqlen;
  const long keys = causal ? (long)a.start_pos + a.n_q : a.max_seqlen;
  if (n_q * a.kv_mul >= (1l << 30)) return false;  // packed rows are ints
  // One or two key tiles: the merge costs more than the split saves (24 rows 5.0 against 5.4).
  if (keys <= 64) return false;
  const long blocks = causal ? sk_blocks<true>(a) : sk_blocks<false>(a);
  // Many short segments already fill the device (8 of 256: 10.6 against 11.3).
  if (!causal && keys <= 256 && blocks > 2l * a.n_cu) return false;
  size_t bytes;
  const bool key_split = causal && fwd_pp_key_split(a, dtype, a.n_cu, &bytes) > 0;
  const long pp_blocks = (causal ? 1 : a.n_seg) * ((n_q + 255) / 256) * a.Hq;
  if (!key_split && pp_blocks < 256) return true;  // the tile kernel would run
  // Few rows behind a long prefix: a workgroup's own chain is the longer one (12/2 heads, 128 rows
  // behind 6000 28.0 against 29.4; 28/4 heads, 112 workgroups, 31.8 against 30.1).
  if (key_split && blocks * 4 < a.n_cu && keys > 4096) return false;
  // Wave tiles (32 rows x 32 keys) in all, each 16 KB through a CU's L2 path (10 KB at head size
  // 64); for segments an upper bound, since the host does not know their lengths.
  const long tiles = causal ? blocks * (2l * a.start_pos + a.n_q) / 64
                            : ((long)a.n_q * a.kv_mul + 31) / 32 * a.Hkv * ((keys + 31) / 32);
  return tiles * (causal && a.head_size == 64 ? 5 : 8) <= 1280l * a.n_cu;
}

hipError_t launch_fwd_sk(const FwdArgs& a, int dtype, bool causal, hipStream_t stream) {
  if (dtype == kF16) return causal ? launch_sk<f16, true>(a, stream) : launch_sk<f16, false>(a, stream);
  return causal ? launch_sk<bf16, true>(a, stream) : launch_sk<bf16, false>(a, stream);
}

}  // namespace orin
