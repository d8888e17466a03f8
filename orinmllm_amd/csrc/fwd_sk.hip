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
// second launch that merges partials.  Where the grid is large enough, a workgroup owns two such
// sets of 32 rows: each K and V fragment read from LDS serves two products.  Rows of the query heads that share a kv head are packed
// (row R of a kv head = query R / kv_mul, head R % kv_mul of its group): short prompts fill the
// 32 rows, and little of a causal diagonal tile is masked.
//
// The price: K and V are read from L2 once per 32 or 64 rows (a CU streams ~110 GB/s from L2), with
// no wave sharing another's tile, so large launches stay on fwd_pp.hip.
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
#include <algorithm>
#include <type_traits>

#include "common.h"
#include "fwd_tile.h"
#include "kernels.h"

namespace orin {

namespace {

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
// K and V tiles of the waves (1 KB per transfer), or O [wave][32 rows][DT * 32] in the merge; then
// the Q fragments of two row sets, or the waves' (m, l).
template <int D, int NW>
constexpr int sk_q_offset() {
  const int tiles = NW * 2 * sk_transfers<D>() * 1024;
  const int merge = NW * 32 * ((D + 31) / 32 * 32) * 4;
  return tiles > merge ? tiles : merge;
}
template <int D, int RS, int NW>
constexpr int sk_lds() {
  const int q = RS > 1 ? RS * ((D + 15) / 16) * 1024 : 0, ml = NW * 32 * RS * 2 * 4;
  return sk_q_offset<D, NW>() + (q > ml ? q : ml);
}
// A lane's 16 weights of one tile may sum to at most this before the row maximum is raised.
constexpr float kSkSumMax = 256.0f;

// FQ: the query rows are raw and the Q producer runs on the fragments (a.rope_sin set).
template <typename T, bool CAUSAL, int D, bool FQ, int RS, int NW>
__global__ void __launch_bounds__(NW * kWave, 2) fwd_sk_kernel(FwdArgs a) {
  constexpr int QS = (D + 15) / 16;  // 16-wide slices of the QK contraction
  constexpr int DT = (D + 31) / 32;  // 32-wide output tiles of O^T
  constexpr int NCH = D / 8;         // valid 16-byte chunks of a K / V row
  constexpr bool kConvV = !std::is_same<T, f16>::value;
  constexpr int kSkRows = 32 * RS;   // rows per workgroup
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
  // This lane's row of each set (rows past the end repeat the last one and are not stored).
  int tok[RS], head[RS], pos[RS];  // pos: the last key the row sees
#pragma unroll
  for (int u = 0; u < RS; ++u) {
    const int R = min(r_first + 32 * u + lq, r_last);
    tok[u] = R / G;
    head[u] = kvh * G + R % G;
    pos[u] = CAUSAL ? a.start_pos + tok[u] : kv_len - 1;
  }
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
  const uint32_t k_addr = __builtin_amdgcn_readfirstlane(lds_addr(my));
  auto issue = [&](const T* x, int t0, auto is_v) __attribute__((always_inline)) {
    constexpr bool V = decltype(is_v)::value;
    const uint32_t dst = k_addr + (V ? kTile : 0);
    const char* base = reinterpret_cast<const char*>(x + (long)t0 * tstr);
    // Rows past the sequence read the last chunk of its last row: finite values, in bounds.
    const uint32_t lim =
        (uint32_t)min(kv_len - 1 - t0, kSkKeys - 1) * row_bytes + (D - 8) * (uint32_t)sizeof(T);
#pragma unroll
    for (int b = 0; b < NI; ++b) {
      const uint32_t off = D == 128 ? (V ? v_off : k_off[b & 3]) + 4 * b * row_bytes : k_off[b % NOK];
      dma16_s(base, min(off, lim), dst + b * 1024);
    }
  };
  auto issue_k = [&](int t0) __attribute__((always_inline)) { issue(kb, t0, std::false_type{}); };
  auto issue_v = [&](int t0) __attribute__((always_inline)) { issue(vb, t0, std::true_type{}); };

  int t = wave;
  const bool any = wave < n_tiles;
  if (any) issue_k(t * kSkKeys);

  // ------------------------------------------------------------ Q fragments
  // One row set: in registers.  Two: wave u loads set u and all waves read the fragments from
  // LDS ([set][slice][lane]), which leaves the registers to O.
  u32x4 qf[QS];
  char* const q_sm = smem + sk_q_offset<D, NW>();
#pragma unroll
  for (int u = 0; u < RS; ++u) {
    if (RS > 1 && wave != u) continue;
    const T* qp = reinterpret_cast<const T*>(a.q) + (long)(seg_start + tok[u]) * a.q_tok_stride +
                  (long)head[u] * a.q_head_stride;
#pragma unroll
    for (int s = 0; s < QS; ++s) {
      u32x4 val = {0u, 0u, 0u, 0u};
      if (16 * s + 8 * hf < D) val = *reinterpret_cast<const u32x4*>(qp + 16 * s + 8 * hf);
      qf[s] = val;
    }
    if constexpr (FQ && CAUSAL && (D == 64 || D == 128))
      fuse_q_producer<T, D>(a, qf, true, pos[u], pos[u], hf);
#pragma unroll
    for (int s = 0; s < QS; ++s) __asm__ volatile("" : "+v"(qf[s]));  // Q has arrived
    if constexpr (RS > 1) {
#pragma unroll
      for (int s = 0; s < QS; ++s)
        *reinterpret_cast<u32x4*>(q_sm + ((u * QS + s) * 64 + lane) * 16) = qf[s];
    }
  }
  if constexpr (RS > 1) __syncthreads();
  const lds_ptr q_p = (lds_ptr)(q_sm + lane * 16);
  auto q_frag = [&](int u, int s) __attribute__((always_inline)) {
    if constexpr (RS > 1) return lds_read128(q_p, (u * QS + s) * 1024);
    return qf[s];
  };
  if (any) issue_v(t * kSkKeys);

  // Fragment addresses.  K fragment s: row lq, chunk 2s + hf.  V^T fragment (chunk ck of 16
  // keys, tile dt): lane L = 16g + 4e + q reads row 16 ck + 4(g/2) + e (+8 for the second half)
  // and columns dt*32 + 16(g&1) + 4q .. +3.
  // At head size 128 (256-byte rows, tiles at multiples of 1 KB) the swizzle makes fragment s
  // (tile dt) the first one's address with 32 s (64 dt) flipped.
  const lds_ptr k_lds = (lds_ptr)my, v_lds = k_lds + kTile;
  uint32_t k_a = lq * RC * 16 + (D == 128 ? hf ^ (lq & 15) : hf) * 16;
  uint32_t v_a;
  {
    const int g = lane >> 4, e = (lane >> 2) & 3, q = lane & 3;
    v_a = (4 * (g >> 1) + e) * RC * 16 + (D == 128 ? e : 0) * 64 + (g & 1) * 32 + q * 8;
  }
  auto k_p = [&](int s) __attribute__((always_inline)) {
    return k_lds + (D == 128 ? k_a ^ (32 * s) : k_a + 32 * s);
  };
  auto v_p = [&](int dt) __attribute__((always_inline)) {
    return v_lds + (D == 128 ? v_a ^ (64 * dt) : v_a + 64 * dt);
  };

  constexpr int kVAhead = DT < 2 ? 2 : 3;  // V fragments read ahead of their products
  f32x16 oacc[RS][DT];
  // Running row maximum times the scale (log2 units) and this half's weights.
  float mc[RS], l[RS];
#pragma unroll
  for (int u = 0; u < RS; ++u) {
    mc[u] = l[u] = 0.f;
#pragma unroll
    for (int d = 0; d < DT; ++d)
#pragma unroll
      for (int r = 0; r < 16; ++r) oacc[u][d][r] = 0.f;
  }
  const float c = a.scale_log2;
  bool first = true;

  if (any)
    for (;;) {
      const int t0 = t * kSkKeys;
      const bool more = t + NW < n_tiles;
      // Two row sets and V's conversion: the fragment addresses are formed where they are used,
      // not kept in registers (24 spilled otherwise).
      if constexpr (RS > 1 && kConvV) __asm__ volatile("" : "+v"(k_a), "+v"(v_a));
      // ---- S^T (K landed; the younger V transfers may be in flight)
      __builtin_amdgcn_sched_barrier(0);
      wait_vmcnt<NI>();
      __builtin_amdgcn_sched_barrier(0);
      f32x16 s[RS];
#pragma unroll
      for (int u = 0; u < RS; ++u)
#pragma unroll
        for (int r = 0; r < 16; ++r) s[u][r] = 0.f;
#pragma unroll
      for (int i = 0; i < QS; ++i) {
        const u32x4 kf = lds_read128(k_p(i), 0);
#pragma unroll
        for (int u = 0; u < RS; ++u) s[u] = mfma32<T>(kf, q_frag(u, i), s[u]);
      }
      __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): the K tile has been read
      if (more) issue_k(t0 + NW * kSkKeys);

      // ---- softmax: P = 2^(c s - mc) with the running maximum left as it is while no weight
      // sum of a lane passes 2^8; else, and on the first tile, the row maximum is taken.
      u32x4 pf[RS][2];
#pragma unroll
      for (int u = 0; u < RS; ++u) {
        if (t0 + kSkKeys - 1 > pos_min) {
          const int rel = pos[u] - t0 - 4 * hf;
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int cr = 8 * (r >> 2) + (r & 3);
            s[u][r] = cr > rel ? -INFINITY : s[u][r];
          }
        }
        float ls;
        auto weights = [&]() __attribute__((always_inline)) {
          float lsp[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int r = 0; r < 16; r += 2) {
            const uint32_t pk = pack2<f16>(fast_exp2(__builtin_fmaf(s[u][r], c, -mc[u])),
                                           fast_exp2(__builtin_fmaf(s[u][r + 1], c, -mc[u])));
            pf[u][r >> 3][(r & 7) >> 1] = pk;
            lsp[(r >> 1) & 3] = sum_pair<f16>(pk, lsp[(r >> 1) & 3]);
          }
          ls = (lsp[0] + lsp[1]) + (lsp[2] + lsp[3]);
        };
        if (!first) weights();
        if (first || __builtin_amdgcn_ballot_w64(!(ls <= kSkSumMax))) {
          float mx = s[u][0];
#pragma unroll
          for (int r = 1; r < 16; ++r) mx = fmaxf(mx, s[u][r]);
          mx = fmaxf(mx, partner32(mx)) * c;
          if (first) {
            mc[u] = mx > -INFINITY ? mx : 0.f;  // no visible key yet: none later either
          } else {
            const float mn = fmaxf(mc[u], mx);
            const float alpha = fast_exp2(mc[u] - mn);
            mc[u] = mn;
            l[u] *= alpha;
#pragma unroll
            for (int d = 0; d < DT; ++d)
#pragma unroll
              for (int r = 0; r < 16; ++r) oacc[u][d][r] *= alpha;
          }
          weights();
        }
        l[u] += ls;
      }
      first = false;

      // ---- O^T (V landed; the younger K transfers may be in flight)
      if (more) wait_vmcnt<NI>();
      else wait_vmcnt<0>();
      __builtin_amdgcn_sched_barrier(0);
      auto v_frag = [&](int i) __attribute__((always_inline)) {
        const int dt = i % DT, row = i / DT * 16;
        const u32x2 lo = lds_read_tr(v_p(dt), row * RC * 16);
        const u32x2 hi = lds_read_tr(v_p(dt), (row + 8) * RC * 16);
        return u32x4{lo[0], lo[1], hi[0], hi[1]};
      };
      u32x4 vr[kVAhead];
#pragma unroll
      for (int i = 0; i < kVAhead; ++i) vr[i] = v_frag(i);
#pragma unroll
      for (int i = 0; i < 2 * DT; ++i) {
        u32x4 vf = vr[i % kVAhead];
        if constexpr (kConvV) vf = bf16x8_to_f16x8(vf);
        if (i + kVAhead < 2 * DT) vr[i % kVAhead] = v_frag(i + kVAhead);
#pragma unroll
        for (int u = 0; u < RS; ++u)
          oacc[u][i % DT] = mfma32<f16>(vf, pf[u][i / DT], oacc[u][i % DT]);
        // Two row sets leave no registers for the scheduler to gather the conversions early.
        if constexpr (RS > 1 && kConvV) __builtin_amdgcn_sched_barrier(0);
      }
      if (!more) break;
      __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): the V tile has been read
      t += NW;
      issue_v(t * kSkKeys);
    }

  // ------------------------------------------------------------ merge the waves and store
  // O [wave][row][DT * 32] of one row set at a time, 4-float chunk ch of a row at ch ^ row within
  // its group of 8; (m, l) [wave][kSkRows][2] take the Q fragments' place.
  constexpr int OW = DT * 32;
  float* s_o = reinterpret_cast<float*>(smem);
  float* s_ml = reinterpret_cast<float*>(q_sm);
#pragma unroll
  for (int u = 0; u < RS; ++u) {
    const float l_row = l[u] + partner32(l[u]);
    const float m_row = l_row > 0.f ? mc[u] : -INFINITY;  // a wave whose keys are all masked
    __syncthreads();  // every wave is done with its tiles (u > 0: with the last set's O)
    if (hf == 0) {
      s_ml[(wave * kSkRows + 32 * u + lq) * 2] = m_row;
      s_ml[(wave * kSkRows + 32 * u + lq) * 2 + 1] = l_row;
    }
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int rg = 0; rg < 4; ++rg) {
        const int ch = dt * 8 + ((2 * rg + hf) ^ (lq & 7));
        *reinterpret_cast<f32x4*>(s_o + (wave * 32 + lq) * OW + ch * 4) =
            f32x4{oacc[u][dt][4 * rg], oacc[u][dt][4 * rg + 1], oacc[u][dt][4 * rg + 2],
                  oacc[u][dt][4 * rg + 3]};
      }
    __syncthreads();
    for (int x = threadIdx.x; x < 32 * NCH; x += NW * kWave) {
      const int row = x / NCH, c8 = x % NCH;  // 8 dimensions of a row
      const int Ro = r_first + 32 * u + row;
      if (Ro > r_last) break;
      float M = -INFINITY, mw[NW];
#pragma unroll
      for (int w = 0; w < NW; ++w) {
        mw[w] = s_ml[(w * kSkRows + 32 * u + row) * 2];
        M = fmaxf(M, mw[w]);
      }
      const float Mu = M > -INFINITY ? M : 0.f;
      float L = 0.f, o[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int w = 0; w < NW; ++w) {
        const float f = fast_exp2(mw[w] - Mu);
        L = __builtin_fmaf(f, s_ml[(w * kSkRows + 32 * u + row) * 2 + 1], L);
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          const int lc = 2 * c8 + q, ch = (lc & ~7) + ((lc & 7) ^ (row & 7));
          const f32x4 y = *reinterpret_cast<const f32x4*>(s_o + (w * 32 + row) * OW + ch * 4);
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
}

template <bool CAUSAL>
long sk_blocks(const FwdArgs& a, int rows) {
  const long tiles = ((long)(CAUSAL ? a.n_q : a.max_seqlen) * a.kv_mul + rows - 1) / rows;
  return tiles * a.Hkv * (CAUSAL ? 1 : a.n_seg);
}

template <typename T, bool CAUSAL, int D, bool FQ, int RS, int NW>
hipError_t launch_sk_t(const FwdArgs& a, hipStream_t stream) {
  const long blocks = sk_blocks<CAUSAL>(a, 32 * RS);
  if (blocks <= 0) return hipSuccess;
  constexpr int lds = sk_lds<D, RS, NW>();
  const void* fn = (const void*)fwd_sk_kernel<T, CAUSAL, D, FQ, RS, NW>;
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
  hipLaunchKernelGGL((fwd_sk_kernel<T, CAUSAL, D, FQ, RS, NW>), dim3((unsigned)blocks), dim3(NW * kWave),
                     lds, stream, a);
  return hipGetLastError();
}

// Two row sets per workgroup: a row costs about 0.8 of what it costs with one, but the units of work
// are twice as large.  Compared is the time of the fullest CU in workgroups times keys: the longest
// workgroup's, or the CU's share of the average one; with one set and more workgroups than CUs some
// CU holds two of them at once.  us, fp16, d 128, one set / two: 32/8 heads, 512 rows 9.6 / 11.0, 1024
// rows 22.1 / 18.6, 2048 rows 60.5 / 49.6; 28/4, 1531 rows 36.7 / 30.6; 12/2, 1792 rows 22.3 / 25.3,
// 2560 rows 36.2 / 34.9, 1000 rows behind 2500 32.9 / 31.7 (bf16 37.4 / 33.5).
template <bool CAUSAL>
bool sk_two_sets(const FwdArgs& a) {
  const long longest = CAUSAL ? a.start_pos + (long)a.n_q : 1;
  const long average2 = CAUSAL ? 2l * a.start_pos + a.n_q : 2;  // twice the average
  const long b1 = sk_blocks<CAUSAL>(a, 32), b2 = sk_blocks<CAUSAL>(a, 64), cu = a.n_cu;
  const long one = b1 <= cu ? 2 * longest * cu : std::max(2 * cu, b1) * average2;
  const long two = std::max(2 * longest * cu, b2 * average2);
  return 8 * two < 5 * one;
}

template <typename T, bool CAUSAL, int D, bool FQ, int RS>
hipError_t launch_sk_w(const FwdArgs& a, hipStream_t stream) {
  // 8 waves where a workgroup has a CU of its own anyway and keys enough for them.
  const int keys = CAUSAL ? a.start_pos + a.n_q : a.max_seqlen;
  // 32/8 heads, 256 rows behind 4000 keys: 32.2 us with 4 waves, 28.6 with 8; 137 rows 5.9 and 6.8.
  return sk_blocks<CAUSAL>(a, 32 * RS) <= a.n_cu && keys >= 512
             ? launch_sk_t<T, CAUSAL, D, FQ, RS, 8>(a, stream)
             : launch_sk_t<T, CAUSAL, D, FQ, RS, 4>(a, stream);
}

template <typename T, bool CAUSAL, int D, bool FQ>
hipError_t launch_sk_r(const FwdArgs& a, hipStream_t stream) {
  return sk_two_sets<CAUSAL>(a) ? launch_sk_w<T, CAUSAL, D, FQ, 2>(a, stream)
                                : launch_sk_w<T, CAUSAL, D, FQ, 1>(a, stream);
}

template <typename T, bool CAUSAL, int D>
hipError_t launch_sk_d(const FwdArgs& a, hipStream_t stream) {
  if constexpr (CAUSAL && (D == 64 || D == 128))
    if (a.rope_sin) return launch_sk_r<T, CAUSAL, D, true>(a, stream);
  return launch_sk_r<T, CAUSAL, D, false>(a, stream);
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
//   causal 32/8 heads: 137 rows 8.2 -> 5.7, 512 rows 23.1 -> 9.6, 1531 rows 42.0 -> 33.1, 2560 rows
//   74.2 -> 73.0, 3072 rows 90.8 against 96.6; 28/4: 1531 rows 40.4 -> 30.6 (bf16 41.2 -> 31.6); 12/2:
//   2560 rows 43.1 -> 34.9, 1000 rows behind 2500 34.1 -> 31.7 (bf16 38.2 -> 33.5)
//   vision, 16 heads, d 72: one image of 1024 27.2 -> 12.7, of 2300 (tile kernel) 67.7 -> 53.0;
//   four of 1024 (fill the device) 30.5 against 36.9
bool fwd_sk_prefers(const FwdArgs& a, int dtype, bool causal) {
  if (!fwd_pp_supports(a, dtype)) return false;
  const long n_q = causal ? a.n_q : a.max_seqlen;
  const long keys = causal ? (long)a.start_pos + a.n_q : a.max_seqlen;
  if (n_q * a.kv_mul >= (1l << 30)) return false;  // packed rows are ints
  // One or two key tiles: the merge costs more than the split saves (24 rows 5.0 against 5.4).
  if (keys <= 64) return false;
  const long blocks = causal ? sk_blocks<true>(a, 32) : sk_blocks<false>(a, 32);
  // Many short segments already fill the device (8 of 256: 10.6 against 11.3).
  if (!causal && keys <= 256 && blocks > 2l * a.n_cu) return false;
  // Wave tiles (32 rows x 32 keys) in all; for segments an upper bound, since the host does not know
  // their lengths.
  const long tiles = causal ? blocks * (2l * a.start_pos + a.n_q) / 64
                            : ((long)a.n_q * a.kv_mul + 31) / 32 * a.Hkv * ((keys + 31) / 32);
  const bool causal_fits = causal && tiles * (a.head_size == 64 ? 5 : 8) <= 3200l * a.n_cu;
  if (causal_fits && keys <= 4096) return true;  // whatever the key split would be
  size_t bytes;
  const long chunk = causal ? fwd_pp_key_split(a, dtype, a.n_cu, &bytes) : 0;
  const long pp_blocks = (causal ? 1 : a.n_seg) * ((n_q + 255) / 256) * a.Hq;
  if (chunk == 0 && pp_blocks < 256) return true;  // the tile kernel would run
  // Few rows behind a long prefix: a workgroup's own chain is the longer one (12/2 heads, 128 rows
  // behind 6000 28.0 against 29.4; 28/4 heads, 112 workgroups, 31.8 against 30.1).
  if (chunk > 0 && blocks * 4 < a.n_cu && keys > 4096) return false;
  if (!causal) return tiles * 8 <= 1280l * a.n_cu;
  // A key split whose chunks cover 84 % of the device, behind a long prefix (700 rows behind 3500: 28/4
  // heads 53.6 against 61.7, 12/2 32.0 against 34.1; 512 behind 6000, 28/4, 82 %, 60.2 against 57.5).
  if (chunk > 0 && a.start_pos >= a.n_q && keys > 4096 &&
      pp_blocks * (2l * a.start_pos + a.n_q) * 100 > 84 * 128 * chunk * a.n_cu)
    return false;
  return causal_fits;
}

hipError_t launch_fwd_sk(const FwdArgs& a, int dtype, bool causal, hipStream_t stream) {
  if (dtype == kF16) return causal ? launch_sk<f16, true>(a, stream) : launch_sk<f16, false>(a, stream);
  return causal ? launch_sk<bf16, true>(a, stream) : launch_sk<bf16, false>(a, stream);
}

}  // namespace orin
