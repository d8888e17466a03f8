"""Attention whose keys are split inside the workgroup (fwd_sk.hip): tiles of 32 or 64 packed
query rows, 32-key tiles over 4 or 8 waves.  Shapes sit at the edges of those tiles and of the dispatch
(up to 64 keys, and launches that fill the device, run elsewhere)."""
import numpy as np
import pytest
import torch

from oracle import oracle
from orinmllm_amd import kernel as K
from tests.test_gpu_prefill import run_prefill, sample_rows
from tests.test_gpu_vision import TORCH, dev, vision_inputs
from tests.util import assert_lowp_close, normal, quantize


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["fp16", "bf16"])
@pytest.mark.parametrize("d", [64, 72, 80, 96, 128])
@pytest.mark.parametrize("Hq,Hkv,start,S", [(4, 2, 0, 65), (3, 1, 63, 2), (7, 1, 64, 33), (5, 5, 95, 1),
                                            (2, 2, 1000, 31), (12, 2, 600, 129)])
def test_sk_causal_tile_edges(kind, d, Hq, Hkv, start, S):
    """4 waves below 512 keys, 8 from there on; row tiles that end inside a position's heads."""
    rng = np.random.default_rng(9000 + d + S + start)
    q, kc, vc, out = run_prefill(kind, start, S, Hq, Hkv, d, start + S + 5, 2, 1, rng)
    rows = sample_rows(S, 16, rng)
    ref = oracle.prefill_causal(start, q, kc, vc, Hq, Hkv, d, rows=rows, nthreads=8)
    assert_lowp_close(out[rows], ref, what=f"{kind} d {d} S {S} start {start}")


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["fp16", "bf16"])
@pytest.mark.parametrize("Hq,Hkv,start,S", [(32, 8, 0, 260), (28, 4, 0, 1100), (12, 2, 300, 1700)])
def test_sk_causal_many_workgroups(kind, Hq, Hkv, start, S):
    """Grids above one, two and more workgroups per CU (the reversed second block among them)."""
    rng = np.random.default_rng(9100 + S)
    q, kc, vc, out = run_prefill(kind, start, S, Hq, Hkv, 128, start + S, 1, 0, rng)
    rows = sample_rows(S, 24, rng)
    ref = oracle.prefill_causal(start, q, kc, vc, Hq, Hkv, 128, rows=rows, nthreads=8)
    assert_lowp_close(out[rows], ref, what=f"{kind} S {S}")


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["fp16", "bf16"])
@pytest.mark.parametrize("d", [64, 72, 80, 96, 128])
@pytest.mark.parametrize("cu", [(0, 65), (0, 1, 33, 33, 130), (0, 700, 731), (0, 31, 63, 95, 1200)])
def test_sk_varlen_segments(kind, d, cu):
    """Segments of one token, none, a whole tile and a tail; 4 and 8 waves."""
    rng = np.random.default_rng(9200 + d + cu[-1])
    H, N = 3, cu[-1]
    q, k, v = vision_inputs(rng, np.array(cu, np.int32), H, d, kind)
    out = torch.zeros(N, H * d, device="cuda", dtype=TORCH[kind])
    K.vision_attention_varlen_cu(dev(q, kind), dev(k, kind), dev(v, kind), out,
                                 torch.tensor(cu, dtype=torch.int32, device="cuda"),
                                 int(np.diff(cu).max()), H, d)
    torch.cuda.synchronize()
    rows = np.unique(np.concatenate([[c for c in cu if c < N], np.array(cu[1:]) - 1,
                                     rng.integers(0, N, 16)]))
    ref = oracle.varlen_bidir(q, k, v, np.array(cu, np.int32), rows=rows, nthreads=8)
    assert_lowp_close(out.float().cpu().numpy()[rows], ref, what=f"{kind} d {d} {cu}")


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["fp16", "bf16"])
@pytest.mark.parametrize("d", [64, 72, 80, 96, 128])
@pytest.mark.parametrize("Hq,Hkv,start,S", [(16, 16, 0, 1501), (9, 3, 2600, 1333), (32, 8, 190, 290)])
def test_sk_causal_two_row_sets(kind, d, Hq, Hkv, start, S):
    """64 rows per workgroup (grids of more than two workgroups of 32 rows per CU, or that little
    above one): last workgroups with one set, or part of one, in range; 4 and 8 waves."""
    rng = np.random.default_rng(9400 + d + S)
    q, kc, vc, out = run_prefill(kind, start, S, Hq, Hkv, d, start + S, 1, 0, rng)
    rows = np.unique(np.concatenate([sample_rows(S, 20, rng), [0, 31, 32, 63, 64, S - 2, S - 1]]))
    ref = oracle.prefill_causal(start, q, kc, vc, Hq, Hkv, d, rows=rows, nthreads=8)
    assert_lowp_close(out[rows], ref, what=f"{kind} d {d} S {S} start {start}")


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["fp16", "bf16"])
@pytest.mark.parametrize("d", [64, 72, 80, 96, 128])
@pytest.mark.parametrize("cu", [(0, 1000, 1001, 1700), (0, 1473)])
def test_sk_varlen_two_row_sets(kind, d, cu):
    rng = np.random.default_rng(9500 + d + cu[-1])
    H, N = 16, cu[-1]
    q, k, v = vision_inputs(rng, np.array(cu, np.int32), H, d, kind)
    out = torch.zeros(N, H * d, device="cuda", dtype=TORCH[kind])
    K.vision_attention_varlen_cu(dev(q, kind), dev(k, kind), dev(v, kind), out,
                                 torch.tensor(cu, dtype=torch.int32, device="cuda"),
                                 int(np.diff(cu).max()), H, d)
    torch.cuda.synchronize()
    rows = np.unique(np.concatenate([[c for c in cu if c < N], np.array(cu[1:]) - 1, [31, 32, 63, 64],
                                     rng.integers(0, N, 16)]))
    ref = oracle.varlen_bidir(q, k, v, np.array(cu, np.int32), rows=rows, nthreads=8)
    assert_lowp_close(out.float().cpu().numpy()[rows], ref, what=f"{kind} d {d} {cu}")


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["fp16", "bf16"])
@pytest.mark.parametrize("Hq,Hkv,d,start,S", [(28, 4, 128, 0, 700), (6, 2, 64, 500, 90), (28, 4, 128, 0, 1110),
                                              (16, 16, 64, 0, 1501), (12, 2, 128, 2500, 1000)])
def test_sk_fused_q_and_aliased_output(kind, Hq, Hkv, d, start, S):
    """The fused Q producer gives the bits of the producer followed by the prefill, and the
    output may be the query."""
    rng = np.random.default_rng(9300 + S)
    t, n = TORCH[kind], start + S
    q, k, v = (dev(quantize(normal(rng, (S, h * d)), kind), kind) for h in (Hq, Hkv, Hkv))
    w = dev(quantize(1 + 0.1 * normal(rng, d), kind), kind)
    sn, cs = (torch.empty(n, d, device="cuda") for _ in range(2))
    K.sin_cos_cache_calc_cu(d, n, sn, cs)
    kc, vc = (dev(quantize(normal(rng, (1, n, Hkv * d)), kind), kind) for _ in range(2))
    raw, fused, plain = q.clone(), torch.empty_like(q), torch.empty_like(q)
    K.qk_norm_rope_cu(q, k, v, w, w, sn, cs, kc, vc, 0, n, start, S, Hq, Hkv, d)
    K.flash_attention_prefill_cu(start, S, Hq, Hkv, d, Hq // Hkv, 0, n, Hkv * d, q, plain, kc, vc)
    K.flash_attention_prefill_qk_norm_rope_cu(start, S, Hq, Hkv, d, Hq // Hkv, 0, n, Hkv * d, raw,
                                              fused, kc, vc, w, sn, cs)
    assert torch.equal(fused, plain)
    K.flash_attention_prefill_cu(start, S, Hq, Hkv, d, Hq // Hkv, 0, n, Hkv * d, q, q, kc, vc)
    assert torch.equal(q, plain)
    assert t == plain.dtype
