"""The matrix-core split decode and the split merge: tile edges, both workgroup shapes, rows of
many splits, the single-sequence split size that follows the row's length, and its workspaces."""
import numpy as np
import pytest
import torch

from oracle import oracle
from orinmllm_amd import _lib
from orinmllm_amd import kernel as K
from tests.test_gpu_decode import TORCH, dev, host, make_paged
from tests.util import assert_fp32_close, assert_lowp_close, normal, quantize

EDGES = np.array([1, 15, 16, 17, 63, 64, 65, 127, 128, 129, 257], np.int32)


def run_both(rng, lens, Hq, Hkv, d, kind, split, maxlen, layout=K.KV_LAYOUT_HEAD_MAJOR, bs=16):
    kc, vc, kp, vp, bt = make_paged(rng, lens, Hkv, d, bs, kind)
    if layout == K.KV_LAYOUT_HEAD_MAJOR:
        kp, vp = kp.transpose(0, 2, 1, 3), vp.transpose(0, 2, 1, 3)
    bt = np.pad(bt, ((0, 0), (0, max(0, (maxlen + bs - 1) // bs - bt.shape[1]))))
    q = quantize(normal(rng, (len(lens), Hq, d)), kind)
    lens_d = torch.from_numpy(lens).cuda()
    op = torch.full((len(lens), Hq, d), 7.0, device="cuda", dtype=TORCH[kind])
    oc = torch.full_like(op, 7.0)
    K.paged_decode_cu(dev(q, kind), dev(kp, kind), dev(vp, kind), op, torch.from_numpy(bt).cuda(),
                      lens_d, maxlen, split_tokens=split, layout=layout)
    K.batched_decode_cu(dev(q, kind), dev(kc, kind), dev(vc, kind), oc, lens_d, maxlen, Hkv,
                        split_tokens=split)
    torch.cuda.synchronize()
    assert torch.equal(op, oc), "paged != contiguous"
    close = assert_fp32_close if kind == "fp32" else None
    ref = oracle.decode_contig(q, kc, vc, lens)
    if close:
        close(host(op), ref, d, what=f"split {split}")
    else:
        assert_lowp_close(host(op), ref, what=f"split {split}")


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["fp16", "bf16"])
@pytest.mark.parametrize("Hq,Hkv,d", [(7, 1, 128), (32, 2, 64), (3, 3, 128), (16, 1, 128)])
@pytest.mark.parametrize("split", [0, 64, 128])
def test_split_decode_tile_edges(kind, Hq, Hkv, d, split):
    """Few workgroups: 8 waves, K straight into the MFMA layout."""
    rng = np.random.default_rng(8100 + Hq + d + split)
    run_both(rng, EDGES, Hq, Hkv, d, kind, split, int(EDGES.max()), bs=8)


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["fp16", "bf16"])
@pytest.mark.parametrize("Hq,Hkv,d,layout", [(28, 4, 128, K.KV_LAYOUT_TOKEN_MAJOR),
                                             (12, 12, 64, K.KV_LAYOUT_HEAD_MAJOR),
                                             (64, 4, 128, K.KV_LAYOUT_HEAD_MAJOR)])
def test_split_decode_many_workgroups(kind, Hq, Hkv, d, layout):
    """More than two workgroups per CU (the bound of 9000 tokens sets the launch): 4 waves, K
    and V through LDS, 16 heads per kv head among them."""
    rng = np.random.default_rng(8200 + Hq + d)
    run_both(rng, EDGES, Hq, Hkv, d, kind, 64, 9000, layout)


@pytest.mark.gpu
@pytest.mark.parametrize("kind,Hq,Hkv,d", [("fp16", 8, 2, 128), ("bf16", 4, 1, 64),
                                           ("fp32", 4, 2, 128), ("fp16", 4, 2, 256)])
def test_merge_of_many_splits(kind, Hq, Hkv, d):
    """Rows of 1, 2, 32, 33 and 101 splits: up to 4 per merge group at first, then a loop."""
    rng = np.random.default_rng(8300 + d)
    run_both(rng, np.array([64, 100, 2048, 2049, 6401], np.int32), Hq, Hkv, d, kind, 64, 6401)


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["fp16", "bf16"])
@pytest.mark.parametrize("Hq,Hkv,d", [(32, 8, 128), (12, 2, 128), (12, 12, 64), (128, 8, 128)])
def test_single_sequence_split_follows_length(kind, Hq, Hkv, d):
    """Host and device positions give the same bits (the split size is the row length's, not the
    launch's) and match the oracle, at the edges of the split-size rule."""
    rng = np.random.default_rng(8400 + Hq)
    cap = 5000
    kc = quantize(normal(rng, (1, cap, Hkv * d)), kind)
    vc = quantize(normal(rng, (1, cap, Hkv * d)), kind)
    q = quantize(normal(rng, Hq * d), kind)
    qd, kd, vd = dev(q, kind), dev(kc, kind), dev(vc, kind)
    p = torch.zeros(1, dtype=torch.int32, device="cuda")
    a, b = (torch.full((Hq * d,), 7.0, device="cuda", dtype=TORCH[kind]) for _ in range(2))
    for pos in [0, 127, 128, 129, 511, 1023, 1024, 2047, 2048, 4999]:
        p.fill_(pos)
        K.flash_attention_decode_cu(pos, Hq, Hkv, d, Hq // Hkv, 0, cap, Hkv * d, qd, a, kd, vd)
        K.flash_attention_decode_fp16_gpu_pos_cu(p, Hq, Hkv, d, Hq // Hkv, 0, cap, Hkv * d, qd, b,
                                                 kd, vd)
        torch.cuda.synchronize()
        assert torch.equal(a, b), pos
        ref, _ = oracle.mha_kernel(pos, Hq, 0, cap, Hkv * d, Hq // Hkv, d, q, kc, vc)
        assert_lowp_close(host(a), ref, what=f"{kind} pos {pos}")


@pytest.mark.gpu
@pytest.mark.parametrize("cap_rows,reserve_rows", [(256, 0), (4096, 256 * 16)])
def test_capture_with_the_fixed_splits_workspace(cap_rows, reserve_rows):
    """A capture whose stream holds no workspace (a cache of up to 256 rows) or only that of
    256-token splits still runs, with those splits."""
    lib = _lib.load()
    rng = np.random.default_rng(8500)
    Hq, Hkv, d = 32, 8, 128
    kc = quantize(normal(rng, (1, cap_rows, Hkv * d)), "fp16")
    vc = quantize(normal(rng, (1, cap_rows, Hkv * d)), "fp16")
    q = quantize(normal(rng, Hq * d), "fp16")
    qd, kd, vd = dev(q, "fp16"), dev(kc, "fp16"), dev(vc, "fp16")
    p = torch.zeros(1, dtype=torch.int32, device="cuda")
    out = torch.full((Hq * d,), 7.0, device="cuda", dtype=torch.float16)
    s = torch.cuda.Stream()
    if reserve_rows:
        n = Hq * (reserve_rows // 256) * (d + 2) * 4
        assert lib.orin_attn_workspace_reserve_stream(n, 0, s.cuda_stream) == _lib.OK
    g = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(g, stream=s):
        K.flash_attention_decode_fp16_gpu_pos_cu(p, Hq, Hkv, d, Hq // Hkv, 0, cap_rows, Hkv * d, qd,
                                                 out, kd, vd)
    for pos in [cap_rows - 1, 3, 200]:
        p.fill_(pos)
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        ref, _ = oracle.mha_kernel(pos, Hq, 0, cap_rows, Hkv * d, Hq // Hkv, d, q, kc, vc)
        assert_lowp_close(host(out), ref, what=f"pos {pos}")


@pytest.mark.gpu
def test_batched_decode_with_the_larger_splits_workspace():
    """An automatic split accepts the workspace of 256-token splits, and refuses less."""
    lib = _lib.load()
    rng = np.random.default_rng(8600)
    B, Hq, Hkv, d, n = 2, 12, 2, 128, 1000
    q = dev(quantize(normal(rng, (B, Hq, d)), "fp16"), "fp16")
    kc = quantize(normal(rng, (B, n, Hkv, d)), "fp16")
    vc = quantize(normal(rng, (B, n, Hkv, d)), "fp16")
    kd, vd = dev(kc, "fp16"), dev(vc, "fp16")
    lens = torch.tensor([1000, 300], dtype=torch.int32, device="cuda")
    out = torch.zeros(B, Hq, d, device="cuda", dtype=torch.float16)
    small = B * Hq * 4 * (d + 2) * 4
    assert lib.orin_attn_decode_workspace_size(B, Hq, Hkv, d, n, 0) > small
    ws = torch.empty(small, dtype=torch.uint8, device="cuda")

    def call(nbytes):
        return lib.orin_attn_decode(q.data_ptr(), kd.data_ptr(), vd.data_ptr(), out.data_ptr(), B,
                                    Hq, Hkv, d, n * Hkv * d, Hkv * d, lens.data_ptr(), n,
                                    _lib.DTYPE_FP16, 0.0, 0, ws.data_ptr(), nbytes,
                                    torch.cuda.current_stream().cuda_stream)

    assert call(small - 4) == _lib.ERR_WORKSPACE
    assert call(small) == _lib.OK
    torch.cuda.synchronize()
    assert_lowp_close(host(out), oracle.decode_contig(host(q), kc, vc, np.array([1000, 300])),
                      what="256-token splits")
