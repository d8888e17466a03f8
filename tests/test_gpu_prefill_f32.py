"""fp32 attention on the matrix-core kernel (fwd_f32.hip): packed rows of a kv head in 16- or
32-row tiles, 16-key tiles split over four waves.  Shapes sit at the edges of those tiles and
of the dispatch (few rows stay on the dot-product kernel), against float64 on the same inputs."""
import numpy as np
import pytest
import torch

from orinmllm_amd import kernel as K
from tests.util import normal


def attend64(q, k, v, lo, hi, kv_mul):
    """q [R, Hq, d], k / v [n, Hkv, d] in float64; row r attends keys lo[r] .. hi[r] - 1."""
    R, Hq, d = q.shape
    out = np.zeros((R, Hq, d))
    for r in range(R):
        for h in range(Hq):
            kk, vv = k[lo[r]:hi[r], h // kv_mul], v[lo[r]:hi[r], h // kv_mul]
            s = kk @ q[r, h] / np.sqrt(d)
            p = np.exp(s - s.max())
            out[r, h] = p @ vv / p.sum()
    return out


def check(got, ref, n):
    """Row-wise 2-norm.  The weighted sum of n terms in fp32 rounds to about sqrt(n) 2^-24 of its
    size; a score of up to 16 (log2 units, 4 standard deviations) rounds by 16 2^-24 and its
    weight by as much relatively.  Four times both."""
    err = np.linalg.norm(got - ref, axis=-1) / np.linalg.norm(ref, axis=-1)
    assert err.max() <= 4 * (np.sqrt(n) + 16) * 2.0 ** -24, err.max()


@pytest.mark.gpu
@pytest.mark.parametrize("Hq,Hkv,d", [(28, 4, 128), (12, 2, 128), (12, 12, 64), (10, 2, 64), (8, 8, 128)])
@pytest.mark.parametrize("start,S", [(0, 1), (0, 3), (0, 33), (15, 2), (16, 32), (401, 7), (0, 129),
                                     (70, 260), (0, 1031)])
def test_prefill_f32_tiles(Hq, Hkv, d, start, S):
    rng = np.random.default_rng(7000 + 31 * S + start + Hq)
    n, pad = start + S, 3
    q = normal(rng, (S, Hq, d))
    k = normal(rng, (2, n + pad, Hkv, d))
    v = normal(rng, (2, n + pad, Hkv, d))
    out = torch.full((S, Hq * d), 7.0, device="cuda")
    K.batched_mha_kernel_cu(start, S, Hq, 1, n + pad, Hq * d, Hkv * d, Hq // Hkv, d, out,
                            torch.from_numpy(q).cuda(), None, torch.from_numpy(k).cuda(),
                            torch.from_numpy(v).cuda())
    rows = np.unique(np.concatenate([[0, S - 1], rng.integers(0, S, 12)]))
    ref = attend64(q[rows].astype(np.float64), k[1].astype(np.float64), v[1].astype(np.float64),
                   np.zeros(len(rows), int), start + rows + 1, Hq // Hkv)
    check(out.view(S, Hq, d).cpu().numpy()[rows].astype(np.float64), ref, n)


@pytest.mark.gpu
def test_prefill_f32_output_over_query():
    rng = np.random.default_rng(7100)
    Hq, Hkv, d, S = 28, 4, 128, 600  # 32-row tiles, more workgroups than CUs
    q = torch.from_numpy(normal(rng, (S, Hq * d))).cuda()
    k, v = (torch.from_numpy(normal(rng, (1, S, Hkv * d))).cuda() for _ in range(2))
    out = torch.empty_like(q)
    K.flash_attention_prefill_cu(0, S, Hq, Hkv, d, Hq // Hkv, 0, S, Hkv * d, q, out, k, v)
    K.flash_attention_prefill_cu(0, S, Hq, Hkv, d, Hq // Hkv, 0, S, Hkv * d, q, q, k, v)
    assert torch.equal(out, q)


@pytest.mark.gpu
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("cu", [(0, 1, 2, 40), (0, 16, 16, 48, 95), (0, 300), (0, 257, 258, 530)])
def test_varlen_f32_segments(d, cu):
    """Tiles that span several segments (an empty one among them) and one-token segments."""
    rng = np.random.default_rng(7200 + cu[-1] + d)
    H, N = 12, cu[-1]
    q, k, v = (normal(rng, (H, N, d)) for _ in range(3))
    out = torch.full((N, H * d), 7.0, device="cuda")
    K.vision_attention_varlen_cu(*(torch.from_numpy(x).cuda() for x in (q, k, v)), out,
                                 torch.tensor(cu, dtype=torch.int32, device="cuda"),
                                 int(np.diff(cu).max()), H, d)
    rows = np.unique(np.concatenate([[c for c in cu if c < N], np.array(cu[1:]) - 1]))
    seg = np.searchsorted(cu, rows, side="right") - 1
    t = [x.transpose(1, 0, 2).astype(np.float64) for x in (q, k, v)]
    ref = attend64(t[0][rows], t[1], t[2], np.array(cu)[seg], np.array(cu)[seg + 1], 1)
    check(out.view(N, H, d).cpu().numpy()[rows].astype(np.float64), ref, N)


@pytest.mark.gpu
@pytest.mark.parametrize("Hq,Hkv,d", [(28, 4, 128), (12, 12, 64)])
@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan])
def test_prefill_f32_nonfinite_value_stays_in_its_rows(Hq, Hkv, d, bad):
    """A non-finite V element of key t reaches the rows that attend to t and no earlier row of
    the same tile."""
    rng = np.random.default_rng(7300)
    S, t = 75, 38
    q, k, v = normal(rng, (S, Hq * d)), normal(rng, (1, S, Hkv, d)), normal(rng, (1, S, Hkv, d))
    run = []
    for x in (None, bad):
        w = v.copy()
        if x is not None:
            w[0, t, :, 5] = x
        out = torch.full((S, Hq * d), 7.0, device="cuda")
        K.batched_mha_kernel_cu(0, S, Hq, 0, S, Hq * d, Hkv * d, Hq // Hkv, d, out,
                                torch.from_numpy(q).cuda(), None, torch.from_numpy(k).cuda(),
                                torch.from_numpy(w).cuda())
        run.append(out.view(S, Hq, d).cpu().numpy())
    clean, got = run
    assert np.array_equal(got[:t], clean[:t])
    others = np.arange(d) != 5
    assert np.array_equal(got[t:, :, others], clean[t:, :, others])
    want = np.full(got[t:, :, 5].shape, bad, np.float32)
    assert np.array_equal(got[t:, :, 5], want, equal_nan=True)
