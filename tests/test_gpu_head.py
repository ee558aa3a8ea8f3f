"""The many-row head top-2 (k_head_top2) at its edges, on heads whose logits are exact."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import qrow as oq

pytestmark = pytest.mark.gpu


# 16-row weight tiles (2, 16 and 17 rows), a full wave round of 8 tiles and its remainder,
# more tiles than the 4096 waves of the largest launch; 8, 10 and 12 chunks of 64 k pick the
# three windows; 16 activation rows fill the tile, 17 and 33 start another launch.
# (Fewer rows of the shorter heads take the one- and two-row kernels, fp32 ones up to 17.)
@pytest.mark.parametrize("v,k", [(2, 512), (16, 640), (17, 768), (129, 1536), (2049, 512), (66000, 512)])
@pytest.mark.parametrize("m", [3, 5, 16, 17, 33])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_head_top2_exact(dev, v, k, m, dtype):
    from mrun_pub_amd import qrow as q

    if v > 60000 and m > 17:
        pytest.skip("one size past the launch is enough")
    rng = np.random.default_rng(v + k + m)
    # products and sums of multiples of 2^-10 below 2^10: exact in fp32, ties included
    codes = rng.integers(-127, 128, size=(v, k), dtype=np.int8)
    scales = np.full(v, 2.0 ** -6, np.float32)
    x = (rng.integers(-8, 9, size=(m, k)) / 16.0).astype(np.float32)
    x[0] = 0.0  # every logit ties at zero: the two lowest rows
    page = q.CompactQRowPage("h", 11, 11 + v, k, torch.from_numpy(codes).to(dev), torch.from_numpy(scales).to(dev))
    cand, vals, _, _ = q.fused_qrow_top2(page, torch.from_numpy(x).to(dev).to(dtype))
    name = {torch.bfloat16: "bf16", torch.float16: "fp16", torch.float32: "fp32"}[dtype]
    ri, rv = oq.qrow_top2(oq.head_logits(codes, scales, x, name), start_row=11)
    assert np.array_equal(cand.cpu().numpy(), ri)
    assert np.array_equal(vals.cpu().numpy(), rv)


def test_head_top2_nonfinite_rows(dev):
    """A NaN row has no candidates, an infinite one keeps its own; the others are untouched."""
    from mrun_pub_amd import qrow as q

    v, k, m = 300, 512, 5
    rng = np.random.default_rng(1)
    codes = rng.integers(-127, 128, size=(v, k), dtype=np.int8)
    codes[:, 3] = np.where(np.arange(v) == 77, 1, -1)
    scales = np.full(v, 2.0 ** -6, np.float32)
    x = (rng.integers(-8, 9, size=(m, k)) / 16.0).astype(np.float32)
    good = x.copy()
    x[1, 0] = np.nan
    x[2, 3] = np.inf
    page = q.CompactQRowPage("h", 0, v, k, torch.from_numpy(codes).to(dev), torch.from_numpy(scales).to(dev))
    cand, vals, _, _ = q.fused_qrow_top2(page, torch.from_numpy(x).to(dev).to(torch.bfloat16))
    cand, vals = cand.cpu().numpy(), vals.cpu().numpy()
    ri, rv = oq.qrow_top2(oq.head_logits(codes, scales, good, "bf16"))
    for r in (0, 3, 4):
        assert np.array_equal(cand[r], ri[r]) and np.array_equal(vals[r], rv[r])
    assert np.array_equal(vals[1], [-np.inf, -np.inf])
    assert cand[2, 0] == 77 and vals[2, 0] == np.inf


@pytest.mark.parametrize("dtype,few,many", [(torch.bfloat16, (1, 2), (3, 5, 16, 17, 33)), (torch.float16, (1, 2), (3, 17)),
                                            (torch.float32, (1, 2, 4), (5, 16, 21))])
def test_head_rows_do_not_depend_on_the_batch_within_a_kernel(dev, dtype, few, many):
    """A row's logits are the same bits in every call of few rows, and in every call of more; the
    rerank of given candidates is the same in all."""
    from mrun_pub_amd import qrow as q

    v, k = 9001, 768  # long enough that the smallest of `many` takes the many-row kernel
    g = torch.Generator(device=dev).manual_seed(4)
    codes = torch.randint(-127, 128, (v, k), dtype=torch.int8, device=dev, generator=g)
    scales = torch.rand(v, device=dev, generator=g) + 0.5
    x = torch.randn(max(many), k, device=dev, generator=g).to(dtype)
    page = q.CompactQRowPage("h", 0, v, k, codes, scales)
    for sizes in (few, many):
        ref = q.fused_qrow_top2(page, x[:sizes[-1]])
        for m in sizes[:-1]:
            got = q.fused_qrow_top2(page, x[:m])
            assert torch.equal(got[0], ref[0][:m]) and torch.equal(got[1], ref[1][:m])
    cand = q.fused_qrow_top2(page, x)[0]
    best, score = q.rerank_qrow_candidates_fp32(page, x, cand)
    for m in few + many:
        b, s = q.rerank_qrow_candidates_fp32(page, x[:m], cand[:m])
        assert torch.equal(b, best[:m]) and torch.equal(s, score[:m])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_head_top2_of_wider_rows(dev, dtype):
    """Activation rows inside wider ones: what lies past k is not read."""
    import mrun_pub_amd._native as nat

    v, k, m, ldx = 300, 640, 21, 640 + 16
    rng = np.random.default_rng(8)
    codes = rng.integers(-127, 128, size=(v, k), dtype=np.int8)
    scales = np.full(v, 2.0 ** -6, np.float32)
    x = (rng.integers(-8, 9, size=(m, k)) / 16.0).astype(np.float32)
    xd = torch.full((m, ldx), float("nan"), dtype=dtype, device=dev)
    xd[:, :k] = torch.from_numpy(x).to(dev).to(dtype)
    c, s = torch.from_numpy(codes).to(dev), torch.from_numpy(scales).to(dev)
    cand = torch.empty((m, 2), dtype=torch.int32, device=dev)
    vals = torch.empty((m, 2), device=dev)
    wsb = int(nat.load().qs_qrow_top2_workspace_bytes(m, v))
    ws = torch.empty(wsb, dtype=torch.uint8, device=dev)
    nat.call("qs_qrow_top2", xd.data_ptr(), nat.dtype_code(dtype), ldx, c.data_ptr(), s.data_ptr(), m, v, k, 0,
             ws.data_ptr(), wsb, cand.data_ptr(), vals.data_ptr(), nat.stream_of(dev))
    ri, rv = oq.qrow_top2(oq.head_logits(codes, scales, x, "bf16" if dtype == torch.bfloat16 else "fp32"))
    assert np.array_equal(cand.cpu().numpy(), ri)
    assert np.array_equal(vals.cpu().numpy(), rv)
