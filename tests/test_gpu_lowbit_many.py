"""Packed int3 / int2 products of many activation rows (k_lowbit_gemm) against the oracle."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import lowbit as ol
from oracle import qrow as oq

pytestmark = pytest.mark.gpu

# Exact bf16 products, fp32 sums: short chains per group, then at most sqrt(groups) roundings
# of the running sums, 1e-7 of rel-L2 on random signs; 1e-6 leaves a factor of ten (the fp32
# contract is 1e-5).
TOL = 1e-6


def _page(bits, G, asym, n, k, dev, seed):
    from mrun_pub_amd.lowbit import LowbitPage

    rng = np.random.default_rng(seed)
    codes = rng.integers(0, 1 << bits, size=(n, k), dtype=np.uint8)
    packed = ol.pack_codes(codes, bits)
    ng = k // G
    scales = (rng.uniform(0.5, 1.5, size=(n, ng)) / 8).astype(np.float16 if asym else np.float32)
    zeros = rng.normal((1 << bits) / 2, 0.5, size=(n, ng)).astype(np.float16) if asym else None
    page = LowbitPage("w", bits, G, k, torch.from_numpy(packed).to(dev), torch.from_numpy(scales).to(dev),
                      None if zeros is None else torch.from_numpy(zeros).to(dev))
    return page, lambda x: ol.lowbit_matmul(packed, scales, x, k, bits, G, zeros)


# 32 / 64-row tiles and their edges, 64-row weight tiles (5, 63, 65 rows), one 128-k step to
# K splits (2048 x few rows), both layouts of both group sizes; K = 320 at G = 64 has an odd
# group count, which the 16-row kernels keep.
@pytest.mark.parametrize("bits", [2, 3])
@pytest.mark.parametrize("G,asym", [(64, True), (64, False), (128, True), (128, False)])
@pytest.mark.parametrize("m,n,k", [(17, 5, 128), (32, 63, 256), (33, 65, 640), (65, 300, 2048), (131, 64, 1024),
                                   (40, 70, 320)])
def test_many_bf16_rows(dev, bits, G, asym, m, n, k):
    from mrun_pub_amd.lowbit import lowbit_matmul

    if k % G:
        pytest.skip("whole groups only")
    page, ref = _page(bits, G, asym, n, k, dev, seed=m + n + k)
    x = oq.round_bf16(np.random.default_rng(m).standard_normal((m, k)).astype(np.float32))
    y = lowbit_matmul(page, torch.from_numpy(x).to(dev).to(torch.bfloat16))
    assert oq.rel_l2(y.cpu().numpy(), ref(x)) <= TOL


# int2 with G = 64: 17 to 32 rows of widths whose 48-row blocks fill most of the chip once run as
# two launches of 16 (8449 to 12288 rows), one row more or a narrower or wider block do not.
@pytest.mark.parametrize("asym", [False, True])
@pytest.mark.parametrize("m", [17, 32, 33])
@pytest.mark.parametrize("n", [8448, 8449, 12288, 12289])
def test_int2_rows_around_the_two_launch_widths(dev, asym, m, n):
    from mrun_pub_amd.lowbit import lowbit_matmul

    page, ref = _page(2, 64, asym, n, 256, dev, seed=m + n)
    x = oq.round_bf16(np.random.default_rng(m).standard_normal((m, 256)).astype(np.float32))
    y = lowbit_matmul(page, torch.from_numpy(x).to(dev).to(torch.bfloat16))
    assert oq.rel_l2(y.cpu().numpy(), ref(x)) <= TOL


@pytest.mark.parametrize("bits,G,asym", [(2, 128, False), (3, 64, True)])
@pytest.mark.parametrize("m,n,k", [(6, 65, 256), (33, 130, 1024), (515, 40, 256)])
def test_many_fp32_rows(dev, bits, G, asym, m, n, k):
    """Three exact bf16 terms per row; 515 rows run as two launches of at most 512."""
    from mrun_pub_amd.lowbit import lowbit_matmul

    page, ref = _page(bits, G, asym, n, k, dev, seed=m + n + k)
    x = np.random.default_rng(m).standard_normal((m, k)).astype(np.float32)
    y = lowbit_matmul(page, torch.from_numpy(x).to(dev))
    assert oq.rel_l2(y.cpu().numpy(), ref(x)) <= TOL


def test_many_rows_into_a_wider_output_with_the_old_workspace(dev):
    """A leading dimension past N (nothing beyond the N columns is written), with the workspace
    of a single row: the call still runs, in smaller pieces where it has to."""
    import mrun_pub_amd._native as nat
    from mrun_pub_amd.lowbit import lowbit_matmul

    m, n, k, ldy = 37, 65, 2048, 100
    for bits, G, asym, dt in ((3, 64, True, torch.bfloat16), (2, 128, False, torch.float32)):
        page, ref = _page(bits, G, asym, n, k, dev, seed=bits)
        x = oq.round_bf16(np.random.default_rng(1).standard_normal((m, k)).astype(np.float32))
        xd = torch.from_numpy(x).to(dev).to(dt)
        y = torch.full((m, ldy), 7.0, device=dev)
        wsb = int(nat.load().qs_lowbit_workspace_bytes(nat.dtype_code(dt), 1, n, k, G))
        ws = torch.empty(wsb, dtype=torch.uint8, device=dev)
        nat.call("qs_lowbit_gemv", xd.data_ptr(), nat.dtype_code(dt), k, page.packed.data_ptr(), page.row_bytes,
                 page.scales.data_ptr(), nat.dtype_code(page.scales.dtype), nat.ptr(page.zeros),
                 nat.QS_F16 if asym else nat.QS_F32, page._offset(), bits, G, y.data_ptr(), ldy, m, n, k,
                 ws.data_ptr(), wsb, nat.stream_of(dev))
        assert oq.rel_l2(y[:, :n].cpu().numpy(), ref(x)) <= TOL
        assert bool((y[:, n:] == 7.0).all())
        assert oq.rel_l2(lowbit_matmul(page, xd).cpu().numpy(), ref(x)) <= TOL


def test_many_rows_nonfinite_stays_in_its_row(dev):
    from mrun_pub_amd.lowbit import lowbit_matmul

    page, ref = _page(3, 64, True, 70, 256, dev, seed=5)
    x = oq.round_bf16(np.random.default_rng(2).standard_normal((40, 256)).astype(np.float32))
    x[3, 9] = np.inf
    x[39, 255] = np.nan
    y = lowbit_matmul(page, torch.from_numpy(x).to(dev).to(torch.bfloat16)).cpu().numpy()
    rows = np.array([r for r in range(40) if r not in (3, 39)])
    assert np.isfinite(y[rows]).all() and not np.isfinite(y[3]).any() and np.isnan(y[39]).all()
    assert oq.rel_l2(y[rows], ref(x[rows])) <= TOL


def test_many_fp32_rows_of_a_wide_block(dev):
    """A block so wide that its partial sums, not the 512 rows, end a launch (319 rows here)."""
    from mrun_pub_amd.lowbit import lowbit_matmul

    page, ref = _page(2, 64, True, 70001, 128, dev, seed=9)
    x = np.random.default_rng(3).standard_normal((330, 128)).astype(np.float32)
    y = lowbit_matmul(page, torch.from_numpy(x).to(dev)).cpu().numpy()
    want = ref(x)
    for rows in (slice(0, 319), slice(319, 330)):
        assert oq.rel_l2(y[rows], want[rows]) <= TOL


# The 64-row tiles, in one K slice and in several, with ragged rows and columns: input rows
# wider than k (not read past it), output rows wider than n (not written past it).
@pytest.mark.parametrize("bits", [2, 3])
@pytest.mark.parametrize("G,asym", [(64, True), (64, False), (128, True), (128, False)])
@pytest.mark.parametrize("dt,m,n,k,split", [
    (torch.bfloat16, 131, 4093, 128, False), (torch.bfloat16, 33, 11007, 256, False),
    (torch.bfloat16, 33, 4093, 4096, True), (torch.bfloat16, 131, 4093, 11008, True),
    (torch.float32, 65, 4093, 128, False), (torch.float32, 33, 2049, 4096, True)])
def test_many_rows_64_row_tiles(dev, bits, G, asym, dt, m, n, k, split):
    import mrun_pub_amd._native as nat

    tile = (nat.ctypes.c_int32 * 4)()
    xdt = nat.dtype_code(dt)
    assert nat.load().qs_lowbit_many_plan(xdt, m, n, k, G, tile) == 0
    assert tile[0] == 64 and (tile[1] > 1) == split  # another size for this tile if this fails
    g = torch.Generator(device=dev).manual_seed(m + n + k + bits)
    codes = torch.randint(0, 1 << bits, (n, k), dtype=torch.uint8, device=dev, generator=g)
    words = sum(codes.view(n, k // 8, 8)[:, :, i].to(torch.int32) << (bits * i) for i in range(8))
    packed = torch.stack([(words >> (8 * b)) & 255 for b in range(bits)], dim=2).to(torch.uint8).reshape(n, -1)
    ng = k // G
    scales = (torch.rand(n, ng, device=dev, generator=g) + 0.5) / 8
    offset = 4.0 if bits == 3 else 1.0
    zeros = None
    if asym:
        scales, zeros = scales.half(), (offset + 0.5 * torch.randn(n, ng, device=dev, generator=g)).half()
    z = zeros.double() if asym else torch.full((n, ng), offset, dtype=torch.float64, device=dev)
    w = ((codes.double().view(n, ng, G) - z[:, :, None]) * scales.double()[:, :, None]).view(n, k)
    ldx, ldy = k + 64, n + 3
    x = torch.full((m, ldx), float("nan"), dtype=dt, device=dev)
    x[:, :k] = torch.randn(m, k, device=dev, generator=g).to(dt)
    y = torch.full((m, ldy), 7.0, device=dev)
    wsb = int(nat.load().qs_lowbit_workspace_bytes(xdt, m, n, k, G))
    ws = torch.empty(wsb, dtype=torch.uint8, device=dev)
    nat.call("qs_lowbit_gemv", x.data_ptr(), xdt, ldx, packed.data_ptr(), packed.shape[1], scales.data_ptr(),
             nat.dtype_code(scales.dtype), nat.ptr(zeros), nat.QS_F16 if asym else nat.QS_F32, offset, bits, G,
             y.data_ptr(), ldy, m, n, k, ws.data_ptr(), wsb, nat.stream_of(dev))
    want = x[:, :k].double() @ w.t()
    assert float((y[:, :n].double() - want).norm() / want.norm()) <= TOL
    assert bool((y[:, n:] == 7.0).all())
