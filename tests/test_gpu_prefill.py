"""GPU parity of the many-row (prefill) W8A16 kernels against the CPU oracle."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import qrow as oq

pytestmark = pytest.mark.gpu

# The oracle rounds the same sums once to 16 bits.  fp32 sums of at most 8960 products in
# another order move a sum by about 1e-6 of its terms' norm, which flips the rounding of
# roughly 1 output in 4000 by one ulp (2^-8 / 2^-11 relative): rel-L2 below 1e-4.
TOL = 1e-3


def _case(n, k, seed):
    rng = np.random.default_rng(seed)
    codes = rng.integers(-127, 128, size=(n, k), dtype=np.int8)
    scales = (rng.uniform(0.5, 1.5, size=n) / 127).astype(np.float32)
    return codes, scales


def _x(m, k, seed, f16):
    x = np.random.default_rng(seed).standard_normal((m, k)).astype(np.float32)
    return oq.round_f16(x) if f16 else oq.round_bf16(x)


def _guarded(m, n, dtype, dev):
    """A contiguous [m, n] output between 256 sentinel elements on both sides."""
    buf = torch.full((m * n + 512,), 7.0, dtype=dtype, device=dev)
    return buf, buf[256:256 + m * n].view(m, n)


def _untouched(buf, m, n):
    return bool((buf[:256] == 7).all()) and bool((buf[256 + m * n:] == 7).all())


# Tile edges (16/32/64/128 activation rows, 128 weight rows), ragged N (N % 4 != 0 also turns
# the vector stores off), one to a few K steps, and K splits.
@pytest.mark.parametrize("m", [33, 64, 65, 129, 300])
@pytest.mark.parametrize("n,k", [(5, 64), (127, 128), (129, 320), (256, 1536), (72, 8960), (1030, 1088)])
@pytest.mark.parametrize("f16", [False, True])
def test_prefill_matmul(dev, m, n, k, f16):
    from mrun_pub_amd import qrow as q

    codes, scales = _case(n, k, seed=m + n + k)
    x = _x(m, k, m + k, f16)
    dt = torch.float16 if f16 else torch.bfloat16
    c, s, xd = torch.from_numpy(codes).to(dev), torch.from_numpy(scales).to(dev), torch.from_numpy(x).to(dev).to(dt)
    assert q._prefill_eligible(xd, [c])
    buf, out = _guarded(m, n, dt, dev)
    y = q.qrow_matmul(c, s, xd, out=out)
    ref = oq.qrow_matmul_w8a16(codes, scales, x, "fp16" if f16 else "bf16")
    assert oq.rel_l2(y.float().cpu().numpy(), ref) <= TOL
    assert _untouched(buf, m, n)
    # without a workspace (no K split): the entry points that take none
    buf, out = _guarded(m, n, dt, dev)
    q.nat.call("qs_qrow_matmul", xd.data_ptr(), q.nat.dtype_code(dt), k, c.data_ptr(), s.data_ptr(), out.data_ptr(), n,
               m, n, k, q.nat.stream_of(dev))
    assert oq.rel_l2(out.float().cpu().numpy(), ref) <= TOL
    assert _untouched(buf, m, n)


@pytest.mark.parametrize("m", [33, 100, 200])
@pytest.mark.parametrize("n,k", [(7, 64), (64, 1024), (200, 384), (68, 4096)])
def test_prefill_swiglu(dev, m, n, k):
    from mrun_pub_amd import qrow as q

    g, u = _case(n, k, seed=m + n), _case(n, k, seed=m + n + 1)
    x = _x(m, k, m + k, False)
    xd = torch.from_numpy(x).to(dev).to(torch.bfloat16)
    pages = [q.CompactQRowPage(nm, 0, n, k, torch.from_numpy(w[0]).to(dev), torch.from_numpy(w[1]).to(dev))
             for nm, w in (("g", g), ("u", u))]
    buf, out = _guarded(m, n, torch.bfloat16, dev)
    y = q.qrow_swiglu_into(pages[0], pages[1], xd, out)
    ref = oq.qrow_swiglu(*g, *u, x)
    # a flipped gate or up rounding is one ulp of the product too: the same bar
    assert oq.rel_l2(y.float().cpu().numpy(), ref) <= TOL
    assert _untouched(buf, m, n)
    buf, out = _guarded(m, n, torch.bfloat16, dev)
    q.nat.call("qs_qrow_swiglu", xd.data_ptr(), k, *(t.data_ptr() for p in pages for t in (p.codes, p.scales)),
               out.data_ptr(), n, m, n, k, q.nat.stream_of(dev))
    assert oq.rel_l2(out.float().cpu().numpy(), ref) <= TOL
    assert _untouched(buf, m, n)


@pytest.mark.parametrize("m", [40, 333])
@pytest.mark.parametrize("ns", [[1536, 256, 256], [130, 3], [64, 128, 16, 4]])
def test_prefill_multi_equals_oracle(dev, m, ns):
    """Linears of different widths in one launch, each with its own tiles."""
    from mrun_pub_amd import qrow as q

    k = 1536
    ws = [_case(n, k, seed=n + i) for i, n in enumerate(ns)]
    x = _x(m, k, m, False)
    xd = torch.from_numpy(x).to(dev).to(torch.bfloat16)
    bufs, outs = zip(*(_guarded(m, n, torch.bfloat16, dev) for n in ns))
    q.qrow_matmul_multi([(torch.from_numpy(c).to(dev), torch.from_numpy(s).to(dev)) for c, s in ws], xd, out=list(outs))
    for (c, s), n, y, buf in zip(ws, ns, outs, bufs):
        assert oq.rel_l2(y.float().cpu().numpy(), oq.qrow_matmul_w8a16(c, s, x)) <= TOL
        assert _untouched(buf, m, n)


def test_prefill_nonfinite_stays_in_its_row(dev):
    """An infinity or NaN in one activation row reaches that row only."""
    from mrun_pub_amd import qrow as q

    n, k, m = 136, 256, 70
    codes, scales = _case(n, k, seed=3)
    x = _x(m, k, 4, False)
    x[5, 17] = np.inf
    x[69, 0] = np.nan
    y = q.qrow_matmul(torch.from_numpy(codes).to(dev), torch.from_numpy(scales).to(dev),
                      torch.from_numpy(x).to(dev).to(torch.bfloat16)).float().cpu().numpy()
    rows = np.array([r for r in range(m) if r not in (5, 69)])
    assert np.isfinite(y[rows]).all() and not np.isfinite(y[5]).any() and np.isnan(y[69]).all()
    assert oq.rel_l2(y[rows], oq.qrow_matmul_w8a16(codes, scales, x[rows])) <= TOL


# fp32: 16 / 32-row tiles, 64-row weight blocks, ragged N, short and split K.  Both sides sum
# exact products of the same fp32 weights in some order; the longest chains here are 16
# products, then about sqrt(K) partial sums, so a result lies within 2 (16 + sqrt(K)) 2^-24 of
# the norm of its terms, 3e-7 of rel-L2 on random signs (1e-5 is the fp32 contract).
@pytest.mark.parametrize("m", [5, 16, 17, 33, 149])
@pytest.mark.parametrize("n,k", [(5, 64), (63, 128), (65, 320), (300, 1536), (72, 8960), (1030, 1088)])
def test_prefill_fp32(dev, m, n, k):
    from mrun_pub_amd import qrow as q

    codes, scales = _case(n, k, seed=m + n + k)
    x = np.random.default_rng(m + k).standard_normal((m, k)).astype(np.float32)
    c, s, xd = (torch.from_numpy(a).to(dev) for a in (codes, scales, x))
    assert q._prefill_eligible(xd, [c])
    ref = x.astype(np.float64) @ oq.dequant_qrow(codes, scales).astype(np.float64).T
    buf, out = _guarded(m, n, torch.float32, dev)
    q.qrow_matmul(c, s, xd, out=out)
    assert oq.rel_l2(out.cpu().numpy(), ref) <= 1e-6
    assert _untouched(buf, m, n)
    buf, out = _guarded(m, n, torch.float32, dev)
    q.nat.call("qs_qrow_matmul", xd.data_ptr(), q.nat.QS_F32, k, c.data_ptr(), s.data_ptr(), out.data_ptr(), n, m, n, k,
               q.nat.stream_of(dev))
    assert oq.rel_l2(out.cpu().numpy(), ref) <= 1e-6
    assert _untouched(buf, m, n)


def test_prefill_fp32_long_rows_and_range(dev):
    """Rows past the decode kernel's 12288 k, values near both ends of fp32, and a non-finite
    activation that reaches its own row only."""
    from mrun_pub_amd import qrow as q

    n, k, m = 40, 14336, 6
    codes, scales = _case(n, k, seed=9)
    x = np.random.default_rng(10).standard_normal((m, k)).astype(np.float32)
    x[1] *= np.float32(1e-38)  # subnormal activations among them
    x[2] *= np.float32(2e33)
    x[3, 7] = np.inf
    c, s, xd = (torch.from_numpy(a).to(dev) for a in (codes, scales, x))
    assert q._prefill_eligible(xd, [c])
    y = q.qrow_matmul(c, s, xd).cpu().numpy()
    ref = x.astype(np.float64) @ oq.dequant_qrow(codes, scales).astype(np.float64).T
    for r in (0, 1, 2, 4, 5):
        assert oq.rel_l2(y[r], ref[r]) <= 1e-6, r
    assert not np.isfinite(y[3]).any()


def test_many_f32_rows_rule(dev):
    """Which fp32 row counts leave the decode kernel: the binding's early answer never differs
    from the library's (whose rule looks at the widths too)."""
    from mrun_pub_amd import qrow as q

    for k in (64, 1024, 4096, 4160, 8192, 8256, 12288, 12352, 16384):
        for m in range(1, 12):
            plans = [q.nat.load().qs_qrow_prefill_plan(q.nat.QS_F32, m, 1, q.nat.int64_array([n]), k, 0, 1, None)
                     for n in (1, 300, 4096, 60000)]
            if not q._many_f32_rows(m, k):
                assert plans == [-1] * 4, (m, k)
            elif k > 12288:
                assert min(plans) >= 0, (m, k)
    assert [m for m in range(1, 9) if not q._many_f32_rows(m, 1024)] == [1, 2, 4]
    assert [m for m in range(1, 9) if not q._many_f32_rows(m, 8192)] == [1, 2]
    assert [m for m in range(1, 9) if not q._many_f32_rows(m, 12288)] == [1, 2]
    assert [m for m in range(1, 9) if not q._many_f32_rows(m, 16384)] == [1]


def _exact(ws, x, dt, swiglu):
    """The result rounded once from 64-bit sums of the weights a product uses (fp32: unrounded)."""
    def mul(w):
        return x.double() @ (w[0].float() * w[1][:, None]).to(dt).double().t()

    if swiglu:
        g, u = (mul(w).to(dt).double() for w in ws)
        return ((g * torch.sigmoid(g)).to(dt).double() * u).to(dt).double()
    return mul(ws[0]) if dt == torch.float32 else mul(ws[0]).to(dt).double()


def _check_entry(dev, dt, m, ns, k, *, swiglu=False, split=True, ldx=None, pad=0, shift=0):
    """``qs_qrow_*_prefill`` on rows of ``ldx`` elements (NaN past k) into rows of n + ``pad``
    that start ``shift`` elements into their buffer."""
    from mrun_pub_amd import qrow as q

    nat = q.nat
    g = torch.Generator(device=dev).manual_seed(m + sum(ns) + k)
    ws = []
    for n in ns * (2 if swiglu else 1):
        c = torch.randint(-127, 128, (n, k), dtype=torch.int8, device=dev, generator=g)
        ws.append((c, (torch.rand(n, device=dev, generator=g) + 0.5) / (73 * k ** 0.5)))
    ldx = ldx or k
    xb = torch.full((m, ldx), float("nan"), dtype=dt, device=dev)
    xb[:, :k] = torch.randn(m, k, device=dev, generator=g).to(dt)
    bufs = [torch.full((shift + m * (n + pad),), 7.0, dtype=dt, device=dev) for n in ns]
    ys = [b[shift:].view(m, n + pad) for b, n in zip(bufs, ns)]
    n_arr, xdt, lib = nat.int64_array(ns), nat.dtype_code(dt), nat.load()
    wsb = int(lib.qs_qrow_prefill_workspace_bytes(xdt, m, len(ns), n_arr, k, int(swiglu))) if split else 0
    work = torch.full((wsb // 4 + 64,), float("nan"), device=dev) if wsb else None
    if swiglu:
        nat.call("qs_qrow_swiglu_prefill", xb.data_ptr(), ldx, *(t.data_ptr() for w in ws for t in w), ys[0].data_ptr(),
                 ns[0] + pad, m, ns[0], k, nat.ptr(work), wsb, nat.stream_of(dev))
    else:
        nat.call("qs_qrow_matmul_prefill", xb.data_ptr(), xdt, ldx, len(ns), nat.pointer_array([c.data_ptr() for c, _ in ws]),
                 nat.pointer_array([s.data_ptr() for _, s in ws]), nat.pointer_array([y.data_ptr() for y in ys]),
                 nat.int64_array([n + pad for n in ns]), n_arr, m, k, nat.ptr(work), wsb, nat.stream_of(dev))
    tol = 1e-6 if dt == torch.float32 else TOL
    for i, (n, y, b) in enumerate(zip(ns, ys, bufs)):
        ref = _exact(ws if swiglu else [ws[i]], xb[:, :k], dt, swiglu)
        err = float((y[:, :n].double() - ref).norm() / ref.norm())
        assert err <= tol, (n, err)
        assert bool((b[:shift] == 7).all()) and bool((y[:, n:] == 7).all())
    if work is not None:
        assert bool(torch.isnan(work[wsb // 4:]).all())
    return wsb


# Ragged widths in K splits: partial rows hold each linear's columns rounded up to 4, alone, in
# a SwiGLU and beside other linears; output rows that allow vector stores (N + pad a multiple of
# 4, aligned) and rows that do not.
@pytest.mark.parametrize("dt,m,ns,k,swiglu", [
    (torch.float32, 3, [1001], 8960, False), (torch.float32, 37, [301, 6, 1], 1536, False),
    (torch.bfloat16, 33, [1001], 8960, False), (torch.float16, 50, [3, 130, 65, 301], 4096, False),
    (torch.bfloat16, 40, [301], 8192, True), (torch.bfloat16, 140, [66], 4096, True)])
@pytest.mark.parametrize("vec", [False, True])
def test_prefill_ragged_widths_split(dev, dt, m, ns, k, swiglu, vec):
    pad = -ns[0] % 4 if vec and len(ns) == 1 else 0
    assert _check_entry(dev, dt, m, ns, k, swiglu=swiglu, pad=pad) > 0
    assert _check_entry(dev, dt, m, ns, k, swiglu=swiglu, pad=pad, split=False) == 0


# Every tile shape, (activation rows, K parts) with one slice and with several, which the sizes
# above reach only in part: ragged rows and columns, wider input rows (not read past k), wider
# output rows (not written past n) that allow vector stores and that start off alignment.
@pytest.mark.parametrize("dt,swiglu,m,n,k,tile,split", [
    (torch.bfloat16, False, 37, 301, 128, (32, 2), False), (torch.bfloat16, False, 37, 1030, 2048, (32, 2), True),
    (torch.bfloat16, False, 1029, 1030, 128, (64, 2), False), (torch.bfloat16, False, 777, 37, 4096, (64, 2), True),
    (torch.bfloat16, False, 300, 1030, 64, (128, 1), False), (torch.bfloat16, False, 65, 4099, 4096, (128, 1), True),
    (torch.bfloat16, False, 200, 8961, 1536, (128, 2), False), (torch.bfloat16, False, 389, 1537, 4096, (128, 2), True),
    (torch.float16, False, 1029, 1030, 128, (64, 2), False), (torch.float16, False, 65, 4099, 4096, (128, 1), True),
    (torch.float16, False, 200, 8961, 1536, (128, 2), False), (torch.float16, False, 389, 1537, 4096, (128, 2), True),
    (torch.bfloat16, True, 37, 301, 128, (32, 2), False), (torch.bfloat16, True, 37, 301, 2048, (32, 2), True),
    (torch.bfloat16, True, 33, 8961, 128, (64, 2), False), (torch.bfloat16, True, 33, 1030, 4096, (64, 2), True),
    (torch.bfloat16, True, 129, 777, 64, (128, 1), False), (torch.bfloat16, True, 65, 2049, 4096, (128, 1), True),
    (torch.bfloat16, True, 65, 8961, 1536, (128, 2), False), (torch.bfloat16, True, 389, 777, 4096, (128, 2), True),
    (torch.float32, False, 37, 301, 128, (16, 2), False), (torch.float32, False, 37, 301, 1536, (16, 2), True),
    (torch.float32, False, 515, 1537, 320, (32, 2), False), (torch.float32, False, 149, 130, 8960, (32, 2), True)])
@pytest.mark.parametrize("layout", ["packed", "wide", "misaligned"])
def test_prefill_every_tile_and_layout(dev, dt, swiglu, m, n, k, tile, split, layout):
    from mrun_pub_amd import qrow as q

    plan = (q.nat.ctypes.c_int32 * 4)()
    q.nat.load().qs_qrow_prefill_plan(q.nat.dtype_code(dt), m, 1, q.nat.int64_array([n]), k, int(swiglu), int(split), plan)
    assert (plan[0], plan[2]) == tile and (plan[3] > 1) == split  # another size for this tile if this fails
    kw = {"packed": {}, "wide": dict(ldx=k + 64, pad=8 - n % 4), "misaligned": dict(ldx=k + 8, pad=-n % 4, shift=1)}[layout]
    assert (_check_entry(dev, dt, m, [n], k, swiglu=swiglu, split=split, **kw) > 0) == split


def test_prefill_rows_past_one_launch(dev):
    """More rows than one grid's 2^32 threads hold: 32-row tiles of one column reach that at 2^28
    rows (a 69 GB input).  All rows are zero but a few on both sides of every edge."""
    from mrun_pub_amd import qrow as q

    m, k = 2**28 + 40, 64
    if torch.cuda.mem_get_info()[0] < 80 << 30:
        pytest.skip("needs 80 GB of free device memory")
    codes, scales = _case(1, k, seed=1)
    c, s = torch.from_numpy(codes).to(dev), torch.from_numpy(scales).to(dev)
    tile = (q.nat.ctypes.c_int32 * 4)()
    assert q.nat.load().qs_qrow_prefill_plan(q.nat.QS_F32, m, 1, q.nat.int64_array([1]), k, 0, 1, tile) == 0
    assert m // tile[0] * 512 >= 2**32  # (8 waves per workgroup)
    rows = torch.tensor([0, 31, 32, 2**28 - 65, 2**28 - 33, 2**28 - 32, 2**28 - 1, 2**28, m - 1], device=dev)
    some = torch.randn(len(rows), k, device=dev, generator=torch.Generator(device=dev).manual_seed(2))
    x = torch.zeros(m, k, device=dev)
    x[rows] = some
    y = q.qrow_matmul(c, s, x)
    del x
    ref = some.double() @ (c.double() * s.double()[:, None]).t()
    assert float((y[rows].double() - ref).norm() / ref.norm()) <= 1e-6
    assert int(torch.count_nonzero(y)) == len(rows)
    torch.cuda.empty_cache()
