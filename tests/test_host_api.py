"""Host-side API behaviour that needs no device: the W8A8 store binding, route-index range
checks on host tensors, embedding row-id normalisation."""

from __future__ import annotations

import numpy as np
import pytest
import torch


class _FakeStore:
    """A store with the two methods enable_w8a8 needs; only non-qrow blocks are called
    here, so no device work happens."""

    def __init__(self):
        self.calls = []

    def block_kind(self, name):
        return "fp32" if name.endswith("norm") else "qrow"

    def compact_page(self, name):  # pragma: no cover - qrow path not exercised on CPU
        raise AssertionError("qrow path needs a device")

    def matmul(self, name, x):
        self.calls.append(name)
        return x


def test_w8a8_binding_enable_twice_and_disable():
    from mrun_pub_amd.w8a8 import disable_w8a8, enable_w8a8

    st = _FakeStore()
    enable_w8a8(st, protect_k=8)
    first = vars(st)["matmul"]
    enable_w8a8(st, protect_k=2, protect_lists={"a": [1]})
    assert vars(st)["matmul"] is first  # no second wrapper around the first
    assert first.protect_k == 2 and first.protect_lists == {"a": [1]}
    x = torch.ones(2)
    assert st.matmul("l0.norm", x) is x and st.calls == ["l0.norm"]
    disable_w8a8(st)
    assert "matmul" not in vars(st) and "_w8a8_binding" not in vars(st)
    assert st.matmul("l0.norm", x) is x and st.calls == ["l0.norm", "l0.norm"]
    disable_w8a8(st)  # no-op when not enabled


def test_w8a8_binding_restores_an_instance_matmul():
    from mrun_pub_amd.w8a8 import disable_w8a8, enable_w8a8

    st = _FakeStore()

    def own(name, x):
        return None

    st.matmul = own
    enable_w8a8(st)
    disable_w8a8(st)
    assert vars(st)["matmul"] is own


def test_w8a8_binding_needs_store_methods():
    from mrun_pub_amd.w8a8 import enable_w8a8

    with pytest.raises(TypeError, match="compact_page"):
        enable_w8a8(object())


@pytest.mark.parametrize("bad", [-1, 16])
def test_route_rejects_out_of_range_host_indices(bad):
    from mrun_pub_amd import moe

    idx = torch.tensor([[0, 3], [bad, 2]], dtype=torch.int64)
    w = torch.ones(2, 2)
    with pytest.raises(ValueError, match="top_indices must lie in"):
        moe.grouped_route_tensors(idx, w, num_experts=16)


def test_row_id_normalisation():
    from mrun_pub_amd.qrow import normalize_row_ids

    flat, shape = normalize_row_ids(np.array([[0, -1], [3, -4]]), 4)
    assert shape == (2, 2) and flat.tolist() == [[0, 3], [3, 0]]
    with pytest.raises(IndexError):
        normalize_row_ids([4], 4)
    with pytest.raises(IndexError):
        normalize_row_ids([-5], 4)
    with pytest.raises(TypeError):
        normalize_row_ids([0.5], 4)


def test_prefill_plan_follows_widths_and_split():
    """The many-row kernel is left alone where the decode kernels are faster: long rows of few
    columns without a K split, and few fp32 rows."""
    import mrun_pub_amd._native as nat

    if not nat.LIB_PATH.exists():
        pytest.skip("library not built")

    def plan(dt, m, ns, k, split, swiglu=0):
        return nat.load().qs_qrow_prefill_plan(dt, m, len(ns), nat.int64_array(ns), k, swiglu, split, None)

    f32, bf16 = nat.QS_F32, nat.QS_BF16
    # without a split (measured, decode kernels against this one): 16 / 61 us, 26 / 62, 33 / 42, 57 / 81, 68 / 82,
    # 20 / 22
    for dt, m, n, k in ((f32, 3, 1536, 8960), (f32, 5, 1001, 8960), (bf16, 33, 1536, 8960), (bf16, 33, 4096, 14336),
                        (bf16, 48, 4096, 14336), (bf16, 33, 4096, 4096)):
        assert plan(dt, m, [n], k, 0) == -1, (m, n, k)
    # 81 / 61, 19 / 10, 62 / 29, 77 / 43, 22 / 12
    for dt, m, n, k in ((f32, 16, 1536, 8960), (f32, 16, 4096, 1024), (bf16, 33, 14336, 4096), (bf16, 96, 1536, 8960),
                        (bf16, 33, 8960, 1536)):
        assert plan(dt, m, [n], k, 0) == 0, (m, n, k)
    # with one: 26 / 16, 20 / 15, 33 / 15; eager calls of few short fp32 rows 12 / 18
    assert plan(f32, 5, [1536], 8960, 1) > 0 and plan(f32, 5, [4096], 4096, 1) > 0
    assert plan(bf16, 33, [1001], 8960, 1) > 0
    assert plan(f32, 3, [4096], 1024, 1) == -1 and plan(f32, 8, [4096], 1024, 1) == -1
    # several linears count together
    assert plan(f32, 3, [14336, 14336], 4096, 0) == 0 and plan(f32, 3, [256, 256], 4096, 0) == -1
    assert plan(bf16, 33, [1536], 8960, 0, swiglu=1) == 0


@pytest.mark.parametrize("dtype", ["QS_F32", "QS_BF16"])
@pytest.mark.parametrize("n,k", [(151936, 1536), (11008, 4096), (4096, 11008), (1 << 22, 128), (512, 1 << 20)])
def test_lowbit_workspace_is_bounded(dtype, n, k):
    """Many rows of a wide block share a launch only as far as a bounded workspace allows."""
    import mrun_pub_amd._native as nat

    if not nat.LIB_PATH.exists():
        pytest.skip("library not built")
    size = nat.load().qs_lowbit_workspace_bytes
    one = size(getattr(nat, dtype), 1, n, k, 64)
    for m in (17, 149, 512, 4096, 100000):
        # partial sums and split rows, or what a single row takes
        assert size(getattr(nat, dtype), m, n, k, 64) <= max((256 + 64) << 20, one + 192 * k) + 512, m


def test_rows_bound_of_the_grouped_products():
    """A bound on one group's rows does not pass for a queue of few tokens, and keeps its row tile
    (16 rows while the mean bound per group is at most 8)."""
    from mrun_pub_amd.moe import _rows_bound

    assert _rows_bound(None, 1024, 128) == 1024 and _rows_bound(0, 1024, 128) == 0
    assert _rows_bound(4, 1024, 128) == 1024 and _rows_bound(4, 104, 128) == 104
    assert _rows_bound(16, 6216, 128) == 8 * 128 and _rows_bound(4000, 1024, 128) == 4000
    with pytest.raises(ValueError, match="non-negative"):
        _rows_bound(-1, 8, 8)
