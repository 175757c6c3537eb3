"""GPU parity: the radix-select kernel (through the C ABI) vs the oracle, bit-exact."""

import json

import numpy as np
import pytest
import torch

from cppmega_mlx_amd.nn._tilelang import topk_selector as tk
from oracle import topk as otopk
from tests._inputs import to_dev, topk_scores

pytestmark = pytest.mark.gpu


def _run(scores_t, k, device, *, starts=None, ends=None, order="index", fill=-7, **kw):
    out = torch.full((scores_t.shape[0], k), fill, dtype=torch.int32, device=device)
    st = None if starts is None else to_dev(np.asarray(starts, np.int32), device)
    en = None if ends is None else to_dev(np.asarray(ends, np.int32), device)
    got = tk.topk_selector_tilelang_direct(scores_t, k, out=out, starts=st, ends=en, order=order, **kw)
    assert got is out
    torch.cuda.synchronize()
    return out.cpu().numpy()


def test_reference_known_answers(device, golden_dir):
    kats = json.loads((golden_dir / "reference_kats.json").read_text())
    c = kats["topk_exact_order_ties"]
    assert _run(to_dev(np.array(c["scores"], np.float32), device), c["k"], device, order="value").tolist() == c["expected_value_order"]
    c = kats["topk_masked_ties"]
    assert _run(to_dev(np.array(c["scores"], np.float32), device), c["k"], device, starts=c["starts"], ends=c["ends"],
                order="value").tolist() == c["expected_value_order"]
    c = kats["topk_short_and_empty_intervals"]
    got = _run(to_dev(np.array(c["scores"], np.float32), device), c["k"], device, starts=c["starts"], ends=c["ends"])
    assert [sorted(set(r)) for r in got.tolist()] == [sorted(s) for s in c["expected_sets"]]
    c = kats["topk_k_one_argmax"]
    assert _run(to_dev(np.array(c["scores"], np.float32), device), 1, device).tolist() == c["expected"]


@pytest.mark.parametrize("rows,width,k", [(4, 64, 8), (3, 512, 64), (5, 2048, 256), (6, 8192, 2048), (2, 8192, 1),
                                          (2, 8192, 8192), (3, 100, 7), (2, 1001, 500), (2, 4096, 2048), (1, 4, 4), (2, 20000, 3000), (1, 65536, 2048), (2, 9001, 100),
                                          (3, 16384, 2048), (2, 12288, 4096), (2, 32768, 2048), (2, 20004, 5000), (1, 30001, 7), (2, 16384, 16384), (2, 16380, 1), (2, 8196, 8000)])
@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("order", ["index", "value"])
def test_random_rows_bit_exact(device, rows, width, k, masked, order):
    rng = np.random.default_rng(rows * 7919 + width * 31 + k + (5 if masked else 0))
    s = topk_scores(rng, rows, width)
    starts = ends = None
    if masked:
        starts = rng.integers(0, max(1, width // 2), rows).astype(np.int32)
        ends = (starts + rng.integers(0, width, rows)).astype(np.int32)
        ends[0] = starts[0]                      # an empty interval
        starts[-1] = -5                          # clipped to 0
    got = _run(to_dev(s, device), k, device, starts=starts, ends=ends, order=order)
    want = otopk.topk_selector_oracle(s, k, starts=starts, ends=ends, order=order)
    np.testing.assert_array_equal(got, want)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_half_precision_scores(device, dtype):
    rng = np.random.default_rng(17)
    t = to_dev(topk_scores(rng, 5, 2048), device).to(dtype)
    s = t.to(torch.float32).cpu().numpy()       # many exact ties after rounding
    for order in ("index", "value"):
        np.testing.assert_array_equal(_run(t, 300, device, order=order), otopk.topk_selector_oracle(s, 300, order=order))


def test_special_values_zero_signs_denormals_infinities_nan(device):
    s = np.array([[0.0, -0.0, 0.0, -0.0, 1e-40, -1e-40, np.inf, -np.inf, np.nan, 3.0, 3.0, -np.inf]], np.float32)
    t = to_dev(s, device)
    for k in (1, 3, 5, 7, 9, 11, 12):
        for order in ("index", "value"):
            np.testing.assert_array_equal(_run(t, k, device, order=order), otopk.topk_selector_oracle(s, k, order=order))
    np.testing.assert_array_equal(_run(t, 12, device, order="value", neg_inf_is_masked=True),
                                  otopk.topk_selector_oracle(s, 12, order="value", neg_inf_is_masked=True))


def test_constant_and_two_valued_rows(device):
    s = np.zeros((3, 8192), np.float32)
    s[1] = 5.0
    s[2, ::3] = 1.0
    np.testing.assert_array_equal(_run(to_dev(s, device), 2048, device), otopk.topk_selector_oracle(s, 2048))
    np.testing.assert_array_equal(_run(to_dev(s, device), 3000, device, order="value"),
                                  otopk.topk_selector_oracle(s, 3000, order="value"))


def test_misaligned_view_takes_the_scalar_load_path(device):
    rng = np.random.default_rng(23)
    s = topk_scores(rng, 4, 1030)
    base = to_dev(np.concatenate([np.zeros(1, np.float32), s.reshape(-1)]), device)
    t = base[1:].view(4, 1030)                   # 4-byte aligned only
    assert t.data_ptr() % 16 != 0
    np.testing.assert_array_equal(_run(t, 77, device), otopk.topk_selector_oracle(s, 77))


def test_headline_config_full_size_bit_exact(device):
    """[4, 1024, 8192] fp32 scores, 5% ties, causal bounds, k = 2048 (both the all-visible and the padded window)."""
    rng = np.random.default_rng(2048)
    B, S, T, k = 4, 1024, 8192, 2048
    s = topk_scores(rng, B * S, T)
    for off in (T - S, 0):
        ends = np.tile(off + np.arange(S, dtype=np.int32) + 1, B)
        masked = s.copy()
        masked[np.arange(T)[None, :] >= ends[:, None]] = -np.inf
        out = tk.topk_selector(to_dev(masked.reshape(B, S, T), device), k, ends=to_dev(ends, device))
        torch.cuda.synchronize()
        assert tuple(out.shape) == (B, S, k)
        got = out.reshape(B * S, k).cpu().numpy()
        want = otopk.topk_selector_oracle(masked, k, ends=ends)
        np.testing.assert_array_equal(got, want)
        valid = np.minimum(ends, k)
        assert ((got >= 0).sum(axis=1) == valid).all()


def test_public_entry_points(device):
    rng = np.random.default_rng(3)
    s = topk_scores(rng, 3, 256)
    t = to_dev(s, device)
    ref = tk.topk_selector_reference(t, 16)
    np.testing.assert_array_equal(ref.cpu().numpy(), otopk.topk_selector_oracle(s, 16, order="value"))
    for backend in ("auto", "hip", "path_c", "mlx"):
        np.testing.assert_array_equal(tk.topk_selector(t, 16, backend=backend).cpu().numpy(), otopk.topk_selector_oracle(s, 16))
    assert tk.topk_selector_path_c_status().available


@pytest.mark.parametrize("rows,width,k", [(32, 65536, 2048), (3, 40000, 4000), (2, 24576, 8192), (5, 16388, 100), (2, 30001, 2000)])
def test_wide_rows_two_stage_and_single_workgroup_paths_agree_with_the_oracle(device, rows, width, k):
    """Rows wider than 16384 columns: k best of every 8192-column segment, then k of those.  Ties that
    straddle segments, bounds that empty whole segments, -inf and NaN entries."""
    import ctypes as C
    from cppmega_mlx_amd import _lib, ops
    rng = np.random.default_rng(rows + width + k)
    s = topk_scores(rng, rows, width, tie_fraction=0.2)
    s[0, ::5] = 1.5                                      # one value far beyond k times, in every segment
    s[1, 100:9000] = np.nan
    s[1, 9000:9500] = -np.inf
    starts = rng.integers(0, width // 3, rows).astype(np.int32)
    ends = rng.integers(width // 2, width + 1, rows).astype(np.int32)
    starts[-1], ends[-1] = 9000, 9000 + k // 2           # fewer selectable columns than k, inside one segment
    t = to_dev(s, device)
    for order in ("index", "value"):
        for bounds in (False, True):
            st = to_dev(starts, device) if bounds else None
            en = to_dev(ends, device) if bounds else None
            want = otopk.topk_selector_oracle(s, k, starts=starts if bounds else None, ends=ends if bounds else None,
                                              order=order, neg_inf_is_masked=True)
            for two_stage in (True, False):
                out = torch.full((rows, k), -7, dtype=torch.int32, device=device)
                ops.topk_select(t, k, out=out, starts=st, ends=en, order=order, neg_inf_is_masked=True, two_stage=two_stage)
                torch.cuda.synchronize()
                np.testing.assert_array_equal(out.cpu().numpy(), want)
    a = _lib.TopkArgs()
    a.struct_size = C.sizeof(a)
    a.rows, a.width, a.row_stride, a.k = rows, width, width, k
    need = C.c_size_t(0)
    assert _lib.load().cppmega_mi355_topk_workspace_bytes(C.byref(a), C.sizeof(a), C.byref(need)) == _lib.OK
    assert need.value > 0                                # two stages, whole 16-byte rows or not
    a.width = a.row_stride = 16384
    assert _lib.load().cppmega_mi355_topk_workspace_bytes(C.byref(a), C.sizeof(a), C.byref(need)) == _lib.OK and need.value == 0


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows,width,k,offset", [(3, 1023, 5, 1), (1, 8191, 2048, 3), (2, 4097, 300, 0), (3, 16383, 1000, 1), (2, 30001, 2047, 1), (1, 17, 16, 2)])
def test_rows_that_start_and_end_anywhere(device, rows, width, k, offset, dtype):
    """Widths that are no multiple of four, at addresses that are none of 16 bytes; the last row ends its buffer."""
    rng = np.random.default_rng(width)
    flat = torch.from_numpy(rng.standard_normal(offset + rows * width).astype(np.float32)).to(device).to(dtype)
    view = flat[offset:].view(rows, width)
    assert (_run(view, k, device) == otopk.topk_selector_oracle(view.float().cpu().numpy(), k, order="index")).all()


@pytest.mark.parametrize("width,k", [(300, 255), (700, 257), (1500, 1025), (4096, 4096), (8192, 513), (16000, 16000), (40000, 3000)])
def test_value_order_around_the_chunks_of_the_sort(device, width, k):
    rng = np.random.default_rng(k)
    scores = np.round(rng.standard_normal((3, width)) * 50).astype(np.float32)       # many equal values: ties by index
    assert (_run(to_dev(scores, device), k, device, order="value") == otopk.topk_selector_oracle(scores, k, order="value")).all()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows,width,pitch,k", [(3, 1023, 1024, 5), (2, 1022, 1031, 1022), (3, 8189, 8192, 300), (2, 16381, 16400, 900), (2, 20003, 20010, 77),
                                                (3, 1, 5, 1), (4, 1, 1, 1), (5, 2, 2, 1), (2, 3, 4, 2)])
def test_rows_with_a_pitch_whose_buffer_ends_with_the_last_row(device, rows, width, pitch, k, dtype):
    """The right-hand columns of a wider matrix through the C interface: nothing lies behind the last row's last column."""
    import ctypes as C
    from cppmega_mlx_amd import _lib
    rng = np.random.default_rng(width)
    whole = torch.from_numpy(rng.standard_normal((rows, pitch)).astype(np.float32)).to(device).to(dtype)
    view = whole[:, pitch - width:]
    out = torch.full((rows, k), -7, dtype=torch.int32, device=device)
    a = _lib.TopkArgs()
    a.struct_size, a.score_dtype = C.sizeof(a), _lib.F32 if dtype is torch.float32 else _lib.BF16
    a.scores, a.indices = view.data_ptr(), out.data_ptr()
    a.rows, a.width, a.row_stride, a.k, a.order = rows, width, pitch, k, _lib.TOPK_ORDER_INDEX
    need = C.c_size_t(0)
    lib = _lib.load()
    assert lib.cppmega_mi355_topk_workspace_bytes(C.byref(a), C.sizeof(a), C.byref(need)) == _lib.OK
    ws = torch.empty(max(need.value, 1), dtype=torch.uint8, device=device)
    a.workspace, a.workspace_bytes = ws.data_ptr(), need.value
    assert lib.cppmega_mi355_topk_select(C.byref(a), C.sizeof(a), _lib.current_stream(view.device)) == _lib.OK
    assert (out.cpu().numpy() == otopk.topk_selector_oracle(view.float().cpu().numpy(), k, order="index")).all()


# one and two keys to a lane of the sort, on 256, 512 and 1024 threads, a key short of a run and not
@pytest.mark.parametrize("width,k", [(256, 256), (900, 129), (2048, 512), (4096, 400), (8000, 200), (8192, 512), (16000, 256), (20000, 511)])
def test_value_order_of_short_lists(device, width, k):
    rng = np.random.default_rng(width + k)
    scores = np.round(rng.standard_normal((3, width)) * 50).astype(np.float32)       # many equal values: ties by index
    ends = np.array([width, k // 2, width - 1], np.int32)
    assert (_run(to_dev(scores, device), k, device, ends=ends, order="value") == otopk.topk_selector_oracle(scores, k, ends=ends, order="value")).all()


# scores of 8 MiB, requested before their bounds, and of a row more, of which only columns inside the bounds are read
@pytest.mark.parametrize("rows,width,k", [(256, 8192, 300), (257, 8192, 300), (2048, 1024, 64), (2049, 1024, 64), (530, 4003, 90), (131, 16384, 700), (60, 40000, 200)])
def test_bounds_of_many_rows(device, rows, width, k):
    rng = np.random.default_rng(rows + width)
    scores = np.round(rng.standard_normal((rows, width)) * 1000).astype(np.float32)
    starts = rng.integers(-5, width // 2, rows).astype(np.int32)
    ends = (starts + rng.integers(0, width, rows)).astype(np.int32)
    ends[0] = starts[0]                                  # an empty interval
    got = _run(to_dev(scores, device), k, device, starts=starts, ends=ends)
    assert (got == otopk.topk_selector_oracle(scores, k, starts=starts, ends=ends, order="index")).all()
