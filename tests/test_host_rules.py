"""Host-side layout rules of the ops layer (no device work): line-pitched
buffers, the paired-product layout and the rule that decides when the
convolution adds its self term inside the SpMM."""
import pytest
import torch

from graph_rws_amd.core import ops
from graph_rws_amd.layers import layer


def test_line_pitched_empty_rows_start_on_lines():
    for cols, dt in ((41, torch.float16), (47, torch.bfloat16), (7, torch.float32), (64, torch.float16),
                     (172, torch.float16)):
        t = ops.line_pitched_empty(10, cols, dt, "cpu", zero=True)
        esz = t.element_size()
        assert t.shape == (10, cols) and t.stride(1) == 1
        assert (t.stride(0) * esz) % 128 == 0 and t.stride(0) >= cols
        assert t.stride(0) - cols < 128 // esz                 # the smallest such pitch
        assert not bool(t.any())


def test_pair_pitch_puts_each_product_on_whole_lines():
    assert ops.pair_pitch(256, 2) == 512
    assert ops.pair_pitch(47, 2) == 128
    assert ops.pair_pitch(41, 2) == 128
    assert ops.pair_pitch(16, 4) == 64
    assert ops.pair_pitch(172, 2) == 384


def test_mm_pair_line_pitched_matches_two_products():
    torch.manual_seed(0)
    a = torch.randn(50, 24)
    w1, w2 = torch.randn(24, 47), torch.randn(24, 47)
    t1, t2 = ops.mm_pair_line_pitched(a, w1, w2)
    assert t1.shape == (50, 47) and t2.shape == (50, 47)
    assert t1.stride(0) == ops.pair_pitch(47, 4)
    torch.testing.assert_close(t1, a @ w1)
    torch.testing.assert_close(t2, a @ w2)


def test_fuse_self_rule():
    # narrow paired rows always pay; wide ones only within the Infinity Cache
    assert ops.fuse_self_pays(2_449_029, 47, 2)
    assert ops.fuse_self_pays(232_965, 256, 2)
    assert not ops.fuse_self_pays(2_449_029, 256, 2)
    assert ops.fuse_self_pays(2708, 16, 4)


@pytest.mark.parametrize("m,n,tiles", [(7, 7, 1), (32, 33, 1), (64, 128, 1), (129, 65, 2), (128, 129, 2), (1024, 256, 16),
                                       (1433, 16, 12), (8415, 41, 66)])
def test_f32_weight_gradient_tiles(m, n, tiles):
    assert ops.gemm_tn_f32_tiles(m, n) == ops.gemm_tn_f32_tiles(n, m) == tiles


# 20 tiles of whole vectors, 21; 10 ragged tiles, 11; wide on either side
@pytest.mark.parametrize("m,n,kernel", [(128, 256, True), (7, 41, True), (2560, 32, True), (2564, 32, False),
                                        (1280, 256, True), (1536, 256, False), (1279, 7, True), (1281, 7, False),
                                        (602, 256, True), (602, 602, False), (16, 8415, False), (2048, 2048, False)])
def test_f32_weight_gradient_leaves_wide_products_to_the_library(monkeypatch, m, n, kernel):
    """The f32 split-K kernel takes products of few output tiles only: with
    more the library is faster and needs no partial sums."""
    monkeypatch.setattr(layer, "F32_TN_ROWS", 8)
    monkeypatch.setattr(ops, "gemm_tn_f32_supported", lambda a, b: True)
    monkeypatch.setattr(ops, "gemm_tn_f32", lambda a, b: "kernel")
    x, g = torch.ones(8, m), torch.ones(8, n)
    with torch.no_grad():
        got = layer._weight_grad(x, g)
    assert (isinstance(got, str) and got == "kernel") == kernel
    if not kernel:
        assert got.shape == (m, n) and bool((got == 8).all())


def test_f32_weight_gradient_counts_misaligned_rows_as_ragged(monkeypatch):
    monkeypatch.setattr(layer, "F32_TN_ROWS", 8)
    monkeypatch.setattr(ops, "gemm_tn_f32_supported", lambda a, b: True)
    monkeypatch.setattr(ops, "gemm_tn_f32", lambda a, b: "kernel")
    wide = torch.ones(8, 2560 + 8)
    g = torch.ones(8, 16)
    with torch.no_grad():
        assert isinstance(layer._weight_grad(wide[:, :2560], g), str)       # 20 tiles, whole vectors
        assert torch.is_tensor(layer._weight_grad(wide[:, 1:2561], g))      # a start 4 bytes off
        assert torch.is_tensor(layer._weight_grad(torch.ones(8, 2562)[:, :2560], g))  # a pitch of 2,562


def _windows(slabs, max_slabs, sampled):
    """A BCSR (host arrays) of short windows and one of `slabs` 16-column slabs."""
    from graph_rws_amd.data import BCSRGraph
    tiles = torch.tensor([1, slabs, 2, 1])
    win = torch.cat([torch.zeros(1, dtype=torch.int64), tiles.cumsum(0)])
    T = int(win[-1])
    g = BCSRGraph(num_nodes=64, num_edges=0, tile_rows=16, tile_cols=16, window_offset=win,
                  original_col_indices=torch.zeros(16 * T, dtype=torch.int32),
                  values_condensed=torch.zeros(256 * T), device="cpu", num_rows=64, num_cols=5000)
    g.max_window_slabs = max_slabs
    if sampled:
        g.sampled = True
    return g


# (longest window, products before the first with a plan): none needed up to a
# plan's own item (16 slabs); 200 slabs walked in excess; past 128 at once
@pytest.mark.parametrize("slabs,before", [(16, None), (17, 201), (40, 9), (128, 2), (129, 0), (400, 0)])
def test_sampled_block_takes_a_plan_when_it_is_kept(monkeypatch, slabs, before):
    from graph_rws_amd.data import bcsr
    built = []
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    monkeypatch.setattr(bcsr, "build_spmm_plan", lambda *a, **k: built.append(1) or "plan")
    g = _windows(slabs, slabs, True)
    assert ops.default_slabs(g.num_windows, g.num_tiles, 16, 128) == 16
    if before is None:
        assert all(g.spmm_plan(128) is None for _ in range(300)) and not built
        return
    for i in range(before):
        assert g.spmm_plan(128) is None, i
    assert g.spmm_plan(128) == "plan" and g.spmm_plan(128) == "plan" and built == [1]
    # other windows in the same buffer: the count starts again
    g.window_offset.add_(0)
    if before:
        assert g.spmm_plan(128) is None
    # not sampled, or of unknown windows: at the first product
    assert _windows(slabs, slabs, False).spmm_plan(128) == "plan"
    assert _windows(slabs, None, True).spmm_plan(128) == "plan"


def test_sampled_block_builds_no_plan_under_capture(monkeypatch):
    from graph_rws_amd.data import bcsr
    monkeypatch.setattr(bcsr, "build_spmm_plan", lambda *a, **k: "plan")
    capturing = [True]
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: capturing[0])
    g = _windows(128, 128, True)
    assert all(g.spmm_plan(64) is None for _ in range(5))
    capturing[0] = False
    assert g.spmm_plan(64) == "plan"
    capturing[0] = True
    assert g.spmm_plan(64) == "plan"  # built before the capture: used in it
