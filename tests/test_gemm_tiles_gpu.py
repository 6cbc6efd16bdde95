"""Prompt GEMM tiles: shapes whose estimated best tile is each of the kernel's
(64 x 128, 128 x 128 with two and with four stages in flight, 256 x 160, 192
and 256), unsplit and with K split over the workspace, one past and one short
of whole tiles, stages and store widths."""
import pytest

from tests.helpers import assert_f16_path, assert_f32_rel, dev_f16, normal, values

SHAPES = [
    (33, 1000, 4097), (65, 4104, 4100), (129, 2568, 7679), (199, 4104, 12289), (257, 64, 260),
    (511, 4096, 4097), (701, 2056, 8191), (1023, 4104, 12292), (1025, 1096, 4095),
    (1500, 4096, 12290), (1501, 2056, 9001), (2047, 4104, 4095), (2049, 1160, 11009),
    # 256 x 192
    (529, 360, 13875),
    # with the workspace: 64 x 128, 128 x 128 (two stages), 256 x 160, 192 and 256
    (17, 904, 35), (67, 9624, 11271), (131, 5624, 5703), (133, 9688, 5435), (137, 9464, 13865)]


def test_shapes_reach_every_tile_unsplit_and_split(tmc):
    """The host's own choice for the shapes below: a change of its figures that
    left a tile or its split form unrun fails here."""
    plans = {tmc.gemm_rows_plan(*shape, ws)
             for shape in SHAPES for ws in (0, tmc.gemm_rows_workspace_bytes())}
    tiles = {(64, 128, 4), (128, 128, 2), (128, 128, 4), (256, 160, 2), (256, 192, 2),
             (256, 256, 2)}
    assert {p[:3] for p in plans if p[3] == 1} == tiles
    assert {p[:3] for p in plans if p[3] > 1} == tiles


@pytest.mark.gpu
@pytest.mark.parametrize("m,k,n", SHAPES)
def test_gemm_rows_tiles_match_fp64(tmc, orc, m, k, n):
    import torch
    x = dev_f16(orc.f16(normal(3001 + m, (m, k))))
    w = torch.empty((n, k), dtype=torch.float16, device="cuda")
    tmc.fill_normal(w, 3002 + n, 0.0, 0.02)
    ref = (x.double() @ w.double().t()).cpu().numpy()
    workspace = torch.empty(tmc.gemm_rows_workspace_bytes() // 4, dtype=torch.int32, device="cuda")
    for ws in (None, workspace):
        y = torch.full((m, n), float("nan"), dtype=torch.float32, device="cuda")
        tmc.gemm_rows(x, w, y, ws)
        assert_f32_rel(values(y), ref, what=f"{m}x{k}x{n}")
        # an output that starts off a store's alignment takes the scalar stores
        flat = torch.full((m * n + 1,), float("nan"), dtype=torch.float16, device="cuda")
        tmc.gemm_rows(x, w, flat[1:].view(m, n), ws)
        assert_f16_path(values(flat[1:]), ref, what=f"{m}x{k}x{n} f16")
        assert bool(torch.isnan(flat[0]))


@pytest.mark.gpu
def test_gemm_rows_keeps_non_finite_inputs_in_their_rows(tmc):
    """An infinity in one row of x reaches that row only: the zeros that stand
    in for rows and k past the operands never meet it."""
    import torch
    x = torch.ones((130, 136), dtype=torch.float16, device="cuda")
    x[129, 135] = float("inf")
    w = torch.ones((260, 136), dtype=torch.float16, device="cuda")
    y = torch.full((130, 260), float("nan"), dtype=torch.float32, device="cuda")
    tmc.gemm_rows(x, w, y, None)
    assert bool((y[:129] == 136).all()) and bool(torch.isinf(y[129]).all())
