"""Packed GEMMs above 16 batch rows: one launch reads every weight for up to
64 rows (16-row tiles), and wide outputs share activation fragments between
three 16-column tiles.  Batches at the edges of the row tiles, widths at the
edges of the column tiles, K with a ragged tail."""
import numpy as np
import pytest

from tests.helpers import assert_f16_path, assert_f32_rel, bits, dev_f16, normal, uniform, values

pytestmark = pytest.mark.gpu



@pytest.fixture(scope="module")
def torch():
    import torch as t
    return t


BATCHES = [17, 32, 33, 48, 49, 64, 65]


def _rows(tmc, torch, x, packed, b, k, n, layout, cfg, residual=None):
    xin = tmc.pack_activations(x) if layout else x
    if residual is None:
        y = torch.full((b, n), float("nan"), dtype=torch.float32, device="cuda")
        tmc.gemm_packed_ex(xin, packed, y, b, k, n, layout, cfg)
    else:
        y = torch.full((b, n), float("nan"), dtype=torch.float16, device="cuda")
        tmc.gemm_packed_residual(xin, packed, residual, y, b, k, n, layout, cfg)
    return y


@pytest.mark.parametrize("batch", BATCHES)
@pytest.mark.parametrize("layout", [0, 1])
@pytest.mark.parametrize("k,n,ks", [(1160, 200, 4), (2048, 520, 16)])
def test_row_tiles_equal_single_passes(tmc, orc, torch, batch, layout, k, n, ks):
    """The same k split gives each row the bits of a launch of its own 16
    rows: fp32 output and fp16 output with the residual."""
    cfg = tmc.GemvConfig(3, 1, 1, ks)
    x = dev_f16(orc.f16(normal(2001 + batch, (batch, k))))
    packed = tmc.pack_weights(dev_f16(orc.f16(normal(2002, (n, k), 0.02))))
    res = dev_f16(orc.f16(normal(2003, (batch, n))))
    for r in (None, res):
        got = _rows(tmc, torch, x, packed, batch, k, n, layout, cfg, r)
        want = torch.cat([
            _rows(tmc, torch, x[a:a + 16].contiguous(), packed, min(16, batch - a), k, n, layout,
                  cfg, None if r is None else r[a:a + 16].contiguous())
            for a in range(0, batch, 16)])
        torch.cuda.synchronize()
        assert torch.equal(got, want)


@pytest.mark.parametrize("batch,n,k", [(17, 12288, 1184), (33, 8208, 1184), (49, 8217, 1184),
                                       (64, 12300, 1184), (48, 12288, 1024), (48, 12288, 1016)])
def test_three_column_tiles_match_fp64(tmc, orc, torch, batch, n, k):
    """Wide outputs (three 16-column tiles per block from K 1024 on, the last
    block short): the fp32 projection within the fp32 rule of 64-bit sums of
    the same fp16 products, and the token-only LM head's tokens from the same
    logits."""
    x = dev_f16(orc.f16(normal(2011 + batch, (batch, k))))
    gamma = dev_f16(orc.f16(uniform(2012, (k,), 0.5, 1.5)))
    w = dev_f16(orc.f16(normal(2013, (n, k), 0.02)))
    packed = tmc.pack_weights(w)
    y = _rows(tmc, torch, x, packed, batch, k, n, 1, None)
    ref = x.double() @ w.double().t()
    assert_f32_rel(values(y), ref.cpu().numpy(), what=f"b{batch} n{n}")
    scaled = tmc.pack_weights(w, gamma=gamma)
    logits = torch.full((batch, n), float("nan"), dtype=torch.float32, device="cuda")
    xin = tmc.pack_activations(x)
    tmc.gemm_packed_norm(xin, scaled, logits, batch, k, n, 1e-6, 1)
    xd = x.double()
    norm = xd / torch.sqrt((xd * xd).mean(-1, keepdim=True) + 1e-6)
    ref = norm @ (w.float() * gamma.float()).half().double().t()
    assert_f32_rel(values(logits), ref.cpu().numpy(), what=f"norm b{batch} n{n}")
    ws = torch.zeros(tmc.lm_head_argmax_workspace_bytes(batch, n) // 4, dtype=torch.float32,
                     device="cuda")
    tok = torch.full((batch,), -7, dtype=torch.int32, device="cuda")
    tmc.lm_head_argmax_packed_norm(xin, scaled, ws, tok, batch, k, n, 1e-6, 1)
    assert torch.equal(tok.long(), logits.argmax(-1))


@pytest.mark.parametrize("batch,n", [(17, 8216), (40, 200), (63, 8216), (65, 8200)])
def test_gated_rows_match_fp64(tmc, orc, torch, batch, n):
    """Gate/up + SiLU*Mul with the folded norm, packed output, at one and
    three tile pairs per block."""
    k = 2088
    x = dev_f16(orc.f16(normal(2021 + batch, (batch, k))))
    one = dev_f16(orc.f16(np.ones(k, np.float32)))
    wg = dev_f16(orc.f16(normal(2022, (n, k), 0.02)))
    wu = dev_f16(orc.f16(normal(2023, (n, k), 0.02)))
    out = torch.zeros(tmc.packed_activation_elements(batch, n), dtype=torch.float16, device="cuda")
    tmc.gate_up_silu_packed_norm(tmc.pack_activations(x), tmc.pack_weights(wg, gamma=one),
                                 tmc.pack_weights(wu, gamma=one), out, batch, k, n, 1e-6, 3)
    got = torch.empty((batch, n), dtype=torch.float16, device="cuda")
    tmc.pack_activations(out, got, unpack=True, rows=batch, cols=n)
    xd = x.double()
    norm = xd / torch.sqrt((xd * xd).mean(-1, keepdim=True) + 1e-6)
    g, u = norm @ wg.double().t(), norm @ wu.double().t()
    assert_f16_path(values(got), (g / (1 + torch.exp(-g)) * u).cpu().numpy(), what=f"b{batch}")


@pytest.mark.parametrize("batch,qh", [(33, 8), (64, 48)])
def test_qkv_rope_rows_equal_unfused(tmc, orc, torch, batch, qh):
    """RoPE + append in the epilogue of several row (and column) tiles writes
    the bits of the packed GEMM followed by the append kernel."""
    kvh, d, hidden, cap, p = qh, 64, 1032, 64, 16
    mp, width = cap // p, 3 * qh * 64
    rng = np.random.default_rng(2031)
    w = tmc.pack_weights(dev_f16(orc.f16(normal(2032, (width, hidden), 0.05))))
    x = tmc.pack_activations(dev_f16(orc.f16(normal(2033, (batch, hidden)))))
    i32 = lambda a: torch.tensor(np.asarray(a, np.int32), device="cuda")  # noqa: E731
    ang = np.arange(cap)[:, None] * 10000.0 ** (-np.arange(0, d, 2) / d)
    cos, sin = (torch.tensor(f(ang).astype(np.float32), device="cuda") for f in (np.cos, np.sin))
    tables = rng.permutation(batch * mp).reshape(batch, mp)
    args = (cos, sin, i32(rng.integers(1, cap + 1, batch)), i32(tables), i32([batch]))
    out = []
    for fused in (True, False):
        q = torch.full((batch, qh * d), float("nan"), dtype=torch.float16, device="cuda")
        kp = torch.zeros((batch * mp, kvh, p, d), dtype=torch.float16, device="cuda")
        vp = torch.zeros_like(kp)
        if fused:
            tmc.qkv_rope_append_packed(x, w, *args, q, kp, vp, batch, hidden, qh, kvh, d, cap, p,
                                       mp, 1)
        else:
            qkv = torch.empty((batch, width), dtype=torch.float16, device="cuda")
            tmc.gemm_packed_ex(x, w, qkv, batch, hidden, width, 1)
            tmc.decode_rope_append(qkv, *args, q, kp, vp, batch, qh, kvh, d, cap, p, mp)
        torch.cuda.synchronize()
        out.append([bits(t) for t in (q, kp, vp)])
    for a, b in zip(*out):
        assert np.array_equal(a, b)


def _norm_ref(x, w, gamma):
    xd = x.double()
    norm = xd / ((xd * xd).mean(-1, keepdim=True) + 1e-6).sqrt()
    return norm @ (w.float() * gamma.float()).half().double().t()


@pytest.mark.parametrize("batch,n", [(65, 12300), (80, 12300), (130, 12288), (70, 20000)])
def test_norm_remainder_rows_match_fp64(tmc, orc, torch, batch, n):
    """Folded norm, a last pass of at most 16 rows after 64-row passes with
    three column tiles: logits and the token-only head's tokens."""
    k = 1096
    x = dev_f16(orc.f16(normal(2041 + batch, (batch, k))))
    gamma = dev_f16(orc.f16(uniform(2042, (k,), 0.5, 1.5)))
    w = dev_f16(orc.f16(normal(2043, (n, k), 0.02)))
    packed, xin = tmc.pack_weights(w, gamma=gamma), tmc.pack_activations(x)
    y = torch.full((batch, n), float("nan"), dtype=torch.float32, device="cuda")
    tmc.gemm_packed_norm(xin, packed, y, batch, k, n, 1e-6, 1)
    assert_f32_rel(values(y), _norm_ref(x, w, gamma).cpu().numpy(), what=f"b{batch} n{n}")
    ws = torch.zeros(tmc.lm_head_argmax_workspace_bytes(batch, n) // 4, dtype=torch.float32,
                     device="cuda")
    tok = torch.full((batch,), -7, dtype=torch.int32, device="cuda")
    tmc.lm_head_argmax_packed_norm(xin, packed, ws, tok, batch, k, n, 1e-6, 1)
    assert torch.equal(tok.long(), y.argmax(-1))


@pytest.mark.parametrize("batch,n", [(65, 11008), (80, 11008), (97, 9600), (112, 9600),
                                     (96, 10400)])
def test_gated_remainder_rows_match_fp64(tmc, orc, torch, batch, n):
    """Gate/up: last passes of one to three row tiles with one column tile
    after passes with three."""
    k = 2056
    x = dev_f16(orc.f16(normal(2051 + batch, (batch, k))))
    one = dev_f16(orc.f16(np.ones(k, np.float32)))
    wg, wu = (dev_f16(orc.f16(normal(s, (n, k), 0.02))) for s in (2052, 2053))
    out = torch.zeros(tmc.packed_activation_elements(batch, n), dtype=torch.float16, device="cuda")
    tmc.gate_up_silu_packed_norm(tmc.pack_activations(x), tmc.pack_weights(wg, gamma=one),
                                 tmc.pack_weights(wu, gamma=one), out, batch, k, n, 1e-6, 3)
    got = torch.empty((batch, n), dtype=torch.float16, device="cuda")
    tmc.pack_activations(out, got, unpack=True, rows=batch, cols=n)
    g, u = _norm_ref(x, wg, one), _norm_ref(x, wu, one)
    assert_f16_path(values(got), (g / (1 + torch.exp(-g)) * u).cpu().numpy(), what=f"b{batch}")


@pytest.mark.parametrize("batch", [65, 80])
def test_norm_qkv_remainder_rows_equal_their_own_call(tmc, orc, torch, batch):
    """Fused q.k.v of 12288 columns: the 64-row pass and the remainder write
    the bits of calls of their own, K/V pages included."""
    qh, d, hidden, cap, p = 32, 128, 1096, 64, 16
    mp, width = cap // p, 3 * qh * d
    rng = np.random.default_rng(2061)
    one = dev_f16(orc.f16(np.ones(hidden, np.float32)))
    w = tmc.pack_weights(dev_f16(orc.f16(normal(2062, (width, hidden), 0.05))), gamma=one)
    x = dev_f16(orc.f16(normal(2063, (batch, hidden))))
    i32 = lambda a: torch.tensor(np.asarray(a, np.int32), device="cuda")  # noqa: E731
    ang = np.arange(cap)[:, None] * 10000.0 ** (-np.arange(0, d, 2) / d)
    cos, sin = (torch.tensor(f(ang).astype(np.float32), device="cuda") for f in (np.cos, np.sin))
    tables, lengths = rng.permutation(batch * mp).reshape(batch, mp), rng.integers(1, cap + 1, batch)
    whole, parts = [], []
    for cuts, out in (([(0, batch)], whole), ([(0, 64), (64, batch)], parts)):
        q = torch.full((batch, qh * d), float("nan"), dtype=torch.float16, device="cuda")
        kp = torch.zeros((batch * mp, qh, p, d), dtype=torch.float16, device="cuda")
        vp = torch.zeros_like(kp)
        for a, b in cuts:
            tmc.rmsnorm_qkv_rope_append_packed(
                tmc.pack_activations(x[a:b].contiguous()), w, cos, sin, i32(lengths[a:b]),
                i32(tables[a:b]), i32([b - a]), q[a:b], kp, vp, b - a, hidden, qh, qh, d, cap, p,
                mp, 1e-6, 1)
        torch.cuda.synchronize()
        out.extend(bits(t) for t in (q, kp, vp))
    for a, b in zip(whole, parts):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("unroll", [1, 2, 4])
@pytest.mark.parametrize("batch,ks", [(24, 2), (40, 16), (64, 3), (70, 1)])
def test_a_chosen_split_is_every_passes_split(tmc, orc, torch, batch, ks, unroll):
    """A caller's k split and unroll hold above 16 rows and at widths whose
    default is three column tiles: the bits of 16-row calls with them, with
    the folded norm (at most 4 waves) as well."""
    k, n = 1160, 12288
    x = dev_f16(orc.f16(normal(2071 + batch, (batch, k))))
    w = dev_f16(orc.f16(normal(2072, (n, k), 0.02)))
    packed = tmc.pack_weights(w)

    def rows(run, cfg):
        return torch.cat([run(x[a:a + 16].contiguous(), cfg) for a in range(0, batch, 16)])

    def plain(rows_x, cfg):
        return _rows(tmc, torch, rows_x, packed, rows_x.shape[0], k, n, 1, cfg)

    def norm(rows_x, cfg):
        y = torch.full((rows_x.shape[0], n), float("nan"), dtype=torch.float32, device="cuda")
        tmc.gemm_packed_norm(tmc.pack_activations(rows_x), packed, y, rows_x.shape[0], k, n, 1e-6, 1,
                             cfg)
        return y

    cfg = tmc.GemvConfig(3, 1, unroll, ks)
    assert torch.equal(plain(x, cfg), rows(plain, cfg))
    cfg = tmc.GemvConfig(3, 1, unroll, min(ks, 4))
    assert torch.equal(norm(x, cfg), rows(norm, cfg))


@pytest.mark.parametrize("ks", [3, 16])
def test_a_chosen_split_of_two_matrices(tmc, orc, torch, ks):
    batch, k, n = 40, 1160, 11008
    x = dev_f16(orc.f16(normal(2081, (batch, k))))
    wg, wu = (tmc.pack_weights(dev_f16(orc.f16(normal(s, (n, k), 0.02)))) for s in (2082, 2083))
    cfg = tmc.GemvConfig(3, 1, 1, ks)

    def run(rows_x):
        y = torch.full((rows_x.shape[0], n), float("nan"), dtype=torch.float16, device="cuda")
        tmc.gate_up_silu_packed(rows_x, wg, wu, y, n, cfg)
        return y

    assert torch.equal(run(x), torch.cat([run(x[a:a + 16].contiguous()) for a in (0, 16, 32)]))
