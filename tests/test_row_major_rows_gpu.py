"""Row-major MFMA linear layers (batch above 1): blocks whose height follows
the output width (heights 8 to 48, one short and one past whole blocks), up to
64 batch rows per launch, ragged k, and configurations chosen by the caller."""
import pytest

from tests.helpers import assert_f16_path, assert_f32_rel, dev_f16, normal, values

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch,k,n", [
    (2, 64, 1), (3, 136, 17), (7, 4104, 5003), (16, 1160, 2049), (17, 520, 4097), (31, 2056, 700),
    (33, 1000, 5121), (48, 264, 12288), (64, 4096, 4095), (65, 136, 12289), (5, 264, 33000),
    (12, 72, 60001)])
def test_row_major_linear_matches_fp64(tmc, orc, batch, k, n):
    import torch
    x = dev_f16(orc.f16(normal(4001 + batch, (batch, k))))
    w = torch.empty((n, k), dtype=torch.float16, device="cuda")
    tmc.fill_normal(w, 4002 + n, 0.0, 0.02)
    y = torch.full((batch, n), float("nan"), dtype=torch.float32, device="cuda")
    tmc.gemv(x, w, y)
    ref = x.double() @ w.double().t()
    assert_f32_rel(values(y), ref.cpu().numpy(), what=f"{batch}x{k}x{n}")


@pytest.mark.parametrize("batch,k,n", [(2, 64, 9), (9, 4096, 11008), (30, 1160, 4097),
                                       (50, 520, 3000), (64, 264, 33000), (40, 264, 9000),
                                       (48, 520, 12288)])
def test_row_major_gated_matches_fp64(tmc, orc, batch, k, n):
    import torch
    x = dev_f16(orc.f16(normal(4011 + batch, (batch, k))))
    wg, wu = (torch.empty((n, k), dtype=torch.float16, device="cuda") for _ in range(2))
    tmc.fill_normal(wg, 4012, 0.0, 0.02)
    tmc.fill_normal(wu, 4013, 0.0, 0.02)
    y = torch.full((batch, n), float("nan"), dtype=torch.float16, device="cuda")
    tmc.gate_up_silu(x, wg, wu, y)
    g, u = x.double() @ wg.double().t(), x.double() @ wu.double().t()
    assert_f16_path(values(y), (g / (1 + torch.exp(-g)) * u).cpu().numpy(), what=f"{batch}x{k}x{n}")


@pytest.mark.parametrize("batch,k,n", [(2, 520, 4096), (7, 4104, 5003), (16, 1160, 9000),
                                       (30, 4104, 5003), (24, 520, 33000), (1, 4096, 4096)])
def test_the_default_configuration_names_the_default(tmc, orc, batch, k, n):
    """tmc_gemv_default_config's result gives the default's bits; so does
    tmc_skinny_gemm_f16_mfma above batch 1."""
    import torch
    x = dev_f16(orc.f16(normal(4031 + batch, (batch, k))))
    w, wu = (torch.empty((n, k), dtype=torch.float16, device="cuda") for _ in range(2))
    tmc.fill_normal(w, 4032, 0.0, 0.02)
    tmc.fill_normal(wu, 4033, 0.0, 0.02)
    y, z, s = (torch.full((batch, n), float("nan"), device="cuda") for _ in range(3))
    tmc.gemv(x, w, y)
    tmc.gemv_config(x, w, z, tmc.default_config(batch, k, n))
    assert torch.equal(y, z)
    if batch > 1:
        tmc.skinny_gemm(x, w, s)
        assert torch.equal(y, s)
    y, z = (torch.full((batch, n), float("nan"), dtype=torch.float16, device="cuda")
            for _ in range(2))
    tmc.gate_up_silu(x, w, wu, y)
    tmc.gate_up_silu_config(x, w, wu, z, tmc.default_config(batch, k, n, True))
    assert torch.equal(y, z)


@pytest.mark.parametrize("cfg", [(3, 1, 4, 16), (3, 2, 4, 8), (3, 4, 2, 9), (3, 4, 1, 16),
                                 (3, 2, 1, 1)])
def test_chosen_row_tiles_match_the_default(tmc, orc, cfg):
    """Configurations with more and with at most 8 waves, against 64 bits."""
    import torch
    batch, k, n = 19, 2184, 1000
    x = dev_f16(orc.f16(normal(4021, (batch, k))))
    w = dev_f16(orc.f16(normal(4022, (n, k), 0.02)))
    y = torch.full((batch, n), float("nan"), dtype=torch.float32, device="cuda")
    tmc.gemv_config(x, w, y, tmc.GemvConfig(*cfg))
    assert_f32_rel(values(y), (x.double() @ w.double().t()).cpu().numpy(), what=str(cfg))
