"""The weight-streaming kernel on narrow outputs of the down projection (512 .. 2048 features, up to 16 rows), where a workgroup
owns 4 or 8 features: feature counts at the edges of those ranges and tails of a workgroup, K from one vector over one and two steps
of every wave to several, both fetches of the activations, both sides of the K from which a workgroup is narrow. Against the fp64 oracle under one rounding (half an ulp, twice, plus 1e-3
for fp32 sums in another order), Y and H inside wider NaN buffers."""
import pytest
import torch

from oracle import oracle

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("D", [511, 512, 514, 1000, 1023, 1024, 1025, 1030, 2041, 2048, 2049])
@pytest.mark.parametrize("M,FF", [(1, 8), (3, 128), (2, 512), (7, 520), (12, 648), (8, 1048), (9, 1024), (16, 2056), (1, 2816), (16, 4360), (5, 8192)])
def test_few_features_a_workgroup(capi, D, M, FF):
    dtype = torch.bfloat16 if (D + M) % 2 else torch.float16
    gen = torch.Generator().manual_seed(D + FF)
    H = (torch.randn(M, FF, generator=gen) * 0.5).to(dtype)
    W2 = (torch.randn(D, FF, generator=gen) / FF ** 0.5).to(dtype)
    wide_h = torch.full((M, FF + 8), float("nan"), dtype=dtype, device=DEV)
    wide_h[:, :FF] = H.to(DEV)
    wide_y = torch.full((M, D + 4), float("nan"), dtype=dtype, device=DEV)
    try:
        capi.set_variant(1, 100)
        capi.down(wide_h[:, :FF], W2.to(DEV), out=wide_y[:, :D])
    finally:
        capi.set_variant(1, -1)
    ref = oracle.ref_down(H, W2, torch.float64)
    err = (wide_y[:, :D].cpu().double() - ref).abs()
    assert (err <= ref.abs() * (2.0 ** -7 if dtype == torch.bfloat16 else 2.0 ** -10) + 1e-3).all(), err.max().item()
    assert torch.isnan(wide_y[:, D:]).all()
