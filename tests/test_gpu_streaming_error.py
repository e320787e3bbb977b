"""Rounding of H x and H^T x in FP32 on the 256^2 rank-16 matrix against the same
matrix in FP64. A chain of n products of random sign rounds to about u / sqrt(3)
sqrt(n / 2) of its result (u = 2^-24); an atom's 1,700 columns over four waves
are chains of 16 and of 27 of their sums, together 1.6e-7. Twice that is
allowed (the projections' own rounding comes on top); one chain of 430 gives
4e-7."""
import pytest

torch = pytest.importorskip("torch")        # before the library: both then share one HIP runtime
import dmhm_amd  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [1, 6])
@pytest.mark.parametrize("seed", [1, 2])
def test_fp32_sums_are_short_chains(k, seed):
    dmhm_amd.init(0)
    H = dmhm_amd.HMat2d.zeros([256, 256], 6, 16, True, dmhm_amd.DMHM_F32)
    H.SetToRandom(seed)
    D = H.Convert(dmhm_amd.DMHM_F64)
    x = torch.randn((k, 65536), generator=torch.Generator().manual_seed(seed)).cuda()
    for op in ("Multiply", "TransposeMultiply"):
        got = getattr(H, op)(1.0, x.t()).double()
        want = getattr(D, op)(1.0, x.double().t())
        assert float((got - want).norm() / want.norm()) <= 3.2e-7, op
