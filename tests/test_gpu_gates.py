"""The gate pre-pass at the lengths and numbers of heads where it changes form: granules of 64 positions, 4 or 16 of them per workgroup,
one launch up to 4096 positions and two beyond, up to the longest sequence; by the stabiliser m_t = F_t + max_{j <= t} (i_j - F_j) in 64 bits."""
import pytest
import torch

from _mlstm_pkg import submodule

pytestmark = pytest.mark.gpu
mm = submodule("mlstm_matmul")


def check(f, i, lf, gate_form="raw"):
    BH, S = f.shape
    q = torch.zeros(1, BH, S, 64, device="cuda", dtype=torch.bfloat16)
    m = mm.mlstm_forward_hip(q, q, q, f.cuda()[None], i.cuda()[None], gate_form=gate_form)[1][0].cpu().double()
    F = torch.cumsum(lf, -1)
    best, at = torch.cummax(i.double() - F, -1)
    want = F + best
    # one logarithm is good to 3e-7 of itself, a sum inside a granule takes eight roundings, and those between the maximum's position and t add up
    bound = 4e-7 * (64 + (torch.gather(F, 1, at) - F).abs() + want.abs() + i.double().abs())
    assert bool(((m - want).abs() <= bound).all()), float(((m - want).abs() / bound).max())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("BH,S", [(2, s) for s in (1, 63, 65, 257, 1024, 1025, 2049, 4033, 4096, 4097, 5121, 8193, 65600, 131072)] + [(70, 1000), (140, 513), (17, 4096), (33, 5000)])
def test_stabiliser(BH, S, dtype):
    g = torch.Generator().manual_seed(S)
    f, i = (torch.randn(BH, S, generator=g) + 3).to(dtype), torch.randn(BH, S, generator=g).to(dtype)
    i[:, ::977] += 20   # (maxima that stay for many granules)
    check(f, i, torch.nn.functional.logsigmoid(f.double()))


@pytest.mark.parametrize("S", [1000, 3000, 9000])
def test_given_sums(S):
    g = torch.Generator().manual_seed(S)
    lf = torch.nn.functional.logsigmoid(torch.randn(3, S, generator=g) + 3)
    i = torch.randn(3, S, generator=g)
    check(lf, i, lf.double(), "logsigmoid")
    F = torch.cumsum(lf, -1)
    check(F, i, torch.diff(F.double(), prepend=torch.zeros(3, 1, dtype=torch.float64)), "cumsum")
