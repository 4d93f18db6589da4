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


# a row kernel that forms the gates of its head by itself (16 bits, D = 128 and 256, sequences that are not cut) against the pre-pass (more heads): every
# type of gates and of layout (values at either half of a dword), one to sixteen granules, and what the backward reads
@pytest.mark.parametrize("gates", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("S,D,layout", [(1, 128, "bns"), (63, 256, "bns"), (65, 128, "bsn"), (255, 128, "bns"), (257, 256, "bsn"), (513, 128, "bns"), (770, 128, "bsn"),
                                        (1023, 256, "bns"), (1023, 128, "bsn")])
def test_gates_formed_by_the_row_kernel(S, D, layout, gates):
    NG = (S + 63) // 64
    g = torch.Generator(device="cuda").manual_seed(S)
    for heads in (1, 128 // NG + 1):   # workgroups of 32 and of 64 rows
        many = (256 + 8 * NG) // NG + 1
        rows = [torch.randn(1, many, S, D, device="cuda", generator=g).bfloat16() for _ in range(4)]
        shape = (1, many, S) if layout == "bns" else (1, S, many)
        f, i = [(torch.randn(shape, device="cuda", generator=g) + c).to(gates) for c in (3, 0)]
        if layout == "bsn":
            f, i = f.transpose(1, 2), i.transpose(1, 2)
        def step(n, offset):
            q, k, v, dh = [t[:, :n] for t in rows]
            # (the same values from an address of either parity, in the same layout)
            def moved(t):
                flat = torch.empty(t.numel() + offset, device="cuda", dtype=gates)[offset:]
                return flat.view(shape[:1] + ((n, S) if layout == "bns" else (S, n))).copy_(t if layout == "bns" else t.transpose(1, 2)).transpose(1, 1 if layout == "bns" else 2)
            a, b = moved(f[:, :n]), moved(i[:, :n])
            h, m, bs, saved = mm.mlstm_forward_save_hip(q, k, v, a, b)
            return [h, m, bs, *mm.mlstm_backward_saved_hip(dh, q, k, v, a, b, h, m, bs, saved)]
        want = step(many, 0)
        for offset in (0, 1):
            for name, x, y in zip(range(8), step(heads, offset), want):
                assert bool(torch.isfinite(y.float()).all()) and torch.equal(x, y[:, :heads]), (name, offset, heads)
