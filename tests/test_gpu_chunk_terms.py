"""Chunk sums of bf16 at D = 64 (weighted values as three bf16 terms) on the forward states and the reverse ones: a last chunk of one position up to a whole
one, heads beside each other in either layout, values that are not finite."""
import pytest
import torch

from _mlstm_pkg import submodule
from oracle import mlstm_oracle as O
from tests.helpers import assert_close, rounding_noise

pytestmark = pytest.mark.gpu
mm = submodule("mlstm_matmul")


def step(q, k, v, f, i, dh):
    h, m, b, saved = mm.mlstm_forward_save_hip(q, k, v, f, i)
    return [h, *mm.mlstm_backward_saved_hip(dh, q, k, v, f, i, h, m, b, saved)]


@pytest.mark.parametrize("S", [1024, 1025, 1279, 1281, 1535])
def test_against_oracle(S):
    # the bound of the 16-bit kernels: literal tolerance plus six predicted sigmas of rounding weights and states
    x = O.make_inputs(1, 3, S, 64, torch.bfloat16, seed=S, f_mean=3.0)
    q, k, v, f, i, dh = x
    hr, _, _ = O.mlstm_forward_dense(q, k, v, f, i)
    want = [hr, *O.mlstm_backward_dense(dh, q, k, v, f, i, zero_first_df=True)]
    sigma = rounding_noise(dh, q, k, v, f, i, torch.bfloat16, chunk_len=256)
    d = [t.cuda() for t in x]
    got = step(*d)
    for name, g, w in zip(("h", "dq", "dk", "dv", "df", "di"), got, want):
        assert_close(g, w, torch.bfloat16, name, sigma[name])
    # the same heads as views of [B,S,NH,D] projections: the same bits
    views = [t.transpose(1, 2).contiguous().transpose(1, 2) for t in d]
    for name, g, w in zip(("h", "dq", "dk", "dv", "df", "di"), step(*views), got):
        assert torch.equal(g, w), name


def test_values_that_are_not_finite():
    # an infinite value in the first chunk makes its own column of every later row not finite, and no other
    x = [t.cuda() for t in O.make_inputs(1, 2, 1100, 64, torch.bfloat16, seed=5, f_mean=6.0)]
    clean = mm.mlstm_forward_hip(*x[:5])[0]
    x[2][0, 1, 100, 37] = float("inf")
    h = mm.mlstm_forward_hip(*x[:5])[0]
    assert torch.equal(h[0, 0], clean[0, 0])
    assert not bool(torch.isfinite(h[0, 1, 256:, 37]).any())
    others = [c for c in range(64) if c != 37]
    # (its block of the state is formed again in another order: one rounding to bf16 of the state apart, 2^-8 of what the sum is made of)
    a, b = h[0, 1][:, others].float(), clean[0, 1][:, others].float()
    assert bool(torch.isfinite(a).all()) and float((a - b).norm() / b.norm()) <= 2.0 ** -8


@pytest.mark.parametrize("S", [1025, 1056, 1279])
def test_an_infinite_last_query_of_a_partial_chunk(S):
    # Column 5 of the last query is infinite, and all that meets it on the way to dK of earlier chunks is positive (values, dh and, by an h that
    # opposes dh, the row's share of the normaliser): dK is infinite there and not NaN, which a row past the end with a weight of zero would make it.
    q, k, v, f, i, dh = [t.cuda() for t in O.make_inputs(1, 2, S, 64, torch.bfloat16, seed=S, f_mean=6.0)]
    v = v.abs() + 0.5
    dh[:, :, -1] = dh[:, :, -1].abs() + 0.5
    h, m, b, saved = mm.mlstm_forward_save_hip(q, k, v, f, i)
    b[:, :, -1] = b[:, :, -1].abs() + 10   # (above the normaliser's floor)
    h[:, :, -1] = -dh[:, :, -1]
    clean = mm.mlstm_backward_saved_hip(dh, q, k, v, f, i, h, m, b, saved)[1]
    assert bool(torch.isfinite(clean).all())
    q[:, :, -1, 5] = float("inf")
    dk = mm.mlstm_backward_saved_hip(dh, q, k, v, f, i, h, m, b, saved)[1]
    assert bool(torch.isposinf(dk[:, :, :1024, 5]).all())
    others = [c for c in range(64) if c != 5]
    assert bool(torch.isfinite(dk[:, :, :1024][..., others]).all())
