"""The generic kernels, row_kernel and col_kernel, at sizes that others serve by default: what the generic switch selects, fp32 against the oracle
and bit by bit against rowf_kernel and colf_kernel, and what is not finite formed again by them too."""
import pytest
import torch
from torch.profiler import ProfilerActivity, profile

from _mlstm_pkg import submodule
from oracle import mlstm_oracle as O
from tests import test_gpu_variants as variants
from tests.helpers import assert_close, assert_matches_oracle

pytestmark = pytest.mark.gpu
ffi, mm = submodule("_ffi"), submodule("mlstm_matmul")


@pytest.fixture
def generic():
    before = ffi.force_generic_kernels(True)
    yield
    ffi.force_generic_kernels(before)


def _step(q, k, v, f, i, dh):
    h, m, b, saved = mm.mlstm_forward_save_hip(q, k, v, f, i)
    return [h, m, b, *mm.mlstm_backward_saved_hip(dh, q, k, v, f, i, h, m, b, saved)]


@pytest.mark.parametrize("D,dtype", [(64, torch.float32), (128, torch.float32), (64, torch.bfloat16), (128, torch.float16), (256, torch.bfloat16)])
@pytest.mark.parametrize("S", [200, 1100])
def test_the_switch_selects_them(generic, S, D, dtype):
    ins = [t.cuda() for t in O.make_inputs(1, 2, S, D, dtype, seed=S, f_mean=3.0)]
    torch.cuda.synchronize()
    with profile(activities=[ProfilerActivity.CUDA]) as p:
        _step(*ins)
        torch.cuda.synchronize()
    recorded = [e.key for e in p.key_averages() if "mlstm" in e.key]
    if not recorded:
        pytest.skip("the profiler records no kernels here")
    names = [key for key in recorded if any(s in key for s in ("row", "col")) and "rowreduce" not in key]
    assert names and all("row_kernel" in n or "col_kernel" in n for n in names), names


# (in chunks of 128 at D = 128 col_kernel is reached by the switch alone)
@pytest.mark.parametrize("S,D", [(33, 64), (200, 64), (450, 64), (65, 128), (230, 128), (450, 128)])
def test_fp32_against_the_oracle(generic, S, D):
    q, k, v, f, i, dh = O.make_inputs(1, 2, S, D, torch.float32, seed=S, f_mean=3.0)
    h, m, b, *grads = _step(*(t.cuda() for t in (q, k, v, f, i, dh)))
    assert_matches_oracle(torch.float32, q, k, v, f, i, dh=dh, h=h, m=m, b=b, grads=grads)


@pytest.mark.parametrize("S,D", [(1, 64), (97, 128), (319, 64), (320, 128), (450, 64), (450, 128), (700, 128), (1025, 64)])
def test_fp32_same_bits_as_the_kernels_for_few_workgroups(S, D):
    ins = [t.cuda() for t in O.make_inputs(1, 2, S, D, torch.float32, seed=S, f_mean=3.0)]
    ours = _step(*ins)
    before = ffi.force_generic_kernels(True)
    try:
        theirs = _step(*ins)
    finally:
        ffi.force_generic_kernels(before)
    for name, a, b in zip(("h", "m", "b", "dq", "dk", "dv", "df", "di"), ours, theirs):
        assert bool(torch.isfinite(a).all()) and torch.equal(a, b), name


@pytest.mark.parametrize("S,at", [(200, 150), (400, 150), (400, 399)])
@pytest.mark.parametrize("D", [64, 128])
def test_fp32_keeps_what_is_not_finite(generic, D, S, at):
    variants.test_fp32_terms_keep_what_is_not_finite(D, S, at, float("inf"))


@pytest.mark.parametrize("B,NH,S,D,at", [(1, 2, 200, 64, 0), (1, 1, 63, 64, 40), (1, 2, 400, 64, 3), (2, 1, 450, 64, 300), (1, 2, 200, 128, 100), (1, 2, 450, 128, 3),
                                         (1, 1, 450, 128, 449)])
def test_fp32_rows_and_keys_formed_again(generic, B, NH, S, D, at):
    variants.test_fp32_rows_and_keys_formed_again(B, NH, S, D, at)


# the same on launches that are large enough for the generic kernels by themselves: one head of many
@pytest.mark.parametrize("S,D,at,heads", [(200, 64, 3, 40), (200, 64, 100, 40), (400, 64, 300, 24), (200, 128, 40, 70), (63, 128, 0, 260)])
def test_fp32_rows_and_keys_of_one_head_formed_again(S, D, at, heads):
    q, k, v, f, i, dh = O.make_inputs(1, 1, S, D, torch.float32, seed=S + at, f_mean=3.0)
    q[..., 7] = 0
    k[..., at, 7] = 0
    dh *= 1e-3
    want = [O.mlstm_forward_dense(q, k, v, f, i)[0], *O.mlstm_backward_dense(dh, q, k, v, f, i, zero_first_df=True)]
    ins = [t.cuda().repeat(1, heads, *([1] * (t.dim() - 2))) for t in (q, k, v, f, i, dh)]
    ins[1][0, 5, at, 7] = 3.4e38
    h, _, _, *grads = _step(*ins)
    keep = [d for d in range(D) if d != 7]
    for name, g, w in zip(("h", "dq", "dk", "dv", "df", "di"), (h, *grads), want):
        for head in (4, 5, 6):
            assert_close(*((t[..., keep] if name == "dq" else t) for t in (g[:, head:head + 1], w)), torch.float32, name)
