"""Which workgroups of a column kernel run together, and which column kernel serves a launch, changes no bit: a head's gradients are the same among
many heads as among three.  Numbers of heads that the XCDs share out evenly (multiples of 8), uncut and in chunks of which the last is short, on
either side of the lines between the kernels."""
import pytest
import torch

from _mlstm_pkg import submodule

pytestmark = pytest.mark.gpu
mm = submodule("mlstm_matmul")
DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}


def _grads(x, dh, precise):
    h, m, b, saved = mm.mlstm_forward_save_hip(*x, precise=precise)
    return mm.mlstm_backward_saved_hip(dh, *x, h, m, b, saved, precise=precise)


@pytest.mark.parametrize("dt,D,precise,NH,S", [
    ("bf16", 64, False, 16, 1700), ("f16", 64, False, 40, 300), ("bf16", 64, True, 16, 1700), ("f32", 64, False, 16, 1700), ("f32", 64, False, 64, 300),
    ("bf16", 128, False, 32, 1700), ("bf16", 128, False, 64, 1000), ("bf16", 128, False, 17, 2048), ("f16", 128, False, 24, 2048), ("bf16", 128, False, 25, 2048),
    ("bf16", 256, False, 32, 1700), ("bf16", 256, False, 40, 1000), ("f16", 256, False, 40, 1000), ("bf16", 256, True, 32, 1700), ("f32", 128, False, 48, 300),
    ("bf16", 256, False, 36, 1000), ("bf16", 256, False, 37, 1000), ("bf16", 256, True, 37, 1000), ("bf16", 256, False, 30, 1100), ("bf16", 256, True, 24, 2048),
    ("bf16", 256, False, 320, 128), ("bf16", 256, False, 321, 128), ("bf16", 256, True, 600, 64), ("f16", 256, False, 40, 1100),
    ("bf16", 128, False, 101, 384), ("f16", 128, False, 102, 384), ("bf16", 128, False, 35, 1100), ("f16", 128, False, 36, 1100), ("f16", 128, True, 30, 1100), ("bf16", 128, True, 24, 2048),
])
def test_a_head_among_many(dt, D, precise, NH, S):
    g = torch.Generator(device="cuda").manual_seed(S + D + NH)
    n = lambda *s: torch.randn(s, device="cuda", generator=g)  # noqa: E731
    rows = lambda: n(1, NH, S, D).to(DTYPES[dt])  # noqa: E731
    x, dh = [rows(), rows(), rows(), n(1, NH, S) + 3, n(1, NH, S)], rows()
    few = [0, NH // 2, NH - 1]
    part = lambda t: t[:, few].contiguous()  # noqa: E731
    for k, (a, b) in enumerate(zip(_grads(x, dh, precise), _grads([part(t) for t in x], part(dh), precise))):
        assert torch.isfinite(a).all(), k
        assert torch.equal(part(a), b), k
