"""Chunk states in one pass (chunk_seq_kernel) against chunk sums and carry: the same bits, in every result.  At the edges of its walk: one state
and several, last chunks of one tile (the reverse walk's first step) down to one row and of whole tiles, heads with and without the order by XCD,
shorter chunks, strided layouts, split mode; and the launches that the rule takes to it."""
import pytest
import torch

from _mlstm_pkg import submodule

pytestmark = pytest.mark.gpu
mm = submodule("mlstm_matmul")
ffi = submodule("_ffi")
DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16}


def _run(x, dh, precise):
    h, m, b, saved = mm.mlstm_forward_save_hip(*x, precise=precise)
    grads = mm.mlstm_backward_saved_hip(dh, *x, h, m, b, saved, precise=precise)
    return [mm.mlstm_forward_hip(*x, precise=precise)[0], h, m, b, *grads, *mm.mlstm_backward_hip(dh, *x, precise=precise)]


@pytest.mark.parametrize("dt,precise", [("bf16", False), ("f16", False), ("bf16", True), ("f16", True)])
@pytest.mark.parametrize("B,NH,S,D,L,strided", [
    (1, 3, 1024, 256, 0, False), (1, 2, 1025, 128, 0, False), (1, 8, 1088, 256, 0, False), (2, 4, 1600, 128, 0, True), (1, 8, 1777, 256, 0, True),
    (1, 5, 2560, 128, 0, False), (1, 2, 1000, 128, 128, False), (1, 3, 1161, 256, 256, False), (1, 3, 1537, 128, 384, True), (2, 8, 1024, 256, 128, False),
])
def test_same_bits_as_two_kernels(dt, precise, B, NH, S, D, L, strided):
    g = torch.Generator(device="cuda").manual_seed(S + D + L)
    n = lambda *s: torch.randn(s, device="cuda", generator=g)  # noqa: E731
    rows = lambda: (n(B, S, NH, D).to(DTYPES[dt]).transpose(1, 2) if strided else n(B, NH, S, D).to(DTYPES[dt]))  # noqa: E731
    x, dh = [rows(), rows(), rows(), n(B, NH, S) + 3, n(B, NH, S)], rows()
    try:
        ffi.set_chunk_length(L)
        outs = []
        for variant in (1, 2, 0):
            ffi.set_state_kernel(variant)
            outs.append(_run(x, dh, precise))
    finally:
        ffi.set_chunk_length(0)
        ffi.set_state_kernel(0)
    assert ffi.lib().mlstm_kernel_error() == 0
    for other in outs[1:]:
        for k, (a, b) in enumerate(zip(outs[0], other)):
            assert torch.equal(a, b), k
