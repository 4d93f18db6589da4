"""Chunk states in one pass (chunk_seq_kernel) against chunk sums and carry: the same bits, in every result.  At the edges of its walk: one state
and several, walks of one tile up to more than it copies ahead, last chunks (the reverse walk's first step) down to one row and of whole tiles, heads with
and without the order by XCD, shorter chunks, strided layouts, split mode (at D = 256: the one-pass kernel has none at 128), as many states as its tables hold
and one more; launches that the rule takes to it; gates and values at the ends of their ranges."""
import pytest
import torch

from _mlstm_pkg import submodule

pytestmark = pytest.mark.gpu
mm = submodule("mlstm_matmul")
ffi = submodule("_ffi")
DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16}


def _run(x, dh, precise, L):
    h, m, b, saved = mm.mlstm_forward_save_hip(*x, precise=precise)
    grads = mm.mlstm_backward_saved_hip(dh, *x, h, m, b, saved, precise=precise)
    B, NH, S, D = x[0].shape
    n = B * NH * ((S - 1) // (L or 512)) * D * D   # the forward's states themselves (behind the header; those of two terms one set behind the other)
    states = saved.view(torch.uint8)[256:256 + 2 * n].clone().view(x[0].dtype)
    return [states, mm.mlstm_forward_hip(*x, precise=precise)[0], h, m, b, *grads, *mm.mlstm_backward_hip(dh, *x, precise=precise)]


def _inputs(dt, B, NH, S, D, strided, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    n = lambda *s: torch.randn(s, device="cuda", generator=g)  # noqa: E731
    rows = lambda: (n(B, S, NH, D).to(DTYPES[dt]).transpose(1, 2) if strided else n(B, NH, S, D).to(DTYPES[dt]))  # noqa: E731
    return [rows(), rows(), rows(), n(B, NH, S) + 3, n(B, NH, S)], rows()


def _same(x, dh, precise, L, variants=(1, 2, 0)):
    """The same bits in every result whichever kernels form the states; what is not a number is so in all of them.  Returns the results."""
    try:
        ffi.set_chunk_length(L)
        outs = []
        for variant in variants:
            ffi.set_state_kernel(variant)
            outs.append(_run(x, dh, precise, L))
    finally:
        ffi.set_chunk_length(0)
        ffi.set_state_kernel(0)
    assert ffi.lib().mlstm_kernel_error() == 0
    for other in outs[1:]:
        for k, (a, b) in enumerate(zip(outs[0], other)):
            assert torch.equal(a.isnan(), b.isnan()), (k, int(a.isnan().sum()), int(b.isnan().sum()))
            assert torch.equal(a.nan_to_num(0.0, float("inf"), float("-inf")), b.nan_to_num(0.0, float("inf"), float("-inf"))), k
    return outs[0]


TYPES = [("bf16", False), ("f16", False), ("bf16", True), ("f16", True)]
SIZES = [
    (1, 3, 1024, 256, 0, False), (1, 2, 1025, 128, 0, False), (1, 8, 1088, 256, 0, False), (2, 4, 1600, 128, 0, True), (1, 8, 1777, 256, 0, True),
    (1, 5, 2560, 128, 0, False), (1, 2, 1000, 128, 128, False), (1, 3, 1161, 256, 256, False), (1, 3, 1537, 128, 384, True), (2, 8, 1024, 256, 128, False),
    # walks of two tiles forward and one, two or four back
    (1, 2, 129, 128, 128, False), (1, 2, 192, 256, 128, False), (1, 3, 256, 256, 128, True), (1, 3, 257, 128, 128, False), (1, 2, 300, 256, 128, False),
    # 256 states and 257 (two kernels)
    (1, 1, 128 * 256 + 1, 128, 128, False), (1, 1, 128 * 257 + 70, 128, 128, False),
    # launches that the rule takes to the one-pass kernel: less than a round of workgroups, a whole one, more
    (1, 32, 1100, 128, 0, False), (2, 8, 1088, 256, 0, True), (1, 64, 1090, 128, 0, False), (5, 8, 1025, 256, 0, False), (2, 32, 1024, 256, 0, False),
]


@pytest.mark.parametrize("B,NH,S,D,L,strided,dt,precise", [(*size, *t) for size in SIZES for t in TYPES if not (t[1] and size[3] == 128)])
def test_same_bits_as_two_kernels(B, NH, S, D, L, strided, dt, precise):
    x, dh = _inputs(dt, B, NH, S, D, strided, S + D + L)
    for t in _same(x, dh, precise, L):
        assert torch.isfinite(t).all()


# A decay between chunks of 0 (in every chunk; behind a position in the middle), input gates that nothing else comes near, values that are not finite in a whole
# chunk and at the sequence's last position, whose tile may be short or the only one of a short chunk.
@pytest.mark.parametrize("B,NH,S,D,L,dt,precise", [(*size, *t) for size in [
    (1, 3, 1088, 256, 0), (1, 2, 1100, 256, 0), (1, 3, 1600, 128, 0), (1, 2, 1777, 128, 0), (1, 26, 1088, 256, 0), (1, 40, 1600, 128, 0), (1, 2, 1088, 128, 256), (1, 3, 700, 256, 384),
] for t in TYPES if not (t[1] and size[3] == 128)])
@pytest.mark.parametrize("what", ["forgets", "forgets once", "large input gates", "infinite", "infinite last", "nan last"])
def test_same_bits_at_the_ends_of_the_ranges(what, B, NH, S, D, L, dt, precise):
    (q, k, v, f, i), dh = _inputs(dt, B, NH, S, D, False, S + D)
    if what == "forgets":
        f -= 60
    elif what == "forgets once":
        f[:, :, 700 % S] = -1000
    elif what == "large input gates":
        i[:, :, ::97] += 80
    elif what == "infinite":
        k[:, 0, 100, 7] = float("inf")
        v[:, 1, 130, 9] = float("-inf")
        q[:, 0, 600, 3] = float("inf")
        dh[:, 1, 640, 11] = float("inf")
    else:
        value = float("inf" if what == "infinite last" else "nan")
        q[:, 0, -1, 5] = value
        dh[:, 1, -1, 11] = value
    _same([q, k, v, f, i], dh, precise, L)


@pytest.mark.parametrize("dt", ["bf16", "f16"])
@pytest.mark.parametrize("variant", [1, 2])
@pytest.mark.parametrize("NH,S,D,L", [(2, 1025, 128, 0), (2, 1088, 256, 0), (40, 1100, 128, 0), (40, 1088, 128, 0), (26, 1279, 256, 0), (26, 1088, 256, 0), (2, 1100, 256, 256), (2, 1088, 128, 384)])
def test_an_infinite_last_query_of_a_partial_chunk(dt, variant, NH, S, D, L):
    # Column 5 of the last query is infinite, and all that meets it on the way to dK of earlier chunks is positive (values, dh and, by an h that
    # opposes dh, the row's share of the normaliser): dK is infinite there and not NaN, which a row past the end with a weight of zero would make it.
    (q, k, v, f, i), dh = _inputs(dt, 1, NH, S, D, False, S)
    f += 3
    v = v.abs() + 0.5
    dh[:, :, -1] = dh[:, :, -1].abs() + 0.5
    full = (S - 1) // (L or 512) * (L or 512)
    try:
        ffi.set_chunk_length(L)
        ffi.set_state_kernel(variant)
        h, m, b, saved = mm.mlstm_forward_save_hip(q, k, v, f, i)
        b[:, :, -1] = b[:, :, -1].abs() + 10   # (above the normaliser's floor)
        h[:, :, -1] = -dh[:, :, -1]
        clean = mm.mlstm_backward_saved_hip(dh, q, k, v, f, i, h, m, b, saved)[1]
        assert bool(torch.isfinite(clean).all())
        q[:, :, -1, 5] = float("inf")
        dk = mm.mlstm_backward_saved_hip(dh, q, k, v, f, i, h, m, b, saved)[1][:, :, :full]
    finally:
        ffi.set_chunk_length(0)
        ffi.set_state_kernel(0)
    assert bool(torch.isposinf(dk[..., 5]).all()), (int(dk[..., 5].isnan().sum()), int(torch.isfinite(dk[..., 5]).sum()))
    assert bool(torch.isfinite(dk[..., [c for c in range(D) if c != 5]]).all())


