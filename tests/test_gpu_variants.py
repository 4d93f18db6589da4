"""Edges of the dispatch rules: chunk lengths, the two carries of the chunk states, fp32 operands as three
bf16 terms, the scan form on the tile kernels and on its own, key ranges that share a partial numerator.  Forward and gradients
against the float64 oracle: fp32 to the fp32 bound of tests/helpers.py, 16-bit types to the predicted rounding noise."""
import pytest
import torch

from _mlstm_pkg import submodule
from oracle import mlstm_oracle as O
from tests.helpers import assert_close, assert_matches_oracle

pytestmark = pytest.mark.gpu
ffi, mm, ms = submodule("_ffi"), submodule("mlstm_matmul"), submodule("mlstm_scan")


def _check(B, NH, S, D, dtype, seed, chunk_len=0):
    q, k, v, f, i, dh = O.make_inputs(B, NH, S, D, dtype, seed=seed, f_mean=3.0)
    ts = [t.cuda().requires_grad_(True) for t in (q, k, v, f, i)]
    out = mm.Triton_mLSTM.apply(*ts)
    assert_matches_oracle(dtype, q, k, v, f, i, dh=dh, h=out.detach(), grads=torch.autograd.grad(out, ts, dh.cuda()), chunk_len=chunk_len)


# (16 bits: 1023 / 1024 are the last length that is not cut and the first in chunks.  The edges of the two carries: test_gpu_small_grids.)
# The last number is the chunk length the rule gives, which the noise prediction needs.
@pytest.mark.parametrize("B,NH,S,D,L", [(1, 2, 959, 64, 0), (1, 2, 1023, 64, 0), (1, 2, 1024, 64, 256), (1, 1, 1536, 64, 256), (1, 2, 1023, 128, 0),
                                        (1, 1, 1023, 256, 0), (1, 9, 1025, 256, 512), (1, 33, 1024, 128, 512), (16, 2, 1100, 128, 512),
                                        (1, 3, 1537, 128, 512)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_16_bit_chunk_lengths_and_carries(B, NH, S, D, L, dtype):
    assert int(ffi.lib().mlstm_chunk_length(B, NH, S, D, ffi.dtype_code(dtype))) == L
    _check(B, NH, S, D, dtype, seed=S + NH, chunk_len=L)


# A head's results are the same bits alone and in a batch, whatever the number of heads around it: with 40 heads the chunk states
# of D = 128 and 256 come from the other carry, with another split of dF's sums over workgroups.
@pytest.mark.parametrize("dtype,S,D", [(torch.bfloat16, 1000, 64), (torch.bfloat16, 1100, 128), (torch.float16, 2050, 128), (torch.bfloat16, 1500, 256),
                                       (torch.float16, 1000, 128), (torch.float32, 400, 64), (torch.float32, 700, 128), (torch.float32, 2048, 64)])
@pytest.mark.parametrize("op", ["Triton_mLSTM", "Triton_mLSTM_precise"])
def test_a_head_is_the_same_bits_in_any_batch(op, dtype, S, D):
    g = torch.Generator(device="cuda").manual_seed(S + D)
    rnd = lambda *s: torch.randn(s, device="cuda", generator=g).to(dtype)  # noqa: E731
    ins, dh = [rnd(1, 40, S, D), rnd(1, 40, S, D), rnd(1, 40, S, D), rnd(1, 40, S) + 3, rnd(1, 40, S)], rnd(1, 40, S, D)

    def step(heads):
        ts = [t[:, :heads].contiguous().requires_grad_(True) for t in ins]
        out = getattr(mm, op).apply(*ts)
        return [t[:, 0] for t in (out.detach(), *torch.autograd.grad(out, ts, dh[:, :heads].contiguous()))]
    alone = step(1)
    for heads in (9, 40):
        for name, a, b in zip(("h", "dq", "dk", "dv", "df", "di"), alone, step(heads)):
            assert torch.equal(a, b), (heads, name)


@pytest.mark.parametrize("B,NH,S,D", [(1, 2, 319, 64), (1, 2, 320, 64), (2, 1, 321, 128), (1, 1, 447, 128), (1, 3, 65, 128), (1, 1, 63, 64)])
def test_fp32_short_chunks(B, NH, S, D):
    _check(B, NH, S, D, torch.float32, seed=S)


# (D = 64, 128: tile kernels.  Key ranges of the scan kernels by heads: 256 two apart, from 32 heads two that share, from 64 one;
# 512 four apart, from 8 in two pairs, from 16 one pair; 1024 eight apart, from 2 heads in four pairs, from 4 in two)
@pytest.mark.parametrize("BH,S,D", [(2, 130, 64), (1, 400, 128), (3, 200, 256), (32, 65, 256), (64, 70, 256), (3, 130, 512), (8, 70, 512), (16, 70, 512),
                                    (1, 65, 1024), (2, 65, 1024), (4, 130, 1024)])
def test_scan_form_every_key_split(BH, S, D):
    q, k, v, f, i, dh = O.make_inputs(1, BH, S, D, torch.float32, seed=S + D, f_mean=3.0)
    o = torch.randn(q.shape, generator=torch.Generator().manual_seed(D))
    od, sg = o.double(), torch.sigmoid(o.double())
    hd, _, _ = O.mlstm_forward_dense(q, k, v, f, i)
    want = [hd * od * sg, *O.mlstm_backward_dense(dh.double() * od * sg, q.double(), k.double(), v.double(), f.double(), i.double(), zero_first_df=True),
            dh.double() * hd * sg * (1 + od * (1 - sg))]
    ts = [t.cuda().requires_grad_(True) for t in (q, k, v, f, i, o)]
    out = ms.mlstm_scan(*ts)
    got = [out.detach(), *torch.autograd.grad(out, ts, dh.cuda())]
    again = ms.mlstm_scan(*ts)
    for name, g, w, g2 in zip(("h", "dq", "dk", "dv", "df", "di", "do"), got, want, [again, *torch.autograd.grad(again, ts, dh.cuda())]):
        assert_close(g, w, torch.float32, name)
        assert torch.equal(g, g2), name   # (two contributions per shared element: the same bits in either order)


def _shifted(t, by):
    buf = torch.zeros(t.numel() + by, dtype=t.dtype, device="cuda")
    buf[by:] = t.flatten()
    return buf[by:].view(t.shape)


# Dense tensors that start off a 16-byte boundary, at the entry points that take no layout and therefore ask for no alignment: the
# scan kernels behind the matmul form in fp32 at D >= 256, every entry point that reaches them; the same bits as on a boundary.
@pytest.mark.parametrize("by", [1, 2])
@pytest.mark.parametrize("BH,S,D", [(2, 300, 256), (32, 140, 256), (1, 1100, 256), (16, 130, 512), (2, 130, 1024), (4, 200, 1024)])
def test_scan_kernels_on_rows_off_a_16_byte_boundary(BH, S, D, by):
    g = torch.Generator(device="cuda").manual_seed(S + D)
    rnd = lambda *s: torch.randn(s, device="cuda", generator=g)  # noqa: E731
    q, k, v, dh, o = (rnd(1, BH, S, D) for _ in range(5))
    f, i = rnd(1, BH, S) + 3, rnd(1, BH, S)
    L, P, null, F32 = ffi.lib(), ffi.ptr, ffi.ptr(None), ffi.F32

    def run(move):
        q_, k_, v_, dh_, o_ = (move(t) for t in (q, k, v, dh, o))
        new = lambda like: move(torch.zeros_like(like))  # noqa: E731
        out, st, shape = [], ffi.stream_ptr(), (1, BH, S, D, F32)
        h, m, b = new(q), torch.zeros_like(f), torch.zeros_like(f)
        ins = (P(q_), P(k_), P(v_), P(f), P(i))
        calls = [lambda: L.mlstm_forward_ex(*ins, P(h), P(m), P(b), *shape, F32, null, 0, st),
                 lambda: L.mlstm_forward_save_ex(*ins, P(h), P(m), P(b), null, 0, *shape, F32, null, 0, st)]
        if L.mlstm_workspace_bytes(ffi.OP_FORWARD, *shape) <= ffi.NOALLOC_MAX_WORKSPACE:
            calls.append(lambda: L.mlstm_forward_noalloc_ex(*ins, P(h), P(m), P(b), *shape, F32, st))
        calls.append(lambda: L.mlstm_scan_forward_ex(*ins, P(o_), P(h), *shape, null, 0, st))
        for call in calls:
            h.zero_()
            ffi.check_rc(call(), "forward")
            out += [h.clone(), m.clone(), b.clone()]
        gr = [new(q), new(q), new(q), torch.zeros_like(f), torch.zeros_like(f)]
        for call in (lambda: L.mlstm_backward_ex(P(dh_), *ins, null, null, null, *(P(t) for t in gr), *shape, F32, null, 0, st),
                     lambda: L.mlstm_backward_saved_ex(P(dh_), *ins, P(h), P(m), P(b), null, 0, *(P(t) for t in gr), *shape, F32, null, 0, st)):
            ffi.check_rc(call(), "backward")
            out += [t.clone() for t in gr]
        return out
    for n, (a, w) in enumerate(zip(run(lambda t: _shifted(t, by)), run(lambda t: t.clone()))):
        assert bool(torch.isfinite(a).all()) and torch.equal(a, w), n


# An output in host memory that the GPU can address: stores reach it, atomic adds may not, so shared partial numerators go elsewhere.
def test_scan_kernels_with_an_output_in_pinned_host_memory():
    q, k, v, f, i, _ = O.make_inputs(1, 16, 70, 512, torch.float32, seed=3, f_mean=3.0)
    dev = [t.cuda() for t in (q, k, v, f, i)]
    h = torch.zeros(q.shape, pin_memory=True)
    null = ffi.ptr(None)
    rc = ffi.lib().mlstm_forward_ex(*(ffi.ptr(t) for t in dev), ffi.ptr(h), null, null, 1, 16, 70, 512, ffi.F32, ffi.F32, null, 0, ffi.stream_ptr())
    ffi.check_rc(rc, "mlstm_forward_ex")
    torch.cuda.synchronize()
    assert_close(h, O.mlstm_forward_dense(q, k, v, f, i)[0], torch.float32, "h")


# Errors against 64 bits, medians over the rows of h, dQ, dK and dV, for inputs that the generator fixes: no larger than the same
# operators had on v_mfma_f32_32x32x2_f32 (the scan form on the scan kernels), which gave the bounds below on these inputs.
@pytest.mark.parametrize("form,S,D,bounds", [("scan", 1000, 64, (2.582e-7, 3.510e-7, 9.778e-7, 3.905e-7)),
                                             ("scan", 1000, 128, (2.748e-7, 3.767e-7, 1.167e-6, 4.359e-7)),
                                             ("matmul", 300, 128, (3.037e-7, 4.530e-7, 1.528e-6, 6.394e-7)),
                                             ("matmul", 1000, 64, (2.720e-7, 3.847e-7, 1.217e-6, 5.665e-7)),
                                             ("scan", 500, 256, (2.838e-7, 4.002e-7, 1.146e-6, 4.859e-7))])
def test_fp32_errors_against_64_bits(form, S, D, bounds):
    q, k, v, f, i, dh, o = O.make_inputs(1, 4, S, D, torch.float32, seed=S + D, f_mean=3.0, with_o=True)
    if form == "scan":
        ts = [t.cuda().requires_grad_(True) for t in (q, k, v, f, i, o)]
        out = ms.mlstm_scan(*ts)
        want = [O.mlstm_scan_dense(q, k, v, f, i, o), *O.mlstm_gated_backward_dense(dh, q, k, v, f, i, o, zero_first_df=True)]
    else:
        ts = [t.cuda().requires_grad_(True) for t in (q, k, v, f, i)]
        out = mm.Triton_mLSTM.apply(*ts)
        want = [O.mlstm_forward_dense(q, k, v, f, i)[0], *O.mlstm_backward_dense(dh, q, k, v, f, i, zero_first_df=True)]
    got = [out.detach(), *torch.autograd.grad(out, ts, dh.cuda())]
    errors = [float(((g.double().cpu() - w.double()).norm(dim=-1) / w.double().norm(dim=-1)).median()) for g, w in zip(got[:4], want[:4])]
    assert all(e <= 1.01 * bound for e, bound in zip(errors, bounds)), (errors, bounds)   # (1.01: the bounds' own digits, and D = 256, level)


# A product of three-term operands keeps fp32's range and precision over magnitudes.
@pytest.mark.parametrize("scale", [1e-30, 1e-12, 1.0, 1e12, 1e30])
def test_fp32_terms_over_magnitudes(scale):
    q, k, v, f, i, _ = O.make_inputs(1, 1, 400, 64, torch.float32, seed=5, f_mean=3.0)
    h, _, _ = O.mlstm_forward_dense(q, k, v * scale, f, i)
    got = mm.mlstm_matmul(q.cuda(), k.cuda(), (v * scale).cuda(), f.cuda(), i.cuda())
    assert_close(got / scale, h / scale, torch.float32, "h")


# An infinite operand makes infinite what it makes infinite in fp32 products, and nothing else: 150 of 200 is in a sequence that
# is not cut, 150 of 400 in a chunk of 128 to 255 (the tile kernels take what lies before a row's chunk from a state, whose infinities
# a row's products with it may turn into NaN, as they always could), 399 the last position.
@pytest.mark.parametrize("value", [float("inf"), float("-inf")])
@pytest.mark.parametrize("S,at", [(200, 150), (400, 150), (400, 399)])
@pytest.mark.parametrize("D", [64, 128, 256])
def test_fp32_terms_keep_what_is_not_finite(D, S, at, value):
    q, k, v, f, i, dh = O.make_inputs(1, 1, S, D, torch.float32, seed=6, f_mean=3.0)
    h, _, b = O.mlstm_forward_dense(q, k, v, f, i)
    v[0, 0, at, 7] = value
    got = mm.mlstm_matmul(q.cuda(), k.cuda(), v.cuda(), f.cuda(), i.cuda()).cpu()
    keep = [d for d in range(D) if d != 7]
    assert_close(got[..., keep], h[..., keep], torch.float32, "the other columns")
    if at > 0:
        assert_close(got[0, 0, :at], h[0, 0, :at], torch.float32, "the rows before")
    own = min(S, (at // 128 + 1) * 128 if S > 320 and D <= 128 else S)
    assert bool(torch.isinf(got[0, 0, at:own, 7]).all()) and not bool(torch.isfinite(got[0, 0, at:, 7]).any())
    # in the output gradient: dV's column, for the keys up to that position; every other column is as if it were not there
    v[0, 0, at, 7] = 0
    dh[0, 0, at, 7] = value
    ts = [t.cuda().requires_grad_(True) for t in (q, k, v, f, i)]
    grads = torch.autograd.grad(mm.Triton_mLSTM.apply(*ts), ts, dh.cuda())
    dh[0, 0, at, 7] = 0
    want = O.mlstm_backward_dense(dh, q, k, v, f, i, zero_first_df=True)
    assert_close(grads[2][..., keep], want[2][..., keep], torch.float32, "dv, the other columns")
    if at + 1 < S:
        assert_close(grads[2][0, 0, at + 1:], want[2][0, 0, at + 1:], torch.float32, "dv, the keys behind")
    first = at // 128 * 128 if S > 320 and D <= 128 else 0
    assert bool(torch.isinf(grads[2][0, 0, first:at + 1, 7]).all())
    rows = [t for t in range(S) if t != at]
    assert_close(grads[0][0, 0, rows], want[0][0, 0, rows], torch.float32, "dq, the other rows")


# The lowest value of the type, as masks use it: it rounds to an infinite bf16.  As a value behind every row that is looked at it
# changes nothing, not a bit.
@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("S", [130, 200, 400])
def test_fp32_terms_and_the_lowest_value(S, D):
    q, k, v, f, i, _ = (t.cuda() for t in O.make_inputs(1, 2, S, D, torch.float32, seed=9, f_mean=3.0))
    o = torch.randn(q.shape, generator=torch.Generator().manual_seed(S)).cuda()
    for tail in (0.0, torch.finfo(torch.float32).min):
        v[..., -3:, :] = tail
        k[..., -1:, :] = tail
        out = [mm.mlstm_matmul(q, k, v, f, i)[..., :-3, :], ms.mlstm_scan(q, k, v, f, i, o)[..., :-3, :]]
        if tail == 0.0:
            want = out
    for a, w in zip(out, want):
        assert bool(torch.isfinite(w).all())
        assert_close(a, w, torch.float32, "the rows before")   # (a tile that had to be formed again: in another order)


# One element of one key that rounds to an infinite bf16, where every query has a zero: scores, outputs and gradients are what
# they are without it.  Every product with it goes wrong in terms, so all rows and keys that see it are formed again: forward, dQ, dK,
# dV, dF and dI of those paths against the oracle, in the first chunk, behind it, and without chunks.
@pytest.mark.parametrize("B,NH,S,D,at", [(1, 2, 200, 64, 0), (1, 1, 63, 64, 40), (1, 2, 400, 64, 3), (2, 1, 450, 64, 300), (1, 2, 200, 128, 100),
                                         (1, 2, 450, 128, 3), (1, 1, 450, 128, 449), (1, 2, 200, 256, 3), (1, 16, 70, 512, 10)])
def test_fp32_rows_and_keys_formed_again(B, NH, S, D, at):
    q, k, v, f, i, dh = O.make_inputs(B, NH, S, D, torch.float32, seed=S + at, f_mean=3.0)
    q[..., 7] = 0
    k[..., at, 7] = 0
    dh *= 1e-3   # (so that what the element itself contributes, to column 7 of dQ, stays finite)
    want = [O.mlstm_forward_dense(q, k, v, f, i)[0], *O.mlstm_backward_dense(dh, q, k, v, f, i, zero_first_df=True)]
    k[..., at, 7] = 3.4e38
    ts = [t.cuda().requires_grad_(True) for t in (q, k, v, f, i)]
    out = mm.Triton_mLSTM.apply(*ts)
    got = [out.detach(), *torch.autograd.grad(out, ts, dh.cuda())]
    keep = [d for d in range(D) if d != 7]
    got[1], want[1] = got[1][..., keep], want[1][..., keep]
    for name, g, w in zip(("h", "dq", "dk", "dv", "df", "di"), got, want):
        assert_close(g, w, torch.float32, name)
    o = torch.randn(q.shape, generator=torch.Generator().manual_seed(S)).cuda()
    assert_close(ms.mlstm_scan(*(t.detach() for t in ts), o), want[0] * (o * torch.sigmoid(o)).cpu().double(), torch.float32, "scan form")
