"""Parity of the sLSTM kernels against the CPU oracle (oracle/slstm_oracle.py), fp32 bound of tests/helpers.py."""
import pytest
import torch

from oracle import slstm_oracle as SO
from tests.helpers import assert_close

pytestmark = pytest.mark.gpu


def gpu(*xs):
    return [x.cuda() for x in xs]


@pytest.mark.parametrize("forget_sigmoid", [False, True])
@pytest.mark.parametrize("B,NH,S,DH", [(1, 1, 1, 32), (2, 2, 17, 32), (2, 3, 130, 64), (1, 2, 96, 128)])
def test_forward_and_backward_against_oracle(B, NH, S, DH, forget_sigmoid):
    from slstm import slstm_backward_hip, slstm_forward_hip
    wx, r, b, dh = SO.make_inputs(B, NH, S, DH, seed=B + S + DH)
    h, saved = slstm_forward_hip(*gpu(wx, r, b), forget_sigmoid=forget_sigmoid)
    assert_close(h, SO.slstm_forward(wx, r, b, forget_sigmoid), torch.float32, "h")
    dwx, dr, db = slstm_backward_hip(dh.cuda(), h, r.cuda(), saved, forget_sigmoid=forget_sigmoid)
    rwx, rr, rb = SO.slstm_backward(dh, wx, r, b, forget_sigmoid)
    assert_close(dwx, rwx, torch.float32, "dwx")
    assert_close(dr, rr, torch.float32, "dr")
    assert_close(db, rb, torch.float32, "db")


@pytest.mark.parametrize("B,NH,S,DH", [(1, 1, 7, 32), (1, 2, 8, 64), (2, 1, 9, 128), (1, 1, 16, 32), (3, 2, 23, 64)])
def test_sequences_around_the_prefetch_depth(B, NH, S, DH):
    # the kernels keep eight steps of inputs under way: sequences shorter than, equal to and just past that depth
    from slstm import slstm_backward_hip, slstm_forward_hip
    wx, r, b, dh = SO.make_inputs(B, NH, S, DH, seed=100 + S)
    want = SO.slstm_forward(wx, r, b, True)
    h, saved = slstm_forward_hip(*gpu(wx, r, b), forget_sigmoid=True)
    assert_close(h, want, torch.float32, "h")
    h_only, none = slstm_forward_hip(*gpu(wx, r, b), forget_sigmoid=True, save=False)
    assert none is None and torch.equal(h_only, h)      # the variant that keeps nothing for a backward: the same bits
    got = slstm_backward_hip(dh.cuda(), h, r.cuda(), saved, forget_sigmoid=True)
    for name, g, w in zip(("dwx", "dr", "db"), got, SO.slstm_backward(dh, wx, r, b, True)):
        assert_close(g, w, torch.float32, name)


@pytest.mark.parametrize("DH", [32, 64, 128])
def test_recurrent_gradient_of_what_is_not_finite(DH):
    # one gradient of one step infinite, or beyond what rounds to a finite bf16, on the way into dR: the sums it enters are
    # infinite or huge, as products in fp32 make them, and not NaN; every other element is as if it were not there
    from slstm import slstm_backward_hip, slstm_forward_hip
    wx, r, b, dh = SO.make_inputs(2, 2, 40, DH, seed=DH)
    h, saved = slstm_forward_hip(*gpu(wx, r, b), forget_sigmoid=True)
    clean = slstm_backward_hip(dh.cuda(), h, r.cuda(), saved, forget_sigmoid=True)
    bad = dh.cuda()
    bad[1, 0, 1, 5] = float("inf")    # (the first step of a sequence: its own gradients are not finite, nothing before it is)
    dwx, dr, db = slstm_backward_hip(bad, h, r.cuda(), saved, forget_sigmoid=True)
    for g, w in zip((dwx, dr, db), clean):
        part = lambda t: t[:, :, :, 0] if t.dim() == 5 else t[0]  # noqa: E731  (head 0)
        assert torch.equal(part(g), part(w))
    assert_close(dr[1], clean[1][1], torch.float32, "dr")   # (h before the first step is zero: it adds nothing to dR)
    assert not bool(torch.isfinite(dwx[1, 0, :, 1, 5]).all()) and not bool(torch.isfinite(db[1]).all())
    # infinite at a later step: the rows of dR it enters are infinite with the sign of h, or NaN where its gradients are NaN
    bad = dh.cuda()
    bad[1, 39, 1, 5] = float("inf")
    dwx, dr, _ = slstm_backward_hip(bad, h, r.cuda(), saved, forget_sigmoid=True)
    last = dwx[1, 39, :, 1, 5]   # [gate]
    for g in range(4):
        if bool(torch.isinf(last[g])) and bool(torch.isfinite(dwx[1, :39, g, 1, 5]).all()):
            assert torch.equal(dr[1, g, 5], torch.sign(last[g]) * torch.sign(h[1, 38, 1]) * float("inf"))


def test_benchmark_shape_twice():
    # B16 NH4 S2048 DH64: two runs give the same bits (nothing depends on when a load lands), and match the oracle
    # (dR and db at a long sequence: test_long_sequence_and_many_heads)
    from slstm import slstm_backward_hip, slstm_forward_hip
    wx, r, b, dh = SO.make_inputs(16, 4, 2048, 64, seed=11, f_mean=2.0)
    dev = gpu(wx, r, b)
    h, saved = slstm_forward_hip(*dev, forget_sigmoid=True)
    got = slstm_backward_hip(dh.cuda(), h, dev[1], saved, forget_sigmoid=True)
    # the second run shares the memory system with a stream of large copies on another (default-priority) stream: the
    # kernels' inputs arrive several steps ahead of their use, later or earlier than before, and nothing may change
    side = torch.cuda.Stream()
    big = torch.empty(64 * 1024 * 1024, device="cuda")
    other = torch.empty_like(big)
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(40):
            other.copy_(big)
    h2, saved2 = slstm_forward_hip(*dev, forget_sigmoid=True)
    got2 = slstm_backward_hip(dh.cuda(), h2, dev[1], saved2, forget_sigmoid=True)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    assert torch.equal(h, h2) and torch.equal(saved, saved2)
    for x, y in zip(got, got2):
        assert torch.equal(x, y)
    # (the oracle on one sequence of the batch: h and dwx of a sequence depend on no other)
    assert_close(h[3:4], SO.slstm_forward(wx[3:4], r, b, True), torch.float32, "h")
    assert_close(got[0][3:4], SO.slstm_backward(dh[3:4], wx[3:4], r, b, True)[0], torch.float32, "dwx")


def test_long_sequence_and_many_heads():
    from slstm import slstm_backward_hip, slstm_forward_hip
    wx, r, b, dh = SO.make_inputs(4, 4, 1024, 64, seed=5, f_mean=1.0)
    h, saved = slstm_forward_hip(*gpu(wx, r, b), forget_sigmoid=True)
    assert_close(h, SO.slstm_forward(wx, r, b, True), torch.float32, "h")
    got = slstm_backward_hip(dh.cuda(), h, r.cuda(), saved, forget_sigmoid=True)
    for name, g, w in zip(("dwx", "dr", "db"), got, SO.slstm_backward(dh, wx, r, b, True)):
        assert_close(g, w, torch.float32, name)


def test_gates_far_from_zero_stay_finite():
    # the stabiliser at work: input gates of e^80, forget gates of e^(+-60) in turn
    from slstm import slstm_forward_hip
    wx, r, b, _ = SO.make_inputs(1, 2, 200, 32, seed=6)
    wx[:, :, 0] += 80.0
    wx[:, ::3, 1] += 60.0
    wx[:, 1::3, 1] -= 60.0
    h, _ = slstm_forward_hip(*gpu(wx, r, b))
    assert bool(torch.isfinite(h).all())
    assert_close(h, SO.slstm_forward(wx, r, b), torch.float32, "h")


@pytest.mark.parametrize("forget_sigmoid", [False, True])
@pytest.mark.parametrize("DH", [32, 64, 128])
def test_a_pre_activation_takes_its_input_last(DH, forget_sigmoid):
    # From the kernel's own h_{t-1}, so that only one step's roundings are left.  A rounding at the size of x has the variance ulp(x)^2 / 12.  There is one of
    # wx + b and one of the whole sum; the recurrent sum, eight chains of DH / 8 multiply-adds and three levels of adds, has at most DH / 8 + 3 on the way of each of
    # its terms, at the size of what it adds up alone.  With the input ahead of the recurrent sum, those are at the size of the whole: 1.8 (DH = 32) to 2.6 (128)
    # times the root mean square that this predicts, where the input last is at 0.9 (both orders on the CPU).
    from slstm import slstm_forward_hip
    B, NH, S = 4, 2, 200
    wx, r, b, _ = (x.double() for x in SO.make_inputs(B, NH, S, DH, seed=DH))
    h, saved = slstm_forward_hip(*gpu(wx.float(), r.float(), b.float()), forget_sigmoid=forget_sigmoid)
    before = torch.cat([torch.zeros(B, 1, NH, DH).double(), h[:, :-1].double().cpu()], 1)
    recurrent = lambda m, v: torch.matmul(m, v.unsqueeze(3).unsqueeze(-1)).squeeze(-1).transpose(2, 3)  # noqa: E731  [B,S,4,NH,DH]
    given = wx + b.transpose(0, 1)
    want = given + recurrent(r, before)
    ulp = lambda x: 2.0 ** (x.abs().clamp_min(1e-30).log2().floor() - 23)  # noqa: E731
    variance = (ulp(given) ** 2 + ulp(want) ** 2 + (DH / 8 + 3) * 2.0 ** -46 * recurrent(r ** 2, before ** 2)) / 12
    kept = saved.view(torch.float32).view(B, S, 7, NH, DH)
    for gate in (0,) if forget_sigmoid else (0, 1):   # what is kept of the other gates has been through their nonlinearity
        error = kept[:, :, gate].double().cpu() - want[:, :, gate]
        assert error.square().mean() <= 1.25 ** 2 * variance[:, :, gate].mean(), (gate, error.square().mean().sqrt(), variance[:, :, gate].mean().sqrt())


def test_autograd_function_and_repeatability():
    from slstm import slstm
    wx, r, b, dh = SO.make_inputs(2, 2, 64, 64, seed=7)
    leaves = [x.cuda().requires_grad_(True) for x in (wx, r, b)]
    h = slstm(*leaves)
    h.backward(dh.cuda())
    for name, x, w in zip(("dwx", "dr", "db"), leaves, SO.slstm_backward(dh, wx, r, b)):
        assert_close(x.grad, w, torch.float32, name)
    again = [x.detach().clone().requires_grad_(True) for x in leaves]
    slstm(*again).backward(dh.cuda())
    for x, y in zip(leaves, again):
        assert torch.equal(x.grad, y.grad)          # the slices of dR and db are added in a fixed order
    with torch.no_grad():
        assert torch.equal(slstm(*leaves), h)


def test_rejects_what_it_cannot_serve():
    from slstm import slstm_forward_hip
    wx, r, b, _ = SO.make_inputs(1, 1, 8, 48, seed=1)
    with pytest.raises(ValueError):
        slstm_forward_hip(*gpu(wx, r, b))
    wx, r, b, _ = SO.make_inputs(1, 1, 8, 32, seed=1)
    with pytest.raises(TypeError):
        slstm_forward_hip(wx.cuda().half(), r.cuda(), b.cuda())
    with pytest.raises(ValueError):
        slstm_forward_hip(wx.cuda(), r.cuda()[:, :3], b.cuda())


@pytest.mark.parametrize("forget_sigmoid", [False, True])
@pytest.mark.parametrize("B,NH,S,DH", [(1, 1, 2, 64), (1, 2, 3, 128), (2, 1, 5, 32), (1, 1, 6, 64), (1, 3, 10, 128), (2, 1, 15, 64)])
def test_short_sequences_of_every_prologue_length(B, NH, S, DH, forget_sigmoid):
    # a step's stores and loads are issued by its successor and the backward takes values two steps ahead: the first and last steps
    from slstm import slstm_backward_hip, slstm_forward_hip
    wx, r, b, dh = SO.make_inputs(B, NH, S, DH, seed=40 + S, f_mean=0.0)
    h, saved = slstm_forward_hip(*gpu(wx, r, b), forget_sigmoid=forget_sigmoid)
    assert_close(h, SO.slstm_forward(wx, r, b, forget_sigmoid), torch.float32, "h")
    assert torch.equal(slstm_forward_hip(*gpu(wx, r, b), forget_sigmoid=forget_sigmoid, save=False)[0], h)
    got = slstm_backward_hip(dh.cuda(), h, r.cuda(), saved, forget_sigmoid=forget_sigmoid)
    for name, g, w in zip(("dwx", "dr", "db"), got, SO.slstm_backward(dh, wx, r, b, forget_sigmoid)):
        assert_close(g, w, torch.float32, name)


@pytest.mark.parametrize("DH", [32, 64, 128])
@pytest.mark.parametrize("S", [1, 2, 3, 4, 5, 6, 7, 8, 9, 16, 17, 18, 19, 21])
def test_backward_at_every_turn_of_the_helpers(S, DH):
    # The waves beside a step's own serve every second or fourth step and keep four of these under way: sequences that end at each
    # of their intervals.  A saved state off a 16-byte boundary is loaded a float a lane: the same values, so the same bits.
    from slstm import slstm_backward_hip, slstm_forward_hip
    B, NH = 2, 3
    wx, r, b, dh = SO.make_inputs(B, NH, S, DH, seed=70 + S, f_mean=0.5)
    h, saved = slstm_forward_hip(*gpu(wx, r, b), forget_sigmoid=True)
    got = slstm_backward_hip(dh.cuda(), h, r.cuda(), saved, forget_sigmoid=True)
    for name, g, w in zip(("dwx", "dr", "db"), got, SO.slstm_backward(dh, wx, r, b, True)):
        assert_close(g, w, torch.float32, name)
    for off in (1, 2):
        def away(x):
            skip = 4 * off // x.element_size()
            return torch.empty(x.numel() + skip, dtype=x.dtype, device="cuda")[skip:].view(x.shape).copy_(x)
        for g, w in zip(slstm_backward_hip(away(dh), h, r.cuda(), away(saved), forget_sigmoid=True), got):
            assert torch.equal(g, w)


@pytest.mark.parametrize("DH", [32, 64, 128])
@pytest.mark.parametrize("S", [1, 2, 3, 7, 8, 9, 10, 11, 17, 26])
def test_forward_at_every_turn_of_the_helpers(S, DH):
    # Waves beside the walk bring its inputs and write out what it keeps, a step and two behind it: sequences that end around the turns of the
    # ring.  Inputs off a 16-byte boundary go a float a lane: the same values, so the same bits.
    from slstm import slstm_forward_hip
    wx, r, b, _ = SO.make_inputs(3, 2, S, DH, seed=90 + S, f_mean=0.5)
    h, saved = slstm_forward_hip(*gpu(wx, r, b), forget_sigmoid=True)
    assert_close(h, SO.slstm_forward(wx, r, b, True), torch.float32, "h")
    flat = torch.empty(wx.numel() + 3, device="cuda")
    for off in (1, 3):
        other = flat[off:off + wx.numel()].view(wx.shape).copy_(wx)
        h2, saved2 = slstm_forward_hip(other, r.cuda(), b.cuda(), forget_sigmoid=True)
        h3, _ = slstm_forward_hip(other, r.cuda(), b.cuda(), forget_sigmoid=True, save=False)
        assert torch.equal(h2, h) and torch.equal(saved2, saved) and torch.equal(h3, h)


@pytest.mark.parametrize("DH", [32, 64, 128])
@pytest.mark.parametrize("B,NH,S", [(40, 2, 15), (21, 1, 16), (18, 3, 17), (5, 4, 333), (2, 1, 1000)])
def test_recurrent_gradients_over_slices(B, NH, S, DH):
    # dR and db from dWx and h, sixteen pairs of (sequence, step) at a time: rounds inside a sequence, across the start of one, at the end of a
    # slice, sequences shorter than a round.  Products of three bf16 terms keep 24 bits, sums are fp32 over at most B S terms in chains of 1/8 of a slice.
    from slstm import slstm_backward_hip, slstm_forward_hip
    wx, r, b, dh = SO.make_inputs(B, NH, S, DH, seed=B + DH, f_mean=1.0)
    h, saved = slstm_forward_hip(*gpu(wx, r, b), forget_sigmoid=True)
    dwx, dr, db = slstm_backward_hip(dh.cuda(), h, r.cuda(), saved, forget_sigmoid=True)
    d, prev = dwx.double().cpu(), torch.nn.functional.pad(h.double().cpu(), (0, 0, 0, 0, 1, 0))[:, :-1]
    d2, p2 = d.permute(3, 2, 4, 0, 1).reshape(NH, 4, DH, B * S), prev.permute(2, 3, 0, 1).reshape(NH, 1, DH, B * S)
    size = d2.abs() @ p2.abs().transpose(-1, -2).contiguous()
    bound = 2.0 ** -24 * (B * S) ** 0.5 * 4
    assert bool(((dr.double().cpu() - d2 @ p2.transpose(-1, -2).contiguous()).abs() <= bound * size + 1e-30).all())
    assert bool(((db.double().cpu() - d2.sum(-1)).abs() <= bound * d2.abs().sum(-1) + 1e-30).all())


@pytest.mark.parametrize("DH", [32, 64, 128])
def test_forward_of_a_full_grid_off_a_16_byte_boundary(DH):
    # Thousands of steps in every workgroup, inputs that no cache holds: a step that took its input from the ring before it was there would take that of
    # eight steps before.
    from slstm import slstm_forward_hip
    B, NH, S = 16, 4, 2048
    g = torch.Generator(device="cuda").manual_seed(DH)
    wx = torch.randn(B, S, 4, NH, DH, device="cuda", generator=g)
    r, b = torch.randn(NH, 4, DH, DH, device="cuda", generator=g) / DH ** 0.5, torch.randn(NH, 4, DH, device="cuda", generator=g)
    h, saved = slstm_forward_hip(wx, r, b, forget_sigmoid=True)
    assert bool(torch.isfinite(h).all())
    for off in (1, 2, 3):
        other = torch.empty(wx.numel() + off, device="cuda")[off:].view(wx.shape).copy_(wx)
        h2, saved2 = slstm_forward_hip(other, r, b, forget_sigmoid=True)
        h3, _ = slstm_forward_hip(other, r, b, forget_sigmoid=True, save=False)
        assert torch.equal(h2, h) and torch.equal(saved2, saved) and torch.equal(h3, h)


def test_a_batch_of_more_threads_than_a_launch_holds():
    # 22.5 million sequences of one step: beyond 2^32 threads of either step kernel, whose batches then take several launches
    from slstm import slstm_backward_hip, slstm_forward_hip
    B, DH = 22_500_000, 32
    if torch.cuda.mem_get_info()[0] < 60e9:
        pytest.skip("needs 60 GB of GPU memory")
    g = torch.Generator(device="cuda").manual_seed(1)
    wx = torch.empty(B, 1, 4, 1, DH, device="cuda").normal_(generator=g)
    r, b = torch.randn(1, 4, DH, DH, device="cuda", generator=g) / DH ** 0.5, torch.randn(1, 4, DH, device="cuda", generator=g)
    dh = torch.empty(B, 1, 1, DH, device="cuda").normal_(generator=g)
    h, saved = slstm_forward_hip(wx, r, b, forget_sigmoid=True)
    dwx, dr, db = slstm_backward_hip(dh, h, r, saved, forget_sigmoid=True)
    del saved
    some = torch.tensor([0, 1, *[n * 2 ** 32 // threads + k for n, threads in ((1, 192), (1, 384), (2, 384)) for k in (-2, -1, 0, 1)], B - 1], device="cuda")
    h1, saved1 = slstm_forward_hip(wx[some], r, b, forget_sigmoid=True)
    assert torch.equal(h[some], h1) and bool(torch.isfinite(h1).all())
    assert torch.equal(dwx[some], slstm_backward_hip(dh[some], h1, r, saved1, forget_sigmoid=True)[0])
    assert not bool(dr.any())   # (h before the first step is zero)
    want = torch.stack([dwx[:, 0, x, 0].double().sum(0) for x in range(4)])
    # (fp32 sums over 128 slices of 176 thousand terms each, in chains of an eighth of a slice)
    size = torch.stack([dwx[:, 0, x, 0].abs().double().sum(0) for x in range(4)])
    assert bool(((db[0].double() - want).abs() <= 2.0 ** -24 * 22000 ** 0.5 * 4 * size).all())
    del wx, dh, h, dwx
    torch.cuda.empty_cache()


@pytest.mark.parametrize("NH", [260_000, 300_000])
def test_recurrent_gradients_of_more_heads_than_a_launch_holds(NH):
    # a workgroup per 64 elements: dR and db of 260 000 heads of 32 units are 2^32 threads together, of 300 000 dR is by itself
    from slstm import slstm_backward_hip, slstm_forward_hip
    S, DH = 2, 32
    if torch.cuda.mem_get_info()[0] < 20e9:
        pytest.skip("needs 20 GB of GPU memory")
    g = torch.Generator(device="cuda").manual_seed(2)
    wx, dh = torch.randn(1, S, 4, NH, DH, device="cuda", generator=g), torch.randn(1, S, NH, DH, device="cuda", generator=g)
    r, b = torch.randn(NH, 4, DH, DH, device="cuda", generator=g).mul_(DH ** -0.5), torch.randn(NH, 4, DH, device="cuda", generator=g)
    h, saved = slstm_forward_hip(wx, r, b, forget_sigmoid=True)
    dwx, dr, db = slstm_backward_hip(dh, h, r, saved, forget_sigmoid=True)
    for lo in (0, NH // 2, NH - 3):   # (a few heads by themselves: the same bits)
        few = slice(lo, lo + 3)
        h1, saved1 = slstm_forward_hip(wx[:, :, :, few].contiguous(), r[few].contiguous(), b[few].contiguous(), forget_sigmoid=True)
        got = slstm_backward_hip(dh[:, :, few].contiguous(), h1, r[few].contiguous(), saved1, forget_sigmoid=True)
        for x, y in zip(got, (dwx[:, :, :, few], dr[few], db[few])):
            assert torch.equal(x, y)
    del wx, dh, r, dwx, dr, saved
    torch.cuda.empty_cache()
