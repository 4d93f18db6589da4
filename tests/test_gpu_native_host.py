"""The native host path (csrc/mlstm_torch.cpp) where an autograd function is passed by: saved-tensor hooks, checkpointing,
forward-mode tangents, function transforms, derived classes, in-place changes, unaligned views.  What is compared is the same
kernels on the same values, so results are the same bits unless noted."""
import pytest
import torch
from torch.utils.checkpoint import checkpoint

from _mlstm_pkg import submodule

pytestmark = pytest.mark.gpu
mm, ms, sl = submodule("mlstm_matmul"), submodule("mlstm_scan"), submodule("slstm")


def _inputs(op, S=100):
    g = torch.Generator(device="cuda").manual_seed(7)
    rnd = lambda *s: torch.randn(s, device="cuda", generator=g)  # noqa: E731
    if op == "slstm":
        return [rnd(2, S, 4, 2, 32), rnd(2, 4, 32, 32) / 6, rnd(2, 4, 32)]
    D, dt = {"scan": (64, torch.float32), "scan_wide": (256, torch.float32)}.get(op, (64, torch.bfloat16))
    ins = [rnd(1, 2, S, D).to(dt) for _ in range(3)] + [(rnd(1, 2, S) + 2).to(dt), rnd(1, 2, S).to(dt)]
    return ins + [rnd(1, 2, S, D).to(dt)] if op in ("gated", "scan", "scan_wide") else ins


OPS = {"matmul": lambda *t: mm.Triton_mLSTM.apply(*t), "precise": lambda *t: mm.Triton_mLSTM_precise.apply(*t),
       "gated": lambda *t: mm.Triton_mLSTM_gated.apply(*t), "scan": ms.mlstm_scan, "scan_wide": ms.mlstm_scan,
       "slstm": lambda *t: sl.slstm(*t, True)}


def _step(op, ins, context=None):
    ts = [t.clone().requires_grad_(True) for t in ins]
    if context is None:
        out = OPS[op](*ts)
    else:
        with context:
            out = OPS[op](*ts)
    g = torch.Generator(device="cuda").manual_seed(9)
    dh = torch.randn(out.shape, device="cuda", generator=g).to(out.dtype)
    return [out.detach(), *torch.autograd.grad(out, ts, dh)]


def _same(got, want):
    for n, (a, b) in enumerate(zip(got, want)):
        assert torch.equal(a, b), n


def _other_layout(t):
    return t.transpose(0, -1).contiguous().transpose(0, -1) if t.dim() > 1 else t.clone()


@pytest.mark.parametrize("op", list(OPS))
def test_saved_tensor_hooks_see_everything_the_backward_reads(op):
    ins = _inputs(op, S=1100 if op in ("matmul", "gated") else 100)   # (1100: in chunks, with saved states)
    want = _step(op, ins)
    moved = []

    def pack(t):
        moved.append(t.numel() * t.element_size())
        return t.cpu()
    _same(_step(op, ins, torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t.cuda())), want)
    _same(_step(op, ins, torch.autograd.graph.saved_tensors_hooks(lambda t: t, _other_layout)), want)
    assert len(moved) >= len(ins[:1]) + 2
    # nothing the backward needs stays on the device beside what the hooks moved away: less than one row tensor more in use
    ts = [t.clone().requires_grad_(True) for t in ins]
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t.cpu(), lambda t: t.cuda()):
        out = OPS[op](*ts)
    held = torch.cuda.memory_allocated() - before - out.numel() * out.element_size()
    assert held < 4096, held


@pytest.mark.parametrize("op", list(OPS))
def test_hooks_that_change_a_saved_tensor_are_an_error(op):
    ts = [t.clone().requires_grad_(True) for t in _inputs(op)]
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, lambda t: t[..., :1].contiguous() if t.dim() > 1 else t):
        out = OPS[op](*ts)
    with pytest.raises(RuntimeError, match="saved for the backward"):
        out.backward(torch.ones_like(out))


@pytest.mark.parametrize("op", list(OPS))
def test_checkpointed_call(op):
    ins = _inputs(op)
    ts = [t.clone().requires_grad_(True) for t in ins]
    out = checkpoint(OPS[op], *ts, use_reentrant=False)
    g = torch.Generator(device="cuda").manual_seed(9)
    dh = torch.randn(out.shape, device="cuda", generator=g).to(out.dtype)
    _same([out.detach(), *torch.autograd.grad(out, ts, dh)], _step(op, ins))


@pytest.mark.parametrize("op", ["matmul", "precise", "gated"])
def test_forward_mode_and_function_transforms_are_refused_as_by_the_autograd_function(op):
    ins = _inputs(op)
    with torch.autograd.forward_ad.dual_level():
        dual = torch.autograd.forward_ad.make_dual(ins[0], torch.ones_like(ins[0]))
        with pytest.raises((RuntimeError, NotImplementedError)):
            OPS[op](dual, *ins[1:])
    with pytest.raises(RuntimeError):
        torch.func.grad(lambda q: OPS[op](q, *ins[1:]).float().sum())(ins[0])


def test_derived_class_runs_its_own_forward():
    class Doubled(mm.Triton_mLSTM):
        @staticmethod
        def forward(ctx, q, k, v, f, i, SB=16, num_warps=8, gate_form="raw"):
            return 2 * mm.Triton_mLSTM.forward(ctx, q, k, v, f, i, SB, num_warps, gate_form)
    ins = _inputs("matmul")
    assert torch.equal(Doubled.apply(*ins), 2 * mm.mlstm_matmul(*ins))


@pytest.mark.parametrize("op", list(OPS))
def test_an_input_changed_in_place_is_noticed(op):
    ts = [t.clone().requires_grad_(True) for t in _inputs(op)]
    out = OPS[op](*ts)
    with torch.no_grad():
        ts[1].mul_(2)   # (k; the sLSTM's recurrent matrices)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        out.backward(torch.ones_like(out))


@pytest.mark.parametrize("op", ["scan", "scan_wide"])
@pytest.mark.parametrize("shift", [1, 2])
def test_scan_form_on_views_that_start_off_a_16_byte_boundary(op, shift):
    ins = _inputs(op, S=700)

    def shifted(t):
        buf = torch.empty(t.numel() + shift, device="cuda")
        buf[shift:] = t.flatten()
        return buf[shift:].view(t.shape)
    views = [shifted(t) for t in ins]
    _same(_step(op, ins)[:1], [ms.mlstm_scan(*views)])
    want = _step(op, ins)
    ts = [t.requires_grad_(True) for t in views]
    out = ms.mlstm_scan(*ts)
    g = torch.Generator(device="cuda").manual_seed(9)
    dh = shifted(torch.randn(out.shape, device="cuda", generator=g))
    _same([out.detach(), *torch.autograd.grad(out, ts, dh)], want)
    # the entry points below torch, which make the copies themselves
    plain = [t.detach() for t in views]
    h, hu, b = ms.mlstm_scan_forward_save_hip(*plain)
    _same([h, *ms.mlstm_scan_backward_hip(dh, *plain, h_ungated=shifted(hu), b=b)], want)


@pytest.mark.parametrize("op", list(OPS))
def test_the_same_bits_without_it(op, monkeypatch):
    # the wrappers' own calls through ctypes, as where the extension has not been built for the torch at hand
    ffi = submodule("_ffi")
    ins = _inputs(op, S=1100 if op in ("matmul", "gated") else 100)
    want = _step(op, ins)
    monkeypatch.setattr(ffi, "_native", ffi._ServesNothing())
    _same(_step(op, ins), want)
