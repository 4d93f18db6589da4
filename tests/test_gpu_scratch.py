"""What scratch memory holds before a call must not show in its results.  Workspaces and kept buffers come from torch's caching
allocator with whatever their last owner left; here that is zeros in one run and NaN in the other, and the results have to be
the same bits.  Ragged lengths: the last granule of 64 positions then has rows that no position stands for."""
import pytest
import torch

from _mlstm_pkg import submodule

pytestmark = pytest.mark.gpu
ffi, mm, ms, sl = submodule("_ffi"), submodule("mlstm_matmul"), submodule("mlstm_scan"), submodule("slstm")

OPS = {"matmul": lambda *t: mm.Triton_mLSTM.apply(*t), "precise": lambda *t: mm.Triton_mLSTM_precise.apply(*t),
       "gated": lambda *t: mm.Triton_mLSTM_gated.apply(*t), "scan": ms.mlstm_scan, "slstm": lambda *t: sl.slstm(*t, True)}


def _leave_behind(value):
    """Free blocks of the caching allocator, small and large, filled with `value`."""
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    blocks = [torch.full((1 << 17,), value, device="cuda") for _ in range(64)] + [torch.full((1 << 24,), value, device="cuda") for _ in range(6)]
    torch.cuda.synchronize()
    del blocks


def _inputs(op, BH, S, D, dtype):
    g = torch.Generator(device="cuda").manual_seed(S + D)
    rnd = lambda *s: torch.randn(s, device="cuda", generator=g)  # noqa: E731
    if op == "slstm":
        return [rnd(BH, S, 4, 2, D), rnd(2, 4, D, D) / D ** 0.5, rnd(2, 4, D)], rnd(BH, S, 2, D)
    ins = [rnd(1, BH, S, D).to(dtype) for _ in range(3)] + [(rnd(1, BH, S) + 3).to(dtype), rnd(1, BH, S).to(dtype)]
    return ins + ([rnd(1, BH, S, D).to(dtype)] if op in ("gated", "scan") else []), rnd(1, BH, S, D).to(dtype)


def _same_on_both(run):
    results = []
    for value in (0.0, float("nan")):
        _leave_behind(value)
        results.append([t.clone() for t in run()])
    for n, (a, b) in enumerate(zip(*results)):
        assert bool(torch.isfinite(a).all()) and torch.equal(a, b), n


def _step(op, ins, dh):
    ts = [t.detach().requires_grad_(True) for t in ins]
    out = OPS[op](*ts)
    return [out.detach(), *torch.autograd.grad(out, ts, dh)]


CASES = [(op, dt, 3, S, D) for op in ("matmul", "precise", "gated") for dt in (torch.bfloat16, torch.float16) for S, D in
         ((70, 64), (1100, 64), (100, 128), (1130, 128), (65, 256), (1090, 256))] + \
        [(op, torch.float32, 3, S, D) for op in ("matmul", "gated", "scan") for S, D in ((200, 64), (500, 64), (65, 128), (500, 128))] + \
        [(op, torch.float32, 3, S, D) for op in ("matmul", "scan") for S, D in ((130, 256), (70, 512), (130, 1024))] + \
        [("scan", torch.float32, 1, 1100, 256), ("slstm", torch.float32, 2, 33, 32), ("slstm", torch.float32, 2, 70, 128)]


@pytest.mark.parametrize("op,dtype,BH,S,D", CASES)
def test_results_do_not_depend_on_what_scratch_memory_held(op, dtype, BH, S, D):
    ins, dh = _inputs(op, BH, S, D, dtype)
    _same_on_both(lambda: _step(op, ins, dh))


# the other kernels behind the same entry points: the column kernels, the generic ones, the one-pass states
@pytest.mark.parametrize("setting", ["col16", "col", "generic", "one_pass"])
@pytest.mark.parametrize("S,D", [(100, 128), (1130, 128), (1090, 256)])
def test_the_same_for_the_kernels_behind_the_switches(setting, S, D):
    ins, dh = _inputs("matmul", 3, S, D, torch.bfloat16)
    try:
        if setting == "generic":
            ffi.force_generic_kernels(True)
        elif setting == "one_pass":
            ffi.set_state_kernel(2)
        else:
            ffi.set_column_kernel(1 if setting == "col16" else 3)
        _same_on_both(lambda: _step("matmul", ins, dh))
    finally:
        ffi.force_generic_kernels(False)
        ffi.set_state_kernel(0)
        ffi.set_column_kernel(0)


# backward passes that form the forward again themselves
@pytest.mark.parametrize("dtype,S,D", [(torch.bfloat16, 1130, 128), (torch.float16, 100, 256), (torch.float32, 500, 64), (torch.float32, 130, 256)])
def test_the_same_for_backward_passes_without_the_forward_s_outputs(dtype, S, D):
    ins, dh = _inputs("matmul", 2, S, D, dtype)
    _same_on_both(lambda: mm.mlstm_backward_hip(dh, *ins))
    ins, dh = _inputs("scan", 2, S, D, torch.float32)
    _same_on_both(lambda: ms.mlstm_scan_backward_hip(dh, *ins))
