"""The C-ABI calls with a caller-provided workspace only launch kernels: a HIP graph can capture them."""
import pytest
import torch

from _mlstm_pkg import submodule
from oracle import mlstm_oracle as O

pytestmark = pytest.mark.gpu

ffi = submodule("_ffi")


@pytest.mark.parametrize("D,dtype,S,save", [(128, torch.float16, 320, False), (256, torch.bfloat16, 320, False),
                                            (256, torch.bfloat16, 1100, True), (128, torch.float16, 1100, False)])
def test_forward_backward_in_a_hip_graph(D, dtype, S, save):
    # forward + backward captured once and replayed several times, with eager work and synchronisations between the
    # replays; every replay must reproduce the eager results bit for bit (new inputs are copied into the same buffers)
    L = ffi.lib()
    # (S = 1100 runs in chunks: state kernels in the graph too; `save`: the forward hands its chunk states to the backward)
    B, NH = 1, 2
    dev = torch.device("cuda:0")
    dt = ffi.dtype_code(dtype)
    ws, n = ffi.workspace(ffi.OP_BACKWARD, B, NH, S, D, dt, dev)
    P = ffi.ptr
    bufs = [torch.empty((B, NH, S, D), device=dev, dtype=dtype) for _ in range(4)]                 # q, k, v, dh
    f, i = (torch.empty((B, NH, S), device=dev, dtype=dtype) for _ in range(2))
    h, dq, dk, dv = (torch.empty_like(bufs[0]) for _ in range(4))
    m, b = (torch.empty((B, NH, S), device=dev, dtype=torch.float32) for _ in range(2))
    df, di = torch.empty_like(f), torch.empty_like(i)
    q, k, v, dh = bufs

    nsaved = int(L.mlstm_saved_state_bytes(B, NH, S, D, dt))
    assert (nsaved > 0) == (S >= 1024)
    saved = torch.empty(max(nsaved, 1), dtype=torch.uint8, device=dev)

    def step():
        st = ffi.stream_ptr()
        if save:
            ffi.check_rc(L.mlstm_forward_save_ex(P(q), P(k), P(v), P(f), P(i), P(h), P(m), P(b), P(saved), nsaved, B, NH, S, D, dt, dt,
                                                 P(ws), n, st), "forward")
            ffi.check_rc(L.mlstm_backward_saved_ex(P(dh), P(q), P(k), P(v), P(f), P(i), P(h), P(m), P(b), P(saved), nsaved, P(dq), P(dk),
                                                   P(dv), P(df), P(di), B, NH, S, D, dt, dt, P(ws), n, st), "backward")
            return
        ffi.check_rc(L.mlstm_forward_ex(P(q), P(k), P(v), P(f), P(i), P(h), P(m), P(b), B, NH, S, D, dt, dt, P(ws), n, st), "forward")
        ffi.check_rc(L.mlstm_backward_ex(P(dh), P(q), P(k), P(v), P(f), P(i), P(h), P(m), P(b), P(dq), P(dk), P(dv), P(df), P(di),
                                         B, NH, S, D, dt, dt, P(ws), n, st), "backward")

    def load(seed):
        src = O.make_inputs(B, NH, S, D, dtype, seed=seed, f_mean=2.0)
        for dst, x in zip((q, k, v, f, i, dh), src):
            dst.copy_(x)

    outs = (h, m, b, dq, dk, dv, df, di)
    load(100)
    step()              # (also sets the kernels' attributes, which must not happen during capture)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        with torch.cuda.graph(graph, stream=side):
            step()
    torch.cuda.synchronize()
    for seed in (101, 102, 103):
        load(seed)
        step()
        torch.cuda.synchronize()
        eager = [x.clone() for x in outs]
        for x in outs:
            x.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        for name, e, x in zip(("h", "m", "b", "dq", "dk", "dv", "df", "di"), eager, outs):
            assert torch.equal(e, x), (seed, name)


@pytest.mark.parametrize("BH,S,D", [(16, 130, 512), (2, 130, 1024), (1, 1100, 256)])
def test_scan_kernels_in_a_hip_graph(BH, S, D):
    # fp32 at D >= 256: shared partial numerators (cleared and added to by kernels), segments, rows off a 16-byte boundary; the
    # workspace is the caller's, nothing is allocated on the way
    L, P, F32 = ffi.lib(), ffi.ptr, ffi.F32
    shape = (1, BH, S, D, F32)
    new = lambda: torch.empty(BH * S * D + 1, device="cuda")[1:].view(1, BH, S, D)  # noqa: E731
    q, k, v, dh, h, dq, dk, dv = (new() for _ in range(8))
    f, i, m, b, df, di = (torch.empty((1, BH, S), device="cuda") for _ in range(6))
    ws, n = ffi.workspace(ffi.OP_BACKWARD, *shape, q.device)

    def step():
        st = ffi.stream_ptr()
        ffi.check_rc(L.mlstm_forward_ex(P(q), P(k), P(v), P(f), P(i), P(h), P(m), P(b), *shape, F32, P(ws), n, st), "forward")
        ffi.check_rc(L.mlstm_backward_ex(P(dh), P(q), P(k), P(v), P(f), P(i), P(h), P(m), P(b), P(dq), P(dk), P(dv), P(df), P(di), *shape, F32,
                                         P(ws), n, st), "backward")

    def load(seed):
        for dst, x in zip((q, k, v, f, i, dh), O.make_inputs(1, BH, S, D, torch.float32, seed=seed, f_mean=2.0)):
            dst.copy_(x)
    outs = (h, m, b, dq, dk, dv, df, di)
    load(7)
    step()
    torch.cuda.synchronize()
    graph, side = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    with torch.cuda.stream(side):
        with torch.cuda.graph(graph, stream=side):
            step()
    torch.cuda.synchronize()
    for seed in (8, 9, 10):
        load(seed)
        step()
        torch.cuda.synchronize()
        eager = [x.clone() for x in outs]
        for x in outs:
            x.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        for name, e, x in zip(("h", "m", "b", "dq", "dk", "dv", "df", "di"), eager, outs):
            assert torch.equal(e, x), (seed, name)
