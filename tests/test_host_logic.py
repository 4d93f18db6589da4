"""Host-side logic of the ctypes layer that needs no GPU: layouts of gradient tensors, overlap detection."""
import os
import subprocess

import pytest
import torch

from _mlstm_pkg import submodule

ffi = submodule("_ffi")


def test_expanded_views_are_recognised_as_overlapping():
    B, NH, S, D = 2, 4, 8, 64
    f = torch.zeros(B, 1, S)
    assert ffi.overlaps(f.expand(B, NH, S))                       # gates shared over the heads: stride 0
    q = torch.zeros(1, NH, S, D)
    assert ffi.overlaps(q.expand(B, NH, S, D))
    assert ffi.overlaps(torch.zeros(S + 3).as_strided((2, 3), (2, 1)))   # rows of 3 that start 2 apart
    proj = torch.zeros(B, S, NH, D)
    assert not ffi.overlaps(proj.transpose(1, 2))                 # [B,S,NH,D] activations seen as [B,NH,S,D]
    fused = torch.zeros(B, S, 3, NH, D)
    assert not ffi.overlaps(fused[:, :, 1].transpose(1, 2))       # one slice of a fused q/k/v projection
    assert not ffi.overlaps(torch.zeros(B, NH, S, D))
    assert not ffi.overlaps(torch.zeros(1, 1, S).expand(1, 1, S))  # size-1 dimensions never overlap


def test_overlapping_inputs_are_replaced_by_dense_copies_together():
    B, NH, S = 2, 4, 8
    f = torch.arange(B * S, dtype=torch.float32).reshape(B, 1, S).expand(B, NH, S)
    i = torch.zeros(B, NH, S)
    f2, i2 = ffi.dense_unless_disjoint(f, i)
    assert f2.is_contiguous() and i2.is_contiguous() and torch.equal(f2, f)
    a, b = torch.zeros(B, NH, S), torch.zeros(B, NH, S)
    a2, b2 = ffi.dense_unless_disjoint(a, b)
    assert a2 is a and b2 is b                                     # disjoint tensors pass through untouched


def test_gradient_buffers_of_a_strided_view_keep_its_strides_and_do_not_alias():
    B, NH, S, D = 2, 3, 5, 8
    proj = torch.zeros(B, S, NH, D)
    q = proj.transpose(1, 2)
    dq, dk = ffi.strided_like(q, 2)
    assert dq.stride() == q.stride() and dk.stride() == q.stride() and dq.data_ptr() != dk.data_ptr()
    assert not ffi.overlaps(dq)
    fused = torch.zeros(B, S, 3, NH, D)[:, :, 0].transpose(1, 2)
    g = ffi.strided_like(fused)[0]
    assert g.stride() == fused.stride() and not ffi.overlaps(g)
    g.fill_(1.0)
    assert float(g.sum()) == B * NH * S * D


def test_chunk_length_query_agrees_with_the_buffers_for_any_number_of_heads():
    """mlstm_chunk_length against what the entry points size their buffers for: the states of a head in the buffer a
    forward keeps for its backward (header, matrix and vector states, the gate pre-pass), on both sides of every length the rule
    names and for few and many heads."""
    L = ffi.lib()
    up = lambda n: (n + 255) // 256 * 256  # noqa: E731
    for code, el, dims in ((ffi.F32, 4, (64, 128)), (ffi.BF16, 2, (64, 128, 256)), (ffi.F16, 2, (64, 128, 256))):
        for D in dims:
            for S in (63, 319, 320, 500, 959, 960, 1023, 1024, 1100, 1535, 1536, 2048, 3071, 3072, 9000):
                for BH in (1, 8, 9, 24, 25, 33, 64):
                    length = int(L.mlstm_chunk_length(1, BH, S, D, code))
                    assert length == int(L.mlstm_chunk_length(BH, 1, S, D, code)) == int(L.mlstm_chunk_length(1, 1, S, D, code))
                    assert S < 1024 or length == int(L.mlstm_chunk_length_for(S, D, code))
                    n = (S - 1) // length if length else 0
                    NG = (S + 63) // 64
                    gates = 3 * up(BH * NG * 256) + up(BH * NG * 8) + up((BH * NG * 2 + 64) * 4)
                    want = 256 + up(BH * n * D * D * el) + up(BH * n * D * 4) + gates if n else 0
                    assert int(L.mlstm_saved_state_bytes(1, BH, S, D, code)) == want, (code, D, S, BH, length)


def test_tile_copy_index_arithmetic_stays_inside_the_tiles():
    """tests/harness/tile_bounds (the kernels' own offset functions, compiled for the host): every block of every tile shape
    is fetched exactly once, lands where the LDS readers expect it, and no fetch ends beyond the tile's last row -- for the
    last tile of the last head that is the end of the caller's tensor; the early touch of the dQ pass stays inside its half row."""
    here = os.path.join(os.path.dirname(os.path.abspath(__file__)), "harness")
    exe = os.path.join(here, "tile_bounds")
    if not os.path.exists(exe):
        subprocess.check_call(["make", "-C", here, "tile_bounds"])
    out = subprocess.run([exe], capture_output=True, text=True)
    assert out.returncode == 0 and "tile_bounds: ok" in out.stdout, out.stdout + out.stderr


def test_gates_formed_in_a_row_kernel_go_to_that_kernel_alone():
    """tests/harness/row_dispatch (the library's own choice of a row kernel, compiled for the host): once the pre-pass is left to roww_kernel no
    other kernel is launched in its place."""
    here = os.path.join(os.path.dirname(os.path.abspath(__file__)), "harness")
    subprocess.check_call(["make", "-C", here, "row_dispatch"])
    out = subprocess.run([os.path.join(here, "row_dispatch")], capture_output=True, text=True)
    assert out.returncode == 0 and "row_dispatch: ok" in out.stdout, out.stdout + out.stderr


def test_the_column_kernel_taken_is_the_one_measured_to_be_faster():
    """tests/harness/col_dispatch (the library's own choice of a column kernel, compiled for the host)"""
    here = os.path.join(os.path.dirname(os.path.abspath(__file__)), "harness")
    subprocess.check_call(["make", "-C", here, "col_dispatch"])
    out = subprocess.run([os.path.join(here, "col_dispatch")], capture_output=True, text=True)
    assert out.returncode == 0 and "col_dispatch: ok" in out.stdout, out.stdout + out.stderr


@pytest.mark.parametrize("scratch", [[], ["scratch"]])
def test_chunk_states_of_a_kernel_with_scratch_memory_go_to_the_two_others(scratch):
    """tests/harness/chunk_dispatch (the library's own choice of the kernels of the chunk states, compiled for the host): a one-pass kernel that a compiler
    gave scratch memory is replaced where the library chose it and refused where the caller named it."""
    here = os.path.join(os.path.dirname(os.path.abspath(__file__)), "harness")
    subprocess.check_call(["make", "-C", here, "chunk_dispatch"])
    out = subprocess.run([os.path.join(here, "chunk_dispatch"), *scratch], capture_output=True, text=True)
    assert out.returncode == 0 and "cases ok" in out.stdout, out.stdout + out.stderr


def test_operators_do_without_the_native_host_path(monkeypatch):
    """The extension belongs to one torch release; missing, or another release's, it is left out with a warning and the calls go
    through ctypes (every function says that it serves nothing)."""
    def missing():
        raise ImportError("no such file")
    monkeypatch.setattr(ffi, "_native", None)
    monkeypatch.setattr(ffi, "_load_native", missing)
    with pytest.warns(RuntimeWarning, match="native host path does not load"):
        stand_in = ffi.native()
    assert ffi.native() is stand_in
    for name in ("matmul", "matmul_train", "gated", "gated_train", "scan", "slstm"):
        assert getattr(stand_in, name)(1, 2, 3) is None
    monkeypatch.undo()
    monkeypatch.setattr(ffi, "_native", None)
    monkeypatch.setattr(torch, "__version__", "1.0.0")
    with pytest.warns(RuntimeWarning, match="built for torch"):
        ffi.native()


def test_library_target_needs_no_torch():
    """The default target where Python has no torch: the library, and nothing that needs torch's headers."""
    csrc = os.path.join(os.path.dirname(os.path.abspath(ffi.__file__)), "csrc")
    for python, native in (("false", False), ("python3", True)):
        plan = subprocess.run(["make", "-n", "-B", "-C", csrc, f"PYTHON={python}"], capture_output=True, text=True)
        assert plan.returncode == 0 and "-o ../libmlstm_hip.so" in plan.stdout, plan.stderr
        assert ("mlstm_torch.cpp" in plan.stdout) == native
