"""The results of one head, bit by bit, against digests in golden/kernel_bits.json: those of the kernels that served launches of every size
before there were others for few workgroups.  Which kernel serves a head depends on the batch it is in and its results do not, nor do
they change with the way a kernel spreads its sums over waves; what rounds a product or adds up a sum in another order shows here.
(dF of a sequence in chunks is pinned where one wave holds all columns of a row: 16 bits at D = 64.)"""
import hashlib
import json
import os

import numpy as np
import pytest
import torch

from _mlstm_pkg import submodule

pytestmark = pytest.mark.gpu
mm = submodule("mlstm_matmul")
with open(os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "kernel_bits.json")) as file:
    GOLDEN = json.load(file)
DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}


def results(case, copies=1):
    """{name: [1, copies, ...]} of `copies` times the same head"""
    op, dtype, S, D = case.split("_")
    S, D = int(S[1:]), int(D[1:])
    rng = np.random.default_rng(S + D)
    rows = [torch.from_numpy(rng.standard_normal((1, 1, S, D)).astype(np.float32)).to(DTYPES[dtype]) for _ in range(4)]
    gates = [torch.from_numpy((rng.standard_normal((1, 1, S)) + m).astype(np.float32)) for m in (3, 0)]
    q, k, v, dh, f, i = [t.cuda().repeat_interleave(copies, 1) for t in rows + gates]
    h, m, b, saved = mm.mlstm_forward_save_hip(q, k, v, f, i, precise=op == "precise")
    grads = mm.mlstm_backward_saved_hip(dh, q, k, v, f, i, h, m, b, saved, precise=op == "precise")
    return dict(zip(("h", "b", "dq", "dk", "dv", "df", "di"), (h, b, *grads)))


def digest(t):
    return hashlib.sha256(t.contiguous().cpu().view(torch.uint8).numpy().tobytes()).hexdigest()[:16]


def check(case, names, copies):
    res = results(case, copies)
    for name in names:
        assert digest(res[name][:, 0]) == GOLDEN[case][name], name
        assert torch.equal(res[name], res[name][:, :1].expand_as(res[name])), name


def copies_of(case, many):   # one head: the kernels for few workgroups; more than 768 workgroups of 64 positions: the others
    return 800 * 64 // int(case.split("_")[2][1:]) + 1 if many else 1


@pytest.mark.parametrize("many", [False, True])
@pytest.mark.parametrize("case", sorted(GOLDEN))
def test_row_pass(case, many):
    check(case, ("b", "h", "dq"), copies_of(case, many))


# fp32 and D = 64: col_kernel and colf_kernel; the products of dD enter the row sums unrounded
@pytest.mark.parametrize("many", [False, True])
@pytest.mark.parametrize("case", [c for c in sorted(GOLDEN) if "f32" in c or c.endswith("D64")])
def test_column_pass_of_fp32_and_of_head_dimension_64(case, many):
    check(case, [n for n in ("dk", "dv", "di", "df") if n in GOLDEN[case]], copies_of(case, many))


# 16 bits at D = 128 and 256: cold_kernel and colw_kernel; one column sum per key, products of dD unrounded in it, and those of G and W in their
# low-order terms
@pytest.mark.parametrize("many", [False, True])
@pytest.mark.parametrize("case", [c for c in sorted(GOLDEN) if "f32" not in c and not c.endswith("D64")])
def test_column_pass_of_16_bits(case, many):
    check(case, [n for n in ("dk", "dv", "di", "df") if n in GOLDEN[case]], copies_of(case, many))
