"""The work that users of these operators have them do, as cases that can be timed and compared.

A case is one operator on one shape: a forward pass as inference runs it, or a training step (forward and the gradients of
every input through autograd).  ``listed`` holds the shapes that stand for typical uses, ``draw`` gives further ones of the
same ranges:

* matmul form (``mlstm_matmul``, ``Triton_mLSTM``, with output gate ``Triton_mLSTM_gated``, in split mode
  ``Triton_mLSTM_precise``): bf16, fp16 and fp32, D = 64, 128, 256 (fp32: 64, 128), 1 to 64 heads over the batch, 64 to 16384
  positions, q / k / v as [B,NH,S,D] or as views of [B,S,NH,D] projections, gates in the tensors' type or in fp32;
* scan form (``mlstm_scan``): fp32, D = 64 ... 1024, 1 to 32 heads over the batch, 64 to 8192 positions;
* sLSTM cell (``slstm``): fp32, DH = 32, 64, 128, batches of 1 to 32, 1 to 8 heads, 16 to 2048 positions.

Inputs are standard normal; the forget gate's pre-activations are shifted by +3 (a trained forget-gate bias), those of the
case ``train_f32`` not at all (a model at initialisation).
"""
import torch

from _mlstm_pkg import submodule
from mlstm_matmul import Triton_mLSTM, Triton_mLSTM_gated, mlstm_matmul
from mlstm_scan import mlstm_scan
from slstm import slstm

Triton_mLSTM_precise = submodule("mlstm_matmul").Triton_mLSTM_precise

DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}


def _mlstm(name, op, B, NH, S, D, dtype, gates=None, layout="bnsd", f_mean=3.0):
    case = {"op": op, "B": B, "NH": NH, "S": S, "D": D, "dtype": dtype, "gates": gates or dtype, "layout": layout, "f_mean": f_mean}
    return dict(case, name=name) if name else case


def _slstm(name, op, B, NH, S, D):
    case = {"op": op, "B": B, "NH": NH, "S": S, "D": D, "dtype": "f32"}
    return dict(case, name=name) if name else case


def listed():
    return [
        # one head of a short sequence: the smallest call, the shape of a single-head forward harness
        _mlstm("forward_f16_one_head", "forward", 1, 1, 640, 128, "f16"),
        # a prompt of odd length through one layer, straight from the projections
        _mlstm("forward_bf16_prompt", "forward", 1, 8, 1777, 256, "bf16", "f32", "bsnd"),
        # a small model in fp32 at initialisation
        _mlstm("train_f32", "train", 1, 4, 2048, 64, "f32", f_mean=0.0),
        # a small model on short sequences, where launches and host work count
        _mlstm("train_bf16_short", "train", 8, 4, 256, 64, "bf16", "f32"),
        # few heads, a length that fits no tile
        _mlstm("train_f16_ragged", "train", 3, 5, 1001, 128, "f16"),
        # a layer of a large model
        _mlstm("train_bf16_layer", "train", 4, 8, 4096, 256, "bf16"),
        # long context
        _mlstm("train_bf16_long", "train", 2, 32, 16384, 128, "bf16"),
        # a layer with the output gate, straight from the projections
        _mlstm("train_gated", "train_gated", 2, 8, 2048, 128, "bf16", "f32", "bsnd"),
        # split mode: 16-bit tensors where fp32-like results are wanted
        _mlstm("train_split_mode", "train_precise", 2, 4, 1500, 256, "bf16"),
        # the scan form at a large head dimension, inference
        _mlstm("scan_forward", "scan", 1, 4, 2048, 1024, "f32"),
        # the scan form of a small model, training, ragged length
        _mlstm("scan_train", "scan_train", 2, 4, 1000, 128, "f32"),
        # the sLSTM cell of a training step
        _slstm("slstm_train", "slstm_train", 16, 4, 2048, 64),
    ]


def _log_int(rng, lo, hi):
    n = int(round(lo * (hi / lo) ** rng.random()))
    return min(hi, max(lo, n))


def _cost(case):
    """Seconds on an ideal card, fp32 products at a fifth of the 16-bit rate: what a drawn case is limited by."""
    w = work(case)
    return max(w["bytes"] / 8e12, w["flops"] / (5e14 if case["dtype"] == "f32" else 2.5e15))


def draw(rng):
    most = max(_cost(c) for c in listed())
    while True:
        op = rng.choice(["forward", "forward", "train", "train", "train", "train", "train_gated", "train_precise", "scan", "scan_train",
                         "slstm", "slstm_train"])
        if op.startswith("slstm"):
            case = _slstm(None, op, _log_int(rng, 1, 32), _log_int(rng, 1, 8), _log_int(rng, 16, 2048), rng.choice([32, 64, 128]))
        else:
            scan = op.startswith("scan")
            heads = _log_int(rng, 1, 32 if scan else 64)
            NH = rng.choice([n for n in range(1, heads + 1) if heads % n == 0])
            S = _log_int(rng, 64, 8192 if scan else 16384)
            if rng.random() < 0.5:   # half of the lengths are whole tiles, as padded batches have them
                S = max(64, S // 64 * 64)
            if scan:
                case = _mlstm(None, op, heads // NH, NH, S, rng.choice([64, 128, 256, 512, 1024]), "f32")
            else:
                dtype = rng.choice(["bf16", "f16"] if op == "train_precise" else ["bf16", "bf16", "f16", "f32"])
                D = rng.choice([64, 128] if dtype == "f32" else [64, 128, 256])
                case = _mlstm(None, op, heads // NH, NH, S, D, dtype, rng.choice([dtype, "f32"]), rng.choice(["bnsd", "bsnd"]))
        if _cost(case) <= most:
            return case


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    B, NH, S, D, op, dtype = case["B"], case["NH"], case["S"], case["D"], case["op"], DTYPES[case["dtype"]]
    train = "train" in op
    normal = lambda *shape: torch.randn(shape, device="cuda", generator=g)  # noqa: E731
    if op.startswith("slstm"):
        ins = [normal(B, S, 4, NH, D), normal(NH, 4, D, D) / D ** 0.5, normal(NH, 4, D)]
        grad = normal(B, S, NH, D) if train else None
    else:
        def rows():
            if case["layout"] == "bsnd":
                return normal(B, S, NH, D).to(dtype).transpose(1, 2)
            return normal(B, NH, S, D).to(dtype)
        gates = DTYPES[case["gates"]]
        ins = [rows(), rows(), rows(), (normal(B, NH, S) + case["f_mean"]).to(gates), normal(B, NH, S).to(gates)]
        if op.startswith("scan") or op == "train_gated":
            ins.append(rows())
        grad = rows() if train else None
    if train:
        for t in ins:
            t.requires_grad_(True)
    return {"op": op, "ins": ins, "grad": grad}


def run(state):
    op, ins, grad = state["op"], state["ins"], state["grad"]
    if op == "forward":
        return mlstm_matmul(*ins)
    if op == "scan":
        return mlstm_scan(*ins)
    if op == "slstm":
        return slstm(*ins, True)
    if op == "train":
        out = Triton_mLSTM.apply(*ins)
    elif op == "train_gated":
        out = Triton_mLSTM_gated.apply(*ins)
    elif op == "train_precise":
        out = Triton_mLSTM_precise.apply(*ins)
    elif op == "scan_train":
        out = mlstm_scan(*ins)
    else:
        out = slstm(*ins, True)
    return (out.detach(), *torch.autograd.grad(out, ins, grad))


def work(case):
    """Bytes: every input and the output gradient once, the output and every gradient once.  Flops: the cheaper of the two
    forms of the function for this length, 2 D multiply-adds per pair of positions or 2 D^2 per position for the state's update
    and read-out; the gradients are five such products to the forward's two.  sLSTM: the recurrent matrices, 4 D^2 per position
    forward, once more each for the gradients of the state and of the matrices."""
    B, NH, S, D, op = case["B"], case["NH"], case["S"], case["D"], case["op"]
    train = "train" in op
    BHS = B * NH * S
    if op.startswith("slstm"):
        weights = 4 * NH * D * (D + 1)
        return {"bytes": 4.0 * ((BHS * 4 * D + weights) * (2 if train else 1) + BHS * D * (2 if train else 1)),
                "flops": 8.0 * D * D * BHS * (3 if train else 1)}
    size = {"f32": 4, "f16": 2, "bf16": 2}
    tensors = 4 if op.startswith("scan") or op == "train_gated" else 3
    row, gate = D * size[case["dtype"]], 2 * size[case["gates"]]
    forward = tensors * row + gate
    nbytes = BHS * (forward + row) if not train else BHS * (2 * forward + 2 * row)
    return {"bytes": float(nbytes), "flops": BHS * min(2.0 * D * (S + 1), 4.0 * D * D) * (3.5 if train else 1.0)}


def tolerance(case):
    """What two correct evaluations in one type differ by.  The 16-bit kernels round the weights of a product to the type (2^-9
    of a bf16, 2^-12 of an fp16 value); rows of the mLSTM whose normaliser nearly cancels enlarge that, in every form of the
    function, as they enlarge the rounding of the fp32 sums."""
    if case["op"].startswith("slstm"):
        return {"rel": 1e-5}
    return {"bf16": {"rel": 1e-2}, "f16": {"rel": 2e-3}, "f32": {"rel": 2e-5}}[case["dtype"]]
