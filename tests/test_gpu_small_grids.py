"""Kernels for launches that would leave the chip part empty (roww_kernel, chunk_sum_narrow_kernel; fp32: rowf_kernel, colf_kernel) against the ones that
serve larger launches: the same products in the same order, so a head alone and the same head in a batch that is large enough for the
other kernels give the same bits.  Lengths at the edges of the 64-row tiles, of the pairs of key tiles, of the 32-row blocks and of the chunks."""
import pytest
import torch

from _mlstm_pkg import submodule

pytestmark = pytest.mark.gpu
mm = submodule("mlstm_matmul")


def _inputs(heads, S, D, dtype, layout):
    g = torch.Generator(device="cuda").manual_seed(S + D)
    shape = (1, heads, S, D) if layout == "bnsd" else (1, S, heads, D)
    rows = [torch.randn(shape, device="cuda", generator=g).to(dtype) for _ in range(5)]
    if layout == "bsnd":
        rows = [t.transpose(1, 2) for t in rows]
    return rows, [(torch.randn(1, heads, S, device="cuda", generator=g) + m).to(dtype) for m in (3, 0)]


def _step(op, rows, gates, heads):
    q, k, v, dh, o = [t[:, :heads] for t in rows]
    f, i = [t[:, :heads].contiguous() for t in gates]
    if op == "gated":
        hg, h, m, b = mm.mlstm_forward_gated_hip(q, k, v, f, i, o)
        return [hg, h, m, b, *mm.mlstm_backward_gated_hip(dh, q, k, v, f, i, o, h, m, b)]
    h, m, b, saved = mm.mlstm_forward_save_hip(q, k, v, f, i, precise=op == "precise")
    return [h, m, b, *mm.mlstm_backward_saved_hip(dh, q, k, v, f, i, h, m, b, saved, precise=op == "precise")]


# heads: enough for more than 256 workgroups of 64 rows, and from 1024 positions on for more than 768 blocks of 64 x 64
@pytest.mark.parametrize("op,S,D,heads,layout", [
    ("plain", 1, 128, 264, "bnsd"), ("plain", 63, 256, 258, "bnsd"), ("plain", 64, 128, 260, "bsnd"), ("plain", 65, 256, 130, "bnsd"),
    ("gated", 127, 128, 131, "bnsd"), ("plain", 129, 128, 90, "bsnd"), ("gated", 200, 256, 70, "bsnd"), ("plain", 640, 128, 27, "bnsd"),
    ("plain", 1023, 256, 17, "bsnd"), ("plain", 1023, 128, 17, "bnsd"), ("plain", 1024, 256, 49, "bnsd"), ("gated", 1025, 128, 65, "bnsd"),
    ("plain", 1601, 256, 25, "bsnd"), ("plain", 2048, 128, 22, "bnsd"), ("precise", 1100, 256, 26, "bnsd"), ("precise", 1537, 128, 30, "bsnd")])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_a_head_alone_is_the_head_of_a_full_chip(op, S, D, heads, layout, dtype):
    rows, gates = _inputs(heads, S, D, dtype, layout)
    for name, a, b in zip(range(10), _step(op, rows, gates, 1), _step(op, rows, gates, heads)):
        assert bool(torch.isfinite(b.float()).all()) and torch.equal(a[:, :1], b[:, :1]), name


# fp32: more than 512 workgroups of 32 rows.  (colf_kernel serves chunks of 128 at D = 128 whatever the number of heads.)
@pytest.mark.parametrize("op,S,D,heads,layout", [
    ("plain", 1, 64, 260, "bnsd"), ("plain", 31, 128, 260, "bnsd"), ("plain", 33, 64, 260, "bsnd"), ("plain", 64, 128, 260, "bnsd"),
    ("gated", 97, 128, 130, "bnsd"), ("plain", 129, 64, 90, "bnsd"), ("plain", 319, 64, 52, "bnsd"), ("gated", 319, 128, 52, "bsnd"),
    ("plain", 320, 64, 52, "bnsd"), ("gated", 450, 64, 33, "bsnd"), ("plain", 700, 128, 24, "bnsd"), ("plain", 1000, 64, 17, "bnsd")])
def test_a_head_alone_is_the_head_of_a_full_chip_fp32(op, S, D, heads, layout):
    test_a_head_alone_is_the_head_of_a_full_chip(op, S, D, heads, layout, torch.float32)


# colw_kernel (few workgroups) against cold_kernel (selected by hand): lengths at the edges of its 32-query tiles, of the pipeline's first and
# last steps, of the 64-key tiles and of the chunks; 1024 queries are the most that a key may meet without chunks
@pytest.mark.parametrize("op,S,D,heads,layout", [
    ("plain", 1, 128, 2, "bnsd"), ("plain", 32, 256, 1, "bnsd"), ("plain", 33, 128, 1, "bsnd"), ("plain", 63, 256, 3, "bsnd"), ("gated", 65, 128, 1, "bnsd"),
    ("precise", 95, 256, 2, "bnsd"), ("precise", 97, 128, 8, "bsnd"), ("plain", 129, 256, 2, "bnsd"), ("precise", 161, 256, 1, "bnsd"),
    ("plain", 1000, 256, 1, "bnsd"), ("precise", 1001, 128, 1, "bnsd"), ("plain", 1025, 256, 3, "bnsd"), ("precise", 1057, 256, 2, "bsnd"),
    ("plain", 1089, 128, 8, "bnsd"), ("precise", 1500, 128, 2, "bnsd"), ("gated", 2047, 256, 2, "bnsd"), ("plain", 2600, 128, 1, "bnsd")])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_few_key_tiles_give_the_bits_of_many(op, S, D, heads, layout, dtype):
    rows, gates = _inputs(heads, S, D, dtype, layout)
    ours = _step(op, rows, gates, heads)
    ffi = submodule("_ffi")
    ffi.set_column_kernel(2)
    try:
        theirs = _step(op, rows, gates, heads)
    finally:
        ffi.set_column_kernel(0)
    for name, a, b in zip(range(10), ours, theirs):
        assert bool(torch.isfinite(a.float()).all()) and torch.equal(a, b), name


# split mode: rowx_kernel against row_kernel (force_generic_kernels), edges of the 64-key tiles, the 32-row blocks, the walk's first steps and the
# chunks' state
@pytest.mark.parametrize("S,D,heads,layout", [
    (1, 128, 1, "bnsd"), (32, 256, 2, "bnsd"), (33, 128, 8, "bsnd"), (64, 256, 1, "bnsd"), (65, 128, 2, "bnsd"), (127, 256, 3, "bsnd"), (130, 256, 1, "bnsd"),
    (200, 128, 1, "bnsd"), (257, 128, 2, "bnsd"), (1000, 256, 2, "bnsd"), (1023, 128, 3, "bsnd"), (1025, 256, 1, "bnsd"), (1089, 128, 2, "bnsd"),
    (1100, 256, 8, "bsnd"), (1665, 256, 2, "bnsd"), (2048, 128, 1, "bnsd")])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_split_mode_few_row_tiles_give_the_bits_of_many(S, D, heads, layout, dtype):
    rows, gates = _inputs(heads, S, D, dtype, layout)
    ours = _step("precise", rows, gates, heads)
    ffi = submodule("_ffi")
    ffi.force_generic_kernels(True)
    try:
        theirs = _step("precise", rows, gates, heads)
    finally:
        ffi.force_generic_kernels(False)
    for name, a, b in zip(range(4), ours, theirs):   # h, m, b, dq
        assert bool(torch.isfinite(a.float()).all()) and torch.equal(a, b), name


# the carry in blocks of 32 x 32 against the one in blocks of 64 x 64 (more than 192, from 6 states on 384, from 12 on 512 of them), and groups of
# four steps: 1 to 5 states, 6, 7, 12, 13 (D = 128 in chunks of 512), 16 and 17 (the edge of what is requested at once)
@pytest.mark.parametrize("op,S,D,heads", [("plain", 1024, 128, 49), ("plain", 1537, 128, 49), ("precise", 2049, 256, 13), ("plain", 2561, 256, 13),
                                          ("plain", 3073, 128, 97), ("precise", 3600, 256, 25), ("plain", 6145, 128, 129), ("plain", 6700, 256, 33),
                                          ("plain", 8193, 128, 129), ("plain", 8705, 128, 129)])
def test_either_carry_gives_a_head_the_same_bits(op, S, D, heads):
    test_a_head_alone_is_the_head_of_a_full_chip(op, S, D, heads, "bnsd", torch.bfloat16)


# D = 128 with more than 512 workgroups of 64 rows (row_kernel, two workgroups per CU) and more than 768 of 64 keys (cold_kernel, likewise; in
# chunks 512): edges of the 128-row and 128-key tiles, of the 64- and 32-row tiles that they walk, and of the chunks
@pytest.mark.parametrize("op,S,heads,layout", [
    ("plain", 1, 772, "bnsd"), ("gated", 32, 770, "bnsd"), ("plain", 33, 769, "bsnd"), ("plain", 64, 776, "bnsd"), ("gated", 65, 390, "bsnd"),
    ("plain", 127, 388, "bnsd"), ("plain", 129, 260, "bnsd"), ("plain", 200, 200, "bsnd"), ("plain", 640, 80, "bnsd"), ("gated", 1023, 50, "bnsd"),
    ("plain", 1024, 41, "bnsd"), ("gated", 1025, 40, "bsnd"), ("plain", 1153, 33, "bnsd"), ("plain", 1601, 24, "bnsd")])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_pairs_of_workgroups_per_cu_give_the_same_bits(op, S, heads, layout, dtype):
    test_a_head_alone_is_the_head_of_a_full_chip(op, S, 128, heads, layout, dtype)


# split mode at D = 128 on row_kernel with two workgroups per CU (more than 256 of 64 rows) against rowx_kernel (one head), the same edges
@pytest.mark.parametrize("S,heads,layout", [(1, 258, "bnsd"), (33, 257, "bsnd"), (65, 130, "bnsd"), (129, 90, "bsnd"), (640, 27, "bnsd"), (1023, 17, "bnsd"),
                                            (1025, 16, "bsnd"), (1601, 25, "bnsd")])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_split_mode_pairs_of_workgroups_per_cu_give_the_same_bits(S, heads, layout, dtype):
    test_a_head_alone_is_the_head_of_a_full_chip("precise", S, 128, heads, layout, dtype)


# D = 64: the forward in chunks of 256 (three workgroups per CU) against the uncut one (two) on the first chunk alone, whose rows take no state
@pytest.mark.parametrize("S,heads,layout", [(1024, 1, "bnsd"), (1025, 9, "bsnd"), (1100, 3, "bnsd"), (1919, 40, "bsnd")])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_the_first_chunk_at_head_dimension_64_is_the_uncut_sequence(S, heads, layout, dtype):
    rows, gates = _inputs(heads, S, 64, dtype, layout)
    L = submodule("_ffi").lib().mlstm_chunk_length_for(S, 64, submodule("_ffi").dtype_code(dtype))
    whole = mm.mlstm_forward_hip(*rows[:3], *gates)
    first = mm.mlstm_forward_hip(*[t[:, :, :L] for t in rows[:3]], *[t[:, :, :L].contiguous() for t in gates])
    for name, a, b in zip(("h", "m", "b"), first, whole):
        assert bool(torch.isfinite(a.float()).all()) and torch.equal(a, b[:, :, :L]), name


# fp32 at D = 64 on row_kernel with two workgroups per CU (more than 256 of 128 rows) against rowf_kernel (one head)
@pytest.mark.parametrize("op,S,heads,layout", [("plain", 1, 520, "bnsd"), ("plain", 97, 514, "bsnd"), ("gated", 129, 260, "bnsd"), ("plain", 320, 176, "bnsd"),
                                               ("plain", 1025, 60, "bsnd")])
def test_fp32_pairs_of_workgroups_per_cu_give_the_same_bits(op, S, heads, layout):
    test_a_head_alone_is_the_head_of_a_full_chip(op, S, 64, heads, layout, torch.float32)


# roww_kernel on 32 rows per workgroup (up to 128 granules of 64 rows) and on 64 (up to 256, uncut sequences a few more) against row8_kernel: rows that end in
# either half of a granule, one to five rounds of 128 keys, diagonal blocks in either half of a round, and the chunks' state in front of them
@pytest.mark.parametrize("op,S,layout", [("plain", 1, "bnsd"), ("gated", 31, "bsnd"), ("plain", 32, "bnsd"), ("plain", 33, "bsnd"), ("plain", 96, "bnsd"),
                                         ("gated", 129, "bnsd"), ("plain", 160, "bsnd"), ("plain", 193, "bnsd"), ("plain", 257, "bnsd"), ("gated", 321, "bnsd"),
                                         ("plain", 385, "bsnd"), ("plain", 450, "bnsd"), ("plain", 545, "bnsd"), ("plain", 990, "bsnd"), ("plain", 1024, "bnsd"),
                                         ("gated", 1025, "bsnd"), ("plain", 1185, "bnsd"), ("plain", 1700, "bnsd")])
@pytest.mark.parametrize("D", [128, 256])
def test_row_workgroups_of_every_size_give_the_same_bits(op, S, D, layout):
    NG = (S + 63) // 64
    sizes = (1, 128 // NG + 1, (256 if S >= 1024 else 256 + 8 * NG) // NG + 1)
    rows, gates = _inputs(sizes[-1], S, D, torch.bfloat16, layout)
    small, middle, large = [_step(op, rows, gates, heads) for heads in sizes]
    for name, a, b, c in zip(range(10), small, middle, large):
        assert bool(torch.isfinite(c.float()).all()) and torch.equal(a, c[:, :1]) and torch.equal(b, c[:, :sizes[1]]), name
