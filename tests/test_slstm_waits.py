"""The sLSTM forward's helper waves wait for their input ring by a count of memory operations (csrc/slstm.hip).  What such a wait is worth depends on
how many operations the compiler issued, so the kernels are compiled for the device here, and the counts read from the listing."""
import os
import re
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "xlstm-triton-cuda-implementation_amd", "csrc")


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """(DH, saved state, sigmoid gate, 16-byte boundaries) -> lines of the kernel"""
    def variable(name):
        return subprocess.run(["make", "-s", "-C", CSRC, f"--eval=show: ; @echo $({name})", "show"], capture_output=True, text=True, check=True).stdout.split()
    out = tmp_path_factory.mktemp("listing") / "slstm.s"
    subprocess.run([*variable("HIPCC"), *variable("FLAGS"), "--cuda-device-only", "-S", "slstm.hip", "-o", str(out)], cwd=CSRC, check=True, capture_output=True)
    found, key = {}, None
    for line in out.read_text().splitlines():
        name = re.match(r"_ZN5slstm20slstm_forward_kernelILi(\d+)ELb(\d)ELb(\d)ELb(\d)E\w*:", line)
        if name:
            key = tuple(int(x) for x in name.groups())
            found[key] = []
        elif line.startswith(".Lfunc_end"):
            key = None
        elif key:
            found[key].append(line.split(";")[0].strip() + (" LOOP" if "Inner Loop Header" in line else ""))
    return found


def loops(lines):
    """the innermost loops: from the first block that is branched back to, to the last branch back"""
    label = {line.split(":")[0]: at for at, line in enumerate(lines) if line.startswith(".LBB")}
    for at, line in enumerate(lines):
        if line.endswith("LOOP"):
            back = [(label[target.group(1)], n) for n, target in enumerate(re.match(r"s_c?branch\w* (\.LBB\w+)", x) for x in lines) if n > at and target]
            back = [(to, n) for to, n in back if to <= at and "s_endpgm" not in lines[to:at]]
            yield lines[min(to for to, _ in back):max(n for _, n in back) + 1]


@pytest.mark.parametrize("DH", [32, 64, 128])
@pytest.mark.parametrize("save,sigmoid,wide", [(s, f, w) for s in (0, 1) for f in (0, 1) for w in (0, 1)])
def test_the_wait_for_an_input_row_covers_it(kernels, DH, save, sigmoid, wide):
    # A row that is waited for in interval t was requested at the end of interval t - (PF - 2): what may stay under way are the operations of the intervals
    # since, at most.  Without the saved state only the first helper wave stores, and the others have a wait of their own.
    ahead = int(re.search(r"constexpr int PF = (\d+);", open(os.path.join(CSRC, "slstm.hip")).read()).group(1)) - 2
    steady = 0
    for body in loops(kernels[DH, save, sigmoid, wide]):
        loads, stores = [sum(line.startswith(op) for line in body) for op in ("global_load_lds", "global_store")]
        waits = sorted({int(n) for line in body for n in re.findall(r"vmcnt\((\d+)\)", line)})
        if not (loads and any(line.startswith("s_barrier") for line in body)):
            continue
        steady += 1
        issued = [loads + stores] if save else [loads, loads + stores]
        assert waits and len(waits) <= len(issued), waits
        assert all(wait <= ahead * most for wait, most in zip(waits, issued)), (loads, stores, waits)
    assert steady


@pytest.mark.parametrize("DH", [32, 64, 128])
@pytest.mark.parametrize("save,sigmoid,wide", [(s, f, w) for s in (0, 1) for f in (0, 1) for w in (0, 1)])
def test_the_first_input_is_read_before_its_place_is_refilled(kernels, DH, save, sigmoid, wide):
    # The rows of the first round are there at a barrier.  The walk reads the first one behind it, the helpers request the row that takes its place: with
    # a barrier more between the two.
    lines = kernels[DH, save, sigmoid, wide]
    at = lambda start, *ops: next(n for n in range(start, len(lines)) if lines[n].startswith(ops))  # noqa: E731
    label = {line.split(":")[0]: n for n, line in enumerate(lines) if line.startswith(".LBB")}

    def passed(start, op):
        """for every line with `op` that a way from `start` comes to first: the lines of a shortest way there"""
        ways, seen, ends = [(start,)], {start}, []
        for way in ways:
            line = lines[way[-1]]
            if line.startswith(op) and len(way) > 1:
                ends.append([lines[n] for n in way])
                continue
            jump = re.match(r"s_(c?)branch\w* (\.LBB\w+)", line)
            following = ([label[jump.group(2)]] if jump else []) + ([] if line == "s_endpgm" or jump and not jump.group(1) else [way[-1] + 1])
            for n in following:
                if n not in seen and n < len(lines):
                    seen.add(n)
                    ways.append(way + (n,))
        return ends
    there = at(at(0, "global_load_lds"), "s_waitcnt vmcnt(0)")
    ways = passed(there, "global_load_lds")
    assert ways and all(sum(x.startswith("s_barrier") for x in way) >= 2 for way in ways)
    first = at(at(0, "global_load_dwordx4"), "s_barrier")   # (the walk begins with its part of R)
    ways = passed(first, "s_barrier")
    assert ways
    for way in ways:
        read = next(n for n, x in enumerate(way) if x.startswith("ds_read_b32"))
        assert any("lgkmcnt(0)" in x for x in way[read:])
