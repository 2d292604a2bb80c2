"""The generated code of dense_pair_kernel, whose output wavefronts count their tile loads.

They issue the loads of a tile (inline assembly, direct to LDS) once per position and wait
with `s_waitcnt vmcnt(N)` until all but the three youngest tiles have landed.  The count holds
only if nothing else of theirs is counted, and the ring only runs ahead if nothing drains it:
a stray vector-memory instruction, or a wait of the compiler's own, would break one or the other.
"""
import re

import pytest

from tests.test_kernel_invariants import _significant, prefill_asm  # noqa: F401  (a fixture)

VMEM = re.compile(r"(global|buffer|scratch|flat)_")
TILE_LOADS = {64: 2, 96: 4, 128: 4}     # K and V instructions of one 32-key tile per wavefront
AHEAD = 6                               # tiles requested before the first position


@pytest.fixture(scope="module")
def pair_kernels(prefill_asm):  # noqa: F811
    kernels = {}
    for m in re.finditer(r"^(_ZN2mi\S*\ddense_pair_kernelI(\S+?)Li(\d+)E\S*):", prefill_asm, re.M):
        body = prefill_asm[m.end():prefill_asm.index(".Lfunc_end", m.end())]
        kernels[(m.group(2), int(m.group(3)))] = [t for _, t in _significant(body.split("\n"))]
    assert len(kernels) == 6, sorted(kernels)          # bf16 / f16  x  64 / 96 / 128
    return kernels


def _roles(code):
    """(output wavefronts up to their stores, score wavefronts from their Q loads on)."""
    first = next(i for i, t in enumerate(code) if t.startswith("global_load_lds"))
    store = next(i for i, t in enumerate(code) if t.startswith("global_store_dwordx4"))
    q = next(i for i, t in enumerate(code) if re.match(r"global_load_dwordx4 v\[\d+:\d+\], v\[\d+:\d+\], off", t))
    assert first < store < q
    return code[first:store], code[q:]


def _problems(output, scores, d):
    """What of the kernel's assumptions the instructions of its two roles do not meet."""
    found = []
    loads = TILE_LOADS[d]
    counted, drained = "s_waitcnt vmcnt(%d)" % (3 * loads), "s_waitcnt vmcnt(0)"
    found += [t for t in output if VMEM.match(t) and not t.startswith("global_load_lds_dwordx4")]
    found += [t for t in output if "vmcnt" in t and t not in (counted, drained)]
    parts, part = [], []
    for t in output:
        if t == "s_barrier":
            parts.append(part)
            part = []
        else:
            part.append(t)
    # first position, positions with output, positions without; what leads to the barrier of each
    if len(parts) != 3:
        found.append("%d barriers" % len(parts))
    sent = [sum(t.startswith("global_load_lds") for t in p) for p in parts + [part]]
    if sent != [AHEAD * loads] + [loads] * 3:
        found.append("loads between barriers: %s" % sent)
    for p in parts[:2] + [sum(parts[2:], part)]:   # (the last loop may be laid out with its waits behind its loads)
        if p.count(counted) != 1 or p.count(drained) != 1:
            found.append("waits before a barrier: %s" % [t for t in p if "vmcnt" in t])
    # the full wait is one arm of a decision: a conditional branch stands directly before it
    for i, t in enumerate(output):
        if t == drained and not output[i - 1].startswith("s_cbranch"):
            found.append("a full wait on the straight path behind %s" % output[i - 1])
    # the score wavefronts load Q and nothing else, and have waited for it before their loop leaves probabilities
    at = [i for i, t in enumerate(scores) if VMEM.match(t) and not t.startswith("global_store_dword ")]
    if len(at) != d // 16:
        found.append("%d loads of Q" % len(at))
    if max(i for i, t in enumerate(scores) if "vmcnt" in t) >= next(i for i, t in enumerate(scores) if t.startswith("ds_write_b128")):
        found.append("a wait for vector memory in the loop of the score wavefronts")
    return found


def test_the_output_wavefronts_count_their_tile_loads_alone(pair_kernels):
    for (dtype, d), code in pair_kernels.items():
        assert not _problems(*_roles(code), d), (dtype, d)


# A listing with one mistake planted in it: each has to be noticed.
@pytest.mark.parametrize("plant", ["stray load", "full wait", "other count", "missing load", "wait in the score loop"])
def test_mistakes_are_noticed(pair_kernels, plant):
    for (dtype, d), code in pair_kernels.items():
        output, scores = (list(part) for part in _roles(code))
        second = [i for i, t in enumerate(output) if t == "s_barrier"][1]
        load = next(i for i in range(second, len(output)) if output[i].startswith("global_load_lds"))
        wait = next(i for i in range(second) if output[i] == "s_waitcnt vmcnt(%d)" % (3 * TILE_LOADS[d]))
        if plant == "stray load":
            output.insert(load, "global_load_dword v1, v[2:3], off")
        elif plant == "full wait":
            output.insert(load, "s_waitcnt vmcnt(0)")
        elif plant == "other count":
            output[wait] = "s_waitcnt vmcnt(%d)" % (4 * TILE_LOADS[d])
        elif plant == "missing load":
            del output[load]
        else:
            scores.append("s_waitcnt vmcnt(0)")
        assert _problems(output, scores, d), (dtype, d, plant)
