"""Scalars that a kernel has no scalar register for are kept by the compiler in lanes of a vector register (v_writelane), from where they
are read back (v_readlane) at their use. Assembly inside the kernels, accumulators moved as a whole and branches of the write stages are
around such places: this follows every way through the built kernels and finds a lane that is read and was not written on all of
them, or whose register something else has written since."""
import re
import subprocess
import tempfile

import foundry_attn as fa
from test_kernel_resources import _code_objects
from test_lds_load_waits import OBJDUMP, functions

NO_VECTOR_RESULT = re.compile(r"s_|ds_(write|store)|(global|buffer|flat|scratch)_store|buffer_(wb|inv)|v_cmp|v_readlane|v_readfirstlane")


def vectors(operand):
    m = re.fullmatch(r"v\[(\d+):(\d+)\]|v(\d+)", operand)
    if not m:
        return set()
    return {int(m[3])} if m[3] else set(range(int(m[1]), int(m[2]) + 1))


def written(op, operands):
    """Vector registers that an instruction writes."""
    if NO_VECTOR_RESULT.match(op) or not operands or (op.startswith("buffer_load") and "lds" in operands):
        return set()
    if "atomic" in op and "sc0" not in operands:  # (nothing comes back)
        return set()
    return vectors(operands[0]) | (vectors(operands[1]) if "swap" in op else set())


def check(code):
    """(reads of such lanes, those that may find something else) of one function."""
    keeping = {min(vectors(x[0])) for _, op, x, _ in code if op.startswith("v_writelane")}
    if not keeping:
        return 0, []
    index = {c[0]: i for i, c in enumerate(code)}
    known, work = {0: frozenset()}, [0]  # lanes that hold what was written to them, on all ways to an instruction
    while work:
        i = work.pop()
        _, op, x, to = code[i]
        after = known[i]
        if op.startswith("v_writelane"):
            after = after | {(min(vectors(x[0])), x[2])}
        else:
            lost = written(op, x) & keeping
            if lost:
                after = frozenset(s for s in after if s[0] not in lost)
        ways = [index[to]] if to in index else []
        if op not in ("s_branch", "s_endpgm", "s_setpc_b64") and i + 1 < len(code):
            ways.append(i + 1)
        for k in ways:
            new = after if k not in known else known[k] & after
            if known.get(k) != new:
                known[k] = new
                work.append(k)
    reads, wrong = 0, []
    for i, (at, op, x, _) in enumerate(code):
        if i in known and op.startswith("v_readlane") and vectors(x[1]) & keeping:
            reads += 1
            if (min(vectors(x[1])), x[2]) not in known[i]:
                wrong.append((hex(at), x))
    return reads, wrong


def test_checker_follows_the_ways():
    def listing(other, back):
        return """0000000000001000 <f>:
	v_writelane_b32 v73, s6, 5   // 000000001000: 0
	s_cbranch_scc0 2 // 000000001008: 0 <f+0x14>
	%s
	v_readlane_b32 s7, v73, 5   // 000000001014: 0
	s_cbranch_scc1 9 // 00000000101C: 0 <f+%s>
	s_endpgm  // 000000001020: 0
	v_writelane_b32 v73, s6, 6   // 000000001024: 0
	s_branch 9   // 00000000102C: 0 <f+0x14>
""" % (other, back)
    for other, back, found in (("v_mov_b32_e32 v72, v1 // 00000000100C: 0", "0x14", 0), ("v_mov_b32_e32 v73, v1 // 00000000100C: 0", "0x14", 1),
                               ("buffer_load_dwordx4 v73, s[4:7], s8 offen lds // 00000000100C: 0", "0x24", 0),
                               ("v_mfma_f32_16x16x32_f16 v[72:75], v[0:3], v[4:7], 0 // 00000000100C: 0", "0x24", 1),
                               ("v_permlane32_swap_b32_e32 v1, v73 // 00000000100C: 0", "0x24", 1)):
        (code,) = functions(listing(other, back))
        reads, wrong = check(code)
        assert reads == 1 and len(wrong) == found, (other, wrong)


def test_scalars_kept_in_vector_lanes_are_read_as_they_were_written():
    reads = 0
    with open(fa.LIB_PATH, "rb") as f:
        data = f.read()
    for co in _code_objects(data):
        with tempfile.NamedTemporaryFile(suffix=".co") as fh:
            fh.write(co)
            fh.flush()
            out = subprocess.run([OBJDUMP, "-d", fh.name], capture_output=True, text=True, check=True).stdout
        for code in functions(out):
            n, wrong = check(code)
            reads += n
            assert not wrong, wrong[:3]
    assert reads > 0
