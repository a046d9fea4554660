"""Loads from a buffer straight into LDS are assembly of this library (fa_lds_dma.h), into which the compiler does not look when it keeps
hazards apart: a vector memory instruction must come five wait states after a vector instruction that wrote a scalar it reads. This
reads the built kernels and looks at what is ahead of every such load, over all ways that lead to it."""
import re
import subprocess
import tempfile

import foundry_attn as fa
from test_kernel_resources import _code_objects

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
STATES = 5


def scalars(operand):
    """Numbers of the scalar registers that an operand names."""
    if operand.startswith("vcc"):
        return {"vcc": {106, 107}, "vcc_lo": {106}, "vcc_hi": {107}}[operand]
    m = re.fullmatch(r"s\[(\d+):(\d+)\]|s(\d+)", operand)
    if not m:
        return set()
    return {int(m[3])} if m[3] else set(range(int(m[1]), int(m[2]) + 1))


def written_by_vector(op, operands):
    if op.startswith(("v_readlane", "v_readfirstlane", "v_cmp")):
        return scalars(operands[0]) if operands else set()
    if "_co_" in op or op.startswith(("v_div_scale", "v_mad_u64", "v_mad_i64")):
        return scalars(operands[1])
    return set()


def functions(listing):
    """Each function of an objdump listing: [(address, instruction, operands, address branched to or None)]."""
    start, out = 0, []
    for line in listing.splitlines():
        head = re.match(r"([0-9a-f]+) <\w+>:", line)
        if head:
            if out:
                yield out
            start, out = int(head[1], 16), []
            continue
        m = re.match(r"\s+(\w+)\s*(.*?)\s*// ([0-9A-F]+):", line)
        if m:
            to = re.search(r"<\w+\+0x([0-9a-f]+)>", line) if "branch" in m[1] else None
            operands = [x for part in m[2].split(",") for x in part.split()]
            out.append((int(m[3], 16), m[1], operands, start + int(to[1], 16) if to else None))
    if out:
        yield out


def check(code):
    """(loads into LDS, those that come too early) of one function."""
    index = {c[0]: i for i, c in enumerate(code)}
    from_branch = {}
    for i, (_, _, _, to) in enumerate(code):
        if to in index:
            from_branch.setdefault(index[to], []).append(i)
    loads, early = 0, []
    for i, (_, op, operands, _) in enumerate(code):
        if not (op.startswith("buffer_load") and "lds" in operands):
            continue
        loads += 1
        reads = set().union(*map(scalars, operands))
        ways, seen = [(i, 0)], {}
        while ways:
            j, states = ways.pop()
            before = list(from_branch.get(j, ()))
            if j and code[j - 1][1] not in ("s_branch", "s_endpgm", "s_setpc_b64"):
                before.append(j - 1)
            for k in before:
                _, o, x, _ = code[k]
                if written_by_vector(o, x) & reads:
                    early.append((hex(code[i][0]), o, x, states))
                after = states + (int(x[0], 0) + 1 if o == "s_nop" else 1)
                if after < STATES and after < seen.get(k, STATES):
                    seen[k] = after
                    ways.append((k, after))
    return loads, early


def test_checker_counts_wait_states():
    def listing(wait):
        return """0000000000001000 <f>:
	v_readlane_b32 s12, v73, s6   // 000000001000: 0
	%s
	s_mov_b32 m0, s3   // 000000001010: 0
	s_nop 0   // 000000001014: 0
	buffer_load_dwordx4 v70, s[44:47], s12 offen lds  // 000000001018: 0
	s_cbranch_scc0 65532 // 000000001020: BF84FFFC <f+0x14>
	v_cmp_lt_u32_e64 s[46:47], s1, v2   // 000000001024: 0
	s_branch 65528 // 000000001028: BF82FFF8 <f+0x18>
""" % wait
    for wait, found in (("s_nop 0  // 000000001008: 0", 2), ("s_nop 1  // 000000001008: 0", 2), ("s_nop 2  // 000000001008: 0", 1)):
        (code,) = functions(listing(wait))
        loads, early = check(code)
        assert loads == 1 and len(early) == found, (wait, early)


def test_loads_into_lds_come_five_wait_states_after_their_scalars():
    loads = 0
    with open(fa.LIB_PATH, "rb") as f:
        data = f.read()
    for co in _code_objects(data):
        with tempfile.NamedTemporaryFile(suffix=".co") as fh:
            fh.write(co)
            fh.flush()
            out = subprocess.run([OBJDUMP, "-d", fh.name], capture_output=True, text=True, check=True).stdout
        for code in functions(out):
            n, early = check(code)
            loads += n
            assert not early, early[:3]
    assert loads > 0
