"""CPU checks of the other FP64 kernels that spill into accumulation registers, beside the delay-line ones of
test_isa_invariants.py: the role-split solve, the direct solve from LDS blocks, and the adjoint's local stage,
tangent and transposes. The wait states are checked the same way. The must-defined analysis is too strict for the
role-split kernel: on the way out of its plane loop the compiler runs through the copies at the loop's end,
some of registers that only the next step would have read. So what is required here is that no value
that may be undefined reaches an instruction that is not a copy, on any path that scalar conditions known to be 0
or -1 leave open."""
import collections
import os
import re
import shutil
import subprocess

import pytest

from astaroth_amd import build as B
from tests import isa_check as I

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
COPIES = ("v_accvgpr_read", "v_accvgpr_mov", "v_accvgpr_write", "v_mov_b32", "v_mov_b64", "scratch_load",
          "scratch_store")
STORES = ("global_store", "ds_write", "buffer_store", "flat_store", "scratch_store")


def vregs(tok):
    m = re.match(r"^-?\|?v\[(\d+):(\d+)\]", tok)
    if m:
        return {f"v{k}" for k in range(int(m.group(1)), int(m.group(2)) + 1)}
    m = re.match(r"^-?\|?(v\d+)\|?$", tok)
    return {m.group(1)} if m else set()


def operands(t):
    """(storage written, storage read) of one instruction: vector registers, and what isa_check tracks."""
    ts = I._toks(t)
    defs, uses = I._effects(t)
    store = ts[0].startswith(STORES)
    for x in ts[1 if store else 2:]:
        uses = uses | vregs(x)
    if not store and len(ts) > 1:
        if ts[0].startswith(("v_fmac", "v_writelane")):
            uses = uses | vregs(ts[1])
        if not ts[0].startswith("v_writelane"):  # one lane of the register
            defs = defs | vregs(ts[1])
    return defs, uses


def scalar_facts(t, facts):
    """Scalar pairs known to be 0 or -1 after the instruction."""
    ts = I._toks(t)
    op, new = ts[0], None
    if op == "s_mov_b64":
        new = int(ts[2]) if ts[2] in ("0", "-1") else facts.get(ts[2])
    elif op in ("s_and_b64", "s_andn2_b64") and ts[1:3] == ["vcc", "exec"] and ts[3] in facts:
        new = facts[ts[3]] if op == "s_and_b64" else -1 - facts[ts[3]]
    if op.startswith(("s_", "v_")) and not op.startswith(("s_cbranch", "s_branch", "s_waitcnt", "s_nop", "s_barrier",
                                                          "s_endpgm", "s_cmp")):
        written = set().union(*(I._sregs(x) for x in ts[1:3 if op[0] == "v" else 2]))
        if re.match(r"v_(cmp|add_co|sub_co|subrev_co|addc_co|subb_co|subbrev_co).*_e32$|v_div_scale", op):
            written |= {"vcc_lo", "vcc_hi"}
        facts = {k: v for k, v in facts.items() if not I._sregs(k) & written}
    if new is not None:
        facts = dict(facts, **{ts[1]: new})
    return facts


def undefined_values(lines):
    """(block, storage, instruction) of every use, other than a copy, of a value that may be undefined. Vector
    registers count as defined at the entry; accumulation registers, spill slots and lanes do not."""
    blocks = I._blocks(lines)
    index = {label: i for i, (label, _) in enumerate(blocks)}

    def run(i, facts, good, found):
        facts, good = dict(facts), set(good)
        for t in blocks[i][1]:
            defs, uses = operands(t)
            bad = uses - good
            if bad and not t.startswith(COPIES):
                found.add((blocks[i][0], ",".join(sorted(bad)), t))
                bad = set()
            good = good - defs if bad else good | defs
            facts = scalar_facts(t, facts)
        last = blocks[i][1][-1] if blocks[i][1] else ""
        target = [index[last.split()[-1]]] if last.startswith(("s_cbranch", "s_branch")) else []
        through = [] if last.startswith(("s_branch", "s_endpgm", "s_setpc")) or i + 1 == len(blocks) else [i + 1]
        if last.startswith("s_cbranch_vcc") and "vcc" in facts:
            jumps = (facts["vcc"] != 0) == last.startswith("s_cbranch_vccnz")
            target, through = (target, []) if jumps else ([], through)
        return frozenset(facts.items()), good, target + through

    start = (0, frozenset())
    state = {start: {f"v{k}" for k in range(256)}}
    work = collections.deque([start])
    while work:
        node = work.popleft()
        facts, good, after = run(*node, state[node], set())
        for nxt in ((j, facts) for j in after):
            meet = good if nxt not in state else state[nxt] & good
            if nxt not in state or meet != state[nxt]:
                state[nxt] = meet
                work.append(nxt)
    found = set()
    for node, good in state.items():
        run(*node, good, found)
    return sorted(found)


LOOP = """\
_Z1ev:
\tv_accvgpr_write_b32 a1, 0
.LBB0_1:
\tv_add_f32_e32 v1, v2, v3
\ts_mov_b64 s[0:1], -1
\ts_cbranch_scc1 .LBB0_2
\tds_read_b32 a0, v4
\ts_mov_b64 s[0:1], 0
.LBB0_2:
\tv_accvgpr_read_b32 v2, a0
\ts_and_b64 vcc, exec, s[0:1]
\ts_cbranch_vccz .LBB0_1
\tv_accvgpr_read_b32 v5, a1
\tv_add_f32_e32 v6, v5, v5
\ts_endpgm
.Lfunc_end0:
"""


def test_checker_follows_values():
    body = I.kernels(LOOP)["_Z1ev"]
    # a0 is copied undefined on the way out, and used by no one there
    assert [x for _, x, _ in I.undefined_reads(body)] == ["a0"]
    assert undefined_values(body) == []
    # used after the loop; the exit condition of that path not known; the copy used in the loop's first pass
    used = LOOP.replace("\tv_accvgpr_read_b32 v5, a1\n", "\tv_mov_b32_e32 v5, v2\n")
    assert undefined_values(I.kernels(used)["_Z1ev"]) == [("#2", "v5", "v_add_f32_e32 v6, v5, v5")]
    unknown = LOOP.replace("\ts_mov_b64 s[0:1], -1\n", "")
    assert undefined_values(I.kernels(unknown)["_Z1ev"]) == [(".LBB0_1", "v2", "v_add_f32_e32 v1, v2, v3")]
    early = LOOP.replace("v_add_f32_e32 v1, v2, v3", "v_accvgpr_mov_b32 a2, a0\n\tv_accvgpr_read_b32 v7, a2\n"
                         "\tglobal_store_dword v8, v7, s[2:3]")
    assert [x for _, x, _ in undefined_values(I.kernels(early)["_Z1ev"])] == ["v7"]


@pytest.fixture(scope="module", params=["solve_split_a.hip", "solve_split_b.hip", "solve_direct.hip", "adjoint.hip"])
def fp64_kernels(request, tmp_path_factory):
    if shutil.which(B._hipcc()) is None and not os.path.exists(B._hipcc()):
        pytest.skip("hipcc not available")
    source = request.param
    out = tmp_path_factory.mktemp("isa") / (source + ".s")
    cmd = ([B._hipcc()] + B.HIP_FLAGS + ["-DAC_DOUBLE_PRECISION=1"] +
           ([] if source in B.DEFAULT_SCHED else B.PRECISION_FLAGS["fp64"]) + B.SOURCE_FLAGS.get(source, []) +
           ["-I", os.path.join(REPO, "include"), "--cuda-device-only", "-S",
            os.path.join(REPO, "astaroth_amd", "csrc", source), "-o", str(out)])
    r = subprocess.run([c for c in cmd if c != "-fPIC"], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    kernels = I.kernels(out.read_text())
    assert len(kernels) >= 4
    return kernels


def test_no_undefined_value_is_used(fp64_kernels):
    bad = {k: found[:5] for k, found in ((k, undefined_values(b)) for k, b in fp64_kernels.items()) if found}
    assert not bad, bad


def test_wait_states_kept(fp64_kernels):
    bad = {k: found[:5] for k, found in ((k, I.wait_state_violations(b)) for k, b in fp64_kernels.items()) if found}
    assert not bad, bad
