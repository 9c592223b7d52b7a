"""The copies into LDS (lds_dma16, lds_dma4, lds_dma16_at in csrc/common.hpp) are inline assembly, which
the compiler's hazard handling does not look into: a memory instruction that reads an SGPR (or m0) needs
five wait states after a VALU instruction that wrote it.  The device assembly that the compiler writes
from every source with the library's own flags holds no such pair, and the copies that move their
scalar operands hold none whatever the compiler puts before them.  Compiles for gfx950, CPU only."""
import concurrent.futures as cf
import os
import re
import subprocess

import pytest

from syntropy_amd import build as B

pytestmark = pytest.mark.skipif(not os.path.exists(B.HIPCC), reason="needs hipcc")
WAIT_STATES = 5
COPY = "global_load_lds_"


def assembly(src, out):
    cmd = [B.HIPCC, *B.FLAGS, *B.FILE_FLAGS.get(os.path.basename(src), []), f"-I{B.CSRC}", "--cuda-device-only", "-S",
           src, "-o", out]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    with open(out) as f:
        return f.read()


def scalars(operand):
    """The scalar registers an operand names: s5, s[4:5], m0, vcc."""
    m = re.fullmatch(r"s\[(\d+):(\d+)\]", operand)
    if m:
        return {f"s{i}" for i in range(int(m[1]), int(m[2]) + 1)}
    if re.fullmatch(r"s\d+|m0|vcc_lo|vcc_hi|ttmp\d+", operand):
        return {operand}
    return {"vcc_lo", "vcc_hi"} if operand == "vcc" else set()


def instructions(asm):
    """(line number, label or None, mnemonic, operands) of each instruction and label."""
    for no, line in enumerate(asm.splitlines(), 1):
        line = line.split(";")[0].strip()
        if re.fullmatch(r"[\w.$]+:", line):
            yield no, line[:-1], "", []
        elif line and not line.startswith("."):
            op, _, rest = line.partition(" ")
            yield no, None, op.strip(), [t for a in re.split(r",\s*", rest.strip()) if a for t in a.split()[:1]]


def hazards(asm):
    """Copies that read a scalar register fewer than five wait states after a VALU instruction wrote
    it, on the straight line before them or at the end of a block that branches to them."""
    found, copies = [], 0
    history = []                 # (VALU-written scalars, wait states it counts) back to front
    at_branch = {}               # label: the histories at the branches to it
    code = list(instructions(asm))
    for walk in (0, 1):          # backward branches are known on the second walk
        found, copies, history = [], 0, [[]]
        for no, label, op, args in code:
            if label is not None:
                history = history + at_branch.get(label, [])
                continue
            if op.startswith(COPY):
                copies += 1
                reads = {"m0"}.union(*(scalars(a) for a in args))
                for h in history:
                    left = WAIT_STATES
                    for written, states in reversed(h):
                        if written & reads:
                            found.append(no)
                        left -= states
                        if left <= 0:
                            break
            if op in ("s_branch",) or op.startswith("s_cbranch"):
                at_branch.setdefault(args[0], []).extend(h[-WAIT_STATES:] for h in history)
                at_branch[args[0]] = [list(h) for h in {tuple((frozenset(w), s) for w, s in h) for h in at_branch[args[0]]}]
            if op in ("s_branch", "s_endpgm", "s_setpc_b64"):
                history = []
                continue
            written = set()
            if op.startswith("v_") and args:
                # v_readlane and compares write the first operand, carries and div_scale the second
                written = scalars(args[0]) | (scalars(args[1]) if len(args) > 3 and "_co_" in op or "div_scale" in op else set())
            elif op.startswith("s_") and args and not re.match(r"s_(cmp|bitcmp|nop|waitcnt|set|barrier|sleep)", op):
                over = scalars(args[0])  # a scalar instruction's own result (it waits for the VALU's)
                history = [[(w - over, s) for w, s in h] for h in history]
            states = 1 + int(args[0], 0) if op == "s_nop" else 1
            history = [(h + [(frozenset(written), states)])[-WAIT_STATES:] for h in history]
            history = [list(h) for h in {tuple(h) for h in history}]
    return sorted(set(found)), copies


PROBE = r"""
#include "common.hpp"
using namespace syn;
template <int FORM>
__global__ void probe(const uint8_t* p, uint32_t* out) {
    extern __shared__ uint8_t lds[];
    const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)(uintptr_t)p + threadIdx.x, 3);
    const uint32_t hi = __builtin_amdgcn_readlane((uint32_t)((uintptr_t)p >> 32) + threadIdx.x, 3);
    const uint8_t* base = (const uint8_t*)(((uint64_t)hi << 32) | lo);
    const uint32_t at = __builtin_amdgcn_readlane(lds_addr(lds) + threadIdx.x, 5);
    if constexpr (FORM == 0) lds_dma16(16 * threadIdx.x, base, at);
    if constexpr (FORM == 1) lds_dma4(4 * threadIdx.x, base, at);
    if constexpr (FORM == 2) lds_dma16_at(p + 16 * threadIdx.x, at);
    if constexpr (FORM == 3) lds_dma16<true>(16 * threadIdx.x, base, at);
    wait_vm<0>();
    lds_barrier();
    out[threadIdx.x] = lds[threadIdx.x];
}
template __global__ void probe<%d>(const uint8_t*, uint32_t*);
"""


@pytest.mark.parametrize("form,safe", [(0, True), (1, True), (2, True), (3, False)])
def test_moved_operands_need_no_wait_states(tmp_path, form, safe):
    """A base and an LDS address straight from v_readlane: the moving forms are safe, and the check
    sees the bare one."""
    src = tmp_path / "probe.hip"
    src.write_text(PROBE % form)
    found, copies = hazards(assembly(str(src), str(tmp_path / "probe.s")))
    assert copies == 1
    assert (not found) == safe


def test_the_check_reads_branches():
    asm = "a:\nv_readlane_b32 s4, v0, 1\ns_cbranch_scc1 b\ns_nop 4\ns_branch c\nb:\ns_nop 0\n" \
          "global_load_lds_dword v1, s[4:5]\nc:\nglobal_load_lds_dword v1, s[4:5]\ns_endpgm\n"
    assert hazards(asm) == ([8, 10], 2)
    assert hazards(asm.replace("b:\n", "b:\ns_mov_b32 s4, s4\n")) == ([], 2)
    assert hazards(asm.replace("b:\n", "b:\ns_nop 3\n")) == ([], 2)


def test_no_copy_follows_a_valu_write_of_its_operands(tmp_path):
    srcs = [s for s in B.sources() if s.endswith(".hip")]
    with cf.ThreadPoolExecutor(max_workers=8) as ex:
        asm = list(ex.map(lambda s: assembly(s, str(tmp_path / (os.path.basename(s) + ".s"))), srcs))
    total = 0
    for src, text in zip(srcs, asm):
        found, copies = hazards(text)
        total += copies
        assert not found, f"{os.path.basename(src)}: assembly lines {found[:8]}"
    assert total > 100  # the copies are there to be checked
