"""Wait states around the instructions that are written as assembly (gemm_tile_k_loop_quad): the compiler keeps them for its own
instructions, and knows nothing of those inside an asm statement.  Looked for in the built library's code:

  * five between the vector unit writing a scalar register and a memory request that is addressed by it;
  * one between a write of M0 and a request into LDS;
  * two between the vector unit writing a register and a matrix product that reads it;
  * eleven between a product of eight passes and any other instruction touching its accumulator.
"""
import functools
import os
import re
import subprocess

import pytest

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PRODUCT = "v_mfma_f32_16x16x32_bf16"


@functools.lru_cache(maxsize=None)
def _regs(operand):
    """The registers an operand names: ("v", 3), ("a", 0), ("s", 28), ("m0", 0) ..."""
    m = re.match(r"([vas])(?:(\d+)$|\[(\d+):(\d+)\])", operand)
    if not m:
        return {(operand, 0)}
    lo = int(m[2] or m[3])
    return {(m[1], i) for i in range(lo, int(m[4] or lo) + 1)}


class _Instruction:
    def __init__(self, text):
        self.name, _, rest = text.partition(" ")
        ops = [o.strip().split(" ")[0] for o in rest.split(",")] if rest else []
        self.states = int(ops[0]) + 1 if self.name == "s_nop" else 1
        self.valu = self.name.startswith("v_")
        self.product = self.name.startswith("v_mfma") or self.name.startswith("v_smfma")
        outs = 2 if "_co_" in self.name or self.name.startswith(("v_div_scale", "v_swap")) else 1
        stores = self.name.startswith(("global_store", "buffer_store", "ds_write", "flat_store"))
        self.lds_request = self.name.startswith(("buffer_load", "global_load_lds")) and (rest.endswith(" lds") or "_lds_" in self.name)
        n = 0 if stores or self.lds_request or self.name.startswith(("s_cmp", "s_cbranch", "s_branch", "s_waitcnt", "s_nop")) else outs
        self.writes = set().union(*map(_regs, ops[:n])) if ops[:n] else set()
        self.reads = set().union(*map(_regs, ops[n:])) if ops[n:] else set()


_instruction = functools.lru_cache(maxsize=None)(_Instruction)


def hazards(listing):
    """Violations in an `llvm-objdump -d` listing of one or more kernels, as (instruction, earlier instruction) lines."""
    found, body = [], []
    for line in listing.splitlines() + ["0 <end>:"]:
        if re.match(r"[0-9a-f]+ <.*>:$", line):
            found += _kernel(body)
            body = []
        elif "//" in line:
            body.append(line)
    return found


def _kernel(lines):
    if not any(" offen lds" in l for l in lines):   # (no request written as assembly)
        return []
    ins, at, sources = [], {}, {}
    for i, l in enumerate(lines):
        text, _, tail = l.partition("//")
        at[int(tail.split(":")[0], 16)] = i
        ins.append(_instruction(re.sub(r"\s+", " ", text.strip())))
    base = min(at)
    for i, l in enumerate(lines):
        m = re.search(r"<[^<>+]*(?:\+0x([0-9a-f]+))?>\s*$", l)
        if m and ins[i].name.startswith(("s_cbranch", "s_branch")):
            sources.setdefault(at[base + int(m[1] or "0", 16)], []).append(i)

    def before(i, limit, wrong):
        """The first instruction within `limit` wait states before i, on any path, that `wrong` says must not be there."""
        todo, seen = [(i, 0)], {}
        while todo:
            j, waited = todo.pop()
            prev = list(sources.get(j, ()))
            if j and not ins[j - 1].name.startswith(("s_branch", "s_endpgm", "s_setpc")):
                prev.append(j - 1)
            for k in prev:
                if wrong(ins[k]):
                    return k
                w = waited + ins[k].states
                if w < limit and seen.get(k, limit) > w:
                    seen[k] = w
                    todo.append((k, w))
        return None

    found = []
    accumulators = set().union(*(x.writes for x in ins if x.name == PRODUCT))
    for i, x in enumerate(ins):
        checks = []
        if x.name.startswith(("buffer_", "global_")):
            scalars = {r for r in x.reads if r[0] == "s"}
            checks.append((5, lambda y: y.valu and y.writes & scalars))
        if x.lds_request:
            checks.append((1, lambda y: ("m0", 0) in y.writes))
        if x.product:
            checks.append((2, lambda y: y.valu and not y.product and y.writes & x.reads))
        elif (x.reads | x.writes) & accumulators:
            checks.append((11, lambda y: y.name == PRODUCT and y.writes & (x.reads | x.writes)))
        for limit, wrong in checks:
            k = before(i, limit, wrong)
            if k is not None:
                found.append((lines[i].strip(), lines[k].strip()))
    return found


@pytest.fixture(scope="module")
def listings(tmp_path_factory):
    """The disassembly of each of the built library's code objects."""
    if not os.path.exists(OBJDUMP):
        pytest.skip("no disassembler")
    tmp = tmp_path_factory.mktemp("code")
    lib = tmp / "lib.so"
    lib.symlink_to(os.path.join(ROOT, "dion_amd", "libdion_amd.so"))
    subprocess.run([OBJDUMP, "--offloading", str(lib)], cwd=tmp, check=True, capture_output=True)
    return {f.name: subprocess.run([OBJDUMP, "-d", "--mcpu=gfx950", str(f)], check=True, capture_output=True, text=True).stdout
            for f in sorted(tmp.glob("*gfx950*"))}


def test_the_built_library_keeps_the_wait_states(listings):
    assert sum(text.count(" offen lds") for text in listings.values()) > 0
    for name, text in listings.items():
        assert hazards(text) == [], name


def test_accumulators_are_cleared_behind_the_first_requests(listings):
    """Not a hazard, but half a microsecond of a tile: the clearing lies under the first stage's trip to memory, where nothing else does."""
    kernels = 0
    for text in listings.values():
        for kernel in re.split(r"^[0-9a-f]+ <.*>:$", text, flags=re.M)[1:]:
            first = kernel.find(" offen lds")
            if first >= 0:
                kernels += 1
                assert not re.search(r"v_accvgpr_write|v_mfma", kernel[:first])
    assert kernels > 0


LOOP = """0000000000001000 <kernel>:
\ts_add_u32 m0, s17, s33                     // 000000001000: 807C2111
\ts_nop 0                                    // 000000001004: BF800000
\tbuffer_load_dwordx4 v128, s[28:31], s25 offen lds // 000000001008: E05D1000 19070080
\tv_mfma_f32_16x16x32_bf16 a[0:3], v[8:11], v[4:7], a[0:3] // 000000001010: D3B50000 04020908
\ts_nop 10                                   // 000000001018: BF80000A
\tv_accvgpr_read_b32 v1, a2                  // 00000000101C: D3D84001 18000102
\ts_cbranch_scc1 65528                       // 000000001024: BF85FFF8 <kernel>
\ts_endpgm                                   // 000000001028: BF810000
"""


@pytest.mark.parametrize("old, new, count", [
    ("s_nop 10", "s_nop 10", 0),
    ("s_nop 10", "s_nop 9", 1),                                                # an accumulator read too early
    ("s_nop 0 ", "s_mov_b32 s1, 0 ", 0),
    ("\ts_nop 0 ", "\tv_mov_b32 v9, 0 ", 1),                                   # a fragment moved, one instruction before its product
    ("v_accvgpr_read_b32 v1, a2 ", "v_readlane_b32 s28, v1, 0 ", 1),           # a buffer's scalar, four before the request, round the loop
    ("s_add_u32 m0, s17, s33", "s_mov_b32 s3, s33     ", 0),
    ("\ts_nop 0  ", "\ts_mov_b32 m0, s3 ", 1),                                 # M0 written right before the request
])
def test_planted_hazards_are_found(old, new, count):
    assert old in LOOP
    assert len(hazards(LOOP.replace(old, new, 1))) == count
