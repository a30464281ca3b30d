"""Wait states in the built library, checked on its disassembly (no GPU needed).

The kernels issue their MFMAs and their global -> LDS copies from inline assembly, so the compiler counts none of the wait states
that gfx950 leaves to software around them: it cannot see what the statements are.  What it puts next to them (a spilled scalar
fetched back with v_readlane, a spilled accumulator stored to scratch, a register move) changes with every change of a kernel, so
the built code itself is looked at.  From every producer all paths are followed until enough wait states have passed:

  * a scalar register written by a vector instruction and read by a vector memory instruction: 5
  * M0 written by a scalar instruction and used by a buffer load to LDS: 1
  * a register written by an MFMA and used by anything but an MFMA that takes exactly it as SrcC: 8 for 4 passes, 12 for 8
  * a vector register written by a vector instruction and read by an MFMA: 2

Every instruction is one wait state, s_nop N is N + 1.  In the kernels whose MFMAs are inline assembly the accumulators must besides be
separated from whatever reads them by an s_nop that is long enough by itself: instructions that happen to stand there would do as
well, until they don't.
"""

import re
import struct
import subprocess
from concurrent.futures import ProcessPoolExecutor
from pathlib import Path

import pytest

LIB = Path(__file__).resolve().parents[1] / "flydsl_amd" / "libpsgemm.so"
OBJDUMP = Path("/opt/rocm/llvm/bin/llvm-objdump")

_REG = re.compile(r"(?<![\w.])([vas])(?:(\d+)\b|\[(\d+):(\d+)\])")
_LINE = re.compile(r"^\t(\S+)(.*?)\s*// ([0-9A-F]+): [0-9A-F ]+(?:<[^>]*?(?:\+0x([0-9a-f]+))?>)?$")
_HEAD = re.compile(r"^[0-9a-f]* ?<(.+)>:$")
_VMEM = ("buffer_", "global_", "flat_", "scratch_")
_BASE = {"v": 0, "a": 1 << 10, "s": 1 << 11}
_M0, _VCC = _BASE["s"] + 500, _BASE["s"] + 501


def _regs(text):
    """Registers named in `text`, one number each."""
    out = set()
    for kind, one, lo, hi in _REG.findall(text):
        b = _BASE[kind]
        out.update(range(b + int(lo), b + int(hi) + 1) if lo else (b + int(one),))
    if "m0" in text:
        out.add(_M0)
    if "vcc" in text:
        out.add(_VCC)
    return out


class Ins:
    __slots__ = ("op", "args", "addr", "target", "_ops")

    def __init__(self, op, args, addr, target):
        self.op, self.args, self.addr, self.target, self._ops = op, args, addr, target, None

    @property
    def ops(self):
        if self._ops is None:
            self._ops = [_regs(x) for x in self.args.split(",")]
        return self._ops

    @property
    def states(self):
        return int(self.args, 0) + 1 if self.op == "s_nop" else 1

    @property
    def mfma(self):
        return self.op.startswith("v_mfma")

    @property
    def valu(self):
        return self.op.startswith("v_") and not self.mfma

    @property
    def vmem(self):
        return self.op.startswith(_VMEM)

    def used(self):
        return set().union(*self.ops)

    def __str__(self):
        return f"{self.addr:x}: {self.op} {self.args.strip()}"


def parse(text):
    """Disassembly -> {symbol: [Ins]}."""
    out, cur, base = {}, None, 0
    for line in text.splitlines():
        h = _HEAD.match(line)
        if h:
            cur, base = out.setdefault(h.group(1), []), None
            continue
        m = _LINE.match(line)
        if m is None or cur is None:
            continue
        addr = int(m.group(3), 16)
        base = addr if base is None else base
        op = m.group(1)
        target = base + int(m.group(4) or "0", 16) if op.startswith(("s_branch", "s_cbranch")) else None
        cur.append(Ins(op, m.group(2), addr, target))
    return out


def _passes(i):
    """Passes of a 16x16 MFMA: fp8 operands take eight, everything narrower or 16-bit four."""
    if "f8f6f4" in i.op:
        code = lambda n: int((re.search(rf"{n}:(\d)", i.args) or [0, 0])[1])
        return 4 if code("cbsz") >= 2 and code("blgp") >= 2 else 8
    return 4


def hazards(code, explicit=False):
    """Messages for one kernel: [Ins] -> [str].  `explicit`: an MFMA's result needs an s_nop, looked for over 32 wait states."""
    at = {i.addr: n for n, i in enumerate(code)}
    found = []

    def follow(n, need, regs, hit, nop=None):
        """All paths behind instruction n until `need` states have passed (or an s_nop of `nop` states) or `regs` are written again: where
        hit() holds, report."""
        todo, seen = [(n + 1, 0, frozenset(regs))], set()
        while todo:
            k, states, live = todo.pop()
            while k < len(code) and states < need and live:
                if (k, states) in seen:
                    break
                seen.add((k, states))
                i = code[k]
                if hit(i, live):
                    found.append(f"{code[n]}  ->  {i}  ({states} of {need} wait states)")
                    break
                states += i.states
                if i.op == "s_endpgm" or (nop and i.states >= nop):
                    break
                if i.target is not None and i.target in at:
                    if i.op == "s_branch":
                        k = at[i.target]
                        continue
                    todo.append((at[i.target], states, live))
                if (i.valu or i.op.startswith("s_")) and i.ops:
                    live = live - i.ops[0]
                k += 1

    for n, i in enumerate(code):
        if i.mfma:
            d = i.ops[0]

            def early(j, live, d=d):
                if not j.mfma:
                    return bool(j.used() & live)
                # exactly the result as SrcC: the hardware waits
                return bool((j.ops[1] | j.ops[2]).union(*j.ops[4:]) & live) or (j.ops[3] != d and bool(j.ops[3] & live))

            need = 12 if _passes(i) == 8 else 8
            follow(n, 32 if explicit else need, d, (lambda j, live: not j.mfma and bool(j.used() & live)) if explicit else early, need if explicit else None)
        elif i.valu:
            d = set().union(*i.ops[:2]) if i.op.startswith(("v_add_co", "v_addc_co", "v_sub_co", "v_subb_co", "v_mad_u64", "v_mad_i64", "v_div_scale")) else i.ops[0]
            sregs = {r for r in d if r >= _BASE["s"]}
            if sregs:
                follow(n, 5, sregs, lambda j, live: j.vmem and bool(j.used() & live))
            vregs = i.ops[0] - sregs
            if vregs:
                follow(n, 2, vregs, lambda j, live: j.mfma and bool(j.used() & live))
        elif i.op.startswith("s_") and i.ops and _M0 in i.ops[0]:
            follow(n, 1, {_M0}, lambda j, live: j.op.startswith("buffer_load") and j.args.rstrip().endswith("lds"))
    return found


def _code_objects():
    data = LIB.read_bytes()
    magic, at = b"__CLANG_OFFLOAD_BUNDLE__", 0
    while (at := data.find(magic, at)) >= 0:
        (count,), o = struct.unpack_from("<Q", data, at + 24), at + 32
        for _ in range(count):
            off, size, tl = struct.unpack_from("<QQQ", data, o)
            if b"gfx950" in data[o + 24:o + 24 + tl]:
                yield data[at + off:at + off + size]
            o += 24 + tl
        at += 24


def _k(text):
    lines, addr = ["0000000000000000 <k>:"], 0
    for t in text.strip().splitlines():
        t, _, target = t.strip().partition(" @")
        lines.append(f"\t{t} // {addr:012X}: 00000000" + (f" <k+0x{int(target) * 4:x}>" if target else ""))
        addr += 4
    return parse("\n".join(lines))["k"]


@pytest.mark.parametrize("text,bad", [
    ("v_readlane_b32 s20, v1, 3\ns_mov_b32 m0, s3\ns_nop 0\nbuffer_load_dwordx4 v2, s[8:11], s20 offen lds", True),
    ("v_readlane_b32 s20, v1, 3\ns_mov_b32 m0, s3\ns_nop 4\nbuffer_load_dwordx4 v2, s[8:11], s20 offen lds", False),
    ("s_mov_b32 s20, s1\ns_mov_b32 m0, s3\ns_nop 0\nbuffer_load_dwordx4 v2, s[8:11], s20 offen lds", False),
    ("s_mov_b32 m0, s3\nbuffer_load_dwordx4 v2, s[8:11], s20 offen lds", True),
    ("v_mfma_f32_16x16x128_f8f6f4 a[0:3], v[0:7], v[8:15], a[0:3]\ns_nop 10\nscratch_store_dwordx4 off, a[0:3], s33", True),
    ("v_mfma_f32_16x16x128_f8f6f4 a[0:3], v[0:7], v[8:15], a[0:3]\ns_nop 11\nscratch_store_dwordx4 off, a[0:3], s33", False),
    ("v_mfma_i32_16x16x64_i8 a[0:3], v[0:3], v[8:11], a[0:3]\ns_nop 6\nv_accvgpr_read_b32 v9, a1", True),
    ("v_mfma_i32_16x16x64_i8 a[0:3], v[0:3], v[8:11], a[0:3]\nv_mfma_i32_16x16x64_i8 a[0:3], v[4:7], v[8:11], a[0:3]", False),
    ("v_mov_b32_e32 v5, v6\ns_nop 0\nv_mfma_i32_16x16x64_i8 a[0:3], v[4:7], v[8:11], a[0:3]", True),
    ("v_mov_b32_e32 v5, v6\ns_nop 1\nv_mfma_i32_16x16x64_i8 a[0:3], v[4:7], v[8:11], a[0:3]", False),
    # the reader sits behind a taken branch
    ("v_readlane_b32 s20, v1, 3\ns_cbranch_scc1 2 @4\ns_nop 4\ns_endpgm\nbuffer_load_dwordx4 v2, s[8:11], s20 offen", True),
])
def test_the_check_itself(text, bad):
    assert bool(hazards(_k(text))) == bad


def _scan(blob):
    text = subprocess.run([str(OBJDUMP), "-d", "--no-leading-addr", "/dev/stdin"], input=blob, capture_output=True, check=True).stdout.decode()
    return {name: bad for name, code in parse(text).items() if (bad := hazards(code) + (hazards(code, True) if "_tiled" in name else []))}


@pytest.mark.skipif(not LIB.exists() or not OBJDUMP.exists(), reason="needs the built library and llvm-objdump")
def test_no_kernel_reads_too_early():
    bad, blobs = {}, sorted(_code_objects(), key=len, reverse=True)
    assert len(blobs) >= 15
    with ProcessPoolExecutor(4) as pool:
        for one in pool.map(_scan, blobs):
            bad.update(one)
    assert not bad, "\n".join(f"{k}: {len(v)}\n  " + "\n  ".join(v[:4]) for k, v in bad.items())
