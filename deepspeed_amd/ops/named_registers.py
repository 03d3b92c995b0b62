"""A look through the compiler's assembly of kernels that keep sums in accumulation
registers which they name in inline assembly (csrc/tile_linear.hip). The compiler
knows neither that these hold anything nor what the assembly does, so a build ends
where its output would not go with it: ``faults`` of every such kernel.

  * An accumulation register outside the kernel's own assembly, or m0, where its
    loads to LDS go; a vector register spilled, scratch memory (both are how the
    compiler would come to take an accumulation register).
  * What the hardware does not wait for and the compiler, which does not read inline
    assembly, does not fill in: a vector register written less than two instructions
    before a product of the assembly reads it, a scalar register written by a vector
    instruction less than five before a load of the assembly does.

It is run by setup.py and stands alone: no import of the package is needed."""

import re
import subprocess
import tempfile

_KERNEL = re.compile(r"^(\w+):\s*; @\1$")
_LABEL = re.compile(r"^(\.L\w+):")
_REGISTER = re.compile(r"\b([asv])(?:(\d+)\b|\[(\w+):(\w+)\])")
_M0 = re.compile(r"\bm0\b")
# written by a vector instruction besides its first operand
_PAIR = re.compile(r"^v_(?:swap|permlane\d+_swap|mad_[ui]64|div_scale|"
                   r"(?:add|sub|subrev)(?:c|b|brev)?_co)")


def _registers(text):
    """Kinds and numbers of the registers that an operand's text names."""
    out = set()
    for kind, one, lo, hi in _REGISTER.findall(text):
        a = int(one or lo, 0)
        out |= {(kind, i) for i in range(a, (a if one else int(hi, 0)) + 1)}
    return out


class _Instruction:
    def __init__(self, text, own):
        self.own = own                          # of the kernel's assembly
        self.name, _, rest = text.partition(" ")
        operands = [o.strip() for o in rest.split(",")]
        self.all = _registers(rest)
        self.written, self.read = set(), set()
        if self.name.startswith(("v_", "ds_read", "buffer_load", "global_load")):
            n = 2 if _PAIR.match(self.name) else 1
            if not (self.name.startswith("buffer_load") and "lds" in rest.split()):
                self.written = _registers(",".join(operands[:n]))
            else:
                n = 0
            if "permlane" in self.name or "swap" in self.name:
                n = 0
            self.read = _registers(",".join(operands[n:]))
        self.waits = 1
        if self.name == "s_nop":
            self.waits = int(rest.split()[0], 0) + 1
        self.vector = self.name.startswith("v_") and "mfma" not in self.name
        self.to = rest.strip() if self.name.startswith(
            ("s_cbranch", "s_branch")) else None
        self.text = text


def _functions(lines):
    """(name, [instructions and labels], following metadata) of every function."""
    name, body = None, []
    for line in lines:
        start = _KERNEL.match(line)
        if start:
            name, body, own = start.group(1), [], False
        elif name is None:
            continue
        elif line.startswith(".Lfunc_end"):
            yield name, body
            name = None
        elif "#ASMSTART" in line:
            own = True
        elif "#ASMEND" in line:
            own = False
        elif _LABEL.match(line):
            body.append(_LABEL.match(line).group(1))
        else:
            for text in line.split(";")[0].split("\n"):
                text = " ".join(text.split())
                if text and not text.startswith("."):
                    body.append(_Instruction(text, own))


def _before(body, at, waits):
    """Instructions that may come less than ``waits`` before the one at ``at``, over
    every branch to a label on the way."""
    came = {}
    for i, b in enumerate(body):
        if isinstance(b, _Instruction) and b.to:
            came.setdefault(b.to, []).append(i)
    found, todo, seen = [], [(at, waits)], set()
    while todo:
        i, left = todo.pop()
        while i > 0 and left > 0 and (i, left) not in seen:
            seen.add((i, left))
            i -= 1
            b = body[i]
            if isinstance(b, str):
                todo += [(j + 1, left) for j in came.get(b, [])]
                continue
            if b.name in ("s_branch", "s_endpgm") and i + 1 != at and \
                    isinstance(body[i + 1], str):
                break               # what follows is come to by its label alone
            found.append(b)
            left -= b.waits
    return found


def faults(assembly: str):
    """What is wrong with the kernels of the assembly that name accumulation
    registers themselves; and the number of these kernels."""
    bad, kernels = [], 0
    meta = dict(re.findall(r"\.amdhsa_kernel (\w+)\n(.*?)\.end_amdhsa_kernel",
                           assembly, re.S))
    spilled = dict(re.findall(r"\.name:\s+(\w+)\n(?:(?!\.name:).)*?"
                              r"\.vgpr_spill_count:\s+(\d+)", assembly, re.S))
    for name, body in _functions(assembly.split("\n")):
        code = [b for b in body if isinstance(b, _Instruction)]
        if not any(b.own and any(k == "a" for k, _ in b.all) for b in code):
            continue
        kernels += 1
        scratch = re.search(r"private_segment_fixed_size (\d+)", meta.get(name, ""))
        if scratch is None or int(scratch.group(1)):
            bad.append(name + ": scratch memory")
        if int(spilled.get(name, 1)):
            bad.append(name + ": vector registers spilled")
        for i, b in enumerate(body):
            if isinstance(b, str):
                continue
            if not b.own:
                if any(k == "a" for k, _ in b.all) or _M0.search(b.text):
                    bad.append("%s: %s, outside of the assembly" % (name, b.text))
                continue
            if "mfma" in b.name:
                bad += ["%s: %s, right after %s" % (name, b.text, p.text)
                        for p in _before(body, i, 2)
                        if p.vector and p.written & b.read]
            elif b.name.startswith("buffer_load"):
                bad += ["%s: %s, right after %s" % (name, b.text, p.text)
                        for p in _before(body, i, 5) if p.vector and
                        {r for r in p.written if r[0] == "s"} & b.read]
    return bad, kernels


class assembly_of:
    """The compiler that writes the source's assembly for the GPU, at work."""

    def __init__(self, source: str, flags, hipcc: str = "hipcc"):
        # by way of files: a full pipe would hold the compiler up
        self._out, self._err = tempfile.TemporaryFile(), tempfile.TemporaryFile()
        self._process = subprocess.Popen(
            [hipcc, *flags, "-fPIC", "--offload-device-only", "-S", source, "-o",
             "-"], stdout=self._out, stderr=self._err)

    def text(self) -> str:
        code = self._process.wait()
        for f in (self._out, self._err):
            f.seek(0)
        if code:
            raise RuntimeError(self._err.read().decode())
        return self._out.read().decode()

    def close(self):
        if self._process.poll() is None:
            self._process.kill()
            self._process.wait()
        self._out.close()
        self._err.close()


def check(assembly: assembly_of, source: str, kernels: int):
    """Ends the build where the assembly will not do, or where there are not
    ``kernels`` of these: another way of naming registers would pass unseen."""
    bad, found = faults(assembly.text())
    if found != kernels:
        bad.append("%d kernels name registers, not %d" % (found, kernels))
    if bad:
        raise RuntimeError("\n".join(["%s:" % source] + bad[:20]))
