"""The gfx950 assembly of the library's own kernels, for the tests that pin
what the compiler made of them: compiled here from csrc/ with the Makefile's
flags."""
import functools
import os
import re
import shlex
import subprocess

PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "kandinsky.cpp_amd")


def _flags(source):
    """The compiler and flags that the Makefile builds `source` with."""
    out = subprocess.run(["make", "-n", "-B", "-C", PKG, "libkd_fa.so"], check=True, capture_output=True, text=True).stdout
    for line in out.splitlines():
        words = shlex.split(line.split(" && ")[0])
        if words and "hipcc" in words[0] and source in words:
            return words[:words.index("-shared" if "-shared" in words else "-c")]
    raise AssertionError(f"the Makefile does not build {source}")


@functools.lru_cache(maxsize=None)
def kernels(source):
    """{mangled name: lines} of every kernel of csrc/`source`: labels end in
    ':', comments without an instruction stay (asm blocks hold markers)."""
    cmd = _flags("csrc/" + source) + ["--cuda-device-only", "-S", "csrc/" + source, "-o", "-"]
    text = subprocess.run(cmd, cwd=PKG, check=True, capture_output=True, text=True).stdout
    found, name = {}, None
    for line in text.splitlines():
        m = re.match(r"(_Z\w+):", line)
        if m:
            name, found[m.group(1)] = m.group(1), []
        elif line.startswith(".Lfunc_end"):
            name = None
        elif name and line.strip():
            found[name].append(re.sub(r"\s+;.*", "", line).strip() if not line.strip().startswith(";") else line.strip())
    return {k: v for k, v in found.items() if any(ln.startswith("s_endpgm") for ln in v)}


def successors(lines):
    """For each line, the indexes that control may reach next."""
    at = {ln[:-1]: i for i, ln in enumerate(lines) if ln.startswith(".L") and ln.endswith(":")}
    out = []
    for i, ln in enumerate(lines):
        op, _, rest = ln.partition(" ")
        if op.split("\t")[0] == "s_endpgm":
            out.append([])
        elif op.split("\t")[0] == "s_branch":
            out.append([at[ln.split()[1]]])
        elif op.startswith("s_cbranch"):
            out.append([i + 1, at[ln.split()[1]]])
        else:
            out.append([i + 1] if i + 1 < len(lines) else [])
    return out
