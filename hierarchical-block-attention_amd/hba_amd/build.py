"""Build libhba_amd.so (the C-ABI + HIP kernels) in-tree for gfx950.

    python -m hba_amd.build        (from hierarchical-block-attention_amd/)

Each csrc/*.hip is compiled to an object under ../_build/ (in parallel), its
assembly checked for register spills that lose lanes (lost_spills), then linked
into hba_amd/libhba_amd.so next to this file.
"""
import concurrent.futures as cf
import glob
import os
import re
import subprocess
import tempfile

HERE = os.path.dirname(os.path.abspath(__file__))
PKG_ROOT = os.path.dirname(HERE)
CSRC = os.path.join(PKG_ROOT, "csrc")
OBJ_DIR = os.path.join(PKG_ROOT, "_build")
LIB_PATH = os.path.join(HERE, "libhba_amd.so")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = "gfx950"

FLAGS = [
    f"--offload-arch={ARCH}", "-O3", "-std=c++17", "-fPIC",
    # every a*b+c is two roundings unless written as fmaf(): the selection
    # kernels reproduce a declared fp32 operation order bit for bit
    "-ffp-contract=off",
    # no packed-fp32 VALU instructions
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
]


# s_or_b64 exec, exec, s[..] and the like: lanes that a branch or a finished
# loop had switched off run again
_WIDEN = re.compile(r"s_or_b64 exec, exec,|s_or_saveexec_b64|s_andn2_saveexec_b64|s_xor_b64 exec, exec,|s_mov_b64 exec,")
_EXEC = re.compile(r"s_\w*saveexec_b64|s_\w+ exec,")
_VECTOR = re.compile(r"(?!v_readlane|v_writelane|v_readfirstlane)(?:v|ds|global|buffer|scratch|flat)_")


def lost_spills(asm):
    """(line number, kernel, instruction) of the vector instructions that come
    before a block's exec restore: lanes that skipped the branch, and after a
    divergent loop all of them, do not execute them.

    The register allocator puts spills and copies at the start of a block and
    has put them before the restore there.  An earlier form of the bf16 query
    gradient, with 16 VGPRs spilled, lost the head index of its LSE rows so: a
    `scratch_store` between `s_cbranch_execnz` (the loop's exit, exec = 0) and
    `s_or_b64 exec, exec`, reloaded 2000 lines later with every lane on.  Within
    a block that no branch reaches, instructions before a restore are the
    branch's own; there only spills count."""
    lines = asm.splitlines()
    targets = {m.group(1) for m in map(re.compile(r"\s+s_cbranch_execz (\S+)").match, lines) if m}
    found, kernel, before, join, last = [], "", [], False, ""
    for no, line in enumerate(lines, 1):
        s = line.strip()
        label = re.match(r"(\.?\w+):", line)
        if label and not label.group(1).startswith("."):
            kernel, before, join = label.group(1), [], False
        elif label or s.startswith("; %bb."):
            before = []
            join = bool(label) and label.group(1) in targets or last.startswith("s_cbranch_execnz")
        elif s and s[0] not in ";.":
            if _EXEC.match(s):
                if _WIDEN.match(s):
                    found += [x for x in before if join or "Folded Spill" in x[2]
                              or ("v_accvgpr_write" in x[2] and "Reload Reuse" in x[2])]
                before, join = [], False
            elif _VECTOR.match(s):
                before.append((no, kernel, s))
            last = s
    return found


def _compile(src):
    name = os.path.basename(src)[:-len(".hip")]
    obj = os.path.join(OBJ_DIR, name + ".o")
    with tempfile.TemporaryDirectory(dir=OBJ_DIR) as tmp:
        out = os.path.join(tmp, name + ".o")
        r = subprocess.run([HIPCC, *FLAGS, "-save-temps=obj", "-c", src, "-o", out], capture_output=True, text=True)
        if r.returncode != 0:
            raise RuntimeError(f"hipcc failed on {src}:\n{r.stderr}")
        asm, = glob.glob(os.path.join(tmp, f"{name}-hip-*{ARCH}.s"))
        with open(asm) as f:
            lost = lost_spills(f.read())
        if lost:
            raise RuntimeError(f"{src}: the compiler placed vector instructions before an exec restore, where not "
                               "every lane executes them; lower the kernel's register pressure:\n" +
                               "\n".join(f"  {k}, line {no}: {s}" for no, k, s in lost[:8]))
        os.replace(out, obj)
    return obj


def build(verbose=False):
    """Compile every kernel source and link the shared library; returns its path."""
    os.makedirs(OBJ_DIR, exist_ok=True)
    srcs = sorted(glob.glob(os.path.join(CSRC, "*.hip")))
    with cf.ThreadPoolExecutor(max_workers=min(8, len(srcs))) as ex:
        objs = list(ex.map(_compile, srcs))
    tmp = LIB_PATH + ".tmp%d" % os.getpid()
    cmd = [HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", tmp, *objs]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stderr}")
    os.replace(tmp, LIB_PATH)
    if verbose:
        print(LIB_PATH)
    return LIB_PATH


if __name__ == "__main__":
    build(verbose=True)
