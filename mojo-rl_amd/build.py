"""Builds libmrl_hip.so for gfx950 with hipcc (cross-compiles without a GPU): one object per
translation unit, compiled side by side, then linked."""
import os
import re
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OBJ = os.path.join(HERE, "build")
LIB = os.path.join(HERE, "libmrl_hip.so")
SOURCES = ["mrl_core.hip", "mrl_env.hip", "mrl_env_many.hip", "mrl_mlp.hip", "mrl_mlp3.hip", "mrl_fb.hip", "mrl_rows.hip", "mrl_ppo.hip", "mrl_policy.hip", "mrl_rollout.hip", "mrl_collect.hip", "mrl_update.hip", "mrl_shuffle.hip"]
# the 16-row collection kernels, a translation unit per hidden width
COLLECT16 = ["mrl_collect%s_h%d.hip" % (k, h) for k in ("16", "_walkers") for h in (256, 128, 64)]
SOURCES = COLLECT16 + SOURCES   # (the longest to compile go first)
# -ffp-contract=off: fp32/fp64 results follow the written order of operations (the GEMM inner
# loops spell out fmaf / MFMA themselves).  The -target-feature pair switches packed-fp32
# code generation off.
FLAGS = ["--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-ffp-contract=off",
         "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-Wno-unused-value"]
# The collection kernels run a long env step inside a loop over the rollout steps.  The machine-level
# loop-invariant code motion lifts the double-precision constants of that step (the polynomial
# coefficients of exp / log / sincos, two registers each) out of the loop into registers of their own,
# the register allocator then spills them, and every use becomes a dependent load from private memory in
# the middle of the solver wavefront's chain.  Without that pass these kernels need no private memory.
# In the stand-alone env kernels the lifted constants push scalar registers out instead.  Where a saved scalar register is
# the first thing in a block, the register allocator of this compiler has been seen to put vector copies next, ahead of the
# instruction that widens the lane mask again, so that lanes outside the mask lose the value.  The flag makes that rarer, it
# does not rule it out: narrow_copies() looks for it in every unit.
EXTRA_FLAGS = {f: ["-mllvm", "-disable-machine-licm"] for f in ["mrl_collect.hip", "mrl_env.hip", "mrl_env_many.hip"] + COLLECT16}


def _run(cmd, verbose):
    if verbose:
        print(" ".join(cmd), flush=True)
    proc = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    out = "\n".join(l for l in proc.stdout.splitlines() if "packed-fp32-ops' is not a recognized feature" not in l)
    if proc.returncode != 0:
        raise RuntimeError("hipcc failed:\n" + out)
    if verbose and out.strip():
        print(out)


def build(verbose=False, incremental=False, jobs=8):
    """Compiles every translation unit (incremental=True: only those older than a source or header
    they could include) and links the library."""
    os.makedirs(OBJ, exist_ok=True)
    headers = [os.path.join(CSRC, f) for f in os.listdir(CSRC) if f.endswith(".hpp")]
    headers.append(os.path.join(HERE, "..", "include", "mrl.h"))
    newest_header = max(os.path.getmtime(h) for h in headers)
    todo, objs = [], []
    for s in SOURCES:
        src, obj = os.path.join(CSRC, s), os.path.join(OBJ, s[:-4] + ".o")
        objs.append(obj)
        fresh = os.path.exists(obj) and os.path.getmtime(obj) > max(os.path.getmtime(src), newest_header)
        if not (incremental and fresh):
            todo.append(["hipcc"] + FLAGS + EXTRA_FLAGS.get(s, []) + ["-c", src, "-o", obj])
    with ThreadPoolExecutor(max_workers=jobs) as pool:
        list(pool.map(lambda c: _run(c, verbose), todo))
    _run(["hipcc", "--offload-arch=gfx950", "-shared", "-fPIC", "-o", LIB] + objs, verbose)
    return LIB


# ---- vector copies ahead of a widening lane mask
# A block where lanes join again opens with exec = exec | saved.  Behind register allocation, before blocks are merged,
# nothing may stand ahead of that but scalar instructions and scalar registers going to and from lanes of a vector register
# (which no mask holds back): a vector copy or a spill there leaves out the lanes that have not joined yet.
_WIDENS = re.compile(r"^\$exec = S_OR_B64(_term)? \$exec\b|= S_OR_SAVEEXEC_B64\b")
_OTHER_EXEC = re.compile(r"^\$exec = |\bimplicit-def (dead )?\$exec\b")
_HARMLESS = re.compile(r"= IMPLICIT_DEF\b|\b(V_READLANE_B32|V_WRITELANE_B32|SI_SPILL_S32_TO_VGPR|SI_RESTORE_S32_FROM_VGPR)\b")


def narrow_copies(lines):
    """(joins, faults) of a unit's machine code behind register allocation, the lines of it."""
    joins, faults, kernel, head, block = 0, [], None, None, None
    for line in lines:
        if line.startswith("name:"):
            kernel = line.split()[1]
        elif line.startswith("  bb."):
            block, head = line.split()[0], []
        elif head is not None and line.startswith("    ") and not line.startswith(("    liveins:", "    successors:")):
            ins = line.strip()
            if _WIDENS.search(ins):
                joins += 1
                faults += [(kernel, block, h) for h in head if re.search(r"\$[va]gpr\d", h) and not _HARMLESS.search(h)]
                head = None
            elif _OTHER_EXEC.search(ins):
                head = None
            else:
                head.append(ins)
    return joins, faults


def check_lane_masks(jobs=8):
    """Compiles every unit up to the end of register allocation; {unit: (joins, faults)}."""
    def one(unit):
        cmd = ["hipcc"] + FLAGS + EXTRA_FLAGS.get(unit, []) + ["--cuda-device-only", "-S", os.path.join(CSRC, unit), "-o", "-",
               "-mllvm", "-stop-after=virtregrewriter,2"]   # (scalar, whole-wavefront and vector registers: three passes)
        with subprocess.Popen(cmd, stdout=subprocess.PIPE, stderr=subprocess.DEVNULL, text=True) as proc:
            found = narrow_copies(proc.stdout)
        if proc.returncode != 0:
            raise RuntimeError("hipcc failed: " + " ".join(cmd))
        return unit, found
    with ThreadPoolExecutor(max_workers=jobs) as pool:
        return dict(pool.map(one, SOURCES))


if __name__ == "__main__":
    print(build(verbose=True, incremental="--incremental" in sys.argv))
    sys.exit(0)
