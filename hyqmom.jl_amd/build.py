"""Build the native libraries in-tree:
  build/libhyqmom_hip.so      the device step, batch kernels, ensemble and warm-start network
                              (hipcc, gfx950; each source compiled in its own process, then linked)
  build/libhyqmom_opcount.so  host build of the cell numerics with FLOP counting (g++)
"""
import glob
import os
import re
import shutil
import subprocess
import sys
import tempfile
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
CXX = os.environ.get("CXX", "g++")
FLAGS = ["-O3", "--offload-arch=gfx950", "-std=c++17", "-fPIC",
         # no packed FP32 instructions: some of their forms have produced wrong results on
         # this hardware without any error
         "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
         # multiply-add fusion within one source expression only: the same cell code then
         # rounds the same way in every kernel it is inlined into (single run, deferred
         # cells, ensemble), which keeps those paths bitwise identical
         "-ffp-contract=on"]
HOST_FLAGS = ["-O2", "-std=c++17", "-fPIC", "-shared", "-ffp-contract=off", "-Wno-unknown-pragmas"]
# (source, object, extra flags): the warm-start network is built once per hidden width
SOURCES = [("hyq_kernels.hip", "hyq_kernels.o", []), ("hyq_ensemble.hip", "hyq_ensemble.o", []),
           ("hyq_ens_fp64.hip", "hyq_ens_fp64.o", []), ("hyq_ens_mixed.hip", "hyq_ens_mixed.o", []),
           ("hyq_ens_newton.hip", "hyq_ens_newton.o", []),
           ("hyq_mlp.hip", "hyq_mlp_h32.o", ["-DHYQ_MLP_HID=32", "-DHYQ_MLP_NS=mlp_h32"]),
           ("hyq_mlp.hip", "hyq_mlp_h128.o", ["-DHYQ_MLP_HID=128", "-DHYQ_MLP_NS=mlp_h128"]),
           ("hyq_mlp_api.hip", "hyq_mlp_api.o", [])]


def _run(cmd, verbose):
    if verbose:
        print(" ".join(cmd), flush=True)
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        sys.stderr.write(r.stderr)
        raise RuntimeError("%s failed" % cmd[0])


def masked_copies(asm):
    """Join blocks of gfx950 assembly whose first vector instructions run before the execution
    mask is restored: [(function, line, instructions)].  The register allocator has placed
    spill copies there, so that only the lanes of the branch before the join were saved and
    the others went on with what the spill slot held.  The joins looked at:
      - the end of an if: the target of s_cbranch_execz, or the block after one that began by
        narrowing the mask and has no branch over it;
      - the end of a loop: the block after `s_andn2_b64 exec` (or s_xor, a loop over the
        distinct values of a register) and s_cbranch_execnz, where no lane is left;
      - an else: a block that ends the then side with s_or_saveexec.  What the then side's
        lanes bring along (v_mov) belongs before it, so only spill copies count there."""
    copy = re.compile(r"(v_accvgpr_|scratch_)")
    vector = re.compile(r"(v_(?!writelane|readlane)|scratch_|global_|flat_|ds_|buffer_)")
    lines = asm.split("\n")
    targets = set(re.findall(r"s_cbranch_execz (\.LBB\d+_\d+)", asm))
    found, fn, last, before = [], None, "", ""
    narrowed = restored = False  # the block began right after the mask was narrowed; it was widened again
    for i, line in enumerate(lines):
        m = re.match(r"^([A-Za-z_]\S*):\s", line)
        if m:
            fn, narrowed = m[1], False
        label, fall = re.match(r"^(\.LBB\d+_\d+):", line), re.match(r"^; %bb\.\d+:", line)
        if label or fall:
            loop_end = last.startswith("s_cbranch_execnz") and re.match(r"s_(andn2|xor)_b64 exec, exec", before)
            if (label and label[1] in targets) or (fall and narrowed and not restored) or loop_end:
                vec = []
                for t in lines[i + 1:]:
                    if t.startswith((".LBB", ".Lfunc", "; %bb")):
                        break
                    t = t.split(";")[0].strip()
                    if re.match(r"s_or_b64 exec, exec|s_mov_b64 exec, (s\[|vcc)|s_or_saveexec", t):
                        if t.startswith("s_or_saveexec"):
                            vec = [v for v in vec if copy.match(v)]
                        if vec:
                            found.append((fn, i + 1, vec))
                        break
                    if "exec" in t or re.match(r"s_(cbranch|branch|swappc|endpgm|setpc)", t):
                        break
                    if vector.match(t):
                        vec.append(t)
            narrowed = bool(re.match(r"s_and_saveexec|s_andn?2?_b64 exec", last))
            restored = False
        t = line.split(";")[0].strip()
        if t and not line.startswith((".", ";")):
            last, before = t, last
            restored = restored or bool(re.match(r"s_(or|mov)_b64 exec", t))
    return found


def _compile(cmd, obj, verbose):
    """One object, with its assembly checked for masked_copies."""
    tmp = tempfile.mkdtemp(dir=os.path.dirname(obj))
    try:
        part = os.path.join(tmp, os.path.basename(obj))
        _run(cmd[:cmd.index("-o") + 1] + [part] + cmd[cmd.index("-o") + 2:] + ["-save-temps=obj"], verbose)
        asm = glob.glob(os.path.join(tmp, "*gfx950*.s"))
        if not asm:
            raise RuntimeError("no device assembly of %s" % obj)
        for f in asm:
            with open(f) as fh:
                bad = masked_copies(fh.read())
            if bad:
                raise RuntimeError("%s: spill copies under a partial execution mask: %s" % (obj, bad))
        os.replace(part, obj)
    finally:
        shutil.rmtree(tmp, ignore_errors=True)


def build(verbose=True):
    out = os.path.join(HERE, "build")
    os.makedirs(out, exist_ok=True)
    objs = [os.path.join(out, o) for _, o, _ in SOURCES]
    cmds = [[HIPCC] + FLAGS + extra + ["-c", "-o", o, os.path.join(HERE, "csrc", f)]
            for (f, _, extra), o in zip(SOURCES, objs)]
    with ThreadPoolExecutor(len(cmds)) as ex:
        list(ex.map(lambda c, o: _compile(c, o, verbose), cmds, objs))
    target = os.path.join(out, "libhyqmom_hip.so")
    _run([HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", target + ".tmp"] + objs, verbose)
    os.replace(target + ".tmp", target)
    oc = os.path.join(out, "libhyqmom_opcount.so")
    _run([CXX] + HOST_FLAGS + ["-o", oc + ".tmp", os.path.join(HERE, "csrc", "hyq_opcount.cpp")], verbose)
    os.replace(oc + ".tmp", oc)
    return target


if __name__ == "__main__":
    build()
