"""Check of compiled kernels for one register-allocation fault of the compiler.

Where lanes rejoin after a branch the block opens by widening the execution
mask (``s_andn2_saveexec``, ``s_or_b64 exec``).  When scalar registers are
short the compiler first puts scalar reloads at the head of that block; it then
no longer takes the mask update for the block's prologue, and the copies and
spills of vector registers that it splits later land before the update, where
only the lanes of the branch execute them.  The other lanes keep stale values:
the 64-lane Levenberg-Marquardt kernel of a 14-parameter plug-in lost the base
point's 1F1 values so, which spoiled the Jacobian columns of the parameters
behind them and rejected most steps, with no error.  A block that a branch on an
empty mask reaches can hold no vector instruction before its mask update for any
other reason, so that is what is looked for.  (Not seen: a branch left out because
its code is short, or too far for a direct jump.)
"""
import os
import re
import subprocess
import tempfile

LLVM = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin")
_WIDEN = ("s_andn2_saveexec_b64", "s_or_saveexec_b64", "s_orn2_saveexec_b64")
_VECTOR = ("v_", "scratch_", "buffer_", "flat_", "global_", "ds_")
_ANY_MASK = ("v_readlane", "v_writelane", "v_readfirstlane", "v_cmp")
_LABEL = re.compile(r"<(L\d+)>:$")


def misplaced(lines):
    """(function, label, vector instruction, mask update) of every block of a
    disassembly (llvm-objdump --symbolize-operands) that has the fault."""
    found, heads, targets = [], {}, set()
    func = label = vec = None

    def close():
        found.extend((func, l) + h for l, h in heads.items() if l in targets)
        heads.clear()
        targets.clear()

    for line in lines:
        if line.startswith("<"):
            m = _LABEL.match(line.rstrip())
            if m:
                label, vec = m.group(1), None
            else:
                close()
                func, label = line.split(">")[0][1:], None
            continue
        s = line.split("//")[0].strip()
        if not s:
            continue
        op = s.split(None, 1)[0]
        if op == "s_cbranch_execz":
            targets.add(s.split()[1])
            label = None
        elif label is None:
            continue
        elif op in _WIDEN or s.startswith("s_or_b64 exec, exec,"):
            if vec:
                heads[label] = (vec, s)
            label = None
        elif op.startswith(("s_cbranch", "s_branch", "s_setpc", "s_endpgm")) or "exec" in s:
            label = None
        elif vec is None and op.startswith(_VECTOR) and not op.startswith(_ANY_MASK):
            vec = s
    close()
    return found


def misplaced_in_object(obj, arch):
    """misplaced() of the device code in a HIP object file ([] without any)."""
    tool = lambda t: os.path.join(LLVM, t)
    with tempfile.TemporaryDirectory() as d:
        fat, co = os.path.join(d, "fat"), os.path.join(d, "co")
        subprocess.run([tool("llvm-objcopy"), "--dump-section=.hip_fatbin=" + fat, obj, os.path.join(d, "o")],
                       capture_output=True)
        if not os.path.exists(fat):
            return []
        subprocess.run([tool("clang-offload-bundler"), "--unbundle", "--type=o", "--input=" + fat, "--output=" + co,
                        "--targets=hipv4-amdgcn-amd-amdhsa--" + arch], check=True, capture_output=True)
        p = subprocess.Popen([tool("llvm-objdump"), "-d", "--symbolize-operands", "--no-show-raw-insn",
                              "--no-leading-addr", co], stdout=subprocess.PIPE, stderr=subprocess.DEVNULL, text=True)
        found = misplaced(p.stdout)
        if p.wait() != 0:
            raise RuntimeError("llvm-objdump failed on the device code of " + obj)
        return found
