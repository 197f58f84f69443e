"""Builds libmi355attn.so (the C-ABI HIP library) for gfx950 with hipcc.

Usage: python build.py            (from anywhere; output lands next to the
Python package so the built library travels with the source tree)
       python build.py --serving  (libmi355attn_serving.so: what serving a model needs and no more --
no training kernels, no checks of the compiler's output; the command line tools run this in a
checkout that has no library yet)
"""
from __future__ import annotations

import os
import re
import subprocess
import sys
import tempfile
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OUT_DIR = os.path.join(HERE, "mi355_attn")
LIB_NAME = "libmi355attn.so"
SERVING_LIB_NAME = "libmi355attn_serving.so"      # without the kernels that only training needs
CALLS_NAME = "_calls.so"                          # ... nor these
TRAINING_ONLY = ("prefill_bwd.hip", "prefill_bwd_short.hip")
SOURCES = ["api.hip", "paged_decode.hip", "prefill_fwd.hip", "prefill_fwd_w64.hip", "prefill_short.hip", "prefill_keys.hip", "prefill_bwd.hip", "prefill_bwd_short.hip", "kv_cache_ops.hip",
           "layer_ops.hip", "paged_attn_any.hip", "ssm_ops.hip", "moe_ops.hip", "rows_linear.hip"]
# prefill_fwd_w64.hip keeps its output accumulators in AGPRs that only its assembly statements touch: its builtin MFMAs
# must therefore be selected in VGPR form, so that the compiler allocates no AGPR for them.
# It is also compiled without the machine-code hoisting of loop invariants: hoisted out of the job loop, a few dozen
# per-lane addresses stayed live across the assembly loop (which owns most vector registers) and pushed the
# prefetched query rows into scratch memory, whose reloads wait for every load in flight.
EXTRA_FLAGS = {"prefill_fwd_w64.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form=1", "-mllvm", "-disable-machine-licm"],
               # prefill_bwd.hip orders its LDS reads and MFMAs by hand (reads two MFMAs ahead, a scheduling barrier after
               # every MFMA); the scheduler that runs after register allocation undoes part of that: 1.5 % (measured).
               # Its kernel on wavefronts of 64 keys has all AGPRs in inline assembly, so the compiler's own MFMAs are in VGPR form.
               "prefill_bwd.hip": ["-mllvm", "-enable-post-misched=0", "-mllvm", "-amdgpu-mfma-vgpr-form=1"]}

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC",
    "-fno-gpu-rdc", "-Wall", "-Wno-unused-function",
    # packed-fp32 VALU forms are kept off for every device pass
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
]


def _run(cmd):
    r = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    out = "\n".join(l for l in r.stdout.splitlines() if "packed-fp32-ops" not in l)
    if r.returncode != 0:
        raise RuntimeError("command failed: %s\n%s" % (" ".join(cmd), out))
    return out


def library_path() -> str:
    return os.path.join(OUT_DIR, LIB_NAME)


def check_w64_registers() -> str:
    """prefill_fwd_w64.hip keeps values in a[0:N_AGPRS-1] across its assembly statements, behind the compiler's back:
    the statements name those registers as clobbered, so the compiler holds nothing of its own in them ACROSS a
    statement, but nothing in the language keeps it from using one BETWEEN two statements (as a spill slot, say).
    This compiles the file to assembly and fails the build if any instruction outside the statements touches one."""
    n_agprs = 0
    with open(os.path.join(CSRC, "prefill_w64_asm.inc")) as f:
        for line in f:
            if line.startswith("#define W64_CLOBBER_ACC"):
                n_agprs = line.count('"a')
    if n_agprs == 0:
        raise RuntimeError("prefill_w64_asm.inc: no W64_CLOBBER_ACC")
    with tempfile.TemporaryDirectory() as tmp:
        asm = os.path.join(tmp, "w64.s")
        _run([HIPCC, *FLAGS, *EXTRA_FLAGS["prefill_fwd_w64.hip"], "-S", "--cuda-device-only",
              os.path.join(CSRC, "prefill_fwd_w64.hip"), "-o", asm])
        inside, bad = False, []
        with open(asm) as f:
            for no, line in enumerate(f, 1):
                if "#ASMSTART" in line:
                    inside = True
                elif "#ASMEND" in line:
                    inside = False
                elif not inside and not line.lstrip().startswith((";", ".")):
                    for m in re.finditer(r"\ba\[(\d+):\d+\]|\ba(\d+)\b", line.split(";")[0]):
                        if int(m.group(1) or m.group(2)) < n_agprs:
                            bad.append("%d: %s" % (no, line.strip()))
        if bad:
            raise RuntimeError("prefill_fwd_w64.hip: compiler-generated code touches AGPRs below a%d, which the "
                               "assembly statements own:\n%s" % (n_agprs, "\n".join(bad[:20])))
    return "prefill_fwd_w64.hip: no compiler-generated instruction touches a[0:%d]" % (n_agprs - 1)


_SREG = re.compile(r"\bs\[(\d+):(\d+)\]|\bs(\d+)\b")


def _sregs(text):
    out = set()
    for m in _SREG.finditer(text):
        if m.group(3) is not None:
            out.add(int(m.group(3)))
        else:
            out.update(range(int(m.group(1)), int(m.group(2)) + 1))
    return out


def issues_memory_from_assembly(src: str) -> bool:
    """Whether kernels of `src` have inline-assembly memory instructions, of their own or through a header's."""
    with open(os.path.join(CSRC, src)) as f:
        text = f.read()
    if re.search(r'\bdma_to_lds_\w+\(|"[^"\n]*\b(global|buffer|flat|scratch)_(load|store|atomic)', text):
        return True
    # (common.hpp defines the direct-to-LDS loads; who calls them is what counts)
    return any(issues_memory_from_assembly(h) for h in re.findall(r'^#include "(\w+\.hpp)"', text, re.M) if h != "common.hpp")


def check_scalar_address_hazards(src: str) -> str:
    """gfx9 wants five wait states between a VECTOR instruction that writes a scalar register (v_readlane restoring a
    spilled value, v_readfirstlane, a compare or a carry-out) and a vector-memory instruction that reads that register
    as its address.  The compiler inserts them for the instructions it emits, but it cannot see inside an
    inline-assembly statement, and the direct-to-LDS loads of these kernels live in such statements.  This compiles
    `src` to assembly and fails the build if a memory instruction inside a statement reads a scalar register that a
    vector instruction wrote fewer than five wait states earlier on the straight-line path in front of it."""
    with tempfile.TemporaryDirectory() as tmp:
        asm = os.path.join(tmp, "k.s")
        _run([HIPCC, *FLAGS, *EXTRA_FLAGS.get(src, []), "-S", "--cuda-device-only", os.path.join(CSRC, src), "-o", asm])
        lines = open(asm).read().splitlines()
    bad, inside, n_checked = [], False, 0
    code = []                     # (line number, text) of instructions, in order
    for no, raw in enumerate(lines, 1):
        text = raw.split(";")[0].strip()
        if "#ASMSTART" in raw:
            inside = True
            continue
        if "#ASMEND" in raw:
            inside = False
            continue
        if not text or text.startswith(".") or text.endswith(":"):
            continue
        code.append((no, text, inside))
    for i, (no, text, in_asm) in enumerate(code):
        op = text.split()[0]
        if not in_asm or not op.startswith(("global_", "buffer_", "flat_", "scratch_")):
            continue
        addr = _sregs(text)
        if not addr:
            continue
        n_checked += 1
        states, j = 0, i - 1
        while j >= 0 and states < 5:
            _, prev, _ = code[j]
            pop = prev.split()[0]
            if pop == "s_nop":
                states += int(prev.split()[1], 0) + 1
            else:
                # destination operands of a vector instruction: everything in front of the first source; an SGPR
                # there (v_readlane sN, v_cmp_* s[a:b], the carry-out of v_mad_u64_u32 / v_add_co) is a vector write
                if pop.startswith("v_"):
                    ops = prev[len(pop):].split(",")
                    n_dst = 2 if pop.startswith(("v_mad_u64", "v_mad_i64", "v_add_co", "v_sub_co", "v_addc", "v_subb",
                                                  "v_div_scale")) else 1
                    written = set()
                    for o in ops[:n_dst]:
                        written |= _sregs(o)
                    if written & addr:
                        bad.append("%s:%d: `%s` reads s%s, written %d wait state(s) earlier by `%s`"
                                   % (src, no, text, sorted(written & addr), states, prev))
                        break
                states += 1
            j -= 1
    if n_checked == 0:
        raise RuntimeError("%s: no memory instruction found in inline assembly" % src)
    if bad:
        raise RuntimeError("scalar address hazard in inline assembly:\n" + "\n".join(bad[:20]))
    return "%s: %d inline-assembly memory instructions, none reads a scalar register within five wait states of a vector write" % (src, n_checked)


_VREG = re.compile(r"\b([va])(?:\[(\d+):(\d+)\]|(\d+)\b)")


def _vregs(text):
    out = set()
    for m in _VREG.finditer(text):
        first, last = (int(m.group(4)),) * 2 if m.group(4) else (int(m.group(2)), int(m.group(3)))
        out.update(m.group(1) + str(i) for i in range(first, last + 1))
    return out


_TRANS = ("v_exp_", "v_log_", "v_rcp_", "v_rsq_", "v_sqrt_", "v_sin_", "v_cos_")


def asm_hazards(lines):
    """Vector instructions in inline assembly (`lines` of compiler output), whose wait states the compiler does not see to: (MFMAs, others, what is wrong).  On
    the straight-line path in front of each: an MFMA may read a register two wait states after a vector instruction wrote it, another one's operand may come
    from a transcendental instruction two instructions earlier, and an MFMA's result is there eleven states behind one of eight passes (it counts as one
    state here, and takes eight), for the compiler's instructions too where the MFMA is in assembly."""
    code, inside, bad, n_mfma, n_other = [], False, [], 0, 0
    for no, raw in enumerate(lines, 1):
        if "#ASMSTART" in raw or "#ASMEND" in raw:
            inside = "#ASMSTART" in raw
            continue
        text = raw.split(";")[0].strip()
        if text and not text.startswith(".") and not text.endswith(":"):
            ops = text.split(None, 1)[1].split(",") if " " in text or "\t" in text else []
            code.append((no, text.split()[0], ops, inside))
    for i, (no, op, ops, in_asm) in enumerate(code):
        own, other = in_asm and op.startswith("v_mfma"), in_asm and op.startswith("v_") and not op.startswith("v_mfma")
        n_mfma += own
        n_other += other
        reads = _vregs(",".join(ops[1:] if own else ops)) if own or other or not in_asm else set()
        states, j = 0, i - 1
        while reads and j >= 0 and states < (2 if own else 11):
            _, prev, prev_ops, prev_asm = code[j]
            written = _vregs(prev_ops[0]) if prev.startswith("v_") and prev_ops else set()
            mfma = prev.startswith("v_mfma")
            if written & reads and (not mfma if own else mfma and (prev_asm or other) and not op.startswith("v_mfma") or other and states < 1 and prev.startswith(_TRANS)):
                bad.append("%d: %s reads or writes %s, written %d wait state(s) earlier by %s" % (no, op, sorted(written & reads)[:4], states, prev))
                break
            states += int(prev_ops[0], 0) + 1 if prev == "s_nop" else 1
            j -= 1
    return n_mfma, n_other, bad


def scratch_before_products(lines, kernel):
    """Accesses to scratch memory in `kernel` (a part of its symbol) from which an MFMA can still be reached: what the loop spills.  None where there is no such
    kernel or it has no MFMA."""
    code, labels, inside = [], {}, False
    for no, raw in enumerate(lines, 1):
        text = raw.split(";")[0].strip()
        if text.endswith(":") and not text.startswith(".L"):
            inside = kernel in text
        elif text.startswith(".Lfunc_end") and inside:
            break
        if not inside:
            continue
        if text.endswith(":"):
            labels[text[:-1]] = len(code)
        elif text and not text.startswith("."):
            code.append((no, text))
    if not any(text.startswith("v_mfma") for _, text in code):
        return None
    follows = [[] for _ in code]                   # instruction -> those that come in front of it
    for i, (_, text) in enumerate(code):
        op = text.split()[0]
        to = [] if op in ("s_branch", "s_endpgm") else [i + 1]
        if op == "s_branch" or op.startswith("s_cbranch"):
            to.append(labels[text.split()[1]])
        for j in to:
            if j < len(code):
                follows[j].append(i)
    reach, todo = set(), [i for i, (_, text) in enumerate(code) if text.startswith("v_mfma")]
    while todo:
        for i in follows[todo.pop()]:
            if i not in reach:
                reach.add(i)
                todo.append(i)
    return ["%d: %s" % (no, text) for i, (no, text) in enumerate(code) if text.startswith("scratch_") and i in reach]


def check_wide_backward() -> str:
    """bwd_dkv_wide_kernel has MFMAs and conversions in inline assembly, and all registers taken: no hazard of theirs, and nothing spilled before the last product,
    where a reload would wait for all rows that are on their way."""
    src = "prefill_bwd.hip"
    with tempfile.TemporaryDirectory() as tmp:
        asm = os.path.join(tmp, "k.s")
        _run([HIPCC, *FLAGS, *EXTRA_FLAGS.get(src, []), "-S", "--cuda-device-only", os.path.join(CSRC, src), "-o", asm])
        lines = open(asm).read().splitlines()
    n_mfma, n_other, bad = asm_hazards(lines)
    if n_mfma < 2 * 64 or n_other < 2 * 64:                           # (two instances: dV, dV and dK, dK of a step; P and dS of two steps)
        raise RuntimeError("%s: %d MFMAs and %d other vector instructions found in inline assembly" % (src, n_mfma, n_other))
    if bad:
        raise RuntimeError("hazards in inline assembly of %s:\n" % src + "\n".join(bad[:20]))
    for mode in (0, 1):
        spilled = scratch_before_products(lines, "bwd_dkv_wide_kernelILi%dE" % mode)
        if spilled is None or spilled:
            raise RuntimeError("%s: bwd_dkv_wide_kernel<%d> %s" % (src, mode, "not found" if spilled is None else "spills in its loop:\n" + "\n".join(spilled[:20])))
    return "%s: %d MFMAs and %d other vector instructions in inline assembly without a hazard, nothing spilled before the last product" % (src, n_mfma, n_other)


def _compile_all(srcs, tag=""):
    """Objects of `srcs`, compiled in parallel: [(object, compiler messages)]."""
    obj_dir = os.path.join(HERE, "build")
    os.makedirs(obj_dir, exist_ok=True)

    def compile_one(src):
        obj = os.path.join(obj_dir, src.replace(".hip", tag + ".o"))
        log = _run([HIPCC, *FLAGS, *EXTRA_FLAGS.get(src, []), "-c", os.path.join(CSRC, src), "-o", obj])
        return obj, log

    with ThreadPoolExecutor(max_workers=8) as ex:
        return list(ex.map(compile_one, srcs))


# ---- the operators' calls from Python (host code against torch, in front of the library) ----
def compile_calls() -> str:
    import sysconfig
    import torch
    root = os.path.dirname(torch.__file__)
    obj = os.path.join(HERE, "build", "calls.o")
    os.makedirs(os.path.dirname(obj), exist_ok=True)
    includes = [os.path.join(root, "include"), os.path.join(root, "include", "torch", "csrc", "api", "include"),
                os.path.join(os.path.dirname(os.path.dirname(HIPCC)), "include"), sysconfig.get_paths()["include"]]
    _run(["g++", "-O2", "-std=c++17", "-fPIC", "-Wall", "-Wno-sign-compare", "-D__HIP_PLATFORM_AMD__", "-DUSE_ROCM",
          "-D_GLIBCXX_USE_CXX11_ABI=%d" % torch._C._GLIBCXX_USE_CXX11_ABI, *[x for d in includes for x in ("-isystem", d)],
          "-c", os.path.join(CSRC, "calls.cpp"), "-o", obj])
    return obj


def link_calls(obj) -> str:
    import torch
    out = os.path.join(OUT_DIR, CALLS_NAME)
    _run(["g++", "-shared", "-o", out, obj, "-L" + OUT_DIR, "-l:" + LIB_NAME, "-Wl,-rpath,$ORIGIN",
          "-L" + os.path.join(os.path.dirname(torch.__file__), "lib"), "-ltorch_python", "-ltorch_cpu", "-lc10", "-lc10_hip"])
    return out


def build_serving_library() -> str:
    tag = ".%d" % os.getpid()                      # (two first calls at once each build their own and the last one stays)
    objs = [o for o, _ in _compile_all([s for s in SOURCES if s not in TRAINING_ONLY], tag)]
    lib = os.path.join(OUT_DIR, SERVING_LIB_NAME)
    _run([HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", lib + tag, *objs])
    os.replace(lib + tag, lib)
    for o in objs:
        os.remove(o)
    return lib


def build_library(verbose: bool = True) -> str:
    # the hand-scheduled assembly of prefill_fwd_w64.hip is generated text: regenerate it so that it cannot go stale
    _run([sys.executable, os.path.join(CSRC, "gen_prefill_w64_loop.py")])
    srcs = [s for s in SOURCES if os.path.exists(os.path.join(CSRC, s))]

    with ThreadPoolExecutor(max_workers=5) as ex:
        calls = ex.submit(compile_calls)
        check = ex.submit(check_w64_registers)
        hazards = [ex.submit(check_scalar_address_hazards, s) for s in srcs if issues_memory_from_assembly(s)]
        hazards.append(ex.submit(check_wide_backward))
        results = _compile_all(srcs)
        notes = [check.result()] + [h.result() for h in hazards]
    if verbose:
        print("\n".join(notes))
    for _, log in results:
        if verbose and log.strip():
            print(log)
    lib = library_path()
    _run([HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", lib, *[o for o, _ in results]])
    link_calls(calls.result())
    if verbose:
        print("built", lib)
    return lib


if __name__ == "__main__":
    if "--serving" in sys.argv[1:]:
        build_serving_library()
    else:
        build_library()
    sys.exit(0)
