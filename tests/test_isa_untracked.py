"""The decode split kernel loads q, the norm weights and the new row with
untracked (inline-asm) vector loads issued ahead of the tile DMA, and awaits
them with one `s_waitcnt vmcnt(D*RPW)` that names their registers.  The
compiler does not know those registers are pending until that wait: any
instruction that touches them in between would read or clobber data still in
flight.  This CPU test compiles decode.hip for gfx950 (the library's flags) and
checks the generated assembly along every control-flow path (branches
followed, so the early return of a slice with no positions is covered as well
as the tile loop) for such an instruction, and that the first vector-memory
wait after the loads leaves the tile DMAs in flight.
"""
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "lfm2-ampere_amd")
HIPCC = "/opt/rocm/bin/hipcc"
FLAGS = ["--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang", "-target-feature", "-Xclang",
         "-packed-fp32-ops", "-DLK_ATTN_SPLIT=256", "-DLK_ATTN_TARGET_N=16", "-DLK_ATTN_SPLIT_MIN=8",
         "-DLK_DEC_TILE=16", "-DLK_DEC_NBUF=4", "-DLK_DEC_ABLATE=0"]


def _vregs(text):
    out = set()
    for m in re.finditer(r"\bv\[(\d+):(\d+)\]|\bv(\d+)\b", text):
        if m.group(3):
            out.add(int(m.group(3)))
        else:
            out.update(range(int(m.group(1)), int(m.group(2)) + 1))
    return out


def _check_paths(name, body):
    """Dataflow over the kernel's instructions: the set of registers of
    untracked loads still in flight at each instruction, joined over every
    path that reaches it; any instruction other than a vector-memory wait that
    names one of them is a hazard.  Returns (number of untracked loads, vmcnt
    of the first wait that retires them)."""
    ins, labels = [], {}
    in_asm = False
    for l in body:
        if l.startswith(";;#ASMSTART"):
            in_asm = True
            continue
        if l.startswith(";;#ASMEND"):
            in_asm = False
            continue
        m = re.match(r"^(\.?[A-Za-z_][\w.$]*):", l)
        if m:
            labels[m.group(1)] = len(ins)
            continue
        if l.startswith(";") or not l or (l.startswith(".") and not in_asm):
            continue
        ins.append((l.split(";")[0].strip(), in_asm))
    loads = sum(1 for t, a in ins if a and t.startswith("global_load_dwordx4") and "lds" not in t)
    state = [None] * (len(ins) + 1)
    state[0] = frozenset()
    work, first_wait = [0], None
    while work:
        k = work.pop()
        if k >= len(ins):
            continue
        t, a = ins[k]
        pend = state[k]
        op = t.split()[0]
        if a and op == "global_load_dwordx4" and "lds" not in t:
            out = pend | _vregs(t.split(None, 1)[1].split(",")[0])
        elif "vmcnt(" in t:
            if pend and first_wait is None:
                first_wait = int(re.search(r"vmcnt\((\d+)\)", t).group(1))
            out = frozenset()
        else:
            hit = _vregs(t) & pend
            assert not hit, "%s: %s touches registers of loads in flight %s" % (name, t, sorted(hit))
            out = pend
        succ = []
        if op == "s_endpgm":
            succ = []
        elif op == "s_branch":
            succ = [labels[t.split()[1]]]
        elif op.startswith("s_cbranch"):
            succ = [k + 1, labels[t.split()[1]]]
        else:
            succ = [k + 1]
        for j in succ:
            new = out if state[j] is None else (state[j] | out)
            if state[j] is None or new != state[j]:
                state[j] = new
                work.append(j)
    return loads, first_wait


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not installed")
def test_untracked_loads_untouched_until_their_wait(tmp_path):
    asm = tmp_path / "decode.s"
    subprocess.run([HIPCC, *FLAGS, "--offload-device-only", "-S", "-x", "hip",
                    os.path.join(PKG, "csrc", "decode.hip"), "-o", str(asm)],
                   check=True, cwd=PKG, capture_output=True)
    txt = asm.read_text()
    for fused in (0, 1):
        name = "_Z15lk_k_attn_splitILb%dE" % fused
        i = txt.index("\n" + name) + 1
        body = [l.strip() for l in txt[i:txt.index(".Lfunc_end", i)].split("\n")]
        loads, first_wait = _check_paths(name, body)
        assert loads == (20 if fused else 4), (name, loads)
        # D = 3 tiles of RPW = 4 rows per wave stay in flight
        assert first_wait == 12, (name, first_wait)


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not installed")
def test_untracked_loads_with_the_makefiles_own_flags(tmp_path):
    """The same on the command line the Makefile builds decode.hip with
    (kernel-argument preload included), whatever its flags become."""
    cmd = next(l for l in subprocess.run(["make", "-n", "-B", "_build/decode.hip.o"], cwd=PKG, check=True,
                                         capture_output=True, text=True).stdout.split("\n") if " -c -x hip " in l)
    args = cmd.split(" 2>&1")[0].replace("-c -x hip", "--offload-device-only -S -x hip").split()
    asm = tmp_path / "decode.s"
    args[args.index("-o") + 1] = str(asm)
    subprocess.run(args, check=True, cwd=PKG, capture_output=True)
    txt = asm.read_text()
    assert "kernarg_preload_length" in txt
    for fused in (0, 1):
        name = "_Z15lk_k_attn_splitILb%dE" % fused
        i = txt.index("\n" + name) + 1
        body = [l.strip() for l in txt[i:txt.index(".Lfunc_end", i)].split("\n")]
        loads, first_wait = _check_paths(name, body)
        assert loads == (20 if fused else 4), (name, loads)
        assert first_wait == 12, (name, first_wait)


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not installed")
@pytest.mark.parametrize("src,floor", [("decode", 16), ("prefill", 100), ("pf_gemm", 40)])
def test_a_wait_state_between_m0_and_the_lds_dma(tmp_path, src, floor):
    """An LDS DMA takes its LDS address from M0 and needs one wait state after the
    scalar write of M0.  The compiler keeps it for its own DMAs but does not look
    inside inline asm, which therefore has to hold the wait state itself."""
    cmd = next(l for l in subprocess.run(["make", "-n", "-B", "_build/%s.hip.o" % src], cwd=PKG, check=True,
                                         capture_output=True, text=True).stdout.split("\n") if " -c -x hip " in l)
    args = cmd.split(" 2>&1")[0].replace("-c -x hip", "--offload-device-only -S -x hip").split()
    asm = tmp_path / (src + ".s")
    args[args.index("-o") + 1] = str(asm)
    subprocess.run(args, check=True, cwd=PKG, capture_output=True)
    ins = [t for t in (l.split(";")[0].strip() for l in asm.read_text().split("\n"))
           if t and not t.startswith(".") and not t.endswith(":")]
    dma = [k for k, t in enumerate(ins) if re.match(r"(global|buffer)_load_lds|buffer_load.* lds\b", t)]
    assert len(dma) >= floor
    for k in dma:
        assert not re.match(r"s_\w+ m0,", ins[k - 1]), ins[k - 1:k + 1]


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not installed")
@pytest.mark.parametrize("knobs", [[], ["TARGET_N=128"], ["SPLIT=128"], ["NBUF=2"], ["NBUF=3"], ["TILE=32", "NBUF=2"],
                                   ["TILE=32", "NBUF=2", "TARGET_N=64"]], ids=lambda k: "_".join(k) or "default")
def test_no_branch_while_untracked_loads_are_pending(tmp_path, knobs):
    """Between the untracked loads and their wait the code is straight: around a
    branch the compiler may copy registers that are still in flight.  Checked,
    with the registers themselves, at the default and at other settings of the
    Makefile's knobs."""
    knob = dict(k.split("=") for k in knobs)
    in_flight = (int(knob.get("NBUF", 4)) - 1) * int(knob.get("TILE", 16)) // 4      # D tiles of TILE/4 rows per wave
    cmd = next(l for l in subprocess.run(["make", "-n", "-B", *knobs, "_build/decode.hip.o"], cwd=PKG, check=True,
                                         capture_output=True, text=True).stdout.split("\n") if " -c -x hip " in l)
    args = cmd.split(" 2>&1")[0].replace("-c -x hip", "--offload-device-only -S -x hip").split()
    asm = tmp_path / "decode.s"
    args[args.index("-o") + 1] = str(asm)
    subprocess.run(args, check=True, cwd=PKG, capture_output=True)
    txt = asm.read_text()
    for fused in (0, 1):
        name = "_Z15lk_k_attn_splitILb%dE" % fused
        i = txt.index("\n" + name) + 1
        body = [l.strip() for l in txt[i:txt.index(".Lfunc_end", i)].split("\n")]
        assert _check_paths(name, body) == (20 if fused else 4, in_flight)
        ins = [l.split(";")[0].strip() for l in body if l and not l.startswith((";", "."))]
        first = next(k for k, t in enumerate(ins) if t.startswith("global_load_dwordx4"))
        wait = next(k for k, t in enumerate(ins) if k > first and "vmcnt(" in t)
        window = ins[first:wait]
        assert not [t for t in window if t.startswith(("s_cbranch", "s_branch")) or t.endswith(":")], (name, window)
