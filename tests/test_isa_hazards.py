"""Static checks of the hazards the compiler cannot see, on the library compiled to assembly.

1. The dK/dV kernel and the 256-query forward and dQ kernels emit their logit MFMAs by hand (accumulators
   pinned to the architectural VGPRs),
   so the compiler's hazard recogniser does not insert the wait states an 8-pass MFMA needs before
   anything else may touch its result.  The kernels are structured so that at least two further MFMAs
   (or, off the hot paths, 11 wait states of s_nop) are issued first.
2. The LDS-DMA copies are emitted by hand as well and take their LDS destination from M0: every one of
   them must find, in its own basic block, an s_mov_b32 to M0 with at least one instruction in between
   (the wait state between a scalar write of M0 and an LDS-DMA that reads it)."""
import os
import re
import shutil
import subprocess
import tempfile

import pytest

from flame_amd import build as fb

SRC = os.path.join(fb.CSRC, "flame_attn.hip")


def _regs(tok, file="v"):
    m = re.match(r"%s\[(\d+):(\d+)\]" % file, tok)
    if m:
        return set(range(int(m.group(1)), int(m.group(2)) + 1))
    m = re.match(r"%s(\d+)$" % file, tok)
    return {int(m.group(1))} if m else set()


@pytest.fixture(scope="module")
def text():
    if shutil.which(fb.HIPCC) is None and not os.path.exists(fb.HIPCC):
        pytest.skip("hipcc not available")
    with tempfile.TemporaryDirectory() as tmp:
        out = os.path.join(tmp, "flame_attn.s")
        flags = [f for f in fb.FLAGS if f not in ("-shared", "-fPIC")]     # the flags the library is built with
        subprocess.run([fb.HIPCC, *flags, "-S", "--cuda-device-only", SRC, "-o", out], check=True,
                       stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL)
        return open(out).read()


def test_checks_run_on_the_compiler_that_built_the_library():
    """The assembly inspected here comes from this machine's hipcc; the shipped library records the hipcc
    that built it.  The checks say nothing about the library unless the two are the same compiler."""
    import ctypes
    lib_path = fb.LIB_PATH
    if not os.path.exists(lib_path):
        pytest.skip("library not built")
    if shutil.which(fb.HIPCC) is None and not os.path.exists(fb.HIPCC):
        pytest.skip("hipcc not available")
    lib = ctypes.CDLL(lib_path)
    lib.flame_attn_version.restype = ctypes.c_char_p
    built_with = lib.flame_attn_version().decode()
    assert f"(hipcc {fb.hipcc_version()})" in built_with, (built_with, fb.hipcc_version())


def test_hand_emitted_mfma_results_are_not_touched_too_early(text):
    """The result of a hand-emitted MFMA (architectural accumulator, or the big-head-dim forward's pinned accumulation
    tuples) may be touched only after two more MFMAs or 11 wait states of s_nop.  Followed along the control flow:
    an unconditional branch to its target, a conditional one both ways."""
    kernels = re.findall(r"^(_ZN5fattn(?:15bwd_dkdv_kernel|21bwd_dkdv_dealt_kernel|18bwd_dq_wide_kernel|24bwd_dq_wide_dealt_kernel|15fwd_wide_kernel|20sage_fwd_wide_kernel|15fwd_bigd_kernel)\w+):.*?\.end_amdhsa_kernel", text, re.S | re.M)
    assert len(kernels) >= 9
    checked = 0
    for name in kernels:
        body = re.search(r"^%s:.*?\.end_amdhsa_kernel" % re.escape(name), text, re.S | re.M).group(0)
        # instructions and labels, in order
        ins = [l.strip() for l in body.split("\n") if re.match(r"^\s+[a-z]", l) or re.match(r"^\.LBB\S+:", l)]
        label_at = {re.match(r"(\.LBB\w+):", l).group(1): i for i, l in enumerate(ins) if l.startswith(".LBB")}
        for idx, l in enumerate(ins):
            if not l.startswith("v_mfma"):
                continue
            ops = [t.strip() for t in l.split(None, 1)[1].split(",")]
            # an accumulator in the accumulation registers is the compiler's own MFMA form, which it guards itself,
            # except in the big-head-dim forward, which emits its O^T MFMAs by hand into pinned a[0:127]
            by_hand_acc = "fwd_bigd_kernel" in name and ops[0].startswith("a[")
            if not ops[0].startswith("v[") and not by_hand_acc:
                continue
            checked += 1
            dst = _regs(ops[0], "a" if by_hand_acc else "v")
            todo = [(idx + 1, 0, 0)]                    # (position, MFMAs since, wait states spent in s_nop since)
            seen = set()
            while todo:
                pos, later_mfma, idle = todo.pop()
                while pos < len(ins) and pos not in seen:
                    seen.add(pos)
                    l2 = ins[pos]
                    pos += 1
                    if l2.startswith(".LBB"):
                        continue
                    if l2.startswith("v_mfma"):
                        later_mfma += 1
                        if later_mfma >= 2:
                            break
                        continue
                    m = re.match(r"s_nop\s+(\d+)", l2)
                    if m:
                        idle += int(m.group(1)) + 1
                        if idle >= 11:                  # an 8-pass result is visible 11 wait states after issue
                            break
                        continue
                    if l2.startswith("s_endpgm"):
                        break
                    m = re.match(r"s_(c?)branch\w*\s+(\.LBB\S+)", l2)
                    if m:
                        if m.group(1):
                            todo.append((label_at[m.group(2)], later_mfma, idle))     # taken; not taken goes on below
                            continue
                        pos = label_at[m.group(2)]
                        continue
                    if l2.startswith("s_") or l2.startswith("global_load_lds"):
                        continue                        # scalar, or vector registers used as addresses only
                    if by_hand_acc:
                        used = set()
                        for t in re.findall(r"\ba\[\d+:\d+\]|\ba\d+\b", l2):
                            used |= _regs(t, "a")
                    else:
                        toks = re.findall(r"v\[\d+:\d+\]|v\d+", l2)
                        if l2.startswith("ds_read"):
                            toks = toks[:1]             # the destination; the other register is an address
                        used = set()
                        for t in toks:
                            used |= _regs(t)
                    assert not (used & dst), f"{name}: `{l2}` touches the result of `{l}` before two more MFMAs"
    assert checked >= 4 * 96


def test_operands_of_hand_emitted_mfmas_are_not_written_just_before(text):
    """An MFMA may read a register the vector ALU wrote two wait states later at the earliest.  The compiler keeps
    that distance for its own MFMAs; for the hand-emitted ones (architectural accumulator, or the big-head-dim
    forward's pinned accumulation tuples) it must come from the statement itself (an s_nop in front) or from where
    the operands live (pinned registers that nothing moves).  Checked on every MFMA of every kernel: no vector-ALU
    instruction within the two wait states in front of it writes one of its source registers."""
    kernels = re.findall(r"^(_ZN5fattn\w+):.*?\.end_amdhsa_kernel", text, re.S | re.M)      # every kernel of the library
    checked = 0
    for name in kernels:
        body = re.search(r"^%s:.*?\.end_amdhsa_kernel" % re.escape(name), text, re.S | re.M).group(0)
        ins = [l.strip() for l in body.split("\n") if re.match(r"^\s+[a-z]", l)]
        for idx, l in enumerate(ins):
            if not l.startswith("v_mfma"):
                continue
            ops = [t.strip() for t in l.split(None, 1)[1].split(",")]      # the compiler's own MFMAs pass by construction
            checked += 1
            src_v, src_a = set(), set()
            for t in ops[1:4]:
                src_v |= _regs(t, "v")
                src_a |= _regs(t, "a")
            states = 0
            for l2 in reversed(ins[max(0, idx - 4):idx]):
                m = re.match(r"s_nop\s+(\d+)", l2)
                if m:
                    states += int(m.group(1)) + 1
                elif l2.startswith("v_") and not l2.startswith("v_mfma"):
                    dst = l2.split(None, 1)[1].split(",")[0].strip()
                    wrote = (_regs(dst, "v") & src_v) | (_regs(dst, "a") & src_a)
                    assert not wrote, f"{name}: `{l2}` writes an operand of `{l}` {states} wait states before it"
                    states += 1
                else:
                    states += 1
                if states >= 2:
                    break
    assert checked >= 4 * 96


def test_every_lds_dma_finds_its_destination_in_m0(text):
    kernels = re.findall(r"^(_ZN5fattn\w+):.*?\.end_amdhsa_kernel", text, re.S | re.M)
    assert kernels
    checked = 0
    for name in kernels:
        body = re.search(r"^%s:.*?\.end_amdhsa_kernel" % re.escape(name), text, re.S | re.M).group(0)
        # instructions and labels, in order
        ins = [l.strip() for l in body.split("\n") if re.match(r"^\s+[a-z]", l) or re.match(r"^\.LBB\S+:", l)]
        for idx, l in enumerate(ins):
            if not l.startswith("global_load_lds"):
                continue
            checked += 1
            between = 0
            for l2 in reversed(ins[:idx]):
                assert not l2.startswith(".LBB"), f"{name}: `{l}` has no M0 write in its basic block"
                if re.match(r"s_mov_b32\s+m0,", l2):
                    break
                assert "m0" not in l2.split(";")[0], f"{name}: `{l2}` uses M0 between its write and `{l}`"
                between += 1
            else:
                raise AssertionError(f"{name}: `{l}` has no M0 write before it")
            assert between >= 1, f"{name}: `{l}` follows its M0 write without a wait state"
    assert checked >= 100


WAIT_PROBE = r"""
#include "attn_common.hpp"
using namespace fattn;
template <class W> __device__ void around(const float* x, float* out, const char* src, int n, W wait) {
    extern __shared__ __attribute__((aligned(1024))) uint16_t lds[];
    dma16u(src, threadIdx.x * 16, lds_addr(lds));
    const float v = x[threadIdx.x];
    wait();
    if (n > 3) out[threadIdx.x] = v;           // the one use: the compiler would rather load there
}
extern "C" __global__ void counted(const float* x, float* out, const char* src, int n) { around(x, out, src, n, [] { wait_vm<1>(); }); }
extern "C" __global__ void drained(const float* x, float* out, const char* src, int n) { around(x, out, src, n, [] { wait_vm<0>(); }); }
"""


def test_no_load_moves_past_a_wait(tmp_path):
    """A counted wait says how many younger operations may still be on their way; a load that the compiler moved past it would
    leave as many copies unfinished."""
    if shutil.which(fb.HIPCC) is None and not os.path.exists(fb.HIPCC):
        pytest.skip("hipcc not available")
    src, out = tmp_path / "probe.hip", tmp_path / "probe.s"
    src.write_text(WAIT_PROBE)
    flags = [f for f in fb.FLAGS if f not in ("-shared", "-fPIC")]
    subprocess.run([fb.HIPCC, *flags, "-I" + fb.CSRC, "-S", "--cuda-device-only", str(src), "-o", str(out)], check=True, stdout=subprocess.DEVNULL,
                   stderr=subprocess.DEVNULL)
    for name, count in (("counted", 1), ("drained", 0)):
        body = re.search(r"^%s:.*?s_endpgm" % name, out.read_text(), re.S | re.M).group(0)
        order = re.findall(r"^\s+(global_load_lds_dwordx4|global_load_dword\b|s_waitcnt vmcnt\(%d\))" % count, body, re.M)
        assert order[:3] == ["global_load_lds_dwordx4", "global_load_dword", f"s_waitcnt vmcnt({count})"], (name, order)


def test_the_bias_counted_out_of_a_wait_is_younger_than_the_copies(text):
    """The forward that requests its bias a step ahead: between a step's last copy and the wait that leaves N operations on their
    way, which the step's barrier follows, there are at least N loads of the bias."""
    checked = 0
    for excl, pieces in ((3, 8), (4, 4)):                # fp32, bf16: loads per lane and tile
        name = "_ZN5fattn10fwd_kernelILi64ELi%dELi4ELi0ELi1ELb1EEEvNS_9FwdParamsE" % excl
        body = re.search(r"^%s:.*?\.end_amdhsa_kernel" % name, text, re.S | re.M).group(0)
        ins = [l.strip() for l in body.split("\n") if re.match(r"^\s+[a-z]", l) or re.match(r"^\.LBB\S+:", l)]
        for i, l in enumerate(ins):
            if not l.startswith(f"s_waitcnt vmcnt({pieces})") or not any(x.startswith("s_barrier") for x in ins[i + 1:i + 8]):
                continue
            loads, skipped = 0, None                     # skipped: the label that a branch over a few instructions goes to
            for l2 in reversed(ins[:i]):
                if l2.startswith(".LBB"):
                    assert skipped is None, f"{name}: more than a branch over a few instructions between copies and wait"
                    skipped = l2.split(":")[0]
                elif l2.startswith("s_cbranch") and l2.endswith(skipped or "-"):
                    skipped = None
                elif l2.startswith("global_load_lds"):
                    break
                elif l2.startswith("global_load_dword"):
                    assert skipped is None, f"{name}: `{l2}` is not always executed"
                    loads += 1
            assert skipped is None and loads >= pieces, (name, loads)
            checked += 1
    assert checked == 4                                  # two steps per trip of the loop in either kernel


def test_words_of_a_mask_are_not_waited_for_within_their_step(text):
    """The forward that walks by a mask's bits: loads return in order, so a step that waits for a word which it has requested itself waits
    for its tile copies as well.  The word is the next step's; the first wait behind it is the one in front of the barrier."""
    for D, mfmas, form in [(*d, f) for d in ((64, 16), (96, 24), (128, 32)) for f in ("10fwd_kernelILi%dELi6ELi4ELi0ELi1ELb0EE", "16fwd_dealt_kernelILi%dELi6ELi4EE")]:
        name = "_ZN5fattn" + form % D + "EvNS_9FwdParamsE"    # (half a step's MFMAs or more are between)
        body = re.search(r"^%s:.*?\.end_amdhsa_kernel" % name, text, re.S | re.M).group(0)
        ins = [l.strip() for l in body.split("\n") if re.match(r"^\s+[a-z]", l)]
        first = next(i for i, l in enumerate(ins) if l.startswith("v_mfma"))
        words = [i for i, l in enumerate(ins) if i > first and l.startswith("global_load_dwordx2")]
        assert len(words) == 2                                # two steps per trip of the loop
        for i in words:
            j = next(j for j in range(i, len(ins)) if ins[j].startswith("s_waitcnt") and "vmcnt" in ins[j])
            assert any(l.startswith("s_barrier") for l in ins[j:j + 8]), (name, ins[i:j + 1])
            assert sum(l.startswith("v_mfma") for l in ins[i:j]) >= mfmas, name


def test_the_key_sharing_forward_keeps_its_state_in_registers(text):
    """Every form of it, the draws of a dropout among them: none of a wavefront's running state in scratch memory."""
    kernels = re.findall(r"^(_ZN5fattn19fwd_keyshare_kernel\w+):.*?\.amdhsa_private_segment_fixed_size (\d+)", text, re.S | re.M)
    assert len(kernels) == 18 and all(int(size) == 0 for _, size in kernels), kernels
