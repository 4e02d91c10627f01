"""CPU-only checks of the generated gfx950 code of the attention kernels.

The kernel's MFMAs are inline assembly, so the compiler knows neither their latency nor the wait states a vector
instruction needs before it may read an MFMA result (the hardware does not interlock that read).  The source keeps
such reads far behind the MFMAs by construction, or puts the wait states into the MFMA's own assembly statement
(at_mfma_acc_settled in csrc/sp_attn.hip).  What the source cannot see is the register allocator: to satisfy a tied
operand it may copy a result register with a vector move right behind the MFMA -- that happened in the pivot
instantiation and gave wrong row sums now and then.  This test compiles the file to assembly and measures, for every
vector / memory instruction that reads a register an MFMA wrote, how many wait states lie between the two.

The short-prompt kernel (csrc/sp_attn_short.hip) reads V with transposing LDS reads in inline assembly.  The compiler
takes their registers as written at once, so whatever it places between such a read and the wait behind it -- a register
copy, a branch to a block with copies of its own -- may see the old contents.  The second test follows every such read to
the s_waitcnt that covers it and lets nothing touch its registers, and no branch or label stand, in between."""

import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "shareprefill_amd", "csrc")
MIN_WAIT_STATES = 12  # an 8-pass MFMA needs 11 before a vector instruction reads its result
WINDOW = 40


def _regs(tok):
    tok = tok.strip().rstrip(",")
    m = re.match(r"v\[(\d+):(\d+)\]$", tok)
    if m:
        return set(range(int(m.group(1)), int(m.group(2)) + 1))
    m = re.match(r"-?\|?v(\d+)\|?$", tok)
    return {int(m.group(1))} if m else set()


def closest_reads(lines):
    """-> sorted [(wait states, mfma, reader)] for reads of MFMA results within WINDOW wait states.  Instructions are
    taken in program order (labels ignored); an s_nop N counts N + 1, an MFMA 4, anything else 1."""
    ins = [l.strip() for l in lines
           if l.strip() and not l.strip().startswith((";", ".")) and not l.strip().endswith(":")]
    found, pending = [], []
    for l in ins:
        op = l.split()[0]
        toks = [t for t in re.split(r"[ ,]+", l)[1:] if t]
        if op.startswith("v_mfma"):
            for p in pending:
                p[1] += 4
            dst = _regs(toks[0])
            pending = [p for p in pending if not (p[0] & dst)]  # accumulating in place: the hardware orders MFMAs
            pending.append([dst, 0, l])
            continue
        wait = int(toks[0]) + 1 if op == "s_nop" else 1
        is_store = op.startswith(("global_store", "ds_write", "buffer_store", "flat_store"))
        reads = set()
        if op.startswith(("v_", "ds_", "global_", "buffer_", "flat_")):
            for t in (toks if is_store else toks[1:]):
                reads |= _regs(t)
        for p in pending:
            if p[0] & reads:
                found.append((p[1], p[2], l))
        if op.startswith("v_") and toks:
            d = _regs(toks[0])
            pending = [p for p in pending if not (p[0] & d)]
        for p in pending:
            p[1] += wait
        pending = [p for p in pending if p[1] < WINDOW]
    return sorted(found)


def test_the_scanner_sees_a_copy_placed_right_behind_an_mfma():
    good = ["v_mfma_f32_16x16x32_bf16 v[8:11], v[0:3], v[4:7], v[8:11]", "s_nop 15", "v_mov_b32_e32 v20, v8"]
    bad = ["v_mfma_f32_16x16x32_bf16 v[8:11], v[0:3], v[4:7], v[8:11]", "s_nop 0", "v_mov_b64_e32 v[20:21], v[10:11]",
           "s_nop 15", "v_sub_f32_e32 v1, v20, v2"]
    assert closest_reads(good)[0][0] == 16
    assert closest_reads(bad)[0][0] == 1
    # an MFMA that accumulates into the same registers is ordered by the hardware and is no reader
    chain = ["v_mfma_f32_16x16x32_bf16 v[8:11], v[0:3], v[4:7], v[8:11]"] * 3
    assert closest_reads(chain) == []


def touched_in_flight(lines):
    """-> (number of transposing LDS reads, [(read, instruction)] that touch a read's registers, branch or end a block
    while it is in flight).  LDS operations return in order: s_waitcnt lgkmcnt(N) leaves the N youngest outstanding."""
    count, found, queue = 0, [], []  # queue: (registers or None, text) of every LDS operation in flight, oldest first
    for l in (line.split(";")[0].strip() for line in lines):
        if not l or (l.startswith(".") and not l.endswith(":")):
            continue
        op, toks = l.split()[0], [t for t in re.split(r"[ ,]+", l)[1:] if t]
        pending = [q for q in queue if q[0] is not None]
        if l.endswith(":") or op.startswith(("s_branch", "s_cbranch", "s_setpc", "s_endpgm")):
            found += [(text, l) for _, text in pending]
            continue
        if op == "s_waitcnt":
            m = re.search(r"lgkmcnt\((\d+)\)", l)
            if m or re.fullmatch(r"s_waitcnt 0", l):
                left = int(m.group(1)) if m else 0
                queue = queue[max(0, len(queue) - left):]
            continue
        regs = set()
        for t in toks:
            regs |= _regs(t)
        found += [(text, l) for r, text in pending if r & regs]
        if op.startswith("ds_"):
            is_read = op.startswith("ds_read_b64_tr_b16")
            count += is_read
            queue.append((_regs(toks[0]) if is_read else None, l))
    return count, found


def test_the_scanner_sees_a_copy_of_a_read_in_flight():
    read = ["ds_read_b64_tr_b16 v[8:9], v1 offset:64", "ds_read_b64_tr_b16 v[10:11], v1"]
    use = ["v_mfma_f32_16x16x32_bf16 v[20:23], v[8:11], v[4:7], v[20:23]"]
    assert touched_in_flight(read + ["s_waitcnt lgkmcnt(0)"] + use) == (2, [])
    assert touched_in_flight(read + ["s_waitcnt lgkmcnt(1)", "v_mov_b32_e32 v3, v8"])[1] == []
    assert len(touched_in_flight(read + ["v_mov_b32_e32 v3, v9", "s_waitcnt lgkmcnt(0)"] + use)[1]) == 1
    assert len(touched_in_flight(read + ["s_waitcnt lgkmcnt(1)"] + use)[1]) == 1
    assert len(touched_in_flight(read + ["s_cbranch_vccnz .LBB0_7", "s_waitcnt lgkmcnt(0)"] + use)[1]) == 2
    assert len(touched_in_flight(read + [".LBB0_3:", "s_waitcnt lgkmcnt(0)"] + use)[1]) == 2
    assert touched_in_flight(["s_waitcnt vmcnt(0)"] + read + ["s_waitcnt vmcnt(0)"] + use)[1] != []


def _kernels(source, name):
    """{mangled name: assembly lines} of the kernels called `name` in csrc/`source`, compiled as the library is."""
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not available")
    out = os.path.join(CSRC, source.replace(".hip", ".isa_check.s"))
    cmd = [hipcc, "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-Xclang", "-target-feature", "-Xclang",
           "-packed-fp32-ops", "-I", os.path.join(ROOT, "include"), "-I", CSRC, "-S", "--cuda-device-only",
           os.path.join(CSRC, source), "-o", out]
    try:
        subprocess.run(cmd, check=True, capture_output=True)
        text = open(out).read()
    finally:
        if os.path.exists(out):
            os.remove(out)
    kernels = {}
    for m in re.finditer(r"^(_Z\S*" + name + r"\S*):.*\n", text, re.M):
        start = m.end()
        kernels[m.group(1)] = text[start:text.index(".Lfunc_end", start)].split("\n")
    return kernels


def test_no_vector_instruction_reads_an_mfma_result_too_early():
    kernels = _kernels("sp_attn.hip", "sp_attn_fwd_kernel")
    assert len(kernels) == 5, "the forward kernel has five instantiations (pivot x half-channel, and small blocks)"
    for name, body in kernels.items():
        assert sum("v_mfma_f32_16x16x32_bf16" in l for l in body) > 100
        reads = closest_reads(body)
        assert not reads or reads[0][0] >= MIN_WAIT_STATES, (
            f"{name}: '{reads[0][2]}' reads the result of '{reads[0][1]}' only {reads[0][0]} wait states behind it")


def test_nothing_touches_a_transposing_read_in_flight():
    kernels = _kernels("sp_attn_short.hip", "sp_attn_short_kernel")
    assert len(kernels) == 4, "64 / 128 channels x with / without the pivots' patterns"
    for name, body in kernels.items():
        count, found = touched_in_flight(body)
        assert count >= 16
        assert not found, f"{name}: '{found[0][1]}' while '{found[0][0]}' is in flight"


def test_nothing_touches_a_transposing_read_in_flight_in_the_decode_ring():
    kernels = _kernels("sp_decode.hip", "sp_decode_ring_kernel")
    assert len(kernels) == 14, "whole and padded rows x 64 channels in 1, 2, 4 tiles, 128 in 1, 2, 4, 8"
    for name, body in kernels.items():
        count, found = touched_in_flight(body)
        assert count >= 2
        assert not found, f"{name}: '{found[0][1]}' while '{found[0][0]}' is in flight"


def test_nothing_touches_a_transposing_read_in_flight_in_the_decode_rings_of_many_pairs():
    kernels = _kernels("sp_decode.hip", "sp_decode_ring_(?:pair|quad)_kernel")
    assert len(kernels) == 8, "whole and padded rows x 64 and 128 channels x two workgroups a CU and four"
    for name, body in kernels.items():
        count, found = touched_in_flight(body)
        assert count >= 2
        assert not found, f"{name}: '{found[0][1]}' while '{found[0][0]}' is in flight"
