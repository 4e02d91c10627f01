"""CPU-only check of the generated code of the short-prompt attention kernel: its K operands are fetched by LDS reads in inline
assembly a group ahead of the matrix instructions, like V's transposing reads (test_isa_hazards.py), and nothing may touch a
read's registers, and no branch or label stand, between the read and the wait that covers it."""

from test_isa_hazards import _kernels, touched_in_flight


def _inline_reads_as_transposing(lines):
    """The scanner follows transposing reads: the 16-byte reads of inline assembly take their place, the compiler's own (which it
    waits for itself) and the transposing ones become reads that only count."""
    out, inline = [], False
    for l in lines:
        if l.strip() in (";APP", ";NO_APP", ";;#ASMSTART", ";;#ASMEND"):
            inline = l.strip() in (";APP", ";;#ASMSTART")
        l = l.replace("ds_read_b64_tr_b16", "ds_read_b64")
        out.append(l.replace("ds_read_b128", "ds_read_b64_tr_b16") if inline else l)
    return out


def test_nothing_touches_an_operand_read_in_flight():
    kernels = _kernels("sp_attn_short.hip", "sp_attn_short_kernel")
    assert len(kernels) == 4, "64 / 128 channels x with / without the pivots' patterns"
    for name, body in kernels.items():
        count, found = touched_in_flight(_inline_reads_as_transposing(body))
        assert count >= 8
        assert not found, f"{name}: '{found[0][1]}' while '{found[0][0]}' is in flight"


def test_nothing_touches_an_operand_read_in_flight_where_the_priority_stays_level():
    kernels = _kernels("sp_attn_short.hip", "sp_attn_short_level_kernel")
    assert len(kernels) == 4
    for name, body in kernels.items():
        assert not any("s_setprio" in l for l in body)
        for lines, least in ((_inline_reads_as_transposing(body), 8), (body, 16)):
            count, found = touched_in_flight(lines)
            assert count >= least
            assert not found, f"{name}: '{found[0][1]}' while '{found[0][0]}' is in flight"


def test_the_first_tile_is_asked_for_before_the_mask_is_there():
    """64 channels: the mask's word is a row's first load, the first tile's the next ones, and nothing in between waits for memory."""
    kernels = _kernels("sp_attn_short.hip", "sp_attn_short_(?:level_)?kernelILi64E")
    assert len(kernels) == 4
    for name, body in kernels.items():
        loads = [i for i, l in enumerate(body) if l.strip().startswith(("global_load", "buffer_load", "flat_load"))]
        first, tile = loads[0], next(i for i in loads if " lds" in body[i])
        assert "global_load_dwordx2" in body[first] and loads.index(tile) == 1, name
        waits = [l.strip() for l in body[first:tile] if "s_waitcnt" in l and "vmcnt" in l]
        assert not waits, f"{name}: '{waits[0]}'"
