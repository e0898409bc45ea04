"""Wait states of gfx950 machine code that the hardware leaves to the program.

The compiler counts them for its own instructions only: not for those inside
inline asm, whose results the next instruction may read too early.  `early`
finds such reads in the text of a disassembly.
"""
import re


def _numbers(token, kind):
    m = re.fullmatch(kind + r"\[(\d+):(\d+)\]", token)
    if m:
        return set(range(int(m[1]), int(m[2]) + 1))
    m = re.fullmatch(kind + r"(\d+)", token)
    return {int(m[1])} if m else set()


def _sgprs(token):
    return {"vcc"} if token.startswith("vcc") else _numbers(token, "s")


def _vgprs(token):
    return _numbers(token, "v")


def _any(tokens, regs):
    return set().union(*map(regs, tokens)) if tokens else set()


def early(text):
    """The VALU reads that come too few wait states after a VALU write:

    2 of a scalar register (a lane mask, VCC) by any VALU instruction; 2 of a
    vector register by an MFMA, a permlane swap or a DPP instruction; 1 by
    v_readlane and v_readfirstlane.  Every instruction between is one wait
    state, s_nop n is n + 1."""
    found, writes = [], []  # writes: [register set, is scalar, wait states since]
    for line in text.splitlines():
        line = re.split(r"//|;", line, maxsplit=1)[0].strip()
        if not line or line.startswith(".") or line.endswith(":"):
            continue
        op, _, rest = line.partition(" ")
        if op == "s_nop":
            n = int(rest, 0) + 1
            writes = [[r, s, d + n] for r, s, d in writes if d + n < 2]
            continue
        if op.startswith("v_"):
            args = [a for a in re.split(r"[,\s|]+", rest.replace("-v", "v")) if a]
            lane_read = op.startswith(("v_readlane", "v_readfirstlane"))
            two = bool(re.search(r"_co_|v_mad_[ui]64|v_div_scale", op))  # a mask is the second result
            swap = op.startswith(("v_permlane", "v_swap"))
            reads = args if swap else args[2:] if two else args[1:]
            sread, vread = _any(reads, _sgprs), _any(reads, _vgprs)
            slow = op.startswith(("v_mfma", "v_permlane")) or op.endswith("_dpp")
            for r, scalar, d in writes:
                need = 2 if scalar or slow else 1 if lane_read else 0
                if d < need and r & (sread if scalar else vread):
                    found.append(line)
                    break
            written = args if swap else args[:2] if two else args[:1]
            fresh = [[_any(written, _sgprs), True, 0], [_any(written, _vgprs) if not op.startswith("v_mfma") else set(), False, 0]]
        else:
            fresh = []
        writes = [[r, s, d + 1] for r, s, d in writes if d < 1] + [w for w in fresh if w[0]]
    return found
