"""LDS exchanged between the lanes of one wave, without a workgroup barrier, is ordered in the source (CPU only).

The hardware runs a wave's LDS accesses in order, but nothing obliges the compiler to keep a lane's store ahead
of its load of another index, and a cell offset read too early would be an arbitrary address.  No run on a GPU
can show that such an ordering is missing while the compiler happens to keep it, so the order is read off the
source: after a store to a wave's own slice of an LDS array, a synchronisation comes before the next read of
that array."""
import os
import re

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "wzy-flash-serve_amd", "csrc")
SYNC = r"wave_lds_sync\(\)|__syncthreads\(\)"


def body(name, fn):
    with open(os.path.join(CSRC, name)) as fh:
        src = re.sub(r"//[^\n]*", "", fh.read())
    at = src.index("{", re.search(r"\b%s\(" % fn, src).start())
    depth = 0
    for i in range(at, len(src)):
        depth += {"{": 1, "}": -1}.get(src[i], 0)
        if depth == 0:
            return src[at:i]
    raise AssertionError("no end of %s" % fn)


def unordered_reads(text, array, store):
    """Reads of `array` that follow a store to it with no synchronisation between, in source order; macros that
    the text defines count where they are used."""
    macros = {}
    for m in re.finditer(r"#define (\w+)\(.*?\)((?:[^\n]*\\\n)*[^\n]*)\n", text):
        macros[m.group(1)] = m.group(2)
    text = re.sub(r"#define (?:[^\n]*\\\n)*[^\n]*\n|#undef[^\n]*\n", "", text)
    for n, b in macros.items():
        text = re.sub(r"\b%s\(" % n, lambda m: b + " (", text)
    pending, bad = False, []
    for m in re.finditer(r"(?P<store>%s)|(?P<sync>%s)|(?P<read>\b%s\b)" % (store, SYNC, array), text):
        if m.group("store"):
            pending = True
        elif m.group("sync"):
            pending = False
        elif pending:
            bad.append(text[max(0, m.start() - 60):m.end() + 20])
    return bad


@pytest.mark.parametrize("name,fn,array,store,stores", [
    ("prefill.hip", "pf_attn_kernel", "sOff", r"sOff\[w\]\[\w+\]\[lane\] =", 2),        # cell offsets of a chunk
    ("wzy_qsa_dev.h", "norm_rope_wave", "s_rot", r"s_rot\[lane(?: \+ 64)?\] =", 2),      # the rotated dims
])
def test_wave_private_lds_is_ordered(name, fn, array, store, stores):
    text = body(name, fn)
    text = text.replace("off_t %s[" % array, "off_t decl_[")                             # the declaration
    assert len(re.findall(store, text)) == stores
    assert unordered_reads(text, array, store) == []


def test_the_check_sees_a_missing_synchronisation():
    text = "{ s[w][lane] = x; y = s[w][3]; wave_lds_sync(); z = s[w][4]; }"
    assert len(unordered_reads(text, "s", r"s\[w\]\[lane\] =")) == 1
