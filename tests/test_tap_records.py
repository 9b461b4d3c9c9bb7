"""Tap records are staged in 16-byte pieces by a fixed number of lanes, and the
records are allocated back to back with nothing behind the last one: no lane may
index a piece past its record.  A wrong index gives right results (the extra
piece is never used), so it is checked here on the host: the index function of
pf_taprec.h, compiled as it stands, over every width, and that the staging
kernels read records through it."""

import ctypes
import itertools
import os
import re
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "pyfourier_amd", "csrc")
WMAX = 8


@pytest.fixture(scope="module")
def rec(tmp_path_factory):
    d = tmp_path_factory.mktemp("taprec")
    src, out = d / "rec.cpp", d / "rec.so"
    src.write_text('#include "pf_taprec.h"\n'
                   'extern "C" int words(int z, int y, int x) { return pf_rec_words(z, y, x); }\n'
                   'extern "C" int piece(int c, int rec4) { return pf_rec_piece(c, rec4); }\n')
    subprocess.run(["g++", "-std=c++17", "-shared", "-fPIC", "-I", CSRC, str(src), "-o", str(out)], check=True)
    return ctypes.CDLL(str(out))


def test_every_staged_piece_lies_in_its_record(rec):
    widths = [w for d in (1, 2, 3) for w in itertools.product(range(1, WMAX + 1), repeat=d)]
    seen = set()
    for w in widths:
        z, y, x = (1,) * (3 - len(w)) + w
        words = rec.words(z, y, x)
        assert words % 4 == 0 and words >= 4 + z + y + x
        pieces = words // 4
        seen.add(pieces)
        # lane & 3 and (lane & 3) + 4 (spread of plain values), lane & 7 (fp16-split spread)
        staged = [rec.piece(c, pieces) for c in range(8)]
        assert all(0 <= c < pieces for c in staged), (w, pieces, staged)
        assert set(range(pieces)) <= set(staged)  # and every piece of the record is among them
    assert seen == {2, 3, 4, 5, 6, 7}


def _body(text, name):
    """From the definition of `name` to the end of its block."""
    start = text.index(name)
    i = text.index("{", text.index(")", start))
    depth = 0
    for k in range(i, len(text)):
        depth += {"{": 1, "}": -1}.get(text[k], 0)
        if depth == 0:
            return text[i:k]
    raise AssertionError(name)


def test_staging_kernels_read_records_through_it():
    text = open(os.path.join(CSRC, "pf_ops.hip")).read()
    body = _body(text, "k_spread_pipe(GeoParams")
    assert re.search(r"float4\* r = reinterpret_cast<const float4\*>\(taprec\)", body)
    reads = re.findall(r"= r\[(.*)\];", body)
    assert len(reads) == 2 and body.count("taprec") == 1
    assert all(re.fullmatch(r"pf_rec_piece\(.*, rec4\)", e) for e in reads), reads
    body = _body(text, "void smfma_issue(")
    assert "4 * cs" in body and body.count("taprec") == 1
    assert re.search(r"int cs = pf_rec_piece\(c, rec4\);", body)
