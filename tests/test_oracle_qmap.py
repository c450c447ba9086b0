"""Pins of the oracle's quantisation maps and code assignment (no GPU).

The reference ships no vectors; what pins these functions is (a) the bit patterns of the two
maps as obtained from the reference's own construction recipe run with PyTorch ops
(tests/golden/qmaps.json), (b) the closed form "code = number of fp32 midpoints < x",
(c) brute force around every map point and midpoint."""
import json
import os
import re
import subprocess
import sys

import numpy as np
import pytest
import torch

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(ROOT, "low-bit-optimizers_amd", "csrc")

GOLD = json.load(open(os.path.join(HERE, "golden", "qmaps.json")))


def bits(a):
    return [int(x) for x in np.asarray(a, dtype=np.float32).view(np.uint32)]


def test_qmap_m_bits(oracle):
    assert bits(oracle.qmap_m()) == [int(h, 16) for h in GOLD["qmap_m_hex"]]
    assert bits(oracle.midpoints(oracle.qmap_m())) == [int(h, 16) for h in GOLD["mid_m_hex"]]


def test_qmap_m_shape_properties(oracle):
    q = oracle.qmap_m()
    assert np.all(np.diff(q) > 0) and q[7] == 0.0 and q[15] == 1.0
    # asymmetric: +1.0 has no negative counterpart, everything else mirrors exactly
    assert np.array_equal(q[:7], -q[8:15][::-1]) and -1.0 not in q


def test_qmap_v_is_k_over_16(oracle):
    q = oracle.qmap_v()
    assert np.array_equal(q, (np.arange(16, dtype=np.float32) + 1) / np.float32(16))
    assert bits(q) == [int(h, 16) for h in GOLD["qmap_v_hex"]]
    assert np.array_equal(oracle.midpoints(q)[0:], (2 * np.arange(0, 15, dtype=np.float32) + 3) / np.float32(32))


def test_product_maps_equal_oracle_maps(oracle):
    """lpmm.functional builds the maps with torch ops (as the reference does); the oracle
    builds them with numpy float32 arithmetic.  Both must give the golden bits."""
    import lpmm.functional as F

    assert bits(F.create_general_qmap("nonlinear", 4, True).numpy()) == bits(oracle.qmap_m())
    assert bits(F.create_general_qmap("power-1", 4, False).numpy()) == bits(oracle.qmap_v())


def test_compiled_in_tables_equal_oracle_maps(oracle):
    txt = open(os.path.join(CSRC, "std_tables.inc")).read()

    def arr(name):
        body = txt.split(name)[1].split("{", 1)[1].split("}", 1)[0]
        return [int(t.strip().rstrip("u"), 16) for t in body.split(",")]

    assert arr("kStdQmapMBits[16]") == bits(oracle.qmap_m())
    assert arr("kStdQmapVBits[16]") == bits(oracle.qmap_v())


def test_generated_table_is_current():
    out = subprocess.check_output([sys.executable, os.path.join(CSRC, "gen_std_tables.py")], text=True)
    assert out == open(os.path.join(CSRC, "std_tables.inc")).read(), "re-run gen_std_tables.py"


def _count_code(mids, x):
    return int(np.sum(mids < np.float32(x)))


@pytest.mark.parametrize("which", ["m", "v"])
def test_qmapping_brute_force(oracle, which):
    q = oracle.qmap_m() if which == "m" else oracle.qmap_v()
    mids = oracle.midpoints(q)
    pts = [np.float32(0.0), np.float32(-0.0), np.float32(2.0), np.float32(-2.0), np.float32(np.inf),
           np.float32(-np.inf), np.float32(1e-45), np.float32(-1e-45)]
    for base in list(q) + list(mids):
        b = np.float32(base)
        pts += [b, np.nextafter(b, np.float32(np.inf)), np.nextafter(b, np.float32(-np.inf))]
    rng = np.random.default_rng(0)
    pts += list(rng.uniform(-1.2, 1.2, 20000).astype(np.float32))
    pts = np.array(pts, dtype=np.float32)
    got = oracle.qmapping(q, pts)
    want = np.array([_count_code(mids, x) for x in pts], dtype=np.uint8)
    assert np.array_equal(got, want)
    # every map point maps to itself; an exact tie goes to the lower code
    assert np.array_equal(oracle.qmapping(q, q), np.arange(16, dtype=np.uint8))
    assert np.array_equal(oracle.qmapping(q, mids), np.arange(15, dtype=np.uint8))
    # monotone
    xs = np.sort(pts[np.isfinite(pts)])
    assert np.all(np.diff(oracle.qmapping(q, xs).astype(int)) >= 0)


def test_qmapping_nan_is_minus_one_then_15(oracle):
    for q in (oracle.qmap_m(), oracle.qmap_v()):
        assert oracle.qmapping_scalar(q, np.nan) == -1
        assert oracle.qmapping(q, np.array([np.nan], np.float32))[0] == 15


def test_pad_codes(oracle):
    # zero padding of the non-fused layout: 0.0 -> code 7 on the m map, code 0 on the v map
    assert oracle.qmapping(oracle.qmap_m(), np.zeros(1, np.float32))[0] == 7
    assert oracle.qmapping(oracle.qmap_v(), np.zeros(1, np.float32))[0] == 0


def test_fast_encoders_exhaustive(tmp_path):
    """The table-driven m encoder and the closed-form v encoder used by the HIP kernels
    (lpmm_encode.hpp) against the reference search on every non-NaN fp32 bit pattern."""
    exe = str(tmp_path / "encode_exhaustive")
    subprocess.check_call(["g++", "-O2", "-fopenmp", "-ffp-contract=off", "-I", CSRC,
                           os.path.join(HERE, "encode_exhaustive.cpp"), "-o", exe])
    out = subprocess.check_output([exe], text=True)
    assert "bad_m 0 bad_v 0" in out, out
    assert "checked 4278190082" in out, out


def test_half_encoders_on_every_half(oracle):
    """The bucket table and the closed form that give the codes of normalised halfs (lpmm_half.hpp: encode8_half_m, encode8_half_v),
    restated, against the search on every half (the closed form: on those from -1 to 1)."""
    txt = open(os.path.join(CSRC, "std_tables.inc")).read()
    body = txt.split("kEncHalfM[256][2]")[1].split("};", 1)[0]
    words = np.array([int(w, 16) for w in re.findall(r"0x[0-9a-f]{8}", body)], dtype=np.uint32).astype(np.int32).astype(np.int64)
    entries = words.reshape(256, 2)
    bits16 = np.arange(1 << 16, dtype=np.uint16)
    x = bits16.view(np.float16)
    e = entries[bits16 >> 8]
    got = (e[:, 0] + e[:, 1] * bits16.view(np.int16).astype(np.int64)) >> 16
    want = oracle.qmapping(oracle.qmap_m(), x.astype(np.float32))
    signalling = np.isnan(x) & ((bits16 & 0x200) == 0)  # arithmetic gives none
    assert np.array_equal(got[~signalling], want[~signalling])
    x = x[np.abs(x.astype(np.float32)) <= 1]
    r = np.maximum((x.astype(np.float64) * 15.9921875 + 1023).astype(np.float16), np.float16(1024))  # one rounding: an fma
    want = oracle.qmapping(oracle.qmap_v(), x.astype(np.float32))
    assert np.array_equal(r.view(np.uint16) - 0x6400, want)
