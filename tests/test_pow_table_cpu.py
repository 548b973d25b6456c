"""The literals of mw_pow_gamma (csrc/stencil_bodies.hpp): x^gamma as 2^(gamma e), from a table, times a polynomial in the
mantissa.  Recomputed here with 50 digits."""
import os
import re
from decimal import Decimal, getcontext

import numpy as np

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SOURCE = open(os.path.join(ROOT, "gpreempt_amd", "csrc", "stencil_bodies.hpp")).read()
getcontext().prec = 50
NUMBER = r"-?\d+\.\d+(?:e[+-]?\d+)?"


def gamma():
    """the exponent: the reference's, rounded to fp32"""
    text = re.search(r"MW_GAMMA = (\d\.\d+)f", SOURCE).group(1)
    assert "MW_GAMMA == %sf" % text in SOURCE  # the assertion in front of the table names the same one
    return Decimal(float(np.float32(text)))


def literals():
    body = SOURCE[SOURCE.index("mw_pow2_gamma[278] = {"):]
    table = [float(x) for x in re.findall(NUMBER, body[:body.index("};")])]
    poly = body[body.index("double q = "):body.index("return q * scale;")]
    first = int(re.search(r"MW_POW_E0 = (-\d+);", SOURCE).group(1))
    return first, table, [float(x) for x in re.findall(NUMBER, poly)]


def test_table_holds_the_powers_of_two():
    first, table, _ = literals()
    assert first == -149 and len(table) == 278 and first + len(table) - 1 == 128  # denormals to the largest fp32 numbers
    ln2 = Decimal(2).ln()
    for i, got in enumerate(table):
        want = (gamma() * (first + i) * ln2).exp()
        assert abs(Decimal(got) - want) <= want * Decimal(2) ** -53, first + i  # correctly rounded, or the neighbour at a tie


def test_polynomial_is_the_power_of_a_mantissa():
    _, _, c = literals()
    assert len(c) == 16
    rng = np.random.default_rng(0)
    m = np.concatenate([[0.5, 0.75, np.nextafter(1.0, 0)], 0.5 + 0.5 * rng.random(3000)])
    w = m - 0.75  # exact
    q = np.full(m.shape, c[0])
    for k in c[1:]:
        q = (q.astype(np.longdouble) * w + k).astype(np.float64)  # a fused multiply-add, but for double rounding
    want = np.array([float((gamma() * Decimal(float(x)).ln()).exp()) for x in m])
    assert np.abs(q / want - 1).max() < 1.6e-15
