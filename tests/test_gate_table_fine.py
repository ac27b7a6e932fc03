"""The scan backward's fine gate table (rp_device.h fill_sincos_fine,
rot_gate_finish_cs), emulated on the CPU from the committed 256-entry records
and the source's constants, against float64 trigonometry."""

import re

import numpy as np

from tests.test_gate_table import CSRC, _constants, _half_ulp, _header_tables

TB, SUB = 2048, 8
AB = 2 * np.pi / TB


def _kc2b():
    text = open(f"{CSRC}/rp_device.h").read()
    return float(np.float32(re.search(r"\bkC2B = (-?[0-9.e+-]+)f", text).group(1)))


def _fine_table():
    """(sign, |m|, t = b (-s a)) as fill_sincos_fine stores them (fp32)."""
    rec, k = _header_tables()["kSinCos"], _constants()
    i = np.arange(TB)
    q = (i + SUB // 2) // SUB
    r = (i - q * SUB) / SUB
    base = rec[q % 256]
    am, sb = np.abs(base[:, 0]).astype(np.float64), base[:, 1].astype(np.float64)
    cm1 = r * r * k["kC2"]
    sx = r * (r * r * k["kS3"] + k["kS1"])
    m = am - cm1 + am * cm1 + sb * sx
    sn = sb + sb * cm1 + sx - am * sx
    sg = np.where(np.signbit(base[:, 0]), -1.0, 1.0)
    flip = m > 1.0
    m, sn, sg = np.where(flip, 2.0 - m, m), np.where(flip, -sn, sn), np.where(flip, -sg, sg)
    return sg, m.astype(np.float32), (sn * -AB).astype(np.float32)


def test_kc2b_is_half_the_squared_step():
    assert abs(_kc2b() / (-AB * AB / 2) - 1) < 2.0 ** -24


def test_fine_expansion_gives_cos_and_its_derivative():
    """b (1 + w) is cos and b v is -a sin at every entry and remainder, to
    half an ulp of the record's terms (the fine entry's and the base entry's)
    plus 2e-9: the base expansion's truncation is below 1e-9, this one's 6e-10,
    the constants' rounding the rest.  Close to |cos| = 1 the record's terms
    are small and the bound is the 2e-9: what the long-memory gates rely on."""
    sg, am, t = (x[:, None] for x in _fine_table())
    r = np.linspace(-0.5, 0.5, 21)[None, :]
    ang = AB * (np.arange(TB)[:, None] + r)
    m64, t64, c2 = am.astype(np.float64), t.astype(np.float64), _kc2b()
    p2 = c2 - m64 * c2
    w = -m64 + r * (t64 + r * p2)
    v = t64 + r * (2 * p2 + r * t64 * c2)
    rec = np.abs(_header_tables()["kSinCos"])
    q = ((np.arange(TB) + SUB // 2) // SUB) % 256
    hm = _half_ulp(am) + _half_ulp(rec[q, 0])[:, None]
    hs = _half_ulp(rec[q, 1])[:, None]
    err_c = np.abs(sg * (1 + w) - np.cos(ang))
    err_s = np.abs(sg * v / -AB - np.sin(ang))
    assert (err_c <= hm + 0.013 * hs + 2e-9).all(), err_c.max()
    assert (err_s <= _half_ulp(t) / AB + hs + 0.013 * hm + 2e-9).all(), err_s.max()
    assert err_c[np.broadcast_to(am <= 0.01, err_c.shape)].max() < 3e-9


def test_a_planted_coefficient_is_refused():
    sg, am, t = (x[:, None].astype(np.float64) for x in _fine_table())
    r = np.linspace(-0.5, 0.5, 21)[None, :]
    ang = AB * (np.arange(TB)[:, None] + r)
    w = -am + r * t  # the quadratic term dropped
    assert np.abs(sg * (1 + w) - np.cos(ang)).max() > 1e-6
