"""The library's IQ lattice tables equal the reference's table fixture (digests of iqtables.npz)."""
import ctypes
import hashlib
import json
import os

import numpy as np
import pytest

from seedpack_amd._lib import check, lib

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LATTICE = {0: 16, 1: 17, 3: 22, 4: 18, 5: 21}      # table -> type
TRIALS = {16: (5, -6, 13, 0.1), 17: (5, -9, 19, 0.1), 22: (5, -9, 19, 0.1), 18: (15, -15, 31, 0.2), 21: (15, -9, 19, 0.2)}
NAMES = ["iq2_data_0", "iq2_data_1", "iq2_data_2", "iq2_data_3", "iq3_data_0", "iq3_data_1"]


def host_table(i):
    g, gn, m, mn, nb, nbn = (ctypes.c_void_p(), ctypes.c_int(), ctypes.c_void_p(), ctypes.c_int(), ctypes.c_void_p(),
                             ctypes.c_int())
    check(lib().spa_iq_table_host(i, ctypes.byref(g), ctypes.byref(gn), ctypes.byref(m), ctypes.byref(mn),
                                  ctypes.byref(nb), ctypes.byref(nbn)))
    grid = np.ctypeslib.as_array(ctypes.cast(g, ctypes.POINTER(ctypes.c_uint8)), (gn.value,)).copy()
    kmap = np.ctypeslib.as_array(ctypes.cast(m, ctypes.POINTER(ctypes.c_int32)), (mn.value,)).copy()
    nbs = np.ctypeslib.as_array(ctypes.cast(nb, ctypes.POINTER(ctypes.c_uint16)), (nbn.value,)).copy()
    return grid, kmap, nbs


@pytest.mark.parametrize("i", range(6))
def test_iq_tables_equal_reference_fixture(i):
    man = json.load(open(os.path.join(ROOT, "tests", "golden", "iqtables_sha256.json")))
    grid, kmap, nbs = host_table(i)
    name = NAMES[i]
    g = grid.view(np.uint64 if i < 4 else np.uint32)
    assert hashlib.sha256(g.tobytes()).hexdigest() == man[name + "_grid"]["sha256"]
    assert hashlib.sha256(kmap.tobytes()).hexdigest() == man[name + "_map"]["sha256"]
    assert nbs.size == man[name + "_nb"]["n"]
    assert hashlib.sha256(nbs.tobytes()).hexdigest() == man[name + "_nb"]["sha256"]


def test_neighbour_lists_are_nearest_by_brute_force():
    """IQ3_XXS: every listed neighbour of an off-grid index is within the nwant nearest distances and
    the list is ordered by (distance, index)"""
    grid, kmap, nbs = host_table(4)
    pts = grid.reshape(-1, 4).astype(np.int64)
    for i in [1, 7, 100, 1000, 4095]:
        if kmap[i] >= 0:
            continue
        pos = 2 * ((i >> (3 * np.arange(4))) & 7) + 1
        d2 = ((pts - pos) ** 2).sum(1)
        o = -kmap[i] - 1
        lst = nbs[o + 1:o + 1 + nbs[o]]
        levels = np.unique(d2)[:2]
        want = [j for d in levels for j in np.flatnonzero(d2 == d)]
        assert list(lst) == want


@pytest.mark.parametrize("i, d, levels, l1, m2, p1, p2", [(0, 8, 3, 20, 128, 24, 144), (1, 8, 3, 20, 128, 24, 144),
                                                          (3, 8, 3, 20, 128, 24, 144), (4, 4, 8, 16, 336, 24, 480),
                                                          (5, 4, 8, 16, 336, 24, 480)])
def test_spread_of_the_neighbour_lists(i, d, levels, l1, m2, p1, p2):
    """the lattice quantizers' bounds (ListBound in csrc/quant_lattice.hip): sums over the coordinates of
    |q - q'| and |q^2 - q'^2| between a list's first point and another, and between any two of its points, over
    every list a rounded group can reach; and the 32-bit ranges that follow from them"""
    grid, kmap, nbs = host_table(i)
    pts = grid.reshape(-1, d).astype(np.int64)
    bits = 2 if d == 8 else 3
    top = np.zeros(4, np.int64)
    for u in range(kmap.size):
        lev = (u >> (bits * np.arange(d))) & ((1 << bits) - 1)
        if lev.max() >= levels or kmap[u] >= 0:
            continue
        o = -int(kmap[u]) - 1
        p = pts[nbs[o + 1:o + 1 + int(nbs[o])]]
        q = p * p
        top = np.maximum(top, [np.abs(p - p[0]).sum(1).max(), np.abs(q - q[0]).sum(1).max(),
                               np.abs(p[:, None] - p[None]).sum(-1).max(), np.abs(q[:, None] - q[None]).sum(-1).max()])
    assert (top <= [l1, m2, p1, p2]).all(), top
    kernel = np.zeros(5, np.float32)
    check(lib().spa_lattice_bound_host(LATTICE[i], np.ones(6, np.float32).ctypes.data, kernel.ctypes.data))
    assert list(kernel[1:]) == [l1, m2, p1, p2]
    vmax = 1 << (23 if d == 8 else 22)
    assert p2 * vmax < 1 << 31 and m2 * vmax < 1 << 31 and (pts * pts).sum(1).max() * vmax < 1 << 32


def numerators(t):
    base, lo, n, step = TRIALS[t]
    return [np.float32(base) + np.float32(lo + k) * np.float32(step) for k in range(n)]


@pytest.mark.parametrize("t", sorted(TRIALS))
def test_trial_scales_divide_exactly(t):
    """the lattice quantizers' trial scales num / max, formed as one remainder step on num * (1 / max), are the
    float32 quotient for every mantissa of max and every num of the type"""
    mx = (np.arange(1 << 23, dtype=np.uint32) | np.uint32(0x3F800000)).view(np.float32)
    got = np.empty_like(mx)
    for k, num in enumerate(numerators(t)):
        check(lib().spa_lattice_trials_host(t, k, mx.ctypes.data, mx.size, got.ctypes.data))
        assert np.array_equal(got, num / mx), k


@pytest.mark.parametrize("t", sorted(TRIALS))
def test_filter_scales_within_four_units(t):
    """the scale that the integer filter takes, max times a reciprocal of num that one step refines, is within
    4 * 2^-24 of 1 / (num / max) as float32 rounds it, the hardware's reciprocal up to one unit off"""
    f, d = np.float32, np.float64
    mx = (np.arange(0, 1 << 23, 7, dtype=np.uint32) | np.uint32(0x3F800000)).view(f)
    for num in numerators(t):
        want = f(1) / (num / mx)
        for r in (np.nextafter(f(1) / num, f(0)), f(1) / num, np.nextafter(f(1) / num, f(9))):
            # the fused steps: exact in float64 but for a rounding far below float32's
            rn = f(f(1 - d(num) * d(r)) * d(r) + d(r))
            assert np.abs((mx * rn).astype(d) / want - 1).max() <= 4 * 2.0 ** -24


@pytest.mark.parametrize("t", sorted(TRIALS))
def test_lead_covers_every_rounding(t):
    """the lead the filter asks of its best point is no less than the sum of what separates the filter's values of
    two points from the reference's float sums (the terms listed at tolerance() in csrc/quant_lattice.hip)"""
    g = np.random.Generator(np.random.PCG64(t))
    u, vmax = 2.0 ** -24, 2.0 ** (22 if t in (18, 21) else 23)
    for _ in range(4000):
        sp = np.exp2(g.uniform(-8, 4))
        c0, a_s = vmax * g.uniform(1, 80), 2.0 ** g.uniform(20, 27)
        b0 = g.uniform(0, 1) * (a_s + sp * c0)
        best = -g.uniform(0, 1.2) * (a_s + sp * c0 - b0) * g.choice([0.01, 1])
        terms = np.array([sp, 1 / sp, a_s * sp, c0, b0, best], np.float32)
        out = np.zeros(5, np.float32)
        check(lib().spa_lattice_bound_host(t, terms.ctypes.data, out.ctypes.data))
        sp, rs, a, c0, b0, best = terms.astype(np.float64)
        l1, m2, p1, p2 = out[1:].astype(np.float64)
        d2 = max(0.0, a * rs + sp * c0 - b0 + best)
        need = (sp * p2 / 2 + p1 + 4 * u * vmax * sp * p2 + 4 * u * (vmax * sp * m2 + 2.0 ** 23 * l1)
                + 28 * u * d2 + 2 * u * a * rs)
        assert out[0] >= need, terms
