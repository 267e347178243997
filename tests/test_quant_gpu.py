"""HIP quantizers vs the golden vectors, the oracle and the reference digests (runs on the MI355X)."""
import hashlib
import json
import os
import sys

import numpy as np
import pytest

from oracle import quants
from seedpack_amd import device as dev
from seedpack_amd import synth
from seedpack_amd.gpuquant import GPUQuant, quantize_into
from seedpack_amd.requant import QFUN, row_size

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIP_TYPES = [8, 2, 3, 6, 7, 42, 10, 11, 12, 13, 14, 20, 23, 16, 17, 18, 19, 21, 22, 29]
NEED_IMX = {16, 17, 19}


def say(*a):
    print(*a, file=sys.stderr, flush=True)


@pytest.fixture(scope="module")
def gq():
    return GPUQuant()


def hip(gq, t, bits, imx, variant=0):
    return gq.quantize_tensors(t, [(bits.reshape(-1), bits.shape[-1])], [imx], variant)[0]


@pytest.mark.parametrize("t", HIP_TYPES)
def test_hip_matches_golden_small(golden_small, gq, t):
    n = 0
    for name in ("normal", "student", "edge"):
        b = golden_small[f"in_{name}"]
        for variant in range(2 if t == 29 else 1):
            for use in ("none", "imx"):
                key = f"q_{name}_{t}_{variant}_{use}"
                if key not in golden_small:
                    continue
                say("case", key)
                got = hip(gq, t, b, golden_small["imatrix"] if use == "imx" else None, variant)
                want = golden_small[key]
                bad = np.flatnonzero(got != want)
                assert bad.size == 0, f"{key}: {bad.size} bytes differ, first at {bad[:8]}"
                n += 1
    assert n >= 3


@pytest.mark.parametrize("t", HIP_TYPES)
def test_hip_matches_oracle_seeded(gq, t):
    g = np.random.Generator(np.random.PCG64(0xA11CE + t))
    b = synth.normal_bf16(g, (96, 2048), 0.02, outlier_frac=0.002)
    imx = g.lognormal(0, 1, 2048).astype(np.float32)
    x = synth.bf16_to_f32(b).reshape(b.shape)
    for w in (None, imx):
        if w is None and t in NEED_IMX:
            continue
        for variant in range(2 if t == 29 else 1):
            say("case seeded", t, "imx" if w is not None else "none", "variant", variant)
            got = hip(gq, t, b, w, variant)
            want = quants.quantize(t, x, w, variant)
            bad = np.flatnonzero(got != want)
            assert bad.size == 0, f"{bad.size} bytes differ, first at {bad[:8]}"


def _manifest():
    p = os.path.join(ROOT, "tests", "golden", "quant_sha256.json")
    return json.load(open(p)) if os.path.exists(p) else {}


@pytest.mark.parametrize("key", sorted(_manifest()))
def test_hip_full_size_matches_reference_digest(gq, key):
    ent = _manifest()[key]
    cfg, ti, t, variant = key.split("_")
    cfg, ti, t, variant = int(cfg[3:]), int(ti[1:]), int(t), int(variant)
    if t not in HIP_TYPES:
        pytest.skip(f"type {t} not built")
    say("case full", key)
    w, imx = synth.tensor(cfg, ti)
    got = hip(gq, t, w, imx, variant)
    assert got.size == ent["nbytes"]
    assert hashlib.sha256(got.tobytes()).hexdigest() == ent["sha256"]


@pytest.mark.parametrize("t", [8, 2, 12, 14])
def test_source_kinds_agree(gq, t):
    """bf16 bits, f32 and f16 copies of the same values give the same bytes"""
    g = np.random.Generator(np.random.PCG64(77))
    b = synth.normal_bf16(g, (16, 1024), 0.02)
    x = synth.bf16_to_f32(b).reshape(b.shape)
    imx = g.lognormal(0, 1, 1024).astype(np.float32)
    ref_bytes = hip(gq, t, b, imx)
    assert hip(gq, t, x, imx).tobytes() == ref_bytes.tobytes()
    xh = x.astype(np.float16)
    if np.array_equal(xh.astype(np.float32), x):
        assert hip(gq, t, xh, imx).tobytes() == ref_bytes.tobytes()


@pytest.mark.parametrize("t", [8, 2, 10, 12])
def test_row_split_invariance(gq, t):
    """rows are quantized independently: any split of the rows gives the same bytes"""
    g = np.random.Generator(np.random.PCG64(5))
    b = synth.normal_bf16(g, (37, 512), 0.02)
    imx = g.lognormal(0, 1, 512).astype(np.float32)
    whole = hip(gq, t, b, imx)
    rb = row_size(t, 512)
    for k in (1, 13, 36):
        a = hip(gq, t, b[:k], imx)
        c = hip(gq, t, b[k:], imx)
        assert np.concatenate([a, c]).tobytes() == whole.tobytes()
        assert a.size == k * rb


def test_zero_rows_is_a_no_op():
    src = dev.DeviceArray(512, np.uint16).zero()
    dst = dev.DeviceArray(16, np.uint8)
    quantize_into(12, dev.DeviceArray(0, np.uint16), 256, dst)
    dev.synchronize()
    del src


@pytest.mark.parametrize("t", [2, 3, 6, 7])
def test_legacy_imatrix_rows_with_half_tile(gq, t):
    """the BF16 row pre-pass of the imatrix legacy quantizers: rows of n_per_row % 64 == 32 (a half
    tile at the end) and a row count that leaves a partial workgroup, against the oracle; the F32 copy
    (the per-lane pre-pass) gives the same bytes"""
    g = np.random.Generator(np.random.PCG64(0xB0 + t))
    b = synth.normal_bf16(g, (70, 1056), 0.02, outlier_frac=0.002)
    imx = g.lognormal(0, 1, 1056).astype(np.float32)
    x = synth.bf16_to_f32(b).reshape(b.shape)
    say("case legacy half tile", t)
    got = hip(gq, t, b, imx)
    want = quants.quantize(t, x, imx)
    bad = np.flatnonzero(got != want)
    assert bad.size == 0, f"{bad.size} bytes differ, first at {bad[:8]}"
    assert hip(gq, t, x, imx).tobytes() == got.tobytes()


@pytest.mark.parametrize("t", [2, 3, 6, 7])
def test_legacy_imatrix_with_and_without_scratch(gq, t):
    """the imatrix Q4_0/Q4_1/Q5_0/Q5_1 with the row mean squares from the first launch (scratch) and
    computed inside the quantizer (no scratch): the same bytes, equal to the oracle's, on row lengths
    that leave a partial 128-column tile (32, 96, 160, 4128) and row counts that leave a partial
    32-row group, for BF16, F16 and F32 sources"""
    from seedpack_amd._lib import check, lib
    g = np.random.Generator(np.random.PCG64(0xC0 + t))
    for rows, npr in ((1, 32), (31, 96), (33, 160), (70, 4128), (5, 12288)):
        b = synth.normal_bf16(g, (rows, npr), 0.02, outlier_frac=0.002)
        x = synth.bf16_to_f32(b).reshape(b.shape)
        imx = dev.DeviceArray.from_host(g.lognormal(0, 1, npr).astype(np.float32))
        want = quants.quantize(t, x, imx.to_host()) if rows * npr <= 70 * 4128 else None
        say("case legacy scratch", t, rows, npr)
        for kind, a in ((0, b), (1, x.astype(np.float16)), (2, x)):
            if kind == 1 and not np.array_equal(a.astype(np.float32), x):
                continue
            src = dev.DeviceArray.from_host(np.ascontiguousarray(a).reshape(-1))
            nbw = lib().spa_quantize_work_bytes(t, rows, npr, 1)
            assert nbw == (rows * 4 + 255) // 256 * 256
            work = dev.DeviceArray(nbw, np.uint8)
            outs = []
            for w in (work.ptr, None):
                dst = dev.DeviceArray(rows * row_size(t, npr), np.uint8)
                check(lib().spa_quantize(t, 0, src.ptr, kind, rows, npr, imx.ptr, dst.ptr, w, None))
                outs.append(dst.to_host())
            assert outs[0].tobytes() == outs[1].tobytes(), (t, rows, npr, kind)
            if want is not None:
                assert outs[0].tobytes() == want.tobytes(), (t, rows, npr, kind)


class _Lazy:
    """a quantized tensor as a quantizer input, dequantized into the launch's buffer (the reference's
    _Dequant, repo3.py:545-557)"""

    def __init__(self, gq, t, raw, npr):
        self.gq, self.t, self.raw, self.npr = gq, t, raw, npr
        self.size = raw.size // row_size(t, npr) * npr
        self.calls = 0

    def into(self, out):
        self.calls += 1
        self.gq.dequantize(self.t, self.raw, self.npr, out=out)


@pytest.mark.parametrize("t", [12, 14, 16])
def test_lazy_sources_and_launch_groups(gq, t):
    """sources written by into(out) (a seed's dequantized tensors) and groups of several tensors per
    device hand-over give the bytes of the same weights quantized one by one as float32 arrays; results
    arrive in order through on_result too"""
    say("case lazy sources", t)
    g = np.random.Generator(np.random.PCG64(40 + t))
    shapes = [(16, 256), (3, 512), (40, 256), (1, 1024), (9, 256)]
    seeds = [quants.quantize(14, (g.standard_normal(s) * 0.02).astype(np.float32), None) for s in shapes]
    lazies = [_Lazy(gq, 14, np.asarray(q, np.uint8), s[1]) for q, s in zip(seeds, shapes)]
    imx = [g.lognormal(0, 1, s[1]).astype(np.float32) for s in shapes]
    f32 = [gq.dequantize(14, np.asarray(q, np.uint8), s[1]).to_host().reshape(s) for q, s in zip(seeds, shapes)]
    want = [quants.quantize(t, x, w) for x, w in zip(f32, imx)]
    for mw in (1 << 28, 5000, 256):
        got = gq.quantize_tensors(t, [(z, s[1]) for z, s in zip(lazies, shapes)], imx, max_weights=mw)
        assert [a.tobytes() for a in got] == [np.asarray(w).tobytes() for w in want]
        seen = []
        gq.quantize_tensors(t, [(x.reshape(-1), s[1]) for x, s in zip(f32, shapes)], imx, max_weights=mw,
                            on_result=lambda k, y: seen.append((k, y.tobytes())))
        assert [k for k, _ in seen] == list(range(len(shapes)))
        assert [y for _, y in seen] == [np.asarray(w).tobytes() for w in want]
    assert all(z.calls == 3 for z in lazies)


def test_blocking_waits_give_the_same_bytes(gq):
    """with the library's waits blocking on an event (as the packer runs), host copies and stream
    waits hand over the same results as the spinning waits"""
    say("case blocking waits")
    g = np.random.Generator(np.random.PCG64(77))
    x = (g.standard_normal((64, 512)) * 0.02).astype(np.float32)
    imx = g.lognormal(0, 1, 512).astype(np.float32)
    want = np.asarray(quants.quantize(12, x, imx)).tobytes()
    prev = dev.set_blocking_waits(True)
    try:
        for _ in range(3):
            assert hip(gq, 12, x, imx).tobytes() == want
            back = dev.DeviceArray.from_host(x.reshape(-1)).to_host()
            assert back.tobytes() == x.tobytes()
    finally:
        dev.set_blocking_waits(prev)
    assert dev.set_blocking_waits(prev) is False
    assert hip(gq, 12, x, imx).tobytes() == want


@pytest.mark.parametrize("use_imx", [True, False])
@pytest.mark.parametrize("t", [20, 23])
def test_iq4_at_codebook_midpoints(gq, t, use_imx):
    """the codebook table of the IQ4 types at its edges: weights that a trial scales onto every midpoint of
    neighbouring codes, a float to each side of it, and the codebook's ends; sub-blocks of zeros and of
    tiny weights beside them"""
    kv = np.array([-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113], np.float32)
    mid = (kv[1:] + kv[:-1]) / 2
    vals = np.concatenate([mid, np.nextafter(mid, np.float32(-1e9)), np.nextafter(mid, np.float32(1e9)), kv[1:],
                           np.float32([113.5, -126.5, 0.0, -0.0, 1e-30])]).astype(np.float32)
    g = np.random.Generator(np.random.PCG64(20 + t))
    x = g.choice(vals, size=(24, 256)).reshape(24, 8, 32)
    x[:, :, 0] = -127                      # the block's largest: trial 0 scales by exactly 2^10
    x[3, 2] = 0
    x[5] = 0
    x[7, 1] *= np.float32(2.0 ** -60)
    x = (x * np.float32(2.0 ** -10)).reshape(24, 256)
    imx = g.lognormal(0, 1, 256).astype(np.float32) if use_imx else None
    got = gq.quantize_tensors(t, [(x.reshape(-1), 256)], [imx])[0]
    want = quants.quantize(t, x, imx)
    bad = np.flatnonzero(got != want)
    assert bad.size == 0, f"{bad.size} bytes differ, first at {bad[:8]}"


@pytest.mark.parametrize("use_imx", [True, False])
@pytest.mark.parametrize("t", [2, 6, 11, 14, 20, 23])
def test_infinite_and_nan_weights(gq, t, use_imx):
    """blocks with infinities, NaN and the largest finite values beside finite ones, and a zero
    importance: the trial searches take the same decisions as the C expressions there"""
    g = np.random.Generator(np.random.PCG64(5))
    x = (g.standard_normal((16, 512)) * 0.02).astype(np.float32)
    x[1, 5], x[2, 300], x[3, 7] = np.inf, -np.inf, np.nan
    x[4, 100:140] = np.inf
    x[5, 40:42] = np.inf, -np.inf
    x[6, 17:19] = 3e38, -3e38
    imx = g.lognormal(0, 1, 512).astype(np.float32)
    imx[17] = 0
    imx = imx if use_imx else None
    got = gq.quantize_tensors(t, [(x.reshape(-1), 512)], [imx])[0]
    with np.errstate(all="ignore"):
        want = quants.quantize(t, x, imx)
    assert np.array_equal(got, want)


def _lattice_edges(g):
    """rows of 256 for the lattice searches: equal magnitudes (every list has ties), two magnitudes, unit and
    zero importance, a huge weight where the importance is zero, sub-blocks scaled far down and up, zeros"""
    x = (g.standard_t(5, size=(40, 256)) * 0.01).astype(np.float32)
    imx = g.lognormal(0, 1, size=256).astype(np.float32)
    imx[37], imx[200:204] = 0, 0
    x[0] = 0.01 * np.sign(x[0])
    x[1] = np.where(np.arange(256) % 3 == 0, 0.01, 0.003) * np.sign(x[1])
    x[2] = np.round(x[2] * 500) / 500
    x[3, 37] = 1e5
    x[4, 37], x[4, 200] = -3e9, 1e30
    x[5] *= np.float32(1e-19)
    x[6] *= np.float32(1e-25)
    x[7] *= np.float32(1e19)
    x[8] *= np.repeat(np.float32([1, 1e-9, 1e-4, 1, 0, 1e-7, 1, 1e-14]), 32)
    x[9, ::2] = 0
    x[10] = np.abs(x[10])
    x[11:16] = np.round(x[11:16] * 64) / 64
    return x.astype(np.float32), imx


@pytest.mark.parametrize("which", ["imatrix", "unit", "none"])
@pytest.mark.parametrize("t", [16, 17, 18, 21, 22])
def test_lattice_searches_at_ties_and_extremes(gq, t, which):
    if which == "none" and t in NEED_IMX:
        pytest.skip("the type needs an importance matrix")
    x, imx = _lattice_edges(np.random.Generator(np.random.PCG64(900 + t)))
    imx = {"imatrix": imx, "unit": np.ones(256, np.float32), "none": None}[which]
    got = gq.quantize_tensors(t, [(x.reshape(-1), 256)], [imx])[0].reshape(len(x), -1)
    compared = 0
    for r in range(len(x)):
        try:
            want = np.asarray(quants.quantize(t, x[r:r + 1], imx))
        except ValueError:                       # no listed point at a finite distance: the reference asserts
            continue
        assert np.array_equal(got[r], want), f"row {r} differs"
        compared += 1
    assert compared >= len(x) - 4


def _on_grid(g, shape, kind):
    """BF16 weights as a model widened from another format has them: 4-bit codes with a scale per 32, three
    values with a scale per 128, and 4-bit codes with a quarter of the weights zero"""
    x = (g.standard_normal(shape) * 0.02).astype(np.float32)
    v = x.reshape(-1, 128 if kind == "ternary" else 32)
    if kind == "ternary":
        d = np.abs(v).mean(1, keepdims=True)
        v = np.clip(np.rint(v / d), -1, 1) * d
    else:
        d = (np.abs(v).max(1, keepdims=True) / 8).astype(np.float16).astype(np.float32)
        v = np.clip(np.rint(v / d), -8, 7) * d
        if kind == "sparse":
            v = np.where(g.random(v.shape) < 0.25, 0, v)
    return synth.bf16_bits(v.reshape(shape).astype(np.float32))


@pytest.mark.parametrize("use_imx", [True, False])
@pytest.mark.parametrize("kind", ["4-bit", "ternary", "sparse"])
@pytest.mark.parametrize("t", [16, 17, 18, 21, 22])
def test_lattice_searches_of_coarse_weights(gq, t, kind, use_imx):
    """equal distances at many trials of many lanes: the float sums decide, trials and lanes side by side"""
    if not use_imx and t in NEED_IMX:
        pytest.skip("the type needs an importance matrix")
    g = np.random.Generator(np.random.PCG64(70 + t))
    b = _on_grid(g, (128, 1024), kind)
    imx = g.lognormal(0, 1, 1024).astype(np.float32) if use_imx else None
    say("case coarse weights", t, kind, use_imx)
    got = hip(gq, t, b, imx)
    want = quants.quantize(t, synth.bf16_to_f32(b).reshape(b.shape), imx)
    bad = np.flatnonzero(got != want)
    assert bad.size == 0, f"{bad.size} bytes differ, first at {bad[:8]}"


@pytest.mark.parametrize("kind", ["4-bit", "ternary"])
@pytest.mark.parametrize("t", [18, 21, 22])
def test_coarse_weights_cost_little_more(gq, t, kind):
    """a matrix of coarse weights, without an importance matrix, within 2.2 times the time of one of the same
    size with normal weights: 1.35 at most when measured, and one search per trial takes the same for both; the
    lists searched one lane at a time made it 3.1 to 11.6"""
    g = np.random.Generator(np.random.PCG64(7))
    ms = []
    for b in (synth.normal_bf16(g, (2048, 4096), 0.02), _on_grid(g, (2048, 4096), kind)):
        src = dev.DeviceArray.from_host(b.reshape(-1))
        dst = dev.DeviceArray(2048 * row_size(t, 4096), np.uint8)
        times = []
        for _ in range(6):
            e0, e1 = dev.Event(), dev.Event()
            e0.record()
            quantize_into(t, src, 4096, dst)
            e1.record()
            dev.synchronize()
            times.append(e0.elapsed_ms(e1))
        ms.append(min(times))
    say("case coarse weights' time", t, kind, ms)
    assert ms[1] < 2.2 * ms[0]
