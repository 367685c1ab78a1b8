"""FP32 3x3x3 convs as three BF16 terms (conv_f3.hip).

With a gather plan made for an FP32 layer (or, in a layer with input
transforms, records of its own) the six term products above 2^-27 of each
product are accumulated in FP32.  Their error against float64 must not exceed
the FP32 matrix instructions' on the same inputs (measured: a quarter to nine
tenths of it), and the FP32 gate (rel-L2 1e-5) holds far off.  Rows in LDS (up
to 719 distinct ones in a tile), rows gathered from memory, and infinities or
NaN, which take FP32 matrix instructions, are all reached.  Tiles of more distinct
rows than the LDS holds (719) are multiplied in two parts, tiles that the plan
keeps no slots for by five offsets' rows at a time (128 columns a workgroup) or
from memory.
"""
import numpy as np
import pytest

from helpers import rel_l2

pytestmark = pytest.mark.gpu


def _ref(x, kmap, w, b, mesh=False):
    """float64 sum over the offsets; w [cout][27][cin], or [27][cout][cin]."""
    w = np.asarray(w, np.float64).transpose(1, 0, 2) if not mesh else np.asarray(w, np.float64)
    y = np.tile(np.asarray(b, np.float64), (kmap.shape[0], 1))
    for o in range(27):
        at = np.flatnonzero((kmap[:, o] >= 0) & (kmap[:, o] < x.shape[0]))
        y[at] += x[kmap[at, o]].astype(np.float64) @ w[o].T
    return y


def _regions(c, runs):
    """Rows so that each 128 of them come from `runs` places of the set."""
    n = c.shape[0] // 128 * 128
    step = 128 // runs
    idx = np.arange(n).reshape(runs, -1, step).transpose(1, 0, 2).reshape(-1)
    return np.ascontiguousarray(c[idx])


def _points(step):
    g = np.stack(np.meshgrid(*(np.arange(0, 60, step),) * 3, indexing="ij"), -1).reshape(-1, 3)
    return np.ascontiguousarray(np.concatenate([np.zeros((len(g), 1), np.int64), g], 1).astype(np.int32))


def _shuffled(c):
    return np.ascontiguousarray(c[np.random.default_rng(5).permutation(len(c))])


def _box(x, y, z):
    g = np.stack(np.meshgrid(np.arange(x), np.arange(y), np.arange(z), indexing="ij"), -1).reshape(-1, 3) + 2
    return np.ascontiguousarray(np.concatenate([np.zeros((len(g), 1), np.int64), g], 1).astype(np.int32))


CASES = {
    # name: (coords, cin, cout, LayerNorm, columns a workgroup)
    "whole_row_ln": (lambda W: W.shells_union(0)[:12801], 128, 128, True, 128),
    "two_blocks": (lambda W: W.shells_union(0)[:9000], 64, 192, False, 64),
    "one_block_ragged_cout": (lambda W: W.shells_union(1)[:6007], 128, 90, False, 32),
    "wide_separate_ln": (lambda W: W.shells_union(2)[:6001], 96, 256, True, None),
    "two_places": (lambda W: _regions(W.shells_union(0)[:12800], 2), 64, 128, False, None),    # 560 to 719 rows
    "four_places": (lambda W: _regions(W.shells_union(0)[:12800], 4), 64, 128, False, None),   # around 719
    "eight_places": (lambda W: _regions(W.shells_union(0)[:12800], 8), 96, 64, False, None),   # above: two parts
    "solid_box": (lambda W: _box(22, 22, 22), 64, 128, False, None),                           # about 560 rows
    "solid_bar": (lambda W: _box(16, 24, 60), 64, 128, False, 128),                            # up to 750: two parts
    "solid_bar_two_k": (lambda W: _box(12, 15, 60), 64, 192, False, 64),
    "solid_bar_four_k": (lambda W: _box(12, 24, 60), 64, 96, False, 32),
    "shuffled_whole_row": (lambda W: _shuffled(W.shells_union(0)[:12801]), 128, 128, True, 128),
    "shuffled_two_k": (lambda W: _shuffled(W.shells_union(0)[:9000]), 64, 192, False, 64),
    "shuffled_four_k": (lambda W: _shuffled(W.shells_union(0)[:9000]), 64, 96, False, 32),
    "shuffled": (lambda W: _shuffled(W.shells_union(0)[:12000]), 64, 128, False, None),        # the plan's global tiles
    "isolated_points": (lambda W: _points(3), 128, 128, False, None),                          # one offset
}


def _layer(s3dx, W, cin, cout, ln, seed=90):
    w, b = W.conv_weight(seed, 2, cin, cout), W.normal_f32(seed, 3, (cout,), 0.1)
    conv = s3dx.SparseConv(cin, cout, 27, s3dx.F32).set_weights(w, s3dx.WEIGHT_SLAT, b)
    if ln:
        conv.set_layernorm(True, 1e-6).set_silu(True)
    return conv, w, b


@pytest.mark.parametrize("name", list(CASES))
def test_error_no_larger_than_fp32(s3dx, O, W, name):
    make, cin, cout, ln, cols = CASES[name]
    coords = make(W)
    n = coords.shape[0]
    kmap = O.kmap_subm3(coords, n)
    conv, w, b = _layer(s3dx, W, cin, cout, ln)
    x, res = W.normal_f32(90, 1, (n, cin)), W.normal_f32(90, 4, (n, cout))
    xd, kd, rd = (s3dx.DeviceArray.from_host(a) for a in (x, kmap, res))
    gp = conv.gather_plan(n, kd, n)
    text = conv.plan(n, n, gp)
    print(f"{name}: n={n} {cin}->{cout}: {text}", flush=True)
    assert text.startswith("mfma tiling=25 terms=3 rows=128") and text.endswith(" plan=128"), text
    assert cols is None or f" cols={cols} " in text, text
    ys = [s3dx.DeviceArray((n, cout), np.float32) for _ in range(3)]
    conv.run(xd, n, kd, n, ys[0], s3dx.F32, rd, plan=gp)
    conv.run(xd, n, kd, n, ys[1], s3dx.F32, rd, plan=gp)
    conv.run(xd, n, kd, n, ys[2], s3dx.F32, rd)  # FP32 matrix instructions
    got, again, fp32 = (y.download() for y in ys)
    assert np.array_equal(got, again), "two runs differ"
    ref = _ref(x, kmap, w, b)
    if ln:
        ref = (ref - ref.mean(1, keepdims=True)) / np.sqrt(ref.var(1, keepdims=True) + 1e-6)
        ref = ref / (1.0 + np.exp(-ref))
    ref += res
    e, f = rel_l2(got, ref), rel_l2(fp32, ref)
    print(f"  rel-L2 three terms {e:.2e}, FP32 {f:.2e}", flush=True)
    assert e <= 1.05 * f and e < 1e-6, (e, f)
    worst = np.max(np.abs(got - ref)) / np.max(np.abs(ref))
    assert worst < 4e-6, worst


@pytest.mark.parametrize("scale", [2.0 ** -100, 2.0 ** 100])
def test_scales(s3dx, O, W, scale):
    # The terms keep FP32's exponent range.
    coords = W.shells_union(0)[:9000]
    n = coords.shape[0]
    kmap = O.kmap_subm3(coords, n)
    conv, w, _ = _layer(s3dx, W, 64, 128, False)
    conv.set_weights(w, s3dx.WEIGHT_SLAT, None)
    x = W.normal_f32(91, 1, (n, 64))
    kd = s3dx.DeviceArray.from_host(kmap)
    gp = conv.gather_plan(n, kd, n)
    y = s3dx.DeviceArray((n, 128), np.float32)
    conv.run(s3dx.DeviceArray.from_host((x * np.float32(scale)).astype(np.float32)), n, kd, n, y, s3dx.F32, plan=gp)
    assert rel_l2(y.download().astype(np.float64) / scale, _ref(x, kmap, w, np.zeros(128))) < 1e-6


@pytest.mark.parametrize("places", [1, 8])
def test_infinities_nan_and_large_values(s3dx, O, W, places):
    coords = _regions(W.shells_union(0)[:9088], places)
    n = coords.shape[0]
    kmap = O.kmap_subm3(coords, n)
    conv, w, b = _layer(s3dx, W, 64, 128, False)
    x = W.normal_f32(92, 1, (n, 64))
    clean = x.copy()
    x[500, 3], x[3000, 9], x[3000, 10], x[6000, 1] = np.inf, -np.inf, np.inf, np.nan
    x[8000, 5] = np.finfo(np.float32).max  # its first term would be infinite
    kd = s3dx.DeviceArray.from_host(kmap)
    gp = conv.gather_plan(n, kd, n)
    ys = [s3dx.DeviceArray((n, 128), np.float32) for _ in range(3)]
    xd = s3dx.DeviceArray.from_host(x)
    conv.run(xd, n, kd, n, ys[0], s3dx.F32, plan=gp)
    conv.run(xd, n, kd, n, ys[1], s3dx.F32)
    conv.run(s3dx.DeviceArray.from_host(clean), n, kd, n, ys[2], s3dx.F32, plan=gp)
    got, want, ok = (y.download() for y in ys)
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isposinf(got), np.isposinf(want))
    assert np.array_equal(np.isneginf(got), np.isneginf(want)) and np.isinf(want).any() and np.isnan(want).any()
    fin = np.isfinite(want)
    assert np.all(np.abs(got[fin].astype(np.float64) - want[fin]) <= 1e-5 * np.maximum(1.0, np.abs(want[fin].astype(np.float64))))
    assert np.isfinite(ok).all()


def test_weights_without_terms(s3dx, O, W):
    # An infinite weight: the layer keeps to FP32 matrix instructions.
    coords = W.shells_union(0)[:9000]
    n = coords.shape[0]
    kmap = O.kmap_subm3(coords, n)
    conv, w, b = _layer(s3dx, W, 64, 128, False)
    w[3, 13, 5] = np.inf
    conv.set_weights(w, s3dx.WEIGHT_SLAT, b)
    kd = s3dx.DeviceArray.from_host(kmap)
    gp = conv.gather_plan(n, kd, n)
    assert "terms=3" not in conv.plan(n, n, gp)
    xd = s3dx.DeviceArray.from_host(W.normal_f32(93, 1, (n, 64)))
    ys = [s3dx.DeviceArray((n, 128), np.float32) for _ in range(2)]
    conv.run(xd, n, kd, n, ys[0], s3dx.F32, plan=gp)
    conv.run(xd, n, kd, n, ys[1], s3dx.F32)
    assert np.array_equal(ys[0].download(), ys[1].download(), equal_nan=True)


def _mesh(s3dx, W, p, cin, cout, parent, seed=95):
    parents = W.shells_union(0)[:p]
    _, kd = s3dx.subdivide2(s3dx.DeviceArray.from_host(parents), p, True)
    rows = p if parent else 8 * p
    x = W.normal_f32(seed, 1, (rows, cin))
    scale, shift = W.normal_f32(seed, 2, (cin,), 0.2) + 1.0, W.normal_f32(seed, 3, (cin,), 0.2)
    w, b = W.conv_weight(seed, 4, cin, cout, layout="mesh"), W.normal_f32(seed, 5, (cout,), 0.1)
    conv = (s3dx.SparseConv(cin, cout, 27, s3dx.F32).set_weights(w, s3dx.WEIGHT_MESH, b).set_gather_parent(parent)
            .set_input_affine_silu(s3dx.DeviceArray.from_host(scale), s3dx.DeviceArray.from_host(shift)))
    v = x.astype(np.float64) * scale + shift
    return conv, kd.download(), x, (v / (1.0 + np.exp(-v))), w, b


def _run(s3dx, conv, x, kmap, cout):
    y = s3dx.DeviceArray((kmap.shape[0], cout), np.float32)
    conv.run(s3dx.DeviceArray.from_host(x), x.shape[0], s3dx.DeviceArray.from_host(kmap), kmap.shape[0], y, s3dx.F32)
    return y.download()


@pytest.mark.parametrize("p,cin,cout,parent", [
    (3001, 192, 96, True),    # folded, a ragged last tile
    (1500, 64, 128, True),
    (2003, 96, 96, False),    # the map's records built in the run
    (1100, 192, 192, False),
])
def test_layers_with_transforms(s3dx, W, monkeypatch, p, cin, cout, parent):
    conv, kmap, x, h, w, b = _mesh(s3dx, W, p, cin, cout, parent)
    text = conv.plan(x.shape[0], 8 * p)
    print(f"p={p} {cin}->{cout} parent={parent}: {text}", flush=True)
    assert (f" fold terms=3 rows=512 cols=32 grid={(p + 127) // 128 * 2}x{cout // 32} else " if parent else " tiling=25 terms=3 rows=128 ") in text
    assert parent or text.endswith(" plan=own")
    got = _run(s3dx, conv, x, kmap, cout)
    assert np.array_equal(got, _run(s3dx, conv, x, kmap, cout)), "two runs differ"
    monkeypatch.setenv("S3DX_CONV_TILING", "11")
    fp32 = _run(s3dx, conv, x, kmap, cout)
    monkeypatch.delenv("S3DX_CONV_TILING")
    assert not np.array_equal(got, fp32)  # (the FP32 kernel, that is)
    km = np.where(kmap >= 0, kmap >> 3, -1) if parent else kmap
    ref = _ref(h, km, w, b, mesh=True)
    e, f = rel_l2(got, ref), rel_l2(fp32, ref)
    print(f"  rel-L2 {e:.2e}, FP32 {f:.2e}", flush=True)
    assert e <= 1.05 * f and e < 2e-6, (e, f)


@pytest.mark.parametrize("shape", [(6, 24, 64), (16, 24, 60)])
def test_folded_solid_sets(s3dx, O, W, monkeypatch, shape):
    # Solid sets name more than 719 parents in a tile: two parts.
    parents = _box(*shape)
    monkeypatch.setattr(W, "shells_union", lambda seed: parents)
    p, cin, cout = parents.shape[0], 64, 96
    km = O.kmap_subm3(parents, p)
    most = max(len(np.unique(km[i:i + 128][km[i:i + 128] < p])) for i in range(0, p, 128))
    conv, kmap, x, h, w, b = _mesh(s3dx, W, p, cin, cout, True)
    print(f"{shape}: {most} rows in a tile; {conv.plan(p, 8 * p)}", flush=True)
    assert most > 719 and " fold terms=3 " in conv.plan(p, 8 * p)
    ref = _ref(h, np.where(kmap >= 0, kmap >> 3, -1), w, b, mesh=True)
    got = _run(s3dx, conv, x, kmap, cout)
    assert rel_l2(got, ref) < 2e-6 and np.max(np.abs(got - ref)) < 1e-5 * np.max(np.abs(ref))


def test_folded_fp32_maps_and_infinities(s3dx, W, monkeypatch):
    # Tiles no subdivide made, and rows with an infinity, run FP32 matrix
    # instructions: near the FP32 kernel's values, the same infinities and NaN.
    p, cin, cout = 3001, 64, 96
    conv, kmap, x, h, w, b = _mesh(s3dx, W, p, cin, cout, True)
    assert " fold terms=3 " in conv.plan(p, 8 * p)
    bad = kmap.copy()
    bad[8 * 130 + 3, 14] = -1
    bad[8 * 300, 26] = 8 * 2000 + 1
    bad[8 * 1500:8 * 1600] = np.random.default_rng(2).integers(-1, 8 * p, (800, 27), dtype=np.int32)
    for m in (bad, np.full_like(kmap, -1)):
        assert rel_l2(_run(s3dx, conv, x, m, cout), _ref(h, np.where(m >= 0, m >> 3, -1), w, b, mesh=True)) < 2e-6
    xi = x.copy()
    xi[700, 3], xi[900, 1] = np.inf, np.nan
    got = _run(s3dx, conv, xi, kmap, cout)
    monkeypatch.setenv("S3DX_CONV_TILING", "11")
    want = _run(s3dx, conv, xi, kmap, cout)
    monkeypatch.delenv("S3DX_CONV_TILING")
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isinf(got), np.isinf(want)) and np.isnan(want).any()
    first = _run(s3dx, conv, x, kmap, cout)
    assert rel_l2(first, _ref(h, np.where(kmap >= 0, kmap >> 3, -1), w, b, mesh=True)) < 2e-6


def test_a_bf16_layers_plan_changes_nothing(s3dx, W):
    # A layer with transforms makes records of its own; with a plan that it cannot
    # read (one made for a BF16 layer) it still does.
    conv, kmap, x, h, w, b = _mesh(s3dx, W, 2003, 96, 96, False)
    n = x.shape[0]
    kd, xd = s3dx.DeviceArray.from_host(kmap), s3dx.DeviceArray.from_host(x)
    other = s3dx.SparseConv(128, 128, 27, s3dx.BF16)
    gp = other.gather_plan(n, kd, n)
    assert conv.plan(n, n, gp) == conv.plan(n, n) and conv.plan(n, n).endswith(" plan=own")
    ys = [s3dx.DeviceArray((n, 96), np.float32) for _ in range(2)]
    conv.run(xd, n, kd, n, ys[0], s3dx.F32)
    conv.run(xd, n, kd, n, ys[1], s3dx.F32, plan=gp)
    assert np.array_equal(ys[0].download(), ys[1].download())


@pytest.mark.parametrize("n,cin,cout", [(12801, 128, 128), (12801, 128, 96), (28265, 256, 512), (10366, 128, 128)])
def test_bf16_layers_over_an_fp32_layers_plan(s3dx, O, W, n, cin, cout):
    # A plan that an FP32 layer made serves BF16 layers as a 64-row plan does.
    coords = W.shells_union(0)[:n]
    kd = s3dx.kmap_subm3(s3dx.DeviceArray.from_host(coords), n, n)
    gp = s3dx.SparseConv(128, 128, 27, s3dx.F32).gather_plan(n, kd, n)
    conv = s3dx.SparseConv(cin, cout, 27, s3dx.BF16).set_weights(W.conv_weight(150, 1, cin, cout), s3dx.WEIGHT_SLAT, None)
    cols = 128 if cout % 128 == 0 else 96
    text = conv.plan(n, n, gp)
    assert text.startswith(f"mfma tiling=21 split-k halo rows=64 cols={cols} ") and text.endswith(" plan=64"), text
    x = s3dx.DeviceArray.from_host(W.f32_to_bf16_bits(W.normal_f32(150, 2, (n, cin))))
    ys = [s3dx.DeviceArray((n, cout), np.uint16) for _ in range(2)]
    conv.run(x, n, kd, n, ys[0], s3dx.BF16)
    conv.run(x, n, kd, n, ys[1], s3dx.BF16, plan=gp)
    assert np.array_equal(ys[0].download(), ys[1].download())


def test_plan_of_a_map_too_long_for_128_row_records(s3dx, W):
    # 15.5M rows: 2.2 GB of 128-row records, whose offsets have 31 bits; the plan is
    # made with the 64-row ones alone, and the FP32 layer ignores it.
    n = 15_500_000
    kd = s3dx.DeviceArray.from_host(np.zeros((n, 27), np.int32))
    conv = s3dx.SparseConv(32, 32, 27, s3dx.F32)
    print("plan of 15.5M rows", flush=True)
    gp = conv.gather_plan(n, kd, n)
    assert "terms=3" not in conv.plan(n, n, gp)
    s3dx.synchronize()


@pytest.mark.parametrize("xs,ws", [(2.0 ** -120, 1.0), (1.0, 2.0 ** -120), (2.0 ** -130, 1.0), (2.0 ** -60, 2.0 ** -60), (2.0 ** 60, 2.0 ** 40)])
def test_small_and_large_values(s3dx, O, W, xs, ws):
    # Values whose third term is subnormal or below (or, at 2^-130, which are
    # subnormal themselves), and sums that overflow at the kernel's scale: no larger
    # an error than the FP32 instructions'.
    coords = W.shells_union(0)[:9000]
    n = coords.shape[0]
    kmap = O.kmap_subm3(coords, n)
    conv, w, _ = _layer(s3dx, W, 64, 128, False)
    w = (w * np.float32(ws)).astype(np.float32)
    conv.set_weights(w, s3dx.WEIGHT_SLAT, None)
    x = (W.normal_f32(91, 1, (n, 64)) * np.float32(xs)).astype(np.float32)
    kd, xd = s3dx.DeviceArray.from_host(kmap), s3dx.DeviceArray.from_host(x)
    gp = conv.gather_plan(n, kd, n)
    assert "terms=3" in conv.plan(n, n, gp)
    ys = [s3dx.DeviceArray((n, 128), np.float32) for _ in range(2)]
    conv.run(xd, n, kd, n, ys[0], s3dx.F32, plan=gp)
    conv.run(xd, n, kd, n, ys[1], s3dx.F32)
    ref = _ref(x, kmap, w, np.zeros(128))
    e, f = (float(np.linalg.norm(y.download() - ref) / np.linalg.norm(ref)) for y in ys)
    print(f"x {xs:.0e} w {ws:.0e}: rel-L2 three terms {e:.2e}, FP32 {f:.2e}", flush=True)
    assert e <= 1.05 * f, (e, f)


@pytest.mark.parametrize("ws", [2.0 ** -120, 2.0 ** 100])
def test_folded_fp32_small_and_large_sums(s3dx, W, monkeypatch, ws):
    p, cin, cout = 3001, 64, 96
    conv, kmap, x, h, w, b = _mesh(s3dx, W, p, cin, cout, True)
    w = (w * np.float32(ws)).astype(np.float32)
    conv.set_weights(w, s3dx.WEIGHT_MESH, None)
    assert " fold terms=3 " in conv.plan(p, 8 * p)
    got = _run(s3dx, conv, x, kmap, cout)
    monkeypatch.setenv("S3DX_CONV_TILING", "11")
    fp32 = _run(s3dx, conv, x, kmap, cout)
    monkeypatch.delenv("S3DX_CONV_TILING")
    ref = _ref(h, np.where(kmap >= 0, kmap >> 3, -1), w, np.zeros(cout), mesh=True)
    e, f = (float(np.linalg.norm(y - ref) / np.linalg.norm(ref)) for y in (got, fp32))
    print(f"w {ws:.0e}: rel-L2 {e:.2e}, FP32 {f:.2e}", flush=True)
    assert e <= 1.05 * f, (e, f)


def test_long_sums(s3dx, O, W):
    # 2048 channels, 55,296 products an output: float64 on sampled rows.
    coords = W.shells_union(0)[:20000]
    n, cin, cout = coords.shape[0], 2048, 128
    kmap = O.kmap_subm3(coords, n)
    conv, w, b = _layer(s3dx, W, cin, cout, True)
    x = np.random.default_rng(160).standard_normal((n, cin), np.float32)
    kd, xd = s3dx.DeviceArray.from_host(kmap), s3dx.DeviceArray.from_host(x)
    gp = conv.gather_plan(n, kd, n)
    assert "terms=3 rows=128 cols=128" in conv.plan(n, n, gp)
    ys = [s3dx.DeviceArray((n, cout), np.float32) for _ in range(2)]
    conv.run(xd, n, kd, n, ys[0], s3dx.F32, plan=gp)
    conv.run(xd, n, kd, n, ys[1], s3dx.F32)
    rows = np.sort(np.random.default_rng(161).choice(n, 600, replace=False))
    ref = _ref(x, kmap[rows], w, b)
    ref = (ref - ref.mean(1, keepdims=True)) / np.sqrt(ref.var(1, keepdims=True) + 1e-6)
    ref = ref / (1.0 + np.exp(-ref))
    e, f = (rel_l2(y.download()[rows], ref) for y in ys)
    print(f"2048 -> 128: rel-L2 three terms {e:.3e}, FP32 {f:.3e}", flush=True)
    assert e <= f, (e, f)
