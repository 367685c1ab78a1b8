"""Convs over repeated parent rows on the folded kernel (conv_fold.hip).

A BF16 layer that gathers parent rows behind an affine + SiLU pass sums the
weights of the offsets that reach one parent (three BF16 terms a sum) and
multiplies 8 parents instead of 27 children.  Against the 27-offset kernel
(S3DX_CONV_TILING=21): both accumulate in FP32 and round once to BF16, and the
folded weights are within 2^-27 of the sums, so the outputs differ by at most
one BF16 step here and there (rel-L2 far below 2^-9).  Parent tiles whose map
is not a subdivide's, or rows that hold an infinity, go to the 27-offset
kernel: those outputs are the same bits.
"""
import ctypes as C

import numpy as np
import pytest

from helpers import check_rel

pytestmark = pytest.mark.gpu


def _setup(s3dx, W, parents, cin, cout, silu=False, seed=70):
    p = parents.shape[0]
    _, kd = s3dx.subdivide2(s3dx.DeviceArray.from_host(parents), p, True)
    x = W.round_bf16(W.normal_f32(seed, 1, (p, cin)))
    scale, shift = W.normal_f32(seed, 2, (cin,), 0.2) + 1.0, W.normal_f32(seed, 3, (cin,), 0.2)
    ds, dh = s3dx.DeviceArray.from_host(scale), s3dx.DeviceArray.from_host(shift)
    w, b = W.conv_weight(seed, 4, cin, cout, layout="mesh"), W.normal_f32(seed, 5, (cout,), 0.1)
    conv = (s3dx.SparseConv(cin, cout, 27, s3dx.BF16).set_weights(w, s3dx.WEIGHT_MESH, b).set_gather_parent(True)
            .set_input_affine_silu(ds, dh).set_silu(silu))
    return conv, kd.download(), x, w, b, scale, shift


def _run(s3dx, W, conv, x, kmap, cout, n_out=None):
    n = kmap.shape[0] if n_out is None else n_out
    y = s3dx.DeviceArray((n, cout), np.uint16)
    conv.run(s3dx.DeviceArray.from_host(W.f32_to_bf16_bits(x)), x.shape[0], s3dx.DeviceArray.from_host(kmap), n, y,
             s3dx.BF16)
    return y.download()


def _general(s3dx, W, monkeypatch, *args, **kw):
    monkeypatch.setenv("S3DX_CONV_TILING", "21")
    y = _run(s3dx, W, *args, **kw)
    monkeypatch.delenv("S3DX_CONV_TILING")
    return y


@pytest.mark.parametrize("p,cin,cout,silu,cols", [
    (6007, 192, 96, False, 32),   # one column block a workgroup; a ragged last parent tile
    (20011, 192, 96, True, 32),   # the same in two passes over the CUs
    (24011, 192, 96, True, 96),   # three
    (12801, 64, 192, False, 96),  # one chunk; a last tile of one parent
    (9000, 128, 128, False, 64),  # column blocks in twos
    (4000, 768, 192, False, 32),  # the mesh decoder's first level
])
def test_folded_matches_general_and_oracle(s3dx, O, W, monkeypatch, p, cin, cout, silu, cols):
    parents = W.shells_union(0)[:p]
    conv, kmap, x, w, b, scale, shift = _setup(s3dx, W, parents, cin, cout, silu)
    print(f"fold p={p} {cin}->{cout} silu={silu}: {conv.plan(p, 8 * p)}", flush=True)
    assert f" fold rows=1024 cols={cols} grid={(p + 127) // 128}x{cout // cols} else mfma tiling=21 " in conv.plan(p, 8 * p)
    got = _run(s3dx, W, conv, x, kmap, cout)
    assert np.array_equal(got, _run(s3dx, W, conv, x, kmap, cout)), "two runs differ"
    want = _general(s3dx, W, monkeypatch, conv, x, kmap, cout)
    g, v = W.bf16_bits_to_f32(got).reshape(got.shape), W.bf16_bits_to_f32(want).reshape(got.shape)
    rel = float(np.linalg.norm(g - v) / np.linalg.norm(v))
    print(f"  against the 27-offset kernel: rel-L2 {rel:.2e}, same bits {np.mean(got == want):.4f}", flush=True)
    assert 0.0 < rel < 2.0 ** -11
    rows = np.sort(np.random.default_rng(1).choice(8 * p, 1500, replace=False))
    rows = np.unique(np.concatenate([rows, [0, 1023, 1024, 8 * p - 1]]))
    a = W.round_bf16(O.silu((x * scale + shift).astype(np.float32)))
    km = np.where(kmap[rows] >= 0, kmap[rows] >> 3, -1).astype(np.int32)
    ref = O.conv(a, km, p, W.round_bf16(w), 1, cout, b)
    check_rel(g[rows], O.silu(ref) if silu else ref, 1e-2, "oracle")


def test_maps_no_subdivide_made(s3dx, W, monkeypatch):
    # Tiles with an entry that does not reach the parent its siblings reach
    # run the 27-offset kernel (the same bits); the other tiles are folded.
    p, cin, cout = 8000, 192, 96
    conv, kmap, x, *_ = _setup(s3dx, W, W.shells_union(1)[:p], cin, cout)
    bad = kmap.copy()
    bad[8 * 130 + 3, 14] = -1            # tile 1: a neighbour taken away
    bad[8 * 300 + 0, 26] = 8 * 4000 + 1  # tile 2: another parent's child
    bad[8 * 4000:8 * 4128] = np.random.default_rng(2).integers(-1, 8 * p, (1024, 27), dtype=np.int32)  # tile 31 and 32
    sib = bad.copy()
    j = sib[8 * 700 + 5, 13]
    sib[8 * 700 + 5, 13] = (j & ~7) | ((j + 3) & 7)  # a sibling: the same parent row, so still foldable
    got, want = _run(s3dx, W, conv, x, bad, cout), _general(s3dx, W, monkeypatch, conv, x, bad, cout)
    for t in (1, 2, 31, 32):
        assert np.array_equal(got[1024 * t:1024 * (t + 1)], want[1024 * t:1024 * (t + 1)]), t
    assert not np.array_equal(got[:1024], want[:1024])  # folded
    assert np.array_equal(got, _run(s3dx, W, conv, x, sib, cout))
    # every tile irregular, then the subdivide's map again
    rnd = np.random.default_rng(3).integers(-1, 8 * p, kmap.shape, dtype=np.int32)
    assert np.array_equal(_run(s3dx, W, conv, x, rnd, cout), _general(s3dx, W, monkeypatch, conv, x, rnd, cout))
    none = np.full_like(kmap, -1)
    assert np.array_equal(_run(s3dx, W, conv, x, none, cout), _general(s3dx, W, monkeypatch, conv, x, none, cout))
    assert np.array_equal(_run(s3dx, W, conv, x, kmap, cout)[:1024], got[:1024])
    # fewer rows than eight per parent: the general kernel
    n = 8 * p - 8
    assert " fold " in conv.plan(p, 8 * p) and " fold " not in conv.plan(p, n)
    assert np.array_equal(_run(s3dx, W, conv, x, kmap[:n], cout, n), _general(s3dx, W, monkeypatch, conv, x, kmap[:n], cout, n))


def test_infinities_new_weights_and_sizes(s3dx, W, monkeypatch):
    # An infinite or NaN row sends the run to the 27-offset kernel (the folded
    # sum's terms may differ in sign); the next run folds again.  New
    # weights are folded anew; a larger set, then the first again.
    cin, cout = 192, 96
    conv, kmap, x, w, b, *_ = _setup(s3dx, W, W.shells_union(2)[:7000], cin, cout)
    first = _run(s3dx, W, conv, x, kmap, cout)
    for v in (np.inf, -np.inf, np.nan):
        xi = x.copy()
        xi[500, 7] = v
        assert np.array_equal(_run(s3dx, W, conv, xi, kmap, cout), _general(s3dx, W, monkeypatch, conv, xi, kmap, cout)), v
    assert np.array_equal(_run(s3dx, W, conv, x, kmap, cout), first)
    conv.set_weights(2.0 * w, s3dx.WEIGHT_MESH, 2.0 * b)  # (twice: exact in BF16)
    twice = _run(s3dx, W, conv, x, kmap, cout)
    assert np.array_equal(W.bf16_bits_to_f32(twice), 2.0 * W.bf16_bits_to_f32(first))
    big, kb, xb, *_ = _setup(s3dx, W, W.shells_union(2)[:12000], cin, cout)
    conv.set_weights(w, s3dx.WEIGHT_MESH, b)
    assert np.array_equal(_run(s3dx, W, conv, xb, kb, cout), _run(s3dx, W, big, xb, kb, cout))
    assert np.array_equal(_run(s3dx, W, conv, x, kmap, cout), first)
    # a weight whose folded sum overflows: the 27-offset kernel
    wh = w.copy()
    wh[:, 0, 0] = 2.0e38
    assert " fold " in conv.plan(7000, 56000)
    conv.set_weights(wh, s3dx.WEIGHT_MESH, b)
    assert " fold " not in conv.plan(7000, 56000)
    assert np.array_equal(_run(s3dx, W, conv, x, kmap, cout), _general(s3dx, W, monkeypatch, conv, x, kmap, cout))


@pytest.mark.parametrize("offsets", [(13, 14, 16), (13, 14, 26), (10, 13, 14)])
def test_folded_sums_keep_fp32s_bits(s3dx, W, offsets):
    # Two input channels with the same rows: one has weights 1, 2^-9 and 2^-17
    # at three offsets that reach slot 0's own parent (or two of them do), the
    # other -1 and -2^-9, so 2^-17 of the rows is left.  FP32 sums of the five
    # products (each rounded at 2^-24 of up to twice the row) keep it within
    # 5 * 2^-24 * 2 / 2^-17 < 2^-3.5 even if every rounding goes one way; the 27-offset
    # kernel's worst is 2^-4.9.  Sums held to 2^-18 lose it whole.
    p, cin, cout = 20011, 192, 96
    parents = W.shells_union(0)[:p]
    _, kd = s3dx.subdivide2(s3dx.DeviceArray.from_host(parents), p, True)
    kmap = kd.download()
    x = np.repeat(np.abs(W.round_bf16(W.normal_f32(130, 1, (p, 1)))) + 1.0, cin, 1).astype(np.float32)
    w = np.zeros((27, cout, cin), np.float32)
    for o, v in zip(offsets, (1.0, 2.0 ** -9, 2.0 ** -17)):
        w[o, :, 5] = v
    w[offsets[0], :, 37], w[offsets[1], :, 37] = -1.0, -2.0 ** -9
    one, none = s3dx.DeviceArray.from_host(np.ones(cin, np.float32)), s3dx.DeviceArray.from_host(np.zeros(cin, np.float32))
    conv = (s3dx.SparseConv(cin, cout, 27, s3dx.BF16).set_weights(w, s3dx.WEIGHT_MESH, None).set_gather_parent(True)
            .set_input_affine_silu(one, none))
    y = W.bf16_bits_to_f32(_run(s3dx, W, conv, W.round_bf16(x), kmap, cout)).reshape(8 * p, cout)
    xb = W.round_bf16(x)[:, 0].astype(np.float64)
    a = W.round_bf16((xb / (1.0 + np.exp(-xb))).astype(np.float32)).astype(np.float64)
    rows = kmap[:, list(offsets)]
    v = np.where(rows >= 0, a[np.maximum(rows, 0) >> 3], 0.0)
    want = v[:, 2] * 2.0 ** -17
    at = np.flatnonzero(rows[:, 2] >= 0)
    err = np.abs(y[at, 0] - want[at]) / np.abs(want[at])
    # (a row's own rounding to BF16 can go the other way where silu ties: 2^-8)
    assert " fold " in conv.plan(p, 8 * p)
    print(f"offsets {offsets}: worst {err.max():.2e}, median {np.median(err):.2e}", flush=True)
    assert err.max() < 2.0 ** -3.5 + 2.0 ** -8


class _Capture:
    """A HIP graph of what is enqueued on a stream inside the with block."""

    def __init__(self, stream):
        with open("/proc/self/maps") as f:
            self.hip = C.CDLL(next(line.split()[-1] for line in f if "libamdhip64" in line))
        self.stream, self.graph, self.exec = C.c_void_p(stream.handle), C.c_void_p(), C.c_void_p()

    def __enter__(self):
        assert self.hip.hipStreamBeginCapture(self.stream, 0) == 0
        return self

    def __exit__(self, *exc):
        assert self.hip.hipStreamEndCapture(self.stream, C.byref(self.graph)) == 0
        if exc[0] is None:
            assert self.hip.hipGraphInstantiate(C.byref(self.exec), self.graph, None, None, C.c_size_t(0)) == 0

    def launch(self):
        assert self.hip.hipGraphLaunch(self.exec, self.stream) == 0
        assert self.hip.hipStreamSynchronize(self.stream) == 0

    def close(self):
        for f, h in ((self.hip.hipGraphExecDestroy, self.exec), (self.hip.hipGraphDestroy, self.graph)):
            if h:
                f(h)


def test_new_weights_then_capture(s3dx, W):
    # The first run after set_weights is captured, and nothing has replayed it
    # when the next run is made: neither may see the weights before.
    p, cin, cout = 20011, 192, 96
    conv, kmap, x, w, b, *_ = _setup(s3dx, W, W.shells_union(0)[:p], cin, cout)
    xd, kd = s3dx.DeviceArray.from_host(W.f32_to_bf16_bits(x)), s3dx.DeviceArray.from_host(kmap)
    ys = [s3dx.DeviceArray((8 * p, cout), np.uint16) for _ in range(2)]
    stream = s3dx.Stream()

    def run(y):
        conv.run(xd, p, kd, 8 * p, y, s3dx.BF16, stream=stream)

    run(ys[0])
    stream.synchronize()
    first = ys[0].download()
    conv.set_weights(2.0 * w, s3dx.WEIGHT_MESH, 2.0 * b)  # (twice: exact in BF16)
    print("capture after set_weights", flush=True)
    with _Capture(stream) as graph:
        run(ys[1])
    for _ in range(3):
        run(ys[0])
        stream.synchronize()
        assert np.array_equal(W.bf16_bits_to_f32(ys[0].download()), 2.0 * W.bf16_bits_to_f32(first))
        ys[1].upload(np.zeros((8 * p, cout), np.uint16))
        graph.launch()
        assert np.array_equal(ys[1].download(), ys[0].download())
    graph.close()


def test_capture_with_no_room_yet(s3dx, W, monkeypatch):
    # A layer whose runs had no map records so far: the captured run can make none
    # and takes the 27-offset kernel; the next eager run is folded.
    p, cin, cout = 20011, 192, 96
    conv, kmap, x, *_ = _setup(s3dx, W, W.shells_union(0)[:p], cin, cout)
    xd, kd, y = s3dx.DeviceArray.from_host(W.f32_to_bf16_bits(x)), s3dx.DeviceArray.from_host(kmap), s3dx.DeviceArray((8 * p, cout), np.uint16)
    general = _general(s3dx, W, monkeypatch, conv, x, kmap, cout)
    stream = s3dx.Stream()
    print("capture before the first folded run", flush=True)
    with _Capture(stream) as graph:
        conv.run(xd, p, kd, 8 * p, y, s3dx.BF16, stream=stream)
    folded = _run(s3dx, W, conv, x, kmap, cout)
    for _ in range(3):
        graph.launch()
        assert np.array_equal(y.download(), general)
        assert np.array_equal(_run(s3dx, W, conv, x, kmap, cout), folded)
    graph.close()
    assert not np.array_equal(folded, general)


def test_refused_plan_leaves_nothing_behind(s3dx, W):
    # A plan of another size is refused before anything is enqueued: rows with an
    # infinity in that call do not send the next one to the 27-offset kernel.
    p, cin, cout = 9000, 192, 96
    conv, kmap, x, *_ = _setup(s3dx, W, W.shells_union(0)[:p], cin, cout)
    first = _run(s3dx, W, conv, x, kmap, cout)
    kd = s3dx.DeviceArray.from_host(kmap)
    gp = conv.gather_plan(p, kd, 8 * p - 8)
    xi = x.copy()
    xi[500, 7] = np.inf
    y = s3dx.DeviceArray((8 * p, cout), np.uint16)
    with pytest.raises(s3dx.S3dxError):
        conv.run(s3dx.DeviceArray.from_host(W.f32_to_bf16_bits(xi)), p, kd, 8 * p, y, s3dx.BF16, plan=gp)
    assert np.array_equal(_run(s3dx, W, conv, x, kmap, cout), first)


def _box(x, y, z):
    g = np.stack(np.meshgrid(np.arange(x), np.arange(y), np.arange(z), indexing="ij"), -1).reshape(-1, 3) + 2
    return np.ascontiguousarray(np.concatenate([np.zeros((len(g), 1), np.int64), g], 1).astype(np.int32))


def _against_both(s3dx, O, W, monkeypatch, parents, cin, cout):
    p = parents.shape[0]
    conv, kmap, x, w, b, scale, shift = _setup(s3dx, W, parents, cin, cout)
    assert " fold " in conv.plan(p, 8 * p)
    got = _run(s3dx, W, conv, x, kmap, cout)
    assert np.array_equal(got, _run(s3dx, W, conv, x, kmap, cout)), "two runs differ"
    want = _general(s3dx, W, monkeypatch, conv, x, kmap, cout)
    g, v = (W.bf16_bits_to_f32(t).reshape(t.shape) for t in (got, want))
    assert np.linalg.norm(g - v) < 2.0 ** -11 * np.linalg.norm(v)
    rows = np.unique(np.concatenate([np.random.default_rng(1).choice(8 * p, 1500, replace=False), [0, 8 * p - 1]]))
    a = W.round_bf16(O.silu((x * scale + shift).astype(np.float32)))
    km = np.where(kmap[rows] >= 0, kmap[rows] >> 3, -1).astype(np.int32)
    check_rel(g[rows], O.conv(a, km, p, W.round_bf16(w), 1, cout, b), 1e-2, "oracle")
    return np.mean((got == want).reshape(-1, 1024 * cout).all(1)) if p % 128 == 0 else None


@pytest.mark.parametrize("shape,cin,cout", [((16, 24, 60), 192, 96), ((16, 24, 64), 128, 128), ((7, 24, 64), 256, 192)])
def test_solid_sets(s3dx, O, W, monkeypatch, shape, cin, cout):
    # Solid sets name more parents in a tile (up to 768) than two halo buffers hold
    # (559): those tiles are folded over one buffer.
    parents = _box(*shape)
    km = O.kmap_subm3(parents, parents.shape[0])
    most = [len(np.unique(t[t < parents.shape[0]])) for t in np.split(km, range(128, len(km), 128))]
    print(f"{shape}: {max(most)} parents, {np.mean(np.array(most) > 559):.2f} of the tiles above 559", flush=True)
    assert max(most) > 700 and np.mean(np.array(most) > 559) > 0.5
    same = _against_both(s3dx, O, W, monkeypatch, parents, cin, cout)
    assert same is None or same < 0.05  # (nearly every tile is folded: none of the general kernel's bits)


def test_rows_in_no_order(s3dx, O, W, monkeypatch):
    # Parents in no order: every tile goes to the general kernel.
    c = W.shells_union(0)[:12800]
    same = _against_both(s3dx, O, W, monkeypatch, np.ascontiguousarray(c[np.random.default_rng(4).permutation(len(c))]), 192, 96)
    assert same == 1.0
