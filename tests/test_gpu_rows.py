"""BF16 convs by 512-row tiles (conv_rows.hip): Cin 96 over many rows, the mesh
decoder's last conv.  Against the split-K kernel (S3DX_CONV_TILING=19): both
accumulate in FP32 and round once to BF16, in different orders, so the outputs
differ by one BF16 step here and there (rel-L2 far below 2^-9).  Tiles without
all 27 offsets, of more rows than the LDS holds, or of rows further apart than
the plan's bitmap run the 64-row split-K kernel: the same bits.
"""
import numpy as np
import pytest

from helpers import check_rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cin,cout,residual,silu", [(96, 96, True, False), (32, 96, False, True), (160, 192, True, False)])
def test_rows_kernel(s3dx, O, W, monkeypatch, cin, cout, residual, silu):
    parents = W.shells_union(0)[:16421]
    p = parents.shape[0]
    n = 8 * p  # 257 tiles, the last of 296 rows
    _, kd = s3dx.subdivide2(s3dx.DeviceArray.from_host(parents), p, True)
    kmap = kd.download()
    whole = kmap.copy()
    kmap[512 * 3:512 * 4, 5] = -1                    # an offset that no row of the tile has
    kmap[100, 20] = n - 1                            # a row far away: 131,367 rows from the tile's first
    rng = np.random.default_rng(1)
    kmap[512 * 9:512 * 10] = rng.integers(-1, 16000, (512, 27), dtype=np.int32)  # too many rows
    kmap[512 * 256 + 3] = -1
    seed = 110
    x = W.round_bf16(W.normal_f32(seed, 1, (n, cin)))
    scale, shift = W.normal_f32(seed, 2, (cin,), 0.2) + 1.0, W.normal_f32(seed, 3, (cin,), 0.2)
    w, b = W.conv_weight(seed, 4, cin, cout, layout="mesh"), W.normal_f32(seed, 5, (cout,), 0.1)
    res = W.round_bf16(W.normal_f32(seed, 6, (p, cout)))
    conv = (s3dx.SparseConv(cin, cout, 27, s3dx.BF16).set_weights(w, s3dx.WEIGHT_MESH, b)
            .set_input_affine_silu(s3dx.DeviceArray.from_host(scale), s3dx.DeviceArray.from_host(shift))
            .set_residual_parent(True).set_silu(silu))
    xd = s3dx.DeviceArray.from_host(W.f32_to_bf16_bits(x))
    rd = s3dx.DeviceArray.from_host(W.f32_to_bf16_bits(res)) if residual else None

    text = conv.plan(n, n)
    print(text, flush=True)
    # (one tile more than the CUs, or two: the split-K kernel's)
    assert f" rows=512 cols=96 grid=256x{cout // 96} else mfma tiling=19 " in text

    def run(m):
        y = s3dx.DeviceArray((n, cout), np.uint16)
        conv.run(xd, n, s3dx.DeviceArray.from_host(m), n, y, s3dx.BF16, rd)
        return y.download()

    a = W.round_bf16(O.silu((x * scale + shift).astype(np.float32)))
    rows = np.unique(np.concatenate([np.sort(rng.choice(n, 1200, replace=False)), np.arange(512 * 3, 512 * 3 + 40),
                                     [100, 512 * 9 + 5, 512 * 256 + 3, n - 1]]))
    for name, m in (("subdivide's map", whole), ("with other tiles", kmap)):
        got = run(m)
        assert np.array_equal(got, run(m)), "two runs differ"
        monkeypatch.setenv("S3DX_CONV_TILING", "19")
        want = run(m)
        monkeypatch.delenv("S3DX_CONV_TILING")
        g, v = (W.bf16_bits_to_f32(t).reshape(t.shape) for t in (got, want))
        rel = float(np.linalg.norm(g - v) / np.linalg.norm(v))
        print(f"{cin}->{cout} {name}: rel-L2 against split-K {rel:.2e}", flush=True)
        assert 0.0 < rel < 2.0 ** -11
        if m is kmap:
            for t in (0, 3, 9, 256):  # the left tiles
                assert np.array_equal(got[512 * t:512 * t + 512], want[512 * t:512 * t + 512]), t
        ref = O.conv(a, m[rows], n, W.round_bf16(w), 1, cout, b)
        ref = O.silu(ref) if silu else ref
        check_rel(g[rows], ref + (res[rows >> 3] if residual else 0.0), 1e-2, "oracle")


def test_source_rows_above_2_24(s3dx, O, W, monkeypatch):
    # Cin 32: rows of 64 bytes, so that x below 2 GiB holds more than 2^24 rows.
    cin, cout, n_in, n = 32, 96, (1 << 24) + 40960, 512 * 512
    far = n_in - 40960  # every row that the map names; the rows 2^24 below are zeros
    rng = np.random.default_rng(3)
    x = np.zeros((n_in, cin), np.uint16)
    x[far:] = W.f32_to_bf16_bits(rng.standard_normal((40960, cin), np.float32)).reshape(-1, cin)
    kmap = (far + (np.arange(n)[:, None] // 64 * 5 + 31 * np.arange(27)) % 40960).astype(np.int32)
    w, b = W.conv_weight(120, 1, cin, cout, layout="mesh"), W.normal_f32(120, 2, (cout,), 0.1)
    one, none = s3dx.DeviceArray.from_host(np.ones(cin, np.float32)), s3dx.DeviceArray.from_host(np.zeros(cin, np.float32))
    conv = s3dx.SparseConv(cin, cout, 27, s3dx.BF16).set_weights(w, s3dx.WEIGHT_MESH, b).set_input_affine_silu(one, none)
    xd, kd, y = s3dx.DeviceArray.from_host(x), s3dx.DeviceArray.from_host(kmap), s3dx.DeviceArray((n, cout), np.uint16)
    print(f"rows above 2^24: {conv.plan(n_in, n)}", flush=True)
    assert " rows=512 " in conv.plan(n_in, n)
    conv.run(xd, n_in, kd, n, y, s3dx.BF16)
    rows = np.sort(rng.choice(n, 500, replace=False))
    a = W.round_bf16(O.silu(W.bf16_bits_to_f32(x[far:]).reshape(-1, cin)))
    ref = O.conv(a, kmap[rows] - far, 40960, W.round_bf16(w), 1, cout, b)
    check_rel(W.bf16_bits_to_f32(y.download()[rows]).reshape(-1, cout), ref, 1e-2, "oracle")


def test_a_plan_changes_nothing(s3dx, W):
    # 512-row tiles read no gather plan: a run that is given one is the same run.
    parents = W.shells_union(0)[:16421]
    p, cin = parents.shape[0], 96
    n = 8 * p
    _, kd = s3dx.subdivide2(s3dx.DeviceArray.from_host(parents), p, True)
    x = s3dx.DeviceArray.from_host(W.f32_to_bf16_bits(W.normal_f32(140, 1, (n, cin))))
    one, none = s3dx.DeviceArray.from_host(np.ones(cin, np.float32)), s3dx.DeviceArray.from_host(np.zeros(cin, np.float32))
    conv = (s3dx.SparseConv(cin, cin, 27, s3dx.BF16).set_weights(W.conv_weight(140, 2, cin, cin, layout="mesh"), s3dx.WEIGHT_MESH, None)
            .set_input_affine_silu(one, none))
    gp = conv.gather_plan(n, kd, n)
    assert conv.plan(n, n, gp) == conv.plan(n, n) and " rows=512 " in conv.plan(n, n)
    ys = [s3dx.DeviceArray((n, cin), np.uint16) for _ in range(2)]
    conv.run(x, n, kd, n, ys[0], s3dx.BF16)
    conv.run(x, n, kd, n, ys[1], s3dx.BF16, plan=gp)
    assert np.array_equal(ys[0].download(), ys[1].download())
