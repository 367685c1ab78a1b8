"""The work that a user of this library has it do, as cases that can be timed.

One sample of the path runs, in order: the occupancy's coordinates ("coords"),
the SLat tables of the voxel set ("tables"), the res blocks of the SLat flow
("slat", in each of the flow's forwards), and for the mesh the subdivide of the
voxel set ("subdivide") and an upsample block per level ("mesh"), the last one
with its linear head.  "conv" is a single 3x3x3 layer, as a program that uses
the operator by itself calls it.

Voxel sets are unions of spherical shells on a 64^3 grid, cut to a stated
number of rows in their (lexicographic) order; the mesh levels are the sets
that the subdivide makes of them.  Features are N(0, 1), weights
N(0, 1/sqrt(fan_in)) in float32, as a checkpoint holds them.

Each case: listed() names it, prepare() makes what a program holds before the
call, run() is one pass through the public entry points, exact() the same in
64 bits by plain torch.
"""
import importlib.util
import math
import random
import sys
from pathlib import Path

import numpy as np
import torch

_PKG = Path(__file__).resolve().parent.parent / "sam3d.cpp_amd"
RES = 64
GROUPS = 32
HEAD = 101


def _lib():
    """The package: a folder whose name holds a dot, imported as `s3dx`."""
    if "s3dx" not in sys.modules:
        spec = importlib.util.spec_from_file_location("s3dx", _PKG / "__init__.py",
                                                      submodule_search_locations=[str(_PKG)])
        mod = importlib.util.module_from_spec(spec)
        sys.modules["s3dx"] = mod
        spec.loader.exec_module(mod)
    return sys.modules["s3dx"]


def listed():
    return [
        # a single small layer: 64 channels on the shell of one sphere of radius 20
        {"name": "conv f32 64 10k", "kind": "conv", "n": 10366, "cin": 64, "cout": 64, "dtype": "f32"},
        # once per sample: the decoder's occupancy to the voxel set
        {"name": "coords 64^3", "kind": "coords", "res": 64, "density": 0.265},
        # once per sample: fine and coarse kernel maps, their gather plans, down/upsample tables
        {"name": "tables 28k", "kind": "tables", "n": 28265},
        # the largest map: the mesh decoder's second subdivide, to 256^3
        {"name": "subdivide 226k", "kind": "subdivide", "n": 28265, "level": 1},
        # the SLat flow's res blocks, 38 times per sample: input_blocks.0 ...
        {"name": "slat bf16 128 28k", "kind": "slat", "n": 28265, "cin": 128, "cout": 128, "dtype": "bf16",
         "join": "none"},
        # ... input_blocks.1, after the mean-pool to the coarse set ...
        {"name": "slat bf16 128-1024 down", "kind": "slat", "n": 5086, "cin": 128, "cout": 1024, "dtype": "bf16",
         "join": "down"},
        # ... out_blocks.0, on the concatenated and upsampled coarse rows
        {"name": "slat bf16 2048-128 up", "kind": "slat", "n": 28265, "cin": 2048, "cout": 128, "dtype": "bf16",
         "join": "up"},
        # the same blocks in the reference's own precision
        {"name": "slat f32 128 28k", "kind": "slat", "n": 28265, "cin": 128, "cout": 128, "dtype": "f32",
         "join": "none"},
        {"name": "slat f32 128-1024 down", "kind": "slat", "n": 5086, "cin": 128, "cout": 1024, "dtype": "f32",
         "join": "down"},
        # the mesh decoder's upsample blocks: 64^3 -> 128^3, and 128^3 -> 256^3 with the head
        {"name": "mesh bf16 768-192 28k", "kind": "mesh", "n": 28265, "level": 0, "cin": 768, "cout": 192,
         "dtype": "bf16", "head": False},
        {"name": "mesh bf16 192-96 226k", "kind": "mesh", "n": 28265, "level": 1, "cin": 192, "cout": 96,
         "dtype": "bf16", "head": True},
        # an upsample block in the reference's own precision, on a small object
        {"name": "mesh f32 768-192 6k", "kind": "mesh", "n": 6001, "level": 0, "cin": 768, "cout": 192,
         "dtype": "f32", "head": False},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["conv", "coords", "tables", "subdivide", "slat", "slat", "slat", "mesh", "mesh"])
    dtype = rng.choice(["bf16", "bf16", "f32"])
    if kind == "coords":
        return {"kind": kind, "res": rng.randint(24, 64), "density": rng.uniform(0.05, 0.3)}
    if kind == "tables":
        return {"kind": kind, "n": _log(rng, 1500, 42000)}
    if kind == "subdivide":
        level = rng.randint(0, 1)
        return {"kind": kind, "n": _log(rng, 1500, 28000 if level else 42000), "level": level}
    if kind == "conv":
        c = [32, 64, 96, 128, 160, 192, 256, 320, 512]
        return {"kind": kind, "n": _log(rng, 1500, 42000), "cin": rng.choice(c), "cout": rng.choice(c),
                "dtype": dtype}
    if kind == "slat":
        cin, cout, join = rng.choice([(128, 128, "none"), (128, 1024, "down"), (2048, 128, "up"),
                                      (256, 128, "cat")])
        n = _log(rng, 300, 8000) if join == "down" else _log(rng, 1500, 42000)
        return {"kind": kind, "n": n, "cin": cin, "cout": cout, "dtype": dtype, "join": join}
    level = rng.randint(0, 1)
    cin, cout = ((768, 192), (192, 96))[level]
    most = (42000, 28000)[level] if dtype == "bf16" else (7000, 4000)[level]
    return {"kind": kind, "n": _log(rng, 1000, most), "level": level, "cin": cin, "cout": cout, "dtype": dtype,
            "head": level == 1}


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
def _dev():
    return torch.device("cuda", 0)


def _shells(n, seed, enough):
    """Rows (0, x, y, z) in lexicographic order: shells of thickness 3 with
    centres in [12, 52]^3 and radii in [6, 14], added until enough(rows)."""
    r = random.Random("voxels %d %d" % (n, seed))
    ax = torch.arange(RES, dtype=torch.float64, device=_dev())
    gx, gy, gz = torch.meshgrid(ax, ax, ax, indexing="ij")
    mask = torch.zeros((RES, RES, RES), dtype=torch.bool, device=_dev())
    while True:
        for _ in range(2):
            c = [r.uniform(12.0, 52.0) for _ in range(3)]
            d = ((gx - c[0]) ** 2 + (gy - c[1]) ** 2 + (gz - c[2]) ** 2).sqrt()
            mask |= (d - r.uniform(6.0, 14.0)).abs() <= 1.5
        xyz = mask.nonzero()
        rows = torch.zeros((xyz.shape[0], 4), dtype=torch.int32, device=_dev())
        rows[:, 1:] = xyz.to(torch.int32)
        if enough(rows):
            return rows


def _voxels(n, seed):
    """A set of n rows: shells, up to row n."""
    return _shells(n, seed, lambda rows: rows.shape[0] >= n)[:n].contiguous()


def _voxels_down(m, seed):
    """A set that has m coarse rows: shells, up to coarse row m."""
    rows = _shells(m, seed, lambda rows: _coarse(rows)[0].shape[0] >= m)
    return rows[_coarse(rows)[1] < m].contiguous()


def _children(rows):
    """The 8 children of each row, (2x + bx, 2y + by, 2z + bz), z fastest."""
    bits = torch.tensor([[0, x, y, z] for x in (0, 1) for y in (0, 1) for z in (0, 1)], dtype=torch.int32,
                        device=rows.device)
    scale = torch.tensor([1, 2, 2, 2], dtype=torch.int32, device=rows.device)
    return (rows[:, None, :] * scale + bits).reshape(-1, 4).contiguous()


def _normal(seed, tag, shape, std=1.0, mean=0.0):
    g = torch.Generator(device=_dev())
    g.manual_seed((seed * 1000003 + tag) & 0x7FFFFFFFFFFF)
    return torch.randn(shape, generator=g, device=_dev(), dtype=torch.float32) * std + mean


def _rows(seed, tag, shape, dtype):
    return _normal(seed, tag, shape).to(torch.bfloat16 if dtype == "bf16" else torch.float32).contiguous()


def _weight(seed, tag, cin, cout, kvol, mesh=False):
    """float32 weights, [cout][kvol][cin], or [kvol][cout][cin] for the mesh layers."""
    return _normal(seed, tag, (kvol, cout, cin) if mesh else (cout, kvol, cin), 1.0 / math.sqrt(kvol * cin))


def _host(t):
    return t.cpu().numpy()


def _empty(shape, dtype):
    return torch.zeros(shape, dtype=dtype, device=_dev())


def _coarse(rows):
    """(coarse rows, fine_to_coarse) by plain torch."""
    c = rows.clone()
    c[:, 1:] //= 2
    u, inv = torch.unique(c, dim=0, return_inverse=True)
    return u.contiguous(), inv


# ---------------------------------------------------------------------------
# prepare
# ---------------------------------------------------------------------------
def prepare(case, seed):
    s3dx = _lib()
    st = {"case": case, "s3dx": s3dx}
    torch.cuda.synchronize()
    {"conv": _prepare_conv, "coords": _prepare_coords, "tables": _prepare_tables, "subdivide": _prepare_subdivide,
     "slat": _prepare_slat, "mesh": _prepare_mesh}[case["kind"]](st, case, seed)
    torch.cuda.synchronize()
    return st


def _ws(s3dx, nbytes):
    return s3dx.DeviceArray(max(int(nbytes), 1), np.uint8)


def _kmap(s3dx, rows, missing):
    n = rows.shape[0]
    out = torch.empty((n, 27), dtype=torch.int32, device=_dev())
    torch.cuda.synchronize()
    s3dx.kmap_subm3(rows.data_ptr(), n, missing, out.data_ptr(), _ws(s3dx, s3dx.kmap_workspace_size(n)))
    s3dx.synchronize()
    return out


def _dt(s3dx, case):
    return (s3dx.BF16, torch.bfloat16) if case["dtype"] == "bf16" else (s3dx.F32, torch.float32)


def _prepare_conv(st, case, seed):
    s3dx = st["s3dx"]
    n, cin, cout = case["n"], case["cin"], case["cout"]
    dt, tdt = _dt(s3dx, case)
    rows = _voxels(n, seed)
    st["kmap"] = _kmap(s3dx, rows, n)
    st["x"] = _rows(seed, 1, (n, cin), case["dtype"])
    st["y"] = _empty((n, cout), tdt)
    st["conv"] = s3dx.SparseConv(cin, cout, 27, dt).set_weights(
        _host(_weight(seed, 2, cin, cout, 27)), s3dx.WEIGHT_SLAT, _host(_normal(seed, 3, (cout,), 0.1)))
    st["plan"] = st["conv"].gather_plan(n, st["kmap"].data_ptr(), n)


def _occupancy(case, seed):
    from statistics import NormalDist
    r = case["res"]
    return _normal(seed, 7, (r, r, r), 1.0, -NormalDist().inv_cdf(1.0 - case["density"])).contiguous()


def _prepare_coords(st, case, seed):
    s3dx = st["s3dx"]
    r = case["res"]
    cells = r ** 3
    st["occ"] = _occupancy(case, seed)
    st["all"] = _empty((cells, 4), torch.int32)
    st["surface"] = _empty((cells, 4), torch.int32)
    st["down"] = _empty((42000, 4), torch.int32)
    st["ws"] = (_ws(s3dx, s3dx.occupancy_workspace_size((r, r, r))),
                _ws(s3dx, s3dx.prune_surface_workspace_size(cells)),
                _ws(s3dx, s3dx.downsample_coords_workspace_size(cells)))


def _prepare_tables(st, case, seed):
    s3dx = st["s3dx"]
    n = case["n"]
    st["rows"] = _voxels(n, seed)
    st["kmap"] = _empty((n, 27), torch.int32)
    st["coarse"] = _empty((n, 4), torch.int32)
    st["f2c"] = _empty((n,), torch.int32)
    st["child"] = _empty((8 * n,), torch.int32)
    st["inv"] = _empty((n,), torch.float32)
    st["kmap_c"] = _empty((n, 27), torch.int32)
    st["ws"] = (_ws(s3dx, s3dx.kmap_workspace_size(n)), _ws(s3dx, s3dx.coarsen2_workspace_size(n)))
    # the layers whose gather plans are kept with the maps: a fine and a coarse block's second conv
    st["conv_f"] = s3dx.SparseConv(128, 128, 27, s3dx.BF16)
    st["conv_c"] = s3dx.SparseConv(1024, 1024, 27, s3dx.BF16)
    torch.cuda.synchronize()
    fine = _kmap(s3dx, st["rows"], n)
    coarse = _coarse(st["rows"])[0]
    cmap = _kmap(s3dx, coarse, coarse.shape[0])
    st["plan_f"] = st["conv_f"].gather_plan(n, fine.data_ptr(), n)
    st["plan_c"] = st["conv_c"].gather_plan(coarse.shape[0], cmap.data_ptr(), coarse.shape[0])
    s3dx.synchronize()


def _prepare_subdivide(st, case, seed):
    s3dx = st["s3dx"]
    rows = _voxels(case["n"], seed)
    for _ in range(case["level"]):
        rows = _children(rows)
    p = rows.shape[0]
    st["rows"], st["p"] = rows, p
    st["child"] = _empty((8 * p, 4), torch.int32)
    st["kmap"] = _empty((8 * p, 27), torch.int32)
    st["ws"] = _ws(s3dx, s3dx.subdivide2_workspace_size(p))


def _slat_inputs(case, seed):
    """What a block is made of, as torch tensors; the float32 parameters whole.
    case["n"]: the rows that the block works on, coarse ones behind a mean-pool."""
    cin, cout, join = case["cin"], case["cout"], case["join"]
    t = {"rows": _voxels_down(case["n"], seed) if join == "down" else _voxels(case["n"], seed)}
    n = t["rows"].shape[0]
    t["coarse"], t["f2c"] = _coarse(t["rows"])
    nc = t["coarse"].shape[0]
    if join == "up":      # [trunk, skip] of the coarse rows, then nearest upsample
        t["a"], t["b"] = _rows(seed, 1, (nc, cin // 2), case["dtype"]), _rows(seed, 2, (nc, cin // 2), case["dtype"])
    elif join == "cat":   # [h, skip] of the fine rows
        t["a"], t["b"] = _rows(seed, 1, (n, cin // 2), case["dtype"]), _rows(seed, 2, (n, cin // 2), case["dtype"])
    else:
        t["a"] = _rows(seed, 1, (n, cin), case["dtype"])
    t["n1w"], t["n1b"] = _normal(seed, 3, (cin,), 0.2, 1.0), _normal(seed, 4, (cin,), 0.2)
    t["ms"], t["mh"] = _normal(seed, 5, (cout,), 0.3), _normal(seed, 6, (cout,), 0.3)
    t["w1"], t["b1"] = _weight(seed, 7, cin, cout, 27), _normal(seed, 8, (cout,), 0.1)
    t["w2"], t["b2"] = _weight(seed, 9, cout, cout, 27), _normal(seed, 10, (cout,), 0.1)
    if cin != cout:
        t["ws"], t["bs"] = _weight(seed, 11, cin, cout, 1), _normal(seed, 12, (cout,), 0.1)
    return t


def _prepare_slat(st, case, seed):
    s3dx = st["s3dx"]
    t = _slat_inputs(case, seed)
    cin, cout, join = case["cin"], case["cout"], case["join"]
    dt, tdt = _dt(s3dx, case)
    n = t["rows"].shape[0]
    st.update(dt=dt, n=n, **{k: t[k] for k in ("a", "n1w", "n1b", "ms", "mh")}, b=t.get("b"))
    st["rows"] = t["rows"]
    st["nc"] = nc = t["coarse"].shape[0]
    m = nc if join == "down" else n
    st["m"] = m
    if join == "down":
        cc, f2c = _empty((n, 4), torch.int32), _empty((n,), torch.int32)
        st["child"], st["inv"] = _empty((8 * n,), torch.int32), _empty((n,), torch.float32)
        torch.cuda.synchronize()
        s3dx.coarsen2(st["rows"].data_ptr(), n, out=(cc.data_ptr(), f2c.data_ptr(), st["child"].data_ptr(),
                                                    st["inv"].data_ptr()),
                      workspace=_ws(s3dx, s3dx.coarsen2_workspace_size(n)))
        s3dx.synchronize()
    st["f2c"] = t["f2c"].to(torch.int32).contiguous()
    st["kmap"] = _kmap(s3dx, t["coarse"] if join == "down" else t["rows"], m)
    st["x"] = _empty((m, cin), tdt) if join != "none" else st["a"]
    st["h"], st["y1"], st["sk"], st["y"] = (_empty((m, cin), tdt), _empty((m, cout), tdt), _empty((m, cout), tdt),
                                            _empty((m, cout), tdt))
    st["conv1"] = (s3dx.SparseConv(cin, cout, 27, dt)
                   .set_weights(_host(t["w1"]), s3dx.WEIGHT_SLAT, _host(t["b1"]))
                   .set_layernorm(True, 1e-6).set_silu(True)
                   .set_modulate(t["ms"].data_ptr(), t["mh"].data_ptr()))
    st["conv2"] = s3dx.SparseConv(cout, cout, 27, dt).set_weights(_host(t["w2"]), s3dx.WEIGHT_SLAT, _host(t["b2"]))
    st["skip"] = (s3dx.SparseConv(cin, cout, 1, dt).set_weights(_host(t["ws"]), s3dx.WEIGHT_SLAT, _host(t["bs"]))
                  if cin != cout else None)
    # one plan per map, kept with it
    st["plan"] = st["conv2"].gather_plan(m, st["kmap"].data_ptr(), m)


def _mesh_inputs(case, seed):
    rows = _voxels(case["n"], seed)
    for _ in range(case["level"]):
        rows = _children(rows)
    cin, cout = case["cin"], case["cout"]
    t = {"rows": rows, "x": _rows(seed, 1, (rows.shape[0], cin), case["dtype"])}
    t["g1"], t["h1"] = _normal(seed, 3, (cin,), 0.2, 1.0), _normal(seed, 4, (cin,), 0.2)
    t["g2"], t["h2"] = _normal(seed, 5, (cout,), 0.2, 1.0), _normal(seed, 6, (cout,), 0.2)
    t["w1"], t["b1"] = _weight(seed, 7, cin, cout, 27, True), _normal(seed, 8, (cout,), 0.1)
    t["w2"], t["b2"] = _weight(seed, 9, cout, cout, 27, True), _normal(seed, 10, (cout,), 0.1)
    t["ws"], t["bs"] = _weight(seed, 11, cin, cout, 1, True), _normal(seed, 12, (cout,), 0.1)
    if case["head"]:
        t["wh"], t["bh"] = _weight(seed, 13, cout, HEAD, 1), _normal(seed, 14, (HEAD,), 0.1)
    return t


def _prepare_mesh(st, case, seed):
    s3dx = st["s3dx"]
    t = _mesh_inputs(case, seed)
    cin, cout = case["cin"], case["cout"]
    dt, tdt = _dt(s3dx, case)
    p = t["rows"].shape[0]
    n = 8 * p
    st.update(dt=dt, p=p, n=n, x=t["x"], **{k: t[k] for k in ("g1", "h1", "g2", "h2")})
    child = _empty((n, 4), torch.int32)
    st["kmap"] = _empty((n, 27), torch.int32)
    torch.cuda.synchronize()
    s3dx.subdivide2(t["rows"].data_ptr(), p, True, out=(child.data_ptr(), st["kmap"].data_ptr()),
                    workspace=_ws(s3dx, s3dx.subdivide2_workspace_size(p)))
    s3dx.synchronize()
    st["y1"], st["ys"], st["y"] = _empty((n, cout), tdt), _empty((p, cout), tdt), _empty((n, cout), tdt)
    st["conv1"] = (s3dx.SparseConv(cin, cout, 27, dt).set_weights(_host(t["w1"]), s3dx.WEIGHT_MESH, _host(t["b1"]))
                   .set_gather_parent(True))
    # the 1x1 skip of the repeated rows, run once per parent
    st["skip"] = s3dx.SparseConv(cin, cout, 1, dt).set_weights(_host(t["ws"]), s3dx.WEIGHT_MESH, _host(t["bs"]))
    st["conv2"] = (s3dx.SparseConv(cout, cout, 27, dt).set_weights(_host(t["w2"]), s3dx.WEIGHT_MESH, _host(t["b2"]))
                   .set_residual_parent(True))
    torch.cuda.synchronize()
    st["gn1"] = s3dx.groupnorm_stats(st["x"].data_ptr(), dt, p, cin, GROUPS, 1e-5, st["g1"].data_ptr(),
                                     st["h1"].data_ptr())
    st["gn2"] = s3dx.groupnorm_stats(st["y1"].data_ptr(), dt, n, cout, GROUPS, 1e-5, st["g2"].data_ptr(),
                                     st["h2"].data_ptr())
    st["conv1"].set_input_affine_silu(st["gn1"][0], st["gn1"][1])
    st["conv2"].set_input_affine_silu(st["gn2"][0], st["gn2"][1])
    if case["head"]:
        st["head"] = s3dx.SparseConv(cout, HEAD, 1, s3dx.F32).set_weights(_host(t["wh"]), s3dx.WEIGHT_SLAT,
                                                                         _host(t["bh"]))
        if case["dtype"] == "bf16":
            st["head"].set_input_dtype(s3dx.BF16)
        st["out"] = _empty((n, HEAD), torch.float32)
    s3dx.synchronize()


# ---------------------------------------------------------------------------
# run
# ---------------------------------------------------------------------------
def run(st):
    return {"conv": _run_conv, "coords": _run_coords, "tables": _run_tables, "subdivide": _run_subdivide,
            "slat": _run_slat, "mesh": _run_mesh}[st["case"]["kind"]](st["s3dx"], st)


def _run_conv(s3dx, st):
    n = st["case"]["n"]
    st["conv"].run(st["x"].data_ptr(), n, st["kmap"].data_ptr(), n, st["y"].data_ptr(), plan=st["plan"])
    return st["y"]


def _run_coords(s3dx, st):
    r = st["case"]["res"]
    n, _ = s3dx.occupancy_coords(st["occ"].data_ptr(), (r, r, r), out=st["all"].data_ptr(), workspace=st["ws"][0])
    k, _ = s3dx.prune_surface(st["all"].data_ptr(), n, out=st["surface"].data_ptr(), workspace=st["ws"][1])
    m = k
    if k > 42000:
        m, _ = s3dx.downsample_coords(st["surface"].data_ptr(), k, 42000, 2, 42, out=st["down"].data_ptr(),
                                      workspace=st["ws"][2])
    return {"counts": [n, k, m], "all": st["all"], "surface": st["surface"], "down": st["down"]}


def _run_tables(s3dx, st):
    n = st["case"]["n"]
    s3dx.kmap_subm3_planned(st["rows"].data_ptr(), n, n, st["kmap"].data_ptr(), st["plan_f"], st["conv_f"],
                            workspace=st["ws"][0])
    nc, *_ = s3dx.coarsen2(st["rows"].data_ptr(), n, out=(st["coarse"].data_ptr(), st["f2c"].data_ptr(),
                                                          st["child"].data_ptr(), st["inv"].data_ptr()),
                           workspace=st["ws"][1])
    s3dx.kmap_subm3_planned(st["coarse"].data_ptr(), nc, nc, st["kmap_c"].data_ptr(), st["plan_c"], st["conv_c"],
                            workspace=st["ws"][0])
    return {"nc": nc, "kmap": st["kmap"], "coarse": st["coarse"], "f2c": st["f2c"], "child": st["child"],
            "inv": st["inv"], "kmap_c": st["kmap_c"]}


def _run_subdivide(s3dx, st):
    s3dx.subdivide2(st["rows"].data_ptr(), st["p"], True, out=(st["child"].data_ptr(), st["kmap"].data_ptr()),
                    workspace=st["ws"])
    return {"child": st["child"], "kmap": st["kmap"]}


def _run_slat(s3dx, st):
    c = st["case"]
    n, m, dt, cin = st["n"], st["m"], st["dt"], c["cin"]
    x = st["x"].data_ptr()
    if c["join"] == "down":
        s3dx.downsample_mean(st["a"].data_ptr(), dt, n, cin, st["child"].data_ptr(), st["inv"].data_ptr(), m, x)
    elif c["join"] == "up":
        s3dx.concat_rows(st["a"].data_ptr(), cin // 2, st["b"].data_ptr(), cin // 2, dt, st["nc"],
                         st["f2c"].data_ptr(), n, x)
    elif c["join"] == "cat":
        s3dx.concat_rows(st["a"].data_ptr(), cin // 2, st["b"].data_ptr(), cin // 2, dt, n, None, n, x)
    h, y1, y, kmap = st["h"].data_ptr(), st["y1"].data_ptr(), st["y"].data_ptr(), st["kmap"].data_ptr()
    s3dx.layernorm_rows(x, dt, m, cin, 1e-6, st["n1w"].data_ptr(), st["n1b"].data_ptr(), silu=True, y=h, y_dtype=dt)
    st["conv1"].run(h, m, kmap, m, y1, dt, plan=st["plan"])
    res = x
    if st["skip"] is not None:
        res = st["sk"].data_ptr()
        st["skip"].run(x, m, None, m, res, dt)
    st["conv2"].run(y1, m, kmap, m, y, dt, residual=res, plan=st["plan"])
    return st["y"]


def _run_mesh(s3dx, st):
    c = st["case"]
    p, n, dt = st["p"], st["n"], st["dt"]
    x, y1, ys, y, kmap = (st[k].data_ptr() for k in ("x", "y1", "ys", "y", "kmap"))
    s3dx.groupnorm_stats(x, dt, p, c["cin"], GROUPS, 1e-5, st["g1"].data_ptr(), st["h1"].data_ptr(), out=st["gn1"])
    st["conv1"].run(x, p, kmap, n, y1, dt)
    st["skip"].run(x, p, None, p, ys, dt)
    s3dx.groupnorm_stats(y1, dt, n, c["cout"], GROUPS, 1e-5, st["g2"].data_ptr(), st["h2"].data_ptr(),
                         out=st["gn2"])
    st["conv2"].run(y1, n, kmap, n, y, dt, residual=ys)
    if not c["head"]:
        return st["y"]
    st["head"].run(y, n, None, n, st["out"].data_ptr(), s3dx.F32)
    return {"rows": st["y"], "out": st["out"]}


# ---------------------------------------------------------------------------
# work and tolerance
# ---------------------------------------------------------------------------
def _pairs(rows):
    """Present (row, offset) pairs of a set, from its dense occupancy."""
    hi = int(rows.max()) + 3
    occ = torch.zeros((hi, hi, hi), dtype=torch.bool, device=rows.device)
    c = rows.long()
    occ[c[:, 1] + 1, c[:, 2] + 1, c[:, 3] + 1] = True
    total = 0
    for dx in (-1, 0, 1):
        for dy in (-1, 0, 1):
            for dz in (-1, 0, 1):
                total += int(occ[c[:, 1] + 1 + dx, c[:, 2] + 1 + dy, c[:, 3] + 1 + dz].sum())
    return total


def work(case):
    """Bytes: each input and output once, at one set's counts (they differ by a
    few per cent from set to set).  flops: a conv's 2 * cin * cout per present
    pair, as the layer is defined."""
    k = case["kind"]
    if k == "coords":
        cells = case["res"] ** 3
        return {"bytes": cells * 4 + cells * case["density"] * 16 * 2, "flops": 0}
    if k == "subdivide":
        p = case["n"] * 8 ** case["level"]
        return {"bytes": p * 16 + 8 * p * (16 + 108), "flops": 0}
    rows = _voxels_down(case["n"], 0) if case.get("join") == "down" else _voxels(case["n"], 0)
    n = rows.shape[0]
    if k == "tables":
        nc = _coarse(rows)[0].shape[0]
        return {"bytes": n * (16 + 108 + 4) + nc * (16 + 108 + 32 + 4), "flops": 0}
    cin, cout, es = case["cin"], case["cout"], 2 if case["dtype"] == "bf16" else 4
    if k == "conv":
        return {"bytes": n * ((cin + cout) * es + 108) + 27 * cin * cout * es, "flops": 2 * cin * cout * _pairs(rows)}
    if k == "slat":
        coarse = _coarse(rows)[0]
        nc = coarse.shape[0]
        m = nc if case["join"] == "down" else n
        src = nc * cin if case["join"] == "up" else n * cin
        pairs = _pairs(coarse if case["join"] == "down" else rows)
        skip = cin * cout if cin != cout else 0
        return {"bytes": (src + m * cout + 27 * cout * (cin + cout) + skip) * es + 108 * m,
                "flops": 2 * cout * (cin + cout) * pairs + 2 * skip * m}
    for _ in range(case["level"]):
        rows = _children(rows)
    p = rows.shape[0]
    pairs = _pairs(_children(rows))
    head = HEAD * cout if case["head"] else 0
    return {"bytes": (p * cin + 8 * p * cout + 27 * cout * (cin + cout) + cin * cout) * es + 8 * p * 108
            + (8 * p * HEAD * 4 if head else 0),
            "flops": 2 * cout * (cin + cout) * pairs + 2 * cin * cout * p + 2 * head * 8 * p}


def tolerance(case):
    if case["kind"] in ("coords", "tables", "subdivide"):
        return "exact"
    # four times what the path shows against exact()
    return {"rel": 1.5e-2} if case["dtype"] == "bf16" else {"rel": 4e-6}


# ---------------------------------------------------------------------------
# exact
# ---------------------------------------------------------------------------
_OFFSETS = [(dx, dy, dz) for dx in (-1, 0, 1) for dy in (-1, 0, 1) for dz in (-1, 0, 1)]


def _conv64(x, rows, w, bias, parent=False):
    """sum over the 27 offsets of w[:, o] x[neighbour], and the bias; w [cout, 27, cin]."""
    n = rows.shape[0]
    hi = int(rows.max()) + 3
    c = rows.long() + 1
    flat = (c[:, 1] * hi + c[:, 2]) * hi + c[:, 3]
    table = torch.full((hi ** 3,), -1, dtype=torch.int32, device=rows.device)
    table[flat] = torch.arange(n, dtype=torch.int32, device=rows.device)
    y = bias.double().expand(n, -1).clone()
    for o, (dx, dy, dz) in enumerate(_OFFSETS):
        j = table[flat + (dx * hi + dy) * hi + dz].long()
        at = (j >= 0).nonzero()[:, 0]
        src = j[at]
        wt = w[:, o].double().t().contiguous()
        for k in range(0, at.shape[0], 1 << 20):
            a, s = at[k:k + (1 << 20)], src[k:k + (1 << 20)]
            y[a] += x[s >> 3 if parent else s] @ wt
    return y


def _ln64(x, eps):
    return (x - x.mean(1, keepdim=True)) / (x.var(1, unbiased=False, keepdim=True) + eps).sqrt()


def _gn64(x, g, b):
    n, c = x.shape
    v = x.reshape(n, GROUPS, c // GROUPS)
    mean = v.mean((0, 2), keepdim=True)
    var = ((v - mean) ** 2).mean((0, 2), keepdim=True)
    return ((v - mean) / (var + 1e-5).sqrt()).reshape(n, c) * g.double() + b.double()


def _silu64(x):
    return x * torch.sigmoid(x)


def exact(case, seed):
    k = case["kind"]
    if k in ("coords", "tables", "subdivide"):
        return None
    if k == "conv":
        n, cin, cout = case["n"], case["cin"], case["cout"]
        return _conv64(_rows(seed, 1, (n, cin), case["dtype"]).double(), _voxels(n, seed),
                       _weight(seed, 2, cin, cout, 27), _normal(seed, 3, (cout,), 0.1))
    if k == "slat":
        t = _slat_inputs(case, seed)
        rows, x = t["rows"], t["a"].double()
        if case["join"] == "down":  # the mean-pool divides by count + 1
            rows, nc = t["coarse"], t["coarse"].shape[0]
            s = torch.zeros((nc, case["cin"]), dtype=torch.float64, device=x.device).index_add_(0, t["f2c"], x)
            x = s / (torch.bincount(t["f2c"], minlength=nc) + 1).double()[:, None]
        elif case["join"] == "up":
            x = torch.cat([x, t["b"].double()], 1)[t["f2c"]]
        elif case["join"] == "cat":
            x = torch.cat([x, t["b"].double()], 1)
        h = _silu64(_ln64(x, 1e-6) * t["n1w"].double() + t["n1b"].double())
        h = _ln64(_conv64(h, rows, t["w1"], t["b1"]), 1e-6)
        h = _silu64(h * (1.0 + t["ms"].double()) + t["mh"].double())
        res = x @ t["ws"][:, 0].double().t().contiguous() + t["bs"].double() if "ws" in t else x
        return _conv64(h, rows, t["w2"], t["b2"]) + res
    t = _mesh_inputs(case, seed)
    child, x = _children(t["rows"]), t["x"].double()
    h = _silu64(_gn64(x, t["g1"], t["h1"]))
    y1 = _conv64(h, child, t["w1"].transpose(0, 1), t["b1"], parent=True)
    y1 = _silu64(_gn64(y1, t["g2"], t["h2"]))
    y = _conv64(y1, child, t["w2"].transpose(0, 1), t["b2"])
    sk = x @ t["ws"][0].double().t().contiguous() + t["bs"].double()
    y += sk.repeat_interleave(8, 0)
    if not case["head"]:
        return y
    return {"rows": y, "out": y @ t["wh"][:, 0].double().t().contiguous() + t["bh"].double()}
