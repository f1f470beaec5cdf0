"""The work whose speed is followed: listed cases, and drawn ones of the same ranges.

  train    one full training step of a hash-grid model (sampler, encoder, network, line integral and loss, their
           backward, Adam) through nect_amd.fused.FusedTrainStep, as nect_amd.trainer drives it
  module   the same step of a QuadCubes model through nect_amd.module_step.ModuleTrainStep
  points   forward and backward of tcnn.NetworkWithInputEncoding on points a caller made itself
  network  forward and backward of tcnn.Network, 128 neurons wide (the dynamic presets' network)
  query    voxels of a trained model through nect_amd.serving.QueryServer
  sample   the reference's own sampling interface, nect_amd.sampling.ct_sampling.sample

The acquisition is a cone beam (source to detector 800 mm, to the origin 400 mm) around a cube of 128 mm, its detector
256 mm wide whatever its pixel count; rays are a random choice of one view's pixels.
"""
import math

import numpy as np
import torch

from nect_amd import tcnn
from nect_amd.fused import FusedTrainStep, xavier_init
from nect_amd.grid import GridDesc
from nect_amd.mlp import MlpDesc
from nect_amd.module_step import ModuleTrainStep
from nect_amd.networks import QuadCubes
from nect_amd.sampling import ct_sampling
from nect_amd.sampling.geometry import Geometry
from nect_amd.serving import QueryRequest, QueryServer

DEVICE = "cuda"
DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}
DSD, DSO, CUBE_MM, DETECTOR_MM = 800.0, 400.0, 128.0, 256.0
KEPT = 0.65          # share of a ray's sample slots that lie in the cube (full views of this geometry)
TABLE = 0.1          # magnitude of the hash-table entries of a model in the middle of its training
ADAM_STEPS, ADAM_V, LR = 1000, 1e-6, 1e-4


def _train(name, det, rays, points, dims, levels, features, log2_t, base, growth, layers, act, out_act, loss, dtype):
    return {"name": name, "kind": "train", "detector": det, "rays": rays, "points": points, "dims": dims,
            "levels": levels, "features": features, "log2_table": log2_t, "base": base, "growth": growth,
            "layers": layers, "activation": act, "output": out_act, "loss": loss, "dtype": dtype}


STATIC_GROWTH = (2 * 256 / 8) ** (1 / 18)
QUAD_GROWTH = (2 * 256 / 16) ** (1 / 22)


def listed():
    return [
        # a quick look at a small scan: 64^2 detector, 1024 rays a step; launches and host work count
        _train("train_cone64", 64, 1024, 64, 3, 16, 2, 19, 16, 1.5, 2, "ReLU", "Softplus", "L2", "fp16"),
        # the headline: 256^3 cone beam, one whole view of 2^16 rays a step
        _train("train_cone256", 256, 65536, 256, 3, 16, 2, 19, 16, 1.5, 2, "ReLU", "Softplus", "L2", "fp16"),
        # a dynamic scan with one 4-D grid, 512^2 detector, half a view's pixels a step
        _train("train_4d", 512, 131072, 128, 4, 16, 2, 21, 16, 1.5, 3, "ReLU", "Softplus", "L2", "bf16"),
        # the reference's default static model at the batch its presets arrive at
        _train("train_static_preset", 256, 6510, 384, 3, 19, 4, 21, 8, STATIC_GROWTH, 6, "LeakyReLU", "ReLU", "L1",
               "fp16"),
        # full precision, a part of a view and a sample count that is no multiple of 32
        _train("train_fp32", 256, 16383, 200, 3, 16, 2, 19, 16, 1.5, 2, "ReLU", "Softplus", "L2", "fp32"),
        # the default dynamic model's structure at its presets' batch (tables of 2^19 entries)
        {"name": "module_quadcubes", "kind": "module", "detector": 512, "rays": 9765, "points": 256, "levels": 23,
         "features": 4, "log2_table": 19, "base": 16, "growth": QUAD_GROWTH, "layers": 4, "dtype": "fp16"},
        # a user's own loop over the encoded network: a million points, and a few thousand
        {"name": "points_1m", "kind": "points", "n": 1000003, "dims": 3, "levels": 16, "features": 2,
         "log2_table": 19, "base": 16, "growth": 1.5, "layers": 2, "dtype": "fp16"},
        {"name": "points_4k", "kind": "points", "n": 4099, "dims": 3, "levels": 16, "features": 2,
         "log2_table": 19, "base": 16, "growth": 1.5, "layers": 2, "dtype": "fp16"},
        # the dynamic presets' network by itself
        {"name": "network_wide", "kind": "network", "n": 262147, "inputs": 372, "layers": 4, "dtype": "fp16"},
        # an exported volume and one slice of a 4-D model
        {"name": "query_volume", "kind": "query", "nz": 512, "ny": 512, "nx": 512, "dims": 4, "log2_table": 21,
         "layers": 3, "dtype": "bf16"},
        {"name": "query_slice", "kind": "query", "nz": 1, "ny": 512, "nx": 512, "dims": 4, "log2_table": 21,
         "layers": 3, "dtype": "bf16"},
        # the reference's sampling call for one view
        {"name": "sample_view", "kind": "sample", "detector": 256, "rays": 65536, "points": 256},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    case = _draw(rng)
    case.pop("name", None)
    return case


def _draw(rng):
    kind = rng.choice(["train", "train", "train", "train", "module", "points", "points", "network", "query", "query",
                       "sample"])
    if kind == "train":
        det = rng.choice([64, 100, 128, 200, 256, 384, 512])
        points = rng.randrange(40, 257)
        style = rng.choice(["3d", "3d", "4d", "static", "fp32"])
        rays = _log_int(rng, 512, min(det * det, 65536))
        if style == "3d":
            return _train(None, det, rays, points, 3, 16, 2, rng.choice([17, 18, 19, 20]), 16, 1.5, rng.choice([1, 2, 3]),
                          "ReLU", "Softplus", rng.choice(["L1", "L2"]), rng.choice(["fp16", "fp16", "bf16"]))
        if style == "4d":
            return _train(None, det, rays, min(points, 128), 4, 16, 2, rng.choice([19, 20, 21]), 16, 1.5,
                          rng.choice([2, 3]), "ReLU", "Softplus", "L2", rng.choice(["fp16", "bf16"]))
        if style == "static":
            return _train(None, det, min(rays, 8192), points, 3, 19, 4, rng.choice([18, 20, 21]), 8, STATIC_GROWTH,
                          rng.choice([3, 6]), "LeakyReLU", "ReLU", "L1", "fp16")
        return _train(None, det, min(rays, 20000), points, 3, 16, 2, rng.choice([17, 19]), 16, 1.5, 2, "ReLU",
                      "Softplus", "L2", "fp32")
    if kind == "module":
        return {"kind": "module", "detector": rng.choice([128, 256, 512]), "rays": _log_int(rng, 512, 10000),
                "points": rng.randrange(64, 257), "levels": 23, "features": 4, "log2_table": rng.choice([17, 18, 19]),
                "base": 16, "growth": QUAD_GROWTH, "layers": rng.choice([2, 4]), "dtype": rng.choice(["fp16", "bf16"])}
    if kind == "points":
        dims = rng.choice([3, 3, 4])
        return {"kind": "points", "n": _log_int(rng, 2000, 2000000), "dims": dims, "levels": 16,
                "features": rng.choice([2, 2, 4]), "log2_table": rng.choice([17, 19]), "base": 16, "growth": 1.5,
                "layers": rng.choice([1, 2, 3]), "dtype": rng.choice(["fp16", "bf16", "fp32"]) if dims == 3 else "fp16"}
    if kind == "network":
        return {"kind": "network", "n": _log_int(rng, 2000, 500000), "inputs": rng.choice([96, 372]),
                "layers": rng.choice([2, 4]), "dtype": rng.choice(["fp16", "bf16"])}
    if kind == "query":
        size = _log_int(rng, 48, 400)
        nz, ny, nx = (max(1, int(size * rng.uniform(0.7, 1.2))) for _ in range(3))
        if rng.random() < 0.5:
            nz = 1
            ny, nx = ny * 2, nx * 2
        return {"kind": "query", "nz": nz, "ny": ny, "nx": nx, "dims": rng.choice([3, 4]),
                "log2_table": rng.choice([19, 21]), "layers": rng.choice([2, 3]), "dtype": rng.choice(["fp16", "bf16"])}
    return {"kind": "sample", "detector": 256, "rays": _log_int(rng, 1000, 65536), "points": rng.randrange(40, 300)}


# ------------------------------------------------------------------- inputs


def _gen(seed):
    return torch.Generator(device=DEVICE).manual_seed(int(seed))


def _geometry(case):
    det = case["detector"]
    pitch = DETECTOR_MM / det
    return Geometry(nDetector=(det, det), dDetector=(pitch, pitch), mode="cone", DSD=DSD, DSO=DSO,
                    nVoxel=(256, 256, 256), dVoxel=(CUBE_MM / 256,) * 3, angles=[0.0])


def _batch(case, seed):
    """One step's rays: view angle and time, pixels, jitters, offsets and measured values (a smooth object with the
    noise of the photon count)."""
    g = _gen(seed)
    det, rays = case["detector"], case["rays"]
    angle = 2 * math.pi * ((seed * 0.6180339887) % 1.0)
    index = torch.randperm(det * det, device=DEVICE, generator=g)[:rays]
    jitter = torch.rand(index.numel(), device=DEVICE, generator=g) - 0.5
    offset = torch.zeros((index.numel(), 2), device=DEVICE)
    r2 = ((index % det).float() / det - 0.5) ** 2 + ((index // det).float() / det - 0.5) ** 2
    target = (0.9 * torch.exp(-6 * r2) + 0.05 * torch.randn(index.numel(), device=DEVICE, generator=g)).contiguous()
    return {"angle": angle, "t": (seed * 0.7548776662) % 1.0, "index": index, "jitter": jitter, "offset": offset,
            "target": target, "rays": int(index.numel())}


def _params(desc, n_table, seed):
    """[network | tables] float32 of a model in the middle of its training."""
    w = xavier_init(desc, torch.Generator().manual_seed(int(seed))).to(DEVICE)
    table = (torch.rand(n_table, device=DEVICE, generator=_gen(seed + 1)) * 2 - 1) * TABLE
    return torch.cat([w, table])


def _encoding(case):
    return {"otype": "HashGrid", "n_levels": case["levels"], "n_features_per_level": case["features"],
            "log2_hashmap_size": case["log2_table"], "base_resolution": case["base"],
            "per_level_scale": case["growth"]}


def _wide(case):
    return {"otype": "FullyFusedMLP", "activation": "LeakyReLU", "output_activation": "None", "n_neurons": 128,
            "n_hidden_layers": case["layers"]}


def prepare(case, seed):
    kind = case["kind"]
    state = {"kind": kind}
    if kind in ("train", "module", "sample"):
        geometry = _geometry(case)
        state["batch"] = _batch(case, seed)
        state["geometry"] = geometry.get_c_geometry()
        state["points"] = case["points"]
        state["l_max"] = geometry.max_distance_traveled
        state["step_mm"] = geometry.max_distance_traveled / case["points"]
    if kind == "train":
        grid = GridDesc(case["dims"], case["levels"], case["features"], case["log2_table"], case["base"], case["growth"])
        mlp = MlpDesc(grid.n_output_dims, 1, 64, case["layers"], case["activation"], case["output"])
        step = FusedTrainStep(grid, mlp, _params(mlp, grid.n_params, seed), DTYPES[case["dtype"]],
                              max_rays=state["batch"]["rays"], max_points_per_ray=case["points"], loss=case["loss"])
        step.v.fill_(ADAM_V)
        step.set_adam_steps(ADAM_STEPS)
        state["step"] = step
    elif kind == "module":
        model = QuadCubes(_encoding(case), _wide(case), include_identity=True, dtype=DTYPES[case["dtype"]]).to(DEVICE)
        net = model.net
        net.params.data.copy_(_params(net.desc, net.n_enc_params, seed))
        step = ModuleTrainStep(model, DTYPES[case["dtype"]], state["batch"]["rays"], case["points"], loss="L1",
                               dynamic=True)
        step.v.fill_(ADAM_V)
        step.set_adam_steps(ADAM_STEPS)
        state["step"] = step
    elif kind == "points":
        net = tcnn.NetworkWithInputEncoding(
            case["dims"], 1, _encoding(case),
            {"otype": "FullyFusedMLP", "activation": "ReLU", "output_activation": "None", "n_neurons": 64,
             "n_hidden_layers": case["layers"]}, dtype=DTYPES[case["dtype"]]).to(DEVICE)
        net.params.data.copy_(_params(net.desc, net.n_enc_params, seed))
        g = _gen(seed + 2)
        state["net"] = net
        state["x"] = torch.rand((case["n"], case["dims"]), device=DEVICE, generator=g)
        state["dy"] = torch.randn((case["n"], 1), device=DEVICE, generator=g) / case["n"]
    elif kind == "network":
        net = tcnn.Network(case["inputs"], 1, _wide(case), dtype=DTYPES[case["dtype"]]).to(DEVICE)
        net.params.data.copy_(_params(net.desc, 0, seed))
        g = _gen(seed + 2)
        state["net"] = net
        state["x"] = (torch.rand((case["n"], case["inputs"]), device=DEVICE, generator=g) * 2 - 1).requires_grad_(True)
        state["dy"] = torch.randn((case["n"], 1), device=DEVICE, generator=g) / case["n"]
    elif kind == "query":
        grid = GridDesc(case["dims"], 16, 2, case["log2_table"], 16, 1.5)
        mlp = MlpDesc(32, 1, 64, case["layers"], "ReLU", "Softplus")
        p = _params(mlp, grid.n_params, seed).to(DTYPES[case["dtype"]])
        state["server"] = QueryServer(grid, mlp, p[: mlp.n_params].clone(), p[mlp.n_params:].clone())
        state["grid"] = _query_grid(case, seed)
    return state


def _query_grid(case, seed):
    """(voxels, first and last coordinate per axis, time): the whole cube, or a slice of it."""
    n = (case["nz"], case["ny"], case["nx"])
    z = (seed * 0.6180339887) % 1.0
    a = (z if n[0] == 1 else 0.0, 0.0, 0.0)
    b = (z if n[0] == 1 else 1.0, 1.0, 1.0)
    return n, a, b, (seed * 0.7548776662) % 1.0


# ---------------------------------------------------------------- one pass


def run(state):
    kind = state["kind"]
    if kind in ("train", "module"):
        s, b = state["step"], state["batch"]
        loss = s.step(state["geometry"], b["angle"], b["index"], 0, b["rays"], state["points"], state["step_mm"], True,
                      b["jitter"], b["offset"], b["target"], state["l_max"], lr=LR, t=b["t"])
        return {"loss": loss, "y": s.y_pred[: b["rays"]], "params": s.params, "m": s.m, "v": s.v}
    if kind == "points":
        net = state["net"]
        net.params.grad = None
        y = net(state["x"])
        y.backward(state["dy"])
        return {"y": y, "grad": net.params.grad}
    if kind == "network":
        net, x = state["net"], state["x"]
        net.params.grad = None
        x.grad = None
        y = net(x)
        y.backward(state["dy"])
        return {"y": y, "grad": net.params.grad, "dx": x.grad}
    if kind == "query":
        n, a, b, t = state["grid"]
        return state["server"].run_alone(QueryRequest(n, a, b, t))
    b = state["batch"]
    return ct_sampling.sample(b["index"], state["geometry"], b["angle"], state["points"], b["rays"], 0,
                              state["step_mm"], True, 0.0, DEVICE, jitter=b["jitter"], detector_offset=b["offset"],
                              return_counts=True)


# ------------------------------------------------- what a pass cannot do without


def _levels(dims, levels, features, log2_t, base, growth):
    """(scale, resolution, entries) per level, by tiny-cuda-nn's rules."""
    growth = float(np.float32(growth))
    out = []
    for l in range(levels):
        scale = np.float32(base * growth ** l - 1.0)
        res = int(math.ceil(float(scale))) + 1
        size = min((res ** dims + 7) // 8 * 8, 1 << log2_t)
        out.append((float(scale), res, size))
    return out


def _layer_flops(inputs, width, layers):
    return 2 * (inputs * width + (layers - 1) * width * width + width)


def work(case):
    kind = case["kind"]
    esz = 4 if case.get("dtype") == "fp32" else 2
    if kind in ("train", "module"):
        grids = 4 if kind == "module" else 1
        dims = case.get("dims", 3)
        lv = _levels(dims, case["levels"], case["features"], case["log2_table"], case["base"], case["growth"])
        n_params = grids * case["features"] * sum(s for _, _, s in lv)
        enc = grids * case["levels"] * case["features"]
        samples = KEPT * min(case["rays"], case["detector"] ** 2) * case["points"]
        net = _layer_flops(enc, 64 if kind == "train" else 128, case["layers"])
        # parameters in the compute dtype read, Adam's three float32 vectors read and written, the dtype's copy written
        return {"bytes": n_params * (2 * esz + 24 if esz == 2 else 24) + case["rays"] * 36,
                "flops": samples * (3 * net + 2 * 2 * enc * 2 ** dims)}
    if kind == "points":
        lv = _levels(case["dims"], case["levels"], case["features"], case["log2_table"], case["base"], case["growth"])
        n_params = case["features"] * sum(s for _, _, s in lv)
        enc = case["levels"] * case["features"]
        return {"bytes": n_params * 8 + case["n"] * (4 * case["dims"] + 8),
                "flops": case["n"] * (3 * _layer_flops(enc, 64, case["layers"]) + 4 * enc * 2 ** case["dims"])}
    if kind == "network":
        return {"bytes": case["n"] * (8 * case["inputs"] + 8),
                "flops": case["n"] * 3 * _layer_flops(case["inputs"], 128, case["layers"])}
    voxels_or_slots = case["rays"] * case["points"] if kind == "sample" else case["nz"] * case["ny"] * case["nx"]
    if kind == "sample":
        return {"bytes": voxels_or_slots * 12 + case["rays"] * 28, "flops": voxels_or_slots * 6}
    lv = _levels(case["dims"], 16, 2, case["log2_table"], 16, 1.5)
    return {"bytes": voxels_or_slots * 2 + 4 * sum(s for _, _, s in lv),
            "flops": voxels_or_slots * (_layer_flops(32, 64, case["layers"]) + 2 * 32 * 2 ** case["dims"])}


# --------------------------------------------------------- the same in 64 bits


PRIMES = (1, 2654435761, 805459861, 3674653429)
CHUNK = 1 << 18


def _corners(level, x):
    """Per corner of x's cell on a level: (entry, weight), x [n, dims] float64."""
    scale, res, size = level
    dims = x.shape[1]
    p = x * scale + 0.5
    c = p.floor()
    f = p - c
    c = c.long()
    dense = res ** dims <= size
    for k in range(1 << dims):
        w = torch.ones_like(f[:, 0])
        idx = torch.zeros_like(c[:, 0])
        for d in range(dims):
            bit = (k >> d) & 1
            w = w * (f[:, d] if bit else 1 - f[:, d])
            cc = c[:, d] + bit
            idx = idx + cc * res ** d if dense else idx ^ ((cc * PRIMES[d]) & 0xFFFFFFFF)
        yield idx % size, w


def _encode64(levels, tables, x):
    """Features of x; tables: one [entries, F] float64 tensor per level."""
    out = []
    for lv, tab in zip(levels, tables):
        acc = 0
        for idx, w in _corners(lv, x):
            acc = acc + w[:, None] * tab[idx]
        out.append(acc)
    return torch.cat(out, dim=1)


def _scatter64(levels, grads, x, dfeat):
    col = 0
    for lv, g in zip(levels, grads):
        F = g.shape[1]
        d = dfeat[:, col:col + F]
        for idx, w in _corners(lv, x):
            g.index_add_(0, idx, w[:, None] * d)
        col += F


def _split_tables(levels, flat, features):
    out, o = [], 0
    for _, _, size in levels:
        out.append(flat[o:o + size * features].view(size, features))
        o += size * features
    return out


def _act64(name, z):
    return {"None": lambda v: v, "ReLU": torch.relu, "Softplus": torch.nn.functional.softplus,
            "LeakyReLU": lambda v: torch.nn.functional.leaky_relu(v, 0.01)}[name](z)


def _net64(weights, h, act, out_act):
    for w in weights[:-1]:
        h = _act64(act, h @ w[:, : h.shape[1]].t())
    return _act64(out_act, h @ weights[-1][:1].t())


def _net_shapes(inputs, width, layers):
    return [(width, (inputs + 15) // 16 * 16)] + [(width, width)] * (layers - 1) + [(16, width)]


def _split_net(flat, inputs, width, layers):
    out, o = [], 0
    for r, c in _net_shapes(inputs, width, layers):
        out.append(flat[o:o + r * c].view(r, c).detach().requires_grad_(True))
        o += r * c
    return out, o


class _Rays64:
    """The cone-beam rays of a batch: double entry and exit points of the cube, float32 samples, as the reference's
    sampler places them."""

    def __init__(self, case, batch, points, step_mm):
        det = case["detector"]
        f32 = lambda v: float(np.float32(v))  # noqa: E731
        pitch = np.float32(DETECTOR_MM / det)
        angle = f32(batch["angle"])
        c, s = f32(math.cos(angle)), f32(math.sin(angle))
        step = f32(step_mm)
        half = np.float32(det - 1) / np.float32(2)
        col = (batch["index"] % det).float()
        row = (batch["index"] // det).float()
        off = batch["offset"]
        u = ((col - float(half)) + off[:, 0]) * float(pitch)
        v = ((row - float(half)) + off[:, 1]) * float(pitch)
        zero = torch.zeros_like(u, dtype=torch.float64)
        d = [zero + (DSD - DSO), -u.double(), v.double()]
        src = [zero - DSO, zero, zero]
        rot = lambda p: [c * p[0] - s * p[1], s * p[0] + c * p[1], p[2]]  # noqa: E731
        a, b = rot(src), rot(d)
        h = float((np.float32(CUBE_MM) - np.float32(CUBE_MM / 256) / np.float32(2)) / np.float32(2))
        lo, hi = [], []
        for k in range(3):
            diff = b[k] - a[k]
            t0, t1 = (-h - a[k]) / diff, (h - a[k]) / diff
            lo.append(torch.minimum(t0, t1).nan_to_num(nan=-math.inf))
            hi.append(torch.maximum(t0, t1).nan_to_num(nan=math.inf))
        t0 = torch.maximum(torch.maximum(lo[0], lo[1]), lo[2])
        t1 = torch.minimum(torch.minimum(hi[0], hi[1]), hi[2])
        self.hit = (t0 <= t1) & (t0 >= 0) & (t0 <= 1) & (t1 >= 0) & (t1 <= 1)
        st = [a[k] + t0 * (b[k] - a[k]) for k in range(3)]
        en = [a[k] + t1 * (b[k] - a[k]) for k in range(3)]
        sp = [en[k] - st[k] for k in range(3)]
        length = torch.sqrt(sp[0] * sp[0] + sp[1] * sp[1] + sp[2] * sp[2]).float().double()
        self.distance = torch.where(self.hit, zero + step, zero)
        sp = [(q / length) * step / CUBE_MM for q in sp]
        j = batch["jitter"].double()
        self.start = [((st[k] / CUBE_MM + 0.5) + j * sp[k]).clamp(0, 1) for k in range(3)]
        self.end = [((en[k] / CUBE_MM + 0.5) + sp[k]).clamp(0, 1) for k in range(3)]
        self.step = sp
        self.points = points

    def samples(self, r0, r1):
        """(float32 positions [r, points, 3] in (z, y, x), which of them are kept) of rays r0..r1."""
        i = torch.arange(self.points, device=DEVICE, dtype=torch.float64)
        stop = ~self.hit[r0:r1, None].expand(-1, self.points)
        pos = []
        for k in range(3):
            sp, en = self.step[k][r0:r1, None], self.end[k][r0:r1, None]
            p = (self.start[k][r0:r1, None] + i * sp).float()
            stop = stop | ((sp > 0) & ((p - 1e-5).double() > en)) | ((sp < 0) & ((p + 1e-5).double() < en))
            pos.append(p.clamp(0, 1))
        kept = stop.long().cumsum(1) == 0
        return torch.stack(pos[::-1], dim=-1), kept


def _step64(case, state, params, parts, net_args):
    """Line integrals, loss and parameter gradient of a training step; parts: (levels, features, first parameter,
    columns of (z, y, x, t)) per grid, then the identity columns."""
    batch, points = state["batch"], state["points"]
    rays = _Rays64(case, batch, points, state["step_mm"])
    weights, n_net = _split_net(params, net_args["inputs"], net_args["width"], net_args["layers"])
    tables = [_split_tables(lv, params[n_net + p0:], F) for lv, F, p0, _ in parts["grids"]]
    grad = torch.zeros_like(params)
    gtables = [_split_tables(lv, grad[n_net + p0:], F) for lv, F, p0, _ in parts["grids"]]
    dl = rays.distance / float(np.float32(state["l_max"]))
    t = float(np.float32(batch["t"]))
    n = batch["rays"]
    per = max(1, CHUNK // points)

    def inputs(r0):
        pos, kept = rays.samples(r0, min(n, r0 + per))
        kept = kept & ~(pos == 0).all(-1)
        x = pos[kept].double()
        return torch.cat([x, torch.full_like(x[:, :1], t)], dim=1), kept

    def features(x):
        f = [_encode64(lv, tab, x[:, cols]) for (lv, _, _, cols), tab in zip(parts["grids"], tables)]
        return torch.cat(f + ([x] if parts["identity"] else []), dim=1)

    y = torch.zeros(n, dtype=torch.float64, device=DEVICE)
    with torch.no_grad():
        for r0 in range(0, n, per):
            x, kept = inputs(r0)
            mu = torch.zeros(kept.shape, dtype=torch.float64, device=DEVICE)
            mu[kept] = _net64(weights, features(x), net_args["act"], net_args["out"])[:, 0]
            y[r0:r0 + per] = mu.sum(1)
    y = y * dl
    diff = y - batch["target"].double()
    loss = (diff * diff).mean() if net_args["loss"] == "L2" else diff.abs().mean()
    gy = (2 * diff if net_args["loss"] == "L2" else torch.sign(diff)) / n
    for r0 in range(0, n, per):
        x, kept = inputs(r0)
        feats = features(x).requires_grad_(True)
        mu = _net64(weights, feats, net_args["act"], net_args["out"])[:, 0]
        mu.backward((gy * dl)[r0:r0 + per, None].expand(kept.shape)[kept])
        col = 0
        for (lv, F, _, cols), g in zip(parts["grids"], gtables):
            _scatter64(lv, g, x[:, cols], feats.grad[:, col:col + F * len(lv)])
            col += F * len(lv)
    grad[:n_net] = torch.cat([w.grad.flatten() for w in weights])
    beta1, beta2, step = 0.9, 0.999, ADAM_STEPS + 1
    m = (1 - beta1) * grad
    v = beta2 * float(np.float32(ADAM_V)) + (1 - beta2) * grad * grad
    size = LR / (1 - beta1 ** step)
    new = params - size * m / (torch.sqrt(v / (1 - beta2 ** step)) + 1e-8)
    return {"loss": loss.reshape(1), "y": y, "params": new, "m": m, "v": v}


def exact(case, seed):
    kind = case["kind"]
    if kind in ("train", "module"):
        state = prepare(case, seed)
        params = state["step"].params.detach().double()
        lv = _levels(case.get("dims", 3), case["levels"], case["features"], case["log2_table"], case["base"],
                     case["growth"])
        n_table = case["features"] * sum(s for _, _, s in lv)
        if kind == "train":
            parts = {"grids": [(lv, case["features"], 0, list(range(case["dims"])))], "identity": False}
            net = {"inputs": case["levels"] * case["features"], "width": 64, "layers": case["layers"],
                   "act": case["activation"], "out": case["output"], "loss": case["loss"]}
        else:
            cols = ([0, 1, 2], [1, 2, 3], [2, 0, 3], [0, 1, 3])
            parts = {"grids": [(lv, case["features"], k * n_table, c) for k, c in enumerate(cols)], "identity": True}
            net = {"inputs": 4 * case["levels"] * case["features"] + 4, "width": 128, "layers": case["layers"],
                   "act": "LeakyReLU", "out": "None", "loss": "L1"}
        batch = {"batch": state["batch"], "points": state["points"], "step_mm": state["step_mm"],
                 "l_max": state["l_max"]}
        del state
        return _step64(case, batch, params, parts, net)
    if kind == "sample":
        state = prepare(case, seed)
        rays = _Rays64(case, state["batch"], state["points"], state["step_mm"])
        pos, kept = rays.samples(0, state["batch"]["rays"])
        return pos.double() * kept[..., None], rays.distance, None
    if kind == "points":
        state = prepare(case, seed)
        params = state["net"].params.detach().double()
        lv = _levels(case["dims"], case["levels"], case["features"], case["log2_table"], case["base"], case["growth"])
        weights, n_net = _split_net(params, case["levels"] * case["features"], 64, case["layers"])
        tables = _split_tables(lv, params[n_net:], case["features"])
        grad = torch.zeros_like(params)
        gtables = _split_tables(lv, grad[n_net:], case["features"])
        ys = []
        for r0 in range(0, case["n"], CHUNK):
            x = state["x"][r0:r0 + CHUNK].double()
            feats = _encode64(lv, tables, x).requires_grad_(True)
            y = _net64(weights, feats, "ReLU", "None")
            y.backward(state["dy"][r0:r0 + CHUNK].double())
            _scatter64(lv, gtables, x, feats.grad)
            ys.append(y.detach())
        grad[:n_net] = torch.cat([w.grad.flatten() for w in weights])
        return {"y": torch.cat(ys), "grad": grad}
    if kind == "network":
        state = prepare(case, seed)
        weights, _ = _split_net(state["net"].params.detach().double(), case["inputs"], 128, case["layers"])
        x = state["x"].detach().double().requires_grad_(True)
        y = _net64(weights, x, "LeakyReLU", "None")
        y.backward(state["dy"].double())
        return {"y": y.detach(), "grad": torch.cat([w.grad.flatten() for w in weights]), "dx": x.grad}
    state = prepare(case, seed)
    n, a, b, t = state["grid"]
    lv = _levels(case["dims"], 16, 2, case["log2_table"], 16, 1.5)
    weights, _ = _split_net(state["server"].weights.double(), 32, 64, case["layers"])
    tables = _split_tables(lv, state["server"].table.double(), 2)
    axes = [torch.linspace(a[k], b[k], n[k], device=DEVICE, dtype=torch.float32).double() for k in range(3)]
    out = torch.empty(n[0] * n[1] * n[2], dtype=torch.float64, device=DEVICE)
    per = 8 * CHUNK
    with torch.no_grad():
        for v0 in range(0, out.numel(), per):
            v = torch.arange(v0, min(out.numel(), v0 + per), device=DEVICE)
            x = [axes[0][v // (n[1] * n[2])], axes[1][v // n[2] % n[1]], axes[2][v % n[2]]]
            x = torch.stack(x + [torch.full_like(x[0], float(np.float32(t)))] * (case["dims"] - 3), dim=1)
            out[v0:v0 + per] = _net64(weights, _encode64(lv, tables, x), "ReLU", "Softplus")[:, 0]
    return out.view(n)
