"""The memory of the table gradient's records: where the device has not enough left for them, every training path works
with less or none, as it does with plenty; a fused step's memory budget holds for them, too; a module step's can be set.

The gradients are the same sums in another order: 1e-4 of the largest (as for batches in chunks)."""
import contextlib
import gc

import pytest
import torch

from tests.helpers import cfg1_geometry, product_struct, seeded_batch

pytestmark = pytest.mark.gpu

MIB = 1 << 20


def held(device):
    gc.collect()
    torch.cuda.synchronize(device)
    torch.cuda.empty_cache()
    return torch.cuda.memory_reserved(device)


@contextlib.contextmanager
def room(device, nbytes):
    """torch's allocator has nbytes more than what is held now."""
    total = torch.cuda.get_device_properties(device).total_memory
    torch.cuda.set_per_process_memory_fraction((held(device) + nbytes) / total, device)
    try:
        yield
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0, device)


def peak(device, f):
    """(f(), bytes it took at most beyond what was held)"""
    before = held(device)
    torch.cuda.reset_peak_memory_stats(device)
    out = f()
    torch.cuda.synchronize(device)
    return out, torch.cuda.max_memory_reserved(device) - before


def same(got, ref):
    assert got.shape == ref.shape and bool(ref.any())
    err = float((got - ref).abs().max() / ref.abs().max())
    assert err <= 1e-4, err


def batch(device, B):
    geo = cfg1_geometry()
    idx, jit, off = (torch.from_numpy(a).to(device) for a in seeded_batch(64 * 64, B, seed=3))
    return geo.max_distance_traveled, product_struct(geo.c_struct_fields()), idx, jit, off, torch.rand(
        B, device=device, generator=torch.Generator(device=device).manual_seed(1))


def fused(device, B, S, batch_, **kw):
    from nect_amd.fused import FusedTrainStep, init_params
    from nect_amd.grid import GridDesc
    from nect_amd.mlp import MlpDesc

    grid = GridDesc(3, 16, 2, 15, 16, 1.5)
    mlp = MlpDesc(32, 1, 64, 2, "ReLU", "Softplus")
    params = init_params(grid, mlp, seed=0, device=device)
    params[mlp.n_params:] = ((torch.rand(grid.n_params, generator=torch.Generator().manual_seed(1)) * 2 - 1) * 0.5).to(device)
    fs = FusedTrainStep(grid, mlp, params, torch.float16, max_rays=B, max_points_per_ray=S, **kw)
    l_max, geo, idx, jit, off, tgt = batch_
    fs.step(geo, 0.4, idx, 0, B, S, l_max / S, True, jit, off, tgt, l_max, lr=0.0, optimizer_step=False)
    return fs


@pytest.mark.parametrize("left", [900, 500, 300])
def test_fused_step_with_little_memory(device, left):
    """2^20 slots: 200 MiB per sample, 1.6 GB of records."""
    print(f"[memory] fused step, {left} MiB", flush=True)
    B, S = 8192, 128
    b = batch(device, B)
    fs = fused(device, B, S, b)
    want, ref, y = fs._bins._buffer.numel(), fs.grad.clone(), fs.y_pred.clone()
    assert want > 900 * MIB
    del fs
    with room(device, left * MIB):
        fs = fused(device, B, S, b)
        assert torch.equal(fs.y_pred, y)
        same(fs.grad, ref)
        assert fs._bins._buffer is None or fs._bins._buffer.numel() < left * MIB


def test_fused_step_memory_budget(device):
    """A batch that the budget cuts in two, one that it leaves no room beside and one that it leaves some: the records lie
    within it, and the gradient is that without a budget."""
    B, S = 16384, 128
    b = batch(device, B)
    fs = fused(device, B, S, b)
    ref, per_ray = fs.grad.clone(), fs.slot_bytes() * S
    del fs
    fixed = None
    for rays, spare, own in [(B // 2, 0, False), (B, 0, False), (B, 1 << 30, True)]:
        budget = per_ray * rays + spare
        print(f"[memory] budget {budget / MIB:.0f} MiB", flush=True)
        fs, used = peak(device, lambda: fused(device, B, S, b, memory_budget=budget))
        assert fs.chunk_rays == rays
        same(fs.grad, ref)
        assert fs._use_bins(rays * S)
        assert (fs._bins._buffer is not None) == own
        # beside the budget: parameters, rays and the like, the same for all
        fixed = used - budget if fixed is None else fixed
        assert used <= budget + fixed + 64 * MIB, (used, budget, fixed)
        assert fixed < 400 * MIB
        del fs


def test_module_step_with_little_memory(device):
    from nect_amd.module_step import ModuleTrainStep
    from nect_amd.networks import QuadCubes

    B, S = 4096, 64
    print("[memory] module step", flush=True)
    l_max, geo, idx, jit, off, tgt = batch(device, B)
    enc = {"otype": "HashGrid", "n_levels": 16, "n_features_per_level": 4, "log2_hashmap_size": 15, "base_resolution": 8,
           "per_level_scale": 1.3}
    net = {"otype": "FullyFusedMLP", "activation": "LeakyReLU", "output_activation": "None", "n_neurons": 128,
           "n_hidden_layers": 2}
    m = QuadCubes(enc, net, include_identity=True, dtype=torch.float16, seed=4).to(device)

    def run(**kw):
        st = ModuleTrainStep(m, torch.float16, B, S, loss="L2", dynamic=True, **kw)
        st.GROUPS_MIN_WORKGROUPS = 0
        st.step(geo, 0.8, idx, 0, B, S, l_max / S, True, jit, off, tgt, l_max, lr=0.0, t=0.6, optimizer_step=False)
        return st

    st = run()
    ref, want = st.grad.clone(), st._bins._buffer.numel()
    del st
    st, used = peak(device, lambda: run(scatter_bytes=0))
    assert not st._use_bins(B * S) and st._bins._buffer is None
    same(st.grad, ref)
    del st
    assert want > 256 * MIB
    with room(device, used + 96 * MIB):
        st = run()
        same(st.grad, ref)


def test_points_with_little_memory(device, monkeypatch):
    from nect_amd import tcnn

    print("[memory] points", flush=True)
    enc = {"otype": "HashGrid", "n_levels": 16, "n_features_per_level": 2, "log2_hashmap_size": 15, "base_resolution": 16,
           "per_level_scale": 1.5}
    m = tcnn.Encoding(3, enc, dtype=torch.float16).to(device)
    x = torch.rand((400_000, 3), device=device, generator=torch.Generator(device=device).manual_seed(2))
    dy = torch.randn((400_000, 32), device=device, generator=torch.Generator(device=device).manual_seed(3)).half()

    def run():
        m.zero_grad()
        m(x).backward(dy)
        return m.params.grad.clone()

    ref = run()
    with monkeypatch.context() as mp:
        mp.setattr(tcnn, "POINTS_SCATTER_BYTES", 0)
        got, used = peak(device, run)
        same(got, ref)
    with room(device, used + 32 * MIB):
        same(run(), ref)
