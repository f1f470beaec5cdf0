"""The MLP backward whose weight gradients stay in registers (one output, piecewise-linear activation, up to 64 inputs and
four hidden layers; beyond that, shared by the waves of a workgroup) against the float64 oracle, where tiles, inputs and layouts are not whole.

Tolerance of the relative 2-norm: a back-propagated value is rounded to the type once per layer (half a unit in the last
place: 2^-12 to 2^-11, 2^-9 to 2^-8), as are the activations; twelve such roundings: 6e-3 and 5e-2; float32 adds the roundings
of the sums, 2e-5.  At the kink of an activation no tolerance
holds: an activation at a rounding boundary lands a unit to either side of it, and a pre-activation that this moves across
zero changes the gradient by a neuron's share.  Samples with a pre-activation so close to zero get dL/dy = 0."""
import pytest
import torch

from oracle import mlp as om

pytestmark = pytest.mark.gpu

TOL = {torch.float32: 2e-5, torch.float16: 6e-3, torch.bfloat16: 5e-2}


def rel(got, ref):
    return (got.cpu().double() - ref).norm().item() / max(ref.norm().item(), 1e-30)


def case(d, dtype, n, seed, hidden=0):
    g = torch.Generator().manual_seed(seed)
    w = (torch.randn(d.n_params, generator=g) / 8).to(dtype)
    x = (torch.rand(n, d.n_input, generator=g) * 2 - 1).to(dtype)
    dy = torch.randn(n, 1, generator=g) / n
    # (pre-activations are taken without the slope: where one is close to zero does not depend on what follows it)
    a = x.double()
    unit = {torch.float32: 2.0 ** -18, torch.float16: 2.0 ** -10, torch.bfloat16: 2.0 ** -7}[dtype]
    for wk in om.split(w.double(), d.n_input_padded, 64, hidden, d.n_output_padded)[:-1] if hidden else []:
        z = a @ wk[:, : a.shape[1]].T
        dy[z.abs().min(1).values < unit * wk.abs().max() * a.abs().max()] = 0.0
        a = (z.clamp(min=0) if d.activation == "ReLU" else torch.where(z > 0, z, z * 0.01)).to(dtype).double()
    return w, x, dy


def oracle(d, w, x, dy, hidden, act, out_act, dtype):
    wr, xr = w.double().requires_grad_(True), x.double().requires_grad_(True)
    y = om.forward(om.split(wr, d.n_input_padded, 64, hidden, d.n_output_padded), xr, act, out_act, 1,
                   round_dtype=None if dtype == torch.float32 else dtype)
    (y * dy.double()).sum().backward()
    return wr.grad, xr.grad


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("hidden", [1, 2, 3, 4])
@pytest.mark.parametrize("act,out_act,n_in,n,pad", [
    ("ReLU", "None", 32, 1, 0), ("LeakyReLU", "Softplus", 64, 33, 0), ("None", "None", 16, 127, 0),
    ("ReLU", "Sigmoid", 48, 129, 8), ("LeakyReLU", "None", 19, 1000, 1), ("ReLU", "Softplus", 64, 40000, 8),
    ("ReLU", "None", 41, 31, 0), ("LeakyReLU", "ReLU", 32, 70001, 3)])
def test_backward(device, dtype, hidden, act, out_act, n_in, n, pad):
    run(device, dtype, hidden, act, out_act, n_in, n, pad)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("hidden,act,out_act,n_in,n,pad", [
    (5, "ReLU", "None", 32, 33, 0), (6, "LeakyReLU", "Softplus", 76, 20001, 4), (7, "ReLU", "None", 64, 129, 0),
    (1, "LeakyReLU", "None", 128, 97, 0), (1, "ReLU", "Sigmoid", 76, 40000, 4), (2, "ReLU", "None", 96, 1, 8),
    (4, "LeakyReLU", "None", 113, 1000, 1), (7, "None", "None", 19, 1500, 0), (5, "LeakyReLU", "ReLU", 48, 31, 0),
    (3, "ReLU", "None", 80, 70001, 0)])
def test_backward_shared(device, dtype, hidden, act, out_act, n_in, n, pad):
    """Deeper networks and wider inputs, whose gradients the waves of a workgroup share."""
    run(device, dtype, hidden, act, out_act, n_in, n, pad)


def run(device, dtype, hidden, act, out_act, n_in, n, pad):
    """Rows of odd strides, inputs that are no multiple of 16 or 32, fewer samples than a tile and more than one pass of the
    device; the gradient is added to, dx written for its rows and columns only."""
    from nect_amd.mlp import MlpDesc, backward

    if dtype == torch.float32 and hidden > 3:
        pytest.skip("float32 networks of more than three hidden layers are refused")
    print(f"[twin] {dtype} H={hidden} {act}/{out_act} in={n_in} n={n}", flush=True)
    d = MlpDesc(n_in, 1, 64, hidden, act, out_act)
    w, x, dy = case(d, dtype, n, hidden * 31 + n_in, hidden if act != "None" else 0)
    assert n < 10000 or hidden > 4 or int((dy != 0).sum()) > n // 200
    ref_w, ref_x = oracle(d, w, x, dy, hidden, act, out_act, dtype)
    xd = torch.full((n, n_in + pad), 9.0, dtype=dtype, device=device)
    xd[:, :n_in] = x.to(device)
    dyd = torch.full((n, 2), 9.0, device=device)
    dyd[:, :1] = dy.to(device)
    dw = torch.zeros(d.n_params, device=device)
    dx = torch.full((n + 1, n_in + 3), 7.0, device=device)
    scale = 1.0 if dtype == torch.float32 else 256.0 * n
    args = dict(loss_scale=scale, grad_scale=1.0)
    backward(d, w.to(device), xd[:, :n_in], dyd[:, :1], dw, dx[:n, :n_in], **args)
    torch.cuda.synchronize()
    assert rel(dw, ref_w) < TOL[dtype]
    assert rel(dx[:n, :n_in], ref_x) < TOL[dtype]
    assert bool((dx[n] == 7.0).all()) and bool((dx[:, n_in:] == 7.0).all())
    first = dw.clone()
    backward(d, w.to(device), xd[:, :n_in], dyd[:, :1], dw, None, **args)   # no dx; added
    torch.cuda.synchronize()
    assert torch.equal(dw, first + first)
    # the tiles past the count on the device are left out
    tiles = torch.tensor([n // 64], dtype=torch.int32, device=device)
    rows = n // 64 * 32
    dw.zero_()
    backward(d, w.to(device), xd[:, :n_in], dyd[:, :1], dw, None, n_tiles_dev=tiles, **args)
    torch.cuda.synchronize()
    if rows:
        assert rel(dw, oracle(d, w, x[:rows], dy[:rows], hidden, act, out_act, dtype)[0]) < TOL[dtype]
    else:
        assert not bool(dw.any())


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("levels,features", [(8, 2), (8, 4), (16, 2), (16, 4), (32, 2)])
def test_grouped_input(device, dtype, levels, features):
    """Inputs in eight planes of 2 to 8 elements: the gradients of the same values in rows."""
    from nect_amd import _lib
    from nect_amd.grid import GridDesc
    from nect_amd.mlp import MlpDesc, workspace_bytes

    n, n_in = 1000, levels * features
    d = MlpDesc(n_in, 1, 64, 2, "LeakyReLU", "Softplus")
    desc = GridDesc(3, levels, features, 10, 4, 1.3)
    w, x, dy = case(d, dtype, n, n_in)
    w, x, dy = w.to(device), x.to(device), dy.to(device)
    vpp = n_in // 8
    planes = torch.empty((8, n, vpp), dtype=dtype, device=device)
    for i in range(n_in):
        level, f = divmod(i, features)
        # level l is entry l // 8 of a plane, the planes taken forwards and backwards in turn
        g, j = (level % 8, level // 8) if (level // 8) % 2 == 0 else (7 - level % 8, level // 8)
        planes[g, :, j * features + f] = x[:, i]
    out = []
    for groups, src in ((None, x.contiguous()), (desc.struct_ref(), planes)):
        dw, dx = torch.zeros(d.n_params, device=device), torch.zeros((n, n_in), device=device)
        need = workspace_bytes(d, dtype, n)
        ws = torch.empty(need, dtype=torch.uint8, device=device)
        _lib.call("nect_mlp_backward", d.struct_ref(), _lib.dtype_code(dtype), w.data_ptr(), src.data_ptr(), n, n_in,
                  groups, None, dy.data_ptr(), 1, 1.0 if dtype == torch.float32 else 1000.0, None, 1.0, dw.data_ptr(),
                  dx.data_ptr(), n_in, ws.data_ptr(), need, _lib.stream_of(device))
        torch.cuda.synchronize()
        out.append((dw, dx))
    tol = TOL[dtype]   # the inputs' order within a sum differs
    assert rel(out[1][0], out[0][0].cpu().double()) < tol and rel(out[1][1], out[0][1].cpu().double()) < tol


@pytest.mark.parametrize("act", ["ReLU", "LeakyReLU"])
@pytest.mark.parametrize("value", [float("nan"), float("inf"), -float("inf")])
def test_not_finite(device, act, value):
    """A sample that is not finite makes the weight gradient not finite and leaves the other samples' dx as it was."""
    from nect_amd.mlp import MlpDesc, backward

    d = MlpDesc(32, 1, 64, 2, act, "None")
    w, x, dy = (v.to(device) for v in case(d, torch.float16, 500, 3))
    res = []
    for bad in (False, True):
        if bad:
            x[77, 5] = value
        dw, dx = torch.zeros(d.n_params, device=device), torch.zeros((500, 32), device=device)
        backward(d, w, x, dy, dw, dx, loss_scale=1000.0, grad_scale=1.0)
        torch.cuda.synchronize()
        res.append((dw, dx))
    keep = torch.arange(500, device=device) != 77
    assert torch.equal(res[0][1][keep], res[1][1][keep])
    assert bool(torch.isfinite(res[0][0]).all()) and not bool(torch.isfinite(res[1][0]).all())


@pytest.mark.parametrize("act", ["ReLU", "LeakyReLU"])
def test_float16_rounding(device, act):
    """dL/dz is the product rounded to float32 and then to float16: with W0 a permutation, dL/dx is dL/dz itself, bit for bit."""
    from nect_amd.mlp import MlpDesc, backward

    d = MlpDesc(64, 1, 64, 1, act, "None")
    g = torch.Generator().manual_seed(4)
    n = 100_000
    wo = torch.randn(64, generator=g).half()
    w = torch.zeros(d.n_params, dtype=torch.float16)
    w[:4096] = torch.eye(64).half().flatten()
    w[4096:4160] = wo
    x = (torch.randn(n, 64, generator=g)).half()
    dy = torch.randn(n, 1, generator=g)
    dw, dx = torch.zeros(d.n_params, device=device), torch.zeros((n, 64), device=device)
    backward(d, w.to(device), x.to(device), dy.to(device), dw, dx, loss_scale=1.0, grad_scale=1.0)
    torch.cuda.synchronize()
    p = dy * wo.float()
    below = p * 0.01 if act == "LeakyReLU" else torch.zeros_like(p)
    assert torch.equal(dx.cpu(), torch.where(x > 0, p, below).half().float())


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("hidden,act,n_in", [(6, "LeakyReLU", 76), (5, "ReLU", 32), (2, "ReLU", 128), (3, "LeakyReLU", 32)])
@pytest.mark.parametrize("tiles", [1, 6, 7, 8, 1029, 1030, 1031])
def test_rows_past_the_count(device, dtype, hidden, act, n_in, tiles):
    """Rows of the tiles past the count on the device hold whatever their memory held: with NaN and infinities there, the
    weight gradient is bit for bit that of zeros there, also where a workgroup's waves have 1, 2 or 3 live tiles."""
    from nect_amd.mlp import MlpDesc, backward

    print(f"[twin] past the count {dtype} H={hidden} {act} in={n_in} tiles={tiles}", flush=True)
    n, rows = 32 * (tiles + 5), 32 * tiles
    d = MlpDesc(n_in, 1, 64, hidden, act, "None")
    w, x, dy = (v.to(device) for v in case(d, dtype, n, tiles))
    count = torch.tensor([tiles], dtype=torch.int32, device=device)
    res = []
    for value in (0.0, float("nan"), float("inf"), -float("inf")):
        x[rows:], dy[rows:] = value, value
        dw = torch.zeros(d.n_params, device=device)
        backward(d, w, x, dy, dw, None, n_tiles_dev=count, loss_scale=256.0 * n, grad_scale=1.0)
        torch.cuda.synchronize()
        res.append(dw)
    assert bool(torch.isfinite(res[0]).all()) and bool(res[0].any())
    for dw in res[1:]:
        assert torch.equal(dw, res[0])
