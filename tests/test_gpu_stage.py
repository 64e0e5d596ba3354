"""Stages (one native call for a run of modules) against the modules called one by one: same bits in
inference, same sums in training, and the cases in which the modules have to be called themselves."""
import copy

import numpy as np
import pytest
import torch

from torchsparse_amd.utils.synthetic import uniform_voxels

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def mods():
    import torchsparse_amd as ts
    from torchsparse_amd import backbones, backend
    from torchsparse_amd import nn as spnn
    from torchsparse_amd.nn.utils import fuse_inference, stage
    return ts, spnn, backbones, backend, stage, fuse_inference


def cloud(n, extent, seed, ascending=True):
    rows = uniform_voxels(n, extent=extent, seed=seed)
    if ascending:
        rows = rows[np.lexsort(rows.T[::-1])]
    return torch.from_numpy(np.ascontiguousarray(rows)).cuda()


def both(stage, fn, monkeypatch):
    """fn() through the modules, and as stages; how many native calls the latter made."""
    monkeypatch.setattr(stage, "enabled", False)
    one = fn()
    monkeypatch.setattr(stage, "enabled", True)
    calls = []
    real = stage.run
    monkeypatch.setattr(stage, "run", lambda *a, **k: (lambda y: (calls.append(y is not None), y)[1])(real(*a, **k)))
    two = fn()
    monkeypatch.setattr(stage, "run", real)
    return one, two, sum(calls)


@pytest.mark.parametrize("n,extent,dtype,segments", [
    (700, 16, torch.float16, False), (9000, 40, torch.bfloat16, "always"), (3000, 24, torch.float32, False),
    (40000, 90, torch.float16, "always")])
def test_inference_networks_give_the_same_bits(mods, n, extent, dtype, segments, monkeypatch):
    ts, _, backbones, backend, stage, fuse_inference = mods
    # (left to itself the form of a layer depends on whether its map's density has arrived yet)
    monkeypatch.setattr(backend, "igemm_through_segments", segments)
    torch.manual_seed(n)
    coords = cloud(n, extent, n)
    for net, cin in ((backbones.SparseResUNet42(in_channels=4), 4), (backbones.VoxelResBackBone8x(in_channels=5), 5)):
        net = fuse_inference(net.cuda().to(dtype).eval())
        feats = torch.randn(n, cin, device="cuda").to(dtype)

        def forward():
            with torch.no_grad():
                out = net(ts.SparseTensor(feats, coords.clone()))
            out = out.values() if isinstance(out, dict) else out
            return [(t.feats.clone(), t.coords, t.stride) for t in out]
        forward()  # (the maps of the passes below are queued ahead alike)
        one, two, calls = both(stage, forward, monkeypatch)
        assert calls >= 5
        for (a, ca, sa), (b, cb, sb) in zip(one, two):
            assert sa == sb and torch.equal(ca, cb) and torch.equal(a, b)


def _grads(module, ts, coords, feats, above=None, seed=0):
    """Output, input gradient, parameter gradients and norm statistics of one training pass."""
    module = copy.deepcopy(module)
    x = feats.clone().requires_grad_()
    t = ts.SparseTensor(x, coords)
    if above is not None:
        t = above(t)
    y = module(t).feats
    g = torch.Generator(device="cuda").manual_seed(seed)
    y.backward(torch.randn(y.shape, device="cuda", generator=g).to(y.dtype))
    out = {"y": y.detach(), "dx": x.grad}
    out.update({"grad " + k: p.grad for k, p in module.named_parameters()})
    out.update({k: b for k, b in module.named_buffers()})
    return out


def _close(one, two, tol):
    assert one.keys() == two.keys()
    for k in one:
        a, b = one[k].double(), two[k].double()
        assert a.shape == b.shape, k
        err = float((a - b).norm() / (a.norm() + 1e-30))
        assert err < tol, (k, err)


@pytest.mark.parametrize("ascending", [True, False])
@pytest.mark.parametrize("cin,cout,n,dtype,tol", [
    (32, 32, 2500, torch.float32, 2e-5), (16, 48, 5000, torch.float32, 2e-5), (4, 32, 300, torch.float32, 2e-5),
    (6, 24, 6001, torch.float32, 2e-5), (128, 256, 700, torch.float32, 2e-5), (64, 128, 13000, torch.bfloat16, 8e-2),
    (64, 64, 9000, torch.float16, 2e-2), (4, 32, 4097, torch.float16, 2e-2)])
def test_training_blocks_have_the_gradients_of_their_modules(mods, cin, cout, n, dtype, tol, ascending, monkeypatch):
    ts, spnn, backbones, backend, stage, _ = mods
    from torchsparse_amd.backbones.modules import SparseConvBlock, SparseResBlock
    if dtype == torch.bfloat16:  # (its wide layer over pair segments, in both directions)
        monkeypatch.setattr(backend, "igemm_through_segments", "always")
    torch.manual_seed(cin + cout)
    coords = cloud(n, max(int((4 * n) ** (1 / 3)), 8), n, ascending)
    feats = torch.randn(n, cin, device="cuda").to(dtype)
    for block in (SparseConvBlock(cin, cout, 3), SparseConvBlock(cin, cout, 2, stride=2),
                  SparseConvBlock(cin, cout, 3, stride=2), SparseResBlock(cin, cout, 3)):
        block = block.cuda().to(dtype).train()
        with torch.no_grad():
            for m in block.modules():
                if isinstance(m, spnn.BatchNorm):
                    m.weight.uniform_(0.5, 1.5), m.bias.normal_()
        one, two, calls = both(stage, lambda: _grads(block, ts, coords, feats), monkeypatch)
        assert calls == 1
        _close(one, two, tol)


# (gradients through ten ReLUs: a rounding that moves a value across zero switches that value's gradient on or off)
@pytest.mark.parametrize("dtype,tol,norm_tol", [(torch.float32, 1e-4, 1e-2), (torch.float16, 2e-2, 1e-1)])
def test_training_a_network_of_stages(mods, dtype, tol, norm_tol, monkeypatch):
    ts, spnn, backbones, _, stage, _ = mods
    torch.manual_seed(3)
    n = 20000
    coords = cloud(n, 70, 5)
    net = backbones.SparseResUNet42(in_channels=4).cuda().to(dtype).train()
    feats = torch.randn(n, 4, device="cuda").to(dtype)

    def step():
        model = copy.deepcopy(net)
        y = model(ts.SparseTensor(feats, coords.clone()))[-1].feats
        (y.float().square().mean() * 64).backward()
        norms = torch.stack([p.grad.float().norm() for p in model.parameters()])
        batches = torch.stack([b for k, b in model.named_buffers() if k.endswith("tracked")])
        stats = torch.cat([b.float() for k, b in model.named_buffers() if "running" in k])
        return {"y": y.detach(), "norms": norms, "stats": stats, "batches": batches.float()}
    one, two, calls = both(stage, step, monkeypatch)
    assert calls >= 9 and bool((two["batches"] == 1).all())
    _close({"norms": one.pop("norms")}, {"norms": two.pop("norms")}, norm_tol)
    _close(one, two, tol)


def test_second_backward_and_frozen_parameters(mods):
    ts, spnn, backbones, _, stage, _ = mods
    from torchsparse_amd.backbones.modules import SparseResBlock
    torch.manual_seed(1)
    coords, feats = cloud(500, 14, 1), torch.randn(500, 16, device="cuda")
    block = SparseResBlock(16, 16, 3).cuda().train()
    y = block(ts.SparseTensor(feats, coords)).feats
    y.sum().backward(retain_graph=True)
    first = block.main[0].kernel.grad.clone()
    y.sum().backward()
    assert torch.allclose(block.main[0].kernel.grad, 2 * first)
    with pytest.raises(RuntimeError):
        y.sum().backward()
    block.main[0].kernel.requires_grad_(False)
    block.zero_grad(set_to_none=True)
    block(ts.SparseTensor(feats, coords)).feats.sum().backward()
    assert block.main[0].kernel.grad is None and block.main[3].kernel.grad is not None
    y = block(ts.SparseTensor(feats, coords)).feats
    with torch.no_grad():
        block.main[3].kernel.add_(1)  # what the backward needs has been written over
    with pytest.raises(RuntimeError):
        y.sum().backward()


def test_changed_weights_replaced_parameters_and_hooks(mods):
    ts, spnn, backbones, _, stage, fuse_inference = mods
    torch.manual_seed(2)
    coords, feats = cloud(3000, 64, 3), torch.randn(3000, 5, device="cuda", dtype=torch.float16)
    net = fuse_inference(backbones.VoxelResBackBone8x(in_channels=5).cuda().half().eval())

    def forward():
        with torch.no_grad():
            return net(ts.SparseTensor(feats, coords))["out"].feats.clone()

    def check():
        got = forward()
        stage.enabled = False
        want = forward()
        stage.enabled = True
        assert torch.equal(got, want)
        return got
    a = check()
    with torch.no_grad():
        net.conv2[0][0].kernel.mul_(1.5)
    b = check()
    net.conv2[0][0].kernel = torch.nn.Parameter(net.conv2[0][0].kernel.detach() * 0.5)
    c = check()
    assert len(a) and not torch.equal(a, b) and not torch.equal(b, c)
    seen = []
    handle = net.conv2[0][0].register_forward_hook(lambda m, i, o: seen.append(o.feats.shape))
    check()
    assert len(seen) == 2  # a hook is called in both forms
    handle.remove()
    net.float()
    feats = feats.float()
    check()


@pytest.mark.parametrize("cin,cout,kernel,stride,n,dtype,tol", [
    (23, 45, 3, 1, 3000, torch.float32, 2e-5), (3, 1, 3, 1, 700, torch.float32, 2e-5), (9, 7, 2, 2, 129, torch.float16, 2e-2),
    (5, 33, 3, 2, 4000, torch.bfloat16, 8e-2), (64, 96, 3, 1, 5000, torch.float16, 2e-2), (1, 17, 5, 1, 65, torch.float16, 2e-2)])
def test_a_layer_on_its_own(mods, cin, cout, kernel, stride, n, dtype, tol, monkeypatch):
    """Rows that are not whole 16-byte pieces, forward and both gradients; the result may be written over."""
    ts, spnn, _, _, stage, _ = mods
    torch.manual_seed(n)
    coords = cloud(n, max(int((4 * n) ** (1 / 3)), 8), n)
    layer = spnn.Conv3d(cin, cout, kernel, stride=stride, padding=1).cuda().to(dtype).train()
    feats = torch.randn(n, cin, device="cuda").to(dtype)

    def step():
        x = feats.clone().requires_grad_()
        layer.zero_grad(set_to_none=True)
        y = layer(ts.SparseTensor(x, coords)).feats
        out = y.detach().clone()
        y.mul_(2)
        y.backward(torch.cos(torch.arange(y.numel(), device="cuda").view_as(y)).to(dtype))
        return {"y": out, "dx": x.grad, "dw": layer.kernel.grad}
    one, two, calls = both(stage, step, monkeypatch)
    assert calls == 1
    _close(one, two, tol)


@pytest.mark.parametrize("dataflow", ["GatherScatter", "FetchOnDemand"])
@pytest.mark.parametrize("cin,cout,kernel,stride,n,dtype,tol", [
    (13, 64, 3, 2, 2651, torch.float16, 2e-2), (23, 45, 3, 1, 3000, torch.float32, 2e-5), (32, 32, 2, 2, 515, torch.float32, 2e-5),
    (64, 128, 3, 1, 5000, torch.bfloat16, 8e-2), (3, 17, 5, 1, 65, torch.float16, 2e-2)])
def test_training_layers_over_pair_lists(mods, cin, cout, kernel, stride, n, dtype, tol, dataflow, monkeypatch):
    """A layer, and where it is strided the transposed one back up, in the dataflows of pair lists."""
    ts, spnn, _, _, stage, _ = mods
    from torchsparse_amd.nn import functional as F
    torch.manual_seed(n)
    config = F.conv_config.get_default_conv_config().copy()
    config.dataflow = getattr(F.Dataflow, dataflow)
    coords = cloud(n, max(int((4 * n) ** (1 / 3)), 8), n)
    layers = [spnn.Conv3d(cin, cout, kernel, stride=stride, padding=kernel // 2 if stride == 1 else 0, config=config)]
    if stride > 1:
        layers.append(spnn.Conv3d(cout, cin, kernel, stride=stride, transposed=True, config=config))
    layers = [m.cuda().to(dtype).train() for m in layers]
    feats = torch.randn(n, cin, device="cuda").to(dtype)

    def step():
        x = feats.clone().requires_grad_()
        y = ts.SparseTensor(x, coords)
        for m in layers:
            m.zero_grad(set_to_none=True)
            y = m(y)
        y = y.feats
        y.backward(torch.cos(torch.arange(y.numel(), device="cuda").view_as(y)).to(dtype))
        return {"y": y.detach(), "dx": x.grad, **{"dw%d" % i: m.kernel.grad for i, m in enumerate(layers)}}
    one, two, calls = both(stage, step, monkeypatch)
    assert calls == len(layers)
    _close(one, two, tol)


def test_layers_given_another_configuration(mods):
    """A plan made before the layers' dataflow was changed is not used again, nor the lack of one afterwards."""
    ts, spnn, backbones, _, stage, fuse_inference = mods
    from torchsparse_amd.nn import functional as F
    torch.manual_seed(4)
    coords, feats = cloud(3000, 64, 3), torch.randn(3000, 4, device="cuda", dtype=torch.float16)
    net = fuse_inference(backbones.SparseResUNet42(in_channels=4).cuda().half().eval())

    def forward():
        with torch.no_grad():
            return net(ts.SparseTensor(feats, coords.clone()))[-1].feats.float()
    want = forward()
    convs = [m for m in net.modules() if isinstance(m, spnn.Conv3d)]
    for config in (F.Dataflow.FetchOnDemand, None):
        for conv in convs:
            conv._config = None
            if config is not None:
                conv._config = F.conv_config.get_default_conv_config().copy()
                conv._config.dataflow = config
        assert (forward() - want).norm() / want.norm() < 2e-2
