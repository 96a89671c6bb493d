"""The native autograd nodes (csrc/autograd.cpp) against the Python classes they
stand in for: the same launches on the same data, so every output and gradient is
the same bits; and the calls that have to stay with the classes do."""
import pytest
import torch
import torch.nn.functional as F

from gs_voxelizer import synthetic as S
from helpers import small_config

pytestmark = pytest.mark.gpu


def _leaves(device, channels=1, n=900, vol=(20, 30, 17), seed=3):
    w = S.make_gaussians(small_config(1, n, vol=vol, channels=channels), seed=seed).to(device)
    return [t.clone().requires_grad_() for t in (w.pos3d, w.scale3d, w.quat, w.intensities)], w.cfg


def _run(leaves, cfg, classes, use, target):
    """One step through the public functions, or through the Python classes."""
    from gs_voxelizer import optim_to_render as o, voxelize as v
    for t in leaves:
        t.grad = None
    pos, scale, quat, inten = leaves
    if classes:
        pr, cn, tmin, tmax, nt = o._OptimToRender.apply(
            pos.contiguous(), scale.contiguous(), quat.contiguous(), inten.contiguous(), cfg.vol,
            cfg.world, cfg.center, None)
    else:
        pr, cn, tmin, tmax, nt = o.optim_to_render(pos, scale, quat, inten, cfg.vol, cfg.world,
                                                   cfg.center)
    args = (pr, cn, inten.contiguous(), cfg.vol, tmin, tmax, nt)
    if use == "volume":
        vol = (v._VoxelizeGaussians.apply(*args, True) if classes
               else v.voxelize_gaussians(*args))
        loss = F.mse_loss(vol, target.view(vol.shape))
        loss.backward()
    else:
        loss, vol = (v._VoxelizeL1.apply(*args, target, True) if classes
                     else v.voxelize_gaussians_l1_loss(*args, target))
        {"l1": loss, "l1_volume_only": vol.square().mean(), "l1_both": loss + vol.mean()}[
            use].backward()
    return [pr, cn, tmin, tmax, nt, vol, loss] + [t.grad for t in leaves]


def _same(a, b):
    for x, y in zip(a, b):
        assert (x is None) == (y is None)
        assert x is None or torch.equal(x, y)


@pytest.mark.parametrize("use", ["volume", "l1", "l1_volume_only", "l1_both"])
@pytest.mark.parametrize("form", ["c1", "c2", "c4", "strided", "some_leaves", "one_gaussian"])
def test_same_bits_as_the_python_classes(device, form, use):
    leaves, cfg = _leaves(device, {"c2": 2, "c4": 4}.get(form, 1),
                          n=1 if form == "one_gaussian" else 900)
    if form == "strided":  # leaves whose rows are not adjacent
        leaves = [torch.stack([t.detach(), t.detach()], 1)[:, 0].requires_grad_() for t in leaves]
        assert not leaves[0].is_contiguous()
    if form == "some_leaves":
        leaves[1].requires_grad_(False)
        leaves[3].requires_grad_(False)
    shape = cfg.vol + (leaves[3].shape[1],)
    target = torch.rand(shape, device=device)
    _run(leaves, cfg, True, use, target)  # records the capacity
    ref = _run(leaves, cfg, True, use, target)
    got = _run(leaves, cfg, False, use, target)
    assert "CppNode" in got[0].grad_fn.name() and "_Voxelize" in ref[5].grad_fn.name()
    assert "CppNode" in got[5].grad_fn.name()
    _same(got, ref)


def test_a_scene_that_outgrows_or_misses_the_volume(device):
    from gs_voxelizer import voxelize as v
    leaves, cfg = _leaves(device)
    target = torch.rand(cfg.vol + (1,), device=device)
    ref = _run(leaves, cfg, True, "volume", target)
    key = leaves[0].device.index or 0
    v._capacity[key] = 8
    _same(_run(leaves, cfg, False, "volume", target), ref)
    assert v._capacity[key] > 8
    away = [t.detach().clone().requires_grad_() for t in leaves]
    with torch.no_grad():
        away[0] += 50.0
    out = _run(away, cfg, False, "volume", target)
    assert not out[5].any() and not any(t.any() for t in out[7:])


def test_hooks_streams_and_refusals(device):
    from gs_voxelizer import optim_to_render as o, voxelize as v
    leaves, cfg = _leaves(device)
    target = torch.rand(cfg.vol + (1,), device=device)
    _run(leaves, cfg, True, "volume", target)
    ref = _run(leaves, cfg, True, "volume", target)
    # saved-tensor hooks see what the nodes keep, and their answer is what is used
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(1) or t.cpu(),
                                                  lambda t: t.to(device)):
        got = _run(leaves, cfg, False, "volume", target)
    assert len(packed) >= 14
    _same(got, ref)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        got = _run(leaves, cfg, False, "volume", target)
    torch.cuda.current_stream().wait_stream(side)
    _same(got, ref)
    pr, cn, tmin, tmax, nt = o.optim_to_render(*leaves, cfg.vol, cfg.world, cfg.center)
    vol = v.voxelize_gaussians(pr, cn, leaves[3], cfg.vol, tmin, tmax, nt)
    vol.sum().backward()
    with pytest.raises(RuntimeError, match="second time"):
        vol.sum().backward()
    # what the classes refuse stays refused
    def volume(inten):
        return v.voxelize_gaussians(pr.detach(), cn.detach(), inten, cfg.vol, tmin, tmax, nt)
    inten = leaves[3].detach()
    with pytest.raises(RuntimeError):
        torch.func.grad(lambda t: volume(t).sum())(inten)
    with pytest.raises(RuntimeError):
        torch.func.vmap(volume)(torch.stack([inten, inten]))
    with pytest.raises(RuntimeError):  # NotImplementedError is one
        with torch.autograd.forward_ad.dual_level():
            volume(torch.autograd.forward_ad.make_dual(inten, inten))
    with pytest.raises(RuntimeError, match="scalar type"):
        volume(inten.double())
    with pytest.raises(ValueError):
        o.optim_to_render(leaves[0][:0], *leaves[1:], cfg.vol, cfg.world, cfg.center)


@pytest.mark.parametrize("change", ["cpu", "half", "shorter"])
@pytest.mark.parametrize("node", ["project", "volume", "l1"])
def test_saved_tensors_that_hooks_exchanged_are_refused(device, node, change):
    """What the hooks hand back is checked on the host, before its address is used."""
    from gs_voxelizer import optim_to_render as o, voxelize as v
    leaves, cfg = _leaves(device)
    target = torch.rand(cfg.vol + (1,), device=device)
    _run(leaves, cfg, True, "volume", target)
    unpack = {"cpu": lambda t: t.cpu(), "half": lambda t: t.half(),
              "shorter": lambda t: t.flatten()[:-1]}[change]
    hooks = torch.autograd.graph.saved_tensors_hooks(lambda t: t, unpack)
    pr, cn, tmin, tmax, nt = o.optim_to_render(*(t.detach() for t in leaves), cfg.vol, cfg.world,
                                               cfg.center)
    args = (pr, cn, leaves[3], cfg.vol, tmin, tmax, nt)
    with hooks:
        if node == "project":
            out = o.optim_to_render(*leaves, cfg.vol, cfg.world, cfg.center)[0]
        elif node == "volume":
            out = v.voxelize_gaussians(*args)
        else:
            out = v.voxelize_gaussians_l1_loss(*args, target)[0]
    assert "CppNode" in out.grad_fn.name()
    with pytest.raises(RuntimeError, match="values of scalar type"):
        out.sum().backward()


def test_what_makes_the_outputs_require_gradients(device):
    """As with the classes: any argument does, also one that gets no gradient."""
    from gs_voxelizer import optim_to_render as o, voxelize as v
    leaves, cfg = _leaves(device)
    target = torch.rand(cfg.vol + (1,), device=device)
    _run(leaves, cfg, True, "volume", target)
    pos, scale, quat, inten = (t.detach() for t in leaves)
    for asks in (False, True):
        pr, cn, tmin, tmax, nt = o.optim_to_render(pos, scale, quat,
                                                   inten.clone().requires_grad_(asks), cfg.vol,
                                                   cfg.world, cfg.center)
        assert pr.requires_grad is asks and cn.requires_grad is asks
        wanted = target.clone().requires_grad_(asks)
        loss, vol = v.voxelize_gaussians_l1_loss(pr.detach(), cn.detach(), inten, cfg.vol, tmin,
                                                 tmax, nt, wanted)
        assert loss.requires_grad is asks and vol.requires_grad is asks
        if asks:
            loss.backward()
            assert wanted.grad is None


@pytest.mark.parametrize("reads", [0, 1])
@pytest.mark.parametrize("use", ["volume", "l1"])
def test_a_count_that_is_late_is_waited_for(device, monkeypatch, use, reads):
    """Out of reads of the pinned count, the native node waits for its stream and
    keeps what it launched; the class does not launch the forward again."""
    from gs_voxelizer import voxelize as v
    leaves, cfg = _leaves(device)
    target = torch.rand(cfg.vol + (1,), device=device)
    _run(leaves, cfg, True, use, target)
    ref = _run(leaves, cfg, True, use, target)

    def entered(*args):
        raise AssertionError("the class launched a forward")
    monkeypatch.setattr(v, "_bin_and_forward", entered)
    monkeypatch.setattr(v, "_NATIVE_SPIN_READS", reads)
    _same(_run(leaves, cfg, False, use, target), ref)


class _Watching(torch.overrides.TorchFunctionMode):
    def __torch_function__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


@pytest.mark.parametrize("use", ["volume", "l1"])
@pytest.mark.parametrize("empty", [False, True])
def test_checkpoint_whose_recomputation_takes_the_other_route(device, use, empty):
    """A checkpointed step runs its forward under a function mode (the classes) and
    is computed again outside it (the native nodes): both keep the same tensors in
    the same order, so the recomputation fits."""
    from gs_voxelizer import optim_to_render as o, voxelize as v
    from torch.utils.checkpoint import checkpoint
    leaves, cfg = _leaves(device)
    target = torch.rand(cfg.vol + (1,), device=device)
    if empty:
        with torch.no_grad():
            leaves[0] += 50.0
        _run(leaves, cfg, True, use, target)
    _run(leaves, cfg, True, use, target)
    ref = _run(leaves, cfg, True, use, target)

    def step(*leaves):
        pr, cn, tmin, tmax, nt = o.optim_to_render(*leaves, cfg.vol, cfg.world, cfg.center)
        args = (pr, cn, leaves[3], cfg.vol, tmin, tmax, nt)
        if use == "l1":
            return v.voxelize_gaussians_l1_loss(*args, target)[0]
        return F.mse_loss(v.voxelize_gaussians(*args), target)

    for t in leaves:
        t.grad = None
    with _Watching():
        loss = checkpoint(step, *leaves, use_reentrant=False)
    loss.backward()
    _same([loss] + [t.grad for t in leaves], ref[6:])


@pytest.mark.parametrize("use", ["volume", "l1", "l1_volume_only", "l1_both"])
def test_an_empty_scene_takes_one_forward(device, monkeypatch, use):
    """No pairs: the native node's own launches give the zero volume (and the loss
    against it); the class does not launch them again."""
    from gs_voxelizer import voxelize as v
    leaves, cfg = _leaves(device)
    target = torch.rand(cfg.vol + (1,), device=device)
    _run(leaves, cfg, True, use, target)  # records a capacity
    with torch.no_grad():
        leaves[0] += 50.0
    cap = v._capacity[device.index or 0]
    ref = _run(leaves, cfg, True, use, target)
    v._capacity[device.index or 0] = cap

    def entered(*args):
        raise AssertionError("the class launched a forward")
    monkeypatch.setattr(v, "_bin_and_forward", entered)
    got = _run(leaves, cfg, False, use, target)
    assert "CppNode" in got[5].grad_fn.name()
    _same(got, ref)
    assert v._capacity[device.index or 0] == v._grow(0)
