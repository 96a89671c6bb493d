"""The voxelizer's work as a program that uses it makes it call: whole training
steps (projection, voxelization, a loss against a target volume, backward to the
four leaves), the step fused with its L1 loss, that step replayed from a HIP
graph, and volumes for display (no gradients).

A case is a dict of plain values:
  call      "l1" | "mse": the drop-in step with torch's loss of that name;
            "fused": voxelize_gaussians_l1_loss; "replayed": the fused step in a
            CapturedStep; "volume": the forward alone under no_grad
  D, H, W   voxels                    n         Gaussians
  channels  1 .. 4                    rotate    random rotations or none
  scale     "axis": each axis log-uniform in 0.5 .. widest voxels; "iso": one such
            draw for all three; "world": REFERENCE_SCALE; "mixture": 9 in 10 small
            (0.5 .. 2 voxels), the rest large (8 .. 32); widest is 0 for the last two
  dim, bright  ends of the uniform intensities
  layout    "uniform" | "clustered" positions
"""
import math
import os
import sys

import numpy as np
import torch
import torch.nn.functional as F

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "gs-voxelizer_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

WORLD = (1.0, 1.0, 1.0)
CENTER = (0.5, 0.5, 0.5)
REFERENCE_SCALE = (0.03, 0.01, 0.02)  # x, y, z in world units: random_gauss_init's


def _case(name, call, vol, n, channels=1, scale=("axis", 4.0), rotate=True,
          bright=(0.0, 1.0), layout="uniform"):
    c = dict(call=call, D=vol[0], H=vol[1], W=vol[2], n=n, channels=channels, scale=scale[0],
             widest=scale[1], rotate=rotate, dim=bright[0], bright=bright[1], layout=layout)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # a first try-out or a unit test: almost only launches and host work
        _case("tiny_40x48x36_2k", "l1", (40, 48, 36), 2_000),
        # the reference's README example: an uneven small volume, few Gaussians
        _case("readme_100x150x80_5k", "l1", (100, 150, 80), 5_000),
        # its multi-channel test: two channels, fixed anisotropic scales, no rotation
        _case("channels2_100x150x80_5k", "mse", (100, 150, 80), 5_000, 2, ("world", 0.0), False,
              (0.1, 1.0)),
        # its value test: 100k Gaussians crowded into a small volume (~500 to a tile)
        _case("crowded_100x150x80_100k", "mse", (100, 150, 80), 100_000, 1, ("world", 0.0), True,
              (0.01, 0.1)),
        # fitting a 128^3 scan from isotropic Gaussians, as optimisation starts out
        _case("cube128_50k", "mse", (128, 128, 128), 50_000, 1, ("iso", 3.0), False,
              (0.0, 0.5)),
        # the same loop with the loss fused and the whole step replayed from a graph
        _case("cube128_50k_replayed", "replayed", (128, 128, 128), 50_000, 1, ("iso", 3.0),
              False, (0.0, 0.5)),
        # the headline workload: one step of fitting a 256^3 scan
        _case("cube256_200k", "mse", (256, 256, 256), 200_000, 1, ("axis", 6.0)),
        # and the same through the fused L1 loss
        _case("cube256_200k_fused", "fused", (256, 256, 256), 200_000, 1, ("axis", 6.0)),
        # a colour volume whose edges no tile and no vector load divides
        _case("rgb_157x203x181_120k", "mse", (157, 203, 181), 120_000, 3, ("axis", 5.0)),
        # the largest scan fitted on one GPU in the benchmark
        _case("cube512_1m", "l1", (512, 512, 512), 1_000_000, 1, ("axis", 8.0), True,
              (0.0, 0.2)),
        # many channels, clustered, with large Gaussians: thousands to a tile
        _case("clustered256_500k_c4", "l1", (256, 256, 256), 500_000, 4, ("mixture", 0.0), True,
              (0.0, 1.0), "clustered"),
        # writing a fitted model out at a high resolution (the volume-scaling test):
        # few, large Gaussians over an odd-sized volume, forward only
        _case("volume_509x515x501_32k", "volume", (509, 515, 501), 32_000, 1, ("world", 0.0),
              False, (0.1, 1.0)),
    ]


def _vol(case):
    return case["D"], case["H"], case["W"]


def _mean_box(case):
    """Mean over the Gaussians of prod_k (6 s_k + 8): the voxels of the tiles that
    a 3-sigma box reaches, s_k in voxels."""
    def log_uniform(lo, hi):
        return (hi - lo) / math.log(hi / lo)
    kind, lo, hi = case["scale"], 0.5, case["widest"]
    if kind == "world":
        return math.prod(6.0 * s * e + 8.0 for s, e in zip(REFERENCE_SCALE, _vol(case)[::-1]))
    if kind == "axis":
        return (6.0 * log_uniform(lo, hi) + 8.0) ** 3
    if kind == "iso":
        r = math.log(hi / lo)
        m = [1.0] + [(hi ** k - lo ** k) / (k * r) for k in (1, 2, 3)]
        return 216.0 * m[3] + 864.0 * m[2] + 1152.0 * m[1] + 512.0
    small, large = 6.0 * log_uniform(0.5, 2.0) + 8.0, 6.0 * log_uniform(8.0, 32.0) + 8.0
    return 0.9 * small ** 3 + 0.1 * large ** 3


def _evaluations(case):
    """(Gaussian, voxel) evaluations of the 3-sigma boxes, about."""
    return case["n"] * min(_mean_box(case), float(math.prod(_vol(case))))


def draw(rng):
    """One more case of the same ranges: volumes from 32 to 512 on an edge, odd or
    even, 1k to 1M Gaussians, every call, channel count and kind of scale."""
    while True:
        call = rng.choice(["l1", "mse", "mse", "fused", "replayed", "volume"])
        edge = math.exp(rng.uniform(math.log(32), math.log(512)))
        vol = [min(512, max(17, round(edge * rng.uniform(0.7, 1.3)))) for _ in range(3)]
        n = round(math.exp(rng.uniform(math.log(1_000), math.log(1_000_000))))
        kind = rng.choice(["axis", "axis", "iso", "world", "mixture"])
        hi = round(rng.uniform(2.0, 8.0), 2)
        scale = (kind, hi if kind in ("axis", "iso") else 0.0)
        layout = "clustered" if kind == "mixture" or rng.random() < 0.2 else "uniform"
        bright = rng.choice([(0.0, 1.0), (0.0, 0.2), (0.1, 1.0)])
        case = _case("", call, vol, n, rng.choice([1, 1, 1, 2, 3, 4]), scale, rng.random() < 0.7,
                     bright, layout)
        c = case["channels"]
        if _evaluations(case) * (2 + c) > 1.2e10 or math.prod(vol) * c > 1.35e8:
            continue  # dearer than the largest listed one
        if n > 4 * math.prod(vol):
            continue  # more Gaussians than anyone fits to so few voxels
        return case


# ------------------------------------------------------------------ the inputs --

def _inputs(case, seed):
    """The four leaves and the target volume (D, H, W, C), on the GPU."""
    D, H, W = _vol(case)
    n, C = case["n"], case["channels"]
    g = torch.Generator(device="cuda").manual_seed(seed)

    def rand(*shape):
        return torch.rand(shape, generator=g, device="cuda", dtype=torch.float32)

    def randn(*shape):
        return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32)

    pos = rand(n, 3)
    if case["layout"] == "clustered":
        centres = rand(16, 3)
        which = torch.randint(0, 16, (n,), generator=g, device="cuda")
        pos = centres[which] + 0.05 * randn(n, 3)
    voxel = torch.tensor([1.0 / W, 1.0 / H, 1.0 / D], device="cuda")

    def log_uniform(k, lo, hi):
        return torch.exp(math.log(lo) + rand(n, k) * math.log(hi / lo))

    kind = case["scale"]
    if kind == "world":
        scale = torch.tensor(REFERENCE_SCALE, device="cuda").expand(n, 3)
    elif kind == "mixture":
        large = rand(n, 1) < 0.1
        scale = torch.where(large, log_uniform(3, 8.0, 32.0), log_uniform(3, 0.5, 2.0)) * voxel
    else:
        k = 3 if kind == "axis" else 1
        scale = log_uniform(k, 0.5, case["widest"]).expand(n, 3) * voxel
    if case["rotate"]:
        quat = randn(n, 4)
        quat = quat / quat.norm(dim=1, keepdim=True)
    else:
        quat = torch.tensor([1.0, 0.0, 0.0, 0.0], device="cuda").expand(n, 4).contiguous()
    bright = case["dim"] + (case["bright"] - case["dim"]) * rand(n, C)
    # a phantom: a dim background and a dozen ellipsoids, clipped at 1
    target = torch.full((D, H, W), 0.1, device="cuda")
    z, y, x = ((torch.arange(e, device="cuda") + 0.5) / e for e in (D, H, W))
    for _ in range(12):
        c, r, v = rand(3), 0.05 + 0.15 * rand(3), 0.5 + 0.5 * rand(1)
        inside = (((x - c[0]) / r[0]) ** 2)[None, None, :] + (((y - c[1]) / r[1]) ** 2)[None, :, None] \
            + (((z - c[2]) / r[2]) ** 2)[:, None, None] <= 1.0
        target += inside * v
    target = target.clamp_(max=1.0)[..., None].expand(D, H, W, C).contiguous()
    return pos, scale.contiguous(), quat, bright, target


class _State:
    pass


def _project(s):
    from gs_voxelizer.optim_to_render import optim_to_render
    pos, scale, quat, bright = s.leaves
    return optim_to_render(pos, scale, quat, bright, s.vol, WORLD, CENTER)


def _step(s):
    """One step of the caller's training loop; its optimiser would follow."""
    from gs_voxelizer.voxelize import voxelize_gaussians, voxelize_gaussians_l1_loss
    for t in s.leaves:
        t.grad = None
    render, conics, tile_min, tile_max, hits = _project(s)
    if s.call in ("fused", "replayed"):
        loss, volume = voxelize_gaussians_l1_loss(render, conics, s.leaves[3], s.vol, tile_min,
                                                  tile_max, hits, s.target)
    else:
        volume = voxelize_gaussians(render, conics, s.leaves[3], s.vol, tile_min, tile_max, hits)
        loss = (F.l1_loss if s.call == "l1" else F.mse_loss)(volume, s.target)
    loss.backward()
    pos, scale, quat, bright = s.leaves
    return {"volume": volume.detach(), "loss": loss.detach(), "d_pos3d": pos.grad,
            "d_scale3d": scale.grad, "d_quat": quat.grad, "d_intensities": bright.grad}


def prepare(case, seed):
    s = _State()
    s.call, s.vol = case["call"], _vol(case)
    *leaves, s.target = _inputs(case, seed)
    s.leaves = [t.requires_grad_(s.call != "volume") for t in leaves]
    if s.call == "replayed":
        from gs_voxelizer.graph import CapturedStep
        s.replay = CapturedStep(lambda: _step(s)).replay
    return s


def run(state):
    if state.call == "replayed":
        return state.replay()
    if state.call == "volume":
        from gs_voxelizer.voxelize import voxelize_gaussians
        with torch.no_grad():
            render, conics, tile_min, tile_max, hits = _project(state)
            return voxelize_gaussians(render, conics, state.leaves[3], state.vol, tile_min,
                                      tile_max, hits)
    return _step(state)


def work(case):
    """Leaves and target in, volume and leaf gradients out; per evaluation that
    passes the gate (about half of the boxes' voxels) the exponent's update, the
    product and the sum per channel, and in the backward ten moments more."""
    n, C = case["n"], case["channels"]
    voxels = math.prod(_vol(case)) * C
    passing = 0.5 * _evaluations(case)
    leaves = n * (40 + 4 * C)
    if case["call"] == "volume":
        return {"bytes": leaves + 4 * voxels, "flops": passing * (3 + 2 * C)}
    return {"bytes": 2 * leaves + 8 * voxels, "flops": passing * (3 + 2 * C + 14 + 4 * C)}


def tolerance(case):
    # Four times the largest errors against exact() over 60 cases of these ranges:
    # 7e-6 (the quaternions' and scales' gradients of thin Gaussians, whose binary32
    # projection backward is ill-conditioned), single elements 4e-4.  The L1 loss's
    # gradient jumps where a voxel meets its target to within rounding: one such
    # voxel moved the gradients of a small scene by 9e-4, and an element fully.
    if case["call"] in ("mse", "volume"):
        return {"rel": 3e-5, "max": 2e-3}
    return {"rel": 4e-3, "max": 0.5}


# ------------------------------------------------- the same values in 64 bits --
#
# The tile boxes are whole numbers defined by binary32 arithmetic in a fixed
# order, so they are formed that way (numpy, one rounding per operation); all
# that follows is binary64.

_EXACT_MOST = 1.5e11  # evaluations and channel sums that take about 10 s
_UNSIGNED = 2e-5      # |volume - target| / target that binary32 leaves without a sign


def _boxes(case, pos, scale, quat, bright):
    """(tile_min, tile_max) per axis x, y, z: (n, 3) integers, empty boxes where
    a Gaussian is dropped."""
    f = np.float32
    D, H, W = _vol(case)
    size = (W, H, D)
    vs = [f(1.0) / f(e) for e in size]  # world extent 1 on every axis
    p = [(pos[:, k] - f(0.5) + f(1.0) * f(0.5)) / vs[k] for k in range(3)]
    q0, q1, q2, q3 = (quat[:, k] for k in range(4))
    inv = f(1.0) / np.sqrt(q3 * q3 + q0 * q0 + q1 * q1 + q2 * q2)
    w, x, y, z = q0 * inv, q1 * inv, q2 * inv, q3 * inv
    one, two = f(1.0), f(2.0)
    R = [[one - two * (y * y + z * z), two * (x * y - w * z), two * (x * z + w * y)],
         [two * (x * y + w * z), one - two * (x * x + z * z), two * (y * z - w * x)],
         [two * (x * z - w * y), two * (y * z + w * x), one - two * (x * x + y * y)]]
    # M = S R^T row by row, cov = M^T M, then the voxel scaling from both sides
    M = [[scale[:, i] * R[j][i] for j in range(3)] for i in range(3)]
    iv = [one / v for v in vs]
    cov = [[(iv[i] * (M[0][i] * M[0][j] + M[1][i] * M[1][j] + M[2][i] * M[2][j])) * iv[j]
            for j in range(3)] for i in range(3)]
    a, b, c, d, e, g = cov[0][0], cov[0][1], cov[0][2], cov[1][1], cov[1][2], cov[2][2]
    det = a * d * g + two * b * c * e - a * e * e - g * b * b - d * c * c
    radius = np.ceil((f(3.0) * scale.max(1)) / min(vs))
    mean = bright[:, 0]
    for k in range(1, bright.shape[1]):
        mean = mean + bright[:, k]
    mean = mean / f(bright.shape[1])
    with np.errstate(all="ignore"):
        reach = np.sqrt(two * np.log((mean * f(1e6)).astype(np.float64)).astype(f))
    reach = np.fmin(f(3.0), reach)
    keep = (det != 0) & (radius > 0)
    lo = np.zeros(pos.shape, np.int64)
    hi = np.zeros(pos.shape, np.int64)
    for k in range(3):
        keep &= ~((p[k] + radius < 0) | (p[k] - radius > f(size[k])))
        r = np.maximum(f(0.0), np.sqrt(cov[k][k]) * reach - f(0.5))
        tiles = (size[k] + 7) // 8
        lo[:, k] = np.clip(np.trunc((p[k] - r) / f(8.0)), 0, tiles)
        hi[:, k] = np.clip(np.trunc((p[k] + r + f(7.0)) / f(8.0)), 0, tiles)
    keep &= (hi > lo).all(1)
    hi[~keep] = lo[~keep]
    return lo, hi, keep


class _Truth:
    """The volume and the gradients, by chunks of (tile, Gaussian) pairs."""

    def __init__(self, case, pos, scale, quat, bright):
        f8 = torch.float64
        self.vol = D, H, W = _vol(case)
        self.tiles = (W + 7) // 8, (H + 7) // 8, (D + 7) // 8
        n = pos.shape[0]
        lo, hi, keep = _boxes(case, *(t.cpu().numpy() for t in (pos, scale, quat, bright)))
        self.lo, self.ext = torch.from_numpy(lo).cuda(), torch.from_numpy(hi - lo).cuda()
        self.keep = torch.from_numpy(keep).cuda()
        self.end = self.ext.prod(1).cumsum(0)
        self.pairs = int(self.end[-1])
        # binary32 voxel sizes, as the API's world units are
        self.vs = torch.tensor([np.float32(1.0) / np.float32(e) for e in (W, H, D)],
                               device="cuda").to(f8)
        self.centre = pos.to(f8) / self.vs
        self.scale, self.bright = scale.to(f8), bright.to(f8)
        q = quat.to(f8)
        self.q = q / q.norm(dim=1, keepdim=True)
        w, x, y, z = self.q.unbind(1)
        self.R = torch.stack([  # columns: the Gaussian's axes in the world
            1 - 2 * (y * y + z * z), 2 * (x * y - w * z), 2 * (x * z + w * y),
            2 * (x * y + w * z), 1 - 2 * (x * x + z * z), 2 * (y * z - w * x),
            2 * (x * z - w * y), 2 * (y * z + w * x), 1 - 2 * (x * x + y * y)], 1).view(n, 3, 3)
        A = self.R * self.scale[:, None, :]
        self.cov = (A[:, :, None, :] * A[:, None, :, :]).sum(-1) / (self.vs[:, None] * self.vs)
        self.conic = torch.linalg.inv(self.cov)
        self.mean = self.bright.mean(1)
        r = torch.arange(8, device="cuda", dtype=f8) + 0.5
        zz, yy, xx = torch.meshgrid(r, r, r, indexing="ij")
        self.local = torch.stack([xx, yy, zz], -1).reshape(512, 3)

    def chunks(self, most=1 << 16):
        Tx, Ty, _ = self.tiles
        for a in range(0, self.pairs, most):
            e = torch.arange(a, min(self.pairs, a + most), device="cuda")
            g = torch.searchsorted(self.end, e, right=True)
            ext, lo = self.ext[g], self.lo[g]
            k = e - (self.end[g] - ext.prod(1))
            tx = lo[:, 0] + k % ext[:, 0]
            ty = lo[:, 1] + (k // ext[:, 0]) % ext[:, 1]
            tz = lo[:, 2] + k // (ext[:, 0] * ext[:, 1])
            origin = 8.0 * torch.stack([tx, ty, tz], 1).double()
            d = [(self.centre[g, j] - origin[:, j])[:, None] - self.local[:, j] for j in range(3)]
            Q = self.conic[g]
            power = -0.5 * (Q[:, 0, 0, None] * d[0] * d[0] + Q[:, 1, 1, None] * d[1] * d[1]
                            + Q[:, 2, 2, None] * d[2] * d[2]) \
                - (Q[:, 0, 1, None] * d[0] * d[1] + Q[:, 0, 2, None] * d[0] * d[2]
                   + Q[:, 1, 2, None] * d[1] * d[2])
            alpha = torch.exp(power)
            alpha[(power > 0) | (alpha * self.mean[g, None] < float(np.float32(1e-6)))] = 0.0
            yield g, (tz * Ty + ty) * Tx + tx, d, alpha

    def volume(self):
        D, H, W = self.vol
        Tx, Ty, Tz = self.tiles
        C = self.bright.shape[1]
        out = torch.zeros(C, Tx * Ty * Tz, 512, device="cuda", dtype=torch.float64)
        for g, tile, _, alpha in self.chunks():
            for c in range(C):
                out[c].index_add_(0, tile, alpha * self.bright[g, c, None])
        out = out.view(C, Tz, Ty, Tx, 8, 8, 8).permute(1, 4, 2, 5, 3, 6, 0)
        return out.reshape(Tz * 8, Ty * 8, Tx * 8, C)[:D, :H, :W].contiguous()

    def gradients(self, d_volume):
        D, H, W = self.vol
        Tx, Ty, Tz = self.tiles
        n, C = self.bright.shape
        padded = torch.zeros(Tz * 8, Ty * 8, Tx * 8, C, device="cuda", dtype=torch.float64)
        padded[:D, :H, :W] = d_volume
        tiled = padded.view(Tz, 8, Ty, 8, Tx, 8, C).permute(6, 0, 2, 4, 1, 3, 5)
        tiled = tiled.reshape(C, Tx * Ty * Tz, 512)
        del padded
        first = torch.zeros(n, 3, device="cuda", dtype=torch.float64)
        second = torch.zeros(n, 6, device="cuda", dtype=torch.float64)
        d_bright = torch.zeros(n, C, device="cuda", dtype=torch.float64)
        for g, tile, d, alpha in self.chunks():
            w = 0.0
            for c in range(C):
                t = alpha * tiled[c][tile]
                d_bright[:, c].index_add_(0, g, t.sum(1))
                w = w + t * self.bright[g, c, None]
            m = [w * v for v in d]
            first.index_add_(0, g, torch.stack([v.sum(1) for v in m], 1))
            second.index_add_(0, g, torch.stack(
                [-0.5 * (m[0] * d[0]).sum(1), -(m[0] * d[1]).sum(1), -(m[0] * d[2]).sum(1),
                 -0.5 * (m[1] * d[1]).sum(1), -(m[1] * d[2]).sum(1),
                 -0.5 * (m[2] * d[2]).sum(1)], 1))
        d_centre = -(self.conic @ first[:, :, None])[..., 0]
        d_scale, d_quat = self.shape_gradients(second)
        drop = ~self.keep
        # the reference multiplies by the voxel size where the chain rule divides
        grads = [d_centre * self.vs, d_scale, d_quat, d_bright]
        for t in grads:
            t[drop] = 0.0
        return grads

    def shape_gradients(self, s):
        """Scales and quaternions from the conic's gradient, with the reference's
        conventions: a 1e-7 beside det^2, no derivative of the normalisation."""
        c = self.cov
        a, b, cc, d, e, f = c[:, 0, 0], c[:, 0, 1], c[:, 0, 2], c[:, 1, 1], c[:, 1, 2], c[:, 2, 2]
        gA, gB, gC, gD, gE, gF = s.unbind(1)
        det = a * d * f + 2 * b * cc * e - a * e * e - f * b * b - d * cc * cc
        adj = [d * f - e * e, cc * e - b * f, b * e - cc * d, a * f - cc * cc, b * cc - a * e,
               a * d - b * b]
        along = sum(x * y for x, y in zip(adj, (gA, gB, gC, gD, gE, gF)))
        slope = [gD * f - gE * e + gF * d,
                 -gB * f + gC * e + gE * cc - 2 * gF * b,
                 gB * e - gC * d - 2 * gD * cc + gE * b,
                 gA * f - gC * cc + gF * a,
                 -2 * gA * e + gB * cc + gC * b - gE * a,
                 gA * d - gB * b + gD * a]
        times = (1, 2, 2, 1, 2, 1)
        by = 1.0 / (det * det + float(np.float32(1e-7)))
        h = [by * (det * slope[k] - times[k] * adj[k] * along) for k in range(6)]
        # to world units; off the diagonal each entry stands for two
        full = torch.stack([h[0], 0.5 * h[1], 0.5 * h[2], 0.5 * h[1], h[3], 0.5 * h[4],
                            0.5 * h[2], 0.5 * h[4], h[5]], 1).view(-1, 3, 3)
        full = full / (self.vs[:, None] * self.vs)
        Rt = self.R.transpose(1, 2)
        t = (2.0 * self.scale)[:, :, None] * (Rt @ full)  # row i: axis i
        d_scale = (Rt * t).sum(2)
        v = t * self.scale[:, :, None]  # v[i][j] = dL / d R[j][i]
        w, x, y, z = self.q.unbind(1)

        def r(i, j):
            return v[:, i, j]

        d_quat = torch.stack([
            2 * (z * (r(0, 1) - r(1, 0)) + y * (r(2, 0) - r(0, 2)) + x * (r(1, 2) - r(2, 1))),
            2 * (y * (r(1, 0) + r(0, 1)) + z * (r(2, 0) + r(0, 2)) + w * (r(1, 2) - r(2, 1)))
            - 4 * x * (r(2, 2) + r(1, 1)),
            2 * (x * (r(1, 0) + r(0, 1)) + w * (r(2, 0) - r(0, 2)) + z * (r(1, 2) + r(2, 1)))
            - 4 * y * (r(2, 2) + r(0, 0)),
            2 * (w * (r(0, 1) - r(1, 0)) + x * (r(2, 0) + r(0, 2)) + y * (r(1, 2) + r(2, 1)))
            - 4 * z * (r(1, 1) + r(0, 0))], 1)
        return d_scale, d_quat


def exact(case, seed):
    if _evaluations(case) * (1 + case["channels"]) > _EXACT_MOST:
        return None
    pos, scale, quat, bright, target = _inputs(case, seed)
    truth = _Truth(case, pos, scale, quat, bright)
    volume = truth.volume()
    if case["call"] == "volume":
        return volume
    diff = volume - target.double()
    if case["call"] == "mse":
        loss, d_volume = (diff * diff).mean(), 2.0 * diff / diff.numel()
    else:
        loss, d_volume = diff.abs().mean(), diff.sign() / diff.numel()
        if bool((diff.abs() <= _UNSIGNED * target).any()):
            # a voxel whose sign rounding decides: the gradients have no such value
            return {"volume": volume, "loss": loss, "d_pos3d": None, "d_scale3d": None,
                    "d_quat": None, "d_intensities": None}
    d_pos, d_scale, d_quat, d_bright = truth.gradients(d_volume)
    return {"volume": volume, "loss": loss, "d_pos3d": d_pos, "d_scale3d": d_scale,
            "d_quat": d_quat, "d_intensities": d_bright}
