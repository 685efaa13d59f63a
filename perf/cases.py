"""Workloads of the voxel framework, each a pass that a user's program makes again and again.

A case names an operation ("op") and its sizes:

  voxelize  a frame of points into an emptied map (clear + insertPointCloud)
  list      a frame of labelled points into an emptied voxel list, then list x map collision
  collide   robot map against environment map, counting or with meanings
  edt       environment map to metric distance field (clear, mergeOccupied, EDT, metric read-out)
  batch     a planner's poses of an arm against the environment in one call
  cost      clearance cost of trajectories and its gradient, for a trajectory optimiser
  sensor    a depth camera's scan cast into a probabilistic map

Everything is seeded; the clouds are depth images of box rooms, noisy box surfaces, arm links of
capsules or uniform obstacle fields, at the sizes of this repository's benchmark and tests.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "gpu-voxels_amd", "python"))

import gvx  # noqa: E402
from gvx.torch_cost import clearance_cost  # noqa: E402

SIDE = 0.01      # voxel side of every map here, metres
LINKS = 7        # joints of the arm
MAPS = {"bit": gvx.BITVECTOR_VOXELMAP, "prob": gvx.PROBAB_VOXELMAP}


def listed():
    return [
        # the small end: a scene of noisy box surfaces at 1 cm in a 1.28 m cube, where launches count
        {"name": "voxelize_bit_128", "op": "voxelize", "dx": 128, "dy": 128, "dz": 128, "map": "bit",
         "cloud": "boxes", "points": 100000},
        # a 640 x 480 depth camera's frame into the 5 m workspace of an arm
        {"name": "voxelize_prob_512", "op": "voxelize", "dx": 512, "dy": 512, "dz": 512, "map": "prob",
         "cloud": "scan", "points": 307200},
        # a labelled cloud (five objects) sorted and merged into a list, then collided with the scene
        {"name": "list_128", "op": "list", "dx": 128, "dy": 128, "dz": 128, "map": "bit", "points": 50000,
         "clouds": 5, "mode": 1},
        # an arm against a camera's map, with the links that collide
        {"name": "collide_bit_prob_512", "op": "collide", "dx": 512, "dy": 512, "dz": 512, "map": "prob",
         "types": True, "threshold": 0.8},
        # two bit vector maps of the whole workspace: the largest data a collision check reads
        {"name": "collide_bit_bit_512", "op": "collide", "dx": 512, "dy": 512, "dz": 512, "map": "bit",
         "types": False, "threshold": 1.0},
        # distance field of a small scene, once per planning cycle
        {"name": "edt_scene_128", "op": "edt", "dx": 128, "dy": 128, "dz": 128, "cloud": "boxes", "points": 100000},
        # distance field of the workspace as a depth camera sees it: thin surfaces, wide free space
        {"name": "edt_scene_512", "op": "edt", "dx": 512, "dy": 512, "dz": 512, "cloud": "scan", "points": 307200},
        # the exact transform at full load: 1 % of all voxels, uniformly spread
        {"name": "edt_uniform_512", "op": "edt", "dx": 512, "dy": 512, "dz": 512, "cloud": "uniform",
         "points": 1342177},
        # a sampling planner's edge check: few poses from the host, answers back to the host
        {"name": "batch_64_host", "op": "batch", "dx": 256, "dy": 256, "dz": 256, "map": "prob", "poses": 64,
         "points": 40000, "device": False},
        # a batch planner: 1024 poses of a finely sampled arm, all in device memory
        {"name": "batch_1024", "op": "batch", "dx": 512, "dy": 512, "dz": 512, "map": "bit", "poses": 1024,
         "points": 150000, "device": True},
        # a trajectory optimiser's step: cost and joint gradient of 256 trajectories
        {"name": "cost_256x32", "op": "cost", "dx": 512, "dy": 512, "dz": 512, "trajectories": 256, "waypoints": 32,
         "spheres": 64},
        # a depth frame with ray casting: free space along every ray, occupied at its end
        {"name": "sensor_512", "op": "sensor", "dx": 512, "dy": 512, "dz": 512, "points": 307200, "rays": True,
         "cut": False},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["voxelize", "list", "collide", "edt", "batch", "cost", "sensor"])
    c = {"op": op}
    c["dx"], c["dy"], c["dz"] = (_log(rng, 64, 512) for _ in range(3))
    if rng.random() < 0.3:  # round sizes are common too
        c["dx"] = c["dy"] = c["dz"] = rng.choice([64, 128, 192, 256, 320, 384, 512])
    nvox = c["dx"] * c["dy"] * c["dz"]
    if op == "voxelize":
        c.update(map=rng.choice(["bit", "prob"]), cloud=rng.choice(["boxes", "scan"]), points=_log(rng, 2000, 307200))
    elif op == "list":
        c.update(map=rng.choice(["bit", "prob"]), points=_log(rng, 2000, 307200), clouds=rng.randint(1, 8),
                 mode=rng.randint(0, 2))
    elif op == "collide":
        c.update(map=rng.choice(["bit", "prob"]), types=rng.random() < 0.5, threshold=round(rng.uniform(0.6, 1.0), 2))
    elif op == "edt":
        c["cloud"] = rng.choice(["boxes", "scan", "uniform"])
        if c["cloud"] == "uniform":
            c["points"] = max(64, int(nvox * math.exp(rng.uniform(math.log(0.001), math.log(0.1)))))
        else:
            c["points"] = _log(rng, 20000, 307200)
    elif op == "batch":
        c.update(map=rng.choice(["bit", "prob"]), poses=_log(rng, 4, 1024), points=_log(rng, 10000, 150000),
                 device=rng.random() < 0.5)
    elif op == "cost":
        c.update(trajectories=_log(rng, 1, 256), waypoints=rng.randint(4, 32), spheres=rng.randint(1, 64))
    else:
        c.update(points=_log(rng, 20000, 307200), rays=rng.random() < 0.8, cut=rng.random() < 0.3)
    return c


# ---------------------------------------------------------------- inputs, from the seed alone
def _gen(seed, what):
    return torch.Generator(device="cuda").manual_seed((int(seed) * 1000003 + what) % (1 << 62))


def _rand(g, *shape):
    return torch.rand(*shape, generator=g, device="cuda", dtype=torch.float64)


def _dims(case):
    return case["dx"], case["dy"], case["dz"]


def _extent(case):
    return torch.tensor(_dims(case), device="cuda", dtype=torch.float64) * SIDE


def _scene(case, seed, n):
    """n boxes of 4 to 23 % of the room, anywhere in it: lower and upper corners."""
    g = _gen(seed, 1)
    ext = _extent(case)
    size = (0.04 + 0.19 * _rand(g, n, 3)) * ext
    lo = _rand(g, n, 3) * (ext - size)
    return lo, lo + size


def _surface(case, seed, n):
    """n points on the surfaces of 20 boxes with 2 mm of noise."""
    lo, hi = _scene(case, seed, 20)
    g = _gen(seed, 2)
    ext = hi - lo
    area = torch.stack([ext[:, 1] * ext[:, 2], ext[:, 0] * ext[:, 2], ext[:, 0] * ext[:, 1]], 1)
    area = area.repeat_interleave(2, dim=1).reshape(-1)
    pick = torch.multinomial(area, n, replacement=True, generator=g)
    box, face = pick // 6, pick % 6
    p = lo[box] + _rand(g, n, 3) * ext[box]
    at = torch.where((face % 2 == 1)[:, None], hi[box], lo[box])
    axis = torch.nn.functional.one_hot(face // 2, 3).bool()
    p = torch.where(axis, at, p)
    p = p + 0.002 * torch.randn(n, 3, generator=g, device="cuda", dtype=torch.float64)
    return p.to(torch.float32).contiguous()


def _camera(case):
    ext = _extent(case)
    return ext * torch.tensor([0.5, 0.02, 0.45], device="cuda", dtype=torch.float64)


def _scan(case, seed, n, keep_nan):
    """A 4:3 depth image of about n pixels of a room with 55 boxes, back-projected; 1 % of the pixels drop out."""
    h = max(8, int(math.sqrt(n * 0.75)))
    w = max(8, n // h)
    ext, cam = _extent(case), _camera(case)
    lo, hi = _scene(case, seed, 55)
    f = w * 525.0 / 640.0
    v, u = torch.meshgrid(torch.arange(h, device="cuda", dtype=torch.float64),
                          torch.arange(w, device="cuda", dtype=torch.float64), indexing="ij")
    ray = torch.stack([(u - w / 2) / f, torch.ones_like(u), -(v - h / 2) / f], -1).reshape(-1, 3)
    inv = 1.0 / torch.where(ray.abs() < 1e-9, torch.full_like(ray, 1e-9), ray)
    margin = 2.5 * SIDE  # the walls stand a little inside the map
    wall = torch.where(inv > 0, (ext - margin - cam) * inv, (margin - cam) * inv)
    depth = wall.min(dim=1).values
    for k in range(lo.shape[0]):
        a, b = (lo[k] - cam) * inv, (hi[k] - cam) * inv
        near, far = torch.minimum(a, b).max(dim=1).values, torch.maximum(a, b).min(dim=1).values
        hit = (far >= near) & (near > 0.05 * float(ext[1]))
        depth = torch.where(hit & (near < depth), near, depth)
    g = _gen(seed, 3)
    depth = torch.where(_rand(g, depth.shape[0]) < 0.01, torch.full_like(depth, float("nan")), depth)
    p = (cam + depth[:, None] * ray).to(torch.float32)
    return p.contiguous() if keep_nan else p[~torch.isnan(depth)].contiguous()


def _uniform(case, seed, n):
    """The centres of n voxels drawn uniformly (some twice)."""
    dx, dy, dz = _dims(case)
    i = torch.randint(0, dx * dy * dz, (n,), generator=_gen(seed, 4), device="cuda")
    p = torch.stack([i % dx, (i // dx) % dy, i // (dx * dy)], 1).to(torch.float64)
    return ((p + 0.5) * SIDE).to(torch.float32).contiguous()


def _cloud(case, seed, cloud, n):
    if cloud == "boxes":
        return _surface(case, seed, n)
    return _scan(case, seed, n, False) if cloud == "scan" else _uniform(case, seed, n)


def _arm(case, seed, n):
    """A 7-joint arm standing in the room: DH rows, n link points on capsules (uneven), base, link lengths."""
    r = np.random.default_rng(int(seed) * 7 + 5)
    reach = 0.12 * min(_dims(case)) * SIDE
    dh = np.zeros((LINKS, 5), np.float32)
    dh[:, 1] = r.uniform(0.3, 1.2, LINKS) * reach
    dh[:, 2] = r.uniform(0.3, 1.2, LINKS) * reach
    dh[:, 3] = r.choice([-math.pi / 2, 0.0, math.pi / 2], LINKS)
    share = r.uniform(0.1, 1.0, LINKS)
    sizes = np.maximum(16, n * share / share.sum()).astype(np.uint32)
    clouds = []
    for k in range(LINKS):
        m = int(sizes[k])
        end = np.array([dh[k, 2], 0.0, dh[k, 1]])
        axis = end / np.linalg.norm(end)
        e1 = np.cross(axis, [0.0, 1.0, 0.0])
        e1 /= np.linalg.norm(e1)
        e2 = np.cross(axis, e1)
        a = r.uniform(0, 2 * math.pi, m)[:, None]
        rad = reach * r.uniform(0.1, 0.25)
        clouds.append(r.uniform(0, 1, m)[:, None] * end + rad * (np.cos(a) * e1 + np.sin(a) * e2))
    base = np.eye(3, 4, dtype=np.float32)
    base[:, 3] = np.array(_dims(case)) * SIDE * np.array([0.5, 0.45, 0.1])
    return dh, np.concatenate(clouds).astype(np.float32), sizes, base.reshape(12)


def _joints(seed, what, n):
    return np.random.default_rng(int(seed) * 11 + what).uniform(-math.pi, math.pi, (n, LINKS)).astype(np.float32)


def _spheres(case, seed):
    dh, _, _, base = _arm(case, seed, 16 * LINKS)
    r = np.random.default_rng(int(seed) * 13 + 1)
    n = case["spheres"]
    t = np.linspace(0.0, 1.0, n)[None, :, None]
    end = np.stack([dh[:, 2], np.zeros(LINKS), dh[:, 1]], 1)[:, None, :]
    sph = np.concatenate([t * end, r.uniform(0.02, 0.08, (LINKS, n, 1))], 2).astype(np.float32)
    return dh, sph, base


def _distance_grid(case, seed):
    """Metric distance of every voxel centre to the nearest of 24 boxes."""
    dx, dy, dz = _dims(case)
    lo, hi = (t.to(torch.float32) for t in _scene(case, seed, 24))
    at = [(torch.arange(n, device="cuda", dtype=torch.float32) + 0.5) * SIDE for n in (dx, dy, dz)]
    d = torch.full((dz, dy, dx), 1e30, device="cuda", dtype=torch.float32)
    for k in range(24):
        ex, ey, ez = ((torch.clamp(torch.maximum(lo[k, a] - at[a], at[a] - hi[k, a]), min=0.0)) ** 2 for a in range(3))
        d = torch.minimum(d, (ez[:, None] + ey[None, :])[:, :, None] + ex)
    return d.sqrt_().reshape(-1)


class _Buffer:
    """The device memory of a map as torch sees it."""

    def __init__(self, owner, shape, kind):
        self.__cuda_array_interface__ = {"data": (int(owner.device_ptr()), False), "shape": shape, "typestr": kind,
                                         "version": 3}


def _voxels(m):
    """The map's voxels without a copy: 4 words of 64 bits per bit vector voxel, else one number."""
    if m.type == gvx.BITVECTOR_VOXELMAP:
        shape, kind = (m.n, 4), "<i8"
    else:
        shape, kind = (m.n,), "|i1" if m.type == gvx.PROBAB_VOXELMAP else "<i4"
    t = torch.as_tensor(_Buffer(m, shape, kind), device="cuda")
    t.owner = m  # whoever holds the voxels holds the map: its memory goes back when the map does
    assert t.data_ptr() == m.device_ptr()
    return t


# ---------------------------------------------------------------- what the program holds before the call
def prepare(case, seed):
    gvx.init(0)
    op, dims = case["op"], _dims(case)
    s = {"case": case}
    if op == "voxelize":
        s["pts"] = _cloud(case, seed, case["cloud"], case["points"])
        s["map"] = gvx.Map(MAPS[case["map"]], dims, SIDE)
        s["out"] = _voxels(s["map"])
    elif op == "list":
        s["pts"] = _surface(case, seed + 1, case["points"])
        n, k = case["points"], case["clouds"]
        ends = np.linspace(0, n, k + 1).astype(np.int64)
        s["sizes"] = np.diff(ends).astype(np.uint32)
        s["meanings"] = np.arange(1, k + 1, dtype=np.uint32)
        s["list"] = gvx.VoxelList(dims, SIDE)
        s["ids"] = torch.zeros(n, device="cuda", dtype=torch.int32)  # at most one entry per point
        s["coords"] = torch.zeros((n, 3), device="cuda", dtype=torch.int32)
        s["bits"] = torch.zeros((n, 4), device="cuda", dtype=torch.int64)
        s["map"] = gvx.Map(MAPS[case["map"]], dims, SIDE)
        scene = torch.cat([_surface(case, seed, 100000), s["pts"][: n // 2]])
        s["mask"] = np.packbits(np.arange(256) % 2 == 0, bitorder="little") if case["mode"] == 2 else None
        torch.cuda.synchronize()
        s["map"].insert_points(scene, gvx.eBVM_OCCUPIED)
    elif op == "collide":
        dh, pts, sizes, base = _arm(case, seed, 80000)
        s["robot"] = gvx.Map(gvx.BITVECTOR_VOXELMAP, dims, SIDE)
        links = np.arange(4, 4 + LINKS, dtype=np.uint32)
        gvx.map_insert_robot(s["robot"], pts, sizes, dh, _joints(seed, 1, 1)[0], base, links)
        s["env"] = gvx.Map(MAPS[case["map"]], dims, SIDE)
        scene = torch.cat([_scan(case, seed, 307200, False), _surface(case, seed, 100000)])
        torch.cuda.synchronize()
        s["env"].insert_points(scene, gvx.eBVM_OCCUPIED)
        if case["map"] == "bit" and case["types"]:  # another arm's swept volume, pose after pose
            for k, q in enumerate(_joints(seed, 2, 8)):
                gvx.map_insert_robot(s["env"], pts, sizes, dh, q, base, links + LINKS * k)
        s["out"] = _voxels(s["robot"])
    elif op == "edt":
        pts = _cloud(case, seed, case["cloud"], case["points"])
        s["env"] = gvx.Map(gvx.PROBAB_VOXELMAP, dims, SIDE)
        s["dist"] = gvx.Map(gvx.DISTANCE_VOXELMAP, dims, SIDE)
        s["metric"] = torch.empty(s["dist"].n, device="cuda", dtype=torch.float32)
        torch.cuda.synchronize()
        s["env"].insert_points(pts, gvx.eBVM_OCCUPIED)
        s["out"] = _voxels(s["dist"])
    elif op == "batch":
        dh, pts, sizes, base = _arm(case, seed, case["points"])
        s["env"] = gvx.Map(MAPS[case["map"]], dims, SIDE)
        scene = torch.cat([_scan(case, seed, 307200, False), _surface(case, seed, 100000)])
        torch.cuda.synchronize()
        s["env"].insert_points(scene, gvx.eBVM_OCCUPIED)
        n = case["poses"]
        s["batch"] = gvx.Batch(s["env"], pts, sizes, dh, base, max_poses=n, threshold=0.7)
        s["q"] = _joints(seed, 3, n)
        if case["device"]:
            s["q"] = torch.from_numpy(s["q"]).cuda()
            s["counts"] = torch.empty(n, device="cuda", dtype=torch.int32)
            s["masks"] = torch.empty((n, 32), device="cuda", dtype=torch.uint8)
        else:
            s["counts"] = s["masks"] = None
    elif op == "cost":
        dh, sph, base = _spheres(case, seed)
        t, w = case["trajectories"], case["waypoints"]
        s["cost"] = gvx.Cost(_distance_grid(case, seed), dims, SIDE, dh, sph, eps=0.05, weight=1.0, base=base)
        s["q"] = torch.from_numpy(_joints(seed, 4, t * w).reshape(t, w, LINKS)).cuda().requires_grad_(True)
        s["up"] = (0.5 + _rand(_gen(seed, 5), t)).to(torch.float32)
    else:
        s["pts"] = _scan(case, seed, case["points"], True)
        s["map"] = gvx.Map(gvx.PROBAB_VOXELMAP, dims, SIDE)
        s["pose"] = _camera(case).cpu().numpy().astype(np.float32)
        s["robot"] = None
        if case["cut"]:
            dh, pts, sizes, base = _arm(case, seed, 80000)
            s["robot"] = gvx.Map(gvx.BITVECTOR_VOXELMAP, dims, SIDE)
            gvx.map_insert_robot(s["robot"], pts, sizes, dh, _joints(seed, 1, 1)[0], base, None, 5)
        s["out"] = _voxels(s["map"])
    torch.cuda.synchronize()
    return s


# ---------------------------------------------------------------- one pass
def run(s):
    c = s["case"]
    op = c["op"]
    if op == "voxelize":
        s["map"].clear()
        outside = s["map"].insert_points(s["pts"], gvx.eBVM_OCCUPIED)
        return {"outside": outside, "voxels": s["out"]}
    if op == "list":
        lst = s["list"]
        lst.clear()
        lst.insert_points(s["pts"], sizes=s["sizes"], meanings=s["meanings"])
        count, mask = lst.collide_map(s["map"], 0.7, mode=c["mode"], typemask=s["mask"])
        # the entries stay on the device for what comes next
        gvx.check(gvx.lib().gvx_list_read(lst.h, s["ids"].data_ptr(), s["coords"].data_ptr(), s["bits"].data_ptr(),
                                          gvx.MEM_DEVICE))
        return {"count": count, "mask": mask, "ids": s["ids"], "coords": s["coords"], "bits": s["bits"]}
    if op == "collide":
        if c["types"]:
            count, mask = s["robot"].collide_types(s["env"], c["threshold"])
            return {"count": count, "mask": mask, "voxels": s["out"]}
        return {"count": s["robot"].collide(s["env"], c["threshold"]), "voxels": s["out"]}
    if op == "edt":
        d = s["dist"]
        d.clear()
        d.merge_occupied(s["env"], threshold=0.5)
        d.pba()
        d.metric(s["metric"])
        return {"nearest": s["out"], "metric": s["metric"]}
    if op == "batch":
        counts, masks = s["batch"].collide(s["q"], s["counts"], s["masks"])
        return {"counts": counts if c["device"] else counts.view(np.int32), "masks": masks}
    if op == "cost":
        cost = clearance_cost(s["q"], s["cost"])
        (dq,) = torch.autograd.grad(cost, s["q"], s["up"])
        return {"cost": cost.detach(), "dq": dq}
    s["map"].insert_sensor_data(s["pts"], s["pose"], raycast=c["rays"], robot=s["robot"], robot_meaning=5)
    return {"voxels": s["out"]}


def work(case):
    op, n = case["op"], case["dx"] * case["dy"] * case["dz"]
    if op == "voxelize":  # the cleared voxels written, the points read, their words updated
        return {"bytes": n * (32 if case["map"] == "bit" else 1) + 20.0 * case["points"], "flops": 0}
    if op == "list":  # the points read, an entry of 48 bytes per two of them written and read out, its voxel read
        return {"bytes": 12.0 * case["points"] + (2 * 48 + 32) * case["points"] / 2, "flops": 0}
    if op == "collide":  # one side whole, the other only where the first holds something
        return {"bytes": n * (32.0 if case["map"] == "bit" else 1.0), "flops": 0}
    if op == "edt":  # log-odds in, nearest obstacle and distance out
        return {"bytes": 9.0 * n, "flops": 0}
    if op == "batch":  # points, occupancy bits, joints, answers
        return {"bytes": 12.0 * case["points"] + n / 8 + case["poses"] * (4.0 * LINKS + 36), "flops": 0}
    if op == "cost":  # eight samples per sphere, forward and backward
        sph = case["trajectories"] * case["waypoints"] * LINKS * case["spheres"]
        return {"bytes": 2 * 32.0 * sph, "flops": 300.0 * sph}
    # the points, and with rays the log-odds of about a third of the map read and written
    return {"bytes": 12.0 * case["points"] + (2.0 * n / 3 if case["rays"] else 2.0 * case["points"]), "flops": 0}


# ---------------------------------------------------------------- the same numbers in 64 bits
def _exact_metric(case, seed):
    dx, dy, dz = _dims(case)
    p = _cloud(case, seed, case["cloud"], case["points"])
    v = torch.from_numpy(np.floor(p.cpu().numpy() / np.float32(SIDE))).cuda()  # correctly rounded division
    ok = ((v >= 0) & (v < torch.tensor([dx, dy, dz], device="cuda"))).all(dim=1)
    v = v[ok].long()
    far = 1 << 28
    f = torch.full((dz, dy, dx), far, device="cuda", dtype=torch.int32)
    f[v[:, 2], v[:, 1], v[:, 0]] = 0
    for axis in range(3):
        out = f.clone()
        n = f.shape[axis]
        for k in range(1, n):
            if k % 16 == 0 and k * k >= int(out.max()):
                break
            a, b = out.narrow(axis, k, n - k), out.narrow(axis, 0, n - k)
            torch.minimum(a, f.narrow(axis, 0, n - k) + k * k, out=a)
            torch.minimum(b, f.narrow(axis, k, n - k) + k * k, out=b)
        f = out
    return f.reshape(-1).to(torch.float64).sqrt_() * float(np.float32(SIDE))


def _exact_cost(case, seed):
    dh, sph, base = (torch.from_numpy(a.astype(np.float64)).cuda() for a in _spheres(case, seed))
    t, w = case["trajectories"], case["waypoints"]
    q = torch.from_numpy(_joints(seed, 4, t * w)).cuda().double().requires_grad_(True)
    up = (0.5 + _rand(_gen(seed, 5), t)).to(torch.float32).double()
    grid = _distance_grid(case, seed)
    rot, pos = base.reshape(3, 4)[:, :3].expand(t * w, 3, 3), base.reshape(3, 4)[:, 3].expand(t * w, 3)
    dims = torch.tensor(_dims(case), device="cuda", dtype=torch.float64)
    side, eps = float(np.float32(SIDE)), float(np.float32(0.05))
    total = torch.zeros(t * w, device="cuda", dtype=torch.float64)
    for k in range(LINKS):
        x = torch.matmul(sph[k, :, :3], rot.transpose(1, 2).contiguous()) + pos[:, None]
        u = torch.minimum(torch.clamp(x / side - 0.5, min=0.0), dims - 1)
        i = torch.minimum(u.detach().floor(), dims - 2)
        fr = u - i
        i = i.long()
        at = (i[..., 2] * case["dy"] + i[..., 1]) * case["dx"] + i[..., 0]
        d = 0.0
        for c in range(8):
            cx, cy, cz = c & 1, (c >> 1) & 1, c >> 2
            wt = 1.0
            for a, hi in enumerate((cx, cy, cz)):
                wt = wt * (fr[..., a] if hi else 1 - fr[..., a])
            d = d + wt * grid[at + (cz * case["dy"] + cy) * case["dx"] + cx].double()
        total = total + (torch.clamp(sph[k, :, 3] + eps - d, min=0.0) ** 2).sum(dim=1)
        th = dh[k, 0] + q[:, k]
        ct, st, ca, sa = th.cos(), th.sin(), dh[k, 3].cos(), dh[k, 3].sin()
        zero = torch.zeros_like(ct)
        turn = torch.stack([ct, -st * ca, st * sa, st, ct * ca, -ct * sa, zero, sa + zero, ca + zero], 1).reshape(-1, 3, 3)
        step = torch.stack([dh[k, 2] * ct, dh[k, 2] * st, dh[k, 1] + zero], 1)
        pos = pos + torch.matmul(rot, step[:, :, None]).squeeze(2)
        rot = torch.matmul(rot, turn)
    cost = total.reshape(t, w).sum(dim=1)
    (dq,) = torch.autograd.grad(cost, q, up)
    return {"cost": cost.detach(), "dq": dq.reshape(t, w, LINKS)}


def exact(case, seed):
    if case["op"] == "edt":
        return {"nearest": None, "metric": _exact_metric(case, seed)}
    return _exact_cost(case, seed) if case["op"] == "cost" else None
