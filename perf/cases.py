"""Performance cases of the framework's public entry points.

Each case is a dict of plain values; `kind` names the path:

  fit       batched plain cylinder RANSAC (CylinderFitPlan.exec)
  learned   proposal network + verified fit with the plain fallback (LearnedCylinderFit.exec)
  train     one Adam step of the proposal network (ProposalNet.train_step)
  pose      batched Levenberg-Marquardt pose solves (PosePlan.exec)
  plane     point-level plane RANSAC (PlaneFitPlan.exec)
  frontend  projection, partition, tree instances, axis lines and ground cells of one scan
            (Frontend.exec: one HIP graph on the plan's buffers)
  keyframe  a keyframe stream's first two scans on the device estimator, from pinned host memory
            (front end, learned tree fits, association and pose as one HIP graph per keyframe)

Inputs are seeded and drawn with torch on the GPU (clusters, poses, plane sets) or ray cast by
sloam_amd.synth (scans).  `exact` restates a path in 64 bits with torch and numpy alone.
"""
import ctypes as C
import math

import numpy as np
import torch

from sloam_amd import _lib, proposal, synth
from sloam_amd.gpu import Context, CylinderFitPlan, Frontend, PlaneFitPlan, PosePlan

SEED = 0x5EED  # Philox key of every RANSAC plan (the library's default)
XYYAW, ZROLLPITCH = 0b100011, 0b011100  # free parameters of the two-step solves


def listed():
    return [
        # the trees of one keyframe: 10 or so short trunks, fitted between two scans, where the
        # launches and the serial refit are the cost (the keyframe stream's plain tree model)
        dict(name="fit_keyframe", kind="fit", clusters=12, n_min=90, n_max=1400, hyp=1024,
             outliers=0.2),
        # the batched-fitting benchmark: 2000 trunks of 50 to 5000 points
        dict(name="fit_2000", kind="fit", clusters=2000, n_min=50, n_max=5000, hyp=1024,
             outliers=0.2),
        # a survey map refitted in one batch: dense trunks of ragged sizes up to 40000 points
        dict(name="fit_dense", kind="fit", clusters=1500, n_min=500, n_max=40000, hyp=1024,
             outliers=0.2),
        # the learned-proposal benchmark: 4096 trunks, 16 verifying hypotheses each
        dict(name="learned_4096", kind="learned", clusters=4096, n_min=50, n_max=5000,
             outliers=0.2),
        # one training step at train_proposal.py's batch size
        dict(name="train_250", kind="train", clusters=250, n_min=50, n_max=5000, outliers=0.2),
        # the two-step solve of one keyframe in FP64: 10 trees x 20 features and 36 ground cells
        # x 5 features, up to 50 iterations
        dict(name="pose_keyframe", kind="pose", problems=1, cyl=10, planes=36, pts_cyl=20,
             pts_plane=5, two_step=True, precision=1, iters=50),
        # the batched-pose benchmark: 64 problems x (500 trunks + 20 ground patches), 10 iterations
        dict(name="pose_64", kind="pose", problems=64, cyl=500, planes=20, pts_cyl=60,
             pts_plane=50, two_step=False, precision=0, iters=10),
        # the ground of one 64-beam scan as one RANSAC set, 200 hypotheses (the small-scan keyframe)
        dict(name="plane_scan", kind="plane", sets=1, n_min=27001, n_max=27001, hyp=200),
        # ground patches of a map segment as one batch
        dict(name="plane_patches", kind="plane", sets=300, n_min=40, n_max=20000, hyp=200),
        # the per-scan front end of a 64-beam and of a 128-beam sensor
        dict(name="frontend_64", kind="frontend", H=64, W=2048, lines=True),
        dict(name="frontend_128", kind="frontend", H=128, W=2048, lines=True),
        # the start of a keyframe stream: the scan that opens the map and the first estimate
        dict(name="keyframe_128", kind="keyframe", H=128, W=2048),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["fit", "fit", "learned", "train", "pose", "pose", "plane", "plane",
                       "frontend", "keyframe"])
    if kind in ("fit", "learned", "train"):
        cap = {"fit": 4000, "learned": 5000, "train": 800}[kind]
        n = _log(rng, {"fit": 1, "learned": 4, "train": 7}[kind], cap)
        n_max = _log(rng, 150, 30000 if kind == "fit" else 6000)
        while n * n_max > 1.5e7:  # at most the largest listed batch's points
            n_max = n_max // 2 + 1
        c = dict(kind=kind, clusters=n, n_min=max(3, int(n_max / rng.uniform(1.5, 120))),
                 n_max=n_max, outliers=round(rng.uniform(0.0, 0.5), 3))
        if kind == "fit":
            c["hyp"] = rng.choice([100, 200, 256, 777, 1024])
        return c
    if kind == "pose":
        return dict(kind=kind, problems=_log(rng, 1, 64), cyl=_log(rng, 4, 400),
                    planes=_log(rng, 2, 40), pts_cyl=rng.randint(5, 60),
                    pts_plane=rng.randint(5, 60), two_step=rng.random() < 0.5,
                    precision=rng.randint(0, 1), iters=rng.choice([10, 50]))
    if kind == "plane":
        sets = _log(rng, 1, 600)
        n_max = max(60, _log(rng, 60, 120000) // max(1, sets // 20))
        return dict(kind=kind, sets=sets, n_min=max(3, int(n_max / rng.uniform(1.0, 100))),
                    n_max=n_max, hyp=rng.choice([64, 200, 333, 512]))
    if kind == "frontend":
        return dict(kind=kind, H=rng.choice([16, 32, 40, 64, 100, 128]),
                    W=rng.choice([512, 900, 1024, 1800, 2048, 4000]), lines=rng.random() < 0.5)
    return dict(kind=kind, H=rng.choice([48, 64, 96, 128]), W=rng.choice([1024, 1500, 2048]))


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
_contexts = {}


def _context(key="plans"):
    """One library context per use; graphs hold their context's scratch, so each scan size has its
    own."""
    if key not in _contexts:
        _contexts[key] = Context(0)
    return _contexts[key]


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(1000003 * int(seed) + 17)
    return g


def _uniform(g, lo, hi, *shape):
    return lo + (hi - lo) * torch.rand(shape, generator=g, device="cuda", dtype=torch.float64)


def _normal(g, *shape):
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float64)


def _offsets(sizes):
    return np.concatenate([[0], np.cumsum(sizes)]).astype(np.int32)


def _sizes(case, count):
    """Ragged set sizes, log-uniform: the case's own, the same for every seed."""
    lo, hi = math.log(case["n_min"]), math.log(case["n_max"] + 1)
    u = np.random.default_rng([count, case["n_min"], case["n_max"]]).uniform(lo, hi, count)
    return np.minimum(np.floor(np.exp(u)), case["n_max"]).astype(np.int64)


def _basis(a):
    ref = torch.zeros_like(a)
    ref[:, 0] = 1.0
    e1 = ref - (ref * a).sum(1, keepdim=True) * a
    e1 = e1 / e1.norm(dim=1, keepdim=True)
    return e1, torch.linalg.cross(a, e1)


def _tilted(g, n, max_deg):
    t = torch.deg2rad(_uniform(g, 0.0, max_deg, n))
    az = _uniform(g, -math.pi, math.pi, n)
    return torch.stack([t.sin() * az.cos(), t.sin() * az.sin(), t.cos()], 1)


def _around(g, owner, axis, base, radius, height, noise, half):
    """Noisy points of the cylinders `owner` (visible half: the side facing the origin)."""
    n = owner.numel()
    e1, e2 = _basis(axis)
    face = -base / base[:, :2].norm(dim=1, keepdim=True)
    phi = torch.atan2((face[:, :2] * e2[:, :2]).sum(1), (face[:, :2] * e1[:, :2]).sum(1))
    th = phi[owner] + _uniform(g, -1.0, 1.0, n) * (math.pi / 2 if half else math.pi)
    rr = radius[owner] + noise * _normal(g, n)
    h = _uniform(g, 0.0, 1.0, n) * height[owner]
    return (base[owner] + h[:, None] * axis[owner] + (rr * th.cos())[:, None] * e1[owner] +
            (rr * th.sin())[:, None] * e2[owner])


def _clusters(case, seed):
    """Trunk clusters as the batched-fitting workload has them: the visible half of a tilted
    cylinder with 2 cm noise and a share of uniform outliers."""
    S = case["clusters"]
    off = _offsets(_sizes(case, S))
    g = _generator(seed)
    o = torch.as_tensor(off).cuda()
    owner = torch.repeat_interleave(torch.arange(S, device="cuda"), (o[1:] - o[:-1]).long())
    axis = _tilted(g, S, 5.0)
    radius = _uniform(g, 0.05, 0.6, S)
    height = _uniform(g, 2.0, 8.0, S)
    dist, bearing = _uniform(g, 1.5, 40.0, S), _uniform(g, -math.pi, math.pi, S)
    base = torch.stack([dist * bearing.cos(), dist * bearing.sin(), _uniform(g, -0.5, 0.5, S)], 1)
    p = _around(g, owner, axis, base, radius, height, 0.02, True)
    n = owner.numel()
    box = torch.stack([radius + 1.0, radius + 1.0], 1)[owner]
    out = base[owner].clone()
    out[:, :2] += _uniform(g, -1.0, 1.0, n, 2) * box
    out[:, 2] += _uniform(g, 0.0, 1.0, n) * height[owner]
    bad = _uniform(g, 0.0, 1.0, n) < case["outliers"]
    xyz = torch.where(bad[:, None], out, p).float().contiguous()
    target = torch.zeros((S, 8), dtype=torch.float64, device="cuda")
    target[:, :3], target[:, 3:6], target[:, 6] = base, axis, radius
    return dict(xyz=xyz, offsets=o, host=off, target=target)


def _plane_sets(case, seed):
    """Ground patches: tilted planes with 2 cm noise, 30 % of the points up to 2 m off."""
    S = case["sets"]
    off = _offsets(_sizes(case, S))
    g = _generator(seed)
    o = torch.as_tensor(off).cuda()
    owner = torch.repeat_interleave(torch.arange(S, device="cuda"), (o[1:] - o[:-1]).long())
    n = owner.numel()
    nrm = _tilted(g, S, 6.0)
    d = _uniform(g, 1.0, 2.0, S)
    xy = _uniform(g, -15.0, 15.0, n, 2)
    z = -((nrm[owner, :2] * xy).sum(1) + d[owner]) / nrm[owner, 2] + 0.02 * _normal(g, n)
    off_plane = _uniform(g, 0.0, 1.0, n) < 0.3
    z = z + torch.where(off_plane, _uniform(g, -2.0, 2.0, n), torch.zeros_like(z))
    return dict(xyz=torch.cat([xy, z[:, None]], 1).float().contiguous(), offsets=o, host=off)


def _quat(v):
    """Unit quaternions (x, y, z, w) of rotation vectors."""
    th = v.norm(dim=1, keepdim=True).clamp_min(1e-12)
    return torch.cat([v / th * (th / 2).sin(), (th / 2).cos()], 1)


def _quat_mul(a, b):
    ax, ay, az, aw = a.unbind(1)
    bx, by, bz, bw = b.unbind(1)
    return torch.stack([aw * bx + ax * bw + ay * bz - az * by, aw * by - ax * bz + ay * bw + az * bx,
                        aw * bz + ax * by - ay * bx + az * bw,
                        aw * bw - ax * bx - ay * by - az * bz], 1)


def _rot(q):
    x, y, z, w = q.unbind(1)
    return torch.stack([
        torch.stack([1 - 2 * (y * y + z * z), 2 * (x * y - z * w), 2 * (x * z + y * w)], 1),
        torch.stack([2 * (x * y + z * w), 1 - 2 * (x * x + z * z), 2 * (y * z - x * w)], 1),
        torch.stack([2 * (x * z - y * w), 2 * (y * z + x * w), 1 - 2 * (x * x + y * y)], 1)], 1)


def _pose_problems(case, seed):
    """Trunks and ground patches around true poses, seen from them with noise, and estimates up to
    0.5 m and 5 degrees off.  two_step: per pose an x / y / yaw problem over the trunks and a
    z / roll / pitch problem over the patches."""
    K, nc, npl = case["problems"], case["cyl"], case["planes"]
    g = _generator(seed)
    t = torch.stack([_uniform(g, -100, 100, K), _uniform(g, -100, 100, K), _uniform(g, 1, 3, K)], 1)
    yaw = torch.zeros((K, 3), dtype=torch.float64, device="cuda")
    yaw[:, 2] = _uniform(g, -math.pi, math.pi, K)
    q = _quat_mul(_quat(yaw), _quat(_uniform(g, -0.05, 0.05, K, 3)))
    ground = t[:, 2] - _uniform(g, 1.2, 2.0, K)

    def spots(n):
        r = 30.0 * _uniform(g, 0.02, 1.0, K * n).sqrt()
        b = _uniform(g, -math.pi, math.pi, K * n)
        own = torch.arange(K, device="cuda").repeat_interleave(n)
        xy = t[own, :2] + torch.stack([r * b.cos(), r * b.sin()], 1)
        return torch.cat([xy, ground[own, None]], 1), own

    root, cown = spots(nc)
    ray, rad = _tilted(g, K * nc, 5.0), _uniform(g, 0.1, 0.4, K * nc)
    cyl = torch.cat([root, ray, rad[:, None], torch.zeros_like(rad)[:, None]], 1)
    cid = torch.arange(K * nc, device="cuda").repeat_interleave(case["pts_cyl"])
    cp = _around(g, cid, ray, root - t[cown], rad, torch.full_like(rad, 6.0), 0.02, True)
    pc, pown = spots(npl)
    nrm = _tilted(g, K * npl, 5.0)
    planes = torch.cat([nrm, -(nrm * pc).sum(1, keepdim=True)], 1)
    pid = torch.arange(K * npl, device="cuda").repeat_interleave(case["pts_plane"])
    e1, e2 = _basis(nrm)
    uv = _uniform(g, -2.0, 2.0, pid.numel(), 2)
    pp = (pc[pid] + uv[:, :1] * e1[pid] + uv[:, 1:] * e2[pid] +
          0.03 * _normal(g, pid.numel(), 1) * nrm[pid])

    def seen(p, own):  # world (relative to the pose's translation) to sensor frame
        return torch.einsum("nij,ni->nj", _rot(q)[own], p)

    cs = torch.cat([seen(cp, cown[cid]), torch.zeros((cid.numel(), 1), device="cuda")], 1).float()
    ps = torch.cat([seen(pp - t[pown[pid]], pown[pid]),
                    torch.zeros((pid.numel(), 1), device="cuda")], 1).float()
    cs.view(torch.int32)[:, 3] = cid.int()
    ps.view(torch.int32)[:, 3] = -pid.int() - 1
    dt = _normal(g, K, 3)
    dt = dt / dt.norm(dim=1, keepdim=True) * _uniform(g, 0.0, 0.5, K, 1)
    dr = _normal(g, K, 3)
    dr = dr / dr.norm(dim=1, keepdim=True) * _uniform(g, 0.0, math.radians(5.0), K, 1)
    init = torch.cat([t + dt, _quat_mul(_quat(dr), q)], 1)
    a, b = nc * case["pts_cyl"], npl * case["pts_plane"]
    pts = torch.cat([cs.view(K, a, 4), ps.view(K, b, 4)], 1).reshape(-1, 4).contiguous()
    if case["two_step"]:
        sizes, mask = [a, b] * K, [XYYAW, ZROLLPITCH] * K
        co, po = [nc, 0] * K, [0, npl] * K
        init = init.repeat_interleave(2, 0)
    else:
        sizes, mask, co, po = [a + b] * K, None, [nc] * K, [npl] * K
    dev = lambda v: torch.as_tensor(_offsets(v)).cuda()  # noqa: E731
    return dict(points=pts, res=_offsets(sizes), cyl=cyl.contiguous(), cyl_off=dev(co),
                planes=planes.contiguous(), plane_off=dev(po), init=init.contiguous(),
                mask=None if mask is None else torch.tensor(mask, dtype=torch.int32).cuda())


def _scan(case, seed, k=0):
    """Scan k of a sensor moving through a forest (clutter, occlusion, sloped ground)."""
    forest = synth.make_forest(seed=int(seed) % 1000, n_trees=300)
    s = 20.0 + 0.5 * k + (int(seed) % 97)
    R, t = synth.trajectory_pose(s, ground=forest["ground"])
    sc = synth.scan_from(forest, R, t, seed=int(seed) * 10 + k, H=case["H"], W=case["W"])
    return sc, forest, R, t


class _Buffer:
    """A plan-owned device buffer, for torch; holds the plan."""

    def __init__(self, owner, ptr, shape, kind):
        self.owner = owner
        self.__cuda_array_interface__ = {"data": (int(ptr), False), "shape": tuple(shape),
                                         "typestr": kind, "version": 2}


def _view(owner, ptr, shape, kind):
    return torch.as_tensor(_Buffer(owner, ptr, shape, kind), device="cuda")


def _pose_plan_args(case):
    return dict(max_iters=case["iters"], stop_on_convergence=case["iters"] == 50,
                parametrization=int(case["two_step"]), precision=case["precision"])


# ---------------------------------------------------------------------------
# prepare / run
# ---------------------------------------------------------------------------
def prepare(case, seed):
    return {"fit": _prepare_fit, "learned": _prepare_learned, "train": _prepare_train,
            "pose": _prepare_pose, "plane": _prepare_plane, "frontend": _prepare_frontend,
            "keyframe": _prepare_keyframe}[case["kind"]](case, int(seed))


def run(state):
    return state["run"](state)


def _ready(ctx, state):
    torch.cuda.synchronize()  # torch's stream made the inputs
    ctx.sync()                # lets go of the tensors of earlier states
    return state


def _prepare_fit(case, seed):
    ctx = _context()
    d = _clusters(case, seed)
    plan = CylinderFitPlan(ctx, d["host"], n_hyp=case["hyp"], seed=SEED)
    return _ready(ctx, dict(d, plan=plan, out=plan.alloc_outputs(), run=_run_fit))


def _run_fit(s):
    return s["plan"].exec(s["xyz"], s["offsets"], s["out"])


def _prepare_learned(case, seed):
    ctx = _context()
    d = _clusters(case, seed)
    net = proposal.ProposalNet(ctx, proposal.load_weights())
    fit = proposal.LearnedCylinderFit(ctx, net, d["host"], seed=SEED)
    return _ready(ctx, dict(d, fit=fit, out=fit.alloc(), run=_run_fit_learned))


def _run_fit_learned(s):
    return s["fit"].exec(s["xyz"], s["offsets"], s["out"])


def _prepare_train(case, seed):
    ctx = _context()
    d = _clusters(case, seed)
    net = proposal.ProposalNet(ctx, proposal.init_params(seed=seed % 1000))
    loss = torch.empty(case["clusters"], dtype=torch.float32, device="cuda")
    return _ready(ctx, dict(d, net=net, loss=loss, cfg=proposal.train_cfg(), run=_run_train))


def _run_train(s):
    n = s["net"]
    n.train_step(s["xyz"], s["offsets"], s["target"], s["cfg"], s["loss"])
    return {"loss": s["loss"], "params": n.params, "m": n.m, "v": n.v}


def _prepare_pose(case, seed):
    ctx = _context()
    d = _pose_problems(case, seed)
    plan = PosePlan(ctx, d["res"], len(d["cyl"]), len(d["planes"]), **_pose_plan_args(case))
    return _ready(ctx, dict(d, plan=plan, out=plan.alloc_outputs(), run=_run_pose))


def _run_pose(s):
    return s["plan"].exec(s["points"], s["cyl"], s["cyl_off"], s["planes"], s["plane_off"],
                          s["init"], s["out"], free_mask=s["mask"])


def _prepare_plane(case, seed):
    ctx = _context()
    d = _plane_sets(case, seed)
    plan = PlaneFitPlan(ctx, d["host"], n_hyp=case["hyp"], seed=SEED)
    return _ready(ctx, dict(d, plan=plan, out=plan.alloc_outputs(), run=_run_plane))


def _run_plane(s):
    return s["plan"].exec(s["xyz"], s["offsets"], s["out"])


def _prepare_frontend(case, seed):
    # the scan and its labels are on the device already (the segmentation network ran there); the
    # plan's first exec sizes its scratch and captures its graph
    ctx = _context(("frontend", case["H"], case["W"], case["lines"]))
    sc, _, _, _ = _scan(case, seed)
    fe = Frontend(ctx, case["H"], case["W"], use_graph=True, host_results=True,
                  fit_lines=case["lines"])
    x = torch.as_tensor(np.ascontiguousarray(sc["xyzi"], np.float32)).cuda()
    lab = torch.as_tensor(np.ascontiguousarray(sc["label"], np.uint8)).cuda()
    torch.cuda.synchronize()
    s = dict(ctx=ctx, fe=fe, xyzi=x, label=lab, out={}, run=_run_frontend)
    _run_frontend(s)
    ctx.sync()
    o, N = fe.out, case["H"] * case["W"]
    shapes = {
        "mask": ((N,), "|u1"), "ground": ((N, 4), "<f4"), "n_ground": ((1,), "<i4"),
        "tree": ((N, 4), "<f4"), "trellis_counts": ((8,), "<i4"),
        "tree_offsets": ((o.cap_trees + 1,), "<i4"), "vertex_int": ((o.cap_vertices, 4), "<i4"),
        "vertex_f64": ((o.cap_vertices, 4), "<f8"), "point_offsets": ((o.cap_vertices + 1,), "<i4"),
        "points": ((o.cap_points, 4), "<f4"), "cell_info": ((o.n_cells, 4), "<i4"),
        "cell_model": ((o.n_cells, 8), "<f8")}
    if case["lines"]:
        shapes.update(line_coeff=((o.cap_trees, 6), "<f4"), line_stats=((o.cap_trees, 4), "<i4"))
    # whole buffers: zero past what a scan fills
    s["out"] = {k: _view(fe, getattr(o, k), *v).zero_() for k, v in shapes.items()}
    return _ready(ctx, s)


def _copy(ctx, dst, t):
    _lib.check(ctx.lib.sloam_memcpy_async(ctx.handle, dst, t.data_ptr(),
                                          t.numel() * t.element_size()), ctx.handle)


def _run_frontend(s):
    _copy(s["ctx"], s["fe"].out.xyzi, s["xyzi"])
    _copy(s["ctx"], s["fe"].out.label, s["label"])
    s["fe"].exec()
    return s["out"]


class _Keyframes:
    """The device keyframe as a host program drives it through the C ABI: counted learned fits and
    the estimator behind the front end, captured as one graph after the first keyframe."""

    TREES, MAP = 512, 256

    def __init__(self, ctx, H, W):
        self.ctx, self.lib = ctx, ctx.lib
        dev = torch.device("cuda")
        self.fe = Frontend(ctx, H, W, use_graph=False, host_results=True)
        o = self.fe.out
        T = self.trees = min(o.cap_trees, self.TREES)
        self.points = o.cap_points
        p = _lib.KfParams(max_lidar_dist=20.0, default_tree_radius=0.2, max_tree_radius=0.45,
                          max_axis_theta=10.0, tree_match_thresh=1.0,
                          add_new_tree_thresh_dist=1.5, min_tree_models=5.0,
                          min_ground_models=36.0, min_planes=o.n_cells * 0.1,
                          features_per_tree=20, num_ground_features=self.fe.nf, two_step=1,
                          pose_precision=1)
        self.est = self._make("sloam_kf_estimator_create", C.byref(p), T, o.n_cells, self.MAP)
        self.input = torch.zeros(8 + 8 * self.MAP, dtype=torch.float64, device=dev)
        self.off = torch.zeros(T + 1, dtype=torch.int32, device=dev)
        self.xyz = torch.zeros((self.points, 3), dtype=torch.float32, device=dev)
        self.n = torch.zeros(4, dtype=torch.int32, device=dev)
        self.prop = torch.zeros((T, 8), dtype=torch.float32, device=dev)
        self.flags = torch.zeros(T + 1, dtype=torch.int32, device=dev)
        self.model = torch.zeros((T, 8), dtype=torch.float64, device=dev)
        self.params = torch.as_tensor(proposal.load_weights()).to(dev)
        torch.cuda.synchronize()
        base = dict(thr=0.05, max_radius=1.0, refit_iters=2, seed=SEED, tile_points=1024,
                    refit_rounds=3)
        plain = _lib.CylFitCfg(n_hyp=1024, stream_tag=0, hyp_chunk=128, **base)
        verify = _lib.CylFitCfg(n_hyp=16, stream_tag=1, hyp_chunk=16, **base)
        n = self.n.data_ptr()
        self.plain = self._make("sloam_cyl_plan_create_counted", T, self.points, n, C.byref(plain))
        self.verify = self._make("sloam_cyl_plan_create_counted", T, self.points, n,
                                 C.byref(verify))
        self.graph = None

    def _make(self, name, *args):
        h = C.c_void_p()
        _lib.check(getattr(self.lib, name)(self.ctx.handle, *args, C.byref(h)), self.ctx.handle)
        return h

    def _call(self, name, *args):
        _lib.check(getattr(self.lib, name)(*args), self.ctx.handle)

    def enqueue(self):
        o, h = self.fe.out, self.ctx.handle
        off, xyz, n, prop, flags, model, inp = (t.data_ptr() for t in (
            self.off, self.xyz, self.n, self.prop, self.flags, self.model, self.input))
        self._call("sloam_frontend_enqueue", self.fe.handle)
        self._call("sloam_kf_tree_points", h, C.byref(o), self.trees, self.points, off, xyz, n)
        self._call("sloam_pn_infer_counted", h, self.params.data_ptr(), xyz, off, self.trees, n,
                   prop)
        self._call("sloam_cyl_learned_exec", self.verify, self.plain, xyz, off, prop,
                   C.c_float(0.5), None, None, flags, flags + 4 * self.trees, None, model)
        i = _lib.KfInputs(n_cells=o.n_cells, num_features=self.fe.nf, tree_fits=model, pose=inp,
                          n_map=inp + 56, map=inp + 64,
                          **{k: getattr(o, k) for k in ("trellis_counts", "tree_offsets",
                                                        "vertex_int", "vertex_f64",
                                                        "point_offsets", "points", "cell_info",
                                                        "cell_model", "cell_features")})
        self._call("sloam_kf_estimator_exec", self.est, C.byref(i))

    def reset(self):
        self._call("sloam_kf_estimator_reset", self.est)

    def keyframe(self, frame):
        _copy(self.ctx, self.fe.out.xyzi, frame["xyzi"])
        _copy(self.ctx, self.fe.out.label, frame["label"])
        _copy(self.ctx, self.input.data_ptr(), frame["input"])
        if self.graph is None:
            self.enqueue()
            self.ctx.sync()
            self.ctx.graph_begin()
            self.enqueue()
            self.graph = self.ctx.graph_end()
        else:
            self.graph.launch()
        self.ctx.sync()
        r = _lib.KfResultView()
        self._call("sloam_kf_estimator_result", self.est, C.byref(r))

        def arr(ptr, n, ctype, room=None):
            a = np.zeros(room or n, ctype)
            if n:
                a[:n] = np.ctypeslib.as_array(C.cast(ptr, C.POINTER(ctype)), shape=(n,))
            return a

        head = arr(r.head, 20, C.c_int32)
        L, T = int(head[2]), self.trees
        return {"head": head, "pose": arr(r.pose, 7, C.c_double),
                "delta": arr(r.delta, 7, C.c_double), "tree": arr(r.lm_tree, L, C.c_int32, T),
                "id": arr(r.lm_id, L, C.c_int32, T), "match": arr(r.lm_match, L, C.c_int32, T),
                "model": arr(r.lm_model, 8 * L, C.c_double, 8 * T)}

    def __del__(self):
        try:
            if self.graph is not None:
                self.graph.close()
            for name, h in (("sloam_kf_estimator_destroy", self.est),
                            ("sloam_cyl_plan_destroy", self.plain),
                            ("sloam_cyl_plan_destroy", self.verify)):
                getattr(self.lib, name)(h)
            self.fe.close()
        except Exception:
            pass


def _prepare_keyframe(case, seed):
    ctx = _context(("keyframe", case["H"], case["W"]))
    rng = np.random.default_rng([seed, 9])
    frames = []
    for k in range(2):
        sc, forest, R, t = _scan(case, seed, k)
        q = synth.R_to_quat(R)
        inp = np.zeros(8 + 8 * _Keyframes.MAP)
        # the estimate: the true pose a few centimetres off; the map: the trunks in range, none
        # on the scan that opens it
        inp[:3] = t + (rng.normal(0, 0.03, 3) if k else 0.0)
        inp[3:7] = q
        near = [tr for tr in forest["trees"] if np.hypot(*(tr["base"][:2] - t[:2])) < 30.0] if k \
            else []
        inp[7:8].view(np.int32)[0] = len(near)
        for i, tr in enumerate(near):
            inp[8 + 8 * i:16 + 8 * i] = [*tr["base"], *tr["axis"], tr["radius"], 0.0]
        frames.append({"xyzi": torch.as_tensor(np.ascontiguousarray(sc["xyzi"])).pin_memory(),
                       "label": torch.as_tensor(np.ascontiguousarray(sc["label"])).pin_memory(),
                       "input": torch.as_tensor(inp).pin_memory()})
    kf = _Keyframes(ctx, case["H"], case["W"])
    s = dict(kf=kf, frames=frames, run=_run_keyframe)
    _run_keyframe(s)  # sizes the scratch and captures the graph, as a stream's first keyframe does
    return _ready(ctx, s)


def _run_keyframe(s):
    s["kf"].reset()
    return [s["kf"].keyframe(f) for f in s["frames"]]


# ---------------------------------------------------------------------------
# work and tolerance
# ---------------------------------------------------------------------------
def _points(case, count):
    return float(_sizes(case, count).sum())


def work(case):
    k = case["kind"]
    if k == "fit":
        S, n = case["clusters"], _points(case, case["clusters"])
        # points in; models, best hypotheses and the inlier bits out; 6 operations per point and
        # hypothesis, 60 per point and Gauss-Newton step
        return {"bytes": 12 * n + n / 8 + 72 * S, "flops": n * (6 * case["hyp"] + 360)}
    if k == "learned":
        S, n = case["clusters"], _points(case, case["clusters"])
        used = min(n, 512 * S)
        return {"bytes": 12 * n + 100 * S + 4 * 75399,
                "flops": 82304 * used + n * (6 * 16 + 360)}
    if k == "train":
        # points and targets in, weights and moments read and written; forward, and the backward
        # of the at most 256 points that the max-pool kept
        S = case["clusters"]
        used = min(_points(case, S), 512 * S)
        return {"bytes": 12 * used + 68 * S + 24 * 75399,
                "flops": 82304 * used + 2 * 82304 * min(256 * S, used)}
    if k == "pose":
        K = case["problems"]
        res = K * (case["cyl"] * case["pts_cyl"] + case["planes"] * case["pts_plane"])
        # the residuals and landmarks read once; ~90 operations per residual and evaluation (a
        # converging solve takes about 6)
        return {"bytes": 16 * res + 64 * K * case["cyl"] + 32 * K * case["planes"] + 200 * K,
                "flops": 90 * res * (case["iters"] + 1 if case["iters"] == 10 else 7)}
    if k == "plane":
        n = _points(case, case["sets"])
        return {"bytes": 12 * n + n / 8 + 72 * case["sets"], "flops": n * (7 * case["hyp"] + 30)}
    # scan and labels in; mask, ground list, dense tree cloud out (trees and cells are small)
    N = case["H"] * case["W"] * (2 if k == "keyframe" else 1)
    return {"bytes": N * (17 + 1 + 16 + 16 * 0.65), "flops": 100 * N}


def tolerance(case):
    k = case["kind"]
    if k == "fit":  # FP32 residuals with compensated sums: 2.2e-7 from an FP64 refit of the same winner
        return {"rel": 1e-6, "max": 1e-5}
    if k == "learned":
        # proposals are 2e-6 from 64 bits (an activation near a BF16 boundary rounds the other
        # way); a changed proposal can send a borderline cluster to the plain fit
        return {"rel": 1e-4, "max": 2e-2, "differ": 0.002}
    if k == "train":  # up to 6e-5 from 64 bits, by activations that round to the other BF16 value
        return {"rel": 3e-4, "max": 0.05}
    if k == "pose":  # 3e-7 from 64 bits in FP32, 3e-15 in FP64
        return {"rel": 1e-6, "max": 1e-3} if case["precision"] == 0 else {"rel": 1e-9, "max": 1e-6}
    if k == "keyframe":  # FP64 solves of features and planes that agree to 1e-12
        return {"rel": 1e-8, "max": 1e-6}
    # FP64 sums over the winner's inliers / a cell's points
    return {"rel": 1e-10, "max": 1e-7}


# ---------------------------------------------------------------------------
# exact: the paths in 64 bits
# ---------------------------------------------------------------------------
def exact(case, seed):
    return {"fit": _exact_fit, "learned": _exact_learned, "train": _exact_train,
            "pose": _exact_pose, "plane": _exact_plane, "frontend": _exact_frontend,
            "keyframe": lambda c, s: None}[case["kind"]](case, int(seed))


def _philox(h, c, tag):
    """Philox4x32-10 words of the counters (h, c, tag, 0) under the key SEED (Salmon et al., 2011)."""
    m = np.uint64(0xFFFFFFFF)
    h, c = np.meshgrid(np.arange(h, dtype=np.uint64), np.arange(c, dtype=np.uint64))
    x = [h, c, np.full_like(h, tag), np.zeros_like(h)]
    k0, k1 = np.uint64(SEED & 0xFFFFFFFF), np.uint64(SEED >> 32)
    for _ in range(10):
        p0, p1 = np.uint64(0xD2511F53) * x[0], np.uint64(0xCD9E8D57) * x[2]
        x = [(p1 >> np.uint64(32)) ^ x[1] ^ k0, p1 & m, (p0 >> np.uint64(32)) ^ x[3] ^ k1, p0 & m]
        k0, k1 = (k0 + np.uint64(0x9E3779B9)) & m, (k1 + np.uint64(0xBB67AE85)) & m
    return x


def _samples(sizes, hyp, tag):
    """Three distinct point indices per (set, hypothesis): int64 [sets, hyp, 3]."""
    x = _philox(hyp, len(sizes), tag)
    n = sizes.astype(np.uint64)[:, None]
    s32 = np.uint64(32)
    a = (x[0] * n) >> s32
    b = (x[1] * (n - np.uint64(1))) >> s32
    b = b + (b >= a)
    lo, hi = np.minimum(a, b), np.maximum(a, b)
    c = (x[2] * (n - np.uint64(2))) >> s32
    c = c + (c >= lo)
    c = c + (c >= hi)
    return torch.as_tensor(np.stack([a, b, c], -1).astype(np.int64)).cuda()


def _winner(count_of, offsets, hyp):
    """The hypothesis of the largest count, the first on ties: (index, count) per set."""
    o = offsets.long()
    best = torch.full((o.numel() - 1,), -1, dtype=torch.int64, device="cuda")
    count = torch.full_like(best, -1)
    for h in range(hyp):
        cum = torch.cat([torch.zeros(1, dtype=torch.int64, device="cuda"),
                         torch.cumsum(count_of(h).to(torch.int64), 0)])
        n = cum[o[1:]] - cum[o[:-1]]
        better = n > count
        best, count = torch.where(better, h, best), torch.where(better, n, count)
    return best, count


def _frames(d):
    o = d["offsets"].long()
    S = o.numel() - 1
    own = torch.repeat_interleave(torch.arange(S, device="cuda"), o[1:] - o[:-1])
    p = d["xyz"].double()
    lo = torch.full((S, 3), math.inf, dtype=torch.float64, device="cuda")
    hi = -lo.clone()
    lo = lo.scatter_reduce(0, own[:, None].expand(-1, 3), p, "amin")
    hi = hi.scatter_reduce(0, own[:, None].expand(-1, 3), p, "amax")
    mid = (0.5 * (lo + hi)).float().double()
    return o, S, own, mid, p - mid[own]


def _sums(own, S, terms):
    return torch.zeros((S,) + tuple(terms.shape[1:]), dtype=torch.float64,
                       device="cuda").index_add_(0, own, terms)


def _signed(v):
    lead = v.gather(1, v.abs().argmax(1, keepdim=True))
    return torch.where(lead < 0, -v, v)


def _covariance(own, S, n, x):
    mean = _sums(own, S, x) / n[:, None]
    y = x - mean[own]
    return mean, _sums(own, S, y[:, :, None] * y[:, None, :])


def _plane_basis(a):
    ref = torch.nn.functional.one_hot(a.abs().argmin(1), 3).double()
    e1 = ref - (ref * a).sum(1, keepdim=True) * a
    e1 = e1 / e1.norm(dim=1, keepdim=True)
    return e1, torch.linalg.cross(a, e1)


def _exact_fit(case, seed, thr=float(np.float32(0.05)), rounds=3, iters=2):
    d = _clusters(case, seed)
    if d["xyz"].shape[0] * case["hyp"] > 4e9:
        return None  # minutes of elementwise passes
    o, S, own, mid, x = _frames(d)
    n = (o[1:] - o[:-1]).double()
    _, cov = _covariance(own, S, n, x)
    a = _signed(torch.linalg.eigh(cov.cpu())[1][:, :, 2].cuda())
    e1, e2 = _plane_basis(a)
    u, v = (x * e1[own]).sum(1), (x * e2[own]).sum(1)
    smp = o[:-1, None, None] + _samples(np.diff(d["host"]).astype(np.int64), case["hyp"], 0)
    U, V = u[smp], v[smp]
    bx, by = U[..., 1] - U[..., 0], V[..., 1] - V[..., 0]
    cx, cy = U[..., 2] - U[..., 0], V[..., 2] - V[..., 0]
    det = 2 * (bx * cy - by * cx)
    b2, c2 = bx * bx + by * by, cx * cx + cy * cy
    ox, oy = (cy * b2 - by * c2) / det, (bx * c2 - cx * b2) / det
    r = (ox * ox + oy * oy).sqrt()
    cu, cv = U[..., 0] + ox, V[..., 0] + oy
    ok = r <= 1.0

    def inside(h):
        hh = h if torch.is_tensor(h) else torch.full((S,), h, device="cuda")
        pick = lambda t: t.gather(1, hh[:, None])[:, 0][own]  # noqa: E731
        return (((u - pick(cu)).square() + (v - pick(cv)).square()).sqrt() -
                pick(r)).abs().lt(thr) & pick(ok)

    best, count = _winner(inside, d["offsets"], case["hyp"])
    take = best.clamp_min(0)
    c = cu.gather(1, take[:, None]) * e1 + cv.gather(1, take[:, None]) * e2
    rad = r.gather(1, take[:, None])[:, 0]
    good = (count >= 3) & ok.gather(1, take[:, None])[:, 0]
    going = good.clone()
    member = inside(take)

    def residual():
        q = x - c[own]
        h = (q * a[own]).sum(1)
        w = q - h[:, None] * a[own]
        rho = w.norm(dim=1)
        return w, h, rho, rho - rad[own]

    for rnd in range(rounds):
        live = going.clone()
        for it in range(iters):
            f1, f2 = _plane_basis(a)
            w, h, rho, dd = residual()
            if rnd and not it:
                member = dd.abs() < thr
            nn = w / rho[:, None]
            n1, n2 = (nn * f1[own]).sum(1), (nn * f2[own]).sum(1)
            J = torch.stack([-h * n1, -h * n2, -n1, -n2, -torch.ones_like(h)], 1)
            J = torch.where(member[:, None], J, torch.zeros_like(J))
            A = _sums(own, S, J[:, :, None] * J[:, None, :])
            g = _sums(own, S, J * dd[:, None])
            cnt = _sums(own, S, member.double())
            enough = cnt >= 5
            going &= enough
            # a failed factorisation leaves the rest of the round out
            info = torch.linalg.cholesky_ex(A.cpu())[1].cuda()
            live &= going & (info == 0)
            A = torch.where(live[:, None, None], A, torch.eye(5, dtype=torch.float64,
                                                              device="cuda"))
            dl = torch.linalg.solve(A.cpu(), -g.cpu()).cuda()
            na = a + dl[:, :1] * f1 + dl[:, 1:2] * f2
            na = na / na.norm(dim=1, keepdim=True)
            upd = live[:, None]
            c = torch.where(upd, c + dl[:, 2:3] * f1 + dl[:, 3:4] * f2, c)
            a = torch.where(upd, na, a)
            rad = torch.where(live, rad + dl[:, 4], rad)
            going &= rad > 0
            live &= going
    _, _, _, dd = residual()
    fin = (dd.abs() < thr) & (rad > 0)[own]
    cnt = _sums(own, S, fin.double())
    mean = _sums(own, S, torch.where(fin[:, None], x, torch.zeros_like(x))) / cnt[:, None]
    root = mid + c + ((mean - c) * a).sum(1, keepdim=True) * a
    model = torch.cat([root, _signed(a), rad[:, None], cnt[:, None]], 1)
    none = torch.zeros_like(model)
    none[:, 5], none[:, 6] = 1.0, -1.0
    none[:, 7] = torch.where(good, cnt, count.double())
    valid = good & (rad > 0) & (cnt >= 3)
    return {"model": torch.where(valid[:, None], model, none), "mask": None, "best": None}


def _network(d, params, bf16):
    """The proposal network in 64 bits.  bf16: weights and activations rounded where the network
    defines them as BF16, with straight-through gradients."""
    def rounded(t):
        return t + (t.float().bfloat16().double() - t).detach() if bf16 else t

    o = d["offsets"].long()
    n = o[1:] - o[:-1]
    m = n.clamp_max(512)
    j = torch.arange(512, device="cuda")
    real = j[None, :] < m[:, None]
    idx = torch.where(real, o[:-1, None] + j[None, :] * n[:, None] // m[:, None], o[:-1, None])
    p = d["xyz"][idx].double()
    inf = torch.tensor(math.inf, dtype=torch.float64, device="cuda")
    lo = torch.where(real[..., None], p, inf).amin(1)
    hi = torch.where(real[..., None], p, -inf).amax(1)
    mid, half = 0.5 * (lo + hi), 0.5 * (hi - lo)
    sh = 1.0 / half[:, :2].amax(1).clamp_min(1e-3)
    scale = torch.stack([sh, sh, 1.0 / half[:, 2].clamp_min(1e-3)], 1)
    x = (p - mid[:, None]) * scale[:, None]
    # the points enter the first layer unrounded
    w = [(rounded(params[a:a + fi * fo]).view(fo, fi), rounded(params[b:b + fo]))
         for fi, fo, a, b in proposal.LAYERS]
    for W, b in w[:2]:
        x = rounded(torch.relu(x @ W.T + b))
    x = torch.relu(x @ w[2][0].T + w[2][1])
    f = torch.where(real[..., None], x, torch.zeros_like(x)).amax(1)
    h = torch.relu(f @ w[3][0].T + w[3][1])
    return h @ w[4][0].T + w[4][1], mid, scale, m


def _exact_learned(case, seed):
    d = _clusters(case, seed)
    params = torch.as_tensor(proposal.load_weights()).cuda().double()
    outs = []
    for k in range(0, case["clusters"], 256):
        part = dict(d, offsets=d["offsets"][k:k + 257])
        outs.append(_network(part, params, True))
    y, mid, scale, m = (torch.cat([o[i] for o in outs]) for i in range(4))
    v = y[:, :3] / scale
    c = mid + y[:, 3:6] / scale
    r = y[:, 6] / scale[:, 0]
    ok = (m >= 3) & (v.norm(dim=1) > 0) & (r > 0)
    up = torch.tensor([0.0, 0.0, 1.0], dtype=torch.float64, device="cuda")
    axis = torch.where(ok[:, None], v / v.norm(dim=1, keepdim=True), up)
    prop = torch.cat([axis, c, torch.where(ok, r, 0.0)[:, None], ok.double()[:, None]], 1)
    return {"model": None, "proposal": prop, "active": None, "n_fallback": None}


def _exact_train(case, seed):
    d = _clusters(case, seed)
    cfg = proposal.train_cfg()
    S = case["clusters"]
    params = torch.as_tensor(proposal.init_params(seed=seed % 1000)).cuda().double()
    params.requires_grad_(True)
    total = torch.zeros_like(params)
    losses = []
    for k in range(0, S, 128):
        part = dict(d, offsets=d["offsets"][k:k + 129])
        y, mid, scale, m = _network(part, params, True)
        tg = d["target"][k:k + 128]
        ax = tg[:, 3:6] * scale
        ax = ax / ax.norm(dim=1, keepdim=True)
        rt = (tg[:, :3] - mid) * scale
        cs = rt - (rt * ax).sum(1, keepdim=True) * ax
        ah = y[:, :3] / (y[:, :3].norm(dim=1, keepdim=True) + 1e-12)
        loss = (cfg.w_axis * (1 - (ah * ax).sum(1).square()) +
                cfg.w_centre * (y[:, 3:6] - cs).square().sum(1) +
                cfg.w_radius * (y[:, 6] - tg[:, 6] * scale[:, 0]).square())
        loss = torch.where(m >= 3, loss, torch.zeros_like(loss))
        total += torch.autograd.grad(loss.sum() / S, params)[0]
        losses.append(loss.detach())
    b1, b2 = cfg.beta1, cfg.beta2
    m1, m2 = (1 - b1) * total, (1 - b2) * total * total
    new = params.detach() - cfg.lr * (m1 / (1 - b1)) / ((m2 / (1 - b2)).sqrt() + cfg.eps)
    return {"loss": torch.cat(losses), "params": new, "m": m1, "v": m2}


def _aa_quat(w):
    th = w.norm(dim=1, keepdim=True)
    s = torch.where(th > 0, (th / 2).sin() / th.clamp_min(1e-300), torch.full_like(th, 0.5))
    return torch.cat([w * s, (th / 2).cos()], 1)


def _exact_pose(case, seed):
    """Levenberg-Marquardt as Ceres documents it (Huber loss 0.1, trust region 1e4, Jacobian
    scaling clamped to [1e-6, 1e32], function / gradient / parameter tolerances 1e-6 / 1e-10 /
    1e-8)."""
    d = _pose_problems(case, seed)
    K = len(d["res"]) - 1
    o = torch.as_tensor(d["res"]).cuda().long()
    own = torch.repeat_interleave(torch.arange(K, device="cuda"), o[1:] - o[:-1])
    p = d["points"][:, :3].double()
    lid = d["points"].view(torch.int32)[:, 3].long()
    tree = lid >= 0
    cyl, pl = d["cyl"][lid.clamp_min(0)], d["planes"][(-lid - 1).clamp_min(0)]
    free = torch.ones((K, 6), dtype=torch.float64, device="cuda")
    if d["mask"] is not None:
        free = ((d["mask"][:, None] >> torch.arange(6, device="cuda")) & 1).double()
    aa = case["two_step"]
    stop = case["iters"] == 50
    eye = torch.eye(3, dtype=torch.float64, device="cuda")

    def left_jacobian(w):
        t2 = w.square().sum(1)[:, None, None].clamp_min(1e-24)
        t = t2.sqrt()
        Kx = torch.linalg.cross(w[:, None].expand(-1, 3, 3), eye[None].expand(len(w), 3, 3), dim=2)
        Kx = Kx.transpose(1, 2)  # columns w x e_j: Kx v = w x v
        return eye + (1 - t.cos()) / t2 * Kx + (t - t.sin()) / (t2 * t) * (Kx @ Kx)

    def evaluate(t, q, w):
        rp = torch.einsum("nij,nj->ni", _rot(q)[own], p)
        lp = rp + t[own]
        vv = lp - cyl[:, :3]
        ray = cyl[:, 3:6] / cyl[:, 3:6].norm(dim=1, keepdim=True)
        ww = vv - (vv * ray).sum(1, keepdim=True) * ray
        rho = ww.norm(dim=1)
        sv = (pl[:, :3] * lp).sum(1) + pl[:, 3]
        r = torch.where(tree, rho - cyl[:, 6], sv.abs())
        dr = torch.where(tree[:, None], ww / rho[:, None], torch.where(sv < 0, -1.0, 1.0)[:, None] *
                         pl[:, :3])
        jt = torch.linalg.cross(rp, dr)
        if aa:
            jt = torch.einsum("ni,nij->nj", jt, left_jacobian(w)[own])
        J = torch.cat([dr, jt], 1) * free[own]
        ar = r.abs()
        wgt = torch.where(ar <= 0.1, torch.ones_like(r), 0.1 / ar)
        cost = torch.where(ar <= 0.1, r * r, 0.2 * ar - 0.01)
        return (_sums(own, K, wgt[:, None, None] * J[:, :, None] * J[:, None, :]).cpu().numpy(),
                _sums(own, K, (wgt * r)[:, None] * J).cpu().numpy(),
                _sums(own, K, 0.5 * cost).cpu().numpy())

    x0 = d["init"]
    t, q = x0[:, :3].clone(), x0[:, 3:].clone()
    sgn = torch.where(q[:, 3:] < 0, -1.0, 1.0)
    vec = q[:, :3] * sgn
    st = vec.norm(dim=1, keepdim=True).clamp_min(1e-300)
    w = vec / st * (2 * torch.atan2(st, q[:, 3:] * sgn))
    if aa:
        q = _aa_quat(w)
    A, g, F = evaluate(t, q, w)
    F0 = F.copy()
    radius, factor = np.full(K, 1e4), np.full(K, 2.0)
    done = np.zeros(K, bool)
    iters, term = np.zeros(K, int), np.ones(K, int)
    small = np.abs(g).max(1) <= 1e-10
    term[small] = 0
    done |= small & stop
    for _ in range(case["iters"]):
        dx = np.zeros((K, 6))
        model = np.zeros(K)
        for k in np.flatnonzero(~done):
            D = np.clip(np.diag(A[k]), 1e-6, 1e32) / radius[k]
            dx[k] = np.linalg.solve(A[k] + np.diag(D), -g[k])
            model[k] = -(g[k] @ dx[k] + 0.5 * dx[k] @ A[k] @ dx[k])
        step = torch.as_tensor(dx).cuda()
        t2 = t + step[:, :3]
        if aa:
            w2 = w + step[:, 3:]
            q2 = _aa_quat(w2)
            xn = torch.cat([t, w], 1).norm(dim=1).cpu().numpy()
        else:
            w2 = w
            q2 = _quat_mul(_aa_quat(step[:, 3:]), q)
            q2 = q2 / q2.norm(dim=1, keepdim=True)
            xn = torch.cat([t, q], 1).norm(dim=1).cpu().numpy()
        A2, g2, F2 = evaluate(t2, q2, w2)
        acc = np.zeros(K, bool)
        for k in np.flatnonzero(~done):
            iters[k] += 1
            gain = (F[k] - F2[k]) / model[k] if model[k] > 0 else -1.0
            flat = np.linalg.norm(dx[k]) <= 1e-8 * (xn[k] + 1e-8)
            if np.isfinite(F2[k]) and gain > 1e-3:
                acc[k] = True
                radius[k] = min(radius[k] / max(1 / 3, 1 - (2 * gain - 1) ** 3), 1e16)
                factor[k] = 2.0
                flat = flat or abs(F[k] - F2[k]) <= 1e-6 * F[k] or np.abs(g2[k]).max() <= 1e-10
                A[k], g[k], F[k] = A2[k], g2[k], F2[k]
            else:
                radius[k] /= factor[k]
                factor[k] *= 2
            if flat:
                term[k] = 0
                done[k] |= stop
        m = torch.as_tensor(acc).cuda()[:, None]
        t, q, w = torch.where(m, t2, t), torch.where(m, q2, q), torch.where(m, w2, w)
        if done.all():
            break
    params = torch.cat([t, w], 1) if aa else None  # the quaternion form's angles follow its pose
    return {"pose": torch.cat([t, q], 1), "params": params, "status": None,
            "cost": torch.as_tensor(np.stack([F0, F], 1))}


def _exact_plane(case, seed, thr=float(np.float32(0.05))):
    d = _plane_sets(case, seed)
    o, S, own, mid, x = _frames(d)
    smp = o[:-1, None, None] + _samples(np.diff(d["host"]).astype(np.int64), case["hyp"], 1)
    P = x[smp]
    nrm = torch.linalg.cross(P[:, :, 1] - P[:, :, 0], P[:, :, 2] - P[:, :, 0])
    size = nrm.norm(dim=2, keepdim=True)
    ok = size[..., 0] > 0
    nrm = nrm / size
    off = -(nrm * P[:, :, 0]).sum(2)

    def inside(h):
        hh = h if torch.is_tensor(h) else torch.full((S,), h, device="cuda")
        k = torch.arange(S, device="cuda")
        return ((x * nrm[k, hh][own]).sum(1) + off[k, hh][own]).abs().lt(thr) & ok[k, hh][own]

    best, _ = _winner(inside, d["offsets"], case["hyp"])
    m = inside(best.clamp_min(0))
    sel = own[m]
    cnt = _sums(sel, S, torch.ones(sel.numel(), dtype=torch.float64, device="cuda"))
    mean, cov = _covariance(sel, S, cnt, x[m])
    a = torch.linalg.eigh(cov.cpu())[1][:, :, 0].cuda()
    a = torch.where(a[:, 2:] < 0, -a, a)
    c = mid + mean
    dd = -(a * c).sum(1)
    fin = ((a[own] * d["xyz"].double()).sum(1) + dd[own]).abs() < thr
    model = torch.cat([a, dd[:, None], c, _sums(own, S, fin.double())[:, None]], 1)
    return {"model": model, "mask": None, "best": None}


def _exact_frontend(case, seed):
    """The ground cells: every beam of these scans owns its pixel, so the ground list is the
    labelled returns of at least one metre, in order."""
    sc, _, _, _ = _scan(case, seed)
    x = sc["xyzi"][:, :3]
    f = np.float32
    far = np.sqrt(x[:, 0] * x[:, 0] + x[:, 1] * x[:, 1] + x[:, 2] * x[:, 2]) >= f(1)
    p = x[(sc["label"] == 1) & far]
    dx, dy = p[:, 0].astype(float), p[:, 1].astype(float)
    r = np.sqrt((dx * dx).astype(f) + (dy * dy).astype(f)).astype(float)
    th = np.arctan2(p[:, 1], p[:, 0]).astype(float)
    pi = 3.14159265
    rb = np.clip(np.floor(r / (25.0 / 2)), 0, 1)
    tb = np.clip(np.floor((pi + th) / (2 * pi / 18)), 0, 17)
    cell = np.where((r < 25.0) & (r > 5.0), rb * 18 + tb, -1).astype(int)
    model = np.zeros((36, 8))
    for c in range(36):
        q = p[cell == c].astype(float)
        if 20.0 < len(q):
            q = q[np.argsort(q[:, 2], kind="stable")][:int(len(q) / (1.0 / 0.05))]
        if len(q) < 5:
            continue
        mu = q.mean(0)
        a = np.linalg.eigh((q - mu).T @ (q - mu))[1][:, 0]
        a = -a if a[2] < 0 else a
        model[c, :3], model[c, 3], model[c, 4:7] = a, -a @ mu, mu
    return {"cell_model": model}  # the rest are selections of the input's values
