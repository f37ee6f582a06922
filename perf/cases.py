"""What a user of this package has it do, as timed cases.

Each case is one pass through the public entry points (changa_amd.engine,
changa_amd.ltw, the request functions of libchanga_gpu.so), on the shapes of
changa_amd.configs: isolated Plummer spheres, isolated clustered halos, and
periodic Zel'dovich boxes with Ewald (optionally with an active rung).

Forms ("form" of a case):

  step      one force evaluation, one launch per list (Evaluation.step)
  batched   one force evaluation through an autotuned plan (step_batched)
  fused     one force evaluation that walks the tree in the force launch
            (step_fused; no interaction lists)
  adjoint   dL/dx, dL/dm of L = sum w . a on resident lists
  lists     moments and interaction lists rebuilt on a resident tree, then
            one force evaluation on them
  timestep  one force evaluation from host positions: a new tree, moments,
            then the fused walk and force
  request   the drop-in route: tree, lists and Ewald record in host memory,
            sent as ChaNGa sends them, results back in host memory
  ltw       one request of the GPU_LOCAL_TREE_WALK build
"""
import ctypes
import math

import numpy as np
import torch

from changa_amd import configs, engine, gpu, ltw

DEVICE = "cuda:0"


def _case(name, form, shape, n, bucket, theta, active=1.0):
    return dict(name=name, form=form, shape=shape, n=n, bucket=bucket, theta=theta, active=active)


def listed():
    return [
        # the smallest evaluation: a few thousand particles, where the launches of the moment
        # build and the host calls count
        _case("step_plummer_4k", "step", "plummer", 4096, 16, 0.7),
        # a small production evaluation of an isolated system
        _case("batched_plummer_64k", "batched", "plummer", 65536, 16, 0.7),
        # the flagship: 2^22 clustered particles, every particle a target
        _case("batched_halos_4m", "batched", "halos", 1 << 22, 32, 0.6),
        # a cosmological box near its start: near-uniform, periodic, with Ewald
        _case("batched_box_128", "batched", "box", 128 ** 3, 16, 0.7),
        # a multistep substep: 10% of a 256^3 box on the active rung
        _case("batched_rung_256", "batched", "box", 256 ** 3, 16, 0.7, 0.1),
        # one evaluation without resident lists (a time step whose tree changed)
        _case("fused_halos_256k", "fused", "halos", 1 << 18, 32, 0.6),
        # gradients through an evaluation: an isolated sphere, every particle a target
        _case("adjoint_plummer_1m", "adjoint", "plummer", 1 << 20, 16, 0.7),
        # gradients through a substep of the large box, Ewald terms included (the largest case)
        _case("adjoint_rung_256", "adjoint", "box", 256 ** 3, 16, 0.7, 0.1),
        # new lists and forces after the particles moved, on the same tree
        _case("lists_box_128", "lists", "box", 128 ** 3, 16, 0.7),
        # the evaluation of a time step: everything anew from host positions
        _case("timestep_box_128", "timestep", "box", 128 ** 3, 16, 0.7),
        # one TreePiece's gravity through the drop-in boundary, everything in host memory
        _case("request_box_64", "request", "box", 64 ** 3, 16, 0.7),
        # the drop-in boundary of the local-tree-walk build
        _case("ltw_halos_128k", "ltw", "halos", 1 << 17, 32, 0.6),
    ]


def draw(rng):
    form = rng.choice(["step", "batched", "batched", "fused", "adjoint", "lists", "timestep",
                       "request", "ltw"])
    shape = rng.choice(["plummer", "halos", "box"])
    most = {"step": 1 << 20, "batched": 1 << 21, "fused": 1 << 20, "adjoint": 1 << 20,
            "lists": 1 << 21, "timestep": 1 << 21, "request": 1 << 17, "ltw": 1 << 19}[form]
    n = int(math.exp(rng.uniform(math.log(4096), math.log(most))))
    active = 1.0
    if shape == "box":
        n = max(16, round(n ** (1.0 / 3.0))) ** 3
        if form in ("step", "batched", "fused", "adjoint") and rng.random() < 0.5:
            active = round(math.exp(rng.uniform(math.log(0.02), math.log(0.8))), 3)
    c = _case("", form, shape, n, rng.randint(8, 32), round(rng.uniform(0.55, 0.8), 2), active)
    del c["name"]
    return c


# ---------------------------------------------------------------------- inputs
def _box_positions(ng, rms, seed):
    """configs.zeldovich's displaced lattice, made on the device from the seed."""
    g = torch.Generator(device=DEVICE).manual_seed(seed)
    dk = torch.fft.rfftn(torch.randn((ng, ng, ng), generator=g, device=DEVICE,
                                     dtype=torch.float64))
    k = 2 * math.pi * torch.fft.fftfreq(ng, d=1.0 / ng, device=DEVICE, dtype=torch.float64)
    kr = 2 * math.pi * torch.fft.rfftfreq(ng, d=1.0 / ng, device=DEVICE, dtype=torch.float64)
    axes = (k[:, None, None], k[None, :, None], kr[None, None, :])
    k2 = axes[0] ** 2 + axes[1] ** 2 + axes[2] ** 2
    k2[0, 0, 0] = 1.0
    dk = dk * k2 ** (-2.5 / 4.0) / k2
    dk[0, 0, 0] = 0.0
    pos = torch.stack([torch.fft.irfftn(1j * a * dk, s=(ng, ng, ng)).reshape(-1) for a in axes],
                      dim=1)
    pos *= rms / pos.square().sum(dim=1).mean().sqrt()
    x = (torch.arange(ng, device=DEVICE, dtype=torch.float64) + 0.5) / ng
    pos += torch.stack(torch.meshgrid(x, x, x, indexing="ij"), dim=-1).reshape(-1, 3)
    pos -= torch.floor(pos)
    pos[pos >= 1.0] = 0.0
    return pos.cpu().numpy()


def _workload(case, seed):
    n, shape = case["n"], case["shape"]
    if shape == "plummer":
        w = configs.plummer(n=n, cfg=seed)
    elif shape == "halos":
        w = configs.halos(n=n, cfg=seed)
    else:
        ng = round(n ** (1.0 / 3.0))
        # the nearly uniform start, or, for a rung of a later step, a clustered box
        pos = _box_positions(ng, 0.02 if case["active"] == 1.0 else 0.15, seed)
        active = None
        if case["active"] < 1.0:
            active = np.zeros(n, dtype=bool)
            rung = np.random.default_rng(seed).permutation(n)[:max(1, round(case["active"] * n))]
            active[rung] = True
        w = dict(name=f"box_{ng}", pos=pos, mass=np.full(n, 1.0 / n),
                 soft=np.full(n, 1.0 / (20.0 * ng)), periodic=True, L=1.0, n_replicas=1,
                 ew_cut=2.6, ewh_cut=math.sqrt(10.0), active=active)
    w["theta"], w["bucket"] = case["theta"], case["bucket"]
    return w


class _Request:
    """One TreePiece's gravity through HostCUDA.h / EwaldCUDA.h: the local
    tree, four requests of cells and four of particles (one ILCell per source
    particle, as ChaNGa serializes them), Ewald, and the results back."""

    def __init__(self, w, parts=4):
        L = self.L = gpu.lib()
        ev = engine.Evaluation(w, precise=False, device=DEVICE, lists="gpu", tree="gpu")
        self.n = ev.n
        self.stream = torch.cuda.current_stream()
        self.moments = ev.d_moments.cpu().numpy()
        self.parts = ev.d_parts.cpu().numpy()
        self.zeros = np.zeros((self.n, 5), dtype=np.float32)
        self.out = torch.empty((self.n, 5), dtype=torch.float32, pin_memory=True)
        self.hip = ctypes.CDLL("libamdhip64.so")
        lists = ev.lists
        pcells, pmarks = engine.expand_parts(lists)
        self.requests = []
        for fn, lst, marks in ((L.TreePieceCellListDataTransferLocal, lists["cells"],
                                lists["cell_marks"]),
                               (L.TreePiecePartListDataTransferLocal, pcells, pmarks)):
            cuts = np.linspace(0, ev.tree["n_buckets"], parts + 1).astype(int)
            for b0, b1 in zip(cuts[:-1], cuts[1:]):
                m = marks[b0:b1 + 1].astype(np.int64)
                keep = (np.ascontiguousarray(lst.reshape(-1, 2)[m[0]:m[-1]]),
                        (m - m[0]).astype(np.int32),
                        np.ascontiguousarray(ev.tree["bucket_start"][b0:b1]),
                        np.ascontiguousarray(ev.tree["bucket_size"][b0:b1]))
                q = gpu.CudaRequest()
                q.stream = self.stream.cuda_stream
                q.list, q.bucketMarkers = keep[0].ctypes.data, keep[1].ctypes.data
                q.bucketStarts, q.bucketSizes = keep[2].ctypes.data, keep[3].ctypes.data
                q.numInteractions = int(m[-1] - m[0])
                q.numBucketsPlusOne = int(b1 - b0) + 1
                q.fperiod = ev.L
                self.requests.append((fn, q, keep))
        self.ewald = None
        if w["periodic"]:
            h = self.ewald = gpu.EwaldData()
            L.EwaldHostMemorySetup(ctypes.byref(h), self.n, len(ev.ewt64), 1)
            np.ctypeslib.as_array(h.EwaldMarkers, shape=(self.n,))[:] = np.arange(self.n)
            ewt = np.ascontiguousarray(ev.ewt64, dtype=np.float32)
            ctypes.memmove(h.ewt, ewt.ctypes.data, ewt.nbytes)
            ctypes.memmove(h.cachedData, ctypes.byref(ev.ewald_ro), ctypes.sizeof(ev.ewald_ro))
            h.EwaldRange[0], h.EwaldRange[1] = 0, self.n - 1

    def run(self):
        L, s = self.L, ctypes.c_void_p(self.stream.cuda_stream)
        dm, dp, dv = ctypes.c_void_p(), ctypes.c_void_p(), ctypes.c_void_p()
        L.DataManagerTransferLocalTree(self.moments.ctypes.data, self.moments.nbytes,
                                       self.parts.ctypes.data, self.parts.nbytes,
                                       self.zeros.ctypes.data, self.zeros.nbytes, ctypes.byref(dm),
                                       ctypes.byref(dp), ctypes.byref(dv), s, self.n, None)
        for fn, q, _ in self.requests:
            q.d_localMoments, q.d_localParts, q.d_localVars = dm, dp, dv
            fn(ctypes.byref(q))
        if self.ewald is not None:
            L.EwaldHost(dp, dv, ctypes.byref(self.ewald), s, None, 0, 1)
        L.TransferParticleVarsBack(self.out.data_ptr(), self.n * 20, dv, s, None)
        # the caller reads the host buffer, and gives the tree back, once the stream is through
        self.stream.synchronize()
        for p in (dm, dp, dv):
            self.hip.hipFree(p)
        return self.out

    def __del__(self):
        if getattr(self, "ewald", None) is not None:
            self.L.EwaldHostMemoryFree(ctypes.byref(self.ewald), 1)


def prepare(case, seed):
    w = _workload(case, seed)
    form = case["form"]
    if form == "timestep":
        return dict(form=form, w=w)
    if form == "request":
        return dict(form=form, request=_Request(w))
    ev = engine.Evaluation(w, precise=form != "ltw", device=DEVICE, tree="gpu",
                           lists="none" if form in ("fused", "ltw") else "gpu")
    s = dict(form=form, ev=ev)
    if form == "batched":
        ev.batch_plan()
    elif form == "fused":
        ev.fused_setup()
    elif form == "adjoint":
        g = torch.Generator(device=DEVICE).manual_seed(seed)
        s["w"] = torch.randn((ev.n_targets, 3), generator=g, device=DEVICE)
    elif form == "ltw":
        nodes, parts = ltw.serialize_evaluation(ev)
        del s["ev"]
        s["walk"] = ltw.LocalWalk(nodes, parts, w["theta"],
                                  int(w["n_replicas"]) if w["periodic"] else 0,
                                  w["L"] if w["periodic"] else 0.0, device=DEVICE)
    return s


# ---------------------------------------------------------------------- one pass
def _vars(v):
    return dict(acc=v[:, 0:3], pot=v[:, 3], dtgrav=v[:, 4])


def run(state):
    form = state["form"]
    if form == "timestep":
        ev = engine.Evaluation(state["w"], precise=True, device=DEVICE, tree="gpu", lists="none")
        ev.step_fused()
        # the results are in tree order: the order goes with them
        return dict(_vars(ev.d_vars), order=ev.tree["perm"])
    if form == "request":
        return _vars(state["request"].run())
    if form == "ltw":
        state["walk"].run()
        return _vars(state["walk"].d_vars)
    ev = state["ev"]
    if form == "adjoint":
        return ev.adjoint(state["w"])
    if form == "lists":
        ev.build_moments()
        ev.ewald_root()
        ev.build_lists()
        ev.step(moments=False)
    elif form == "step":
        ev.step()
    elif form == "batched":
        ev.step_batched()
    else:
        ev.step_fused()
    return _vars(ev.d_vars)


# ---------------------------------------------------------------------- work
def _per_target(case):
    """(cells, particles) a target interacts with: the counts of the host
    walk on these shapes, as straight lines in log2 n, with the opening angle
    (cells ~ theta^-3) and the bucket size (particles ~ bucket)."""
    lg, shape = math.log2(case["n"]), case["shape"]
    if shape == "plummer":
        pc, pp, th, b = 80.0 * (lg - 10.4), 650.0, 0.7, 16
    elif shape == "halos":
        pc, pp, th, b = 60.0 * (lg - 10.8), min(1250.0, 633.0 + 100.0 * (lg - 12.0)), 0.6, 32
    else:
        pc, pp, th, b = 25.0 * (lg - 6.0), 280.0, 0.7, 16
        if case["active"] < 1.0:
            pc, pp = 1.5 * pc, 1.3 * pp
    pp = min(pp * case["bucket"] / b, case["n"])
    return max(pc, 25.0) * (th / case["theta"]) ** 3 * (b / case["bucket"]) ** 0.5, pp


def work(case):
    form, n = case["form"], case["n"]
    periodic = case["shape"] == "box"
    nt = case["active"] * n
    pc, pp = _per_target(case)
    leaf = 0.7 * case["bucket"]  # mean bucket
    nodes = 2.0 * n / leaf
    buckets = min(n / leaf, nt)
    # a bucket has about its targets' cells and, per run, one source bucket
    lists = buckets * (8.0 * pc + 12.0 * pp / leaf)
    force = nt * (183.0 * pc + 23.0 * pp + ((74 * 333.0 + 146 * 58.0) if periodic else 0.0))
    moments = 500.0 * n + 2000.0 * nodes
    parts = n * 40.0 + nt * 64.0  # FP64 positions, mass, softening; the targets and results
    walk = buckets * 30.0 * (2.0 * pc + 2.0 * pp / leaf)  # about two tests per accepted entry
    if form == "timestep":
        return dict(bytes=n * 84.0 + nodes * 304.0, flops=force + moments + walk)
    if form == "lists":
        return dict(bytes=parts + nodes * 336.0 + lists, flops=force + moments + walk)
    if form == "adjoint":
        return dict(bytes=parts + nodes * 272.0 + lists + n * 32.0, flops=4.0 * force)
    if form == "request":
        return dict(bytes=n * 40.0 + nodes * 108.0 + buckets * 8.0 * (pc + pp), flops=force)
    if form == "ltw":
        return dict(bytes=n * 44.0 + nodes * 160.0, flops=force)
    if form == "fused":
        return dict(bytes=parts + nodes * 272.0, flops=force + moments + walk)
    return dict(bytes=parts + nodes * 272.0 + lists, flops=force + moments)


# ---------------------------------------------------------------------- 64 bits
def _kernels(r2, twoh):
    """Potential, force and force-gradient kernels (a, b, c = -(1/r) db/dr)
    of the Hernquist-Katz spline at squared distance r2 > 0, softening sum
    twoh; Newtonian outside."""
    ir = r2.rsqrt()
    a, b = ir, ir ** 3
    c = 3.0 * ir ** 5
    near = r2 < twoh * twoh
    if bool(near.any()):
        i, d = ir[near], 2.0 / twoh.expand_as(r2)[near]
        u = d / i
        u1 = u < 1.0
        sa = torch.where(
            u1, d * (7 / 5 + u ** 2 * (-2 / 3 + u ** 2 * (3 / 10 - u / 10))),
            -i / 15 + d * (8 / 5 + u ** 2 * (-4 / 3 + u * (1 + u * (-3 / 10 + u / 30)))))
        sb = torch.where(
            u1, d ** 3 * (4 / 3 + u ** 2 * (-6 / 5 + u / 2)),
            -i ** 3 / 15 + d ** 3 * (8 / 3 + u * (-3 + u * (6 / 5 - u / 6))))
        sc = torch.where(u1, d ** 5 * (12 / 5 - 3 / 2 * u),
                         -i ** 5 / 5 + d ** 5 * (3 / u - 12 / 5 + u / 2))
        a, b, c = a.clone(), b.clone(), c.clone()
        a[near], b[near], c[near] = sa, sb, sc
    return a, b, c


def _tree_order(pos):
    """Indices along the Morton curve the tree follows (21 bits per axis, x
    on top), over the cube of the particles' extent."""
    lo, hi = pos.min(axis=0), pos.max(axis=0)
    scale = float(1 << 21) / (float((hi - lo).max()) * (1 + 1e-12) + 1e-300)
    c = np.clip(np.floor((pos - lo) * scale).astype(np.int64), 0, (1 << 21) - 1)
    key = np.zeros(len(pos), dtype=np.int64)
    for bit in range(20, -1, -1):
        for k in range(3):
            key = (key << 1) | ((c[:, k] >> bit) & 1)
    return np.argsort(key, kind="stable")


def exact(case, seed):
    """Isolated systems: the direct sum over all pairs (its distance from a
    tree result is the tree's truncation) for at most 2^18 particles, 2^16
    for gradients. dtGrav depends on the cells used and has no value here."""
    form, n = case["form"], case["n"]
    if case["shape"] == "box" or n > (1 << 16 if form == "adjoint" else 1 << 18):
        return None
    w = _workload(case, seed)
    order = _tree_order(w["pos"])
    x, m, h = (torch.from_numpy(np.ascontiguousarray(w[k][order])).to(DEVICE)
               for k in ("pos", "mass", "soft"))
    step = max(1, (1 << 25) // n)
    if form == "adjoint":
        g = torch.Generator(device=DEVICE).manual_seed(seed)
        wt = torch.randn((n, 3), generator=g, device=DEVICE).double()
        grad = torch.zeros((n, 4), dtype=torch.float64, device=DEVICE)
    acc = torch.empty((n, 3), dtype=torch.float64, device=DEVICE)
    pot = torch.empty(n, dtype=torch.float64, device=DEVICE)
    for i in range(0, n, step):
        d = [x[None, :, k] - x[i:i + step, None, k] for k in range(3)]
        r2 = d[0] ** 2 + d[1] ** 2 + d[2] ** 2
        apart = (r2 > 0.0).double()
        a, b, c = _kernels(r2 + (1.0 - apart), h[i:i + step, None] + h[None, :])
        b = b * apart
        if form == "adjoint":
            t = wt[i:i + step]
            dw = d[0] * t[:, 0:1] + d[1] * t[:, 1:2] + d[2] * t[:, 2:3]
            grad[:, 3] += (b * dw).sum(dim=0)
            c = c * apart * dw
            for k in range(3):
                p = (b * t[:, k:k + 1] - c * d[k]) * m
                grad[:, k] += p.sum(dim=0)
                grad[i:i + step, k] -= p.sum(dim=1)
            continue
        b = b * m
        for k in range(3):
            acc[i:i + step, k] = (b * d[k]).sum(dim=1)
        pot[i:i + step] = -(a * apart * m).sum(dim=1)
    if form == "adjoint":
        return grad
    out = dict(acc=acc, pot=pot, dtgrav=None)
    return dict(out, order=order) if form == "timestep" else out
