"""The work a user of this package has it do, as cases that can be timed and compared.

A case is a dict of plain values.  Its "kind" says which public entry points one pass goes through:

  icd     one ICD iteration of a resident stage (Stage.icd_iteration: the HICD phases, offset solves,
          line selection, variance, convergence check), the loop every reconstruction spends its
          time in; the object, the offsets, the variance and the ratio come back.  NHICD is off
          (tb_options.no_nhicd, as in the package's parity tests): which lines NHICD visits is an
          order statistic of the updates, which a difference in the last bit decides otherwise, so
          whole iterations with it cannot be compared between two correct programs
  chunk   one of the ten chunks of an iteration, phase by phase (Stage.update_colour, the HICD phase
          of each colour and then the NHICD phase of each on lines selected beforehand from a given
          update map, Stage.offset_update after each): both kinds of phases in their real proportion
  batch   an ICD iteration of many small scans in lockstep (Batch.iteration)
  resid   the error sinogram of an object (Stage.init_error_sino, Stage.error_sino): the start of
          every stage
  fbp     the filtered back-projection start (Stage.init_fbp)
  cost    the MAP cost (Stage.cost), evaluated after every iteration by convergence runs
  unet    the learned start: the network's forward pass over a few frames (UNet.forward)
  train   one training step of that network up to its gradients (forward, loss, backward)

Scans are synthetic: drifting ellipses, closed-form line integrals, Poisson counts, and where the scan
has them zingers and ring offsets, with the models and parameters of timbir_amd.datagen's workloads.
The prior's c is 1, as in the package's smoke and trajectory tests: with the workloads' 1e-2 the first
iterations on a small scan amplify a difference in the last bit some hundred times, and the work is
the same.
"""
import math

import numpy as np
import torch

import timbir_amd as tb
from timbir_amd.devmem import DevArray, synchronize
from timbir_amd.learned import ARCH, SCALE, UNet, init_params

I0 = 1e4
HUBER_T, HUBER_DELTA = 4.0, 0.5
ALPHA, CHUNKS = 1.5, 10
RING_SIGMA, ZINGER_FRAC, ZINGER_GAIN = 0.01, 1e-3, 5.0


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def icd(n, rows, frames, views, K, rings, mult=1, kind="icd"):
    """A stage of a scan: n x n pixels, `rows` detector rows, `frames` time frames, `views` views in
    all (K interlaced sub-frames, 0: one sweep); rings: ring correction, the generalized-Huber data
    term and the variance update (the 4D scans), else the quadratic term.  mult: the stage's
    multiplier (1: the finest stage)."""
    return {"kind": kind, "n": n, "rows": rows, "frames": frames, "views": views, "K": K,
            "rings": rings, "mult": mult}


def listed():
    return [
        # the smallest scans: a single slab, where launches and latency count
        {"name": "icd_small_3d", **icd(64, 4, 1, 90, 0, False)},
        # an ordinary small 4D scan with a ragged width
        {"name": "icd_4d_100", **icd(100, 6, 5, 240, 8, True)},
        # the 256^2 interlaced 4D scan's finest stage
        {"name": "chunk_4d_256", **icd(256, 8, 16, 1024, 8, True, kind="chunk")},
        # a coarse stage of a larger 4D scan
        {"name": "icd_4d_384_coarse", **icd(384, 16, 8, 1024, 8, True, 2)},
        # the deployment scan's finest stage
        {"name": "chunk_deploy", **icd(512, 32, 16, 2048, 8, True, kind="chunk")},
        # a single-frame scan with many views
        {"name": "icd_single_frame", **icd(192, 8, 1, 1440, 0, True)},
        # several small single-frame scans at once
        {"name": "batch_small", "kind": "batch", "n": 128, "rows": 4, "views": 180, "count": 12},
        # a stage's start: the residual of an object
        {"name": "resid_384", "kind": "resid", "n": 384, "rows": 12, "frames": 6, "views": 720,
         "mult": 1},
        # a filtered back-projection start
        {"name": "fbp_512", "kind": "fbp", "n": 512, "rows": 16, "frames": 8, "views": 1024},
        # the cost evaluated while a run converges
        {"name": "cost_512", "kind": "cost", "n": 512, "rows": 16, "frames": 8, "views": 512},
        # the learned start of two frames
        {"name": "unet_2x16x256", "kind": "unet", "samples": 2, "d": 16, "h": 256, "w": 256},
        # training on the default batch of crops
        {"name": "train_4x8x128", "kind": "train", "samples": 4, "d": 8, "h": 128, "w": 128},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["icd", "icd", "icd", "icd", "icd", "coarse", "single", "batch", "resid",
                       "fbp", "cost", "unet", "train"])
    if kind == "icd":
        n, frames = _log_int(rng, 48, 420), _log_int(rng, 1, 16)
        per = rng.choice([8, 16, 24, 32, 48, 64, 72, 96, 128, 160])
        return icd(n, 2 * rng.randint(2, 10), frames, frames * per, 8, frames > 1,
                   kind="chunk" if n > 160 else rng.choice(["icd", "chunk"]))
    if kind == "coarse":
        mult = rng.choice([2, 4])
        n, frames = mult * _log_int(rng, 32, 128), rng.randint(2, 12)
        return icd(n, mult * rng.randint(2, 5), frames, frames * 8 * rng.randint(4, 18), 8, True,
                   mult)
    if kind == "single":
        return icd(_log_int(rng, 48, 200), 2 * rng.randint(2, 6), 1, 8 * rng.randint(20, 180), 0,
                   rng.random() < 0.5)
    if kind == "batch":
        return {"kind": "batch", "n": 4 * rng.randint(16, 40), "rows": 4,
                "views": 6 * rng.randint(20, 60), "count": rng.randint(3, 14)}
    if kind == "resid":
        mult = rng.choice([1, 1, 2])
        return {"kind": "resid", "n": 2 * _log_int(rng, 40, 250), "rows": 2 * rng.randint(2, 8),
                "frames": rng.randint(1, 8), "views": 8 * rng.randint(12, 90), "mult": mult}
    if kind in ("fbp", "cost"):
        return {"kind": kind, "n": _log_int(rng, 80, 500), "rows": rng.randint(4, 16),
                "frames": rng.randint(1, 8), "views": 8 * rng.randint(12, 100)}
    side = [4 * rng.randint(8, 64) for _ in range(2)] if kind == "unet" else \
        [4 * rng.randint(8, 32) for _ in range(2)]
    return {"kind": kind, "samples": rng.randint(1, 2 if kind == "unet" else 4),
            "d": 4 * rng.randint(1, 4 if kind == "unet" else 2), "h": side[0], "w": side[1]}


# ---------------------------------------------------------------------------
# scans
# ---------------------------------------------------------------------------
def _views(views, K):
    """Angles and times: one uniform sweep over [0, pi), or K interlaced sub-frames of it."""
    i = np.arange(views)
    if K == 0 or views % K:
        return (i * (np.pi / views)).astype(np.float32), i.astype(np.float32)
    bits = K.bit_length() - 1
    rev = np.array([int(format(s, "0%db" % bits)[::-1], 2) for s in range(K)])
    a = (i * K + rev[(i // (views // K)) % K]).astype(np.float32)
    return (a * np.float32(np.pi / views)).astype(np.float32), (a / np.float32(K)).astype(np.float32)


class _Phantom:
    """Seeded ellipses in a disk, drifting with time and differing from slice to slice."""

    def __init__(self, n, rows, seed):
        r = np.random.default_rng(seed)
        m, R = 12, 0.5 * n
        self.a, self.b = r.uniform(0.06, 0.3, m) * R, r.uniform(0.06, 0.3, m) * R
        self.x, self.y = r.uniform(-0.45, 0.45, m) * R, r.uniform(-0.45, 0.45, m) * R
        self.t, self.v = r.uniform(0, np.pi, m), r.uniform(0.2, 1.0, m)
        self.vx, self.vy = r.normal(0, 0.03 * R, m), r.normal(0, 0.03 * R, m)
        self.a[0] = self.b[0] = 0.92 * R
        self.x[0] = self.y[0] = self.vx[0] = self.vy[0] = 0.0
        self.v *= 2.5 / (0.8 * n)  # line integrals up to about 5
        ph = r.uniform(0, 2 * np.pi, m)
        z = (np.arange(rows) + 0.5) / rows
        self.z = 0.7 + 0.3 * np.cos(np.pi * z[:, None] + ph[None, :])  # [rows][m]
        self.z[:, 0] = 1.0
        self.n, self.rows = n, rows

    def lines(self, angles, tau):
        """[views][rows][n] line integrals; tau in [0, 1): each view's time."""
        dev, f = "cuda", torch.float32
        th = torch.tensor(angles, dtype=f, device=dev)[:, None]
        tt = torch.tensor(tau, dtype=f, device=dev)[:, None]
        c, s = torch.cos(th), torch.sin(th)
        u = torch.arange(self.n, dtype=f, device=dev)[None] + 0.5 - self.n / 2
        out = torch.zeros(len(angles), self.rows, self.n, device=dev)
        for k in range(len(self.a)):
            n1 = c * math.cos(self.t[k]) - s * math.sin(self.t[k])
            n2 = -c * math.sin(self.t[k]) - s * math.cos(self.t[k])
            s2 = (self.a[k] * n1) ** 2 + (self.b[k] * n2) ** 2
            x0, y0 = self.x[k] + self.vx[k] * tt, self.y[k] + self.vy[k] * tt
            d = u - (x0 * c - y0 * s)
            chord = (2 * self.a[k] * self.b[k] * self.v[k] / s2) * torch.sqrt(
                torch.clamp(s2 - d * d, min=0))
            zk = torch.tensor(self.z[:, k], dtype=f, device=dev)
            out += zk[None, :, None] * chord[:, None, :]
        return out

    def raster(self, frames, nx, rows):
        """[frames][rows][nx][nx], edges a few pixels soft: what a coarser stage hands on."""
        dev, f = "cuda", torch.float32
        h = self.n / nx
        u = (torch.arange(nx, dtype=f, device=dev) + 0.5) * h - self.n / 2
        X, Y = u[None, :], u[:, None]
        z = self.z.reshape(rows, -1, len(self.a)).mean(axis=1)
        out = torch.zeros(frames, rows, nx, nx, device=dev)
        for i in range(frames):
            tau = (i + 0.5) / frames
            for k in range(len(self.a)):
                x, y = X - (self.x[k] + self.vx[k] * tau), Y - (self.y[k] + self.vy[k] * tau)
                p = x * math.cos(self.t[k]) + y * math.sin(self.t[k])
                q = -x * math.sin(self.t[k]) + y * math.cos(self.t[k])
                rho = torch.sqrt((p / self.a[k]) ** 2 + (q / self.b[k]) ** 2)
                soft = torch.sigmoid((1 - rho) * (0.5 * (self.a[k] + self.b[k]) / (2.0 * h)))
                zk = torch.tensor(z[:, k] * self.v[k], dtype=f, device=dev)
                out[i] += zk[:, None, None] * soft
        return out


def _scan(case, seed):
    """(scan dict as reconstruct()'s arguments, phantom)."""
    n, rows, frames, views = case["n"], case["rows"], case.get("frames", 1), case["views"]
    ph = _Phantom(n, rows, seed)
    angles, times = _views(views, case.get("K", 8 if frames > 1 else 0))
    g = torch.Generator(device="cuda").manual_seed(int(seed) + 1)
    lam = I0 * torch.exp(-ph.lines(angles, times / views))
    counts = torch.clamp(torch.poisson(lam, generator=g), min=1)
    proj = -torch.log(counts / I0)
    rings = bool(case.get("rings", frames > 1))
    if rings:
        proj += RING_SIGMA * torch.randn(1, rows, n, generator=g, device="cuda")
        hit = torch.rand(proj.shape, generator=g, device="cuda") < ZINGER_FRAC
        proj = torch.where(hit, proj * ZINGER_GAIN, proj)
    scan = dict(projections=proj.cpu().numpy(), weights=counts.cpu().numpy(), proj_angles=angles,
                proj_times=times, recon_times=np.linspace(0, views, frames + 1).astype(np.float32),
                proj_rows=rows, proj_cols=n, proj_num=views, recon_num=frames, vox_wid=1.0,
                rot_center=n / 2, sig_s=0.02 if rings else 0.01, sig_t=5e-4 if rings else 1.0,
                c_s=1.0, c_t=1.0, convg_thresh=0.0, remove_rings=int(rings),
                quad_convex=0 if rings else 1, huber_delta=HUBER_DELTA, huber_T=HUBER_T)
    return scan, ph


def _stage_args(case):
    """A stage in the middle or at the end of a schedule: offsets and variance on where the scan
    has them."""
    m = case.get("mult", 1)
    return dict(mult_xy=m, mult_z=m, stage_idx=1, prev_mult_z=2 * m)


def _update_map(case, seed):
    """An update-magnitude map: largest at the object's edges, where NHICD goes."""
    m, n, rows = case["mult"], case["n"] // case["mult"], case["rows"] // case["mult"]
    x = _Phantom(case["n"], case["rows"], seed).raster(case["frames"], n, rows)
    p = torch.nn.functional.pad(x, (1, 1, 1, 1))
    g = (p[..., 2:, 1:-1] - p[..., :-2, 1:-1]).abs() + (p[..., 1:-1, 2:] - p[..., 1:-1, :-2]).abs()
    r = torch.Generator(device="cuda").manual_seed(int(seed) + 2)
    return (0.1 * g + 2e-4 * torch.rand(x.shape, generator=r, device="cuda")).cpu().numpy()


class _Memory:
    """Device memory of the library as torch sees it, with what owns it."""

    def __init__(self, owner, addr, shape, typestr="<f4"):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": typestr,
                                         "data": (int(addr), False), "version": 2}


def _tensor(owner, addr, shape):
    return torch.as_tensor(_Memory(owner, addr, shape), device="cuda")


def _stage(case, seed):
    tb.set_options(verbose=0, write_files=0, no_nhicd=1)
    scan, ph = _scan(case, seed)
    st = tb.Stage(scan, **_stage_args(case))
    f, nz, _, nx = st.obj_shape
    st.set_object(ph.raster(f, nx, nz).cpu().numpy())
    return st, _tensor(st, st.object_device()[0], st.obj_shape)


def _crop_volume(case, seed):
    """Back-projection-like volumes (a soft phantom plus noise), their mean and the clean target,
    attenuation per pixel as the network meets it."""
    s, d, h, w = case["samples"], case["d"], case["h"], case["w"]
    side = max(h, w)
    ph = _Phantom(side, d, seed)
    t = ph.raster(s, side, d)[:, :, :h, :w] * (0.015 / (2.5 / (0.8 * side)))
    g = torch.Generator(device="cuda").manual_seed(int(seed) + 1)
    x = t + 0.003 * torch.randn(t.shape, generator=g, device="cuda")
    return x.contiguous(), x.mean(0).contiguous(), t.contiguous()


def _params(seed):
    """Weights of the network: He-normal as at the start of training, a head and biases that are
    not zero."""
    p = init_params(1234 + int(seed) % 7)
    r = np.random.default_rng(77)
    out = {}
    for k, (w, b) in p.items():
        b = r.normal(0, 0.02, b.shape).astype(np.float32)
        out[k] = ((r.normal(0, 0.1, w.shape).astype(np.float32) if k == "head" else w), b)
    return out


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("icd", "chunk", "resid", "fbp", "cost"):
        st, obj = _stage(case, seed)
        if kind in ("icd", "chunk", "cost"):
            st.init_error_sino()
        if kind == "chunk":
            st.set_magmap(_update_map(case, seed))
            st.vsc_select()
        return {"kind": kind, "st": st, "obj": obj, "it": 0, "rings": case.get("rings", False)}
    if kind == "batch":
        sts, objs = [], []
        for k in range(case["count"]):
            n = case["n"] + (64 if k % 3 == 2 else 0)
            st, obj = _stage({**case, "n": n, "frames": 1}, seed * 100 + k)
            st.init_error_sino()
            sts.append(st)
            objs.append(obj)
        return {"kind": kind, "b": tb.Batch(), "sts": sts, "objs": objs, "it": 0}
    x, mean, target = _crop_volume(case, seed)
    net = UNet(params=_params(seed))
    shape = tuple(x.shape)
    out = DevArray(shape, "f32")
    state = {"kind": kind, "net": net, "x": DevArray.from_numpy(x.cpu().numpy()),
             "mean": DevArray.from_numpy(mean.cpu().numpy()), "dev": out,
             "out": _tensor(out, out.addr, shape)}
    if kind == "train":
        state["target"] = DevArray.from_numpy(target.cpu().numpy())
        state["grads"] = {"%s.%s" % k: _tensor(v, v.addr, v.shape) for k, v in net.grad.items()}
    synchronize()
    return state


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(state):
    kind = state["kind"]
    if kind == "icd":
        state["it"] += 1
        st = state["st"]
        _, ratio = st.icd_iteration(state["it"])
        return {"object": state["obj"], "offset": st.offset(), "var": st.var_est, "ratio": ratio}
    if kind == "chunk":
        it, st = state["it"], state["st"]
        state["it"] += 1
        for nhicd in (0, 1):
            for colour in (0, 1):
                st.update_colour(colour, 2 + it // CHUNKS, it % CHUNKS, nhicd)
                if state["rings"]:
                    st.offset_update(1)
        return {"object": state["obj"], "offset": st.offset()}
    if kind == "batch":
        state["it"] += 1
        _, ratio = state["b"].iteration(state["sts"], state["it"])
        return {"objects": list(state["objs"]), "ratio": ratio}
    if kind == "resid":
        state["st"].init_error_sino()
        return state["st"].error_sino()
    if kind == "fbp":
        state["st"].init_fbp()
        return state["obj"]
    if kind == "cost":
        return state["st"].cost()
    net = state["net"]
    if kind == "unet":
        net.forward(state["x"], state["mean"], out=state["dev"])
        return state["out"]
    net.forward(state["x"], state["mean"], keep=True, out=state["dev"])
    loss, g = net.loss_and_grad(state["dev"], state["target"])
    net.backward(g)
    return {"loss": loss, "out": state["out"], "grads": state["grads"]}


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _mean_bins(m):
    """Nonzero bins of a pixel's column in a view, averaged over angles."""
    return 4 / math.pi * m + 1


def work(case):
    kind = case["kind"]
    if kind in ("unet", "train"):
        vox = case["samples"] * case["d"] * case["h"] * case["w"]
        lv = {"x": 1, "e1a": 1, "e1": 1, "e2a": 8, "e2": 8, "b1": 64, "b2": 64, "d2a": 8, "d2": 8,
              "d1a": 1, "d1": 1}
        flops = sum(2 * 27 * ci * co * vox / lv[name] for name, _, ci, co in ARCH)
        par = sum(27 * ci * co for _, _, ci, co in ARCH)
        if kind == "unet":
            return {"bytes": 4 * (2 * vox + vox / case["samples"]) + 2 * par, "flops": flops}
        return {"bytes": 4 * (3 * vox + par) + 2 * par, "flops": 3 * flops}
    m = case.get("mult", 1)
    n = case["n"] // m
    frames, views = case.get("frames", 1), case["views"]
    nobj, nsino = frames * case["rows"] // m * n * n, views * case["rows"] * case["n"]
    pix = math.pi / 4 * n * n * frames * (case["rows"] // m)
    ent = views / frames * _mean_bins(m) * m
    if kind in ("icd", "chunk", "batch"):
        k = case.get("count", 1)
        upd = pix if kind != "chunk" else pix / 5  # a chunk visits a tenth of the voxels twice
        return {"bytes": k * 4.0 * (3 * nsino + 4 * nobj), "flops": k * upd * (8 * ent + 28 * 12)}
    if kind == "resid":
        return {"bytes": 4.0 * (2 * nsino + nobj), "flops": 2 * pix * views / frames * _mean_bins(m)}
    if kind == "fbp":
        return {"bytes": 4.0 * (nsino + nobj), "flops": 4 * pix * views / frames + nsino * case["n"]}
    return {"bytes": 4.0 * (2 * nsino + nobj), "flops": 6 * nsino + 14 * 12.0 * nobj}


# ---------------------------------------------------------------------------
# the same values in 64 bits
# ---------------------------------------------------------------------------
class _Model:
    """A stage's geometry and model (XT_Init.c:211-669, XT_Profile.c:47-218, XT_AMatrix.c:50-110)."""

    def __init__(self, scan, m):
        self.n, self.m, self.rows = scan["proj_cols"], m, scan["proj_rows"]
        self.nx, self.nz = self.n // m, self.rows // m
        n, d = self.n, float(m)
        self.frames = scan["recon_num"]
        th = scan["proj_angles"].astype(np.float64)
        self.cos, self.sin = np.cos(th), np.sin(th)
        t, rt = scan["proj_times"], scan["recon_times"]
        self.views = [np.nonzero((t >= rt[i]) & (t < rt[i + 1]))[0] for i in range(self.frames)]
        self.R0 = -float(scan["rot_center"])
        self.off = (d / math.sqrt(2.0) + 0.5) / 64
        self.pos = self.R0 + (np.arange(self.nx) + 0.5) * d
        yy, xx = np.meshgrid(self.pos, self.pos, indexing="ij")
        self.mask = xx * xx + yy * yy < (n / 2) ** 2
        self.H = self._response(th, d)
        per = sum(len(v) for v in self.views) / self.frames
        self.sS, self.sT = float(np.float32(scan["sig_s"])) * m, float(np.float32(scan["sig_t"])) * per
        self.cS, self.cT = float(np.float32(scan["c_s"])), float(np.float32(scan["c_t"]))
        w = np.zeros((3, 3, 3))
        for i in range(27):
            q = (i // 9 - 1) ** 2 + (i // 3 % 3 - 1) ** 2 + (i % 3 - 1) ** 2
            w[i // 9, i // 3 % 3, i % 3] = 1 / math.sqrt(q) if q else 0.0
        k = m ** 3 * per / (w.sum() + 2)
        self.g, self.gt = w * k, k
        quad = scan["quad_convex"] == 1
        self.T, self.delta = (100000.0, 1.0) if quad else (scan["huber_T"], scan["huber_delta"])

    def _response(self, th, d):
        beam = 0.54 - 0.46 * np.cos(2 * np.pi / 512 * np.arange(512))
        beam /= beam.sum()
        r = -0.5 + np.arange(512) / 512
        H = np.zeros((len(th), 65))
        j2 = 2.0 * np.arange(1536) / 1536
        for k, a in enumerate(th):
            a = a % (np.pi / 2)
            peak = d / math.cos(a if a <= np.pi / 4 else np.pi / 2 - a)
            d1 = math.cos(np.pi / 4) * math.cos(np.pi / 4 - a)
            d2 = math.cos(np.pi / 4) * abs(math.cos(np.pi / 4 + a))
            up = (j2 - (1 - d1)) / max(d1 - d2, 1e-300)
            down = ((1 + d1) - j2) / max(d1 - d2, 1e-300)
            prof = np.where((j2 <= 1 - d1) | (j2 >= 1 + d1), 0.0, peak * np.clip(np.minimum(up, down), 0, 1))
            prof = prof.astype(np.float32).astype(np.float64)
            idx = np.floor((r[None, :] - (np.arange(64) * self.off - d)[:, None]) * (1536 / (2 * d))).astype(int)
            ok = (idx >= 0) & (idx < 1536)
            H[k, :64] = ((prof[np.clip(idx, 0, 1535)] * ok) @ beam).astype(np.float32)
        return H

    def columns(self, v, pix):
        """Window start and the 2 m + 1 A values of pixels `pix` in views `v`: [pixels][views](, bins)."""
        r = self.pos[pix % self.nx][:, None] * self.cos[v] - self.pos[pix // self.nx][:, None] * self.sin[v]
        lo = np.floor(r - self.m - self.R0).astype(int)
        j = lo[..., None] + np.arange(2 * self.m + 1)
        q = np.abs(r[..., None] - (self.R0 + j + 0.5)) / self.off
        b = np.minimum(q.astype(int), 64)
        h = self.H[v][None, :, :]
        h = np.broadcast_to(h, (len(pix),) + h.shape[1:])
        h0 = np.take_along_axis(h, np.minimum(b, 64), 2)
        h1 = np.take_along_axis(h, np.minimum(b + 1, 64), 2)
        a = np.where((b < 64) & (j >= 0) & (j < self.n), h0 + (q - b) * (h1 - h0), 0.0)
        return np.clip(j, 0, self.n - 1), a

    def project(self, obj):
        """A x: [views][slices][bins] of obj [frames][slices][nx][nx], float64."""
        out = torch.zeros(len(self.cos), self.nz, self.n, dtype=torch.float64, device="cuda")
        x = torch.as_tensor(obj, dtype=torch.float64, device="cuda").reshape(self.frames, self.nz, -1)
        pos = torch.as_tensor(self.pos, device="cuda")
        H = torch.as_tensor(self.H, device="cuda")
        for f, vs in enumerate(self.views):
            for v in vs:
                r = (pos[None, :] * self.cos[v] - pos[:, None] * self.sin[v]).reshape(-1)
                lo = torch.floor(r - self.m - self.R0)
                for k in range(2 * self.m + 1):
                    j = (lo + k).long()
                    q = torch.abs(r - (self.R0 + j + 0.5)) / self.off
                    b = torch.clamp(q.long(), max=63)
                    a = H[v][b] + (q - b) * (H[v][b + 1] - H[v][b])
                    a = torch.where((q < 64) & (j >= 0) & (j < self.n), a, torch.zeros_like(a))
                    out[v].index_add_(1, torch.clamp(j, 0, self.n - 1), x[f] * a)
        return out

    def rho(self, d, sig, c):
        a = d.abs()
        return (a * a / sig ** 2) / (c + a ** 0.8 / sig ** 0.8)


def _mix(x):
    x = np.asarray(x, np.uint64) & np.uint64(0xFFFFFFFF)
    m = np.uint64(0xFFFFFFFF)
    x ^= x >> np.uint64(16)
    x = (x * np.uint64(0x7FEB352D)) & m
    x ^= x >> np.uint64(15)
    x = (x * np.uint64(0x846CA68B)) & m
    return x ^ (x >> np.uint64(16))


def _order(N, it, f, z):
    """The keyed Feistel permutation of a cell's pixels in an iteration."""
    k = _mix(0x5BD1E995 ^ ((it * 0x9E3779B1) & 0xFFFFFFFF))
    k = _mix(int(k) ^ ((f * 0x85EBCA77) & 0xFFFFFFFF))
    key = int(_mix(int(k) ^ ((z * 0xC2B2AE3D) & 0xFFFFFFFF)))
    bits = 1
    while (1 << bits) < N:
        bits += 1
    h = (bits + 1) // 2
    msk = np.uint64((1 << h) - 1)
    n = np.arange(N, dtype=np.uint64)
    todo = np.ones(N, bool)
    while todo.any():
        L, R = n[todo] >> np.uint64(h), n[todo] & msk
        for r in range(4):
            L, R = R, L ^ (_mix(R ^ np.uint64((key + r * 0x9E3779B9) & 0xFFFFFFFF)) & msk)
        n[todo] = (L << np.uint64(h)) | R
        todo = n >= N
    return n.astype(np.int64)


class _Icd:
    """ICD iterations (XT_ICD_update.c:936-1105) in 64 bits: the cells of a colour side by side, the
    voxels of a cell one after another."""

    def __init__(self, scan, m, x0):
        M = self.M = _Model(scan, m)
        F, Z, n = M.frames, M.nz, M.nx
        self.x = np.full((F + 2, Z + 2, n + 2, n + 2), np.nan)
        self.x[1:-1, 1:-1, 1:-1, 1:-1] = x0
        self.mag = np.zeros((F, Z, n * n))
        y = scan["projections"].astype(np.float64)  # [views][rows][bins]
        self.e = y - np.repeat(M.project(x0).cpu().numpy(), m, axis=1)
        self.w = scan["weights"].astype(np.float64)
        self.d = np.zeros((M.n, M.rows))
        self.var = 1.0
        self.offsets = scan["remove_rings"] > 0
        self.use_var = scan["quad_convex"] == 0
        nv = max(len(v) for v in M.views)
        self.vi = np.zeros((F, nv), int)
        self.j, self.a = [], []
        for f, v in enumerate(M.views):
            self.vi[f, :len(v)] = v
            j, a = M.columns(v, np.arange(n * n))
            self.j.append(np.pad(j, ((0, 0), (0, nv - len(v)), (0, 0))))
            self.a.append(np.pad(a, ((0, 0), (0, nv - len(v)), (0, 0))))
        self.j, self.a = np.stack(self.j), np.stack(self.a)
        self.lines = {}

    def sweep(self, cells, lists, it, count):
        M, n, m = self.M, self.M.nx, self.M.m
        f, z = cells[:, 0], cells[:, 1]
        lens = np.array([len(q) for q in lists])
        if not len(lens) or not lens.max():
            return 0.0
        pad = np.full((len(lists), lens.max()), -1)
        for c, q in enumerate(lists):
            pad[c, :len(q)] = q
        dz, dy, dx = [q.ravel() for q in np.meshgrid([-1, 0, 1], [-1, 0, 1], [-1, 0, 1], indexing="ij")]
        g = np.concatenate([M.g.ravel(), [M.gt, M.gt]])
        s2 = np.r_[np.full(27, M.sS ** 2), [M.sT ** 2] * 2]
        sp = np.r_[np.full(27, M.sS ** 0.8), [M.sT ** 0.8] * 2]
        cc = np.r_[np.full(27, M.cS), [M.cT] * 2]
        mag = 0.0
        for s in range(pad.shape[1]):
            on = np.nonzero(pad[:, s] >= 0)[0]
            p, ff, zz = pad[on, s], f[on], z[on]
            py, px = p // n, p % n
            nb = np.concatenate([
                self.x[ff[:, None] + 1, zz[:, None] + 1 + dz, py[:, None] + 1 + dy, px[:, None] + 1 + dx],
                self.x[ff[:, None] + np.array([0, 2]), zz[:, None] + 1, py[:, None] + 1, px[:, None] + 1]], 1)
            V = nb[:, 13].copy()
            nb[:, 13] = np.nan
            ok = np.isfinite(nb)
            skip = (V == 0) & (it > 1) & ~np.any(nb > 0, axis=1)
            dl = np.where(ok, V[:, None] - nb, 0.0)
            t1 = np.abs(dl) ** 0.8 / sp
            b = np.where(ok, g, 0.0) * (2 - 0.8 * t1 / (cc + t1)) / ((cc + t1) * s2)
            A = self.a[ff, p][:, :, None, :]
            at = (self.vi[ff][:, :, None, None], (zz[:, None] * m + np.arange(m))[:, None, :, None],
                  self.j[ff, p][:, :, None, :])
            e, w = self.e[at], self.w[at]
            with np.errstate(divide="ignore", invalid="ignore"):
                cw = np.where(np.abs(e) * np.sqrt(w) < M.T, w, M.T * M.delta * np.sqrt(w) / np.abs(e))
            th1, th2 = -(A * e * cw).sum((1, 2, 3)), (A * A * cw).sum((1, 2, 3))
            step = ALPHA * (-(b * dl).sum(1) - th1) / (b.sum(1) + th2)
            step = np.where(skip, 0.0, step)
            self.x[ff + 1, zz + 1, py + 1, px + 1] = V + step
            self.mag[ff, zz, p] = np.abs(step)
            # bins off the detector hold a zero A value and the index of an edge bin: add, not set
            np.subtract.at(self.e, tuple(np.broadcast_arrays(*at)), A * step[:, None, None, None])
            if count:
                mag += np.abs(V + step)[~skip].sum()
        return mag

    def offset(self):
        if not self.offsets:
            return
        M = self.M
        sw = np.sqrt(self.w)
        b = np.abs(self.e) * sw < M.T
        td = M.T * M.delta
        with np.errstate(divide="ignore"):
            den = np.where(b, self.w, td * sw / np.abs(self.e)).sum(0)
        num = np.where(b, self.e * self.w, td * sw * np.sign(self.e)).sum(0)
        self.d += (num / den).T
        self.e -= num / den

    def select(self):
        M, n = self.M, self.M.nx
        tap = np.array([[0.0064, 0.0432, 0.08, 0.0432, 0.0064], [0.0432, 0.2916, 0.54, 0.2916, 0.0432],
                        [0.08, 0.54, 1.0, 0.54, 0.08], [0.0432, 0.2916, 0.54, 0.2916, 0.0432],
                        [0.0064, 0.0432, 0.08, 0.0432, 0.0064]])
        want = int(M.mask.sum()) // CHUNKS
        for f in range(M.frames):
            for z in range(M.nz):
                q = np.pad(self.mag[f, z].reshape(n, n), 2)
                v = sum(tap[a, c] * q[a:a + n, c:c + n] for a in range(5) for c in range(5)).ravel()
                v = v.astype(np.float32)
                thr = np.partition(v, n * n - want - 1)[n * n - want - 1]
                sel = np.nonzero(v > thr)[0][:max(want, 1)]
                inside = M.mask.ravel()[sel]
                self.mag[f, z][sel[~inside]] = 0.0
                self.lines[f, z] = sel[inside]

    def chunk(self, it, j, nhicd):
        M = self.M
        N = M.nx ** 2
        per, msk = N // CHUNKS, M.mask.ravel()
        cells = [(f, z) for f in range(M.frames) for z in range(M.nz)]
        col = [np.array([k for k in cells if sum(k) % 2 == c]).reshape(-1, 2) for c in (0, 1)]
        mag = 0.0
        end = N if j == CHUNKS - 1 else (j + 1) * per
        for c in (0, 1):
            lists = [_order(N, it, f, z)[j * per:end] for f, z in col[c]]
            mag += self.sweep(col[c], [q[msk[q]] for q in lists], it, True)
            self.offset()
        for c in (0, 1) if nhicd else ():
            self.sweep(col[c], [self.lines[tuple(k)] for k in col[c]], it, False)
            self.offset()
        return mag

    def iteration(self, it):
        M = self.M
        msk = M.mask.ravel()
        for j in range(CHUNKS):
            mag = self.chunk(it, j, False)
        if self.use_var:
            raw, sw = self.w * self.var, np.sqrt(self.w)
            b = np.abs(self.e) * sw < M.T
            new = np.where(b, self.e ** 2 * raw,
                           np.abs(self.e) * M.T * M.delta * np.sqrt(raw * self.var)).mean()
            self.w, self.var = raw / new, new
        return 100 * (self.mag * msk).sum() / mag


def _exact_icd(case, seed):
    chunk = case["kind"] == "chunk"
    m, F = case["mult"], case["frames"]
    n, rows = case["n"] // m, case["rows"] // m
    steps = (0.4 if chunk else 2.0) * math.pi / 4 * n * n  # voxels one after another
    entries = F * rows / 2 * case["views"] / F * (2 * m + 1) * m  # of one voxel of each cell
    if steps * (3e-4 + 6e-8 * entries) > 15 or case["views"] / F * n * n * F > 4e7:
        return None
    scan, ph = _scan(case, seed)
    s = _Icd(scan, m, ph.raster(F, n, rows).cpu().numpy().astype(np.float64))
    if chunk:
        s.mag = _update_map(case, seed).astype(np.float64).reshape(F, rows, n * n)
        s.select()
        s.chunk(2, 0, True)
        return {"object": s.x[1:-1, 1:-1, 1:-1, 1:-1].copy(), "offset": s.d}
    ratio = s.iteration(1)
    return {"object": s.x[1:-1, 1:-1, 1:-1, 1:-1].copy(), "offset": s.d, "var": s.var, "ratio": ratio}


def _exact_fbp(scan, M):
    n = M.n
    p = torch.as_tensor(scan["projections"], dtype=torch.float64, device="cuda")
    k = torch.arange(n, device="cuda", dtype=torch.float64)
    dk = k[:, None] - k[None, :]
    ramp = torch.where(dk.abs() % 2 == 1, -1 / (math.pi * dk.abs().clamp(min=1)) ** 2, torch.zeros_like(dk))
    ramp += 0.25 * torch.eye(n, device="cuda", dtype=torch.float64)
    q = p @ ramp.T  # [views][rows][bins]
    pos = torch.as_tensor(M.pos, device="cuda")
    out = torch.zeros(M.frames, M.rows, n * n, dtype=torch.float64, device="cuda")
    for f, vs in enumerate(M.views):
        for v in vs:
            u = (pos[None, :] * M.cos[v] - pos[:, None] * M.sin[v]).reshape(-1) - M.R0 - 0.5
            j = torch.floor(u)
            t, j = u - j, j.long()
            qp = torch.nn.functional.pad(q[v], (1, 1))
            a, b = qp[:, (j + 1).clamp(0, n + 1)], qp[:, (j + 2).clamp(0, n + 1)]
            out[f] += (1 - t) * a + t * b
        out[f] *= math.pi / max(len(vs), 1)
    out *= torch.as_tensor(M.mask.ravel().astype(np.float64), device="cuda")
    return out.reshape(M.frames, M.rows, n, n)


def _exact_cost(scan, M, obj):
    e = torch.as_tensor(scan["projections"], dtype=torch.float64, device="cuda") - M.project(obj)
    u = e.abs() * torch.sqrt(torch.as_tensor(scan["weights"], dtype=torch.float64, device="cuda"))
    fwd = torch.where(u < M.T, u * u, 2 * M.delta * M.T * u + M.T ** 2 * (1 - 2 * M.delta)).sum() / 2
    pri = 0.0
    F, Z, n, _ = obj.shape
    for f in range(F):
        x = obj[f].double()
        for dz in (0, 1):
            for dy in (-1, 0, 1):
                for dx in (-1, 0, 1):
                    if (dz, dy, dx) <= (0, 0, 0):
                        continue
                    a = x[:Z - dz, max(0, -dy):n - max(0, dy), max(0, -dx):n - max(0, dx)]
                    b = x[dz:, max(0, dy):n - max(0, -dy), max(0, dx):n - max(0, -dx)]
                    pri = pri + M.g[dz + 1, dy + 1, dx + 1] * M.rho(a - b, M.sS, M.cS).sum()
        if f + 1 < F:
            pri = pri + M.gt * M.rho(x - obj[f + 1].double(), M.sT, M.cT).sum()
    fwd, pri = float(fwd), float(pri)
    return fwd + pri, fwd, pri


def _conv(x, w, b):
    """3 x 3 x 3 convolution with zero padding, channels last, by 27 matrix products."""
    N, D, H, W, _ = x.shape
    p = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1, 1, 1))
    out = b.expand(N, D, H, W, -1)
    for t in range(27):
        z, y, q = t // 9, t // 3 % 3, t % 3
        out = out + p[:, z:z + D, y:y + H, q:q + W] @ w[t].T
    return out


def _exact_net(case, seed):
    x, mean, target = _crop_volume(case, seed)
    train = case["kind"] == "train"
    P = {}
    for k, (w, b) in _params(seed).items():
        w = torch.as_tensor(w, device="cuda")
        w = w.double() if k == "head" else w.bfloat16().double()  # the weights the layers hold
        P[k] = [w.requires_grad_(train), torch.as_tensor(b, device="cuda").double().requires_grad_(train)]
    xd, md = x.double(), mean.double()
    inp = torch.zeros(x.shape + (32,), dtype=torch.float64, device="cuda")
    inp[..., 0], inp[..., 1] = SCALE * xd, SCALE * md
    acts = {"x": inp}
    for name, src, _, _ in ARCH:
        if src.startswith("pool:"):
            a = acts[src[5:]]
            N, D, H, W, C = a.shape
            a = a.reshape(N, D // 2, 2, H // 2, 2, W // 2, 2, C).mean((2, 4, 6))
        elif src.startswith("cat:"):
            p, q = src[4:].split(",")
            up = acts[p]
            for dim in (1, 2, 3):
                up = up.repeat_interleave(2, dim)
            a = torch.cat([up, acts[q]], -1)
        else:
            a = acts[src]
        acts[name] = torch.relu(_conv(a, *P[name]))
    w, b = P["head"]
    out = xd + ((acts["d1"] @ w) + b) / SCALE
    if not train:
        return out
    loss = ((out - target.double()) ** 2).mean()
    loss.backward()
    return {"loss": float(loss), "out": out.detach(),
            "grads": {"%s.%s" % (k, n): t.grad for k, v in P.items() for n, t in zip("wb", v)}}


def exact(case, seed):
    kind = case["kind"]
    if kind in ("icd", "chunk"):
        return _exact_icd(case, seed)
    if kind == "batch":
        return None  # minutes, one voxel after another
    if kind in ("unet", "train"):
        return _exact_net(case, seed)
    scan, ph = _scan(case, seed)
    M = _Model(scan, case.get("mult", 1))
    if kind == "fbp":
        return _exact_fbp(scan, M)
    obj = ph.raster(M.frames, M.nx, M.nz)
    if kind == "cost":
        return _exact_cost(scan, M, obj)
    y = torch.as_tensor(scan["projections"], dtype=torch.float64, device="cuda")
    e = y - M.project(obj).repeat_interleave(M.m, 1)
    return e.permute(0, 2, 1).contiguous()
