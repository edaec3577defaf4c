"""The work whose speed is tracked: Langevin dynamics without and with
hydrodynamics (TEA, MLP-HI), network training and inference, and the
feature/label extraction, each through mt_amd.engine.Engine as a program of a
user calls it.

Sizes follow the repository's workloads (mt_amd/workloads.py, bench.py): 13-PF
microtubules of 12 to 95 dimers per protofilament, batches of 1 to 256
trajectories, periodic boxes with thousands of free dimers, 100-step list and
epsilon intervals, 8192-sample training batches.  A dynamics pass runs `steps`
steps and reads the state back, as an output stride does; the state goes on
from pass to pass.
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

from mt_amd import lattice, params, workloads
from mt_amd.engine import Engine, HI_MLP, MLP_IN, MLP_NPARAM, MLP_OUT, TEA_SYMMETRIC

GEOMETRY_SEED = 4242            # tube lengths and free-dimer places of a mixed batch
PLAIN_FLOPS = 600               # per bead and step: bonded terms, 8 LJ pairs, 6 normals, one rotation
TEA_PAIR_FLOPS = 50             # per unordered pair: RPY coefficients and both products
EPS_PAIR_FLOPS = 40             # per unordered pair of an epsilon refresh
NET_FLOPS = 2 * (96 * 128 + 2 * 128 * 128 + 128 * 9)   # per sample, forward
STATE_BYTES = 112               # per bead: six state floats and two generator states, in and out
HIDDEN = 128
MOST_UM = 30.0                  # largest free-dimer concentration


def listed():
    return [
        # one short tube: the smallest run, bound by latency
        dict(name="plain_one_tube", kind="plain", layout="tubes", ntraj=1, dimers=12, steps=100),
        # a batch of tubes over several list intervals: the throughput run
        dict(name="plain_batch", kind="plain", layout="tubes", ntraj=256, dimers=40, steps=1000),
        # a batch with frequent output: short windows, where set-up counts
        dict(name="plain_windows", kind="plain", layout="tubes", ntraj=96, dimers=21, steps=20),
        # tubes among free dimers in periodic boxes, sizes uneven: cell lists
        dict(name="plain_free_dimers", kind="plain", layout="mixed", ntraj=4, dimers=95, free=20000, steps=200),
        # TEA on one short tube: launches count
        dict(name="tea_one_tube", kind="tea", layout="tubes", ntraj=1, dimers=12, steps=100),
        # TEA on a batch of tubes, one epsilon refresh per 100 steps
        dict(name="tea_batch", kind="tea", layout="tubes", ntraj=64, dimers=40, steps=100),
        # TEA on uneven periodic batches: the O(N^2) pair sums at their largest
        dict(name="tea_free_dimers", kind="tea", layout="mixed", ntraj=4, dimers=95, free=20000, steps=100),
        # MLP-HI on full-size periodic systems, the judge once per 100 steps
        dict(name="mlp_free_dimers", kind="mlp", layout="mixed", ntraj=8, dimers=95, free=20000, steps=100),
        # network training, the batch size of the deployed network
        dict(name="mlp_train", kind="train", samples=32768, batch=8192, iters=20),
        # loss and gradient of a small ragged sample (checks, other optimisers)
        dict(name="mlp_loss_grad", kind="grad", samples=777),
        # inference on host rows
        dict(name="mlp_forward", kind="forward", samples=20011),
        # features and exact labels of a batch: one frame of training data
        dict(name="mlp_features", kind="local", layout="mixed", ntraj=2, dimers=60, free=5000),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["plain"] * 5 + ["tea"] * 3 + ["mlp", "train", "grad", "forward", "local"])
    if kind == "train":
        batch = _log_int(rng, 500, 8192)
        return dict(kind=kind, samples=batch * rng.randint(1, 4) + rng.randint(0, 99), batch=batch,
                    iters=rng.randint(3, 20))
    if kind == "grad":
        return dict(kind=kind, samples=_log_int(rng, 100, 8192))
    if kind == "forward":
        return dict(kind=kind, samples=_log_int(rng, 100, 60000))
    mixed = kind in ("mlp", "local") or rng.random() < 0.4
    steps = _log_int(rng, 20, 100)
    if mixed:
        top = 4 if kind in ("plain", "tea") else 6
        free = _log_int(rng, 2000, 20000 if kind != "local" else 8000)
        case = dict(kind=kind, layout="mixed", ntraj=rng.randint(1, top), dimers=rng.randint(21, _longest(free)),
                    free=free)
    else:
        case = dict(kind=kind, layout="tubes", ntraj=_log_int(rng, 1, 256 if kind == "plain" else 64),
                    dimers=rng.randint(12, 40))
    return case if kind == "local" else dict(case, steps=steps)


def _longest(free):
    """Longest tube (dimers) that the smallest box of `free` free dimers holds."""
    return int((lattice.box_side_nm(max(1000, free // 2), MOST_UM) - 33.0) / 8.0)


# ------------------------------------------------------------------ inputs
@functools.lru_cache(maxsize=4)
def _geometry(layout, ntraj, dimers, free):
    if layout == "tubes":
        return workloads.plain(ntraj, dimers, seed=GEOMETRY_SEED)
    # tube lengths and free-dimer counts spread below the stated largest ones;
    # the free dimers and their concentration set the box
    return workloads.uneven(ntraj, dimers=(max(12, dimers // 2), dimers), free=(max(1000, free // 2), free),
                            conc=(10.0, MOST_UM), seed=GEOMETRY_SEED)


def _batch(case, seed):
    """The case's structure with thermal displacements drawn from the seed."""
    b = _geometry(case["layout"], case["ntraj"], case["dimers"], case.get("free", 0)).copy()
    rng = np.random.default_rng([seed, 1])
    b.coords[:, :3] += rng.normal(0.0, 0.03, (b.nb, 3)).astype(np.float32)
    return b


def _params(case):
    return params.derive(dict(params.BASE if case["kind"] == "plain" else params.TEA))


def _streams(nb, seed):
    """HybridTaus states of a resumed run: any words >= 128."""
    return np.random.default_rng([seed, 2]).integers(128, 2 ** 32, 8 * nb, dtype=np.uint64).astype(np.uint32)


def _weights(seed, out_scale=1.0, diag=0.0):
    """Network weights of the usual initial scale; diag: the mean of the
    three diagonal outputs (a trained network's is near the local tensor's)."""
    rng = np.random.default_rng([seed, 3])
    shapes = [(MLP_IN, HIDDEN), (HIDDEN,), (HIDDEN, HIDDEN), (HIDDEN,), (HIDDEN, HIDDEN), (HIDDEN,),
              (HIDDEN, MLP_OUT), (MLP_OUT,)]
    parts = [rng.normal(0, 1 / np.sqrt(s[0]), s) if len(s) == 2 else rng.normal(0, 0.02, s) for s in shapes]
    parts[6] *= out_scale
    parts[7] = diag * np.eye(3).ravel() + out_scale * parts[7]
    return np.concatenate([v.ravel() for v in parts]).astype(np.float32)


def _samples(n, seed, tea_a=2.0):
    """Feature rows of n beads, their neighbours placed at random in the 12 nm
    ball (dilute beads with a few, tube beads with 32), nearest first, and the
    local hydrodynamic tensors of those neighbours as labels."""
    rng = np.random.default_rng([seed, 4])
    count = np.where(rng.random(n) < 0.7, rng.integers(1, 9, n), 32)
    d = rng.normal(size=(n, 32, 3))
    d *= (12.0 * rng.uniform(0.04, 1.0, (n, 32, 1)) ** (1 / 3)) / np.linalg.norm(d, axis=2, keepdims=True)
    d = np.take_along_axis(d, np.argsort((d * d).sum(2), axis=1)[:, :, None], axis=1)
    have = np.arange(32)[None, :] < count[:, None]
    r = np.linalg.norm(d, axis=2)
    w = np.where(have, _taper(r), 0.0)
    cii, crr = _rpy(r, tea_a)
    e = d / r[:, :, None]
    label = np.einsum("nk,nka,nkb->nab", w * crr, e, e)
    label += (w * cii).sum(1)[:, None, None] * np.eye(3)
    feat = np.where(have[:, :, None], d / 12.0, 0.0)
    return feat.reshape(n, MLP_IN).astype(np.float32), label.reshape(n, MLP_OUT).astype(np.float32)


def _taper(r):
    x = r.clip(8.0, 12.0) if isinstance(r, np.ndarray) else r.clamp(8.0, 12.0)
    cos = np.cos if isinstance(r, np.ndarray) else torch.cos
    return 0.5 * (1.0 + cos(math.pi * (x - 8.0) / 4.0))


def _rpy(r, a):
    """Coefficients of the Rotne-Prager-Yamakawa block cii I + crr e e^T."""
    where = np.where if isinstance(r, np.ndarray) else torch.where
    ra = r / a
    near = ra <= 2.0
    u = 1.0 / where(near, 2.0 + 0.0 * ra, ra)
    return (where(near, 1.0 - 9.0 * ra / 32.0, 0.75 * u * (1.0 + 2.0 / 3.0 * u * u)),
            where(near, 3.0 * ra / 32.0, 0.75 * u * (1.0 - 2.0 * u * u)))


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("train", "grad", "forward"):
        # the network's work needs no dynamics: an engine of the smallest batch
        eng = Engine(params.derive(dict(params.TEA)), workloads.plain(1, 12), max_lj=48)
        eng.mlp_set_weights(_weights(seed))
        x, y = _samples(case["samples"], seed)
        return dict(case=case, eng=eng, x=x, y=y)
    b = _batch(case, seed)
    eng = Engine(_params(case), b, max_lj=48)
    eng.set_rng(_streams(b.nb, seed))
    if kind == "tea":
        # the pair kernel that the autotuner keeps at these sizes, named so
        # that every run has the same one
        eng.set_tuning(tea_chunk=TEA_SYMMETRIC)
    if kind == "mlp":
        eng.mlp_set_weights(_weights(seed, out_scale=0.02, diag=0.8))
        eng.set_hi_mode(HI_MLP, check_every=100, tolerance=1e9)   # no trained network here: the judge only reports
    return dict(case=case, eng=eng)


def run(state):
    case, eng = state["case"], state["eng"]
    kind = case["kind"]
    if kind == "train":
        losses = eng.mlp_train(state["x"], state["y"], case["iters"], case["batch"], 1e-3)
        return dict(weights=eng.mlp_get_weights(), losses=[float(v) for v in losses])
    if kind == "grad":
        loss, grad = eng.mlp_loss_grad(state["x"], state["y"])
        return dict(loss=loss, grad=grad)
    if kind == "forward":
        return eng.mlp_forward(state["x"])
    if kind == "local":
        feat, label = eng.mlp_local()
        return dict(features=feat, labels=label)
    eng.run(case["steps"])
    return eng.get_state()


def work(case):
    kind = case["kind"]
    weights = 4.0 * MLP_NPARAM
    if kind in ("train", "grad", "forward"):
        n = case["samples"]
        if kind == "forward":
            return dict(bytes=4.0 * n * (MLP_IN + MLP_OUT) + weights, flops=float(NET_FLOPS) * n)
        rows = n if kind == "grad" else case["batch"] * case["iters"]
        # backward: the same products again for the weights and, without the first layer, for the inputs
        flops = rows * (2.0 * NET_FLOPS + (NET_FLOPS - 2 * MLP_IN * HIDDEN))
        return dict(bytes=4.0 * rows * (MLP_IN + MLP_OUT) + 2 * weights, flops=flops)
    b = _geometry(case["layout"], case["ntraj"], case["dimers"], case.get("free", 0))
    n = b.sizes().astype(np.float64)
    if kind == "local":
        return dict(bytes=b.nb * 4.0 * (3 + MLP_IN + MLP_OUT), flops=30.0 * 20 * b.nb)
    steps = case["steps"]
    pairs = float((n * (n - 1)).sum()) / 2
    flops = float(PLAIN_FLOPS) * b.nb * steps
    refreshes = -(-steps // 100) if kind != "plain" else 0
    flops += EPS_PAIR_FLOPS * pairs * refreshes
    if kind == "tea":
        flops += TEA_PAIR_FLOPS * pairs * steps
    if kind == "mlp":
        flops += float(NET_FLOPS) * b.nb * steps
    return dict(bytes=float(STATE_BYTES) * b.nb, flops=flops)


# ------------------------------------------------- the same in 64 bits
def exact(case, seed):
    """What run() returns for prepare(case, seed), in 64-bit torch; None for
    dynamics whose pair or neighbour sums would take minutes in 64 bits."""
    kind = case["kind"]
    if kind in ("train", "grad", "forward"):
        return _exact_network(case, seed)
    b = _batch(case, seed)
    if kind == "local":
        # the 32 nearest are ordered by 32-bit squared distances: near ties
        # may fall otherwise in 64 bits, so features have no value here
        return dict(features=None, labels=_exact_labels(b))
    if kind == "mlp" or (kind == "tea" and case["layout"] == "mixed"):
        return None
    return _Dynamics(_params(case), b, _streams(b.nb, seed)).run(case["steps"])


def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _f64(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(_device()).double()


def _split_params(w):
    shapes = [(MLP_IN, HIDDEN), (HIDDEN,), (HIDDEN, HIDDEN), (HIDDEN,), (HIDDEN, HIDDEN), (HIDDEN,),
              (HIDDEN, MLP_OUT), (MLP_OUT,)]
    out, k = [], 0
    for s in shapes:
        n = int(np.prod(s))
        out.append(w[k:k + n].view(s))
        k += n
    return out


def _net(w, x):
    p = _split_params(w)
    for k in (0, 2, 4):
        x = torch.tanh(x @ p[k] + p[k + 1])
    return x @ p[6] + p[7]


def _exact_network(case, seed):
    x, y = (_f64(v) for v in _samples(case["samples"], seed))
    w32 = _weights(seed)
    if case["kind"] == "forward":
        # inference takes the weights rounded to bfloat16
        return _net(_f64(torch.from_numpy(w32).bfloat16().float().numpy()), x).cpu().numpy()
    w = _f64(w32)

    def loss_grad(w, x, y):
        w = w.detach().requires_grad_(True)
        loss = ((_net(w, x) - y) ** 2).mean()
        return float(loss.detach()), torch.autograd.grad(loss, w)[0]

    if case["kind"] == "grad":
        loss, grad = loss_grad(w, x, y)
        return dict(loss=loss, grad=grad.cpu().numpy())
    m, v, losses, pos, batch = torch.zeros_like(w), torch.zeros_like(w), [], 0, case["batch"]
    for t in range(1, case["iters"] + 1):   # Adam over consecutive batches, from the top again where one would not fit
        if pos + batch > case["samples"]:
            pos = 0
        loss, g = loss_grad(w, x[pos:pos + batch], y[pos:pos + batch])
        pos += batch
        losses.append(loss)
        m = 0.9 * m + 0.1 * g
        v = 0.999 * v + 0.001 * g * g
        w = w - 1e-3 * (m / (1 - 0.9 ** t)) / (torch.sqrt(v / (1 - 0.999 ** t)) + 1e-8)
    return dict(weights=w.cpu().numpy(), losses=losses)


def _exact_labels(b, tea_a=2.0):
    out = torch.zeros((b.nb, 3, 3), dtype=torch.float64, device=_device())
    x = _f64(b.coords)[:, :3]
    for t in range(b.ntraj):
        lo, hi, side = int(b.off[t]), int(b.off[t + 1]), float(b.box[t])
        xt = x[lo:hi]
        for i0 in range(0, hi - lo, 1024):
            d = xt[None, :, :] - xt[i0:i0 + 1024, None, :]
            if side > 0:
                d = d - side * torch.round(d / side)
            i, j = torch.nonzero((d * d).sum(2) < 144.0, as_tuple=True)
            keep = j != i + i0
            i, j = i[keep], j[keep]
            e = d[i, j]
            r = e.norm(dim=1)
            e = e / r[:, None]
            cii, crr = _rpy(r, tea_a)
            g = crr[:, None, None] * e[:, :, None] * e[:, None, :] + cii[:, None, None] * torch.eye(3).to(e)
            out[lo + i0:lo + i0 + 1024].index_add_(0, i, _taper(r)[:, None, None] * g)
    return out.view(b.nb, 9).cpu().numpy()


class _Dynamics:
    """Forces, list rebuilds, HybridTaus noise and the Euler-Maruyama step of
    a batch (with TEA's pair sums where the parameters ask for them)."""

    def __init__(self, p, b, seeds):
        dev = _device()
        self.p, self.b, self.nb = p, b, b.nb
        self.c = _f64(b.coords)[:, :6].clone()   # x, y, z, fi, theta, psi
        sizes = b.sizes()
        self.tid = torch.from_numpy(np.repeat(np.arange(b.ntraj), sizes)).to(dev)
        self.base = torch.from_numpy(np.repeat(b.off[:-1], sizes)).to(dev)
        self.local = torch.arange(self.nb, device=dev) - self.base
        self.side = _f64(np.repeat(b.box, sizes))
        self.extra = torch.from_numpy(b.extra).to(dev) != 0
        self.mobile = ~self.extra & (torch.from_numpy(b.fixed).to(dev) == 0)
        self.mon, self.gtp, self.tub = (torch.from_numpy(v).to(dev) for v in (b.mon_type, b.gtp, b.on_tub))
        self.hraw = torch.from_numpy(b.harm).to(dev).long()
        self.s = torch.from_numpy(seeds.astype(np.int64).reshape(2 * self.nb, 4).T.copy()).to(dev)
        c, s = math.cos(2 * math.pi / 13), math.sin(2 * math.pi / 13)
        self.p1 = [0.5 * 8.12 * (c - 1.0), 0.5 * 8.12 * s, -6.0 / 13.0]
        self.p2 = [0.5 * 8.12 * (c - 1.0), -0.5 * 8.12 * s, 6.0 / 13.0]

    # HybridTaus, four uniforms (and so two Box-Muller pairs) per draw; `who`: the streams that advance
    def normals(self, who):
        z = [v[who] for v in self.s]
        full = 0xFFFFFFFF

        def taus(v, a, q, c, m):
            return (((v & m) << c) & full) ^ ((((v << a) & full) ^ v) >> q)

        u = []
        for _ in range(4):
            z = [taus(z[0], 13, 19, 12, 4294967294), taus(z[1], 2, 25, 4, 4294967288),
                 taus(z[2], 3, 11, 17, 4294967280), (1664525 * z[3] + 1013904223) & full]
            f = ((z[0] ^ z[1] ^ z[2] ^ z[3]) & 0x7FFFFF).double() / 8388608.0
            u.append(torch.where(f == 0, f + float(np.float32(1e-8)), f))
        for v, n in zip(self.s, z):
            v[who] = n
        r0, r1 = torch.sqrt(-2 * torch.log(u[0])), torch.sqrt(-2 * torch.log(u[2]))
        a0, a1 = 2 * math.pi * u[1], 2 * math.pi * u[3]
        return torch.stack([r0 * torch.sin(a0), r0 * torch.cos(a0), r1 * torch.sin(a1)], 1)

    def frames(self):
        f, t, p = self.c[:, 3], self.c[:, 4], self.c[:, 5]
        cf, sf, ct, st, cp, sp = f.cos(), f.sin(), t.cos(), t.sin(), p.cos(), p.sin()
        rows = [[cp * ct, cp * st * sf - sp * cf, cp * st * cf + sp * sf],
                [sp * ct, sp * st * sf + cp * cf, sp * st * cf - cp * sf], [-st, ct * sf, ct * cf]]
        R = torch.stack([torch.stack(r, 1) for r in rows], 1)
        self.n = R[:, :, 2]
        self.a1, self.a2 = (R @ torch.tensor(v, dtype=torch.float64, device=R.device) for v in (self.p1, self.p2))
        self.uphi = torch.stack([cp * ct, sp * ct, -st], 1)
        self.uth = torch.stack([-sp, cp], 1)

    def image(self, d, i):
        side = self.side[i][:, None]
        return torch.where(side > 0, d - side * torch.round(d / torch.where(side > 0, side, 1.0)), d)

    def gap(self, i, j, a, b):
        return self.image(self.c[i, :3] - self.c[j, :3], i) + a - b

    def rebuild(self):
        """Ordered pairs within the list cutoff, and the bonds among them."""
        cut, found = max(float(self.p.ljpairscutoff), 6.75), []
        for t in range(self.b.ntraj):
            lo, hi, side = int(self.b.off[t]), int(self.b.off[t + 1]), float(self.b.box[t])
            x = self.c[lo:hi, :3]
            for i0 in range(0, hi - lo, 2048):
                d = x[i0:i0 + 2048, None, :] - x[None, :, :]
                if side > 0:
                    d = d - side * torch.round(d / side)
                i, j = torch.nonzero((d * d).sum(2) < cut * cut, as_tuple=True)
                keep = (j != i + i0) & ~self.extra[lo + i0 + i]
                found.append((i[keep] + (lo + i0), j[keep] + lo))
        i, j = torch.cat([f[0] for f in found]), torch.cat([f[1] for f in found])
        d = self.image(self.c[i, :3] - self.c[j, :3], i).norm(dim=1)
        near = d < float(self.p.ljpairscutoff)
        self.lj = (i[near], j[near])
        bond = (d < 6.75) & (self.hraw[i].abs() != self.local[j])
        i, j = i[bond], j[bond]
        rp = torch.where(self.hraw[i] < 0, -2.0, 2.0).double()[:, None]
        on = (self.mon[i] != self.mon[j]) & (self.gap(i, j, rp * self.n[i], -rp * self.n[j]).norm(dim=1) < 2.5)
        pos = (self.hraw[i] >= 0) & (self.local[j] != 0)
        self.lon = (i[on], j[on], torch.where(pos[on], 2.0, -2.0).double()[:, None])
        one = self.gap(i, j, self.a1[i], self.a2[j]).norm(dim=1) < 2.5
        two = self.gap(i, j, self.a2[i], self.a1[j]).norm(dim=1) < 2.5
        self.lat = (torch.cat([i[one], i[two]]), torch.cat([j[one], j[two]]),
                    torch.cat([one.new_ones(int(one.sum())), one.new_zeros(int(two.sum()))])[:, None])

    def add(self, i, g, a, scale, bend=None):
        """-scale times the gradient of |g|^2 / 2 onto beads i, and bending torques."""
        t = torch.linalg.cross(a, g)
        tor = torch.stack([(self.uphi[i] * t).sum(1), (self.uth[i] * t[:, :2]).sum(1), t[:, 2]], 1)
        f = -scale[:, None] * torch.cat([g, tor], 1)
        self.F.index_add_(0, i, f if bend is None else f + bend)

    def bending(self, i, j, dr, rm, th0):
        p, sg = self.p, torch.sign(rm[:, 0])
        d = self.c[j] - self.c[i]
        out = torch.zeros((len(i), 6), dtype=torch.float64, device=d.device)
        out[:, 3] = sg * p.B_fi * torch.sin(sg * d[:, 3] - p.fi_0)
        out[:, 4] = sg * p.B_theta * torch.sin(sg * d[:, 4] - th0)
        out[:, 5] = sg * p.B_psi * torch.sin(sg * d[:, 5] - p.psi_0)
        return out * (dr < 1.0)[:, None]

    def slope(self, i, j, dr, D, A, barrier):
        e = torch.exp(-A * dr)
        s = 2 * A * D * (1 - e) * e
        if self.p.barrier:
            h, r, w = barrier
            b = -h * torch.exp(-0.5 * (dr - r) ** 2 / w ** 2) * (dr - r) / w ** 2
            s = s + torch.where((self.tub[i] == 0) & (self.tub[j] == 0), b, 0.0)
        return torch.where(dr > 0, s / dr.clamp(min=1e-300), 0.0)

    def forces(self):
        p, c = self.p, self.c
        self.F = torch.zeros_like(c)
        theta0 = torch.where(self.gtp == 1, p.theta0_gtp, p.theta0_gdp).double()
        has = torch.from_numpy(self.b.harm_count).to(c.device) > 0
        i = torch.nonzero(has & ~self.extra)[:, 0]
        j = self.hraw[i].abs() + self.base[i]
        rm = torch.where(self.hraw[i] < 0, 2.0, -2.0).double()[:, None]
        g = self.gap(i, j, rm * self.n[i], -rm * self.n[j])
        self.add(i, g, rm * self.n[i], torch.full_like(g[:, 0], p.C),
                 self.bending(i, j, g.norm(dim=1), rm, theta0[i]))
        i, j, rm = self.lon
        g = self.gap(i, j, rm * self.n[i], -rm * self.n[j])
        dr = g.norm(dim=1)
        last = torch.where(c[i, 2] > c[j, 2], i, j)
        self.add(i, g, rm * self.n[i],
                 self.slope(i, j, dr, p.D_long, p.A_long, (p.a_barr_long, p.r_barr_long, p.w_barr_long)),
                 self.bending(i, j, dr, rm, theta0[last]))
        i, j, sw = self.lat
        a = torch.where(sw, self.a1[i], self.a2[i])
        g = self.gap(i, j, a, torch.where(sw, self.a2[j], self.a1[j]))
        D = torch.where(self.mon[i] != self.mon[j], p.D_lat / p.seam_coeff, p.D_lat).double()
        self.add(i, g, a, self.slope(i, j, g.norm(dim=1), D, p.A_lat, (p.a_barr_lat, p.r_barr_lat, p.w_barr_lat)))
        if p.lj_on:
            i, j = self.lj
            d = self.image(c[i, :3] - c[j, :3], i)
            r2 = (d * d).sum(1)
            s = torch.where(r2 < 36.0, 6.0 * p.ljscale * p.ljsigma6 / r2 ** 4, 0.0)
            self.F[:, :3].index_add_(0, i, s[:, None] * d)

    # TEA on batches of equal open trajectories
    def blocks(self):
        x = self.c[:, :3].view(self.b.ntraj, -1, 3)
        d = x[:, None, :, :] - x[:, :, None, :]
        r = (d * d).sum(3).sqrt()
        cii, crr = _rpy(r, self.p.tea_a)
        inv = torch.where(r > 0, 1.0 / torch.where(r > 0, r, 1.0), 0.0)
        on = (r > 0).double()
        return cii * on, crr * on, d * inv[..., None]

    def refresh(self):
        cii, crr, e = self.blocks()
        n = e.shape[1]
        ci = ((cii ** 2)[..., None] + (crr * (2 * cii + crr))[..., None] * e ** 2).sum(2)
        eps = (3 * cii + crr * e.sum(3) ** 2).sum((1, 2)) / (3.0 * n * (3.0 * n - 3.0))
        eps = eps.clamp(max=1.0)
        a = (3.0 * n - 1) * eps ** 2 - (3.0 * n - 2) * eps
        self.beta = ((1 - torch.sqrt(1 - a)) / a)[:, None, None]
        self.C = 1.0 / torch.sqrt(1 + self.beta ** 2 * ci)

    def tea(self, xi):
        p = self.p
        F = self.F[:, :3].view(self.b.ntraj, -1, 3)
        R = xi.view_as(F) * math.sqrt(2 * 0.0019872041 * p.temp * p.gammaR / p.dt)
        cii, crr, e = self.blocks()
        drift = cii @ F + torch.einsum("tij,tija,tij->tia", crr, e, (e * F[:, None]).sum(3))
        bc = self.beta * self.C
        # beta C_i acts on the components of R_j before the block
        noise = bc * (cii @ R) + torch.einsum("tij,tija,tij->tia", crr, e, (e * (bc[:, :, None] * R[:, None])).sum(3))
        return (F + self.C * R + drift + noise).reshape(-1, 3)

    def run(self, steps):
        p = self.p
        mob = torch.nonzero(self.mobile)[:, 0]
        every = torch.arange(self.nb, device=mob.device)
        drawn = every if p.tea_on else mob
        vta = p.varTheta * math.sqrt(p.freeze_temp / p.alpha)
        for step in range(steps):
            self.frames()
            if step % p.ljpairsupdatefreq == 0:
                self.rebuild()
            self.forces()
            both = self.normals(torch.cat([drawn, drawn + self.nb]))
            lin, ang = both[:len(drawn)], both[len(drawn):]
            if p.tea_on:
                if step % p.tea_epsilon_freq == 0:
                    self.refresh()
                move = (p.dt / p.gammaR) * self.tea(lin)[mob]
                ang = ang[mob]
            else:
                move = (p.dt / p.gammaR) * self.F[mob, :3] + p.varR * lin
            dta, dtt = p.dt / (p.gammaTheta * p.alpha), p.dt / p.gammaTheta
            F = self.F[mob]
            turn = torch.stack([dta * F[:, 3] + vta * ang[:, 0], dtt * F[:, 4] + p.varTheta * ang[:, 2],
                                dta * F[:, 5] + vta * ang[:, 1]], 1)
            self.c[mob] += torch.cat([move, turn], 1)
        return torch.cat([self.c, torch.zeros_like(self.c[:, :1])], 1).cpu().numpy()
