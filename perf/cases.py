"""What a user of this framework has it do, at the sizes it is used at.

Every case goes through the public Python entry points: whole simulation steps
(BarnesHut.update, Batch.step, Batch.graph_step), the evaluation of the
accelerations at given positions (rebuild and forces), their gradient
(BarnesHut.vjp, BarnesHutAccel, rollout) and the key stages (computeKeys,
sortKeys).  Sizes run from a small disk, where the launches count, to the 4M
headline workload; odd sizes, the unsoftened and the uncompensated force, several
opening angles and uneven ensembles are among them.

listed() gives the cases by name, draw(rng) one more of the same ranges,
prepare(case, seed) the inputs and handles a program keeps, run(state) one pass,
work(case) the bytes and operations no implementation can do without, and
exact(case, seed) the same results in 64 bits from plain torch.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import nns_amd
from nns_amd.adjoint import BarnesHutAccel, Slots, rollout

DEV = "cuda"


def listed():
    return [
        # the smallest runs: a disk of a few thousand bodies stepped many times (the reference's demo sizes)
        {"name": "step_disk_2k", "path": "step", "kind": "star_disk", "n": 2000, "theta": 0.5},
        # the plain CPU configuration: star outside the tree, coupled directly, and 32,767 disk bodies
        {"name": "step_suns_32k", "path": "step", "kind": "star_disk", "n": 32768, "theta": 0.5, "suns": 1},
        # an ordinary odd-sized cluster run at a looser opening angle
        {"name": "step_plummer_150k", "path": "step", "kind": "plummer", "n": 150001, "theta": 0.7},
        # the Plummer sphere of a million bodies
        {"name": "step_plummer_1m", "path": "step", "kind": "plummer", "n": 1048576, "theta": 0.5},
        # the headline workload: circular binary and Keplerian disk
        {"name": "step_binary_4m", "path": "step", "kind": "binary_disk", "n": 4194304, "theta": 0.5},
        # accelerations at given positions, as an integrator of the user's own asks for them: a tight
        # opening angle, unsoftened, plain accumulation
        {"name": "accel_disk_300k", "path": "accel", "kind": "binary_disk", "n": 300007, "theta": 0.3,
         "softening": 0.0, "kahan": 0},
        # an ensemble of small clusters replayed as a graph (parameter studies)
        {"name": "batch_96_small", "path": "batch", "systems": 96, "lo": 200, "hi": 4000, "graph": 1},
        # the ensemble of large uneven clusters with their own opening angles
        {"name": "batch_512", "path": "batch", "systems": 512, "lo": 1024, "hi": 65536, "graph": 0},
        # gradient of the accelerations at a modest size: forward and backward of the autograd function
        {"name": "grad_plummer_20k", "path": "grad", "kind": "plummer", "n": 20011, "theta": 0.5},
        # vector-Jacobian product over the tree in hand, the backward step of the large adjoint run
        {"name": "vjp_plummer_262k", "path": "vjp", "kind": "plummer", "n": 262144, "theta": 0.5},
        # gradient of a checkpointed rollout with respect to the initial state and the masses
        {"name": "rollout_65k", "path": "rollout", "kind": "plummer", "n": 65536, "theta": 0.5, "steps": 12},
        # space-filling-curve keys and their stable sort alone (domain decomposition, neighbour lists)
        {"name": "hilbert_sort_1m", "path": "sort", "kind": "plummer", "n": 1000003},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    path = rng.choice(("step", "step", "step", "accel", "batch", "grad", "vjp", "rollout", "sort"))
    kind = rng.choice(("star_disk", "plummer", "binary_disk"))
    theta = rng.choice((0.4, 0.5, 0.6, 0.7, 0.8))
    if path == "step":
        c = {"path": path, "kind": kind, "n": _log_int(rng, 1500, 2000000), "theta": theta}
        if kind == "star_disk" and rng.random() < 0.5:
            c["suns"] = 1
        return c
    if path == "accel":
        return {"path": path, "kind": kind, "n": _log_int(rng, 1500, 1000000),
                "theta": rng.choice((0.3, 0.5, 0.7)), "softening": rng.choice((0.0, 1e-3)),
                "kahan": rng.choice((0, 1))}
    if path == "batch":
        lo = _log_int(rng, 100, 2000)
        return {"path": path, "systems": _log_int(rng, 16, 400), "lo": lo, "hi": _log_int(rng, 4 * lo, 16 * lo),
                "graph": rng.choice((0, 1))}
    if path == "grad":
        return {"path": path, "kind": kind, "n": _log_int(rng, 2000, 200000), "theta": theta}
    if path == "vjp":
        return {"path": path, "kind": kind, "n": _log_int(rng, 8000, 400000), "theta": theta}
    if path == "rollout":
        return {"path": path, "kind": "plummer", "n": _log_int(rng, 4000, 100000), "theta": theta,
                "steps": rng.randint(4, 12)}
    return {"path": path, "kind": kind, "n": _log_int(rng, 2000, 4000000)}


# ------------------------------------------------------------------ inputs
EVERY = 8      # checkpoint distance of the rollout
DT = 1e-3


def _params(case):
    return nns_amd.default_params(theta=case.get("theta", 0.5), softening=case.get("softening", 1e-3),
                                  kahan=case.get("kahan", 1), timestep=DT)


def _bodies(case, seed):
    """Host arrays x, y, z, vx, vy, vz, mass (single systems)."""
    return nns_amd.initial_conditions(case["kind"], case["n"], seed + 1)


def _ensemble(case, seed):
    """Host arrays of the concatenated clusters, their sizes (spread evenly over the logarithm, shuffled by the
    seed) and opening angles."""
    rng = np.random.default_rng(seed)
    s = case["systems"]
    sizes = np.exp(np.linspace(math.log(case["lo"]), math.log(case["hi"]), s)).astype(np.int32)
    sizes = sizes[rng.permutation(s)]
    thetas = np.array([0.3, 0.5, 0.7] * (s // 3 + 1), np.float32)[:s]
    parts = [nns_amd.initial_conditions("plummer", int(k), seed * 1000 + j + 1) for j, k in enumerate(sizes)]
    return [np.concatenate([p[k] for p in parts]) for k in range(7)], sizes, thetas


def _cotangents(n, seed):
    g = torch.Generator(device=DEV).manual_seed(seed + 77)
    return [torch.randn(n, device=DEV, generator=g) for _ in range(3)]


def _split_suns(case, arrs):
    """(bodies in the tree, stars outside it): the star of the disk is its first body."""
    k = case.get("suns", 0)
    return [a[k:] for a in arrs], [a[:k] for a in arrs] if k else None


def prepare(case, seed):
    path = case["path"]
    if path == "batch":
        arrs, sizes, thetas = _ensemble(case, seed)
        s = {"path": path, "batch": nns_amd.Batch(*arrs, sizes, thetas, _params(case))}
        if case["graph"]:
            torch.cuda.synchronize()  # the arrays were filled on the current stream
            s["stream"] = torch.cuda.Stream()
        return s
    arrs = _bodies(case, seed)
    n = case["n"]
    if path in ("step", "accel"):
        body, stars = _split_suns(case, arrs)
        return {"path": path, "bh": nns_amd.BarnesHut(*body, params=_params(case), stars=stars)}
    if path == "vjp":
        bh = nns_amd.BarnesHut(*arrs, params=_params(case))
        bh.rebuild()
        return {"path": path, "bh": bh, "u": _cotangents(n, seed)}
    if path == "grad":
        ins = [torch.tensor(arrs[k], device=DEV, requires_grad=True) for k in (0, 1, 2, 6)]
        return {"path": path, "slots": Slots(n, 1, _params(case)), "ins": ins, "u": _cotangents(n, seed)}
    if path == "rollout":
        ins = [torch.tensor(a, device=DEV, requires_grad=True) for a in arrs]
        tgt = [torch.as_tensor(a, device=DEV) for a in _bodies(case, seed + 500)[:3]]
        return {"path": path, "slots": Slots(n, EVERY, _params(case)), "ins": ins, "tgt": tgt,
                "steps": case["steps"]}
    pos = [torch.as_tensor(a, device=DEV) for a in arrs[:3]]
    ctx = nns_amd.Context(n, params=_params({}))
    f = torch.zeros(7, dtype=torch.float32, device=DEV)
    return {"path": path, "n": n, "kw": nns_amd.KernelsWrapper(ctx), "pos": pos, "box": [f[k:k + 1] for k in range(7)],
            "keys": torch.empty(n, dtype=torch.int64, device=DEV),
            "skeys": torch.empty(n, dtype=torch.int64, device=DEV),
            "perm": torch.empty(n, dtype=torch.int32, device=DEV)}


# ------------------------------------------------------------------ one pass
STATE = ("x", "y", "z", "vx", "vy", "vz", "ax", "ay", "az")


def run(s):
    path = s["path"]
    if path == "step":
        bh = s["bh"]
        bh.update()
        out = {k: bh.arr[k][:bh.n] for k in STATE}
        if bh.nstars:
            out.update({k: bh.arr[k] for k in ("sx", "sy", "sz", "svx", "svy", "svz", "sax", "say", "saz")})
        return out
    if path == "accel":
        bh = s["bh"]
        bh.rebuild()
        bh.forces()
        return {k: bh.arr[k][:bh.n] for k in ("ax", "ay", "az", "sorted")}
    if path == "batch":
        b = s["batch"]
        if "stream" in s:
            b.graph_step(s["stream"])
        else:
            b.step()
        return {k: b.arr[k] for k in STATE}
    if path == "vjp":
        return list(s["bh"].vjp(*s["u"]))
    if path == "grad":
        for t in s["ins"]:
            t.grad = None
        a = BarnesHutAccel.apply(*s["ins"], s["slots"])
        torch.autograd.backward(a, s["u"])
        return [t.detach() for t in a] + [t.grad for t in s["ins"]]
    if path == "rollout":
        for t in s["ins"]:
            t.grad = None
        out = rollout(s["slots"], *s["ins"], steps=s["steps"], dt=DT, every=EVERY)
        loss = sum(((o - t) ** 2).mean() for o, t in zip(out[:3], s["tgt"]))
        loss.backward()
        return [loss.detach()] + [o.detach() for o in out] + [t.grad for t in s["ins"]]
    kw, n = s["kw"], s["n"]
    kw.computeBoundingBox(s["box"][6], *s["pos"], *s["box"][:6], n)
    kw.computeKeys(*s["pos"], n, s["keys"], nns_amd.KEY_HILBERT)
    kw.sortKeys(s["keys"], n, s["skeys"], s["perm"])
    return [s["keys"], s["skeys"], s["perm"]]


# ------------------------------------------------------------------ necessary work
def _interactions(kind, n, theta):
    """Interactions per body, as counted at theta = 0.5 (disk 703 at 1M, 906 at 4M; sphere 1080 at 64K, 2330 at
    1M): linear in the logarithm of n; list lengths go about as theta^-2."""
    per = 2330 + 310 * math.log2(n / 1048576) if kind == "plummer" else 703 + 100 * math.log2(n / 1048576)
    return max(60.0, min(per * (0.5 / max(theta, 0.05)) ** 2, n - 1.0))


def work(case):
    path = case["path"]
    if path == "sort":
        # positions in; keys, sorted keys and the permutation out
        return {"bytes": case["n"] * (12 + 8 + 8 + 4), "flops": 0}
    if path == "batch":
        sizes = np.exp(np.linspace(math.log(case["lo"]), math.log(case["hi"]), case["systems"]))
        flops = sum(20 * k * _interactions("plummer", k, (0.3, 0.5, 0.7)[j % 3]) for j, k in enumerate(sizes))
        return {"bytes": float(sizes.sum()) * (28 + 36), "flops": flops}
    n = case["n"]
    inter = n * _interactions(case["kind"], n, case["theta"])
    if path == "step":
        return {"bytes": n * (28 + 36), "flops": 20 * inter}
    if path == "accel":
        return {"bytes": n * (16 + 16), "flops": 20 * inter}
    if path == "vjp":  # about twice a forward interaction: h and the two sums it goes to
        return {"bytes": n * (28 + 16), "flops": 40 * inter}
    if path == "grad":
        return {"bytes": n * (28 + 28), "flops": 60 * inter}
    return {"bytes": n * (28 + 12 + 24 + 28), "flops": 60 * inter * case["steps"]}


# ------------------------------------------------------------------ the same in 64 bits
LEVELS = 21


def _spread(v):
    for s, mask in ((32, 0x001f00000000ffff), (16, 0x001f0000ff0000ff), (8, 0x100f00f00f00f00f),
                    (4, 0x10c30c30c30c30c3), (2, 0x1249249249249249)):
        v = (v | (v << s)) & mask
    return v


def _add_runs(out, ids, values):
    """out[ids] += values (a column each), ids ascending: differences of one running sum per column (atomics on few
    addresses would queue)."""
    if ids.numel() == 0:
        return
    end = torch.ones(ids.numel(), dtype=torch.bool, device=ids.device)
    end[:-1] = ids[1:] != ids[:-1]
    at = torch.nonzero(end).flatten()
    to = ids[at]
    for k, v in enumerate(values):
        c = torch.cumsum(v, 0)[at]
        c[1:] -= c[:-1].clone()
        out[to, k] += c


class _Tree64:
    """Key-prefix octree of float64 bodies: nodes level by level, a node's children consecutive.  A cell of level L
    holds the bodies that share L key digits (two or more; the root always); a body alone is a leaf."""

    def __init__(self, p, m):
        n = p.shape[0]
        lo, hi = p.amin(0), p.amax(0)
        span = (hi - lo).max()
        q = ((2.0 ** LEVELS - 1) * (p - lo) / span).to(torch.int64) if n > 1 else torch.zeros_like(p, dtype=torch.int64)
        key = _spread(q[:, 0]) | (_spread(q[:, 1]) << 1) | (_spread(q[:, 2]) << 2)
        key, self.perm = torch.sort(key, stable=True)
        self.p, self.m = p[self.perm], m[self.perm]
        self.n = n
        side0 = float(span) * 2.0 ** LEVELS / (2.0 ** LEVELS - 1)
        mp = torch.cat([self.m[:, None], self.m[:, None] * self.p], 1)
        dev = p.device
        level = [(torch.zeros(1, dtype=torch.int64, device=dev), torch.full((1,), n, device=dev))]
        sums, sides, first, count, body, self.parent = [mp.sum(0, keepdim=True)], [side0], [], [], [], [None]
        base = 0
        inside = torch.ones(n, dtype=torch.bool, device=dev)   # bodies inside a cell of the current level
        cell_of = torch.zeros(n, dtype=torch.int64, device=dev)  # that cell, counted from the level's first node
        body.append(torch.full((1,), -1, dtype=torch.int64, device=dev))
        for L in range(1, LEVELS + 2):
            nodes = level[-1][0].numel()
            idx = torch.nonzero(inside).flatten()
            if idx.numel() == 0:
                first.append(torch.zeros(nodes, dtype=torch.int64, device=dev))
                count.append(torch.zeros(nodes, dtype=torch.int64, device=dev))
                break
            par = cell_of[idx]
            new = torch.ones(idx.numel(), dtype=torch.bool, device=dev)
            if L <= LEVELS:
                pre = key[idx] >> (3 * (LEVELS - L))
                new[1:] = (pre[1:] != pre[:-1]) | (par[1:] != par[:-1])
            run = torch.cumsum(new, 0) - 1
            k = int(run[-1]) + 1
            start = idx[new]
            cnt = torch.bincount(run, minlength=k)
            s = torch.zeros(k, 4, dtype=torch.float64, device=dev)
            _add_runs(s, run, mp[idx].unbind(1))
            pn = par[new]
            nc = torch.bincount(pn, minlength=nodes)
            first.append(torch.cumsum(nc, 0) - nc + base + nodes)
            count.append(nc)
            self.parent.append(pn + base)
            base += nodes
            level.append((start, cnt))
            sums.append(s)
            sides.append(side0 * 0.5 ** L)
            body.append(torch.where(cnt == 1, start, -1))
            keep = cnt[run] > 1
            inside = torch.zeros(n, dtype=torch.bool, device=dev)
            inside[idx[keep]] = True
            cell_of = torch.zeros(n, dtype=torch.int64, device=dev)
            cell_of[idx] = run
        else:
            first.append(torch.zeros(level[-1][0].numel(), dtype=torch.int64, device=dev))
            count.append(torch.zeros(level[-1][0].numel(), dtype=torch.int64, device=dev))
        self.sizes = [lv[0].numel() for lv in level]
        self.first, self.count = torch.cat(first), torch.cat(count)
        self.body = torch.cat(body)
        s = torch.cat(sums)
        self.M, self.X = s[:, 0], s[:, 1:] / s[:, :1]
        self.side = torch.cat([torch.full((k,), v, dtype=torch.float64, device=dev) for k, v in zip(self.sizes, sides)])
        leaf = self.body >= 0
        self.side[leaf] = 0.0
        self.X[leaf] = self.p[self.body[leaf]]
        self.M[leaf] = self.m[self.body[leaf]]
        self.count[leaf] = 0

    def pairs(self, theta, chunk=32768):
        """(body, node, X_node - x_body) of every interaction, in portions; bodies by sorted position."""
        for a in range(0, self.n, chunk):
            i = torch.arange(a, min(self.n, a + chunk), device=self.p.device)
            node = torch.zeros_like(i)
            while i.numel():
                d = self.X[node] - self.p[i]
                take = self.side[node] < theta * d.square().sum(1).sqrt()
                take |= self.body[node] >= 0
                yield i[take], node[take], d[take]
                i, node = i[~take], node[~take]
                k = self.count[node]
                at = torch.repeat_interleave(torch.cumsum(k, 0) - k, k)
                i = torch.repeat_interleave(i, k)
                node = torch.repeat_interleave(self.first[node], k) + torch.arange(i.numel(), device=i.device) - at

    def accel(self, theta, eps2):
        acc = torch.zeros(self.n, 3, dtype=torch.float64, device=self.p.device)
        for i, node, d in self.pairs(theta):
            r2 = d.square().sum(1)
            w = torch.where(r2 > 0, self.M[node] * (r2 + eps2) ** -1.5, 0.0)
            _add_runs(acc, i, [w * d[:, k] for k in range(3)])
        out = torch.empty_like(acc)
        out[self.perm] = acc
        return out

    def vjp(self, theta, eps2, u):
        """dL/dx and dL/dm for u = dL/da, the interaction lists held."""
        u = u[self.perm]
        gx = torch.zeros(self.n, 3, dtype=torch.float64, device=self.p.device)
        G = torch.zeros(self.M.numel(), 4, dtype=torch.float64, device=self.p.device)
        for i, node, d in self.pairs(theta):
            other = self.body[node] != i
            i, node, d = i[other], node[other], d[other]
            r2 = d.square().sum(1) + eps2
            s = torch.where(r2 > 0, r2 ** -1.5, 0.0)
            ui = u[i]
            ud = (ui * d).sum(1)
            h = (self.M[node] * s)[:, None] * (ui - (3 * ud / torch.where(r2 > 0, r2, 1.0))[:, None] * d)
            _add_runs(gx, i, (-h).unbind(1))
            node, order = torch.sort(node)
            _add_runs(G, node, [h[order, k] for k in range(3)] + [(s * ud)[order]])
        # a cell's terms go down to its bodies through its centre of mass
        A = G[:, :3] / self.M[:, None]
        B = G[:, 3] - (A * self.X).sum(1)
        leaf = self.body >= 0
        A[leaf] = 0.0
        B[leaf] = 0.0
        lo = 1
        for pn, k in zip(self.parent[1:], self.sizes[1:]):
            A[lo:lo + k] += A[pn]
            B[lo:lo + k] += B[pn]
            lo += k
        at = self.body[leaf]
        gm = torch.zeros(self.n, dtype=torch.float64, device=self.p.device)
        gx.index_add_(0, at, G[leaf, :3] + self.m[at][:, None] * A[leaf])
        gm.index_add_(0, at, G[leaf, 3] + B[leaf] + (A[leaf] * self.p[at]).sum(1))
        ox, om = torch.empty_like(gx), torch.empty_like(gm)
        ox[self.perm], om[self.perm] = gx, gm
        return ox, om


def _f64(a):
    return torch.as_tensor(np.stack(a, 1) if isinstance(a, (list, tuple)) else a, device=DEV).double()


def _accel64(p, m, theta, eps2):
    if p.shape[0] < 2:
        return torch.zeros_like(p)
    return _Tree64(p, m).accel(theta, eps2)


def _moved(p, v, a):
    v = v + DT * a
    return p + DT * v, v


def _cols(*mats):
    return [m[:, k] for m in mats for k in range(3)]


def exact(case, seed):
    path = case["path"]
    if path == "sort":
        return None  # whole numbers
    if case.get("systems", 0) > 300 or work(case)["flops"] > 2e11:
        return None  # too long in 64 bits
    eps2 = float(np.float32(case.get("softening", 1e-3))) ** 2
    if path == "batch":
        arrs, sizes, thetas = _ensemble(case, seed)
        p, v, m = _f64(arrs[:3]), _f64(arrs[3:6]), _f64(arrs[6])
        off = np.concatenate([[0], np.cumsum(sizes)])
        a = torch.cat([_accel64(p[off[j]:off[j + 1]], m[off[j]:off[j + 1]], float(thetas[j]), eps2)
                       for j in range(len(sizes))])
        return dict(zip(STATE, _cols(*_moved(p, v, a), a)))
    arrs = _bodies(case, seed)
    theta = float(np.float32(case["theta"]))
    body, stars = _split_suns(case, arrs)
    p, v, m = _f64(body[:3]), _f64(body[3:6]), _f64(body[6])
    if path in ("step", "accel"):
        a = _accel64(p, m, theta, eps2)
        if path == "accel":
            return {"ax": a[:, 0], "ay": a[:, 1], "az": a[:, 2], "sorted": None}
        out = {}
        if stars:
            sp, sv, sm = _f64(stars[:3]), _f64(stars[3:6]), _f64(stars[6])
            sa = torch.zeros_like(sp)
            for j in range(sp.shape[0]):
                d = sp[j] - p
                w = ((d.square().sum(1) + eps2) ** -1.5)[:, None] * d
                a = a + sm[j] * w
                sa[j] = -(m[:, None] * w).sum(0)
                for k in range(sp.shape[0]):
                    if k != j:
                        e = sp[k] - sp[j]
                        sa[j] += sm[k] * (e.square().sum() + eps2) ** -1.5 * e
            out.update(zip(("sx", "sy", "sz", "svx", "svy", "svz", "sax", "say", "saz"),
                           _cols(*_moved(sp, sv, sa), sa)))
        out.update(zip(STATE, _cols(*_moved(p, v, a), a)))
        return out
    if path in ("vjp", "grad"):
        t = _Tree64(p, m)
        gx, gm = t.vjp(theta, eps2, torch.stack(_cotangents(case["n"], seed), 1).double())
        grads = _cols(gx) + [gm]
        return grads if path == "vjp" else _cols(t.accel(theta, eps2)) + grads
    tgt = _f64(_bodies(case, seed + 500)[:3])
    trees = []
    for _ in range(case["steps"]):
        trees.append(_Tree64(p, m))
        p, v = _moved(p, v, trees[-1].accel(theta, eps2))
    loss = (p - tgt).square().mean(0).sum()
    lx, lv, lm = 2.0 * (p - tgt) / case["n"], torch.zeros_like(p), torch.zeros_like(m)
    for t in reversed(trees):
        lv = lv + DT * lx
        gx, gm = t.vjp(theta, eps2, lv)
        lx, lm = lx + DT * gx, lm + DT * gm
    return [loss] + _cols(p, v) + _cols(lx, lv) + [lm]
