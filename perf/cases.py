"""Workloads of the closed-shell (T) library, through its Python entry points.

Each case is one thing that a user's program does after a CCSD calculation:

  run     CCSDTriples.run: E[4], E[5] and every task's contribution, all tasks in one
          graph-captured launch (FP64 and mixed precision);
  tasks   CCSDTriples.run_tasks: a subset of the tasks, as a resumed or sharded run or
          the benchmark's samples do;
  dropin  the per-task path of the unchanged fused driver: gather_task into the packed
          buffers, then fully_fused_ccsd_t_gpu on them, for each task of a share;
  gather  gather_task alone (the operand blocks of the per-task path);
  expand  expand_amplitudes: dense spin-orbital T1 / T2 for code that keeps them;
  train   CostModel.train: the schedule's cost model on timed tasks.

Inputs: orbital energies, T1, T2 = (ai|bj)/D (MP2-like) and the two-electron integrals
from Cholesky vectors of random sign and magnitude, uploaded with upload_cholesky.  All
sizes are those of the repository's tests and benchmark, or lie between them.
"""
import functools

import numpy as np
import torch

import exachem_amd as xt

NCHOL = 48  # Cholesky vectors of the inputs: enough for full-rank-looking integrals, quick to ship
NAMES = ("d1_t2", "d1_v2", "d2_t2", "d2_v2", "s1_t1", "s1_v2")


def _case(name, op, O, V, occ, vir, tile_seed=20241202, prec="fp64", tasks=0, restricted=True,
          schedule="driver"):
    return dict(name=name, op=op, O=O, V=V, occ_lo=occ[0], occ_hi=occ[1], vir_lo=vir[0],
                vir_hi=vir[1], tile_seed=tile_seed, prec=prec, tasks=tasks, restricted=restricted,
                schedule=schedule)


def listed():
    return [
        # a small molecule, every spin block kept: one launch's fixed costs
        _case("run_fp64_o7_v22", "run", 7, 22, (3, 4), (5, 9), restricted=False),
        # the reference's CPU-sized case (uniform tiles 8 / 16) in both precisions
        _case("run_fp64_o8_v48", "run", 8, 48, (8, 8), (16, 16)),
        _case("run_mixed_o8_v48", "run", 8, 48, (8, 8), (16, 16), prec="mixed"),
        # ordinary whole calculations, uneven tiles
        _case("run_fp64_o16_v96", "run", 16, 96, (4, 12), (16, 40), tile_seed=7),
        _case("run_mixed_o20_v120", "run", 20, 120, (6, 20), (16, 48), tile_seed=7, prec="mixed",
              schedule="analytic"),
        # a share of a large calculation, uniform tiles 16 / 32
        _case("tasks_mixed_o40_v300", "tasks", 40, 300, (16, 16), (32, 32), prec="mixed", tasks=24),
        # the same size with uneven tiles in FP64
        _case("tasks_fp64_o40_v300", "tasks", 40, 300, (6, 20), (16, 48), tasks=12),
        # a share of the benchmark's workload: uneven tiles, mixed precision
        _case("tasks_mixed_o48_v384", "tasks", 48, 384, (6, 20), (16, 48), prec="mixed", tasks=40),
        # the unchanged driver's per-task loop: gather, fused kernel, partials
        _case("dropin_o24_v160", "dropin", 24, 160, (6, 20), (16, 48), tile_seed=7, tasks=6),
        # operand blocks alone
        _case("gather_o40_v300", "gather", 40, 300, (6, 20), (16, 48), tasks=6),
        # dense spin-orbital amplitudes
        _case("expand_o20_v120", "expand", 20, 120, (6, 20), (16, 48)),
        # the schedule's cost model: 256 tasks timed at both precisions
        dict(name="train_512x200", op="train", n=512, steps=200),
    ]


def _log_int(rng, lo, hi):
    return int(round(float(np.exp(rng.uniform(np.log(lo), np.log(hi))))))


def draw(rng):
    op = rng.choice(["run", "run", "run", "tasks", "tasks", "tasks", "dropin", "gather", "expand",
                     "train"])
    if op == "train":
        return dict(op="train", n=_log_int(rng, 64, 640), steps=_log_int(rng, 20, 200))
    prec = rng.choice(["fp64", "mixed"])
    schedule = rng.choice(["driver", "analytic"])
    seed = rng.randrange(1 << 20)
    if op == "run":
        O = _log_int(rng, 5, 16 if prec == "mixed" else 13)
        V = int(O * rng.uniform(3.0, 6.0)) + 1
        occ = (rng.randint(2, 4), rng.randint(5, 12))
        vir = (rng.randint(5, 14), rng.randint(16, 32))
        c = _case("", op, O, V, occ, vir, seed, prec, 0, rng.random() < 0.85, schedule)
    elif op == "tasks":
        O = _log_int(rng, 16, 40)
        V = int(O * rng.uniform(4.0, 7.5))
        occ, vir = ((6, 20), (16, 48)) if rng.random() < 0.7 else ((16, 16), (32, 32))
        c = _case("", op, O, V, occ, vir, seed, prec, rng.randint(1, 8 if prec == "fp64" else 20),
                  True, schedule)
    else:
        O = _log_int(rng, 8, 20 if op == "expand" else 24)
        V = int(O * rng.uniform(3.0, 6.0))
        n = 0 if op == "expand" else rng.randint(1, 6)
        c = _case("", op, O, V, (rng.randint(3, 6), rng.randint(8, 20)),
                  (rng.randint(6, 16), rng.randint(20, 48)), seed, "fp64", n)
    del c["name"]
    return c


# ------------------------------------------------------------------ tilings and tasks
def _tiling(c):
    occ, vir = (c["occ_lo"], c["occ_hi"]), (c["vir_lo"], c["vir_hi"])
    if occ[0] == occ[1] and vir[0] == vir[1]:
        return xt.Tiling.uniform(c["O"], c["V"], occ[0], vir[0])
    return xt.Tiling.uneven(c["O"], c["V"], occ, vir, seed=c["tile_seed"])


def _key(c):
    return tuple(sorted((k, v) for k, v in c.items() if k != "name"))


@functools.lru_cache(maxsize=64)
def _tasks(key):
    """(tiling, tiles[], spins[], tasks (n x 6), factors, which) of a case."""
    c = dict(key)
    t = _tiling(c)
    ctx = xt.CCSDTriples(-1)
    ctx.set_tiling(t, c["restricted"])
    tasks, fac = ctx.task_list()
    ctx.close()
    tiles, spins = t.spin_orbital()
    n = len(tasks)
    if c["tasks"]:
        rng = np.random.default_rng(c["tile_seed"] + 1)
        which = np.sort(rng.choice(n, min(c["tasks"], n), replace=False))
    else:
        which = np.arange(n)
    return t, np.array(tiles), np.array(spins), tasks, fac, which


def _slots(s):
    """Enabled (d1, d2, s1) equations of a task of tile spins s[6], from spin conservation."""
    n1 = n2 = n0 = 0
    for h in range(3):
        for p in range(3):
            n1 += s[3] + s[4] + s[5] - s[3 + p] - s[h] in (1, 2)
            n2 += s[0] + s[1] + s[2] - s[h] - s[3 + p] in (1, 2)
            n0 += s[h] == s[3 + p]
    return n1, n2, n0


def _unique(d, b):
    """Distinct elements of three positions of extents d on tiles b (equal tiles: i < j)."""
    if b[0] == b[1] == b[2]:
        return max(d[0] * (d[0] - 1) * (d[0] - 2) / 6.0, 1.0)
    if b[0] == b[1]:
        return d[0] * (d[0] - 1) / 2.0 * d[2]
    if b[1] == b[2]:
        return d[1] * (d[1] - 1) / 2.0 * d[0]
    return float(d[0] * d[1] * d[2])


# ------------------------------------------------------------------ inputs
def _inputs(c, seed):
    """Cholesky vectors and amplitudes on the GPU, FP64, from the seed alone."""
    O, V = c["O"], c["V"]
    n = O + V
    g = torch.Generator(device="cuda")
    g.manual_seed(1000 + seed)

    def normal(*shape):
        return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float64)

    L = normal(n, n, NCHOL)
    L = (L + L.transpose(0, 1)) * (0.5 * (0.05 / NCHOL ** 0.5) ** 0.5)
    eo = torch.sort(torch.rand(O, generator=g, device="cuda", dtype=torch.float64) * 1.7 - 2.0)[0]
    ev = torch.sort(torch.rand(V, generator=g, device="cuda", dtype=torch.float64) * 2.9 + 0.1)[0]
    t1 = 1e-3 * normal(V, O)
    vo = L[O:, :O].reshape(V * O, NCHOL)
    t2 = torch.empty(V, V, O, O, device="cuda", dtype=torch.float64)
    den = eo[:, None] + eo[None, :]
    for a in range(V):  # (ai|bj) of one a at a time, symmetrised below
        row = (L[O + a, :O] @ vo.T).reshape(O, V, O).permute(1, 0, 2)  # [b][i][j]
        t2[a] = row / (den[None] - (ev[a] + ev)[:, None, None])
    for a in range(V):
        t2[a, a] = 0.5 * (t2[a, a] + t2[a, a].T)
        t2[a + 1:, a] = t2[a, a + 1:].transpose(1, 2)
    return dict(eo=eo, ev=ev, t1=t1, t2=t2.contiguous(), L=L.contiguous())


def prepare(c, seed):
    if c["op"] == "train":
        rng = np.random.default_rng(seed)
        x = rng.uniform(0.1, 1.0, (c["n"], 7)).astype(np.float32)
        x[:, 6] = np.arange(c["n"]) % 2
        y = (0.8 * np.sin(3.0 * x[:, 0] + x[:, 3]) - x[:, 6] + 0.5 * x[:, 4] * x[:, 5]
             + 0.05 * rng.normal(size=c["n"])).astype(np.float32)
        m = xt.CostModel(0, seed=5)
        return dict(op="train", model=m, p0=_params0(seed), x=x, t=y, steps=c["steps"])
    t, tiles, spins, tasks, fac, which = _tasks(_key(c))
    s = _inputs(c, seed)
    ctx = xt.CCSDTriples(0)
    ctx.set_tiling(t, c["restricted"])
    ctx.upload_cholesky(*[s[k].cpu().numpy() for k in ("eo", "ev", "t1", "t2", "L")])
    prec = xt.PREC_MIXED if c["prec"] == "mixed" else xt.PREC_FP64
    st = dict(op=c["op"], ctx=ctx, which=which, prec=prec,
              sched=xt.SCHED_ANALYTIC if c["schedule"] == "analytic" else xt.SCHED_DRIVER)
    if c["op"] in ("run", "tasks"):
        ctx.prepare(prec)
        return st
    stream = torch.cuda.current_stream().cuda_stream
    st["stream"] = stream if stream else None
    if c["op"] == "expand":
        O, V = c["O"], c["V"]
        st["t1"] = torch.empty(2 * V, 2 * O, device="cuda", dtype=torch.float64)
        st["t2"] = torch.empty(2 * V, 2 * V, 2 * O, 2 * O, device="cuda", dtype=torch.float64)
        return st
    sz = ctx.packed_sizes()
    st["bufs"] = {n: torch.zeros(sz[n], device="cuda", dtype=torch.float64) for n in NAMES}
    st["ptrs"] = {n: st["bufs"][n].data_ptr() for n in NAMES}
    st["tasks"] = [[int(b) for b in tasks[k]] for k in which]
    if c["op"] == "dropin":
        st["max"] = {n: sz[n] // (9 if n.startswith("s1") else sz["max_" + n[:2]]) for n in NAMES}
        st["noab"], st["nvab"] = 2 * len(t.occ), 2 * len(t.vir)
        evl = torch.cat([s["eo"], s["eo"], s["ev"], s["ev"]])
        offs = np.concatenate([[0], np.cumsum(tiles)])
        st["evl"] = evl
        st["ev"] = [[evl.data_ptr() + 8 * int(offs[b]) for b in k] for k in st["tasks"]]
        st["dims"] = [[int(tiles[b]) for b in k] for k in st["tasks"]]
        st["nb"] = [int(np.prod([(d + 3) // 4 for d in dims])) for dims in st["dims"]]
        st["part"] = [torch.zeros(2 * nb, device="cuda", dtype=torch.float64) for nb in st["nb"]]
    return st


def run(st):
    op = st["op"]
    if op == "train":
        st["model"].set_params(st["p0"])
        hist = st["model"].train(st["x"], st["t"], st["steps"], 3e-3)
        return dict(hist=hist, params=st["model"].get_params())
    ctx = st["ctx"]
    if op == "run":
        r = ctx.run(precision=st["prec"], schedule=st["sched"], use_graph=1)
        return dict(e4=r["e4"], e5=r["e5"], partials=r["task_partials"])
    if op == "tasks":
        r = ctx.run_tasks(st["which"], precision=st["prec"], schedule=st["sched"], use_graph=1)
        return dict(e4=r["e4"], e5=r["e5"], partials=r["task_partials"])
    if op == "expand":
        ctx.expand_amplitudes(st["t1"].data_ptr(), st["t2"].data_ptr(), st["stream"])
        return dict(t1=st["t1"], t2=st["t2"])
    if op == "gather":
        for k in st["tasks"]:
            ctx.gather_task(k, st["ptrs"], st["stream"])
        return {n: st["bufs"][n] for n in NAMES}
    for k, dims, nb, ev, part in zip(st["tasks"], st["dims"], st["nb"], st["ev"], st["part"]):
        meta, _ = ctx.gather_task(k, st["ptrs"], st["stream"])
        xt.fully_fused_ccsd_t_gpu(st["stream"], nb, dims, [st["ptrs"][n] for n in NAMES], meta,
                                  st["noab"], st["nvab"], st["max"], ev, part.data_ptr())
    return list(st["part"])


# ------------------------------------------------------------------ required work
def work(c):
    if c["op"] == "train":
        # forward 7-64-64-1, backward of the same, Adam on 4,737 parameters
        per = 2.0 * (7 * 64 + 64 * 64 + 64)
        return dict(bytes=4.0 * (8 * c["n"] + 2 * 4737 + c["steps"]),
                    flops=c["steps"] * (3 * per * c["n"] + 12 * 4737))
    O, V = c["O"], c["V"]
    if c["op"] == "expand":
        return dict(bytes=8.0 * (16 * (V * O) ** 2 + 4 * V * O + (V * O) ** 2 + V * O),
                    flops=2.0 * (V * O) ** 2)
    t, tiles, spins, tasks, fac, which = _tasks(_key(c))
    flops = read = written = 0.0
    for k in which:
        b = tasks[k]
        d, s = tiles[b], spins[b]
        n1, n2, n0 = _slots(s)
        flops += 2.0 * _unique(d[:3], b[:3]) * _unique(d[3:], b[3:]) * (n1 * O + n2 * V + n0)
        t2, v2 = set(), set()
        for h in range(3):
            for p in range(3):
                hA, hB = [x for x in range(3) if x != h]
                pA, pB = [3 + x for x in range(3) if x != p]
                if s[pA] + s[pB] - s[h] in (1, 2):
                    t2.add((1, b[h], b[pA], b[pB], d[h] * d[pA] * d[pB] * O))
                    v2.add((1, b[hA], b[hB], b[3 + p], d[hA] * d[hB] * d[3 + p] * O))
                if s[hA] + s[hB] - s[3 + p] in (1, 2):
                    t2.add((2, b[hA], b[hB], b[3 + p], d[hA] * d[hB] * d[3 + p] * V))
                    v2.add((2, b[h], b[pA], b[pB], d[h] * d[pA] * d[pB] * V))
                if s[h] == s[3 + p]:
                    t2.add((0, b[h], b[3 + p], 0, d[h] * d[3 + p]))
                    v2.add((0, b[h], b[3 + p], 1, d[hA] * d[hB] * d[pA] * d[pB]))
        n = float(sum(x[-1] for x in t2) + sum(x[-1] for x in v2))
        read += n
        written += n if c["op"] == "gather" else 2.0 * np.prod(-(-d // 4)) if c["op"] == "dropin" else 2.0
    whole = float(V * V * O * O * 2 + O ** 3 * V + V ** 3 * O)
    if c["op"] == "gather":
        return dict(bytes=8.0 * (read + written), flops=read)
    if c["op"] == "dropin":  # packed operands written by the gather, read by the kernel
        return dict(bytes=8.0 * (3 * read + written), flops=flops)
    return dict(bytes=8.0 * (min(read, whole) + written), flops=flops)


# ------------------------------------------------------------------ values in 64 bits
def _params0(seed):
    rng = np.random.default_rng(seed + 77)
    p = np.zeros(4737, dtype=np.float32)
    p[:448] = rng.normal(0.0, (2.0 / 7) ** 0.5, 448)
    p[512:4608] = rng.normal(0.0, (2.0 / 64) ** 0.5, 4096)
    p[4672:4736] = rng.normal(0.0, (2.0 / 64) ** 0.5, 64)
    return p


def _exact_train(c, seed):
    st_x = np.random.default_rng(seed)
    x = st_x.uniform(0.1, 1.0, (c["n"], 7)).astype(np.float32)
    x[:, 6] = np.arange(c["n"]) % 2
    y = (0.8 * np.sin(3.0 * x[:, 0] + x[:, 3]) - x[:, 6] + 0.5 * x[:, 4] * x[:, 5]
         + 0.05 * st_x.normal(size=c["n"])).astype(np.float32)
    x, y = x.astype(np.float64), y.astype(np.float64)
    p = _params0(seed).astype(np.float64)
    m, v, hist = np.zeros_like(p), np.zeros_like(p), []
    n, lr = c["n"], float(np.float32(3e-3))
    b1, b2 = float(np.float32(0.9)), float(np.float32(0.999))
    for k in range(c["steps"]):
        w1, c1, w2, c2, w3, c3 = (p[:448].reshape(7, 64), p[448:512], p[512:4608].reshape(64, 64),
                                  p[4608:4672], p[4672:4736], p[4736])
        z1 = x @ w1 + c1
        a1 = np.maximum(z1, 0)
        z2 = a1 @ w2 + c2
        a2 = np.maximum(z2, 0)
        r = a2 @ w3 + c3 - y
        hist.append(np.mean(r * r))
        dy = 2 * r / n
        d2 = dy[:, None] * w3 * (z2 > 0)
        d1 = (d2 @ w2.T) * (z1 > 0)
        g = np.concatenate([(x.T @ d1).ravel(), d1.sum(0), (a1.T @ d2).ravel(), d2.sum(0),
                            a2.T @ dy, [dy.sum()]])
        m = b1 * m + (1 - b1) * g
        v = b2 * v + (1 - b2) * g * g
        p = p - lr * (m / (1 - b1 ** (k + 1))) / (np.sqrt(v / (1 - b2 ** (k + 1))) + 1e-8)
    return dict(hist=np.array(hist), params=p)


class _Blocks:
    """Spatial blocks of one calculation: t2 and (pq|rs) from the Cholesky vectors."""

    def __init__(self, c, seed):
        self.O, self.V = c["O"], c["V"]
        self.s = _inputs(c, seed)

    def eri(self, p, q, r, t):
        """(pq|rt) over index ranges of the orbitals, occupied first."""
        L = self.s["L"]
        a, b = L[p, q], L[r, t]
        na, nb = a.shape[:2], b.shape[:2]
        return (a.reshape(-1, NCHOL) @ b.reshape(-1, NCHOL).T).reshape(*na, *nb)


def _task_terms(B, dims, offs, s):
    """(t3 doubles, t3 singles, D) of a task as [h1, h2, h3, p4, p5, p6] tensors: the
    antisymmetrised connected triples and disconnected singles terms of spin-orbital (T)
    on tiles of spatial extents dims, first orbitals offs and spins s."""
    O, V, t2 = B.O, B.V, B.s["t2"]
    hr = [slice(offs[k], offs[k] + dims[k]) for k in range(3)]          # occupied ranges
    pr = [slice(offs[k], offs[k] + dims[k]) for k in range(3, 6)]       # virtual ranges
    pm = [slice(O + offs[k], O + offs[k] + dims[k]) for k in range(3, 6)]  # in the orbital list
    occ, vir = slice(0, O), slice(O, O + V)
    t3 = torch.zeros(*dims, device="cuda", dtype=torch.float64)
    s3 = torch.zeros_like(t3)

    def diff(on1, x, on2, y):
        return x() - y() if on1 and on2 else x() if on1 else -y() if on2 else None

    for h in range(3):
        hA, hB = [k for k in range(3) if k != h]
        for p in range(3):
            pA, pB = [k for k in range(3) if k != p]
            sg = (-1.0) ** (h + p)
            sH, sA, sB = s[h], s[hA], s[hB]
            sP, sC, sD = s[3 + p], s[3 + pA], s[3 + pB]
            left, right = [], []
            m = sC + sD - sH  # spin of the contracted occupied index
            if m in (1, 2):
                a = diff(sC == sH and sD == m, lambda: t2[pr[pA], pr[pB], hr[h]],
                         sC == m and sD == sH,
                         lambda: t2[pr[pB], pr[pA], hr[h]].transpose(0, 1))   # [pA][pB][h][m]
                b = diff(sA == m and sB == sP,
                         lambda: B.eri(hr[hA], occ, hr[hB], pm[p]).permute(0, 2, 3, 1),
                         sB == m and sA == sP,
                         lambda: B.eri(hr[hB], occ, hr[hA], pm[p]).permute(2, 0, 3, 1))
                if a is not None and b is not None:                          # b: [hA][hB][p][m]
                    left.append(-a.permute(2, 0, 1, 3).reshape(-1, O))
                    right.append(b.reshape(-1, O))
            e = sA + sB - sP  # spin of the contracted virtual index
            if e in (1, 2):
                a = diff(sH == sC and e == sD,
                         lambda: B.eri(hr[h], pm[pA], vir, pm[pB]).permute(0, 1, 3, 2),
                         sH == sD and e == sC,
                         lambda: B.eri(hr[h], pm[pB], vir, pm[pA]).permute(0, 3, 1, 2))
                b = diff(sP == sA and e == sB, lambda: t2[pr[p], :, hr[hA], hr[hB]].permute(2, 3, 0, 1),
                         sP == sB and e == sA,
                         lambda: t2[pr[p], :, hr[hB], hr[hA]].permute(3, 2, 0, 1))
                if a is not None and b is not None:
                    left.append(-a.reshape(-1, V))
                    right.append(b.reshape(-1, V))
            # [h, pA, pB, hA, hB, p] -> [h1, h2, h3, p4, p5, p6]
            at = {h: 0, 3 + pA: 1, 3 + pB: 2, hA: 3, hB: 4, 3 + p: 5}
            if left:
                w = torch.cat(left, 1).contiguous() @ torch.cat(right, 1).contiguous().T
                w = w.reshape(dims[h], dims[3 + pA], dims[3 + pB], dims[hA], dims[hB], dims[3 + p])
                t3 += sg * w.permute(*[at[k] for k in range(6)])
            if sH == sP:
                v = diff(sB == sD and sA == sC,
                         lambda: B.eri(hr[hB], pm[pB], hr[hA], pm[pA]).permute(3, 1, 2, 0),
                         sB == sC and sA == sD,
                         lambda: B.eri(hr[hB], pm[pA], hr[hA], pm[pB]).permute(1, 3, 2, 0))
                if v is not None:  # [pA][pB][hA][hB]
                    w = torch.einsum("ai,bcjk->iabcjk", B.s["t1"][pr[p], hr[h]], v)
                    at = {h: 0, 3 + p: 1, 3 + pA: 2, 3 + pB: 3, hA: 4, hB: 5}
                    s3 += sg * w.permute(*[at[k] for k in range(6)])
    eo, ev = B.s["eo"], B.s["ev"]
    dh = eo[hr[0], None, None] + eo[None, hr[1], None] + eo[None, None, hr[2]]
    dp = ev[pr[0], None, None] + ev[None, pr[1], None] + ev[None, None, pr[2]]
    D = dh[:, :, :, None, None, None] - dp[None, None, None]
    return t3, s3, D


def _block_sums(x):
    """Sums over blocks of 4 along every position, h1's block index fastest."""
    for k in range(6):
        pad = (-x.shape[k]) % 4
        if pad:
            shape = list(x.shape)
            shape[k] = pad
            x = torch.cat([x, x.new_zeros(shape)], k)
        x = x.unflatten(k, (x.shape[k] // 4, 4)).sum(k + 1)
    return x.permute(5, 4, 3, 2, 1, 0).reshape(-1)


def exact(c, seed):
    if c["op"] == "train":
        return _exact_train(c, seed)
    if c["op"] == "gather":
        return None  # copies and one subtraction per value
    if c["op"] == "expand":
        s = _inputs(c, seed)
        O, V = c["O"], c["V"]
        t1, t2 = s["t1"], s["t2"]
        e1 = torch.zeros(2, V, 2, O, device="cuda", dtype=torch.float64)
        e2 = torch.zeros(2, V, 2, V, 2, O, 2, O, device="cuda", dtype=torch.float64)
        for a in range(2):
            e1[a, :, a] = t1
            for b in range(2):
                if a == b:
                    e2[a, :, a, :, a, :, a] = t2 - t2.transpose(2, 3)
                else:
                    e2[a, :, b, :, a, :, b] = t2
                    e2[a, :, b, :, b, :, a] = -t2.transpose(2, 3)
        return dict(t1=e1.reshape(2 * V, 2 * O), t2=e2.reshape(2 * V, 2 * V, 2 * O, 2 * O))
    t, tiles, spins, tasks, fac, which = _tasks(_key(c))
    off = np.concatenate([[0], np.cumsum(tiles)[:-1]])
    first = np.where(np.arange(len(tiles)) < 2 * len(t.occ), off % c["O"], (off - 2 * c["O"]) % c["V"])
    B = _Blocks(c, seed)
    part, blocks = [], []
    for k in which:
        b = tasks[k]
        t3, s3, D = _task_terms(B, [int(x) for x in tiles[b]], [int(x) for x in first[b]],
                                [int(x) for x in spins[b]])
        w = t3 / D
        if c["op"] == "dropin":
            e4 = w * t3
            blocks.append(torch.cat([_block_sums(e4), _block_sums(e4 + w * s3)]))
        else:
            e4 = torch.dot(w.reshape(-1), t3.reshape(-1))
            e5 = e4 + torch.dot(w.reshape(-1), s3.reshape(-1))
            part.append([fac[k] * float(e4), fac[k] * float(e5)])
    if c["op"] == "dropin":
        return blocks
    part = np.array(part)
    return dict(e4=float(part[:, 0].sum()), e5=float(part[:, 1].sum()), partials=part)
