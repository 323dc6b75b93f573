"""The work that programs have this package do, as cases that can be timed: dense Evals, dense plans, kernel
matrices, batches of near-field blocks, the near-field operator and near lists, from calls of a few microseconds
to the largest direct sum of the benchmark.

listed() names the cases, draw() gives others of the same ranges, prepare() makes what a program holds before the
call (torch tensors on the GPU, plans), run() is one pass through the package's functions, work() counts what a
pass cannot do without, and exact() gives the values in plain torch, in 64 bits.  Sizes (numbers of points and
blocks, points per block) belong to a case; positions, normals and densities come from the seed.

Programs hand device memory over as torch tensors on one stream of their own.  A mixed-precision caller goes on in
single precision, which is what that path's sums are worth.
"""
import ctypes
import math

import numpy as np
import torch

import sctl_amd as S

F64 = torch.float64
KERNELS = {"Laplace3D_FxU": S.LAPLACE3D_FXU, "Laplace3D_DxU": S.LAPLACE3D_DXU, "Laplace3D_FxdU": S.LAPLACE3D_FXDU,
           "Stokes3D_FxU": S.STOKES3D_FXU, "Stokes3D_DxU": S.STOKES3D_DXU, "Helmholtz3D_FxU": S.HELMHOLTZ3D_FXU}
# densities per source, values per target, normal words per source, flop per pair (FMA = 2, rsqrt = 1)
DIMS = {"Laplace3D_FxU": (1, 1, 0, 11), "Laplace3D_DxU": (1, 1, 3, 19), "Laplace3D_FxdU": (1, 3, 0, 17),
        "Stokes3D_FxU": (3, 3, 0, 29), "Stokes3D_DxU": (3, 3, 3, 30), "Helmholtz3D_FxU": (2, 2, 0, 40)}
WAVENUMBER = 3.0


def listed():
    return [
        # A C++ or numpy caller's Eval on host arrays, at the size of one element against a few thousand points:
        # copies, allocations and launches, little arithmetic.
        dict(name="eval_host_small", kind="eval_host", kernel="Laplace3D_FxU", nt=2000, ns=3000, where="cube",
             precision="fp64"),
        # The far field of a small GMRES solve: one matrix-free product with resident geometry per iteration.
        dict(name="dense_plan_small", kind="dense_plan", kernel="Laplace3D_DxU", nt=2503, ns=3001, where="sphere",
             precision="fp64"),
        # 20 000 particles on 20 000 targets, to seven digits.
        dict(name="eval_cube_20k_mixed", kind="eval", kernel="Laplace3D_FxU", nt=20000, ns=20000, where="cube",
             precision="mixed"),
        # The largest direct sum: 2^20 surface sources on 2^20 volume targets.
        dict(name="eval_sphere_1M_mixed", kind="eval", kernel="Laplace3D_FxU", nt=1 << 20, ns=1 << 20,
             where="sphere", precision="mixed"),
        # A double layer in full precision at an ordinary, odd size.
        dict(name="eval_dxu_130k_fp64", kind="eval", kernel="Laplace3D_DxU", nt=100003, ns=130001, where="sphere",
             precision="fp64"),
        # Clustered Stokeslets (suspensions), to seven digits.
        dict(name="eval_stokes_150k_mixed", kind="eval", kernel="Stokes3D_FxU", nt=131072, ns=150001,
             where="clusters", precision="mixed"),
        # A dense matrix for a direct solver or a preconditioner block.
        dict(name="matrix_stokes_2k", kind="matrix", kernel="Stokes3D_FxU", nt=2003, ns=3001, where="cube"),
        # The direct part of a boundary integral's near field: thousands of uneven blocks in one call.
        dict(name="blocks_dxu_4096_fp64", kind="blocks", kernel="Laplace3D_DxU", blocks=4096, precision="fp64"),
        dict(name="blocks_stokes_2048_mixed", kind="blocks", kernel="Stokes3D_DxU", blocks=2048, precision="mixed"),
        # Setting up the near-field corrections: the direct part is taken out of the singular quadrature's matrices.
        dict(name="near_subtract_dxu_512", kind="near_subtract", kernel="Laplace3D_DxU", blocks=512),
        # Applying the stored near-field corrections once per GMRES iteration.
        dict(name="near_interac_dxu_512", kind="near_interac", kernel="Laplace3D_DxU", blocks=512),
        # Finding each element's near targets when a geometry moves.
        dict(name="near_list_2048", kind="near_list", elements=2048, nt=500009),
    ]


def draw(rng):
    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["eval_host", "dense_plan", "eval", "eval", "eval", "eval", "matrix", "blocks", "blocks",
                       "near_subtract", "near_interac", "near_list"])
    kernel = rng.choice(sorted(KERNELS))
    where = rng.choice(["cube", "sphere", "clusters"])
    precision = rng.choice(["fp64", "mixed"])
    if kind in ("eval_host", "dense_plan"):
        return dict(kind=kind, kernel=kernel, nt=size(200, 30000), ns=size(200, 30000), where=where,
                    precision=precision)
    if kind == "eval":
        return dict(kind=kind, kernel=kernel, nt=size(2000, 300000), ns=size(2000, 300000), where=where,
                    precision=precision)
    if kind == "matrix":
        return dict(kind=kind, kernel=kernel, nt=size(300, 4000), ns=size(300, 4000), where=where)
    if kind == "blocks":
        return dict(kind=kind, kernel=kernel, blocks=size(64, 4096), precision=precision)
    if kind == "near_list":
        return dict(kind=kind, elements=size(64, 2048), nt=size(10000, 500000))
    kernel = rng.choice(["Laplace3D_FxU", "Laplace3D_DxU", "Stokes3D_FxU", "Stokes3D_DxU"])
    return dict(kind=kind, kernel=kernel, blocks=size(16, 500 if kernel.startswith("Laplace") else 60))


# ------------------------------------------------------------------ inputs
def uniform(g, n, lo=0.0, hi=1.0):
    return torch.rand(n, generator=g, dtype=F64, device="cuda") * (hi - lo) + lo


def normal(g, n):
    return torch.randn(n, generator=g, dtype=F64, device="cuda")


def directions(g, n):
    x = normal(g, 3 * n).view(n, 3)
    return x / x.norm(dim=1, keepdim=True)


def points(case, seed):
    """(xt, xs, normals, densities) of a dense case, flat.
    cube      both sets uniform in the unit cube
    sphere    sources on the unit sphere, targets in the shell 1.05 < r < 2 around it
    clusters  both sets from 64 Gaussian clusters of width 0.02 in the unit cube"""
    g = torch.Generator(device="cuda").manual_seed(seed)
    nt, ns, k0 = case["nt"], case["ns"], DIMS[case["kernel"]][0]
    nrm = directions(g, ns)
    if case["where"] == "cube":
        xt, xs, f = uniform(g, 3 * nt), uniform(g, 3 * ns), uniform(g, k0 * ns, -1.0, 1.0)
    elif case["where"] == "sphere":
        r = (uniform(g, nt) * (2.0 ** 3 - 1.05 ** 3) + 1.05 ** 3) ** (1.0 / 3.0)
        xt, xs, f = directions(g, nt) * r[:, None], nrm.clone(), normal(g, k0 * ns)
    else:
        c = uniform(g, 3 * 64).view(64, 3)
        xt, xs = (c[torch.randint(0, 64, (n,), generator=g, device="cuda")] + 0.02 * normal(g, 3 * n).view(n, 3)
                  for n in (nt, ns))
        f = normal(g, k0 * ns)
    return xt.reshape(-1).contiguous(), xs.reshape(-1).contiguous(), nrm.reshape(-1).contiguous(), f.contiguous()


def starts(cnt):
    return np.concatenate([[0], np.cumsum(cnt)[:-1]]).astype(np.int64)


def block_sizes(blocks):
    """Sources (p^2 nodes of a patch) and targets of each block: p^2 log-uniform in 64..4096, targets in 16..2048."""
    r = np.random.RandomState(blocks)
    p = np.clip(np.rint(np.exp(r.uniform(math.log(8), math.log(64), blocks))), 8, 64).astype(np.int64)
    nt = np.rint(np.exp(r.uniform(math.log(16), math.log(2048), blocks))).astype(np.int64)
    return p, nt


def patches(n):
    """How a torus is cut into about n patches along its two angles."""
    nv = max(1, int(round(math.sqrt(n / 2.0))))
    return -(-n // nv), nv


def torus(u, v, R=1.0, r=0.3):
    cv, sv, cu, su = torch.cos(v), torch.sin(v), torch.cos(u), torch.sin(u)
    return (torch.stack([(R + r * cv) * cu, (R + r * cv) * su, r * sv], 1),
            torch.stack([cv * cu, cv * su, sv], 1))


def patch_nodes(p, turn):
    """Nodes (Gauss-Legendre grids of p[e] x p[e] points) and normals of the patches, the torus turned by an angle."""
    nu, nv = patches(p.size)
    rule = np.zeros((int(p.max()) + 1, int(p.max())))
    for q in np.unique(p):
        rule[q, :q] = (np.polynomial.legendre.leggauss(int(q))[0] + 1) / 2
    rule = torch.from_numpy(rule).cuda()
    cnt = torch.from_numpy(p * p).cuda()
    e = torch.repeat_interleave(torch.arange(p.size, device="cuda"), cnt)
    k = torch.arange(int((p * p).sum()), device="cuda") - torch.from_numpy(starts(p * p)).cuda()[e]
    pe = torch.from_numpy(p).cuda()[e]
    u = ((e // nv) + rule[pe, k // pe]) * (2 * math.pi / nu) + turn
    v = ((e % nv) + rule[pe, k % pe]) * (2 * math.pi / nv) + turn
    return torus(u, v)


def near_points(g, p, nt, turn, off=0.05):
    """nt[e] targets within `off` of each patch's surface."""
    nu, nv = patches(p.size)
    e = torch.repeat_interleave(torch.arange(p.size, device="cuda"), torch.from_numpy(nt).cuda())
    n = e.numel()
    x, m = torus(((e // nv) + uniform(g, n)) * (2 * math.pi / nu) + turn, ((e % nv) + uniform(g, n)) * (2 * math.pi / nv) + turn)
    return x + uniform(g, n, -off, off)[:, None] * m, m


def block_inputs(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    p, nt = block_sizes(case["blocks"])
    turn = float(uniform(g, 1))
    xs, xn = patch_nodes(p, turn)
    xt, tn = near_points(g, p, nt, turn)
    f = normal(g, DIMS[case["kernel"]][0] * xs.shape[0])
    w = uniform(g, xs.shape[0], 0.5, 1.5) * 1e-3
    return p, nt, *(a.reshape(-1).contiguous() for a in (xt, tn, xs, xn, f, w))


def matrices(case, seed, n):
    """The stored near-field corrections of a case's blocks, n entries."""
    return uniform(torch.Generator(device="cuda").manual_seed(seed + 7919), n, -1.0, 1.0)


def near_pairs(nt):
    """Near targets of each element of a stored near field: nt[e] consecutive targets around the element's place,
    so that a target is near about four elements.  Returns (number of targets, target of each pair)."""
    n = max(1, int(nt.sum()) // 4)
    first = np.clip((starts(nt) + nt // 2) // 4 - nt // 2, 0, np.maximum(n - nt, 0))
    pair = np.repeat(first, nt) + np.arange(int(nt.sum())) - np.repeat(starts(nt), nt)
    return n, pair % n


def list_inputs(case, seed):
    """Elements (nodes, radius of each node) and targets of a near-list build: a body that moves as a whole, so that
    the seed gives its place (a rotation and a shift) and the order of the targets, and the case its shape."""
    g = torch.Generator(device="cuda").manual_seed(case["elements"])
    r = np.random.RandomState(case["elements"])
    p = r.randint(8, 33, case["elements"]).astype(np.int64)
    share = r.multinomial(case["nt"], np.full(case["elements"], 1.0 / case["elements"])).astype(np.int64)
    xs, _ = patch_nodes(p, 0.0)
    xt, _ = near_points(g, p, share, 0.0)
    rad = uniform(g, xs.shape[0], 0.03, 0.05)
    g.manual_seed(seed)
    turn = torch.linalg.qr(normal(g, 9).view(3, 3).cpu())[0].cuda()
    shift = uniform(g, 3, -1.0, 1.0)
    xs, xt = xs @ turn + shift, xt[torch.randperm(xt.shape[0], generator=g, device="cuda")] @ turn + shift
    return p, xt.reshape(-1).contiguous(), xs.reshape(-1).contiguous(), rad


# ------------------------------------------------------------------ running
class View(S.DeviceArray):
    """A torch tensor's memory as the package's functions take it (the tensor keeps it)."""

    def __init__(self, t):
        self.t, self.shape, self.nbytes = t, (t.numel(),), t.numel() * t.element_size()
        self.dtype, self.ptr = None, ctypes.c_void_p(t.data_ptr())

    def free(self):
        pass


_stream = None


def stream():
    """The program's own stream."""
    global _stream
    if _stream is None:
        _stream = torch.cuda.Stream()
    return _stream


def prepare(case, seed):
    kind = case["kind"]
    s = dict(case=case)
    if kind == "near_list":
        p, xt, xs, rad = list_inputs(case, seed)
        s.update(xt=View(xt), xs=View(xs), rad=View(rad), cnt=View(torch.from_numpy(p * p).cuda()),
                 dsp=View(torch.from_numpy(starts(p * p)).cuda()), ne=p.size)
        torch.cuda.synchronize()
        return s
    name = case["kernel"]
    kernel, (k0, k1, nd, _) = KERNELS[name], DIMS[name]
    ctx = WAVENUMBER if name.startswith("Helmholtz") else None
    prec = S.MIXED if case.get("precision") == "mixed" else S.FP64
    s.update(kernel=kernel, ctx=ctx, prec=prec, k1=k1)
    if kind in ("blocks", "near_subtract", "near_interac"):
        p, nt, xt, tn, xs, xn, f, w = block_inputs(case, seed)
        cnt = p * p
        plan = S.Plan(kernel, starts(nt), nt, starts(cnt), cnt, int(nt.sum()), int(cnt.sum()),
                      precision=prec, ctx=ctx)
        torch.cuda.synchronize()
        plan.set_geometry(View(xt), View(xs), View(xn) if nd else None)
        S.synchronize()
        s.update(plan=plan, f=View(f), w=View(w), n=int(nt.sum()))
        if kind != "blocks":
            s["K"] = View(matrices(case, seed, plan.near_layout()))
        if kind == "near_interac":
            s["ntrg"], pair = near_pairs(nt)
            tc = np.bincount(pair, minlength=s["ntrg"]).astype(np.int64)
            s.update(tc=View(torch.from_numpy(tc).cuda()), td=View(torch.from_numpy(starts(tc)).cuda()),
                     sc=View(torch.from_numpy(np.argsort(pair, kind="stable")).cuda()))
        torch.cuda.synchronize()
        return s
    xt, xs, xn, f = points(case, seed)
    s.update(nt=case["nt"], ns=case["ns"])
    if kind == "eval_host":
        s.update({k: v.cpu().numpy() for k, v in dict(xt=xt, xs=xs, xn=xn, f=f).items()})
        s["op"] = S.GenericKernel(kernel)
        s["op"].SetCtxPtr(ctx)
    else:
        s.update(xt=View(xt), xs=View(xs), xn=View(xn), f=View(f))
    torch.cuda.synchronize()
    if kind == "dense_plan":
        s["plan"] = S.DensePlan(kernel, s["xt"], s["xs"], s["xn"], precision=prec, ctx=ctx)
    if kind == "matrix":
        s["M"] = torch.empty(case["ns"] * k0, case["nt"] * k1, dtype=F64, device="cuda")
    torch.cuda.synchronize()
    return s


def result(s, v):
    return v.float() if s["prec"] == S.MIXED else v


def run(s):
    kind = s["case"]["kind"]
    if kind == "eval_host":
        v = s["op"].Eval(None, s["xt"], s["xs"], s["xn"], s["f"], precision=s["prec"])
        return v.astype(np.float32) if s["prec"] == S.MIXED else v
    st = stream()
    h = st.cuda_stream
    with torch.cuda.stream(st):
        if kind == "eval":
            v = torch.zeros(s["nt"] * s["k1"], dtype=F64, device="cuda")
            S.eval(s["kernel"], s["xt"], s["xs"], s["xn"], s["f"], View(v), precision=s["prec"], stream=h,
                   ctx=s["ctx"])
            return result(s, v)
        if kind == "dense_plan":
            v = torch.zeros(s["nt"] * s["k1"], dtype=F64, device="cuda")
            s["plan"].apply(s["f"], View(v), stream=h)
            return result(s, v)
        if kind == "matrix":
            S.kernel_matrix(s["kernel"], s["xt"], s["xs"], s["xn"], M=View(s["M"]), stream=h, ctx=s["ctx"])
            return s["M"]
        if kind == "blocks":
            v = torch.zeros(s["n"] * s["k1"], dtype=F64, device="cuda")
            s["plan"].apply(s["f"], View(v), stream=h)
            return result(s, v)
        if kind == "near_subtract":
            s["plan"].near_matrix(s["K"], s["w"], None, S.NEAR_SUBTRACT, stream=h)
            return s["K"].t
        if kind == "near_interac":
            un = torch.empty(s["n"] * s["k1"], dtype=F64, device="cuda")
            u = torch.zeros(s["ntrg"] * s["k1"], dtype=F64, device="cuda")
            s["plan"].near_gemv(s["K"], s["f"], View(un), stream=h)
            S.near_accumulate(View(u), s["k1"], s["tc"], s["td"], s["sc"], View(un), s["n"], stream=h)
            return [u, un]
        # near_list, results in tensors of this program's own
        L, nt, ne, lst, n = S.lib(), s["case"]["nt"], s["ne"], ctypes.c_void_p(), ctypes.c_int64()
        S.check(L.sctl_amd_near_list_build(ctypes.byref(lst), s["xt"].ptr, nt, None, s["xs"].ptr, s["xs"].shape[0] // 3,
                                           s["rad"].ptr, ne, s["cnt"].ptr, s["dsp"].ptr, 0, h))
        S.check(L.sctl_amd_near_list_size(lst, ctypes.byref(n)))
        x = torch.empty(3 * n.value, dtype=F64, device="cuda")
        i64 = [torch.empty(k, dtype=torch.int64, device="cuda") for k in (ne, ne, n.value, nt, nt)]
        S.check(L.sctl_amd_near_list_get(lst, x.data_ptr(), None, *[t.data_ptr() for t in i64], 0, h))
        S.check(L.sctl_amd_near_list_destroy(lst))
        return [x] + i64


# ------------------------------------------------------------------ counting and checking
def work(case):
    """Inputs read once, outputs written once; the arithmetic of every pair."""
    kind = case["kind"]
    if kind == "near_list":
        r = np.random.RandomState(case["elements"])
        p = r.randint(8, 33, case["elements"]).astype(np.int64)
        nodes = int((p * p).sum())
        # every target is near its own patch at least: the pairs written, two words and a position each
        return {"bytes": 24 * case["nt"] + 32 * nodes + (16 + 24 + 32) * case["nt"], "flops": 8 * case["nt"]}
    k0, k1, nd, flop = DIMS[case["kernel"]]
    if kind in ("eval", "eval_host", "dense_plan"):
        nt, ns = case["nt"], case["ns"]
        return {"bytes": 8 * (nt * (3 + k1) + ns * (3 + nd + k0)), "flops": flop * nt * ns}
    if kind == "matrix":
        nt, ns = case["nt"], case["ns"]
        return {"bytes": 8 * (3 * nt + (3 + nd) * ns + nt * k1 * ns * k0), "flops": flop * nt * ns}
    p, nt = block_sizes(case["blocks"])
    cnt = p * p
    pairs, ns, n = int((nt * cnt).sum()), int(cnt.sum()), int(nt.sum())
    if kind == "blocks":
        return {"bytes": 8 * (n * (3 + k1) + ns * (3 + nd + k0)), "flops": flop * pairs}
    entries = pairs * k0 * k1
    if kind == "near_subtract":
        return {"bytes": 16 * entries + 8 * (3 * n + (4 + nd) * ns), "flops": flop * pairs}
    return {"bytes": 8 * entries + 8 * ns * k0 + 8 * n * (2 * k1 + 1) + 8 * (n // 4) * (k1 + 2), "flops": 2 * entries}


def pair_matrix(name, xt, xs, xn):
    """The kernel's values K[t, s, k0, k1] for r = xt - xs (coincident points give 0)."""
    r = xt[:, None, :] - xs[None, :, :]
    r2 = (r * r).sum(-1)
    z = torch.where(r2 > 0, r2.rsqrt(), torch.zeros_like(r2))
    eye = torch.eye(3, dtype=F64, device="cuda")
    if name == "Laplace3D_FxU":
        return (z / (4 * math.pi))[..., None, None]
    if name == "Laplace3D_DxU":
        return ((r * xn[None]).sum(-1) * z ** 3 / (4 * math.pi))[..., None, None]
    if name == "Laplace3D_FxdU":
        return (r * (-z ** 3 / (4 * math.pi))[..., None])[..., None, :]
    if name == "Stokes3D_FxU":
        return (eye * z[..., None, None] + r[..., :, None] * r[..., None, :] * (z ** 3)[..., None, None]) / (8 * math.pi)
    if name == "Stokes3D_DxU":
        return r[..., :, None] * r[..., None, :] * ((r * xn[None]).sum(-1) * z ** 5 * (3 / (4 * math.pi)))[..., None, None]
    c, d = (q * z / (4 * math.pi) for q in (torch.cos(WAVENUMBER * r2 * z), torch.sin(WAVENUMBER * r2 * z)))
    return torch.stack([torch.stack([c, d], -1), torch.stack([-d, c], -1)], -2)


def pair_sum(name, xt, xs, xn, f, chunk=1 << 24):
    """sum_s K(xt, xs) f, without the matrices of the scalar kernels."""
    k0, k1 = DIMS[name][:2]
    out = torch.empty(xt.shape[0], k1, dtype=F64, device="cuda")
    scalar = {"Laplace3D_FxU": (1, 1 / (4 * math.pi)), "Laplace3D_DxU": (3, 1 / (4 * math.pi)),
              "Laplace3D_FxdU": (3, -1 / (4 * math.pi)), "Stokes3D_FxU": (3, 1 / (8 * math.pi)),
              "Stokes3D_DxU": (5, 3 / (4 * math.pi))}
    F = f.view(-1, k0)
    col = [F[:, k].contiguous() for k in range(k0)]
    far = xt.shape[0] * xs.shape[0] > 1 << 38  # sets apart from each other: |t|^2 + |s|^2 - 2 t.s is exact enough
    step = max(1, (chunk << 3 if far else chunk) // max(1, xs.shape[0]))
    for a in range(0, xt.shape[0], step):
        x = xt[a:a + step]
        if far and name == "Laplace3D_FxU":
            q = torch.addmm((xs * xs).sum(1)[None, :], x, xs.t().contiguous(), alpha=-2.0).add_((x * x).sum(1)[:, None])
            out[a:a + step, 0] = q.rsqrt_().mv(col[0]) / (4 * math.pi)
            continue
        d = [x[:, k, None] - xs[None, :, k] for k in range(3)]
        r2 = d[0] * d[0]
        r2.addcmul_(d[1], d[1]).addcmul_(d[2], d[2])
        z = torch.where(r2 > 0, r2.rsqrt(), torch.zeros_like(r2))
        if name == "Helmholtz3D_FxU":
            c, e = torch.cos(WAVENUMBER * r2 * z) * z, torch.sin(WAVENUMBER * r2 * z) * z
            out[a:a + step, 0] = (c.mv(col[0]) - e.mv(col[1])) / (4 * math.pi)
            out[a:a + step, 1] = (e.mv(col[0]) + c.mv(col[1])) / (4 * math.pi)
            continue
        power, scale = scalar[name]
        dot = lambda y: d[0] * y[:, 0] + d[1] * y[:, 1] + d[2] * y[:, 2]  # noqa: E731
        zp = z ** power
        if name == "Laplace3D_FxU":
            v = zp.mv(col[0])[:, None]
        elif name == "Laplace3D_DxU":
            v = (dot(xn) * zp).mv(col[0])[:, None]
        elif name == "Laplace3D_FxdU":
            v = torch.stack([(d[k] * zp).mv(col[0]) for k in range(3)], 1)
        else:
            q = dot(F) * zp * (dot(xn) if name == "Stokes3D_DxU" else 1.0)
            v = torch.stack([(d[k] * q).sum(1) for k in range(3)], 1)
            if name == "Stokes3D_FxU":
                v += torch.stack([z.mv(y) for y in col], 1)
        out[a:a + step] = v * scale
    return out.reshape(-1)


def exact(case, seed):
    kind = case["kind"]
    if kind == "near_list":
        return None  # whole numbers and copied positions
    name = case["kernel"]
    k0, k1, _, _ = DIMS[name]
    if kind in ("eval", "eval_host", "dense_plan", "matrix"):
        xt, xs, xn, f = points(case, seed)
        xt, xs, xn = xt.view(-1, 3), xs.view(-1, 3), xn.view(-1, 3)
        if kind != "matrix":
            v = pair_sum(name, xt, xs, xn, f)
            return v.cpu().numpy() if kind == "eval_host" else v
        M = torch.empty(case["ns"] * k0, case["nt"] * k1, dtype=F64, device="cuda")
        for a in range(0, case["ns"], 256):
            m = pair_matrix(name, xt, xs[a:a + 256], xn[a:a + 256])
            M[a * k0:(a + m.shape[1]) * k0] = m.permute(1, 2, 0, 3).reshape(m.shape[1] * k0, -1)
        return M
    p, nt, xt, tn, xs, xn, f, w = block_inputs(case, seed)
    xt, xs, xn, f = xt.view(-1, 3), xs.view(-1, 3), xn.view(-1, 3), f.view(-1, k0)
    cnt = p * p
    td, sd = starts(nt), starts(cnt)
    if kind == "blocks":
        out = torch.empty(int(nt.sum()) * k1, dtype=F64, device="cuda")
        for b in range(p.size):
            t, s = slice(td[b], td[b] + nt[b]), slice(sd[b], sd[b] + cnt[b])
            out[td[b] * k1:(td[b] + nt[b]) * k1] = pair_sum(name, xt[t], xs[s], xn[s], f[s].reshape(-1))
        return out
    size = nt * cnt * k0 * k1
    K, off = matrices(case, seed, int(size.sum())), starts(size)
    un = torch.empty(int(nt.sum()), k1, dtype=F64, device="cuda")
    for b in range(p.size):
        t, s = slice(td[b], td[b] + nt[b]), slice(sd[b], sd[b] + cnt[b])
        Kb = K[off[b]:off[b] + size[b]].view(nt[b] * k1, cnt[b] * k0)
        if kind == "near_interac":
            un[t] = Kb.mv(f[s].reshape(-1)).view(-1, k1)
            continue
        for a in range(0, int(nt[b]), 256):
            m = pair_matrix(name, xt[t][a:a + 256], xs[s], xn[s]) * w[s][None, :, None, None]
            Kb[a * k1:(a + m.shape[0]) * k1] -= m.permute(0, 3, 1, 2).reshape(m.shape[0] * k1, -1)
    if kind == "near_subtract":
        return K
    n, pair = near_pairs(nt)
    u = torch.zeros(n, k1, dtype=F64, device="cuda").index_add_(0, torch.from_numpy(pair).cuda(), un)
    return [u.reshape(-1), un.reshape(-1)]
