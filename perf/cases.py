"""The work that performance of this framework is measured on.

Each case is one call (or one training step) that a program makes through the
public entry points of `hddm_lb`, over the range that the package's own
workloads cover: D from 4 to 59, grids from a hundred to 281,077 nodes, 7 to
128 dofs, one point to 2^20 points, one state or many, the FP64 path and the
mixed ones, forward, adjoint and both.

A case holds
  kind      host     forward_host: numpy in and out, synchronous (what the
                     plugin's Interpolator::interpolate calls)
            forward  Context.forward on device tensors
            plan     Plan.launch, a forward captured into a hipGraph
            adjoint  Context.adjoint, dx and dsurplus
            step     forward and adjoint of one batch
            grad     hddm_lb_autograd.interpolate and its backward
  dim, points, states, precision
  grid      regular: all nodes with sum(l - 1) <= start_sum; adaptive: seeded
            refinement from start_sum up to max_level until `nodes` are there
  nodes     of an adaptive grid; with several states, log-uniform from
            nodes / 100 up to it
  dofs      of every state; with mixed_dofs, each state draws dofs, dofs / 2 or
            dofs / 4

Results of the mixed paths are F32-accurate numbers in FP64 buffers; a program
that asks for them goes on in float32, so those are returned as float32. FP64
results are returned as they are.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "hddm-solver-postprocessors_amd"))
import hddm_lb  # noqa: E402
import hddm_lb_autograd  # noqa: E402

PRECISION = {"fp64": hddm_lb.FP64, "f32": hddm_lb.F32, "f16x2": hddm_lb.F16X2, "bf16x3": hddm_lb.BF16X3}


def case(name, kind, dim, points, precision, nodes=0, dofs=32, states=1, start_sum=1, max_level=6, mixed_dofs=False):
    c = dict(kind=kind, dim=dim, points=points, precision=precision, grid="adaptive" if nodes else "regular",
             nodes=nodes, dofs=dofs, states=states, start_sum=start_sum, max_level=max_level, mixed_dofs=mixed_dofs)
    return dict(c, name=name) if name else c


def listed():
    return [
        # one point per call through host buffers, the solver's per-point
        # interpolation: latency, launches and copies
        case("host_point_d59_fp64", "host", 59, 1, "fp64", dofs=118, start_sum=1),
        # the CPU-sized regular grid of the small tests, one eager call
        case("forward_small_d4_fp64", "forward", 4, 4096, "fp64", dofs=8, start_sum=4),
        # a launch-bound loop over a captured forward, odd sizes
        case("plan_d8_f32", "plan", 8, 1000, "f32", nodes=2000, dofs=17),
        # a large single-state evaluation, mixed
        case("forward_d16_f32", "forward", 16, 1 << 20, "f32", nodes=60000, start_sum=2, max_level=7),
        # the same grid in full precision, a batch that fills no block evenly
        case("forward_d16_fp64", "forward", 16, 100003, "fp64", nodes=60000, start_sum=2, max_level=7),
        # twelve uneven states in one call, as a solver with many regimes has
        case("multistate_d20_f32", "forward", 20, 262144, "f32", nodes=200000, dofs=64, states=12, mixed_dofs=True),
        # a wide state through the split-f16 path, odd batch
        case("forward_d24_f16x2", "forward", 24, 30011, "f16x2", nodes=12000, dofs=128),
        # forward and adjoint of a differentiated model, mixed
        case("step_d20_f32", "step", 20, 65536, "f32", nodes=100000),
        # a small differentiable layer in a torch program (FP64 backward)
        case("grad_d8_fp64", "grad", 8, 4099, "fp64", nodes=2000, dofs=16),
        # the high-dimensional multistate model: forward, mixed
        case("forward_d59_f32", "forward", 59, 65536, "f32", dofs=128, states=4, start_sum=3, max_level=4),
        # its adjoint, mixed
        case("adjoint_d59_f32", "adjoint", 59, 32768, "f32", dofs=128, states=2, start_sum=3, max_level=4),
        # its training step in full precision, a smaller ragged batch
        case("step_d59_fp64", "step", 59, 12345, "fp64", dofs=128, start_sum=3, max_level=4),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["host", "forward", "forward", "forward", "plan", "adjoint", "step", "grad"])
    precision = "fp64" if kind == "grad" else rng.choice(["fp64", "f32"])
    if kind in ("forward", "plan") and rng.random() < 0.3:
        precision = rng.choice(["f16x2", "bf16x3"])
    if kind == "host":
        return case("", kind, rng.choice([4, 8, 20, 59]), _log(rng, 1, 300), precision, dofs=rng.randint(7, 128),
                    start_sum=1 if rng.random() < 0.5 else 2)
    if kind != "plan" and rng.random() < 0.25:
        # the high-dimensional model, 7,081 or 281,077 nodes
        s = rng.choice([2, 3])
        states = 1 if kind == "grad" else rng.randint(1, 2)
        return case("", kind, rng.randint(50, 59), _log(rng, 300, 16000), precision, dofs=rng.randint(33, 128),
                    states=states, start_sum=s, max_level=4)
    dim = rng.randint(4, 32)
    # adaptive grids of up to 100k nodes (a low dimension holds fewer)
    nodes = _log(rng, 300, {True: 1500, False: 100000 if dim >= 12 else 8000}[dim < 8])
    dofs = rng.choice([_log(rng, 7, 128), 16, 32, 64])
    top = 200000 if kind == "forward" else 40000
    points = _log(rng, 64, 2000 if kind == "plan" else max(100, min(top, int(1.5e11 / (nodes * max(dofs, 32))))))
    states = rng.choice([1, 1, 1, rng.randint(2, 12)]) if kind in ("forward", "adjoint", "step") else 1
    return case("", kind, dim, points, precision, nodes=nodes, dofs=dofs, states=states, mixed_dofs=states > 1)


def _inputs(c, seed):
    """Grids, surpluses, points, state ids and upstream gradients (numpy), from the seed alone."""
    rng = np.random.default_rng([seed, 20])
    shape = np.random.default_rng([c["states"], 40])
    dim, n, states = c["dim"], c["points"], c["states"]
    grids = []
    for s in range(states):
        nodes, dofs = c["nodes"], c["dofs"]
        if states > 1 and nodes:
            nodes = int(np.exp(shape.uniform(np.log(max(1, nodes / 100)), np.log(nodes))))
        if c["mixed_dofs"]:
            dofs = max(1, int(dofs // shape.choice([1, 2, 4])))
        if nodes:
            # the model's grid stays; its values and the points change with the seed
            ii, jj, lv, _ = hddm_lb.generate_grid(dim, c["start_sum"], c["max_level"], 0.3, 300 + s, nodes)
        else:
            ii, jj, lv, _ = hddm_lb.generate_grid(dim, c["start_sum"], c["start_sum"] + 1, 0.0, 1, 0)
        grids.append((ii, jj, hddm_lb.synthetic_surplus(lv, dofs, [seed, 30, s])))
    x = rng.uniform(0.0, 1.0, size=(n, dim))
    sid = rng.integers(0, states, size=n).astype(np.int32) if states > 1 else None
    width = max(g[2].shape[1] for g in grids)
    g = rng.standard_normal((n, width)) if c["kind"] in ("adjoint", "step", "grad") else None
    return grids, x, sid, g


def prepare(c, seed):
    grids, x, sid, g = _inputs(c, seed)
    ctx = hddm_lb.Context(0)
    for s, (ii, jj, S) in enumerate(grids):
        ctx.upload_state(s, ii, jj, S)
    st = {"kind": c["kind"], "ctx": ctx, "precision": PRECISION[c["precision"]], "half": c["precision"] != "fp64"}
    width = max(S.shape[1] for _, _, S in grids)
    n = c["points"]
    if c["kind"] == "host":
        st.update(x=x, sid=sid, y=np.zeros((n, width)))
        return st
    st["x"] = torch.from_numpy(x).cuda()
    st["sid"] = torch.from_numpy(sid).cuda() if sid is not None else None
    if c["kind"] in ("forward", "plan", "step"):
        # columns past a state's own dofs are the caller's
        st["y"] = torch.zeros((n, width), dtype=torch.float64, device="cuda")
    if c["kind"] == "plan":
        st["plan"] = ctx.plan(st["x"], st["y"], st["sid"], st["precision"])
    if c["kind"] in ("adjoint", "step"):
        st["g"] = torch.from_numpy(g).cuda()
        st["dx"] = torch.empty((n, c["dim"]), dtype=torch.float64, device="cuda")
        st["ds"] = torch.empty((ctx.surplus_offset(-1)[1],), dtype=torch.float64, device="cuda")
    if c["kind"] == "grad":
        st["x"].requires_grad_(True)
        st["s"] = torch.from_numpy(grids[0][2]).cuda().requires_grad_(True)
        st["g"] = torch.from_numpy(g).cuda()
    return st


def run(st):
    kind, ctx, prec = st["kind"], st["ctx"], st["precision"]
    if kind == "host":
        y = ctx.forward_host(st["x"], st["y"], st["sid"], prec)
        return y.astype(np.float32) if st["half"] else y
    if kind == "grad":
        y = hddm_lb_autograd.interpolate(ctx, st["x"], st["s"], 0, prec)
        dx, ds = torch.autograd.grad(y, (st["x"], st["s"]), st["g"])
        return {"y": y.detach(), "dx": dx, "ds": ds}
    out = {}
    if kind == "plan":
        st["plan"].launch(torch.cuda.current_stream())
        out["y"] = st["y"]
    if kind in ("forward", "step"):
        ctx.forward(st["x"], st["y"], st["sid"], prec, torch.cuda.current_stream())
        out["y"] = st["y"]
    if kind in ("adjoint", "step"):
        ctx.adjoint(st["x"], st["g"], st["dx"], st["ds"], st["sid"], prec, torch.cuda.current_stream())
        out["dx"], out["ds"] = st["dx"], st["ds"]
    return {k: v.float() for k, v in out.items()} if st["half"] else out


def _grid_size(c):
    """(mean nodes, non-zero nodes of a point) of one state."""
    d = c["dim"]
    if not c["nodes"]:
        # nodes with f active dims of level sums adding up to s: the number of
        # 1-D hats of level l (2, 2, 4, 8, ... from l = 2), of which a point
        # meets one per level
        nodes, nnz = 0, 0
        hats = [1] + [max(2, 2 ** (k - 1)) for k in range(1, c["start_sum"] + 1)]
        ways = [1.0] + [0.0] * c["start_sum"]
        meets = list(ways)
        for _ in range(d):
            ways = [sum(ways[s - k] * hats[k] for k in range(s + 1)) for s in range(c["start_sum"] + 1)]
            meets = [sum(meets[s - k] for k in range(s + 1)) for s in range(c["start_sum"] + 1)]
        nodes, nnz = sum(ways), sum(meets)
        return nodes, nnz
    nodes = c["nodes"] if c["states"] == 1 else c["nodes"] * 0.99 / math.log(100)
    return nodes, 0.078 * nodes


def work(c):
    """Every grid, point and result moved once; two operations a dof for the non-zero (point, node) pairs of the
    forward, four for the adjoint (grids met in 7.8 % of their nodes by a point, as the D=16 and D=20 ones are)."""
    nodes, nnz = _grid_size(c)
    dofs = c["dofs"] * ((1 + 0.5 + 0.25) / 3 if c["mixed_dofs"] else 1)
    n, d, fp64 = c["points"], c["dim"], c["precision"] == "fp64"
    table = c["states"] * nodes * (dofs * (8 if fp64 else 4) + 16)
    fwd = {"bytes": table + n * (d + dofs) * 8, "flops": 2.0 * n * nnz * dofs}
    adj = {"bytes": table + c["states"] * nodes * dofs * 8 + n * (2 * d + dofs) * 8, "flops": 4.0 * n * nnz * dofs}
    if c["kind"] in ("host", "forward", "plan"):
        return fwd
    if c["kind"] == "adjoint":
        return adj
    return {k: fwd[k] + adj[k] for k in fwd}


def _exact_state(ii, jj, S, x, g, want_y, want_grad):
    """y, dx and dS of one state in float64 on the GPU, from the definition."""
    dev = "cuda"
    ii, jj = torch.from_numpy(ii).to(dev), torch.from_numpy(jj).to(dev)
    S, x = torch.from_numpy(S).to(dev), torch.from_numpy(x).to(dev)
    n, d = x.shape
    nno, dofs = S.shape
    active = (ii != 0) | (jj != 0)
    most = max(1, int(active.sum(1).max()))
    # active dims of each node first, in ascending order
    order = torch.argsort((~active).to(torch.int32), dim=1, stable=True)[:, :most]
    on = active.gather(1, order)
    fi, fj = ii.gather(1, order).to(torch.int64), jj.gather(1, order).to(torch.int64)
    # distinct 1-D hats; a padding slot is the hat that is 1 everywhere
    key = torch.where(on, (order + 1) * (1 << 44) + (fi << 22) + fj, torch.zeros_like(order))
    hats, slot = torch.unique(key, return_inverse=True)
    hd = torch.clamp((hats >> 44) - 1, min=0)
    hi = ((hats >> 22) & ((1 << 22) - 1)).double()
    hj = (hats & ((1 << 22) - 1)).double()
    pad = hats == 0
    y = torch.zeros((n, dofs), dtype=torch.float64, device=dev)
    dx = torch.zeros((n, d), dtype=torch.float64, device=dev)
    ds = torch.zeros((nno, dofs), dtype=torch.float64, device=dev)
    gd = torch.from_numpy(g).to(dev)[:, :dofs].contiguous() if want_grad else None
    for p0 in range(0, n, 4096):
        u = x[p0:p0 + 4096][:, hd] * hi - hj
        phi = torch.clamp(1.0 - u.abs(), min=0.0)
        phi[:, pad] = 1.0
        dphi = torch.where(phi > 0, -hi * torch.sign(u), torch.zeros_like(u))
        dphi[:, pad] = 0.0
        for k0 in range(0, nno, 16384):
            sl = slot[k0:k0 + 16384]
            f = [phi[:, sl[:, t]] for t in range(most)] if want_grad else None
            B = f[0].clone() if want_grad else phi[:, sl[:, 0]]
            for t in range(1, most):
                B *= f[t] if want_grad else phi[:, sl[:, t]]
            if want_y:
                y[p0:p0 + 4096] += B @ S[k0:k0 + 16384]
            if want_grad:
                gp = gd[p0:p0 + 4096]
                ds[k0:k0 + 16384] += B.t().contiguous() @ gp
                w = gp @ S[k0:k0 + 16384].t().contiguous()
                for t in range(most):
                    term = w * dphi[:, sl[:, t]]
                    for q in range(most):
                        if q != t:
                            term *= f[q]
                    to = torch.zeros((sl.shape[0], d), dtype=torch.float64, device=dev)
                    to[torch.arange(sl.shape[0], device=dev), hd[sl[:, t]]] = 1.0
                    dx[p0:p0 + 4096] += term @ to
    return y, dx, ds


def exact(c, seed):
    grids, x, sid, g = _inputs(c, seed)
    n, d = x.shape
    want_y, want_grad = c["kind"] != "adjoint", c["kind"] in ("adjoint", "step", "grad")
    width = max(S.shape[1] for _, _, S in grids)
    y = torch.zeros((n, width), dtype=torch.float64, device="cuda")
    dx = torch.zeros((n, d), dtype=torch.float64, device="cuda")
    ds = []
    for s, (ii, jj, S) in enumerate(grids):
        sel = np.arange(n) if sid is None else np.flatnonzero(sid == s)
        ys, dxs, dss = _exact_state(ii, jj, S, np.ascontiguousarray(x[sel]), g[sel] if g is not None else None,
                                    want_y, want_grad)
        at = torch.from_numpy(sel).cuda()
        y[at, :S.shape[1]] = ys
        dx[at] = dxs
        ds.append(dss.reshape(-1))
    if c["kind"] == "host":
        return y.cpu().numpy()
    if c["kind"] == "grad":
        return {"y": y, "dx": dx, "ds": ds[0].reshape(grids[0][2].shape)}
    out = {"y": y} if want_y else {}
    if want_grad:
        out.update(dx=dx, ds=torch.cat(ds))
    return out
