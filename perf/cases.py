"""Timed workloads of the ORB build: what a program that uses this library has it do.

Three kinds of case, all through the public Python binding of the C-ABI:

build  A context holds the particles in HBM (as a simulation does between steps) and a snapshot of
       their input order.  One pass brings that order back (`restore_particles`: the stand-in for new
       particles, a device copy), builds the tree and reads what the caller of a domain decomposition
       needs: the pass counts, the cell heap and the cell-to-range map, for small sets the reordered
       particles too, with ids the leaf of every input particle.
serve  A server (continuous batching) gets particle arrays that already live in device memory and
       reorders them in place; the trees come back to the host.
count  One count-left service call over the cells of a finished level: the reference's hot service.

Particle sets: "uniform" in [-0.5, 0.5)^3 as the reference generator draws them, "plummer" (64 spheres of
scale radius 0.01 with a 10% uniform background, spread over the array), "grid" (512 coordinate values: many equal keys).
Floats come back as their bit patterns: a build moves coordinates and compares them, so every bit counts.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "gpu-load-balance_amd"))
import orb_amd as orb  # noqa: E402

# the reference's option o (src/orbit.cpp:48-66): CPU, GPU count, GPU count and partition
PARAMS = {0: (False, False, False), 1: (True, False, False), 2: (True, True, False)}


def _build(n, d, dist="uniform", o=0, form="batched", levels="full", ids=False, weights=False,
           read="tree"):
    return {"kind": "build", "n": n, "d": d, "dist": dist, "o": o, "form": form, "levels": levels,
            "ids": ids, "weights": weights, "read": read}


def listed():
    return [
        # a small rank's share, rebuilt every step: launches and latency decide
        dict(_build(1 << 16, 64, read="particles"), name="small_64k"),
        # odd sizes, clustered, ids tracked, the leaf of every input particle read back
        dict(_build(100003, 100, "plummer", ids=True, read="members"), name="odd_100k_ids"),
        # the reference's own first configuration, `orbit 20 10`, with its level schedule
        dict(_build(1 << 20, 1 << 10, levels="reference"), name="orbit_20_10"),
        # the drop-in form of the reference's o=1 loop: a count launch per bisection pass
        dict(_build(1 << 20, 64, o=1, form="plain"), name="plain_1m_o1"),
        # workload weights on a ragged set
        dict(_build(2000003, 250, weights=True), name="weights_2m"),
        # the reference's o=2 (<= counts, stable partition)
        dict(_build(1 << 24, 256, o=2), name="stable_16m"),
        # coarse coordinates: many keys equal to a cut
        dict(_build(5000011, 48, "grid"), name="grid_5m"),
        # clustered 2^26 into many leaves
        dict(_build(1 << 26, 1 << 14, "plummer"), name="plummer_64m"),
        # small leaves (256 particles): most levels are deep ones; the ranges are read back
        dict(_build(1 << 26, 1 << 18, read="ranges"), name="deep_64m"),
        # the headline workload: 2^27 uniform particles into 2^10 leaves
        dict(_build(1 << 27, 1 << 10), name="uniform_128m"),
        # a queue of device requests, N log-uniform in [2^16, 2^22], d in [2^4, 2^12], half of them
        # clustered: the serving mix with all requests waiting
        {"kind": "serve", "name": "serve_mix", "requests": 12, "lo": 16.0, "hi": 22.0,
         "dlo": 4.0, "dhi": 12.0},
        # the count-left service over the 512 cells of a level
        {"kind": "count", "name": "count_64m", "n": 1 << 26, "cells": 512, "o": 0},
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    """One more case: sizes log-uniform and rarely round, options as they are used."""
    u = rng.random()
    if u < 0.12:
        lo = rng.uniform(14.0, 18.0)
        dlo = rng.uniform(2.0, 6.0)
        return {"kind": "serve", "requests": rng.randint(1, 12), "lo": lo,
                "hi": min(22.0, lo + rng.uniform(1.0, 6.0)), "dlo": dlo,
                "dhi": dlo + rng.uniform(1.0, 5.0)}
    if u < 0.22:
        n = int(_log(rng, 1 << 14, 1 << 26))
        return {"kind": "count", "n": n, "cells": 1 << rng.randint(0, 9), "o": rng.randint(0, 1)}
    plain = u < 0.30
    n = int(_log(rng, 1 << 14, 1 << (22 if plain else 26)))
    dist = rng.choice(["uniform", "uniform", "plummer", "plummer", "grid"])
    most = 64 if dist == "grid" else 256 if plain else 1 << 17
    d = max(2, int(_log(rng, 2, max(4, min(most, n // 128)))))
    ids = rng.random() < 0.2
    small = n <= 1 << 18
    return _build(n, d, dist, o=rng.choice([0, 0, 0, 1, 2]), form="plain" if plain else "batched",
                  levels="full", ids=ids, weights=not plain and not ids and rng.random() < 0.15,
                  read="particles" if small and not ids else "members" if small else
                  "tree" if d <= 1 << 14 else "ranges")


# ---- particle sets, made on the GPU from the seed
def _uniform(n, g):
    return torch.rand(3, n, device="cuda", generator=g) - 0.5


def _plummer(n, g, spheres=64, a=0.01, background=0.1):
    centre = torch.rand(3, spheres, device="cuda", generator=g) - 0.5
    p = _uniform(n, g)
    todo = torch.nonzero(torch.rand(n, device="cuda", generator=g) >= background).view(-1)
    while todo.numel():
        m = todo.numel()
        u = torch.rand(m, device="cuda", generator=g).clamp_(1e-6, 1.0 - 1e-6)
        r = a / torch.sqrt(u.pow(-2.0 / 3.0) - 1.0)
        c = torch.rand(m, device="cuda", generator=g) * 2.0 - 1.0
        phi = torch.rand(m, device="cuda", generator=g) * (2.0 * math.pi)
        s = torch.sqrt((1.0 - c * c).clamp_(min=0.0))
        q = centre[:, todo % spheres] + r * torch.stack((s * torch.cos(phi), s * torch.sin(phi), c))
        p[:, todo] = q
        todo = todo[((q < -0.5) | (q >= 0.5)).any(0)]  # draws outside the box are drawn again
    return p


def _grid(n, g, values=512):
    return torch.randint(0, values, (3, n), device="cuda", generator=g).float() / values - 0.5


def _particles(dist, n, g):
    return {"uniform": _uniform, "plummer": _plummer, "grid": _grid}[dist](n, g)


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) + 20221)
    return g


def _requests(case, seed):
    """Sizes of a serving mix: fixed by the case, so that every seed asks for the same work."""
    k = case["requests"]
    out = []
    for i in range(k):
        f = (i * 0.6180339887498949 + 0.37) % 1.0  # spread over the log range, ragged
        h = (i * 0.7548776662466927 + 0.11) % 1.0
        n = int(2.0 ** (case["lo"] + f * (case["hi"] - case["lo"])))
        d = max(2, int(2.0 ** (case["dlo"] + h * (case["dhi"] - case["dlo"]))))
        out.append((n, min(d, max(2, n // 64)), "plummer" if i % 2 else "uniform"))
    return out


def prepare(case, seed):
    g = _generator(seed)
    if case["kind"] == "serve":
        reqs = _requests(case, seed)
        total = sum(n for n, _, _ in reqs)
        cells = sum(int(orb.lib().orb_heap_capacity(d)) for _, d, _ in reqs)
        home = [_particles(dist, n, g).contiguous() for n, _, dist in reqs]
        work = [torch.empty_like(h) for h in home]
        torch.cuda.synchronize()
        server = orb.Server(particle_capacity=total + 64 * len(reqs), cell_capacity=2 * cells + 64,
                            max_active=64)
        return {"case": case, "reqs": reqs, "home": home, "work": work, "server": server}
    n = case["n"]
    d = case["cells"] * 2 if case["kind"] == "count" else case["d"]
    p = _particles(case.get("dist", "uniform"), n, g)
    x, y, z = p.cpu().numpy()
    del p
    ctx = orb.Context(n, d, generate=False, params=PARAMS[case["o"]])
    ctx.set_particles(x, y, z)
    if case["kind"] == "count":
        # a level's cells at their margins' midpoints, as the bisection controller asks for them
        ctx.build(orb.FORM_BATCHED, orb.LEVELS_FULL)
        first = case["cells"] - 1
        return {"case": case, "ctx": ctx, "cells": _reset(ctx.heap()[first:first + case["cells"]])}
    if case["ids"]:
        ctx.enable_ids()
    if case["weights"]:
        w = torch.randint(1, 1000, (n,), device="cuda", generator=g).cpu().numpy()
        ctx.set_weights(w.astype(np.uint32))
    ctx.save_particles()
    return {"case": case, "ctx": ctx}


def _reset(cells):
    """The cells as a level starts them: margins at the box, no cut found."""
    cells = cells.copy()
    k = np.arange(len(cells))
    axis = np.clip(cells["cutAxis"], 0, 2)
    cells["cutMarginLeft"] = cells["lower"][k, axis]
    cells["cutMarginRight"] = cells["upper"][k, axis]
    cells["foundCut"] = 0
    return cells


def _bits(a):
    return a.view(np.int32)


def run(state):
    case = state["case"]
    if case["kind"] == "count":
        ctx = state["ctx"]
        left = ctx.count_left if case["o"] == 0 else ctx.count_left_gpu
        return left(state["cells"]).astype(np.int64)
    if case["kind"] == "serve":
        return _serve(state)
    ctx = state["ctx"]
    ctx.restore_particles()
    info = ctx.build(orb.FORM_PLAIN if case["form"] == "plain" else orb.FORM_BATCHED,
                     orb.LEVELS_REFERENCE if case["levels"] == "reference" else orb.LEVELS_FULL)
    out = {"passes": np.array(info["level_passes"], np.int64), "ranges": _bits(ctx.ranges())}
    if case["read"] != "ranges":
        out["heap"] = ctx.heap().view(np.uint8)
    if case["read"] == "particles":
        out["x"], out["y"], out["z"] = (_bits(a) for a in ctx.get_particles())
    elif case["read"] == "members":
        out["leaf_of"] = ctx.membership(by_input_order=case["ids"])
    return out


def _serve(state):
    server, reqs = state["server"], state["reqs"]
    for w, h in zip(state["work"], state["home"]):
        w.copy_(h)
    torch.cuda.current_stream().synchronize()  # the server works on a stream of its own
    ids = {}
    for k, ((n, d, _), w) in enumerate(zip(reqs, state["work"])):
        ids[server.submit_device(w[0].data_ptr(), w[1].data_ptr(), w[2].data_ptr(), n, d)] = k
    trees = [None] * len(reqs)
    while ids:
        server.step()
        while True:
            rid = server.next_done()
            if rid is None:
                break
            k = ids.pop(rid)
            res = server.fetch(rid, reqs[k][0], reqs[k][1], particles=False)
            trees[k] = {"passes": np.array(res["level_passes"], np.int64),
                        "ranges": _bits(res["ranges"]), "heap": res["heap"].view(np.uint8)}
    return {"particles": [w.view(torch.int32) for w in state["work"]], "trees": trees}


def work(case):
    """Each input read once and each output written once."""
    if case["kind"] == "count":
        return {"bytes": 4 * case["n"] + 56 * case["cells"], "flops": 0}
    reqs = _requests(case, 0) if case["kind"] == "serve" else [(case["n"], case["d"], "")]
    row = 12 + (4 if case.get("ids") else 0) + (4 if case.get("weights") else 0)
    total = 0
    for n, d, _ in reqs:
        cap = max(2 * d - 1, 2 ** (math.ceil(math.log2(d)) + 1) - 1)
        total += 2 * row * n + cap * (8 if case.get("read") == "ranges" else 60)
    return {"bytes": total, "flops": 0}


def exact(case, seed):
    """Counts follow from the inputs and the cells alone; a build's outputs are the inputs' own bits
    and whole numbers, which are compared bit for bit and have no nearer value in 64 bits."""
    return None
