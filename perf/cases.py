"""The work whose speed is followed: what a user of this package has it do,
over the range of sizes, forms and directions it is used at.

Three kinds of case, each through the package's public entry points:

* ``flow``: a time loop from an initial temperature, as a program that studies
  convection runs it (``Citcom.initialize``, the step-0 solve
  ``general_stokes_solver``, then ``timestep`` several times; ``steps`` 0: the
  step-0 solve alone), the fields downloaded at the end.  The Uzawa loop runs to
  its cap (``piterations``, here ``cap``) on the larger boxes, as it does in
  earnest on them, so the amount of work is set by the case.  ``form`` is the
  package's arithmetic: 0 the reference's, 1 FP32 multigrid cycles inside FP64
  refinement, 2 the same with FP16 fine-level stiffness; ``warm`` the initial
  guess of each solve (0 previous solution, 1 extrapolated, 2 extrapolated and
  corrected by the trained U-Net).
* ``energy``: one SUPG energy step and the Nusselt numbers from a given state
  (``PG_timestep``, ``heat_flux``), which a drop-in user calls on uploaded
  fields and which every timestep contains.
* ``unet`` / ``convnet``: the warm start's networks: inference (``grad`` 0)
  and one gradient evaluation of training (``grad`` 1: forward, loss,
  backward; the optimizer's update is left out so that a repeated pass does
  the same work).

The context of a mesh is what a user's program builds once and keeps, so one is
kept here per problem; each pass starts from its own temperature.  The plain
form's velocity and pressure come back in FP64, as it holds them; the forms
with FP32 cycles give the fields as snapshots hold them, in FP32.
"""
from __future__ import annotations

import functools
import math
import os

import numpy as np
import torch

from citcom_amd import deck, learn, unet
from citcom_amd.hip import Citcom

NOUT = 4          # channels the networks' losses read


def listed():
    return [
        # the smallest run: the 16^3 isoviscous box, launches and latency count
        flow("iso16_run", "iso16", 0, cap=20, steps=3),
        # the published benchmark boxes: rigid lids, 32x16x32 elements, a few
        # iterations a step; and 32^3 with Arrhenius viscosity on a graded grid,
        # the stiffness rebuilt in every step
        flow("busse1a_run", "busse1a", 0, cap=10, steps=5),
        flow("busse2_run_mixed16", "busse2", 2, cap=10, steps=3),
        # the 64^3 workload in the reference's arithmetic
        flow("tdep64_solve", "tdep64", 0, cap=60),
        # a box that is no power of two on any axis, FP32 cycles
        flow("box80x48x40_solve_mixed", "", 1, cap=60, levels=4, mx=10, my=6, mz=5),
        # the largest workload: the step-0 solve in the reference's arithmetic
        # and in the fastest form, and the time loop of the latter with the
        # learned warm start (rebuild, energy step, U-Net, solve)
        flow("tdep128_solve", "tdep128", 0, cap=60),
        flow("tdep128_solve_mixed16", "tdep128", 2, cap=60),
        flow("tdep128_run_learned", "tdep128", 2, cap=20, steps=4, warm=2),
        # the energy step and heat flux of the largest workload
        {"name": "tdep128_energy", "kind": "energy", "base": "tdep128"},
        # the warm start's network on the largest workload's nodes, and a
        # training gradient at the size it is trained at
        {"name": "unet_forward_129x129x65", "kind": "unet", "grad": 0, "nb": 1, "nx": 129, "ny": 129, "nz": 65},
        {"name": "unet_gradient_65", "kind": "unet", "grad": 1, "nb": 4, "nx": 65, "ny": 65, "nz": 65},
        # the small network of the step-0 guess, at its training size
        {"name": "convnet_gradient_17", "kind": "convnet", "grad": 1, "nb": 16, "nx": 17, "ny": 17, "nz": 17},
    ]


def flow(name, base, form, cap, steps=0, warm=0, **grid):
    return {"name": name, "kind": "flow", "base": base, "form": form, "cap": cap, "steps": steps, "warm": warm, **grid}


def draw(rng):
    pick = rng.random()
    if pick < 0.6:
        # boxes of 8 to 80 elements a side; at most 90 iterations over the
        # pass's solves
        levels, steps = rng.randint(3, 5), rng.randint(0, 2)
        m = [rng.randint(2, 5) for _ in range(3)]
        cap = round(math.exp(rng.uniform(math.log(8), math.log(90 // (steps + 1)))))
        case = flow("", "", rng.randint(0, 2), cap, steps, 0, levels=levels, mx=m[0], my=m[1], mz=m[2])
        case["warm"] = rng.randint(0, 1) if steps else 0
        del case["name"]
        return case
    if pick < 0.7:
        m = [rng.randint(2, 5) for _ in range(3)]
        return {"kind": "energy", "base": "", "levels": rng.randint(3, 5), "mx": m[0], "my": m[1], "mz": m[2]}
    grad = rng.randint(0, 1)
    if pick < 0.9:   # grids whose sides are a multiple of 8 plus one
        n = [8 * round(math.exp(rng.uniform(math.log(2), math.log(9)))) + 1 for _ in range(3)]
        return {"kind": "unet", "grad": grad, "nb": rng.randint(1, 3), "nx": n[0], "ny": n[1], "nz": n[2]}
    n = [round(math.exp(rng.uniform(math.log(5), math.log(40)))) for _ in range(3)]
    return {"kind": "convnet", "grad": grad, "nb": rng.randint(1, 16), "nx": n[0], "ny": n[1], "nz": n[2]}


# ---------------------------------------------------------------------------
# problems and inputs


def problem(case):
    """The workload's problem, or the 64^3 workload's viscosity law on a box of
    (mx, my, mz) 2^(levels-1) elements."""
    base = case["base"]
    keys = deck.workload(base or "tdep64")
    if not base:
        m, f = (case["mx"], case["my"], case["mz"]), 1 << (case["levels"] - 1)
        keys["levels"] = case["levels"]
        for ax, n in zip("xyz", m):
            keys["mgunit" + ax] = n
            size = n / case["mz"]
            keys["dimen" + ax] = size
            keys[2 * ax] = f"0,{size}"
            keys["n" + ax] = f"1,{n * f + 1}"
    if "cap" in case:
        keys["piterations"] = case["cap"]
    return deck.problem_from_deck({k: str(v) for k, v in keys.items()})


@functools.lru_cache(maxsize=12)
def context(items, form, net):
    c = Citcom(problem(dict(items)), mixed=form)
    if net:
        w, b, _ = unet.load()
        c.set_warm_net(w, b)
    return c


def context_of(case):
    grid = ("base", "cap", "levels", "mx", "my", "mz")
    return context(tuple((k, case[k]) for k in grid if k in case), case.get("form", 0), case.get("warm") == 2)


def smooth(shape, seed, device="cpu", points=6):
    """A smooth random field of the order of 1 on a grid [..., ny, nx, nz]."""
    g = torch.Generator(device=device).manual_seed(seed)
    lead = shape[:-3]
    x = torch.randn((math.prod(lead), 1, points, points, points), generator=g, device=device)
    x = torch.nn.functional.interpolate(x, size=shape[-3:], mode="trilinear", align_corners=True)
    return x.reshape(shape)


def energy_fields(case, seed):
    """T, its rate and a velocity as convection has them: cold and hot boundary
    layers with a smooth disturbance, free-slip walls."""
    p = problem(case)
    nox, noy, noz = p.dims()
    x, y, z = (torch.from_numpy(c).double() for c in p.coords)
    shape = (noy, nox, noz)
    wall = torch.sin(math.pi * z / z[-1])
    T = 1.0 - z / z[-1] + 0.1 * wall * smooth(shape, seed)
    T = T.clamp(0.0, 1.0).float()
    T[..., 0], T[..., -1] = p.bottbcval, p.toptbcval
    Tdot = (50.0 * wall * smooth(shape, seed + 1)).float()
    Tdot[..., 0] = Tdot[..., -1] = 0.0
    V = 300.0 * smooth((3,) + shape, seed + 2).double()
    V[0, :, 0, :] = V[0, :, -1, :] = 0.0
    V[1, 0] = V[1, -1] = 0.0
    V[2, ..., 0] = V[2, ..., -1] = 0.0
    return p, T, Tdot, V.float()


def net_inputs(case, seed):
    """A network's input as the warm start forms it, 16 channels of the order of
    1, smooth with some roughness, and a target."""
    shape = (case["nb"], 16, case["ny"], case["nx"], case["nz"])
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = smooth(shape, seed, "cuda") + 0.1 * torch.randn(shape, generator=g, device="cuda")
    x = x.reshape(case["nb"], 16, -1).transpose(1, 2).contiguous().bfloat16()
    channels = 16 if case["kind"] == "convnet" else NOUT
    y = torch.randn((case["nb"], x.shape[1], channels), generator=g, device="cuda")
    return x, y


def net_weights(case, seed):
    """Layer by layer (weights bf16 [co][27][ci], biases FP32 [co]): the trained
    network for inference of the U-Net, else the spread training starts from."""
    if case["kind"] == "unet" and not case["grad"]:
        with np.load(os.path.join(os.path.dirname(unet.__file__), "weights", "warm_unet.npz")) as f:
            w, b = f["weights"], f["bias"]
        out, ow, ob = [], 0, 0
        for ci, co in unet.LAYERS:
            n = co * 27 * ci
            bits = torch.from_numpy(w[ow:ow + n].view(np.int16).copy()).view(torch.bfloat16)
            out.append((bits.reshape(co, 27, ci).cuda(), torch.from_numpy(b[ob:ob + co].copy()).cuda()))
            ow, ob = ow + n, ob + co
        return out
    layers = unet.LAYERS if case["kind"] == "unet" else [(16, 16)] * 4
    g = torch.Generator(device="cuda").manual_seed(seed + 7)
    return [((torch.randn((co, 27, ci), generator=g, device="cuda") * math.sqrt(2.0 / (27 * ci))).bfloat16(),
             0.1 * torch.randn(co, generator=g, device="cuda")) for ci, co in layers]


def prepare(case, seed):
    if case["kind"] == "flow":
        c = context_of(case)
        return {"case": case, "c": c, "T": deck.seeded_temperature(c.p, seed)}
    if case["kind"] == "energy":
        _, T, Tdot, V = energy_fields(case, seed)
        return {"case": case, "c": context_of(case), "T": T.reshape(-1).numpy(), "Tdot": Tdot.reshape(-1).numpy(),
                "V": V.reshape(-1).numpy()}
    net = unet.UNet() if case["kind"] == "unet" else learn.ConvNet(layers=4)
    weights = net_weights(case, seed)
    net.w = [w.float() for w, _ in weights]
    net.wbf = [w for w, _ in weights]
    net.b = [b for _, b in weights]
    x, y = net_inputs(case, seed)
    return {"case": case, "net": net, "x": x, "y": y, "dims": (case["nx"], case["ny"], case["nz"]),
            "wch": torch.tensor([1.0, 1.0, 1.0, 2.0], device="cuda")}


def run(state):
    case = state["case"]
    if case["kind"] == "flow":
        c = state["c"]
        c.set_option("warm_start", case["warm"])
        c.initialize(state["T"])
        c.general_stokes_solver()
        steps = [c.timestep() for _ in range(case["steps"])]
        out = {"V": c.download("V")}
        if case["form"] == 0:
            out["U"], out["P"] = c.download("U"), c.download("P")
        else:
            out["P"] = c.download("P").astype(np.float32)
        if steps:
            out["T"] = c.download("T")
            out["dt"] = [s["pg"]["timestep"] for s in steps]
            out["Nu"] = [s["Nu_top"] for s in steps]
        return out
    if case["kind"] == "energy":
        c = state["c"]
        for name in ("T", "Tdot", "V"):
            c.upload(name, state[name])
        st = c.PG_timestep()
        nu = c.heat_flux()
        return {"T": c.download("T"), "Tdot": c.download("Tdot"), "dt": st["timestep"], "Nu": list(nu)}
    net, x, dims = state["net"], state["x"], state["dims"]
    out = net.forward(x, dims)
    if not case["grad"]:
        return out
    if case["kind"] == "unet":
        loss, dy = net.loss_grad(out, state["y"], state["wch"])
    else:
        loss, dy = net.loss_grad(out, state["y"])
    return {"loss": loss, "grads": net.backward(dy)}


# ---------------------------------------------------------------------------
# the work a pass cannot do without


def nodes(p, lev):
    return math.prod(p.dims(lev))


def work(case):
    kind = case["kind"]
    if kind in ("unet", "convnet"):
        # per convolution: input and weights read, output written (bf16); a
        # gradient evaluation reads input and output gradient again and writes
        # the input's
        if kind == "unet":
            at = [0, 0, 1, 1, 2, 2, 3, 3, 2, 2, 1, 1, 0, 0, 0]
            layers = [(ci, co, s) for (ci, co), s in zip(unet.LAYERS, at)]
        else:
            layers = [(16, 16, 0)] * 4
        total_b = total_f = 0.0
        for ci, co, s in layers:
            nv = case["nb"] * math.prod((case[k] - 1) // (1 << s) + 1 for k in ("nx", "ny", "nz"))
            total_b += 2.0 * nv * (ci + co) * (3 if case["grad"] else 1)
            total_f += 2.0 * 27 * ci * co * nv * (3 if case["grad"] else 1)
        return {"bytes": total_b, "flops": total_f}
    p = problem(case)
    n = nodes(p, p.levmax)
    if kind == "energy":
        # T, Tdot, V read, T, Tdot written; two passes over 8 Gauss points
        return {"bytes": n * 28.0, "flops": n * 2 * 8 * 8 * 24.0}
    # one multigrid call per Uzawa iteration: on each level, the smoother's
    # sweeps and one product with the 27-neighbour rows on the way down and up of
    # every cycle through it
    total_b = total_f = 0.0
    vec = 4 if case["form"] else 8
    for lev in range(1, p.levels):
        coef = 2 if case["form"] == 2 and lev >= p.levmax - 1 else 4
        visits = 2 * (p.levels - lev) * p.mg_cycle
        rows = visits * (p.down_heavy + 1) * nodes(p, lev)
        total_b += rows * (243.0 * coef + 12 * vec)
        total_f += rows * 2.0 * 243
    if case["form"]:
        total_b += n * (243.0 * 4 + 48)
        total_f += n * 2.0 * 243
    its = case["cap"] * (case["steps"] + 1)
    return {"bytes": its * total_b, "flops": its * total_f}


# ---------------------------------------------------------------------------
# the same in 64 bits, with torch alone


def exact(case, seed):
    """The energy step's fields and the networks' outputs and gradients; the
    flow solves have no value that plain code reaches in the time."""
    if case["kind"] == "flow":
        return None
    if case["kind"] == "energy":
        return exact_energy(case, seed)
    x, y = net_inputs(case, seed)
    weights = [(w.double().requires_grad_(bool(case["grad"])), b.double().requires_grad_(bool(case["grad"])))
               for w, b in net_weights(case, seed)]
    grid = (case["nb"], case["ny"], case["nx"], case["nz"])
    with torch.set_grad_enabled(bool(case["grad"])):
        net = exact_unet if case["kind"] == "unet" else exact_convnet
        out = net(x.double().reshape(grid + (16,)), weights).reshape(case["nb"], -1, 16)
        if not case["grad"]:
            return out
        e = out[..., :NOUT] - y.double()[..., :NOUT]
        if case["kind"] == "unet":
            e2 = (e * e * torch.tensor([1.0, 1.0, 1.0, 2.0], device="cuda", dtype=torch.float64)).sum()
        else:
            e2 = (e * e).sum()
        loss = e2 / (out.shape[0] * out.shape[1] * NOUT)
        loss.backward()
    return {"loss": float(loss), "grads": [torch.cat([w.grad.reshape(-1), b.grad]) for w, b in weights]}


def conv(x, wb):
    """3x3x3, zero padding, x [nb][y][x][z][c]; tap (dz+1) + 3(dx+1) + 9(dy+1)."""
    w, b = wb
    nb, ny, nx, nz, _ = x.shape
    xp = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1, 1, 1))
    out = b.expand(nb, ny, nx, nz, b.shape[0])
    for t in range(27):
        k, i, j = t % 3, (t // 3) % 3, t // 9
        out = out + torch.nn.functional.linear(xp[:, j:j + ny, i:i + nx, k:k + nz], w[:, t])
    return out


def restrict(x):
    for d in (1, 2, 3):
        n = x.shape[d]
        even = x.index_select(d, torch.arange(0, n, 2, device=x.device))
        odd = x.index_select(d, torch.arange(1, n, 2, device=x.device))
        zero = torch.zeros_like(odd.narrow(d, 0, 1))
        x = 0.5 * even + 0.25 * (torch.cat([zero, odd], d) + torch.cat([odd, zero], d))
    return x


def interp(x):
    for d in (1, 2, 3):
        n = x.shape[d]
        mid = 0.5 * (x.narrow(d, 0, n - 1) + x.narrow(d, 1, n - 1))
        pairs = torch.stack([x.narrow(d, 0, n - 1), mid], d + 1).flatten(d, d + 1)
        x = torch.cat([pairs, x.narrow(d, n - 1, 1)], d)
    return x


def exact_unet(x, w):
    def layer(k, v, skip=0.0):
        return torch.relu(conv(v, w[k]) + skip)
    s0 = layer(1, layer(0, x))
    s1 = layer(3, layer(2, restrict(s0)))
    s2 = layer(5, layer(4, restrict(s1)))
    b3 = layer(7, layer(6, restrict(s2)))
    d2 = layer(9, layer(8, interp(b3), s2))
    d1 = layer(11, layer(10, interp(d2), s1))
    d0 = layer(13, layer(12, interp(d1), s0))
    return conv(d0, w[14])


def exact_convnet(x, w):
    for k, wb in enumerate(w):
        x = conv(x, wb)
        if k < len(w) - 1:
            x = torch.relu(x)
    return x


def exact_energy(case, seed):
    """One predictor and two corrector passes of the streamline-upwind energy
    step on a grid of bricks, 2x2x2 Gauss points, lumped mass."""
    p, T, Tdot, V = energy_fields(case, seed)
    T, Tdot, V = (a.double().cuda() for a in (T, Tdot, V))
    h = [torch.from_numpy(np.diff(c.astype(np.float64))).cuda() for c in p.coords]
    dx, dy, dz = h[0][None, :, None], h[1][:, None, None], h[2][None, None, :]
    jac = dx * dy * dz / 8.0

    def corners(f):
        """[..., node of an element (oy, ox, oz)], elements [y][x][z]"""
        ny, nx, nz = f.shape[-3] - 1, f.shape[-2] - 1, f.shape[-1] - 1
        return [f[..., a:a + ny, b:b + nx, c:c + nz] for a in (0, 1) for b in (0, 1) for c in (0, 1)]

    def assemble(parts):
        out = torch.zeros_like(T)
        ny, nx, nz = (n - 1 for n in T.shape)
        for part, (a, b, c) in zip(parts, [(a, b, c) for a in (0, 1) for b in (0, 1) for c in (0, 1)]):
            out[a:a + ny, b:b + nx, c:c + nz] += part
        return out

    s = 1.0 / math.sqrt(3.0)
    line = {q: ((1 - q) / 2, (1 + q) / 2) for q in (-s, s)}
    corner = [(a, b, c) for a in (0, 1) for b in (0, 1) for c in (0, 1)]
    mass = assemble([jac.expand([n - 1 for n in T.shape])] * 8)
    uc = [sum(corners(V[d])) / 8.0 for d in range(3)]
    courant = (uc[0].abs() / dx + uc[1].abs() / dy + uc[2].abs() / dz).max()
    size = min(float(a.min()) for a in h)
    dt = min(p.finetunedt * 0.5 / float(courant), 0.5 * size * size)
    if p.fixed_timestep:
        dt = p.fixed_timestep
    peclet = [(uc[0] * dx).abs(), (uc[1] * dy).abs(), (uc[2] * dz).abs()]
    up = sum(q * torch.where(q > 2.0, 1.0 - 2.0 / q, 0.0) for q in peclet)
    norm = uc[0] ** 2 + uc[1] ** 2 + uc[2] ** 2
    tau = torch.where(norm > 1e-6, up / (2.0 * norm), 0.0)
    free = torch.ones_like(T)
    free[..., 0] = free[..., -1] = 0.0
    T = T + free * (1.0 - p.gamma) * dt * Tdot
    Tdot = torch.zeros_like(T)
    vc = [corners(V[d]) for d in range(3)]
    for _ in range(p.temp_iterations):
        tc, rc = corners(T), corners(Tdot * free)
        parts = [0.0] * 8
        for qy in line:
            for qx in line:
                for qz in line:
                    N = [line[qy][a] * line[qx][b] * line[qz][c] for a, b, c in corner]
                    gx = [line[qy][a] * (2 * b - 1) * line[qz][c] / dx for a, b, c in corner]
                    gy = [(2 * a - 1) * line[qx][b] * line[qz][c] / dy for a, b, c in corner]
                    gz = [line[qy][a] * line[qx][b] * (2 * c - 1) / dz for a, b, c in corner]
                    u = [sum(n * f for n, f in zip(N, vc[d])) for d in range(3)]
                    grad = [sum(w * f for w, f in zip(g, tc)) for g in (gx, gy, gz)]
                    rate = sum(n * f for n, f in zip(N, rc)) - p.Q0 + sum(a * b for a, b in zip(u, grad))
                    for m in range(8):
                        weight = N[m] + tau * (u[0] * gx[m] + u[1] * gy[m] + u[2] * gz[m])
                        parts[m] = parts[m] - jac * (weight * rate + gx[m] * grad[0] + gy[m] * grad[1] + gz[m] * grad[2])
        step = assemble(parts) / mass
        T = T + free * p.gamma * dt * step
        Tdot = Tdot + step
    T[..., 0], T[..., -1] = p.bottbcval, p.toptbcval
    return {"T": T.reshape(-1), "Tdot": Tdot.reshape(-1), "dt": dt, "Nu": None}
