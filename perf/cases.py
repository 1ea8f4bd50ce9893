"""The work whose speed is followed: what programs on this package run, from one small cloud
stepped in a Python loop to the largest batched state, each through the public entry points.

A pass advances the radiation field by a number of steps (or takes a gradient over them), as
between two saves of a longer run, and reads the state back as a save does.  The FP64 entry
points return 64-bit results; a batch holds its state in 32 bits, so what comes out of it is
kept in 32 bits here, except the luminosity, which is formed from the 64-bit sources alone.
"""
from __future__ import annotations

import dataclasses
import functools
import math

import numpy as np
import torch

from lydion_amd import _lib
from lydion_amd import constants as K
from lydion_amd import m1lya as M
from lydion_amd import workloads as W
from lydion_amd.adjoint import adjoint_run
from lydion_amd.batch import M1LyaBatch
from lydion_amd.grid import setup_cylindrical_grid
from lydion_amd.lya_arrays import VoigtLUT, compute_a, compute_sigma0, generate_lya_arrays, reference_freq_grid
from lydion_amd.static_cloud import (DEFAULT_SEED, StaticCloud, cfl_time_step, config_grid, developed_state,
                                     point_source_cloud, setup_static_cloud)

REFLECT, OUTFLOW = _lib.REFLECT, _lib.OUTFLOW


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
# A case: what is called ("call"), the medium ("kind"), its sizes and options, and the steps of a pass.
def _static(name, call, n_r, n_z, n_nu, steps, tau0=1e6, tau_abs=0.0, theta=0.0, umax=0.0, hll=False,
            open_bottom=False, grid="bins", graph=False):
    c = dict(call=call, kind="static", n_r=n_r, n_z=n_z, n_nu=n_nu, steps=steps, tau0=tau0, tau_abs=tau_abs,
             theta=theta, umax=umax, hll=hll, open_bottom=open_bottom, grid=grid, graph=graph)
    return dict(c, name=name) if name else c


def listed():
    pi4 = math.pi / 4
    return [
        # The static-cloud test at its smallest configuration, the time loop on the host: one fused FP64
        # step per turn, its scalars read every turn.  Launches and the synchronisation count.
        _static("fp64 loop 32x32x64", "step", 32, 32, 64, 50),
        # FP64 steps queued without a turn of the host, on the reference's default frequency grid
        # (194 bins), an odd-sized expanding dusty cloud with the HLL flux and an open bottom.
        _static("fp64 run 77x90x194", "run", 77, 90, 194, 50, tau0=1e8, tau_abs=0.5, umax=200.0, hll=True,
                open_bottom=True, grid="reference"),
        # The benchmark's cone cloud through the plain FP64 step.
        _static("fp64 run 256x256x128", "run", 256, 256, 128, 120, tau0=1e8, tau_abs=1.0, theta=pi4),
        # The operators one by one, as the radiation-hydrodynamics solvers call them: the coefficients of
        # the new gas state, then the RT sub-cycles on a turbulent medium, then the forces and diagnostics.
        dict(name="operators 128x192x64", call="operators", kind="turbulent", n_r=128, n_z=192, n_nu=64, steps=24),
        # Gradients through an expanding lognormal cloud: a small odd grid, and the benchmark's.
        dict(name="gradient 45x61x64", call="gradient", kind="expanding", n_r=45, n_z=61, n_nu=64, steps=16,
             umax=800.0),
        dict(name="gradient 128x128x128", call="gradient", kind="expanding", n_r=128, n_z=128, n_nu=128, steps=64,
             umax=200.0),
        # One small cloud through the mixed-precision step with its launches replayed from a graph.
        _static("batch 32x32x64", "batch", 32, 32, 64, 400, graph=True),
        # The reference's frequency grid in the mixed-precision step (four bins per lane), HLL flux.
        _static("batch 100x84x194", "batch", 100, 84, 194, 200, tau0=1e8, tau_abs=0.5, umax=200.0, hll=True,
                grid="reference"),
        # The benchmark's headline: the cone cloud through the mixed-precision step.
        _static("batch 256x256x128", "batch", 256, 256, 128, 400, tau0=1e8, tau_abs=1.0, theta=pi4),
        # A parameter study: clouds of uneven size, depth, temperature and 32 to 128 bins in one batch.
        dict(name="batch sweep of 16", call="batch", kind="sweep", first=0, clouds=16, steps=120),
        # The radiation-hydrodynamics state of the benchmark: new gas coefficients, then its sub-steps in a
        # sheared velocity field.
        dict(name="batch turbulent 256x512x128", call="batch", kind="turbulent", n_r=256, n_z=512, n_nu=128,
             steps=300),
    ]


def draw(rng):
    """One more case: sides 24 to 256 and 18 to 256 bins, spread over their logarithms, odd sides among
    them, every option, and steps for a fixed amount of work."""
    def side(hi=256):
        return int(round(math.exp(rng.uniform(math.log(24), math.log(hi)))))

    def bins(hi):
        return 2 * int(round(math.exp(rng.uniform(math.log(9), math.log(hi // 2)))))

    def steps(n, lo, hi):
        return max(lo, min(hi, int(5e8 / n)))

    call = rng.choice(("step", "run", "operators", "gradient", "batch", "batch", "batch"))
    if call == "gradient":
        n_r, n_z, n_nu = side(128), side(128), bins(128)
        return dict(call=call, kind="expanding", n_r=n_r, n_z=n_z, n_nu=n_nu,
                    steps=max(4, min(48, int(4e7 / (n_r * n_z * n_nu)))), umax=rng.choice((10.0, 200.0, 800.0)))
    if call == "operators":
        n_r, n_z, n_nu = side(192), side(192), bins(128)
        return dict(call=call, kind="turbulent", n_r=n_r, n_z=n_z, n_nu=n_nu, steps=rng.randint(8, 24))
    if call == "batch" and rng.random() < 0.35:
        return dict(call=call, kind="sweep", first=rng.randint(1, 48), clouds=rng.randint(2, 12),
                    steps=rng.randint(40, 80))
    n_r, n_z, n_nu = side(), side(), bins(256)
    n = n_r * n_z * n_nu
    if call == "batch" and rng.random() < 0.35:
        return dict(call=call, kind="turbulent", n_r=n_r, n_z=n_z, n_nu=n_nu, steps=steps(n, 40, 200))
    return _static(None, call, n_r, n_z, n_nu, steps(n, 20, 50 if call == "step" else 200),
                   tau0=10.0 ** rng.uniform(5, 9), tau_abs=rng.choice((0.0, 1.0)),
                   theta=rng.choice((0.0, math.pi / 4)), umax=rng.choice((0.0, 200.0)), hll=rng.random() < 0.4,
                   open_bottom=rng.random() < 0.4, graph=call == "batch" and rng.random() < 0.4)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
@functools.lru_cache(maxsize=1)
def _lut():
    return VoigtLUT()


@functools.lru_cache(maxsize=4)
def _static_medium(n_r, n_z, n_nu, tau0, tau_abs, theta, umax, open_bottom, grid):
    bc = OUTFLOW if open_bottom else REFLECT
    if grid == "reference":
        nu = reference_freq_grid()
        assert len(nu) - 1 == n_nu
        return setup_static_cloud(tau0, 1e4, tau_abs=tau_abs, rs=0.5 * (1.1 / n_r), umax=umax, theta_cone=theta,
                                  dmu_cone=0.025, tmax_unitless=4.0, bc_z_bot=bc, n_r=n_r, n_z=n_z, nu=nu, lut=_lut())
    return point_source_cloud(n_r, n_z, n_nu, tau0, tau_abs=tau_abs, theta_cone=theta, umax=umax, lut=_lut(),
                              bc_z_bot=bc)


@functools.lru_cache(maxsize=2)
def _uniform_arrays(n_r, n_z, n_nu, n_mean):
    geom = setup_cylindrical_grid(1.1 * K.pc, 1.1 * K.pc, n_r, n_z)
    tau0 = n_mean * compute_sigma0(1e4) * 1.1 * K.pc
    nu = config_grid(n_nu, tau0)
    return geom, tau0, generate_lya_arrays(K.c, geom.r, geom.Z, np.full((n_z, n_r), 1e4), nu, lut=_lut())


def _turbulent(case, seed):
    """The RHD-like medium of the benchmark (lognormal density, T 1e2..1e4 K, Mach 2 turbulence, dust, open
    Z ends), its gas state in `gas` for the device-side coefficient refresh."""
    n_r, n_z, n_nu, n_mean = case["n_r"], case["n_z"], case["n_nu"], 1e3
    geom, tau0, base = _uniform_arrays(n_r, n_z, n_nu, n_mean)
    L = dataclasses.replace(base, arrays=dict(base.arrays))
    n_H = n_mean * W.lognormal_density(n_z, n_r, 1.0, seed=seed)
    T = np.clip(1e4 * (n_H / n_H.min()) ** -(math.log(100.0) / math.log(n_H.max() / n_H.min())), 1e2, 1e4)
    dust = W.KAPPA_ABS_LYA_DUST * 0.01 * 0.1 * W.MU_H * K.mH * n_H
    Zc = 0.5 * geom.Z[-1]
    js = np.zeros((n_z, n_r))
    j0 = int(np.argmin(np.abs(geom.ZCoM - Zc)))
    js[j0, 0] = 1e5 * K.Lsun / (K.Four_pi * geom.dV[j0, 0])
    pd = np.full((n_z, n_r), 1e-8)
    gas = dict(T=T, n_HI=n_H, alpha_c=dust, alpha_c_F=dust, js=js, pd=pd)
    rc, zc = geom.rCoM, geom.ZCoM
    u_r = W.gaussian_field(n_z, n_r, seed=seed + 1) * (1.0 - np.exp(-rc[None, :] / (2.0 * (geom.r[1] - geom.r[0]))))
    u_z = W.gaussian_field(n_z, n_r, seed=seed + 2)
    s = 2.0 * math.sqrt(K.kB * 1e4 / (W.MU_GAS * K.mH)) / math.sqrt(np.mean(u_r * u_r + u_z * u_z))
    u_r, u_z = u_r * s, u_z * s
    L["dur_dz"], L["dur_dr"] = (np.ascontiguousarray(v) for v in np.gradient(u_r, zc, rc))
    L["duz_dz"], L["duz_dr"] = (np.ascontiguousarray(v) for v in np.gradient(u_z, zc, rc))
    L["ur_over_r"] = u_r / rc[None, :]
    L["ur_star"] = np.concatenate([np.zeros((n_z, 1)), 0.5 * (u_r[:, :-1] + u_r[:, 1:]), u_r[:, -1:]], axis=1)
    L["uz_star"] = np.concatenate([u_z[:1], 0.5 * (u_z[:-1] + u_z[1:]), u_z[-1:]], axis=0)
    L["T"], L["js"], L["pd"], L["alpha_c"] = T, js, pd, dust
    L["alpha"] = n_H * compute_sigma0(T)
    cloud = StaticCloud(geometry=geom, lya=L, T=T, vel={}, c_tilde=K.c, dt=cfl_time_step(geom, K.c, u_r, u_z, 0.4),
                        tdiff=0.0, tmax=0.0, Zc=Zc, bc_z_bot=OUTFLOW, params=dict(tau_cl=tau0, T0=1e4))
    cloud.gas = gas
    return cloud


def _clouds(case, seed):
    """The clouds of a case in a developed radiation field drawn from the seed."""
    kind = case["kind"]
    if kind == "sweep":
        params = W.sweep_params(case["first"] + case["clouds"], DEFAULT_SEED)[case["first"]:]
        media = [W.sweep_cloud(p, _lut()) for p in params]
    elif kind == "turbulent":
        media = [_turbulent(case, seed)]
    elif kind == "expanding":
        media = [W.expanding_cloud(case["n_r"], case["n_z"], case["n_nu"], u_max=case["umax"], seed=seed, lut=_lut())]
    else:
        m = _static_medium(case["n_r"], case["n_z"], case["n_nu"], case["tau0"], case["tau_abs"], case["theta"],
                           case["umax"], case["open_bottom"], case["grid"])
        m = dataclasses.replace(m, lya=dataclasses.replace(m.lya, arrays=dict(m.lya.arrays)))
        m.lya.hll = bool(case["hll"])
        media = [m]
    return [developed_state(m, seed=seed + i) for i, m in enumerate(media)]


def _seeds(case, n_nu, seed):
    """Cotangents of a gradient: the force multipliers of every step and the escaping spectrum."""
    rng = np.random.Generator(np.random.PCG64(seed))
    return rng.uniform(0.5, 1.5, (case["steps"], 3)), rng.uniform(0.5, 1.5, n_nu)


def prepare(case, seed):
    clouds = _clouds(case, seed)
    s = dict(case=case, step=[(c.c_tilde, c.dt, c.Zc) for c in clouds], bc=[c.bc_z_bot for c in clouds])
    if case["call"] == "batch":
        s["batch"] = M1LyaBatch(clouds)
        s["batch"].set_graph(bool(case.get("graph")))
        if case["kind"] == "turbulent":
            s["batch"].set_voigt_lut(_lut())
            s["gas"] = clouds[0].gas
        return s
    c = clouds[0]
    s["ctx"] = M.M1LyaContext(c.lya, c.geometry)
    if case["call"] == "operators":
        s["ctx"].set_voigt_lut(_lut())
        s["gas"] = c.gas
    if case["call"] == "gradient":
        s["mf"], s["spec"] = _seeds(case, c.lya.n_nu, seed)
    return s


# ---------------------------------------------------------------------------
# a pass
# ---------------------------------------------------------------------------
_SCALARS = ("M_F", "M_F_radial_net", "M_F_radial_out", "L_Lya", "f_esc")


def _history(h, f=np.float64):
    """The columns of a history of step scalars; the active bins are whole numbers."""
    out = {k: h[..., i].astype(np.float64 if k == "L_Lya" else f) for i, k in enumerate(_SCALARS)}
    out["bins"] = h[..., 5:7].astype(np.int64)
    return out


def run(s):
    case = s["case"]
    call, n = case["call"], case["steps"]
    (c, dt, zc), bc = s["step"][0], s["bc"][0]
    if call == "batch":
        b = s["batch"]
        if "gas" in s:
            b.prepare_subcycling(0, **s["gas"])
        out = _history(b.run_steps(n), np.float32)
        for i in range(len(b)):
            for k in ("J", "H_r", "H_z"):
                out[f"{k}{i}"] = b.download(i, k).astype(np.float32)
        return out
    ctx = s["ctx"]
    if call == "gradient":
        r = adjoint_run(ctx, n, c, dt, zc, mf_seed=s["mf"], spec_seed=s["spec"], bc_z_bot=bc)
        return dict(_history(r.history), objective=float(r.objective), state=r.grad_state, cell=r.grad_cell,
                    bin=r.grad_bin)
    if call == "operators":
        ctx.prepare_subcycling(**s["gas"])
        for _ in range(n):
            M.advect_lya(c * dt, ctx, bc_z_bot=bc)
            M.lya_emission_absorption_update(ctx, c, dt)
            M.frequency_update_j_lya_all_cells(c * dt, ctx)
        mf = M.update_f_lya_mf_l_lya(ctx, n * dt, zc, bc)
        out = dict(zip(_SCALARS, mf), f_esc=M.compute_f_esc_lya_cylindrical(ctx, mf[3], bc), e_lya=M.update_e_lya(ctx))
        out["f_r"], out["f_z"] = ctx.download("f_r"), ctx.download("f_z")
        M.reset_drhou(ctx)
    elif call == "step":
        rows = [M.step(ctx, c, dt, zc, bc_z_bot=bc) for _ in range(n)]
        out = _history(np.array([list(r.values()) for r in rows]))
    else:
        out = _history(M.run_steps(ctx, n, c, dt, zc, bc_z_bot=bc))
    for k in ("J", "H_r", "H_z"):
        out[k] = ctx.download(k)
    return out


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _cells(case):
    if case["kind"] == "sweep":
        p = W.sweep_params(case["first"] + case["clouds"], DEFAULT_SEED)[case["first"]:]
        return sum(q["n_r"] * q["n_z"] * q["n_nu"] for q in p)
    return case["n_r"] * case["n_z"] * case["n_nu"]


def work(case):
    """Bytes and floating-point operations of a pass, N cell bins and S steps.

    A step reads J, H_r, H_Z, α_F, Hvoigt, ϕ_ν once and writes J, H_r, H_Z once (9 words).  A
    gradient also reads a step's input and the cotangent of its output and writes the cotangent
    of its input: 6 + 9 words.  The operators each pass over the state: advection 7 words,
    emission 8, the frequency update 7.  A step's formulas take about 330 operations per cell
    bin (two interfaces of 90, the cell update 30, emission 20, the frequency factors 60, the
    tridiagonal solve 20, the flux correction and sums 20), a step's reverse about twice that.
    """
    n, steps = _cells(case), case["steps"]
    word = 4 if case["call"] == "batch" else 8
    words = {"gradient": 9 + 15, "operators": 22}.get(case["call"], 9)
    flops = 330 * (3 if case["call"] == "gradient" else 1)
    return {"bytes": float(word * words * n * steps), "flops": float(flops * n * steps)}


# ---------------------------------------------------------------------------
# the same in plain 64-bit torch
# ---------------------------------------------------------------------------
_JEPS, _FMIN, _PMIN, _PMAX = 1e-60, 1e-10, 1e-3, 40.0


def _max(x, v):
    return torch.where(x < v, torch.full_like(x, v), x)


def _minmod(a, b):
    return torch.where(a * b <= 0.0, torch.zeros_like(a), torch.where(a.abs() < b.abs(), a, b))


def _chi(f):
    return (3.0 + 4.0 * f * f) / (5.0 + 2.0 * torch.sqrt(4.0 - 3.0 * f * f))


def _closure(f, nr, nz):
    chi = _chi(f.clamp(_FMIN, 1.0 - _FMIN))
    a, b = 0.5 * (1.0 - chi), 0.5 * (3.0 * chi - 1.0)
    iso = f <= _FMIN
    third = torch.full_like(f, 1.0 / 3.0)
    return (torch.where(iso, third, a + b * nr * nr), torch.where(iso, third, a + b * nz * nz),
            torch.where(iso, torch.zeros_like(f), b * nr * nz))


def _cell_closure(hr, hz, j):
    h2 = hr * hr + hz * hz
    iso = (j <= _JEPS) | (h2 <= 1e-200) | (h2 <= _FMIN * _FMIN * j * j)
    h = torch.sqrt(torch.where(iso, torch.ones_like(h2), h2))
    f = (h / torch.where(iso, torch.ones_like(j), j)).clamp(_FMIN, 1.0 - _FMIN)
    rr, zz, rz = _closure(torch.where(iso, torch.full_like(f, 0.5), f), hr / h, hz / h)
    third = torch.full_like(f, 1.0 / 3.0)
    return torch.where(iso, third, rr), torch.where(iso, third, zz), torch.where(iso, torch.zeros_like(f), rz)


def _work_rate(d, v):
    """D:∇u of the closure d for the velocity gradients v."""
    rr, zz, rz = d
    return rr * v["dur_dr"] + rz * (v["dur_dz"] + v["duz_dr"]) + zz * v["duz_dz"] + _max(1.0 - rr - zz, 0.0) * v["ur_over_r"]


def _eigen(f, mu):
    f, mu = f.clamp(_FMIN, 1.0 - _FMIN), mu.clamp(-1.0, 1.0)
    s = torch.sqrt(4.0 - 3.0 * f * f)
    q = torch.sqrt(_max((2.0 / 3.0) * (4.0 - 3.0 * f * f - s) + 2.0 * mu * mu * (2.0 - f * f - s), 0.0))
    return ((mu * f - q) / s).clamp(-1.0, 1.0), ((mu * f + q) / s).clamp(-1.0, 1.0)


def _ghosts(x, normal, dim, low, high):
    """x with two ghost cells on each side of dim; normal: the flux component along dim."""
    n = x.shape[dim]
    s = lambda a, m: a.narrow(dim, m, 1)  # noqa: E731
    if low == REFLECT:
        lo = [-s(x, 1), -s(x, 0)] if normal else [s(x, 1), s(x, 0)]
    else:
        g = s(x, 0)
        lo = [g.clamp(max=0.0) if normal else g] * 2
    if high == REFLECT:
        hi = [-s(x, n - 1), -s(x, n - 2)] if normal else [s(x, n - 1), s(x, n - 2)]
    else:
        g = s(x, n - 1)
        hi = [g.clamp(min=0.0) if normal else g] * 2
    return torch.cat(lo + [x] + hi, dim)


def _faces(J, Hr, Hz, aF, iv, u, dim, low, high, hll):
    """Fluxes of J, H_r, H_Z through every interface along dim (0: Z, 1: r) and K_ϕϕ on its two sides."""
    n = J.shape[dim]
    at = lambda x, m: x.narrow(dim, m, n + 1)  # noqa: E731
    shape = [n + 1 if d == dim else 1 for d in range(3)]
    dL, dR, im1, ip1, ip2 = (iv[:, m].reshape(shape) for m in range(5))
    P = _ghosts(J, False, dim, low, high)
    iP = 1.0 / _max(P, _JEPS)
    fr = _ghosts(Hr, dim == 1, dim, low, high) * iP
    fz = _ghosts(Hz, dim == 0, dim, low, high) * iP

    def sides(x):
        c = (at(x, 2) - at(x, 1)) * ip1
        return (at(x, 1) + _minmod((at(x, 1) - at(x, 0)) * im1, c) * dL,
                at(x, 2) - _minmod((at(x, 3) - at(x, 2)) * ip2, c) * dR)

    state = []
    for j, r, z in zip(sides(P), sides(fr), sides(fz)):
        j = _max(j, _JEPS)
        f2 = r * r + z * z
        zero = f2 <= 0.0
        f = torch.sqrt(torch.where(zero, torch.ones_like(f2), f2))
        nr, nz = torch.where(zero, f2, r / f), torch.where(zero, f2, z / f)
        f = torch.where(zero, f2, f)
        over = f > 1.0
        r, z, f = torch.where(over, nr, r), torch.where(over, nz, z), torch.where(over, torch.ones_like(f), f)
        rr, zz, rz = _closure(f, nr, nz)
        flux = (r * j, rr * j, rz * j) if dim == 1 else (z * j, rz * j, zz * j)
        state.append(dict(U=(j, r * j, z * j), F=flux, f=f, mu=nr if dim == 1 else nz, kphi=(1.0 - rr - zz).clamp(0.0, 1.0) * j))
    a, b = state
    first, last = aF.narrow(dim, 0, 1), aF.narrow(dim, n - 1, 1)
    tau = torch.cat([first, aF], dim) * dL + torch.cat([aF, last], dim) * dR
    tau = torch.where(tau == 0.0, tau.detach(), tau)   # an empty cell's opacity is no parameter
    den = 1.0 / (0.2 + tau + tau * tau)
    eps, ome = (0.2 + tau) * den, tau * tau * den
    diff = -(1.0 / 3.0) * (at(P, 2) - at(P, 1)) * tau * den   # (1 - ϵ) times Fick's flux
    if hll:
        (l1a, l3a), (l1b, l3b) = _eigen(a["f"], a["mu"]), _eigen(b["f"], b["mu"])
        sr, sl = _max(torch.maximum(l3a, l3b), 0.0), torch.minimum(l1a, l1b).clamp(max=0.0)
        ids = 1.0 / _max(sr - sl, 1e-300)
        G = [(sr * p - sl * q + sr * sl * (v - w)) * ids for p, q, v, w in zip(a["F"], b["F"], b["U"], a["U"])]
        F = [eps * G[0] + diff] + [eps * G[m] + 0.5 * ome * (a["F"][m] + b["F"][m]) for m in (1, 2)]
    else:
        G = 0.5 * (a["F"][0] + b["F"][0]) - 0.5 * (b["U"][0] - a["U"][0])
        F = [eps * G + diff] + [0.5 * (a["F"][m] + b["F"][m]) - 0.5 * eps * (b["U"][m] - a["U"][m]) for m in (1, 2)]
    up = u < 0.0
    F = [x + u * torch.where(up, q, p) for x, p, q in zip(F, a["U"], b["U"])]
    kphi_R = b["kphi"]
    if dim == 1:   # the axis: the closure of the flux along Z alone
        j, z = b["U"][0].narrow(1, 0, 1), b["U"][2].narrow(1, 0, 1)
        q = (z / j).clamp(-1.0, 1.0)
        rr, zz, _ = _closure(q.abs(), torch.zeros_like(q), torch.sign(q))
        kphi_R = torch.cat([(1.0 - rr - zz).clamp(0.0, 1.0) * j, kphi_R.narrow(1, 1, n)], 1)
    return F, a["kphi"], kphi_R


class _Exact:
    """One cloud and its step, with tensors in `p` that a gradient can be taken of."""

    def __init__(self, cloud):
        dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
        t = lambda a: torch.as_tensor(np.ascontiguousarray(a, dtype=np.float64), device=dev)  # noqa: E731
        L, g = cloud.lya, cloud.geometry
        self.t, self.L = t, L
        self.c, self.dt, self.zc, self.bc = cloud.c_tilde, cloud.dt, cloud.Zc, cloud.bc_z_bot
        self.X = tuple(t(L[k]) for k in ("J", "H_r", "H_z"))
        self.p = {k: t(L[k]) for k in ("alpha_F", "Hvoigt", "phi", "alpha", "alpha_c", "pd", "js", "dnuD", "T")}
        self.v = {k: t(L[k])[..., None] for k in ("dur_dr", "dur_dz", "duz_dr", "duz_dz", "ur_over_r", "ur_star", "uz_star")}
        self.g = {k: t(getattr(g, k)) for k in ("dV", "inv_dV", "A_r", "A_Z", "inv_r_cell", "rCoM", "ZCoM")}
        self.nu, self.nuC, self.dnu = t(L.nu), t(L["nuC"]), t(L["dnu"])

        def intervals(d):
            dL, dR, a, b, e, inner, outer = d
            mid = np.stack([dL, dR, a, b, e], axis=1)[:-1]
            return t(np.concatenate([inner[None], mid, outer[None]]))

        self.ivr, self.ivz = intervals(g.dr), intervals(g.dZ)

    def refresh(self, gas):
        """The coefficients of a gas state: Voigt tables, ϕ_ν over all bins, α, α_F."""
        t, lut = self.t, _lut()
        T, n = t(gas["T"]), t(gas["n_HI"])
        tab = t(lut.t)
        b = K.b_PREFACT * torch.sqrt(T)
        ic, a = (1.0 / (b * K.nu_Lya_over_c))[..., None], (K.a_PREFACT / b)[..., None]

        def fn(m, x):
            xs = torch.where(x.abs() < lut.xmax, x, torch.zeros_like(x))
            s = (xs - lut.xmin) * lut.inv_dx
            i = torch.floor(s).long().clamp(max=lut.nx - 2)
            w = (i + 1).double() - s
            far = {0: lambda: torch.sign(x), 1: lambda: 0.5 / x + 0.25 / x ** 3}.get(m, lambda: torch.zeros_like(x))()
            return torch.where(x.abs() < lut.xmax, w * tab[m][i] + (1.0 - w) * tab[m][i + 1], far)

        h = math.sqrt(math.pi) / 2.0
        prim = lambda x: h * fn(0, x) - (1.0 / h) * a * fn(1, x) + a * a * fn(3, x)  # noqa: E731
        e, x = t(self.L["dnu_rel"]) * ic, t(self.L["dnuC_rel"]) * ic
        dx = e[..., 1:] - e[..., :-1]
        q = prim(e)
        Hv = torch.where(dx > 1e-5, (q[..., 1:] - q[..., :-1]) / dx,
                         fn(2, x) + (1.0 / h) * a * (2.0 * x * fn(1, x) - 1.0) + a * a * fn(4, x))
        p = self.p
        p["alpha"] = n * (K.sigma0_PREFACT / b)
        p["phi"] = Hv / (self.dnu * Hv).sum(-1, keepdim=True)
        p["Hvoigt"], p["dnuD"], p["T"] = Hv, b * K.nu_Lya_over_c, T
        p["alpha_F"] = p["alpha"][..., None] * Hv + t(gas["alpha_c_F"])[..., None]
        p["alpha_c"], p["js"], p["pd"] = t(gas["alpha_c"]), t(gas["js"]), t(gas["pd"])

    def active(self, J):
        w = self.g["dV"][..., None] * self.dnu
        J = J.detach()
        e1 = (w * _max(J - _JEPS, 0.0)).sum((0, 1))
        on = torch.nonzero((w * _max(J - 10 * _JEPS, 0.0)).sum((0, 1)) > 1e-10 * e1.sum()).flatten().tolist()
        lo, hi = (on[0], on[-1]) if on else (len(self.dnu) - 1, 0)
        return min(lo, self.L.kcore[0]), max(hi, self.L.kcore[1])

    def advect(self, X, cdt):
        lo, hi = self.active(X[0])
        J, Hr, Hz = (x[..., lo:hi + 1] for x in X)
        aF, g, v = self.p["alpha_F"][..., lo:hi + 1], self.g, self.v
        hll = bool(self.L.hll)
        Fr, kl, kr = _faces(J, Hr, Hz, aF, self.ivr, v["ur_star"] / K.c, 1, REFLECT, OUTFLOW, hll)
        Fz, _, _ = _faces(J, Hr, Hz, aF, self.ivz, v["uz_star"] / K.c, 0, self.bc, OUTFLOW, hll)
        w, nr = cdt * g["inv_dV"][..., None], J.shape[1]
        Ar, Az = g["A_r"][..., None], g["A_Z"][..., None]

        def div(m):
            a, b = Ar * Fr[m], Az * Fz[m]
            return (a[:, 1:] - a[:, :-1]) + (b[1:] - b[:-1])

        Ddu = _work_rate(_cell_closure(Hr, Hz, J), v)
        Jn = _max(J - w * div(0), _JEPS)
        Hrn = Hr - w * div(1) + cdt * 0.5 * (kr[:, :nr] + kl[:, 1:]) * g["inv_r_cell"][None, :, None]
        Hrn = Hrn - cdt / K.c * (Hr * v["dur_dr"] + Hz * v["dur_dz"])
        Hzn = Hz - w * div(2) - cdt / K.c * (Hr * v["duz_dr"] + Hz * v["duz_dz"])
        Jn = _max(Jn - cdt / K.c * Ddu * J, _JEPS)
        Y = self.causal(Jn, Hrn, Hzn)
        return tuple(torch.cat([x[..., :lo], y, x[..., hi + 1:]], -1) for x, y in zip(X, Y)), (lo, hi)

    @staticmethod
    def causal(J, Hr, Hz):
        h2 = Hr * Hr + Hz * Hz
        over = h2 > J * J
        s = torch.where(over, J / torch.sqrt(torch.where(over, h2, torch.ones_like(h2))), torch.ones_like(J))
        return J, Hr * s, Hz * s

    def emit(self, X):
        """Emission and absorption; also the momentum the cells took up."""
        J, Hr, Hz = X
        p, cdt = self.p, self.c * self.dt
        aJ = p["alpha_c"][..., None] + (p["alpha"] * p["pd"])[..., None] * p["Hvoigt"]
        Jn = (J + p["js"][..., None] * cdt * p["phi"]) / (1.0 + aJ * cdt)
        q = 1.0 + p["alpha_F"] * cdt
        Hrn, Hzn = Hr / q, Hz / q
        s = K.Four_pi / K.c / self.c
        return (Jn, Hrn, Hzn), (s * ((Hr - Hrn) * self.dnu).sum(-1), s * ((Hz - Hzn) * self.dnu).sum(-1))

    def diffuse(self, X, cdt):
        """Frequency diffusion and drift: the exponentially fitted rows, their solve, the fluxes' correction."""
        J, Hr, Hz = X
        p, nu, nuC = self.p, self.nu, self.nuC
        Hv = p["Hvoigt"]
        pre = (0.5 * torch.clamp(p["alpha"], min=self.L.alpha_floor) * p["dnuD"] ** 2)[..., None]
        vel = _work_rate(_cell_closure(Hr, Hz, J), self.v)[..., 1:-1] / K.c
        recoil = (K.h / K.kB / p["T"])[..., None] if self.L.recoil else None
        mid, low, up = slice(1, -1), slice(0, -2), slice(2, None)

        def expo(s, half):
            k = pre * Hv[..., s]
            c = vel * nuC[s]
            if recoil is not None:
                c = c + k * (recoil - 2.0 / nuC[s])
            q = half / k
            return (c * q).clamp(-_PMAX, _PMAX), q

        def fit(x, sign):
            small = x.abs() < _PMIN
            xs = torch.where(small, torch.ones_like(x), x)
            o = torch.where(small, 1.0 + sign * x + 0.5 * x * x, torch.exp(sign * xs))
            return o, torch.where(small, -sign - 0.5 * x, -torch.expm1(sign * xs) / xs)

        P, q = expo(mid, nu[2:-1] - nuC[mid])
        Pp, qp = expo(up, nuC[up] - nu[2:-1])
        Pm, qm = expo(low, nu[1:-2] - nuC[low])
        oL, xL = fit(P, -1.0)
        oR, xR = fit(P, 1.0)
        oRp, xRp = fit(Pp, 1.0)
        oLm, xLm = fit(Pm, -1.0)
        idn = 1.0 / self.dnu[mid]
        gp, gm = idn / (xL * q - xRp * qp), idn / (xLm * qm - xR * q)
        dw = 1.0 / cdt
        rows = lambda x: x.reshape(-1, x.shape[-1]).t().contiguous().unbind(0)  # noqa: E731
        A, B, C, D = (rows(x) for x in (oLm * gm, -(oL * gp + oR * gm + dw), oRp * gp, -dw * J[..., mid]))
        n = len(B)
        cs, ds = [C[0] / B[0]], [D[0] / B[0]]
        for r in range(1, n):
            m = B[r] - A[r] * cs[-1]
            cs.append(C[r] / m)
            ds.append((D[r] - A[r] * ds[-1]) / m)
        x = [ds[-1]]
        for r in range(n - 2, -1, -1):
            x.append(ds[r] - cs[r] * x[-1])
        x = torch.stack(x[::-1], 0).t().reshape(J[..., mid].shape)
        Jn = _max(torch.cat([J[..., :1], x, J[..., -1:]], -1), _JEPS)
        ratio = Jn / _max(J, _JEPS)
        return self.causal(Jn, Hr * ratio, Hz * ratio)

    def scalars(self, momentum, dt, H):
        g, L = self.g, K.Four_pi * (self.g["dV"] * self.p["js"]).sum()
        fr, fz = momentum[0] / dt, momentum[1] / dt
        d = torch.stack(torch.broadcast_tensors(g["rCoM"][None, :], (g["ZCoM"] - self.zc)[:, None]))
        frad = (fr * d[0] + fz * d[1]) / torch.sqrt((d * d).sum(0))
        f2 = fr * fr + fz * fz
        f = torch.where(f2 > 0.0, torch.sqrt(torch.where(f2 > 0.0, f2, torch.ones_like(f2))), f2)
        MF = [K.c / L * (g["dV"] * x).sum() for x in (f, frad, _max(frad, 0.0))]
        Ltot = 2.0 * L if self.bc == REFLECT else L
        return MF + [Ltot, (self.spectrum(*H) * self.dnu).sum()]

    def spectrum(self, Hr, Hz):
        g, L = self.g, K.Four_pi * (self.g["dV"] * self.p["js"]).sum()
        s = (g["A_r"][:, -1, None] * _max(Hr[:, -1], 0.0)).sum(0) + (g["A_Z"][-1][:, None] * _max(Hz[-1], 0.0)).sum(0)
        if self.bc == OUTFLOW:
            s = s + (g["A_Z"][0][:, None] * _max(-Hz[0], 0.0)).sum(0)
        return K.Four_pi * s / L

    def step(self, X):
        X, bins = self.advect(X, self.c * self.dt)
        X, mom = self.emit(X)
        X = self.diffuse(X, self.c * self.dt)
        return X, self.scalars(mom, self.dt, X[1:]), bins

    def gradient(self, n, mf, spec):
        """Objective and gradients over n steps, one step's graph at a time."""
        names = ("alpha", "alpha_c", "js", "dnuD", "T", "alpha_F", "Hvoigt", "phi")
        tape, rows, bins, X = [], [], [], self.X
        with torch.no_grad():
            for _ in range(n):
                tape.append(X)
                X, s, b = self.step(X)
                rows.append(torch.stack(s))
                bins.append(b)
        for k in names:
            self.p[k] = self.p[k].clone().requires_grad_(True)
        leaves = [self.p[k] for k in names]
        mf, spec = self.t(mf), self.t(spec)
        obj = float((torch.stack(rows)[:, :3] * mf).sum())
        X = [x.clone().requires_grad_(True) for x in X]
        end = (self.spectrum(*X[1:]) * spec).sum()
        obj += float(end.detach())
        g = torch.autograd.grad(end, list(X) + leaves, allow_unused=True)
        z = lambda v, w: torch.zeros_like(w) if v is None else v  # noqa: E731
        lam = [z(a, b) for a, b in zip(g[:3], X)]
        tot = [z(a, b) for a, b in zip(g[3:], leaves)]
        for s in range(n - 1, -1, -1):
            Y = [x.clone().requires_grad_(True) for x in tape.pop()]
            Z, sc, _ = self.step(Y)
            out = sum((a * b).sum() for a, b in zip(Z, lam)) + sum(sc[m] * mf[s, m] for m in range(3))
            g = torch.autograd.grad(out, Y + leaves, allow_unused=True)
            lam = [z(a, b) for a, b in zip(g[:3], Y)]
            tot = [a + z(b, c) for a, b, c in zip(tot, g[3:], leaves)]
        grads = dict(zip(names, tot))
        cell = {k: grads[k] for k in names[:5]}
        return rows, bins, obj, dict(zip(("J", "H_r", "H_z"), lam)), cell, {k: grads[k] for k in names[5:]}


def _columns(rows, bins, f=torch.float64):
    h = torch.stack([r if torch.is_tensor(r) else torch.stack(r) for r in rows])
    out = {k: h[:, i].to(torch.float64 if k == "L_Lya" else f) for i, k in enumerate(_SCALARS)}
    out["bins"] = torch.tensor(bins, dtype=torch.int64)
    return out


def exact(case, seed):
    # a step takes a few milliseconds per million cell bins here, a gradient's several times that
    cost = _cells(case) / 1e6 * case["steps"] * (6 if case["call"] == "gradient" else 1) + 15 * case["steps"] / 8
    if cost > 6000:
        return None
    clouds = _clouds(case, seed)
    n, call = case["steps"], case["call"]
    if call == "gradient":
        e = _Exact(clouds[0])
        rows, bins, obj, state, cell, per_bin = e.gradient(n, *_seeds(case, e.L.n_nu, seed))
        # between cells of a small opacity the formulas as written form 1 - ϵ by cancellation, and the
        # derivative along α_F, divided by the opacity, has no digits to compare there
        per_bin["alpha_F"] = None
        return dict(_columns(rows, bins), objective=obj, state=state, cell=cell, bin=per_bin)
    with torch.no_grad():
        if call == "operators":
            e = _Exact(clouds[0])
            e.refresh(clouds[0].gas)
            X, mom = e.X, None
            for _ in range(n):
                X, _ = e.advect(X, e.c * e.dt)
                X, m = e.emit(X)
                mom = m if mom is None else (mom[0] + m[0], mom[1] + m[1])
                X = e.diffuse(X, e.c * e.dt)
            out = dict(zip(_SCALARS, (float(v) for v in e.scalars(mom, n * e.dt, X[1:]))))
            out["e_lya"] = K.Four_pi / K.c * (X[0] * e.dnu).sum(-1)
            out["f_r"], out["f_z"] = mom[0] / (n * e.dt), mom[1] / (n * e.dt)
            return dict(out, J=X[0], H_r=X[1], H_z=X[2])
        if call != "batch":
            e = _Exact(clouds[0])
            X, rows, bins = e.X, [], []
            for _ in range(n):
                X, s, b = e.step(X)
                rows.append(s)
                bins.append(b)
            return dict(_columns(rows, bins), J=X[0], H_r=X[1], H_z=X[2])
        out, cols = {}, []
        for i, c in enumerate(clouds):
            e = _Exact(c)
            if case["kind"] == "turbulent":
                e.refresh(c.gas)
            X, rows = e.X, []
            for _ in range(n):
                X, s, b = e.step(X)
                rows.append(torch.stack(s))
            cols.append(torch.stack(rows))
            for k, x in zip(("J", "H_r", "H_z"), X):
                out[f"{k}{i}"] = x
        h = torch.stack(cols, 1)
        out.update({k: h[..., i] for i, k in enumerate(_SCALARS)})
        return dict(out, bins=None)
