"""Workloads of the super-droplet step that are timed: what programs have this library do.

A simulation case is one member of an ensemble, from its initial drops to what is written at the
end: the drops go to the store (which sorts them), the gridbox State and the random stream are
set, some coupling intervals of steps run, the observers read their moments after each, and at the
end State and drops are read back.  The other cases are single entry points with device arrays on
both sides: the sort without allocation, and the learned warm start's gradient, inference and
training.
"""
import ctypes as C
import math

import numpy as np
import torch

from cleo_amd import abi, lib
from cleo_amd import populations as P

# Tilings: "default" is a context as cleo_create leaves it, which the examples and most programs on
# small domains keep; the other is the one cleo_autotune picks for large domains (a program tunes once
# and keeps it; written out here so that every run times the same kernels).
TUNED = (1, 1, 1, 1, 1, 65536, 0, 32768, 1, 8)

_SOLUTE = {"golovin": P.NACL, "coal_breakup": P.NACL, "condensation": P.AMMONIUM_SULPHATE,
           "coupled": P.AMMONIUM_SULPHATE}


def listed():
    return [
        # The Golovin box model of the reference's examples: one gridbox of 8192 drops, one minute of
        # 1 s steps between two outputs.
        _sim("golovin_box_8192", "golovin", (1, 1, 1), 8192, steps=60, host=True),
        # A Low-List box model (coalescence, then breakup) with few drops, stepped one call at a
        # time: launch latency.
        _sim("lowlist_box_501", "golovin", (1, 1, 1), 501, steps=30, eager=True, chain="lowlist", host=True),
        # A rain shaft of 40 gridboxes whose observers read every step, as the observer example does.
        _sim("column_observed", "coupled", (40, 1, 1), 48, steps=1, intervals=20, eager=True, observe=True, host=True),
        # A 2-D flow of ordinary size with the default tiling, coupled every 10 steps.
        _sim("coupled_2d_75x50", "coupled", (75, 50, 1), 128, steps=10, intervals=3, observe=True),
        # The ordinary 3-D domain.
        _sim("coupled_32cubed", "coupled", (32, 32, 32), 64, steps=20, intervals=3, observe=True, tuned=True),
        # Ragged extents and gridboxes of more than 255 drops.
        _sim("coupled_ragged_300", "coupled", (37, 29, 23), 300, steps=20, observe=True, tuned=True),
        # The large coupled domain (33.5M drops), one minute between outputs.
        _sim("coupled_33m", "coupled", (128, 64, 64), 64, steps=60, observe=True, tuned=True),
        # The coupled step with the learned warm start.
        _sim("coupled_learned_8m", "coupled", (64, 64, 32), 64, steps=30, observe=True, tuned=True, learned=True),
        # Collisions alone: coalescence and breakup on 64 cubed gridboxes of Poisson(128) drops.
        _sim("collisions_64cubed", "coal_breakup", (64, 64, 64), 128, steps=120, tuned=True),
        # Condensation alone: 64 cubed gridboxes of Poisson(122) drops.
        _sim("condensation_64cubed", "condensation", (64, 64, 64), 122, steps=60, tuned=True),
        # The generic sort between device arrays, drops in random order.
        dict(name="sort_1m", kind="sort", n=1000003, ngbx=32768),
        # The warm start's network: gradient and inference on a large batch, and a short training.
        dict(name="mlp_train_2m", kind="mlp", n=2097152, batch=65536, epochs=1, seed0=7),
    ]


def _sim(name, pop, ndims, mean, steps, intervals=1, eager=False, observe=False, tuned=False, learned=False,
         chain="standard", host=False, spacing=25.0):
    if pop in ("coal_breakup", "condensation"):
        spacing = 50.0
    return dict(name=name, kind="sim", pop=pop, nz=ndims[0], nx=ndims[1], ny=ndims[2], mean=mean, steps=steps,
                intervals=intervals, eager=eager, observe=observe, tuned=tuned, learned=learned, chain=chain,
                host=host, spacing=spacing)


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    pick = rng.random()
    if pick < 0.10:
        return dict(kind="sort", n=_log_int(rng, 5, 1 << 20), ngbx=_log_int(rng, 1, 1 << 20))
    if pick < 0.22:
        n = _log_int(rng, 4096, 1 << 21)
        return dict(kind="mlp", n=n, batch=min(n, _log_int(rng, 1000, 65536)), epochs=1, seed0=rng.randint(1, 1000))
    if pick < 0.42:  # boxes
        low = rng.random() < 0.5
        c = _sim("", "golovin", (1, 1, 1), _log_int(rng, 100, 20000), steps=rng.randint(5, 60), eager=low,
                 chain="lowlist" if low else "standard", host=True)
    else:
        pop = rng.choice(["coupled", "coupled", "coupled", "coal_breakup", "condensation"])
        drops = math.exp(rng.uniform(math.log(2e3), math.log(2e7)))
        mean = _log_int(rng, 8, 400)
        ngbx = max(1.0, drops / mean)
        shape = rng.choice([1, 2, 3])
        side = ngbx ** (1.0 / shape)
        dims = [1, 1, 1]
        for i in range(shape):
            dims[i] = max(1, int(round(side * rng.uniform(0.7, 1.4))))
        small = dims[0] * dims[1] * dims[2] * mean < 3e5
        c = _sim("", pop, tuple(dims), mean, steps=rng.randint(3, 20), intervals=rng.randint(1, 2),
                 eager=rng.random() < 0.3, observe=rng.random() < 0.7, tuned=(not small) or rng.random() < 0.3,
                 learned=pop == "coupled" and not small and rng.random() < 0.25)
    del c["name"]
    return c


# ---- inputs ------------------------------------------------------------------------------------
def _drops(case, seed):
    """(device arrays of the drops, State as numpy arrays, faces)"""
    nd = (case["nz"], case["nx"], case["ny"])
    dev = torch.device("cuda:0")
    if case["pop"] == "golovin":
        pop = P.golovin_box(seed=seed, nsupers=int(case["mean"]))
        if case["chain"] == "lowlist":  # radii in the range of the Low-List fit, a trace of solute
            pop.supers["radius"] = np.clip(pop.supers["radius"], 0.1, 90.0)
            pop.supers["msol"] = np.full(pop.n, 4.0 / 3.0 * np.pi * 1e-30 * P.NACL["rho"] / P.RHO0)
        view = {"uint32": np.int32, "uint64": np.int64}
        sup = {k: torch.from_numpy(v.view(view.get(str(v.dtype), v.dtype)).copy()).to(dev) for k, v in
               pop.supers.items()}
        return sup, pop.state, pop.halves
    gen = dict(coupled=P.coupled_device, coal_breakup=P.coal_breakup_device, condensation=P.condensation_device)
    return gen[case["pop"]](torch, dev, seed=seed, ndims=nd, spacing_m=case["spacing"], mean=case["mean"])


def _soa(arrays):
    s = abi.SupersSoA()
    for (name, _), (_, ctype) in zip(abi.SUPER_FIELDS, abi.SupersSoA._fields_):
        setattr(s, name, C.cast(C.c_void_p(arrays[name].data_ptr()), ctype))
    return s


def _gbx(arrays):
    s = abi.GbxState()
    for name, ctype in abi.GbxState._fields_:
        setattr(s, name, C.cast(C.c_void_p(arrays[name].data_ptr()), ctype))
    return s


def _like(n, dtype):
    return torch.empty(n, dtype=dtype, pin_memory=True)


def _params(case):
    """The chain of microphysical processes and the motion of a simulation case."""
    cond = abi.CondParams(100, 1, 50, 1e-6, 1e-8, 0.001, int(case["learned"]), 10)
    coll = abi.CollParams(100, abi.PROB_LONG, 1.0, abi.ENACT_COALBURE, 5.0, 0.85)
    if case["chain"] == "lowlist":
        coal = abi.CollParams(100, abi.PROB_LOWLIST_COAL, 1.0, abi.ENACT_COAL, 5.0, 0.85, prob_tv=abi.TV_ROGERS_GK)
        bu = abi.CollParams(100, abi.PROB_LOWLIST_BU, 1.0, abi.ENACT_BREAKUP, 5.0, 0.85, prob_tv=abi.TV_ROGERS_GK)
        return [abi.coll_process(coal), abi.coll_process(bu)], None
    if case["pop"] == "golovin":
        return [abi.coll_process(abi.CollParams(100, abi.PROB_GOLOVIN, 0.0, abi.ENACT_COAL, 0.0, 0.0))], None
    if case["pop"] == "coal_breakup":
        return [abi.coll_process(coll)], None
    if case["pop"] == "condensation":
        return [abi.cond_process(cond)], None
    return [abi.cond_process(cond), abi.coll_process(coll)], abi.MotionParams(100, abi.TV_SIMMEL)


def prepare(case, seed):
    return {"sim": _prepare_sim, "sort": _prepare_sort, "mlp": _prepare_mlp}[case["kind"]](case, seed)


def run(state):
    return state["run"](state)


def _prepare_sim(case, seed):
    b = lib.load()
    sup, gbx, halves = _drops(case, seed)
    if case["host"]:
        sup = {k: v.cpu() for k, v in sup.items()}
    torch.cuda.synchronize()
    n = sup["xi"].numel()
    d = abi.Domain(b, n, (case["nz"], case["nx"], case["ny"]), *halves)
    d.set_solute(*P.solute_dimless(_SOLUTE[case["pop"]]))
    if case["tuned"]:
        d.check(b.set_tiles(d.h, C.byref(abi.Tiles(*TUNED))), "set_tiles")
    procs, motion = _params(case)
    d.check(d.set_sdm_chain(procs, motion), "set_sdm_chain")
    gbx_in = {k: torch.from_numpy(np.ascontiguousarray(gbx[k])).pin_memory() for k in abi.STATE_FIELDS}
    # what is read back goes to arrays of the program's capacity: the number of drops is random
    expected = case["mean"] * d.ngbx
    cap = expected if case["pop"] == "golovin" else int(expected + 8.0 * math.sqrt(expected) + 64.0)
    out = {k: _like(max(n, cap), v.dtype).zero_() for k, v in sup.items()}
    out_gbx = {k: _like(d.ngbx, torch.float64) for k in abi.STATE_FIELDS}
    mom = [[_like(d.ngbx, torch.int64), _like(d.ngbx, torch.float32), _like(d.ngbx, torch.float32)] for _ in range(2)]
    s = dict(run=_run_sim, case=case, d=d, n=n, seed=int(seed), sup=sup, gbx_in=gbx_in, out=out, out_gbx=out_gbx,
             mom=mom, c_sup=_soa(sup), c_gbx=_gbx(gbx_in), c_out=_soa(out), c_out_gbx=_gbx(out_gbx))
    if case["learned"]:  # the network learns the plain solver on this population
        L = b.lib
        _start(s)
        cap = min(n, 1 << 20)
        x = torch.zeros((cap, 8), device="cuda", dtype=torch.float32)
        y = torch.zeros(cap, device="cuda", dtype=torch.float32)
        torch.cuda.synchronize()
        got = C.c_uint64()
        plain = abi.CondParams(100, 1, 50, 1e-6, 1e-8, 0.001, 0, 10)
        d.check(L.cleo_mlp_make_samples(d.h, C.byref(plain), x.data_ptr(), y.data_ptr(), cap, C.byref(got)), "samples")
        tp = abi.MLPTrainParams(40, min(8192, int(got.value)), 2e-3, 0.9, 0.999, 1e-8, 11)
        loss = C.c_float()
        d.check(L.cleo_mlp_train(d.h, x.data_ptr(), y.data_ptr(), got.value, C.byref(tp), C.byref(loss)), "train")
    return s


def _start(s):
    """The initial drops, State and random stream."""
    d, b = s["d"], s["d"].b
    if s["case"]["host"]:
        d.check(b.upload_supers(d.h, C.byref(s["c_sup"]), s["n"]), "upload_supers")
    else:
        d.check(b.lib.cleo_upload_supers_device(d.h, C.byref(s["c_sup"]), s["n"]), "upload_supers_device")
    d.check(b.upload_gbx_state(d.h, C.byref(s["c_gbx"])), "upload_gbx_state")
    d.rng_counter(s["seed"], 0)


def _moments(s, rain):
    d, m = s["d"], s["mom"][rain]
    u64, f32 = C.POINTER(C.c_uint64), C.POINTER(C.c_float)
    p = [C.cast(C.c_void_p(t.data_ptr()), u64 if i == 0 else f32) for i, t in enumerate(m)]
    d.check(d.b.mass_moments(d.h, rain, *p), "mass_moments")


def _run_sim(s):
    d, case = s["d"], s["case"]
    b = d.b
    _start(s)
    t = 0
    for _ in range(case["intervals"]):
        if case["eager"]:
            for _ in range(case["steps"]):
                d.check(d.run_step(t, t + 100), "run_step")
                t += 100
        else:
            d.check(b.lib.cleo_run_steps_graph(d.h, t, 100, case["steps"]), "run_steps_graph")
            t += 100 * case["steps"]
        if case["observe"]:
            _moments(s, 0)
            _moments(s, 1)
    d.check(b.download_gbx_state(d.h, C.byref(s["c_out_gbx"])), "download_gbx_state")
    ntot, ndom = C.c_uint64(), C.c_uint64()
    d.check(b.download_supers(d.h, C.byref(s["c_out"]), C.byref(ntot), C.byref(ndom)), "download_supers")
    return dict(supers=s["out"], state=s["out_gbx"], ndomain=int(ndom.value), moments=s["mom"] if case["observe"] else None)


def _sort_inputs(case, seed):
    """Drops in random order, one in a hundred out of the domain."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed))
    n = case["n"]
    key = torch.randint(0, case["ngbx"], (n,), device="cuda", generator=gen)
    gone = torch.rand(n, device="cuda", generator=gen) < 0.01
    f = lambda: torch.rand(n, device="cuda", dtype=torch.float64, generator=gen)  # noqa: E731
    return dict(sdgbxindex=torch.where(gone, torch.full_like(key, -1), key).to(torch.int32), coord3=f(), coord1=f(),
                coord2=f(), xi=torch.randint(1, 10 ** 8, (n,), device="cuda", generator=gen), radius=f(), msol=f(),
                sdid=torch.arange(n, device="cuda"))


def _prepare_sort(case, seed):
    b = lib.load()
    fn = b.lib.cleo_sort_supers_noalloc
    fn.restype = C.c_int
    fn.argtypes = [C.c_void_p, C.c_void_p, C.c_void_p, C.c_uint64, C.c_uint32, C.c_void_p]
    inp = _sort_inputs(case, seed)
    out = {k: torch.empty_like(v) for k, v in inp.items()}
    refs = torch.empty(case["ngbx"] + 1, device="cuda", dtype=torch.int32)
    return dict(run=_run_sort, case=case, fn=fn, inp=inp, out=out, refs=refs, c_in=_soa(inp), c_out=_soa(out))


def _run_sort(s):
    stream = torch.cuda.current_stream().cuda_stream
    rc = s["fn"](C.byref(s["c_in"]), C.byref(s["c_out"]), s["refs"].data_ptr(), s["case"]["n"], s["case"]["ngbx"], stream)
    if rc != 0:
        raise RuntimeError("cleo_sort_supers_noalloc: %d" % rc)
    return dict(out=s["out"], refs=s["refs"])


def _mlp_inputs(case, seed):
    """Features with the ranges of the coupled population and a smooth growth to learn, and the
    weights (bf16-representable, so that 64-bit references start from the same numbers)."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed))
    n = case["n"]
    u = lambda lo, hi: lo + (hi - lo) * torch.rand(n, device="cuda", generator=gen)  # noqa: E731
    x = torch.zeros((n, 8), device="cuda", dtype=torch.float32)
    x[:, 0] = u(-3.0, 4.0)
    x[:, 1] = u(-2.0, 6.0)
    x[:, 2] = u(0.95, 1.01)
    x[:, 3] = u(0.99, 1.10)
    x[:, 4] = u(0.7, 1.0)
    x[:, 5] = 0.001
    y = 0.1 * torch.tanh(x[:, 2] * 40.0 - 40.0) * torch.exp(-x[:, 0]) + 0.02 * torch.sin(x[:, 1])
    rng = np.random.default_rng(int(seed) + 1)
    blob = np.zeros(abi.MLP_NBLOB, dtype=np.float32)
    h = abi.MLP_HID
    blob[:h * 6] = rng.uniform(-1.0, 1.0, h * 6)
    o = h * 6
    blob[o:o + h] = rng.uniform(-0.2, 0.2, h)
    o += h
    blob[o:o + h * h] = rng.uniform(-0.3, 0.3, h * h)
    o += h * h
    blob[o:o + h] = rng.uniform(-0.2, 0.2, h)
    o += h
    blob[o:o + h] = rng.uniform(-0.3, 0.3, h)
    blob[:o + h] = torch.from_numpy(blob[:o + h]).to(torch.bfloat16).to(torch.float32).numpy()
    o = abi.MLP_NPARAMS
    blob[o:o + 6] = [0.5, 2.0, 0.98, 1.05, 0.85, 0.001]
    blob[o + 6:o + 12] = [2.0, 2.3, 0.017, 0.03, 0.09, 1e-3]
    blob[o + 12:o + 14] = [0.0, 0.05]
    return x, y.contiguous(), blob


def _prepare_mlp(case, seed):
    b = lib.load()
    x, y, blob = _mlp_inputs(case, seed)
    d = abi.Domain(b, 64, (1, 1, 1), *P.uniform_grid((1, 1, 1), 100.0))
    torch.cuda.synchronize()
    return dict(run=_run_mlp, case=case, d=d, x=x, y=y, blob=blob, yp=torch.empty_like(y),
                grad=np.zeros(abi.MLP_NPARAMS, dtype=np.float32), trained=np.zeros(abi.MLP_NBLOB, dtype=np.float32))


def _run_mlp(s):
    d, L, case = s["d"], s["d"].b.lib, s["case"]
    fp = C.POINTER(C.c_float)
    ptr = lambda a: a.ctypes.data_as(fp)  # noqa: E731
    d.check(L.cleo_mlp_set_weights(d.h, ptr(s["blob"])), "mlp_set_weights")
    loss, final = C.c_float(), C.c_float()
    d.check(L.cleo_mlp_loss_grad(d.h, s["x"].data_ptr(), s["y"].data_ptr(), case["n"], C.byref(loss), ptr(s["grad"])),
            "mlp_loss_grad")
    d.check(L.cleo_mlp_forward(d.h, s["x"].data_ptr(), s["yp"].data_ptr(), case["n"]), "mlp_forward")
    tp = abi.MLPTrainParams(case["epochs"], case["batch"], 1e-3, 0.9, 0.999, 1e-8, case["seed0"])
    d.check(L.cleo_mlp_train(d.h, s["x"].data_ptr(), s["y"].data_ptr(), case["n"], C.byref(tp), C.byref(final)),
            "mlp_train")
    d.check(L.cleo_mlp_get_weights(d.h, ptr(s["trained"])), "mlp_get_weights")
    return dict(y=s["yp"], loss=float(loss.value), grad=s["grad"], trained=s["trained"], final_loss=float(final.value))


# ---- 64-bit references ---------------------------------------------------------------------------
def exact(case, seed):
    """The sort and the network's output and gradient in 64 bits.  A simulation has none: its steps
    in plain numpy (serial shuffles, a Newton solve per drop) take minutes; nor has a training."""
    if case["kind"] == "sort":
        inp = _sort_inputs(case, seed)
        key = inp["sdgbxindex"].to(torch.int64)
        key = torch.where(key < 0, torch.full_like(key, case["ngbx"]), key)
        at = torch.sort(key, stable=True).indices
        refs = torch.searchsorted(key[at].contiguous(), torch.arange(case["ngbx"] + 1, device="cuda"))
        return dict(out={k: v[at] for k, v in inp.items()}, refs=refs.to(torch.int32))
    if case["kind"] == "mlp":
        x, y, blob = _mlp_inputs(case, seed)
        w = torch.from_numpy(blob).cuda().double()
        h, npar = abi.MLP_HID, abi.MLP_NPARAMS
        mean, std, ym, ys = w[npar:npar + 6], w[npar + 6:npar + 12], w[npar + 12], w[npar + 13]
        p = w[:npar].clone().requires_grad_(True)
        out, grad, loss, n = [], torch.zeros(npar, device="cuda", dtype=torch.float64), 0.0, case["n"]
        for i in range(0, n, 1 << 18):
            xb = (x[i:i + (1 << 18), :6].double() - mean) / std
            sizes = [h * 6, h, h * h, h, h, 1]
            w1, b1, w2, b2, w3, b3 = torch.split(p, sizes)
            h1 = torch.nn.functional.silu(xb @ w1.view(h, 6).T + b1)
            h2 = torch.nn.functional.silu(h1 @ w2.view(h, h).T + b2)
            yn = h2 @ w3 + b3
            out.append((yn * ys + ym).detach())
            part = ((yn - (y[i:i + (1 << 18)].double() - ym) / ys) ** 2).sum() / n
            grad += torch.autograd.grad(part, p)[0]
            loss += float(part.detach())
        return dict(y=torch.cat(out), loss=loss, grad=grad, trained=None, final_loss=None)
    return None


def work(case):
    if case["kind"] == "sort":  # each 60-byte record read and written once, the references written
        return {"bytes": 120.0 * case["n"] + 4.0 * (case["ngbx"] + 1), "flops": 0.0}
    if case["kind"] == "mlp":
        fwd = 2.0 * (6 * 64 + 64 * 64 + 64)  # per sample; a gradient costs three of these
        trained = case["epochs"] * max(1, case["n"] // case["batch"]) * case["batch"]
        return {"bytes": 28.0 * (case["n"] * 2 + trained) + 4.0 * case["n"], "flops": fwd * (4 * case["n"] + 3 * trained)}
    ngbx = case["nz"] * case["nx"] * case["ny"]
    n = case["mean"] if case["pop"] == "golovin" else case["mean"] * ngbx
    steps = case["steps"] * case["intervals"]
    # per step: the coupled step reads and writes the sorted 60-byte record; condensation reads radius,
    # solute and multiplicity and writes the radius; collisions read those three
    per = {"coupled": 120.0, "condensation": 32.0, "coal_breakup": 24.0, "golovin": 24.0}[case["pop"]]
    ops = {"coupled": 1700.0, "condensation": 1050.0, "coal_breakup": 150.0, "golovin": 60.0}[case["pop"]]
    observed = case["intervals"] * (48.0 * n + 32.0 * ngbx) if case["observe"] else 0.0
    return {"bytes": n * (240.0 + per * steps) + ngbx * (4 * 88.0 + 24.0 * steps) + observed, "flops": n * ops * steps}
