"""What the speed of this framework is measured on: twelve listed cases, and more drawn from the same ranges.

Each case is one call, or one check interval, of a program that uses the framework through its public entry points:

  interval  gasp_sweep_grids on device int32 grids that the caller owns
  swarm     one check interval of an Engine: sweeps with the threshold check, then the counts, the magnetisations and
            the grids (as a gridstates.bin record body, and as int8 snapshots where the case asks for some)
  shoot     committor shooting: input grids, frozen decided replicas, intervals until all are decided or the last one,
            then the bootstrap error bars on the GPU
  driver    a whole mc_driver_gpu run with the largest cluster as its collective variable
  predict, gradient, epoch   the committor surrogate: inference, one gradient, one training epoch

Spins are whole numbers that every build computes alike; a magnetisation is such a sum over L^2.
"""
import math

import numpy as np
import torch

import gpu_2dising_amd as G

BETA, H = 0.54, 0.07  # the reference's metastable point
DN, UP = -0.9, 0.9    # its default thresholds


def listed():
    return [
        # the smallest call: one sweep of one 64-replica group, all launches and latency
        dict(name="interval_L32_R64", kind="interval", method=2, L=32, R=64, sweeps=1),
        # a large lattice beyond the whole-word LDS path, few replicas (the batched workload's largest group)
        dict(name="interval_L256_R256", kind="interval", method=0, L=256, R=256, sweeps=20),
        # the multispin throughput workload: 16384 replicas of 64 x 64, checked every 100 sweeps
        dict(name="swarm_L64_R16384", kind="swarm", method=2, L=64, R=16384, sweeps=100, check=1, rng="philox", snaps=0),
        # ragged: a lattice side and a replica count that fill neither words nor workgroups, fates as in itask 1
        dict(name="swarm_L75_R3001", kind="swarm", method=2, L=75, R=3001, sweeps=20, check=2, rng="philox", snaps=0),
        # gpu_method 1, with the grid history's int8 snapshots
        dict(name="swarm_bits_L100_R2000", kind="swarm", method=1, L=100, R=2000, sweeps=20, check=1, rng="philox", snaps=64),
        # the bit-sliced engine on the throughput workload
        dict(name="swarm_sliced_L64_R16384", kind="swarm", method=3, L=64, R=16384, sweeps=100, check=1, rng="philox", snaps=0),
        # the plain reference run on the reference's own MT19937 streams: 256 replicas, a check every 100 sweeps
        dict(name="swarm_mt_L32_R256", kind="swarm", method=2, L=32, R=256, sweeps=100, check=1, rng="mt19937", snaps=0),
        # committor shooting from droplets, decided replicas frozen
        dict(name="shoot_L64_32x256", kind="shoot", L=64, inputs=32, shots=256, sweeps=100, intervals=10),
        # a whole driver run with the largest cluster as the collective variable and grid output
        dict(name="driver_cluster_L64_R1024", kind="driver", method=2, L=64, inputs=16, shots=64, total=200, mag=20, grid=100),
        # surrogate inference on a batch of 4096 grids
        dict(name="predict_L64_n4096", kind="predict", L=64, n=4096, batch=4096),
        # a small ragged gradient, where the launches count
        dict(name="gradient_L32_n37", kind="gradient", L=32, n=37),
        # a training epoch over resident data in batches of 256, the last one smaller
        dict(name="epoch_L64_n2000", kind="epoch", L=64, n=2000, batch=256),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["interval", "swarm", "swarm", "swarm", "shoot", "driver", "predict", "gradient", "epoch"])
    if kind in ("interval", "swarm"):
        method = rng.choice([0, 1, 2, 2, 2, 3])
        L = {0: _log(rng, 100, 400), 1: _log(rng, 12, 128), 2: _log(rng, 12, 140), 3: _log(rng, 12, 96)}[method]
        R = _log(rng, 16, 600) if method == 0 else _log(rng, 50, 12000)
        # up to 2e9 attempts, and up to 500000 of one replica (they follow one another)
        most = min(100, 2_000_000_000 // (R * L * L), max(1, 500_000 // (L * L)))
        case = dict(kind=kind, method=method, L=L, R=R, sweeps=_log(rng, 1, max(1, most)))
        if kind == "swarm":
            mt = method != 3 and R * L * L < 4_000_000 and rng.random() < 0.3
            case.update(check=rng.randrange(3), rng="mt19937" if mt else "philox", snaps=rng.choice([0, 0, 17]))
        return case
    if kind == "shoot":
        return dict(kind=kind, L=_log(rng, 24, 72), inputs=rng.randrange(3, 40), shots=_log(rng, 16, 256),
                    sweeps=rng.choice([20, 50, 100]), intervals=rng.randrange(2, 9))
    if kind == "driver":
        return dict(kind=kind, method=rng.choice([1, 2]), L=_log(rng, 20, 72), inputs=rng.randrange(1, 20),
                    shots=_log(rng, 10, 60), total=rng.choice([60, 100, 200]), mag=rng.choice([10, 20]), grid=50)
    L = rng.choice([16, 32, 64, 128])
    n = _log(rng, 2, 2_000_000 // (L * L))
    if kind == "predict":
        return dict(kind=kind, L=L, n=n, batch=max(1, n // rng.choice([1, 1, 3])))
    if kind == "gradient":
        return dict(kind=kind, L=L, n=n)
    return dict(kind=kind, L=L, n=max(n, 8), batch=max(4, n // rng.choice([1, 2, 5])))


# ------------------------------------------------------------------ inputs
class Held:
    """A case's inputs and handles; the engine, network and streams go with it."""

    def __init__(self, **kw):
        self.__dict__.update(kw)

    def __del__(self):
        for name in ("engine", "net"):
            if name in self.__dict__:
                self.__dict__[name].close()
        if "rng" in self.__dict__:
            self.rng.free()


def _swarm_grids(L, R, seed):
    """int32 [R, L, L] on the GPU: a swarm half way through its nucleation, each replica in the metastable -1 phase
    (a few spins up) or already in the +1 phase."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    phase = torch.rand(R, 1, 1, device="cuda", generator=g) < 0.5
    odd = torch.rand(R, L, L, device="cuda", generator=g) < 0.03
    return torch.where(phase ^ odd, 1, -1).to(torch.int32).contiguous()


def _droplets(L, n, seed):
    """int32 [n, L, L] on the host: a -1 sea with a +1 droplet (radius up to 0.22 L) at a random centre and 5% of the
    spins flipped, as committor shooting starts from."""
    rs = np.random.default_rng(seed)
    x = np.arange(L)
    c = rs.integers(0, L, (n, 2))
    d = np.abs(x[None, :] - c[:, :1])
    e = np.abs(x[None, :] - c[:, 1:])
    d, e = np.minimum(d, L - d), np.minimum(e, L - e)
    rad = rs.uniform(0.06 * L, 0.22 * L, n)[:, None, None]
    g = np.where(d[:, :, None] ** 2 + e[:, None, :] ** 2 <= rad ** 2, 1, -1)
    return np.where(rs.random(g.shape) < 0.05, -g, g).astype(np.int32)


SHAPES = [(9, 32), (32,)] + [(9, 32, 32), (32,)] * 3 + [(32, 64), (64,), (64,), (1,)]


def _net_inputs(case, seed):
    """Parameters as a network under training has them, int8 grids and labels."""
    rs = np.random.default_rng(seed)
    fan = [9, 0] + [288, 0] * 3 + [32, 0, 64, 0]
    p = [rs.normal(0, math.sqrt(2 / f), s) if f else rs.normal(0, 0.05, s) for s, f in zip(SHAPES, fan)]
    params = np.concatenate([x.ravel() for x in p]).astype(np.float32)
    spins = _droplets(case["L"], case["n"], seed + 1).astype(np.int8)
    m = spins.reshape(case["n"], -1).mean(1)
    labels = np.clip(1 / (1 + np.exp(-20 * (m + 0.75))) + rs.normal(0, 0.02, case["n"]), 0, 1).astype(np.float32)
    return params, spins, labels, rs.permutation(case["n"]).astype(np.int32)


def prepare(case, seed):
    kind, L = case["kind"], case["L"]
    if kind == "interval":
        return Held(case=case, grids=_swarm_grids(L, case["R"], seed), rng=G.RngState(case["R"], seed + 1),
                    mag=torch.empty(case["R"], device="cuda"))
    if kind == "swarm":
        rng = G.RngState(case["R"], seed + 1, mt=case["rng"] == "mt19937")
        engine = G.Engine(L, case["R"], case["method"], rng, BETA, H)
        grids = _swarm_grids(L, case["R"], seed)
        torch.cuda.synchronize()
        G.check(G.lib().gasp_engine_set_grids(engine.ptr, grids.data_ptr(), 1))
        snaps = np.random.default_rng(seed).integers(0, case["R"], case["snaps"]).astype(np.int32)
        return Held(case=case, rng=rng, engine=engine, snaps=snaps)
    if kind == "shoot":
        R = case["inputs"] * case["shots"]
        rng = G.RngState(R, seed + 1)
        engine = G.Engine(L, R, 2, rng, BETA, H)
        engine.set_freeze(True)
        return Held(case=case, rng=rng, engine=engine, inputs=_droplets(L, case["inputs"], seed),
                    open=np.full(R, -1, np.int32))
    if kind == "driver":
        R = case["inputs"] * case["shots"]
        grids = np.repeat(_droplets(L, case["inputs"], seed), case["shots"], axis=0)
        return Held(case=case, rng=G.RngState(R, seed + 1), grids=grids)
    params, spins, labels, order = _net_inputs(case, seed)
    net = G.Surrogate(L, case.get("batch", case["n"]))
    net.set_params(params)
    if kind == "epoch":
        net.set_data(spins, labels)
    return Held(case=case, net=net, spins=spins, labels=labels, order=order)


# ------------------------------------------------------------------ one pass
def run(s):
    case = s.case
    kind, L = case["kind"], case["L"]
    if kind == "interval":
        G.check(G.lib().gasp_sweep_grids(L, case["R"], case["method"], s.rng.ptr, BETA, H, s.grids.data_ptr(),
                                         case["sweeps"], s.mag.data_ptr(), torch.cuda.current_stream().cuda_stream))
        return {"grids": s.grids, "mag": s.mag}
    if kind == "swarm":
        e = s.engine
        e.sweep(case["sweeps"], case["check"], DN, UP)
        out = {"mag": e.magnetisation(), "grids": e.gridstates()}
        if case["check"]:
            out["counts"] = e.counts()[:1] if case["check"] == 1 else e.counts()[1:]
        if case["check"] == 2:
            out["fates"] = e.fates()
        if case["snaps"]:
            out["snaps"] = e.gather(s.snaps)
        return out
    if kind == "shoot":
        e = s.engine
        e.set_inputs(s.inputs)
        e.set_fates(s.open)
        for _ in range(case["intervals"]):
            e.sweep(case["sweeps"], G.CHECK_FATES, DN, UP)
            if e.counts()[1:].sum() == e.R:
                break
        fates = e.fates()
        return {"fates": fates, "mag": e.magnetisation(),
                "errbar": G.bootstrap_gpu(fates.reshape(case["inputs"], -1), 256)}
    if kind == "driver":
        r = G.run_driver(L, s.grids, beta=BETA, h=H, rng=s.rng, method=case["method"], tot_nsweeps=case["total"],
                         mag_output_int=case["mag"], grid_output_int=case["grid"], itask=1, dn_thr=0.005 * L * L,
                         up_thr=0.6 * L * L, ninputs=case["inputs"], cv="largest_cluster", outfunc=lambda *a: 0)
        return {k: r[k] for k in ("result", "fates", "host_grids", "final_grids")}
    if kind == "predict":
        return s.net.predict(s.spins)
    if kind == "gradient":
        loss, grad = s.net.gradient(s.spins, s.labels)
        return {"loss": loss, "grad": grad}
    loss = s.net.train_epoch(s.order, case["batch"], 1e-3)
    return {"loss": loss, "params": s.net.params()}


# ------------------------------------------------------------------ work
def work(case):
    kind, N = case["kind"], case["L"] ** 2
    if kind in ("interval", "swarm"):
        R, attempts = case["R"], case["R"] * N * case["sweeps"]
        # integer operations of an attempt: its share of the random numbers (half a Philox4x32-10 block, 10 products
        # and 20 xors; three MT19937 words), the site, its neighbours, the sum, the comparison
        ops = attempts * (60 if case.get("rng") == "mt19937" else 44)
        if case["method"] == 3:
            # per word of 64 replicas: the site's block, about 7 bit planes of random numbers, adders and comparisons
            ops = attempts / 64 * (60 + 4 * 60 + 2 * (20 + 7 * 10))
        data = R * N * (8 if kind == "interval" else 2 / 8) + R * 4 + case.get("snaps", 0) * N
        return {"bytes": data, "flops": ops}
    if kind in ("shoot", "driver"):
        R = case["inputs"] * case["shots"]
        sweeps = case["sweeps"] * case["intervals"] if kind == "shoot" else case["total"]
        data = R * N / 8 + R * 12 if kind == "shoot" else 3 * 4 * R * N
        # at least half of the replicas of a shooting run are undecided on average
        return {"bytes": data, "flops": 44 * R * N * sweeps * (0.5 if kind == "shoot" else 1)}
    n = case["n"]
    flops = n * N * (2 * 9 * 32 + 3 * 2 * 9 * 32 * 32)
    if kind == "predict":
        return {"bytes": n * (N + 4) + 4 * 30241, "flops": flops}
    # backward: the weight gradients, and the data gradients of all but the first layer
    return {"bytes": n * (N + 4) + 8 * 30241, "flops": 3 * flops - n * N * 2 * 9 * 32}


# ------------------------------------------------------------------ the same in 64 bits
def _net_loss(params, spins, labels):
    """Predictions and mean loss in float64 by plain torch; a convolution is a sum of nine shifted products."""
    p, at = [], 0
    for s in SHAPES:
        n = math.prod(s)
        p.append(params[at:at + n].reshape(s))
        at += n
    a = spins.double().unsqueeze(-1)
    for k in range(4):
        w, b = p[2 * k], p[2 * k + 1]
        z = b
        for t in range(9):
            z = z + torch.roll(a, (1 - t // 3, 1 - t % 3), (1, 2)) @ w[t].reshape(a.shape[-1], 32)
        a = torch.relu(z)
    z = torch.relu(a.mean((1, 2)) @ p[8] + p[9]) @ p[10] + p[11]
    loss = None if labels is None else torch.nn.functional.binary_cross_entropy_with_logits(z, labels.double())
    return torch.sigmoid(z), loss


def _net_gradient(params, spins, labels):
    """Mean loss and its gradient, in pieces that bound the memory."""
    q = params.clone().requires_grad_()
    step, total = max(1, 262144 // spins[0].numel()), 0.0
    for i in range(0, len(spins), step):
        loss = _net_loss(q, spins[i:i + step], labels[i:i + step])[1] * (len(spins[i:i + step]) / len(spins))
        loss.backward()
        total += float(loss)
    return total, q.grad


def exact(case, seed):
    if case["kind"] not in ("predict", "gradient", "epoch"):
        return None  # spins, their sums and counts: whole numbers of a chain that only its sequential walk gives
    params, spins, labels, order = _net_inputs(case, seed)
    p = torch.from_numpy(params).cuda().double()
    x, y = torch.from_numpy(spins).cuda(), torch.from_numpy(labels).cuda()
    if case["kind"] == "predict":
        with torch.no_grad():
            step = max(1, 262144 // x[0].numel())
            return torch.cat([_net_loss(p, x[i:i + step], None)[0] for i in range(0, len(x), step)])
    if case["kind"] == "gradient":
        loss, grad = _net_gradient(p, x, y)
        return {"loss": loss, "grad": grad}
    m, v, losses = torch.zeros_like(p), torch.zeros_like(p), 0.0
    for k, i in enumerate(range(0, len(order), case["batch"]), 1):
        j = torch.from_numpy(order[i:i + case["batch"]]).long().cuda()
        loss, g = _net_gradient(p, x[j], y[j])
        losses += loss * len(j)
        m, v = 0.9 * m + 0.1 * g, 0.999 * v + 0.001 * g * g
        p = p - 1e-3 * (m / (1 - 0.9 ** k)) / (torch.sqrt(v / (1 - 0.999 ** k)) + 1e-8)
    return {"loss": losses / len(order), "params": p}
