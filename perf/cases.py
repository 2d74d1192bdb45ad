"""Performance cases of the engine: the work its users have it do, through the
package's public entry points (Network, Batch).

A case is one network (or one batch of networks) in its steady regime and one
pass of a program that runs it: advance it by `steps` simulated milliseconds
and read back what such a program reads (the neurons' state and the counters;
the step's spikes; the plastic synapses).  Networks are the package's own
renderings (workloads.py): grids of columns with a 3x3 stencil, connection
probabilities that give 0.9 synapses per source and column neuron on average,
0.5 mV bath events.

prepare(case, seed) builds the network (connectome and bath from the seed) and
runs it past its start-up transient, so that a pass works at the activity the
network has in a long run.  A pass continues the simulation where the last one
left it.
"""
import importlib
import math
import os
import tempfile

import numpy as np

PKG = importlib.import_module("201812realtimecortsim_amd")
W = importlib.import_module("201812realtimecortsim_amd.workloads")

FOREVER_MS = 1_000_000_000   # env_totalSimTime_ms: the caller decides when to stop
SETTLE_MS = 60               # past the gather-form start (32 ms) and the first bursts


def network(name, side, steps, exc=500, inh=250, nu_ext=3.0, stdp=False, drive="philox", files=False,
            spikes=False, synapses=False, generator="device", settle=SETTLE_MS):
    """side x side columns of 2 * exc + inh neurons; a pass is `steps` ms."""
    case = {"kind": "network", "side": side, "exc": exc, "inh": inh, "nu_ext": nu_ext, "stdp": stdp, "drive": drive,
            "files": files, "spikes": spikes, "synapses": synapses, "generator": generator, "steps": steps,
            "settle": settle}
    return dict(case, name=name) if name else case


def batch(name, count, min_side, max_side, steps, stdp_share=0.5, settle=SETTLE_MS):
    """`count` independent networks of min_side..max_side columns a side, bath
    rates of 2-6 Hz per input, a share of them plastic (the batching mix)."""
    case = {"kind": "batch", "count": count, "min_side": min_side, "max_side": max_side, "stdp_share": stdp_share,
            "steps": steps, "settle": settle}
    return dict(case, name=name) if name else case


def listed():
    return [
        # one column, one ms at a time, the state after each: a closed loop
        # (a robot, a live plot); launches and latency are all of it
        network("column 1 ms", 1, 1, generator="host"),
        # 2x2 columns, the reference's canonical small network, 10 ms between
        # looks at it
        network("2x2", 2, 10, generator="host"),
        # the same network as the reference runs it: its own random stream
        # for the bath, raster and rate files written
        network("2x2 reference run", 2, 20, drive="replay", files=True, generator="host"),
        # the same, with each ms's spikes handed to the caller
        network("2x2 spikes", 2, 1, spikes=True, generator="host"),
        # plasticity on a small network, with the synapses read back: short
        # learning runs and parameter scans
        network("2x2 small stdp", 2, 12, exc=50, inh=25, stdp=True, synapses=True, generator="host"),
        # odd column sizes: no tile of 64 neurons is whole, denser bath
        network("3x3 ragged", 3, 12, exc=203, inh=101, nu_ext=4.3, generator="host"),
        # a plastic network of the batching mix's middle size
        network("5x5 stdp", 5, 20, stdp=True),
        # 45,000 neurons: the largest class below the stencil-window form
        network("6x6", 6, 20),
        # 80,000 neurons: the smallest class in it
        network("8x8", 8, 20),
        # plasticity at scale
        network("12x12 stdp", 12, 20, stdp=True),
        # the headline network: 720,000 neurons, 810 M synapses
        network("24x24", 24, 20),
        # many networks advancing together
        batch("batch of 16", 16, 1, 4, 10),
    ]


def draw(rng):
    what = rng.random()
    if what < 0.12:
        lo = rng.randint(1, 2)
        return batch(None, rng.randint(4, 20), lo, lo + rng.randint(0, 3), rng.randint(5, 25),
                     stdp_share=rng.choice([0.0, 0.3, 0.5, 1.0]))
    side = min(14, int(math.exp(rng.uniform(0.0, math.log(15.0)))))
    if rng.random() < 0.5:
        exc, inh = 500, 250
    else:  # odd column sizes
        exc = int(math.exp(rng.uniform(math.log(40.0), math.log(540.0))))
        inh = max(8, exc // 2 + rng.randint(-3, 3))
    small = side * side * (2 * exc + inh) <= 12_000
    kind = rng.random()
    stdp = kind < 0.35
    return network(None, side, rng.randint(1, 40) if small else rng.randint(10, 25), exc=exc, inh=inh,
                   nu_ext=round(rng.uniform(2.0, 6.0), 3), stdp=stdp,
                   synapses=stdp and side * side * (2 * exc + inh) <= 1_500,
                   drive="replay" if small and kind > 0.9 else "philox",
                   files=small and kind > 0.95, spikes=small and 0.8 < kind <= 0.9,
                   generator="host" if small else "device", settle=rng.randint(50, 90))


# ---- building -------------------------------------------------------------
def _members(case, seed):
    """(network case, seed) of each member of a batch."""
    rng = np.random.default_rng([seed, 64])
    n = case["count"]
    # sides spread evenly over the range, so that a batch's work depends
    # little on the seed
    span = case["max_side"] - case["min_side"] + 1
    sides = [case["min_side"] + i * span // n for i in range(n)]
    plastic = np.zeros(n, bool)
    plastic[np.linspace(0, n - 1, round(n * case["stdp_share"])).astype(int)] = True
    return [(network(None, sides[i], 0, nu_ext=round(float(rng.uniform(2.0, 6.0)), 4), stdp=bool(plastic[i])),
             seed * 64 + i) for i in range(n)]


def _write(case, seed, d):
    npc = 2 * case["exc"] + case["inh"]
    # a learning run that reads its synapses back keeps one connectome and
    # varies the bath (the lists of two connectomes differ in length)
    cseed = 1 if case["synapses"] else 1 + seed % 29_989
    env = W.instance_env(case["side"], cseed, FOREVER_MS, case["stdp"], raster=case["files"])
    W.write_network(d, env, W.column_txt(case["nu_ext"], (case["exc"], case["exc"], case["inh"])),
                    W.connectivity_txt(case["side"], npc, 0.9 * npc), plasticity=W.STDP if case["stdp"] else None)
    return env


def _options(case, seed, env, out=None):
    return dict(drive=PKG.DRIVE_REPLAY if case["drive"] == "replay" else PKG.DRIVE_PHILOX, philox_seed=7000 + seed,
                output_dir=out, keep_spikes=case["spikes"], env=env,
                generator=PKG.GENERATOR_DEVICE if case["generator"] == "device" else PKG.GENERATOR_HOST,
                generator_seed=9000 + seed)


class _State:
    pass


def prepare(case, seed):
    s = _State()
    s.case = case
    if case["kind"] == "batch":
        with tempfile.TemporaryDirectory(prefix="dpsnn_perf_") as tmp:
            specs = []
            for i, (m, mseed) in enumerate(_members(case, seed)):
                d = os.path.join(tmp, f"n{i:02d}")
                env = _write(m, mseed, d)
                specs.append((d, dict(_options(m, mseed, env), drop_host_synapses=True)))
            s.nets = PKG.Network.build_many(specs, host_threads=2)
        s.batch = PKG.Batch()
        for n in s.nets:
            s.batch.add(n)
        s.batch.step(case["settle"])
        s.batch.sync()
        return s
    s.out = tempfile.TemporaryDirectory(prefix="dpsnn_perf_out_") if case["files"] else None
    with tempfile.TemporaryDirectory(prefix="dpsnn_perf_") as tmp:
        env = _write(case, seed, tmp)
        # a network too large to be dumped to text keeps no host copy of its synapses
        drop = case["side"] * case["side"] * (2 * case["exc"] + case["inh"]) > 20_000
        s.net = PKG.Network(tmp, drop_host_synapses=drop, **_options(case, seed, env, s.out.name if s.out else None))
    s.net.step(case["settle"])
    s.net.sync()
    return s


# ---- one pass -------------------------------------------------------------
def _look(net):
    """The neurons' state and the counters of what was delivered so far."""
    st = net.stats()
    return dict(net.state(), **{k: int(st[k]) for k in ("steps", "spikes", "synaptic_events", "external_events")})


def run(s):
    case = s.case
    if case["kind"] == "batch":
        s.batch.step(case["steps"])
        states = [net.state() for net in s.nets]
        return {k: np.concatenate([st[k] for st in states]) for k in states[0]}
    net = s.net
    net.step(case["steps"])
    if case["files"]:
        net.sync()
    out = _look(net)
    if case["spikes"]:
        ids, te = net.last_spikes()
        # the spike list's length differs from ms to ms: as arrays over the neurons
        out["spike_ms"] = np.full(net.n, -1.0)
        out["spike_ms"][ids] = te
    if case["synapses"]:
        syn = net.synapses()
        out.update({k: syn[k] for k in ("weight", "tderiv", "last")})
    return out


# ---- what a pass cannot do without ----------------------------------------
RATE = 0.41  # spikes per neuron and ms in the steady regime (about 410 Hz)


def _size(case):
    """(neurons, synapses) of a network case."""
    side, npc = case["side"], 2 * case["exc"] + case["inh"]
    p = [[float(v) for v in line.split()[6:]] for line in
         W.connectivity_txt(side, npc, 0.9 * npc).splitlines()][0]
    syn = 0.0
    for dx in (-1, 0, 1):
        for dy in (-1, 0, 1):
            cells = max(0, side - abs(dx)) * max(0, side - abs(dy))
            syn += cells * npc * npc * p[abs(dx) + 2 * abs(dy)]
    return side * side * npc, syn


def _work(case, steps):
    n, syn = _size(case)
    events = RATE * syn * steps
    # each delivered synapse's word (source and weight) once per ms it is
    # delivered; per ms and neuron its state (v, c, Tr, Te, bath time and
    # counter) read and written and its spike recorded; the state read back
    b = 4.0 * events + n * (steps * (2 * 48.0 + 8.0) + 33.0)
    if case["stdp"]:  # each synapse's derivative and last activation, once a pass
        b += syn * 2 * 8.0
    if case["synapses"]:
        b += syn * 10.0
    # the two exponential decays, the membrane's two half steps and the threshold
    return b, 35.0 * events


def work(case):
    if case["kind"] == "batch":
        parts = [_work(m, case["steps"]) for m, _ in _members(case, 0)]
    else:
        parts = [_work(case, case["steps"])]
    return {"bytes": sum(p[0] for p in parts), "flops": sum(p[1] for p in parts)}


# ---- the same pass in plain numpy, 64 bits --------------------------------
def exact(case, seed):
    """What run(prepare(case, seed)) returns, simulated with numpy from the
    prepared network's synapses and checkpoint; None for the cases that
    would take too long (and for the replayed bath, whose stream is the
    host's), and for passes so long that the rounding of the bath's
    logarithm grows to spikes of its own (the dynamics are chaotic)."""
    if case["kind"] == "batch" or case["drive"] == "replay" or case["steps"] > 12:
        return None
    n, syn = _size(case)
    if n > 5_000 or syn * RATE * case["steps"] > 5e7:
        return None
    s = prepare(case, seed)
    sim = _Simulation(case, s.net, 7000 + seed)
    for _ in range(case["steps"]):
        sim.step()
    out = {"v": sim.v, "c": sim.c, "Tr": sim.Tr, "Te": sim.Te, "fired": None, "steps": None, "spikes": None,
           "synaptic_events": None, "external_events": None}
    if case["spikes"]:
        # the spikes of the last step's scan: those of the dynamics before it
        out["spike_ms"] = np.where(sim.fired_before, sim.te_before, -1.0)
    if case["synapses"]:
        out.update(weight=None, tderiv=sim.td, last=None)
    return out


def _read_checkpoint(net):
    """The arrays of dpsnn_checkpoint's file that a simulation needs."""
    with tempfile.TemporaryDirectory(prefix="dpsnn_perf_") as tmp:
        path = os.path.join(tmp, "state")
        net.checkpoint(path)
        raw = open(path, "rb").read()
    head = np.frombuffer(raw, np.uint32, 12, 8)
    n, rs, nw, stdp, t = (int(head[i]) for i in (0, 1, 2, 4, 5))
    at = 8 + 12 * 4 + 16
    d = {"t": t, "rs": rs}

    def take(name, dtype, count):
        nonlocal at
        d[name] = np.frombuffer(raw, dtype, count, at).copy()
        at += d[name].nbytes

    for name in ("v", "c", "Tr", "Te", "bath"):
        take(name, np.float64, n)
    take("counter", np.uint64, n)
    take("bits", np.uint64, rs * nw)
    take("hist", np.float64, rs * n)
    take("counters", np.uint64, 256)
    if stdp:
        take("last_spike", np.int32, n)
    d["hist"] = d["hist"].reshape(rs, n)
    return d


class _Simulation:
    def __init__(self, case, net, philox_seed):
        ck = _read_checkpoint(net)
        syn = net.synapses()
        self.t, self.rs, self.hist = ck["t"], ck["rs"], ck["hist"]
        self.v, self.c, self.Tr, self.Te, self.a, self.ctr = (ck[k] for k in ("v", "c", "Tr", "Te", "bath", "counter"))
        n = self.n = len(self.v)
        inh = np.arange(n) % (2 * case["exc"] + case["inh"]) >= 2 * case["exc"]
        self.tau = np.where(inh, 10.0, 20.0)
        self.alpha = np.where(inh, 0.0, 1.0)
        self.gc = np.where(inh, 0.0, float(np.float32(0.05)))
        self.theta, self.h, self.tarp, self.tauc = 20.0, 15.0, 2.0, 500.0
        self.bath_mean = 1000.0 / float(np.float32(case["nu_ext"]) * np.float32(800.0))
        self.key = ((philox_seed >> 32) ^ np.arange(n, dtype=np.uint64)) & np.uint64(0xFFFFFFFF)
        self.key0 = np.uint64(philox_seed & 0xFFFFFFFF)
        w2f = np.float32(-6.0) / np.float32(-32767.0)
        self.pre, self.post, self.delay = (syn[k].astype(np.int64) for k in ("pre", "post", "delay"))
        self.val = (syn["weight"].astype(np.float32) * w2f).astype(np.float64)
        self.buckets = [np.flatnonzero(self.delay == d) for d in range(int(self.delay.max()) + 1)]
        self.stdp = case["stdp"]
        if self.stdp:
            self.td, self.last = syn["tderiv"].astype(np.float64), syn["last"].astype(np.int64)
            self.last_spike = ck["last_spike"].astype(np.int64)
            self.causal = 0.1 * 1.2 * 0.95 ** np.arange(128)
            self.anti = -0.12 * 1.2 * 0.95 ** np.arange(128)

    def _bath(self, who):
        """One Philox4x32-10 block of each neuron of `who`: its second
        uniform in [0, 1) is the event's lapse."""
        m32, one = np.uint64(0xFFFFFFFF), np.uint64(32)
        x = [self.ctr[who] & m32, self.ctr[who] >> one, np.zeros(len(who), np.uint64),
             np.full(len(who), 0x44505300, np.uint64)]
        k0, k1 = np.full(len(who), self.key0), self.key[who]
        for _ in range(10):
            p0, p1 = np.uint64(0xD2511F53) * x[0], np.uint64(0xCD9E8D57) * x[2]
            x = [(p1 >> one) ^ x[1] ^ k0, p1 & m32, (p0 >> one) ^ x[3] ^ k1, p0 & m32]
            k0, k1 = (k0 + np.uint64(0x9E3779B9)) & m32, (k1 + np.uint64(0xBB67AE85)) & m32
        self.ctr[who] += np.uint64(1)
        return (((x[2] << np.uint64(21)) ^ x[3]) & np.uint64((1 << 53) - 1)).astype(np.float64) * 2.0 ** -53

    def step(self):
        t, n = self.t, self.n
        # internal events, each target's in delivery order: delay descending, source ascending
        who, when, val = [], [], []
        for d in range(len(self.buckets) - 1, -1, -1):
            te = self.hist[(t - d) % self.rs]
            b = self.buckets[d]
            b = b[te[self.pre[b]] >= 0.0]
            k = te[self.pre[b]]
            who.append(self.post[b])
            when.append(t + (k - np.trunc(k)))
            val.append(self.val[b])
            if self.stdp:
                dt = t - self.last_spike[self.post[b]]
                self.last[b] = t
                self.td[b] += np.where(dt < 128, self.anti[np.minimum(dt, 127)], 0.0)
        # bath events, after the internal ones of the same time
        while True:
            due = np.flatnonzero(self.a < t + 1.0)
            if not len(due):
                break
            who.append(due)
            when.append(self.a[due])
            val.append(np.full(len(due), 0.5))
            u = (1.0 - self._bath(due)).astype(np.float32).astype(np.float64)
            self.a[due] += -np.log(u).astype(np.float32).astype(np.float64) * self.bath_mean
        who, when, val = np.concatenate(who), np.concatenate(when), np.concatenate(val)
        order = np.lexsort((when, who))  # stable
        when, val = when[order], val[order]
        count = np.bincount(who, minlength=n)
        first = np.concatenate(([0], np.cumsum(count)[:-1]))
        fired = np.zeros(n, bool)
        by_count = np.argsort(-count, kind="stable")
        sorted_count = count[by_count]
        for r in range(int(count.max())):
            j = by_count[:np.searchsorted(-sorted_count, -r, side="left")]  # neurons with more than r events
            fired[j] |= self._event(j, when[first[j] + r], val[first[j] + r])
        # the scan of the next ms
        self.fired_before, self.te_before = (self.hist[t % self.rs] >= 0.0), self.hist[t % self.rs].copy()
        self.hist[(t + 1) % self.rs] = np.where(fired, self.Te, -1.0)
        if self.stdp:
            hit = fired[self.post] & (self.last != 0)
            dt = t - self.last
            self.td += np.where(hit & (dt < 128), self.causal[np.clip(dt, 0, 127)], 0.0)
            self.last_spike[fired] = t + 1
        self.t += 1

    def _event(self, j, t, val):
        v, c, Te, tau = self.v[j], self.c[j], self.Te[j], self.tau[j]
        dt, since = t - self.Tr[j], t - Te
        active = since > self.tarp
        leaving = active & (self.Tr[j] - Te < self.tarp)
        c = np.where(leaving, c * np.exp(-(dt - since + self.tarp) / self.tauc), c)
        dt = np.where(leaving, since - self.tarp, dt)
        half = dt / 2
        for _ in range(2):
            v = np.where(active, v - v * (half / tau) - self.gc[j] * c * half, v)
        v = np.where(active, v + val, v)
        rc = dt / self.tauc
        c = c * (1 - rc + rc * rc / 2)
        fire = active & (v >= self.theta)
        self.v[j] = np.where(fire, self.h, v)
        self.c[j] = np.where(fire, c + self.alpha[j], c)
        self.Te[j] = np.where(fire, t, Te)
        self.Tr[j] = t
        return fire
