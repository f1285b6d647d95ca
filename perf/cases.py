"""The work that users of this framework have it do, as measurable cases.

Nine kinds of case, each through a public entry point:

  izfc       two Izhikevich layers, fully connected, run by the engine with
             the input current drawn on the device
  izfc_io    the same pair with an input and an output callback every step
  sheet      the excitatory/inhibitory Izhikevich sheet (delays, STDP,
             short-term plasticity; optionally a sparse E->E connection)
  learn      the same sheet, run and then read back: the learned weights and
             the neurons' state through the getters
  rate       a rate-encoded classifier: relay image -> fully connected and
             convergent hidden layers -> outputs
  gol        game of life on one board through the engine
  gol_steps  game-of-life steps on device buffers through the kernel C-ABI
  ensemble   batched rate networks (synaptogenesis_amd.ensemble)
  adjoint    forward and backward of the differentiable leaky network
             (synaptogenesis_amd.adjoint)

listed() gives the measured cases, draw() more of the same ranges.
"""

import ctypes
import os

import numpy as np
import torch

import synaptogenesis_amd
from synaptogenesis_amd import adjoint, syngen
from synaptogenesis_amd.ensemble import RateEnsemble

LIB_DIR = os.path.dirname(os.path.abspath(synaptogenesis_amd.__file__))


def listed():
    return [
        # The plain two-layer network at its stated size: launch latency
        # and small dependent kernels, voltages and rasters looked at now
        # and then.
        {"name": "izfc_1000", "kind": "izfc", "size": 1000, "steps": 500,
         "every": 100},
        # A closed loop: a stimulus comes in and spikes go out every step.
        {"name": "izfc_1000_io", "kind": "izfc_io", "size": 1000,
         "steps": 200},
        # A small sheet trained for a second of model time, then its
        # learned weights read back.
        {"name": "learn_32x40", "kind": "learn", "rows": 32, "cols": 40,
         "steps": 1000},
        # The full sheet: 102,400 neurons, 24 M synapse visits a step.
        {"name": "sheet_256x320", "kind": "sheet", "rows": 256, "cols": 320,
         "steps": 100, "every": 50, "density": 1.0, "learning": True},
        # The same with half of the E->E synapses dropped (SPARSE).
        {"name": "sheet_sparse_256x320", "kind": "sheet", "rows": 256,
         "cols": 320, "steps": 100, "every": 50, "density": 0.5,
         "learning": True},
        # A 28x28 image presented to a rate-encoded classifier until its
        # outputs have settled.
        {"name": "rate_784_1024_10", "kind": "rate", "side": 28,
         "hidden": 1024, "field": 5, "outputs": 10, "steps": 20},
        # The 1024 board: a long run, then the board read back.
        {"name": "gol_1024", "kind": "gol", "rows": 1024, "cols": 1024,
         "steps": 8000, "wrap": True, "rule": "life"},
        # A board of 1 GiB of words, past every cache.
        {"name": "gol_steps_16384", "kind": "gol_steps", "rows": 16384,
         "cols": 16384, "steps": 32, "wrap": True, "rule": "life"},
        # A few narrow rate networks: one launch a step is all latency.
        {"name": "ensemble_8", "kind": "ensemble", "n": 8, "low": 128,
         "high": 512, "precision": "bf16", "rectify": False, "steps": 200},
        # The full ensemble: 256 networks, 2.2 G synapses a step.
        {"name": "ensemble_256", "kind": "ensemble", "n": 256, "low": 128,
         "high": 4096, "precision": "bf16", "rectify": False, "steps": 20},
        # One training iteration of the spiking network at its stated size.
        {"name": "adjoint_spike_784_1024_10", "kind": "adjoint",
         "mode": "spike", "batch": 128, "steps": 100, "n_in": 784,
         "n_hid": 1024, "n_out": 10, "checkpoint": 10},
        # The rate mode at sizes off the 64- and 256-wide tiles.
        {"name": "adjoint_rate_784_500_10", "kind": "adjoint",
         "mode": "rate", "batch": 50, "steps": 25, "n_in": 784,
         "n_hid": 500, "n_out": 10, "checkpoint": 5},
    ]


def _log(rng, low, high):
    """A whole number in [low, high], spread over its logarithm."""
    return max(low, min(high, int(round(low * (high / low) ** rng.random()))))


def draw(rng):
    kind = rng.choice(["izfc", "izfc_io", "sheet", "learn", "rate", "gol",
                       "gol_steps", "ensemble", "adjoint", "adjoint"])
    if kind == "izfc":
        every = rng.randint(10, 100)
        return {"kind": kind, "size": _log(rng, 33, 3000),
                "steps": every * rng.randint(2, 5), "every": every}
    if kind == "izfc_io":
        return {"kind": kind, "size": _log(rng, 33, 3000),
                "steps": rng.randint(50, 200)}
    if kind == "sheet":
        # E has even sides: I is at half its resolution
        every = rng.randint(10, 50)
        return {"kind": kind, "rows": 2 * _log(rng, 9, 128),
                "cols": 2 * _log(rng, 9, 160),
                "steps": every * rng.randint(1, 2), "every": every,
                "density": rng.choice([1.0, 1.0, 0.3, 0.5, 0.8]),
                "learning": rng.random() < 0.75}
    if kind == "learn":
        return {"kind": kind, "rows": 2 * _log(rng, 9, 32),
                "cols": 2 * _log(rng, 9, 32), "steps": rng.randint(200, 1000)}
    if kind == "rate":
        return {"kind": kind, "side": rng.randint(8, 40),
                "hidden": _log(rng, 48, 4096), "field": rng.choice([3, 5, 7]),
                "outputs": rng.randint(2, 100), "steps": rng.randint(5, 20)}
    if kind == "gol":
        return {"kind": kind, "rows": _log(rng, 20, 1024),
                "cols": _log(rng, 20, 1024), "steps": rng.randint(500, 4000),
                "wrap": rng.random() < 0.7,
                "rule": rng.choice(["life", "life", "wide"])}
    if kind == "gol_steps":
        return {"kind": kind, "rows": _log(rng, 64, 16384),
                "cols": _log(rng, 64, 16384), "steps": rng.randint(8, 32),
                "wrap": rng.random() < 0.7,
                "rule": rng.choice(["life", "life", "wide"])}
    if kind == "ensemble":
        high = _log(rng, 128, 2048)
        return {"kind": kind, "n": _log(rng, 1, 64),
                "low": rng.randint(max(16, high // 16), high), "high": high,
                "precision": rng.choice(["bf16", "bf16", "bf16", "fp32"]),
                "rectify": rng.random() < 0.3, "steps": rng.randint(10, 100)}
    checkpoint = rng.choice([5, 10, 16])
    n_hid = _log(rng, 64, 1100)
    if rng.random() < 0.5:          # widths are often multiples of 64
        n_hid = (n_hid + 63) // 64 * 64
    return {"kind": kind, "mode": rng.choice(["spike", "spike", "rate"]),
            "batch": _log(rng, 8, 128),
            "steps": checkpoint * rng.randint(2, 100 // checkpoint),
            "n_in": rng.choice([784, 784, _log(rng, 40, 1000)]),
            "n_hid": n_hid, "n_out": rng.choice([10, 10, rng.randint(2, 16)]),
            "checkpoint": checkpoint}


# ---- networks run by the engine ---------------------------------------------

def _layer(name, model, rows, cols, **more):
    return {"name": name, "neural model": model, "rows": rows,
            "columns": cols, **more}


def _conn(name, source, dest, kind, **more):
    d = {"name": name, "from layer": source, "to layer": dest, "type": kind,
         "opcode": "add", "plastic": "false", "delay": 0}
    d.update(more)
    return d


_filling = None       # {connection id: (weights, delays)} of a state's build
_running = None       # the Sim whose run() is under way


def _fill_weights(ID, size, ptr):
    w = _filling[ID][0]
    assert w.size == size
    ctypes.memmove(ptr, w.ctypes.data, 4 * size)


def _fill_delays(ID, size, weights, ptr):
    d = _filling[ID][1]
    assert d.size == size
    ctypes.memmove(ptr, d.ctypes.data, 4 * size)


def _give(ID, size, ptr):
    """Input callback: the next row of the stimulus."""
    s = _running
    row = s.stimulus[s.given % len(s.stimulus)]
    s.given += 1
    ctypes.memmove(ptr, row.ctypes.data, 4 * size)


def _take(ID, size, ptr):
    """Output callback: one more row of watched value ID."""
    s = _running
    record = s.records[ID]
    ctypes.memmove(record[s.taken[ID]].ctypes.data, ptr, 4 * size)
    s.taken[ID] += 1


_library = None


def _syngen():
    global _library
    if _library is None:
        _library = syngen.load_library()
        _library.set_suppress_output(True)
        _library.set_warnings(False)
        _library.create_weight_callback("perf_weights", _fill_weights)
        _library.create_delay_weight_callback("perf_delays", _fill_delays)
        _library.create_io_callback("perf_give", _give)
        _library.create_io_callback("perf_take", _take)
    return _library


class Sim:
    """A network with its state, an environment and run arguments, moved to
    the GPU by one short run.

    weights, delays: {connection: array}; init: {(layer, key): array};
    stimulus: rows fed to layer `fed`, one a step, or one row held for the
    whole run (held); watched: [(layer, key, dtype)], recorded every `every`
    steps of a run (step 0 included)."""

    def __init__(self, layers, conns, weights, init, delays=None, fed=None,
                 stimulus=None, held=False, watched=(), every=1, steps=1,
                 learning=True):
        global _filling
        lib = _syngen()
        delays = delays or {}
        _filling = {}
        for i, c in enumerate(conns):
            if c["name"] not in weights:
                continue
            config = {"type": "flat", "weight": "0", "id": i,
                      "callback": "perf_weights"}
            if c["name"] in delays:
                config["delay callback"] = "perf_delays"
            c["weight config"] = config
            _filling[i] = (weights[c["name"]], delays.get(c["name"]))
        self.net = syngen.Network(
            {"structures": [{"name": "s", "type": "parallel",
                             "layers": layers}], "connections": conns}, lib)
        self.net.build_state()
        _filling = None
        for (name, key), values in init.items():
            self.read(name, key, np.float32, copy=False)[:] = \
                values.view(np.float32)
        modules = []
        if fed:
            # a held stimulus: the module calls back once and the value
            # stays
            modules.append({"type": "callback",
                            "rate": 1 << 30 if held else 1,
                            "layers": [{"structure": "s", "layer": fed,
                                        "input": True,
                                        "function": "perf_give", "id": 0}]})
        if watched:
            modules.append({"type": "callback", "layers": [
                {"structure": "s", "layer": name, "output": True,
                 "function": "perf_take", "id": i, "output keys": [key]}
                for i, (name, key, _) in enumerate(watched)]})
        self.env = syngen.Environment({"modules": modules}, lib)
        self.stimulus, self.given = stimulus, 0
        self.watched = list(watched)
        sizes = {l["name"]: l["rows"] * l["columns"] for l in layers}
        rows = len(range(0, steps, every))
        self.shapes = [(rows, sizes[name]) for name, _, _ in self.watched]
        self.args = {"worker threads": 0, "multithreaded": False,
                     "learning flag": learning, "verbose": False,
                     "environment rate": every}
        self.steps = steps
        self.run(2)
        self.given = 0

    def run(self, steps=None):
        global _running
        steps = steps or self.steps
        self.records = [np.empty(shape, dtype) for shape, (_, _, dtype) in
                        zip(self.shapes, self.watched)]
        self.taken = [0] * len(self.records)
        _running = self
        report = self.net.run(self.env, dict(self.args, iterations=steps))
        _running = None
        if report.get("iterations") != str(steps):
            raise RuntimeError("run failed")
        report.free()
        return {"%s %s" % (name, key): r for (name, key, _), r in
                zip(self.watched, self.records)}

    def read(self, layer, key, dtype, copy=True):
        view = self.net.get_neuron_data("s", layer, key)
        a = np.ctypeslib.as_array(
            ctypes.cast(view.data, ctypes.POINTER(ctypes.c_float)),
            shape=(view.size,)).view(dtype)
        return a.copy() if copy else a

    def __del__(self):
        if getattr(self, "env", None):
            self.env.free()
        if getattr(self, "net", None):
            self.net.free()


def _uniform(rng, n, low, high):
    return rng.random(n, dtype=np.float32) * np.float32(high - low) + \
        np.float32(low)


def _resting(layers):
    init = {}
    for l in layers:
        n = l["rows"] * l["columns"]
        init[(l["name"], "voltage")] = np.full(n, -65.0, np.float32)
        init[(l["name"], "recovery")] = np.full(
            n, np.float32(0.2) * np.float32(-65.0), np.float32)
    return init


def _izfc(case, seed):
    rng = np.random.default_rng(seed)
    n = case["size"]
    io = case["kind"] == "izfc_io"
    first = {} if io else {"init config": {"type": "normal", "mean": 5,
                                           "std dev": 2}}
    layers = [_layer("L1", "izhikevich", 1, n, params="regular", **first),
              _layer("L2", "izhikevich", 1, n, params="regular")]
    conns = [_conn("fc", "L1", "L2", "fully connected", direct=True,
                   myelinated=True)]
    weights = {"fc": _uniform(rng, n * n, 0.0, 0.5)}
    if io:
        return Sim(layers, conns, weights, _resting(layers), fed="L1",
                   stimulus=(rng.standard_normal((256, n), np.float32) *
                             np.float32(2) + np.float32(5)),
                   watched=[("L2", "output", np.int32),
                            ("L2", "voltage", np.float32)],
                   every=1, steps=case["steps"])
    return Sim(layers, conns, weights, _resting(layers),
               watched=[("L1", "output", np.int32),
                        ("L2", "output", np.int32),
                        ("L2", "voltage", np.float32)],
               every=case["every"], steps=case["steps"] + 1)


def _sheet(case, seed):
    rng = np.random.default_rng(seed)
    rows, cols = case["rows"], case["cols"]
    ne, ni = rows * cols, (rows // 2) * (cols // 2)
    noise = {"init config": {"type": "normal", "mean": 0, "std dev": 3}}
    layers = [_layer("E", "izhikevich", rows, cols, params="regular",
                     **noise),
              _layer("I", "izhikevich", rows // 2, cols // 2, params="fast",
                     **noise)]
    density = case.get("density", 1.0)
    ee = {"plastic": True, "learning rate": 0.01,
          "arborized config": {"field size": 15, "stride": 1, "wrap": True}}
    if density < 1.0:
        ee["sparse"] = True
    direct = {"direct": True, "myelinated": True}
    conns = [
        _conn("EE", "E", "E", "convergent", **ee),
        _conn("EI", "E", "I", "convergent", **direct, **{
            "arborized config": {"field size": 15, "stride": 2,
                                 "wrap": True}}),
        _conn("IE", "I", "E", "divergent", **dict(direct, opcode="sub"), **{
            "arborized config": {"field size": 9, "stride": 2,
                                 "wrap": True}})]
    weights = {"EE": _uniform(rng, ne * 225, 0.0, 0.5),
               "EI": _uniform(rng, ni * 225, 0.0, 0.5),
               "IE": _uniform(rng, ne * 81, 0.0, 0.5)}
    if density < 1.0:
        weights["EE"][rng.random(ne * 225, np.float32) >= density] = 0.0
    delays = {"EE": rng.integers(0, 32, ne * 225, np.int32)}
    if case["kind"] == "learn":
        return Sim(layers, conns, weights, _resting(layers), delays,
                   steps=case["steps"])
    # the conductances sum the plastic weights of the spiking synapses
    return Sim(layers, conns, weights, _resting(layers), delays,
               watched=[("E", "output", np.int32),
                        ("I", "output", np.int32),
                        ("E", "voltage", np.float32),
                        ("I", "voltage", np.float32),
                        ("E", "ampa", np.float32),
                        ("E", "nmda", np.float32)],
               every=case["every"], steps=case["steps"] + 1,
               learning=case["learning"])


def _rate_inputs(case, seed):
    """Image, weights by connection and the convergent layer's side."""
    rng = np.random.default_rng(seed)
    side, hidden, out = case["side"], case["hidden"], case["outputs"]
    conv = (side - case["field"]) // 2 + 1
    image = rng.random((1, side * side), np.float32)

    def normal(rows, cols):
        return (rng.standard_normal(rows * cols, np.float32) /
                np.float32(cols ** 0.5))
    return image, {"in_h": normal(hidden, side * side),
                   "in_c": normal(conv * conv, case["field"] ** 2),
                   "h_o": normal(out, hidden),
                   "c_o": normal(out, conv * conv)}, conv


def _rate(case, seed):
    image, weights, conv = _rate_inputs(case, seed)
    layers = [_layer("in", "relay", case["side"], case["side"]),
              _layer("h", "rate_encoding", 1, case["hidden"]),
              _layer("c", "rate_encoding", conv, conv),
              _layer("o", "rate_encoding", 1, case["outputs"])]
    conns = [_conn("in_h", "in", "h", "fully connected"),
             _conn("in_c", "in", "c", "convergent", **{
                 "arborized config": {"field size": case["field"],
                                      "stride": 2, "offset": 0}}),
             _conn("h_o", "h", "o", "fully connected"),
             _conn("c_o", "c", "o", "fully connected", opcode="sub")]
    return Sim(layers, conns, weights, {}, fed="in", stimulus=image,
               held=True, watched=[("h", "output", np.float32),
                                   ("c", "output", np.float32),
                                   ("o", "output", np.float32)],
               every=case["steps"], steps=case["steps"] + 1)


# survive on 2-3 and born on 3, or a wider rule
RULES = {"life": (2, 3, 3, 3), "wide": (1, 4, 3, 5)}


def _gol(case, seed):
    rng = np.random.default_rng(seed)
    rows, cols = case["rows"], case["cols"]
    smin, smax, bmin, bmax = RULES[case["rule"]]
    layers = [_layer("board", "game_of_life", rows, cols, survival_min=smin,
                     survival_max=smax, birth_min=bmin, birth_max=bmax)]
    conns = [_conn("life", "board", "board", "convergent",
                   convolutional=True, **{
                       "arborized config": {"field size": 3,
                                            "wrap": case["wrap"]},
                       "weight config": {"type": "flat", "weight": 1,
                                         "diagonal": False}})]
    words = (rng.random(rows * cols, np.float32) < 0.5).astype(
        np.uint32) << 31
    return Sim(layers, conns, {}, {("board", "output"): words},
               steps=case["steps"])


# ---- game-of-life steps on device buffers -----------------------------------

_kernels = None


def _kernel_library():
    global _kernels
    if _kernels is None:
        _kernels = ctypes.CDLL(os.path.join(LIB_DIR, "libsg_hip.so"))
        i, p = ctypes.c_int, ctypes.c_void_p
        _kernels.sg_hip_gol_steps.argtypes = [p, p, p, i, i, i, p, i, i, i,
                                              i, i, p]
        _kernels.sg_hip_gol_max_steps.argtypes = [p, i, i]
    return _kernels


class Board:
    def __init__(self, case, seed):
        lib = _kernel_library()
        self.rows, self.cols = case["rows"], case["cols"]
        self.wrap, self.rule = case["wrap"], RULES[case["rule"]]
        self.steps = case["steps"]
        gen = torch.Generator("cuda").manual_seed(seed)
        n = self.rows * self.cols
        alive = torch.rand(n, generator=gen, device="cuda") < 0.5
        self.words = alive.to(torch.int32) << 31
        self.other = torch.empty_like(self.words)
        self.sums = torch.empty(n, device="cuda")
        self.kernel = (ctypes.c_float * 9)(1, 1, 1, 1, 0, 1, 1, 1, 1)
        self.most = lib.sg_hip_gol_max_steps(self.kernel, self.rows,
                                             self.cols)

    def run(self):
        lib = _kernel_library()
        stream = torch.cuda.current_stream().cuda_stream
        left = self.steps
        while left:
            k = min(left, self.most)
            left -= k
            rc = lib.sg_hip_gol_steps(
                self.words.data_ptr(), self.other.data_ptr(),
                None if left else self.sums.data_ptr(), self.rows, self.cols,
                int(self.wrap), self.kernel, *self.rule, k, stream)
            if rc:
                raise RuntimeError("sg_hip_gol_steps: %d" % rc)
            self.words, self.other = self.other, self.words
        return {"words": self.words, "sums": self.sums}


# ---- ensembles ----------------------------------------------------------------

def _widths(case, seed):
    return np.random.default_rng(seed).integers(
        case["low"], case["high"] + 1, (case["n"], 3)).astype(np.int32)


class Ensemble:
    LEAK = 0.1

    def __init__(self, case, seed):
        self.steps = case["steps"]
        # widths are the network's, the seed gives inputs and weights
        self.e = RateEnsemble(_widths(case, 4), case["precision"],
                              leak=self.LEAK, rectify=case["rectify"],
                              seed=seed)

    def run(self):
        self.e.run(self.steps)
        n = len(self.e.widths)
        return {"h%d" % k: np.concatenate([self.e.state(i, k)
                                           for i in range(n)])
                for k in (1, 2)}

    def __del__(self):
        self.e.close()


def _philox(index, stream, seed, workload=4):
    """x0 and x1 of Philox4x32-10 with key (seed, workload) and counter
    (0, index, stream, 0), as int64."""
    low = 0xFFFFFFFF
    zero = torch.zeros_like(index)
    c = [zero, index & low, zero + stream, zero]
    k0, k1 = seed & low, workload
    for _ in range(10):
        p = []
        for m, v in ((0xD2511F53, c[0]), (0xCD9E8D57, c[2])):
            # 32 x 32 bits in two halves: the product does not fit int64
            a, b = m * (v & 0xFFFF), m * (v >> 16)
            t = (a >> 16) + b
            p.append((t >> 16, ((t & 0xFFFF) << 16) | (a & 0xFFFF)))
        c = [p[1][0] ^ c[1] ^ k0, p[1][1], p[0][0] ^ c[3] ^ k1, p[0][1]]
        k0, k1 = (k0 + 0x9E3779B9) & low, (k1 + 0xBB67AE85) & low
    return c[0], c[1]


def _ensemble_weights(case, seed, inst, layer, rows, cols):
    """W of one instance's layer as the kernels use it, in 64 bits."""
    out = torch.empty(rows * cols, dtype=torch.float64, device="cuda")
    for at in range(0, rows * cols, 1 << 24):
        index = torch.arange(at, min(rows * cols, at + (1 << 24)),
                             device="cuda")
        x0, x1 = _philox(index, 4 * inst + layer, seed)
        u1 = ((x0 >> 8).double() + 1.0) * 2.0 ** -24
        u2 = (x1 >> 8).double() * 2.0 ** -24
        z = torch.sqrt(-2.0 * torch.log(u1)) * torch.cos(
            2.0 * np.pi * u2) / cols ** 0.5
        z = z.float()
        if case["precision"] == "bf16":
            z = z.bfloat16()
        out[at:at + len(index)] = z.double()
    return out.reshape(rows, cols)


def _exact_ensemble(case, seed):
    result = {"h1": [], "h2": []}
    for i, (w0, w1, w2) in enumerate(_widths(case, 4).tolist()):
        x0 = (_philox(torch.arange(w0, device="cuda"), 4 * i, seed)[0]
              >> 8).double() * 2.0 ** -24
        W1 = _ensemble_weights(case, seed, i, 1, w1, w0)
        W2 = _ensemble_weights(case, seed, i, 2, w2, w1)

        def rate(v):
            r = torch.tanh(v)
            return torch.where(v > 0, r, 0.0) if case["rectify"] else r
        leak = Ensemble.LEAK
        drive = rate(W1 @ x0)
        h1 = torch.zeros(w1, dtype=torch.float64, device="cuda")
        h2 = torch.zeros(w2, dtype=torch.float64, device="cuda")
        for _ in range(case["steps"]):
            h1, h2 = ((1 - leak) * h1 + leak * drive,
                      (1 - leak) * h2 + leak * rate(W2 @ h1))
        result["h1"].append(h1.cpu())
        result["h2"].append(h2.cpu())
    return {k: torch.cat(v) for k, v in result.items()}


# ---- the differentiable network -----------------------------------------------

def _config(case):
    return adjoint.Config.make(
        batch=case["batch"], steps=case["steps"], n_in=case["n_in"],
        n_hid=case["n_hid"], n_out=case["n_out"],
        checkpoint=case["checkpoint"],
        mode=adjoint.SPIKE if case["mode"] == "spike" else adjoint.RATE)


class Training:
    def __init__(self, case, seed):
        self.cfg = _config(case)
        gen = torch.Generator("cuda").manual_seed(seed)

        def rand(*shape):
            return torch.rand(*shape, generator=gen, device="cuda")
        B, T, I = case["batch"], case["steps"], case["n_in"]
        pixels = rand(B, I)
        self.x = (rand(T, B, I) < pixels).to(torch.bfloat16)
        self.labels = torch.randint(0, case["n_out"], (B,), generator=gen,
                                    device="cuda", dtype=torch.int32)
        self.w = [(torch.randn(rows, cols, generator=gen, device="cuda") /
                   cols ** 0.5).requires_grad_()
                  for rows, cols in ((case["n_hid"], I),
                                     (case["n_out"], case["n_hid"]))]

    def run(self):
        loss, counts = adjoint.snn_loss(self.x, *self.w, self.labels,
                                        self.cfg)
        dw1, dw2 = torch.autograd.grad(loss, self.w)
        return {"loss": loss.detach(), "counts": counts, "dw1": dw1,
                "dw2": dw2}


def _exact_adjoint(case, seed):
    t = Training(case, seed)
    cfg = t.cfg
    spike = case["mode"] == "spike"
    slope, beta, theta, reset = cfg.slope, cfg.beta, cfg.theta, cfg.reset
    # the constants as the kernels hold them
    x = t.x.double()
    w1, w2 = (w.detach().bfloat16().double() for w in t.w)

    def unit(u):
        if spike:
            return (u >= 0).double()
        return 0.5 * (1 + slope * u / (1 + slope * u.abs()))

    def unit_grad(u):
        g = 1 / (1 + slope * u.abs()) ** 2
        return g if spike else 0.5 * slope * g
    T = case["steps"]
    v1 = s1 = torch.zeros(case["batch"], case["n_hid"], dtype=torch.float64,
                          device="cuda")
    v2 = s2 = torch.zeros(case["batch"], case["n_out"], dtype=torch.float64,
                          device="cuda")
    V1, S1, V2 = [], [], []
    counts = torch.zeros_like(v2)
    current = (x.reshape(-1, case["n_in"]) @ w1.T.contiguous()).reshape(
        T, case["batch"], -1)
    w2t = w2.T.contiguous()
    for i in range(T):
        v1 = beta * v1 - reset * theta * s1 + current[i]
        s1 = unit(v1 - theta)
        v2 = beta * v2 - reset * theta * s2 + s1 @ w2t
        s2 = unit(v2 - theta)
        counts = counts + s2
        V1.append(v1)
        S1.append(s1)
        V2.append(v2)
    logp = torch.log_softmax(counts, 1)
    labels = t.labels.long()
    loss = -logp.gather(1, labels[:, None]).mean()
    dc = logp.exp()
    dc[torch.arange(len(labels)), labels] -= 1
    dc /= case["batch"]
    dw1, dw2 = torch.zeros_like(w1), torch.zeros_like(w2)
    d1, d2 = torch.zeros_like(v1), torch.zeros_like(v2)
    for i in reversed(range(T)):
        # ds[t] = dL/ds[t]; the reset reads s[t] at t + 1
        ds2 = dc - reset * theta * d2
        d2 = beta * d2 + ds2 * unit_grad(V2[i] - theta)
        ds1 = d2 @ w2 - reset * theta * d1
        d1 = beta * d1 + ds1 * unit_grad(V1[i] - theta)
        dw2 += d2.T.contiguous() @ S1[i]
        dw1 += d1.T.contiguous() @ x[i]
    return {"loss": loss, "counts": counts, "dw1": dw1, "dw2": dw2}


# ---- the interface ----------------------------------------------------------------

def prepare(case, seed):
    kind = case["kind"]
    if kind in ("izfc", "izfc_io"):
        return _izfc(case, seed)
    if kind == "sheet":
        return _sheet(case, seed)
    if kind == "learn":
        sim = _sheet(case, seed)
        sim.reads = ([(l, k, d) for l in ("E", "I") for k, d in
                      (("output", np.int32), ("voltage", np.float32),
                       ("post trace", np.float32))],
                     ["weights", "weight derivatives", "presyn trace"])
        return sim
    if kind == "rate":
        return _rate(case, seed)
    if kind == "gol":
        sim = _gol(case, seed)
        sim.reads = ([("board", "output", np.int32)], [])
        return sim
    if kind == "gol_steps":
        return Board(case, seed)
    if kind == "ensemble":
        return Ensemble(case, seed)
    return Training(case, seed)


def run(state):
    out = state.run()
    for layer, key, dtype in getattr(state, "reads", [[]])[0]:
        out["%s %s" % (layer, key)] = state.read(layer, key, dtype)
    for key in getattr(state, "reads", [[], []])[1]:
        out["EE " + key] = state.net.get_weight_matrix(
            "EE", key).to_np_array().copy()
    return out


def work(case):
    kind, steps = case["kind"], case.get("steps")
    if kind in ("izfc", "izfc_io"):
        # the weights once and each step's neurons: 112 B read and written
        # a neuron, one addition a synapse of a spiking source (about 1 in
        # 20) and 60 operations a neuron
        n = case["size"]
        return {"bytes": 4 * n * n + steps * 2 * n * 112,
                "flops": steps * (n * n / 20 + 2 * n * 60)}
    if kind in ("sheet", "learn"):
        # a step reads and writes a plastic synapse's weight, derivative
        # and two traces and reads its delay (33 B), reads the other
        # weights, and 112 B a neuron; about 12 operations a synapse
        ne = case["rows"] * case["cols"]
        ni = ne // 4
        ee = ne * 225 * case.get("density", 1.0)
        other = ni * 225 + ne * 16
        return {"bytes": steps * (33 * ee + 4 * other + 112 * (ne + ni)),
                "flops": steps * (12 * ee + other + 60 * (ne + ni))}
    if kind == "rate":
        conv = (case["side"] - case["field"]) // 2 + 1
        weights = (case["hidden"] * case["side"] ** 2 +
                   conv ** 2 * case["field"] ** 2 +
                   case["outputs"] * (case["hidden"] + conv ** 2))
        return {"bytes": 4 * weights, "flops": 2 * weights * steps}
    if kind in ("gol", "gol_steps"):
        # each word read and written once, the sums written once, about 12
        # operations a cell and step
        n = case["rows"] * case["cols"]
        return {"bytes": 12 * n, "flops": 12 * n * steps}
    if kind == "ensemble":
        w = _widths(case, 4).astype(np.int64)
        weights = int((w[:, 0] * w[:, 1] + w[:, 1] * w[:, 2]).sum())
        size = 2 if case["precision"] == "bf16" else 4
        # weights that no cache holds are read again every step
        again = steps if weights * size > 256e6 else 1
        return {"bytes": again * weights * size + 8 * int(w.sum()),
                "flops": 2 * weights * steps}
    B, T, I = case["batch"], case["steps"], case["n_in"]
    H, O = case["n_hid"], case["n_out"]
    return {"bytes": 2 * (T * B * I) + 8 * (H * I + H * O),
            "flops": 2 * B * T * (2 * I * H + 3 * H * O)}


def _exact_rate(case, seed):
    image, weights, conv = _rate_inputs(case, seed)
    W = {k: torch.from_numpy(v).double() for k, v in weights.items()}
    side, field = case["side"], case["field"]
    x = torch.from_numpy(image[0]).double()
    W["in_h"] = W["in_h"].reshape(-1, side * side)
    W["h_o"] = W["h_o"].reshape(case["outputs"], -1)
    W["c_o"] = W["c_o"].reshape(case["outputs"], -1)
    patches = x.reshape(side, side).unfold(0, field, 2).unfold(1, field, 2)
    patches = patches.reshape(conv * conv, field * field)

    def rate(v):
        return torch.where(v > 0, torch.tanh(v), 0.0)
    h = rate(W["in_h"] @ x)
    c = rate((W["in_c"].reshape(conv * conv, -1) * patches).sum(1))
    o = rate(W["h_o"] @ h - W["c_o"] @ c)
    # recorded at the first step and at the last; a pass begins where the
    # last one ended, with every layer settled on the held image
    return {"h output": torch.stack([h, h]), "c output": torch.stack([c, c]),
            "o output": torch.stack([o, o])}


def exact(case, seed):
    """The spiking and cellular runs have no 64-bit value: their float
    state is defined by the 32-bit arithmetic that decides each spike."""
    kind = case["kind"]
    if kind == "rate":
        return _exact_rate(case, seed)
    if kind == "ensemble":
        return _exact_ensemble(case, seed)
    if kind == "adjoint":
        return _exact_adjoint(case, seed)
    return None
