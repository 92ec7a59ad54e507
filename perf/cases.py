"""The calls this framework is used for, from one amplitude of a small circuit to a
49-qubit batch, each through the package's public entry points.

Every case is a dict of plain values; `kind` says which call it is:

* amplitudes  -- `Executor.amplitudes` on a saved plan (`qxtools.jl_amd/workloads`),
  all slices of the plan or the range that one worker of a sharded run takes;
* sample      -- `Executor.sample_rejection` on a saved plan (device-side sampling);
* gradient    -- `ParamCircuit.loss_and_grad` of a parameterised grid circuit;
* variational -- one iteration of a variational loop: new angles, loss and gradient;
* simulate    -- `run_simulation` of a circuit, planning and lowering included.

The saved plans' circuits are fixed, as a program that serves one circuit has them; a
seed draws the bitstrings, the angles, the sampling stream or the circuit's gates."""

import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "qxtools.jl_amd")
if PKG not in sys.path:
    sys.path.insert(0, PKG)

from qxhip import workloads  # noqa: E402
from qxhip.circuits import create_param_rqc_circuit, create_rqc_circuit  # noqa: E402
from qxhip.gradients import ParamCircuit  # noqa: E402
from qxhip.simulation import Executor, run_simulation  # noqa: E402

PLANS = {"3x3": "rqc_3x3_d16", "5x5": "rqc_5x5_d20", "6x6": "rqc_6x6_d12_s6", "7x7": "rqc_7x7_d12_s10_open5"}


def _amplitudes(name, plan, bitstrings, precision="c128", graph=True, autotune=False, slices=0, first_slice=0):
    """`slices` 0: every slice of the plan, else the range that starts at first_slice."""
    return dict(name=name, kind="amplitudes", plan=plan, bitstrings=bitstrings, precision=precision, graph=graph,
                autotune=autotune, slices=slices, first_slice=first_slice)


def _gradient(name, kind, rows, cols, depth, bitstrings, sliced=0, precision="c128"):
    return dict(name=name, kind=kind, rows=rows, cols=cols, depth=depth, bitstrings=bitstrings, sliced=sliced,
                precision=precision)


def listed():
    return [
        # a service that answers one amplitude of a small circuit at a time: latency
        _amplitudes("one_3x3", "3x3", 1),
        # a short list of outputs of the same circuit (the plain method, small)
        _amplitudes("list64_3x3", "3x3", 64),
        # sampling a small device: rounds of candidates and the acceptance test
        dict(name="sample_3x3", kind="sample", plan="3x3", num_samples=100),
        # a whole simulation as a first-time user calls it: plan, lower, every amplitude
        dict(name="simulate_3x3", kind="simulate", rows=3, cols=3, depth=8),
        # the headline: 25 qubits at depth 20, 256 outputs, the kernels tuned beforehand
        _amplitudes("list256_5x5", "5x5", 256, autotune=True),
        # the same circuit in complex64, an odd number of outputs, launched eagerly
        _amplitudes("list100_5x5_c64", "5x5", 100, precision="c64_4m", graph=False),
        # 36 qubits with cut bonds, complex64: more outputs than one batch holds
        _amplitudes("list512_6x6_c64", "6x6", 512, precision="c64_4m"),
        # one worker's share of a sharded run: 8 of the 64 slices, looped, odd batch
        _amplitudes("share_6x6", "6x6", 37, slices=8, first_slice=16),
        # 49 qubits with five open outputs: 1024 amplitudes in double precision
        _amplitudes("open32_7x7", "7x7", 32),
        # the same in the split bf16 product, the fastest precision offered
        _amplitudes("open32_7x7_split", "7x7", 32, precision="c64_bf16x3"),
        # loss and gradient of a 36-qubit parameterised circuit with cut bonds
        _gradient("gradient_6x6", "gradient", 6, 6, 6, 64, sliced=4),
        # one iteration of a variational loop on a small circuit
        _gradient("variational_3x4", "variational", 3, 4, 5, 21),
    ]


def draw(rng):
    """One more case of the same ranges; plans, precisions and counts as listed."""
    log = lambda lo, hi: int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))  # noqa: E731
    kind = rng.choice(["small", "medium", "medium", "sliced", "sliced", "share", "open", "sample", "simulate",
                       "gradient", "variational"])
    graph = rng.random() < 0.7
    if kind == "small":
        c = _amplitudes("", "3x3", log(1, 512), rng.choice(["c128", "c64_4m"]), graph)
    elif kind == "medium":
        c = _amplitudes("", "5x5", log(1, 512), rng.choice(["c128", "c128", "c64_4m", "c64_3m"]), graph,
                        rng.random() < 0.3)
    elif kind == "sliced":
        c = _amplitudes("", "6x6", log(1, 512), rng.choice(["c128", "c64_4m", "c64_3m"]), graph)
    elif kind == "share":
        n = rng.choice([1, 2, 3, 5, 8, 12])
        c = _amplitudes("", "6x6", log(4, 128), rng.choice(["c128", "c64_4m"]), graph, False, n, rng.randrange(64 - n))
    elif kind == "open":
        c = _amplitudes("", "7x7", log(1, 32), rng.choice(["c128", "c64_4m", "c64_bf16x3"]), graph)
    elif kind == "sample":
        c = dict(kind="sample", plan="3x3", num_samples=log(10, 400))
    elif kind == "simulate":
        rows, cols = rng.choice([(2, 3), (2, 4), (3, 3), (2, 5)])
        c = dict(kind="simulate", rows=rows, cols=cols, depth=rng.randint(4, 12))
    elif kind == "gradient":
        rows, cols = rng.choice([(4, 4), (4, 5), (5, 5), (5, 6)])
        c = _gradient("", "gradient", rows, cols, rng.randint(4, 6), log(8, 64), rng.choice([0, 2, 4]),
                      rng.choice(["c128", "c128", "c64_4m"]))
    else:
        rows, cols = rng.choice([(2, 3), (3, 3), (3, 4), (4, 4)])
        c = _gradient("", "variational", rows, cols, rng.randint(3, 6), log(4, 64))
    c.pop("name", None)
    return c


# ---------------------------------------------------------------------- inputs
def _bitstrings(num, qubits, seed):
    draws = np.random.Generator(np.random.PCG64(seed)).integers(0, 2, size=(num, qubits))
    return ["".join("01"[b] for b in row) for row in draws]


def _angles(count, seed):
    return np.random.Generator(np.random.PCG64(seed + 1)).uniform(0.0, 2 * math.pi, size=count)


def _param_circuit(case):
    """The parameterised circuit's plan; its structure does not depend on a seed."""
    circ = create_param_rqc_circuit(case["rows"], case["cols"], case["depth"], seed=workloads.PARAM_SEED)
    return ParamCircuit(circ, planner="greedy", nslice=case["sliced"], precision=case["precision"],
                        batch=1 << (case["bitstrings"] - 1).bit_length(), trials=4, min_fill_trials=4)


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("amplitudes", "sample"):
        w = workloads.WORKLOADS[PLANS[case["plan"]]]
        dsl, data, _ = w.load()
        if kind == "sample":
            return {"case": case, "ex": Executor(dsl, data, graph=1), "seed": seed}
        ex = Executor(dsl, data, precision=case["precision"], graph=int(case["graph"]), batch_last=w.batch_last,
                      autotune=int(case["autotune"]))
        bits = _bitstrings(case["bitstrings"], w.qubits, seed)
        if case["autotune"]:
            ex.amplitudes(bits)
        return {"case": case, "ex": ex, "bits": bits}
    if kind in ("gradient", "variational"):
        pc = _param_circuit(case)
        theta = _angles(pc.num_params, seed)
        if kind == "gradient":
            pc.set_params(theta)
        bits = _bitstrings(case["bitstrings"], case["rows"] * case["cols"], seed)
        return {"case": case, "pc": pc, "theta": theta, "bits": bits}
    return {"case": case, "circuit": create_rqc_circuit(case["rows"], case["cols"], case["depth"], seed=seed)}


def run(state):
    """Results of the complex64 precisions are kept as such: their values carry no more."""
    case = state["case"]
    kind = case["kind"]
    single = case.get("precision", "c128") != "c128"
    if kind == "amplitudes":
        if case["slices"]:
            amps = state["ex"].amplitudes(state["bits"], case["first_slice"], case["first_slice"] + case["slices"])
        else:
            amps = state["ex"].amplitudes(state["bits"])
        return amps.astype(np.complex64) if single else amps
    if kind == "sample":
        bits, amps, m, used = state["ex"].sample_rejection(case["num_samples"], state["seed"])
        return np.frombuffer("".join(bits).encode(), dtype=np.uint8), amps, np.float64(m), used
    if kind == "variational":
        state["pc"].set_params(state["theta"])
    if kind in ("gradient", "variational"):
        loss, grad, amps = state["pc"].loss_and_grad(state["bits"])
        if single:
            return np.float32(loss), grad.astype(np.float32), amps.astype(np.complex64)
        return np.float64(loss), grad, amps
    amps = run_simulation(state["circuit"])
    return np.array(list(amps.values()))


# ----------------------------------------------------------- a saved plan's text
def _labels(text):
    return [] if text == "0" else [int(x) for x in text.split(",")]


def _program(dsl):
    return [s.split() for s in dsl.splitlines() if s.strip() and not s.startswith("#")]


def _variables(prog):
    names = {f[3]: int(f[5]) for f in prog if f[0] == "view"}
    return sorted(names.items(), key=lambda kv: int(kv[0][1:]))


def _chosen_slices(case, prog):
    """Assignments (first variable fastest) of the case's slice range; None: all."""
    if not case.get("slices"):
        return None
    out = []
    for s in range(case["first_slice"], case["first_slice"] + case["slices"]):
        a = {}
        for name, dim in _variables(prog):
            a[name] = s % dim
            s //= dim
        out.append(a)
    return out


def _plan_of(case):
    w = workloads.WORKLOADS[PLANS[case["plan"]]]
    with open(w.prefix() + ".qx") as f:
        return w, _program(f.read())


def _plan_work(prog, batch, slices):
    """Complex multiply-adds x 8 of the plan, steps that no bitstring and no slice
    changes counted once, and the bytes of its tensors and results."""
    dims, dep, cut, flops, elems, seen = {}, {}, {}, 0.0, 0, set()
    fused = slices is None
    for f in prog:
        op = f[0]
        if op == "load":
            dims[f[1]] = [int(x) for x in f[3].split(",")] if len(f) > 3 else []
            dep[f[1]] = cut[f[1]] = False
            if f[2] not in seen:
                seen.add(f[2])
                elems += math.prod(dims[f[1]])
        elif op == "output":
            dims[f[1]], dep[f[1]], cut[f[1]] = [int(f[3])], True, False
        elif op == "view":
            dims[f[1]] = list(dims[f[2]])
            dep[f[1]], cut[f[1]] = dep[f[2]], True
            if not fused:
                dims[f[1]][int(f[4]) - 1] = 1
        elif op == "ncon":
            size = dict(zip(_labels(f[4]), dims[f[3]]))
            size.update(zip(_labels(f[6]), dims[f[5]]))
            dep[f[1]], cut[f[1]] = dep[f[3]] or dep[f[5]], cut[f[3]] or cut[f[5]]
            times = (batch if dep[f[1]] else 1) * (1 if fused or not cut[f[1]] else len(slices))
            flops += 8.0 * math.prod(size.values()) * times
            dims[f[1]] = [size[x] for x in _labels(f[2])]
        else:
            elems += batch * math.prod(dims[f[2]])
    return flops, elems


def work(case):
    kind = case["kind"]
    if kind in ("amplitudes", "sample"):
        _, prog = _plan_of(case)
        # a sample takes five to six candidates here: the bound is the largest ratio seen
        batch = case["bitstrings"] if kind == "amplitudes" else 5.5 * case["num_samples"]
        flops, elems = _plan_work(prog, batch, _chosen_slices(case, prog))
        return {"bytes": 16.0 * elems, "flops": flops}
    n, depth = case["rows"] * case["cols"], case["depth"]
    if kind == "simulate":   # one pass of every gate over the state, every amplitude out
        return {"bytes": 16.0 * 2 ** n, "flops": 8.0 * 2 ** n * 3 * n * depth}
    # forward and two adjoint products of every bitstring's smallest known contraction;
    # inputs: one tensor per gate, outputs: one gradient per angle and the amplitudes
    nb = case["bitstrings"]
    return {"bytes": 16.0 * (6 * n * depth + 3 * n * depth + nb), "flops": 24.0 * nb * n * depth * 4}


# -------------------------------------------- the same values by plain torch, FP64
_DEVICE = "cuda" if torch.cuda.is_available() else "cpu"
_S2 = 1.0 / math.sqrt(2.0)


def _ordered(t, order):
    """t's legs in the given order, contiguous.  A few legs are moved to the front at a
    time, neighbours kept together, since a copy on the device takes few dimensions."""
    legs = list(range(t.dim()))
    shape = list(t.shape)
    t = t.contiguous()
    for at in range((len(order) - 1) // 6 * 6 if order else -1, -1, -6):
        front = order[at:at + 6]
        target = front + [x for x in legs if x not in front]
        if target == legs:
            continue
        runs, where = [], {x: i for i, x in enumerate(target)}   # neighbours in both orders
        for x in legs:
            if runs and where[runs[-1][-1]] + 1 == where[x]:
                runs[-1].append(x)
            else:
                runs.append([x])
        by = sorted(range(len(runs)), key=lambda i: where[runs[i][0]])
        t = t.reshape([math.prod(shape[x] for x in r) for r in runs]).permute(by).contiguous()
        legs = target
    return t.reshape([shape[x] for x in order])


def _pair(a, al, b, bl, cl):
    """C[cl] = sum of A[al] B[bl] over the labels that C does not have."""
    da, db = dict(zip(al, a.shape)), dict(zip(bl, b.shape))
    h = [x for x in al if x in db and x in cl]
    k = [x for x in al if x in db and x not in cl]
    m = [x for x in al if x not in db]
    n = [x for x in bl if x not in da]
    size = lambda ls, d: math.prod(d[x] for x in ls)  # noqa: E731
    x = _ordered(a, [al.index(l) for l in h + m + k]).reshape(size(h, da), size(m, da), size(k, da))
    y = _ordered(b, [bl.index(l) for l in h + k + n]).reshape(size(h, db), size(k, db), size(n, db))
    c = x * y if not k and (size(m, da) == 1 or size(n, db) == 1) else torch.bmm(x, y)
    got = h + m + n
    c = c.reshape([da.get(l, db.get(l)) for l in got])
    return _ordered(c, [got.index(l) for l in cl])


def _contract(prog, tensors, bits, assign):
    """The program for all bitstrings at once (label -1: the bitstring).  Slice variables
    outside `assign` are summed by leaving their legs whole."""
    value = {"0": (1.0, 0.0), "1": (0.0, 1.0), "+": (_S2, _S2), "-": (_S2, -_S2)}
    last = {}
    for i, f in enumerate(prog):
        for name in f[2:]:
            last[name] = i
    env, result = {}, None
    for i, f in enumerate(prog):
        op = f[0]
        if op == "load":
            env[f[1]] = (tensors[f[2]], False)
        elif op == "output":
            v = [value[s[int(f[2]) - 1]] for s in bits]
            env[f[1]] = (torch.tensor(v, dtype=torch.complex128, device=_DEVICE), True)
        elif op == "view":
            t, dep = env[f[2]]
            if f[3] in assign:
                t = t.narrow(int(f[4]) - 1 + int(dep), assign[f[3]], 1)
            env[f[1]] = (t, dep)
        elif op == "ncon":
            (a, da), (b, db) = env[f[3]], env[f[5]]
            al, bl, cl = ([-1] * dep + _labels(s) for dep, s in ((da, f[4]), (db, f[6]), (da or db, f[2])))
            env[f[1]] = (_pair(a, al, b, bl, cl), da or db)
            a = b = None
        else:
            result = env[f[2]]
        for name in set(f[2:]):
            if last.get(name) == i:
                env.pop(name, None)
    t, dep = result
    t = t if dep else t.expand((len(bits),) + tuple(t.shape))
    return t.reshape(len(bits), -1) if t.dim() < 3 else t.permute([0] + list(range(t.dim() - 1, 0, -1))).reshape(len(bits), -1)


def _tensors(data):
    return {k: torch.as_tensor(np.asarray(v, dtype=np.complex128), device=_DEVICE) for k, v in data.items()}


def _plan_amplitudes(case, bits):
    w, prog = _plan_of(case)
    with np.load(w.prefix() + ".npz", allow_pickle=False) as z:
        tensors = _tensors({k: z[k] for k in z.files})
    chosen = _chosen_slices(case, prog)
    if chosen is None:   # a few variables are looped where whole legs would take too much memory
        looped = _variables(prog)[:4 if case["plan"] == "7x7" else 0]
        chosen = [{n: (i >> j) & 1 for j, (n, _) in enumerate(looped)} for i in range(1 << len(looped))]
    out = None
    for a in chosen:
        v = _contract(prog, tensors, bits, a)
        out = v if out is None else out + v
    out = out.cpu().numpy()
    return out[:, 0] if out.shape[1] == 1 else out


def _rotation(which, angle):
    """Rz as its diagonal, Ry as its matrix."""
    half = angle / 2
    if which == "ry":
        c, s = torch.cos(half), torch.sin(half)
        return torch.stack([torch.stack([c, -s]), torch.stack([s, c])]).to(torch.complex128)
    return torch.stack([torch.polar(torch.ones_like(half), -half), torch.polar(torch.ones_like(half), half)])


def _exact_gradient(case, seed):
    pc = _param_circuit(case)
    theta = torch.tensor(_angles(pc.num_params, seed), dtype=torch.float64, requires_grad=True)
    tensors = _tensors(pc.graph.data)
    for p, key, _ in pc.terms:   # the angles are those of Rz Ry Rz, qubit after qubit
        tensors[key] = _rotation(("rz", "ry", "rz")[p % 3], theta[p]).to(_DEVICE)
    bits = _bitstrings(case["bitstrings"], case["rows"] * case["cols"], seed)
    amps = _contract(_program(pc.dsl), tensors, bits, {})[:, 0]
    loss = amps.abs().square().sum()
    loss.backward()
    return np.float64(loss.item()), theta.grad.numpy(), amps.detach().cpu().numpy()


_GATES = None


def _gate(name):
    global _GATES
    if _GATES is None:
        x = np.array([[0, 1], [1, 0]], dtype=np.complex128)
        y = np.array([[0, -1j], [1j, 0]], dtype=np.complex128)
        root = lambda g: 0.5 * ((1 + 1j) * np.eye(2) + (1 - 1j) * g)  # noqa: E731
        _GATES = {"sx": root(x), "sy": root(y), "sw": root(_S2 * (x + y))}
    return _GATES[name]


def _state(circuit):
    """The circuit's amplitudes, first qubit most significant."""
    n = circuit.num_qubits
    v = np.zeros((2,) * n, dtype=np.complex128)
    v[(0,) * n] = 1.0
    for g in circuit.ops:
        if g.name == "cz":
            at = [slice(None)] * n
            at[g.qubits[0] - 1] = at[g.qubits[1] - 1] = 1
            v[tuple(at)] *= -1
        else:
            v = np.moveaxis(np.tensordot(_gate(g.name), v, axes=(1, g.qubits[0] - 1)), 0, g.qubits[0] - 1)
    return v.reshape(-1)


def _exact_sample(case, seed):
    """Candidate j is bit q of the Philox4x64-10 block at counter j, key (seed, 0), its
    uniform the top 53 bits of the block at key (seed, 1); accepted where u M < r."""
    w, _ = _plan_of(case)
    num, n = case["num_samples"], w.qubits
    every = [format(x, f"0{n}b") for x in range(2 ** n)]
    table = dict(zip(every, _plan_amplitudes(case, every)))
    m, bits, amps, used = 1e-4, [], [], 0
    block = 4096
    while len(bits) < num:
        word = [np.random.Philox(counter=(used - 1) % 2 ** 256, key=seed + (k << 64)).random_raw(4 * block)[::4]
                for k in (0, 1)]
        for c, u in zip(word[0], word[1]):
            s = "".join("01"[(int(c) >> q) & 1] for q in range(n))
            a = table[s]
            r = (a.real * a.real + a.imag * a.imag) * 2.0 ** n
            used += 1
            m = max(m, r)
            if float(int(u) >> 11) * 2.0 ** -53 * m < r:
                bits.append(s)
                amps.append(a)
                if len(bits) == num:
                    break
    return np.frombuffer("".join(bits).encode(), dtype=np.uint8), np.array(amps), np.float64(m), used


def exact(case, seed):
    kind = case["kind"]
    if kind == "amplitudes":
        w = workloads.WORKLOADS[PLANS[case["plan"]]]
        return _plan_amplitudes(case, _bitstrings(case["bitstrings"], w.qubits, seed))
    if kind == "sample":
        return _exact_sample(case, seed)
    if kind == "simulate":
        return _state(create_rqc_circuit(case["rows"], case["cols"], case["depth"], seed=seed))
    return _exact_gradient(case, seed)
