"""Gradients of amplitude losses with respect to gate angles.

`qx_amplitudes_vjp` returns, per data key, grad = sum_b amp_cot_b conj(d amp_b / dT)
(the ChainRulesCore pullback of a holomorphic map).  For a parameterised gate T(theta)
the chain rule gives dL/dtheta = Re(sum_i conj(grad_i) dT_i/dtheta) for a real loss L
whose cotangent is amp_cot = dL/d(Re amp) + i dL/d(Im amp), e.g. amp_cot = 2 amp for
L = sum |amp|^2.  dT/dtheta is the derivative matrix pushed through the same
circuit-to-tensor conversion as the gate itself (diagonal gates stay rank-1 on
their wire).  Every gate tensor gets its own data key (no dedupe).  No
counterpart exists in the reference, which is forward-only.
"""

from __future__ import annotations

import numpy as np

from . import _native
from .circuits import Circuit, param_gate_tensors
from .compute_graph import build_compute_graph
from .planning import contraction_scheme, sweep_contraction_plan
from .simulation import Executor
from .tn import gate_tensor_map


class ParamCircuit:
    """A parameterised circuit compiled to a saved plan with per-gate data keys."""

    def __init__(self, circ: Circuit, planner: str = "sweep", nslice: int = 0, precision: str = "c128",
                 batch: int | None = None, device: int = 0, graph: int = 1, **plan_kwargs):
        self._circ, self._angles = circ, None
        tnc, names = gate_tensor_map(circ)
        tnc.add_input()
        tnc.add_output()
        if planner == "sweep":
            plan, groups = sweep_contraction_plan(tnc, **plan_kwargs), []
        else:
            groups, plan, _ = contraction_scheme(tnc, nslice, **plan_kwargs)
        self.graph = build_compute_graph(tnc, plan, groups, dedupe=False)
        key_of = {c.name: c.args[0] for c in self.graph.commands if c.kind == "load"}
        self._pgates = []   # (gate index, data key) of every parameterised gate
        for gi, (g, tn_names) in enumerate(zip(circ.ops, names)):
            if g.param is None:
                continue
            if len(tn_names) != 1:
                raise ValueError("parameterised gates must convert to one tensor")
            self._pgates.append((gi, key_of[tn_names[0]]))
        self._index_gates()
        self._set_terms([circ.ops[gi].theta for gi, _ in self._pgates])
        self.dsl = self.graph.to_dsl()
        self.executor = Executor(self.dsl, self.graph.data, precision=precision, device=device, batch=batch,
                                 graph=graph)
        at = {k: i for i, k in enumerate(self.executor.plan.keys_needed())}
        self._pkeys = np.array([at[k] for k in self._tkeys], dtype=np.int64)
        self.num_params = circ.num_params

    @property
    def circ(self) -> Circuit:
        """The circuit at the current angles."""
        if self._angles is not None:
            self._circ, self._angles = self._circ.with_params(self._angles), None
        return self._circ

    @circ.setter
    def circ(self, circ: Circuit) -> None:
        self._circ, self._angles = circ, None

    @property
    def terms(self) -> list:
        """Chain-rule terms (param index, key, dT/dtheta in the key's array layout)."""
        return [(int(p), k, d) for p, k, d in zip(self._tp, self._tkeys, self._arrays(self._td))]

    def _index_gates(self) -> None:
        """Where each parameterised gate's tensor lies in the flat arrays of all of them,
        gates of a kind together, so that a new set of angles is a few array operations."""
        ops = self._circ.ops
        self._tkeys = [k for _, k in self._pgates]
        self._tp = np.array([ops[gi].param for gi, _ in self._pgates], dtype=np.int64)
        self._shapes = [self.graph.data[k].shape for k in self._tkeys]
        sizes = np.array([int(np.prod(s)) for s in self._shapes], dtype=np.int64)
        self._tstart = np.cumsum(sizes) - sizes
        self._tsize = int(sizes.sum())
        self._kinds = []   # (gate name, its positions among the gates, flat index of every value)
        for name in sorted({ops[gi].name for gi, _ in self._pgates}):
            at = np.array([i for i, (gi, _) in enumerate(self._pgates) if ops[gi].name == name], dtype=np.int64)
            shape = {"rz": (2,), "ry": (2, 2)}[name]
            if any(self._shapes[i] != shape for i in at):
                raise ValueError(f"derivative of gate {name} has a different tensor structure")
            self._kinds.append((name, at, (self._tstart[at][:, None] + np.arange(int(np.prod(shape)))).reshape(-1)))

    def _tensors(self, angles, deriv: bool) -> np.ndarray:
        """Every parameterised gate's tensor (or dT/dtheta), flat, one after the other.  A
        rotation whose tensor has no off-diagonal value has another structure there."""
        out = np.zeros(self._tsize, dtype=np.complex128)
        for name, at, index in self._kinds:
            t = param_gate_tensors(name, [angles[i] for i in at], deriv)
            if t.shape[1] == 4 and np.any((t[:, 1] == 0) & (t[:, 2] == 0)):
                raise ValueError(f"derivative of gate {name} has a different tensor structure" if deriv else
                                 f"gate {name} at the new angle has a different tensor structure")
            out[index] = t.reshape(-1)
        return out

    def _arrays(self, flat: np.ndarray) -> list:
        return [flat[a:a + int(np.prod(s))].reshape(s, order="F") for a, s in zip(self._tstart.tolist(), self._shapes)]

    def _set_terms(self, angles) -> None:
        """dT/dtheta of every gate at the given angles, for one segmented reduction."""
        self._td = self._tensors(angles, True)

    def params(self) -> np.ndarray:
        return self.circ.params()

    def set_params(self, theta) -> None:
        """Move the plan to new angles: every parameterised gate's tensor is rebuilt and
        all of them re-uploaded in one copy (`qx_plan_update_tensors`), so the lowering,
        tuning and captured graphs are kept; the chain-rule terms follow."""
        theta = np.asarray(theta, dtype=np.float64)
        if theta.shape != (self.num_params,):
            raise ValueError(f"need {self.num_params} angles, got shape {theta.shape}")
        angles = theta[self._tp].tolist()
        flat = self._tensors(angles, False)
        if self._tkeys:
            self.executor.plan.update_tensors(self._pkeys, flat)
        for key, arr in zip(self._tkeys, self._arrays(flat)):
            self.graph.data[key] = arr
        self._angles = theta.copy()
        self._set_terms(angles)

    def amplitudes(self, bits) -> np.ndarray:
        return self.executor.amplitudes(bits)

    def param_grad(self, key_grad: dict) -> np.ndarray:
        """dL/dtheta_p = sum over the gate tensors T of parameter p of
        Re <dL/dT, dT/dtheta_p> (the cotangent is conj-linear)."""
        out = np.zeros(self.num_params)
        if not self._tkeys:
            return out
        g = np.concatenate([key_grad[k] for k in self._tkeys])
        per_term = np.add.reduceat(np.real(np.conj(g) * self._td), self._tstart)
        np.add.at(out, self._tp, per_term)
        return out

    def _param_grad_flat(self, g_flat: np.ndarray) -> np.ndarray:
        """`param_grad` from the pullback's flat gradient (layout of the plan's
        `key_offsets`): the terms' entries gathered by one precomputed index."""
        out = np.zeros(self.num_params)
        if not self._tkeys:
            return out
        if getattr(self, "_tidx", None) is None:
            offs = self.executor.plan.key_offsets()
            self._tidx = np.concatenate([np.arange(offs[k][0], offs[k][0] + offs[k][1]) for k in self._tkeys])
        per_term = np.add.reduceat(np.real(np.conj(g_flat[self._tidx]) * self._td), self._tstart)
        np.add.at(out, self._tp, per_term)
        return out

    def loss_and_grad(self, bits) -> tuple:
        """L = sum_b |amp_b|^2 and dL/dtheta: one pass of forward and pullback when
        every slice variable is contracted inline, else the amplitudes first and the
        pullback of the cotangent 2 amp after."""
        try:
            amps, g_flat = self.executor.plan.norm_vjp(bits, flat=True)
        except _native.QxError as e:
            if e.status != _native.QX_ERR_UNSUPPORTED:
                raise
            amps = self.amplitudes(bits)
            kg = self.executor.vjp(bits, 2.0 * amps)
            return float(np.sum(np.abs(amps) ** 2)), self.param_grad(kg), amps
        loss = float(np.sum(np.abs(amps) ** 2))
        return loss, self._param_grad_flat(g_flat), amps
