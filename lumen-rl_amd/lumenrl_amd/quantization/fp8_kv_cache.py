"""Per-step FP8 KV-cache scale recalibration on MI355X kernels.

Behaviour of ``FP8KVCacheQuantizer`` (lumenrl/quantization/fp8_kv_cache.py:26-80):
each RL step, every ``nn.Linear`` whose last name component is ``q_proj``,
``k_proj`` or ``v_proj`` gets a float32 0-dim buffer
``_lumenrl_fp8_kv_scale_<q_proj|k_proj|v_proj>`` equal to
``max(|W|.max(), FLT_MIN) / 448``.  A buffer that exists is updated in place,
and a missing one is registered on the weight's device.

The reference runs one torch reduction per projection.  Here all projections
of a model share one ``TensorScalePlan``: two kernel launches for the whole
model, bit-identical to the torch ops on x86.  The plan is kept while the
weights' storage stays put (the optimizer updates parameters in place).
Buffers this class registers are views of the plan's scale vector, so a later
recalibration writes them with no per-module copy.
"""

from __future__ import annotations

import logging
from typing import Any, Optional

import torch
import torch.nn as nn
from torch import Tensor

from lumenrl_amd.quantization import ops
from lumenrl_amd.quantization.fp8_config import FP8Config

logger = logging.getLogger(__name__)

_KV_PROJECTIONS = frozenset({"q_proj", "k_proj", "v_proj"})
_BUFFER_PREFIX = "_lumenrl_fp8_kv_scale_"


def _atom_quant_spec() -> Any:
    """ATOM's quant_spec module if that engine is installed (it reads the buffers)."""
    try:
        from atom import quant_spec  # type: ignore[attr-defined]
    except ImportError:
        return None
    return quant_spec


class _ScaleGroup:
    """A TensorScalePlan over one dtype's projections, with staging for
    weights the kernels cannot read in place (host memory, float64)."""

    def __init__(self, sources: list[Tensor], device: torch.device) -> None:
        self.sources = sources
        self.staged: list[Optional[Tensor]] = []
        inputs = []
        for w in sources:
            if w.device == device and w.dtype != torch.float64:
                view, *_ = ops.matrix_view(w)
                if view.data_ptr() == w.data_ptr():
                    self.staged.append(None)
                    inputs.append(w)
                    continue
            buf = torch.empty(w.shape, dtype=_kernel_dtype(w), device=device)
            self.staged.append(buf)
            inputs.append(buf)
        self.plan = ops.TensorScalePlan(inputs)

    def run(self) -> Tensor:
        for src, buf in zip(self.sources, self.staged):
            if buf is not None:
                buf.copy_(src, non_blocking=True)  # float64 -> float32 rounds like w.to(float32)
        return self.plan.run()


def _kernel_dtype(w: Tensor) -> torch.dtype:
    return torch.float32 if w.dtype == torch.float64 else w.dtype


def _signature(w: Tensor) -> tuple:
    """What the plan's table holds of a weight."""
    return w.data_ptr(), w.shape, w.stride(), w.dtype, w.device


def _projections(model: nn.Module) -> list[tuple[str, nn.Linear]]:
    """(last name component, module) of every q/k/v projection, in the order and
    with the names of ``model.named_modules()``: each module once, under the
    first path that reaches it."""
    found, seen, usual = [], set(), nn.Module.named_modules

    def walk(module: nn.Module, short: str) -> None:
        # a class or an instance may have its own traversal, and a model may be a
        # proxy that only delegates to a module
        if getattr(type(module), "named_modules", None) is not usual or "named_modules" in module.__dict__:
            raise _OwnNames
        if module in seen:
            return
        seen.add(module)
        if short in _KV_PROJECTIONS and isinstance(module, nn.Linear):
            found.append((short, module))
        for name, child in module._modules.items():
            if child is not None:
                walk(child, name.rpartition(".")[2] if "." in name else name)

    try:
        walk(model, "")
    except _OwnNames:  # a module with a traversal of its own is asked for it
        found = []
        for name, module in model.named_modules():
            short = name.rpartition(".")[2]
            if isinstance(module, nn.Linear) and short in _KV_PROJECTIONS:
                found.append((short, module))
    return found


class _OwnNames(Exception):
    pass


class FP8KVCacheQuantizer:
    """Maintains the per-step q/k/v projection FP8 scales the inference KV caches use."""

    def __init__(self, config: FP8Config) -> None:
        self._config = config
        self._enabled = False
        self._atom_spec = _atom_quant_spec()
        if self._atom_spec is None:
            logger.debug("atom.quant_spec not available; KV cache path uses torch heuristics only.")
        self._groups: dict[torch.dtype, _ScaleGroup] = {}
        self._signature: list[tuple] = []
        self._slots: list[tuple[torch.dtype, int]] = []  # each weight's group and place in it

    def _run(self, weights: list[Tensor]) -> dict[torch.dtype, Tensor]:
        """Each group's scale vector, recomputed; weight i's is at ``_slots[i]``."""
        sig = [_signature(w) for w in weights]
        if sig != self._signature:
            weights = [w.detach() for w in weights]
            dev = next((w.device for w in weights if w.is_cuda), None) or ops.require_device()
            by_dtype: dict[torch.dtype, list[Tensor]] = {}
            slots = []
            for w in weights:
                ws = by_dtype.setdefault(_kernel_dtype(w), [])
                slots.append((_kernel_dtype(w), len(ws)))
                ws.append(w)
            self._groups = {dt: _ScaleGroup(ws, dev) for dt, ws in by_dtype.items()}
            self._slots = slots
            self._signature = sig
        return {dt: g.run() for dt, g in self._groups.items()}

    def recalibrate_scales(self, model: nn.Module) -> None:
        """Recompute every q/k/v projection's scale from its current weight."""
        if not self._config.is_fp8_enabled():
            logger.debug("FP8 disabled; skipping KV scale recalibration.")
            return
        targets = _projections(model)
        if not targets:
            logger.warning("recalibrate_scales: no q_proj/k_proj/v_proj Linear layers found on model.")
            return
        vecs = self._run([m.weight for _, m in targets])
        base = {dt: (v.data_ptr(), v.device) for dt, v in vecs.items()}
        for (short, module), (dt, i) in zip(targets, self._slots):
            name = _BUFFER_PREFIX + short
            buf = module._buffers.get(name)
            there = buf is not None or hasattr(module, name)  # a failing look-up takes 1 us
            if there and buf is None:
                buf = getattr(module, name)
            at, dev = base[dt]
            if isinstance(buf, Tensor) and buf.data_ptr() == at + 4 * i and buf.device == dev:
                continue  # a view of the vector the kernels have just written
            s = vecs[dt][i]
            if there:
                buf.copy_(s.to(buf.device))
            else:
                home = module.weight.device
                module.register_buffer(name, s if home == s.device else s.to(home))
        logger.debug("recalibrate_scales: updated %d projection layers.", len(targets))

    def enable(self, model: nn.Module) -> None:
        """Flag the model for FP8 KV caches and create/refresh the scale buffers."""
        if not self._config.is_fp8_enabled():
            logger.info("FP8 disabled; FP8KVCacheQuantizer.enable is a no-op.")
            return
        setattr(model, "_lumenrl_fp8_kv_cache_enabled", True)
        self._enabled = True
        self.recalibrate_scales(model)
        if self._atom_spec is not None:
            logger.debug("atom.quant_spec present; ATOM engine may consume _lumenrl_fp8_kv_scale_* buffers.")

    @property
    def enabled(self) -> bool:
        return self._enabled
