"""Particle state: integer mesh anchors plus float displacements (single device).

Mirrors ``src/pmpp/nbody/particles.py``: the fields of ``Particles`` (:33-127), ``gen_grid``
(:615-727, single-device branch), ``from_pos`` (:440-478) and ``pos`` (:773-798).  Arrays are
torch tensors; ``pmid`` is (N,3) int16, ``disp``/``vel``/``acc`` are (N,3) float32 and
``unused_index`` is (N,) bool (True marks padding; all False on one device, :686-692).
"""

from __future__ import annotations

from dataclasses import dataclass, fields, replace as dc_replace
from typing import Any, Optional

import numpy as np
import torch


@dataclass(frozen=True, eq=False)
class Particles:
    conf: Any
    pmid: torch.Tensor
    disp: torch.Tensor
    vel: Optional[torch.Tensor] = None
    acc: Optional[torch.Tensor] = None
    unused_index: Optional[torch.Tensor] = None

    def __post_init__(self):
        object.__setattr__(self, "pmid", self.pmid.to(torch.int16))
        for name in ("disp", "vel", "acc"):
            v = getattr(self, name)
            if v is not None and v.dtype != torch.float32:
                object.__setattr__(self, name, v.to(torch.float32))
        if self.unused_index is not None and self.unused_index.dtype != torch.bool:
            object.__setattr__(self, "unused_index", self.unused_index.to(torch.bool))

    def __len__(self):
        return self.pmid.shape[0]

    def replace(self, **changes):
        if type(self) is not Particles or not changes.keys() <= _FIELDS:
            return dc_replace(self, **changes)
        # three of these per step of a run: the fields are set as __init__ and __post_init__ do, which
        # leaves the unchanged ones as they are
        p = object.__new__(Particles)
        d = p.__dict__
        for name in _FIELDS:
            v = changes[name] if name in changes else self.__dict__[name]
            dtype = _DTYPES.get(name)
            if dtype is not None and (v is not None or name == "pmid") and v.dtype != dtype:
                v = v.to(dtype)
            d[name] = v
        return p

    @property
    def valid_mask(self):
        return None if self.unused_index is None else ~self.unused_index

    @classmethod
    def gen_grid(cls, conf, vel=False, acc=False, device="cuda", lpt=None):
        """Particles on the uniform Lagrangian grid with exact integer anchors (:615-727).

        On a GPU they are made there (``pm_ic_lpt_particles``), the same values bit for bit.
        ``lpt`` (GPU only) adds LPT terms: (grad1, grad2, D1, V1, D2, V2), the displacements D1 grad1 +
        D2 grad2 and the velocities V1 grad1 + V2 grad2 of (3, *grid) gradient meshes (None: none)."""
        dev = torch.device(device)
        if dev.type == "cuda" and conf.dim == 3:
            from .. import _lib
            from .._torch import ptr, stream_handle

            n = conf.ptcl_num
            pm_t = torch.empty((n, 3), dtype=torch.int16, device=dev)
            dp_t = torch.empty((n, 3), dtype=torch.float32, device=dev)
            v = torch.empty_like(dp_t) if vel else None
            g1, g2, *factors = lpt if lpt is not None else (None, None, 0.0, 0.0, 0.0, 0.0)
            with torch.cuda.device(dev):  # a default stream's handle names the current device's
                _lib.call("pm_ic_lpt_particles", _lib.int3(conf.ptcl_grid_shape), _lib.int3(conf.mesh_shape),
                          float(conf.cell_size), ptr(g1), ptr(g2), *factors, ptr(pm_t), ptr(dp_t), ptr(v),
                          stream_handle(dev))
            unused = torch.zeros(n, dtype=torch.bool, device=dev)
            return cls(conf, pm_t, dp_t, vel=v, acc=torch.zeros_like(dp_t) if acc else None, unused_index=unused)
        pmid, disp = [], []
        for sp, sm in zip(conf.ptcl_grid_shape, conf.mesh_shape):
            p = np.rint(np.linspace(0, sm, num=sp, endpoint=False)).astype(np.int64)
            d = (np.arange(sp) * sm - p * sp).astype(np.float64) * (conf.cell_size / sp)
            pmid.append(p.astype(np.int16))
            disp.append(d.astype(np.float32))
        pm = np.stack(np.meshgrid(*pmid, indexing="ij"), axis=-1).reshape(-1, conf.dim)
        dp = np.stack(np.meshgrid(*disp, indexing="ij"), axis=-1).reshape(-1, conf.dim)
        pm_t = torch.from_numpy(pm).to(device)
        dp_t = torch.from_numpy(dp).to(device)
        unused = torch.zeros(pm.shape[0], dtype=torch.bool, device=device)
        v = torch.zeros_like(dp_t) if vel else None
        a = torch.zeros_like(dp_t) if acc else None
        return cls(conf, pm_t, dp_t, vel=v, acc=a, unused_index=unused)

    @classmethod
    def from_pos(cls, conf, pos, vel=None, acc=None, wrap=True):
        """pmid = rint(pos / cell), disp = pos - pmid * cell (:470-478)."""
        pos = torch.as_tensor(pos)
        cell = conf.cell_size
        pmid = torch.round(pos / cell)
        disp = pos - pmid * cell
        pmid = pmid.to(torch.int16)
        if wrap:
            shape = torch.tensor(conf.mesh_shape, dtype=torch.int16, device=pmid.device)
            pmid = torch.remainder(pmid, shape)
        return cls(conf, pmid, disp.to(torch.float32), vel=vel, acc=acc, unused_index=None)

    def pos(self, dtype=torch.float64, wrap=True):
        """pmid * cell + disp, wrapped into the box (:773-798)."""
        p = self.pmid.to(dtype) * self.conf.cell_size + self.disp.to(dtype)
        if wrap:
            box = torch.tensor(self.conf.box_size, dtype=dtype, device=p.device)
            p = torch.remainder(p, box)
        return p


_FIELDS = {f.name: None for f in fields(Particles)}.keys()
_DTYPES = {"pmid": torch.int16, "disp": torch.float32, "vel": torch.float32, "acc": torch.float32,
           "unused_index": torch.bool}
