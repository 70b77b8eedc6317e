"""One full xi step of the plasma (plasma3d/solver.py:9-78) as one native call.

``step_dxi`` keeps the reference's signature and value semantics (fresh
particle, field and current objects every step) but runs the free stream, the
three pushes, three deposits and two field solves as one stream-ordered
sequence of HIP kernels (lc3d_plasma_step), with no host round trip."""
from __future__ import annotations

import torch

from .. import _native, runtime
from .._native import ptr, stream_ptr
from ..config import Config
from . import _bind
from .data import Arrays
from .fields import FIELD_KEYS, get_field_computer, new_fields
from .move import get_plasma_particles_mover
from .rhoj import get_rhoj_computer


class Plane2d3vPlasmaSolver:
    def __init__(self, config: Config):
        self.config = config
        self.ctx = runtime.context(config)
        self.dt = runtime.Dtypes(config.precision())
        self.N = config.getint('window-width-steps')
        self.ion_model = config.get('ion-model')
        # The reference's per-stage factories, for callers that use them.
        self.compute_rhoj = get_rhoj_computer(config)
        self.compute_fields = get_field_computer(config)
        self.move_particles_wo_fields, self.move_particles = get_plasma_particles_mover(config)
        # The electrons' noise filter after the last push (solver.py:16-17,
        # 69-73) runs inside the native step.
        self.declustering_enabled = config.getbool('declustering-enabled')
        if self.declustering_enabled:
            from .noise_filter import get_noise_filter
            self.noise_filter = get_noise_filter(config)

    def step_dxi(self, particles_prev: dict, fields_prev: Arrays, currents_prev: Arrays,
                 const_arrays: Arrays, rho_beam_full, rho_beam_prev):
        N, dt, dev = self.N, self.dt, runtime.device()
        sorts = list(const_arrays.sorts.items())
        particles_full = {}
        structs = (_native.Sort * len(sorts))()
        for i, (sort, column) in enumerate(sorts):
            prev = particles_prev[sort]
            x_init, y_init, x_offt, y_offt, px, py, pz, q, m = _bind.checked_pointers(prev, dt)
            full = Arrays.wrap(
                x_init=prev.x_init, y_init=prev.y_init, m=prev.m,
                x_offt=torch.empty_like(prev.x_offt), y_offt=torch.empty_like(prev.y_offt),
                px=torch.empty_like(prev.px), py=torch.empty_like(prev.py),
                pz=torch.empty_like(prev.pz), q=torch.empty_like(prev.q),
                **{k: getattr(prev, k) for k in prev.names()
                   if k not in _bind.PARTICLE_KEYS})
            particles_full[sort] = full
            # The arrays of layer k+1 are fresh, and m is the same tensor.
            structs[i] = _native.Sort(
                prev.m.numel(), x_init, y_init, m, x_offt, y_offt, px, py, q, pz,
                full.x_offt.data_ptr(), full.y_offt.data_ptr(), full.px.data_ptr(),
                full.py.data_ptr(), full.q.data_ptr(), full.pz.data_ptr(), column)
            if self.declustering_enabled and i == 0:
                z = lambda: torch.zeros_like(prev.x_offt, dtype=torch.float64)
                dxp = getattr(prev, 'dx_chaotic', None)
                dyp = getattr(prev, 'dy_chaotic', None)
                dxp = z() if dxp is None else dxp.to(torch.float64).contiguous()
                dyp = z() if dyp is None else dyp.to(torch.float64).contiguous()
                full.dx_chaotic, full.dy_chaotic = z(), z()
                s = structs[i]
                s.dx_chaotic_prev, s.dy_chaotic_prev = dxp.data_ptr(), dyp.data_ptr()
                s.dx_chaotic, s.dy_chaotic = full.dx_chaotic.data_ptr(), full.dy_chaotic.data_ptr()
        fields_full = new_fields(N, dt.full)
        # The half-step fields are the step's own: seven grids of one tensor.
        half = torch.empty(7, N, N, dtype=dt.half, device=dev)
        grid_bytes = half.stride(0) * half.element_size()
        fields_half = _native.Fields(*range(half.data_ptr(), half.data_ptr() + 7 * grid_bytes,
                                            grid_bytes))
        cur = Arrays.wrap(**{k: torch.empty(2, N, N, dtype=dt.current, device=dev)
                             for k in ('ro', 'jx', 'jy', 'jz')})
        bg = None
        if self.ion_model == 'background':
            bg = const_arrays.ro_initial
            if bg.dtype != dt.current:
                bg = bg.to(dt.current)
            bg = bg.contiguous()
        elif len(sorts) == 1:
            for k in ('ro', 'jx', 'jy', 'jz'):
                getattr(cur, k)[1].zero_()
        rbf = rho_beam_full.to(dt.beam_rho).contiguous()
        rbp = rho_beam_prev.to(dt.beam_rho).contiguous()
        self.ctx.check(self.ctx.lib.lc3d_plasma_step(
            self.ctx.handle, len(sorts), structs, _bind.fields7(fields_prev),
            _bind.currents(currents_prev), ptr(rbf), ptr(rbp), ptr(bg),
            _native.Fields(*[getattr(fields_full, k).data_ptr() for k in FIELD_KEYS]),
            fields_half, _native.Currents(cur.ro.data_ptr(), cur.jx.data_ptr(),
                                          cur.jy.data_ptr(), cur.jz.data_ptr()),
            stream_ptr()), 'lc3d_plasma_step')
        return particles_full, fields_full, cur
