"""Fused field gather + Boris push (PyPIC3D/pusher/particle_push.py:13-175).

One HIP kernel gathers the six Yee-staggered components with the particle
shape (CIC or TSC, reduced axes collapsed to index g) and applies the
non-relativistic (boris.py:14-56) or relativistic (boris.py:60-124) Boris
update, or the Higuera-Cary update (higuera_cary.py:57-113) when
``particle_pusher == "higuera_cary"`` (particle_push.py:109-132).
"""

from __future__ import annotations

from .. import _native as N
from .._tensors import (PUSH, as_field3, binned_workspace, check_fields, is_f64, make_desc, make_species, new_soa,
                        particle_planes, pic_particles)
from ..particles.particle_class import TiledParticles


def check_pusher(static_parameters):
    if static_parameters.particle_pusher not in ("boris", "higuera_cary"):
        raise ValueError(f"Unknown particle_pusher: {static_parameters.particle_pusher}")


# The push through tiles brings the launches of the binning (20 us of host time), so first-order sets take it from
# 2^20 slots on.  us in slot order / through tiles, random order: 2^18 slots 58 / 76, 2^19 60 to 96 / 90 to 97, 2^20 114,
# 186, 329 / 119, 142, 192 (32, 4, 1 particles a cell), 2^21 371, 787 / 181, 304; cell order 56 to 80 / 75 to 83
# throughout.  Second order, 2^18: random 170 to 195 / 92 to 97, cell order 89 / 82, but with 40 work items (16^3 cells)
# 98 / 118: a tile's 8192 records are an item and an item a block, and fewer than 64 leave most CUs idle.
_TILE_SLOTS_1, _TILE_SLOTS_2, _TILE_ITEMS = 1 << 20, 1 << 18, 64


def _through_tiles(desc, slots):
    tiles = 1
    for a in range(3):
        tiles *= -(-desc.n[a] // 8)
    least = _TILE_SLOTS_1 if desc.shape_factor == 1 else _TILE_SLOTS_2
    return slots >= least and tiles + slots // 8192 >= _TILE_ITEMS


def push_into(desc, sp, xp, up, act, E3, B3, Ee, Be, u_planes, stream):
    """Pushed velocities into u_planes; E3, B3 are 3-D components, Ee, Be the
    external fields' pointers or None."""
    f64 = is_f64(xp[0])
    pp = pic_particles(xp, up, act)
    ws = None
    if not f64 and _through_tiles(desc, xp[0].numel()):
        ws = binned_workspace(desc, sp, PUSH, xp[0].device)
    if ws is not None:
        N.call("pic_push_binned", desc, sp, pp, N.p3(E3), N.p3(B3), Ee, Be, N.p3(u_planes), N.ptr(ws), ws.numel(),
               stream)
    else:
        N.call(N.op("pic_push", f64), desc, sp, pp, N.p3(E3), N.p3(B3), Ee, Be, N.p3(u_planes), stream)


def particle_push(particles, species_config, E_tiles, B_tiles, static_parameters, dynamic_parameters,
                  E_external=None, B_external=None):
    """Returns TiledParticles with the pushed velocities; x and active are passed through."""
    check_pusher(static_parameters)
    desc = make_desc(static_parameters, dynamic_parameters)
    xp, up, act = particle_planes(particles)
    S, P = xp[0].shape
    sp = make_species(species_config, P)
    E3 = [as_field3(c, "E") for c in E_tiles]
    B3 = [as_field3(c, "B") for c in B_tiles]
    E_external = None if E_external is None else [as_field3(c, "E_ext") for c in E_external]
    B_external = None if B_external is None else [as_field3(c, "B_ext") for c in B_external]
    Ee = None if E_external is None else N.p3(E_external)
    Be = None if B_external is None else N.p3(B_external)
    check_fields(desc, *E3, *B3, *(E_external or ()), *(B_external or ()), dtype=xp[0].dtype)
    store, view = new_soa(S, P, xp[0].device, xp[0].dtype)
    push_into(desc, sp, xp, up, act, E3, B3, Ee, Be, [store[0], store[1], store[2]], N.stream_handle())
    return TiledParticles(x=particles.x, u=view, active=particles.active)
