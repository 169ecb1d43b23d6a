"""Charge density (PyPIC3D/deposition/rho.py:29-196).

rho += q w / (dx dy dz) * S_x S_y S_z at node points, fold + refresh with the
particle codes, digital filter (+ refresh) when current_filter == "digital".
"""

from __future__ import annotations

from .. import _native as N
from .._tensors import RHO, as_field3, binned_workspace, check_fields, is_f64, like_input, make_desc, make_species, particle_planes, pic_particles


def deposit_rho_into(desc, sp, pp, rho3, current_filter, stream, scratch=None, tile=None, starts=None):
    """tile/starts: tile-ordered deposit for particles sorted by pic_tile_keys
    (FP32 only); float64 rho runs the FP64 path."""
    f64 = is_f64(rho3)
    filtered = current_filter == "digital"
    raw = rho3      # the filter reads the raw deposit from an array of its own
    if filtered:
        raw = scratch if scratch is not None else rho3.new_empty(rho3.shape)
    N.call(N.op("pic_zero_fields", f64), desc, N.p1(raw), stream)
    if tile and not f64:
        N.call("pic_deposit_rho_tiled", desc, sp, pp, N.ptr(raw), int(tile), N.ptr(starts), stream)
    else:
        ws = None if f64 else binned_workspace(desc, sp, RHO, raw.device)
        if ws is not None:
            N.call("pic_deposit_rho_binned", desc, sp, pp, N.ptr(raw), N.ptr(ws), ws.numel(), stream)
        else:
            N.call(N.op("pic_deposit_rho", f64), desc, sp, pp, N.ptr(raw), stream)
    N.call(N.op("pic_finish_current", f64), desc, N.p1(raw), 1, stream)
    if filtered:
        N.call(N.op("pic_filter_refresh", f64), desc, N.p1(raw), N.p1(rho3), 0, float(desc.alpha), 1, 0, stream)


def compute_rho(particles, species_config, rho, static_parameters, dynamic_parameters):
    desc = make_desc(static_parameters, dynamic_parameters)
    xp, up, act = particle_planes(particles)
    sp = make_species(species_config, xp[0].shape[1])
    templ = as_field3(rho, "rho")
    check_fields(desc, templ, dtype=xp[0].dtype)
    out = templ.new_empty(templ.shape)
    deposit_rho_into(desc, sp, pic_particles(xp, up, act), out, static_parameters.current_filter,
                     N.stream_handle())
    return like_input(out, rho)
