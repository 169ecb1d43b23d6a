"""Direct current J = q v S (PyPIC3D/deposition/J_from_rhov.py:31-260).

Node weights along the other axes, face weights along the current's axis with
the face offset (x - grid0) - (anchor + 1/2) dx (:139-141) -- these
extrapolate, as in the reference.  Then fold + refresh with the particle
codes, and the optional bilinear / digital filter (+ refresh).
"""

from __future__ import annotations

from .. import _native as N
from .._tensors import DIRECT, as_field3, binned_workspace, check_fields, is_f64, like_input, make_desc, make_species, particle_planes, pic_particles


def raw_direct_current(J3, current_filter, scratch=None):
    """The arrays that take the raw deposit: J3, or, as the filter reads it from
    other arrays than it writes, scratch (new ones where it is None)."""
    if current_filter not in ("bilinear", "digital"):
        return J3
    return scratch if scratch is not None else [c.new_empty(c.shape) for c in J3]


def deposit_direct_into(desc, sp, pp, J3, current_filter, stream, scratch=None, tile=None, starts=None,
                        workspace=binned_workspace):
    """tile/starts: tile-ordered deposit for particles sorted by pic_tile_keys
    (FP32 only); float64 J runs the FP64 path.  workspace(desc, sp, kind, device):
    where the scratch of a deposit in any order comes from."""
    f64 = is_f64(J3[0])
    raw = raw_direct_current(J3, current_filter, scratch)
    N.call(N.op("pic_zero_fields", f64), desc, N.p3(raw), stream)
    if tile and not f64:
        N.call("pic_deposit_direct_tiled", desc, sp, pp, N.p3(raw), int(tile), N.ptr(starts), stream)
    else:
        ws = None if f64 else workspace(desc, sp, DIRECT, J3[0].device)
        if ws is not None:
            N.call("pic_deposit_direct_binned", desc, sp, pp, N.p3(raw), N.ptr(ws), ws.numel(), stream)
        else:
            N.call(N.op("pic_deposit_direct", f64), desc, sp, pp, N.p3(raw), stream)
    finish_direct_current(desc, raw, J3, current_filter, stream)


def finish_direct_current(desc, raw, J3, current_filter, stream):
    """Fold + refresh of the raw direct deposit (raw_direct_current), then the
    optional filter into J3 (J_from_rhov.py:224-258)."""
    f64 = is_f64(J3[0])
    N.call(N.op("pic_finish_current", f64), desc, N.p3(raw), 1, stream)
    if raw is not J3:
        N.call(N.op("pic_filter_refresh", f64), desc, N.p3(raw), N.p3(J3), int(current_filter == "bilinear"),
               float(desc.alpha), 1, 0, stream)


def J_from_rhov(particles, species_config, J, static_parameters, dynamic_parameters):
    desc = make_desc(static_parameters, dynamic_parameters)
    xp, up, act = particle_planes(particles)
    sp = make_species(species_config, xp[0].shape[1])
    templ = [as_field3(c, "J") for c in J]
    check_fields(desc, *templ, dtype=xp[0].dtype)
    out = [t.new_empty(t.shape) for t in templ]
    deposit_direct_into(desc, sp, pic_particles(xp, up, act), out, static_parameters.current_filter,
                        N.stream_handle())
    return tuple(like_input(o, t) for o, t in zip(out, J))
