"""The M2L of an octree folded by the kernel's reflection symmetry
(``csrc/m2l_fold.hip``; reference ``sumpy/fmm.py:777-920``).

Serves the translation-class M2L of a whole traversal where every class
vector is an integer multiple of its level's box size with components of at
most 3 (any octree's list 2), for PDE-compressed expansions of orders 1..12 in
FP64 and FP32.  Other traversals, orders and operator calls on single levels
take the class-matrix contraction of :mod:`sumpy_amd.e2e`.

The plan (tiles of 16 target boxes, the sources of every (tile, vector), the
vectors of every block of tiles) is built on the GPU without a host
synchronisation but the last, and is held on the traversal; the class data of
the canonical vectors are held on the wrangler, like the class data they come
from.
"""

from __future__ import annotations

import ctypes
import math
from functools import lru_cache
from operator import is_

import numpy as np
import torch

from sumpy_amd import _capi
from sumpy_amd.expansion import m2l_device_tables
from sumpy_amd.profiling import kernel_span
from sumpy_amd.tools import as_i32

WAVES, TCOL, NVEC = 4, 16, 343  # as in the kernels
MAX_ORDER, MAX_LEVELS = 12, 32
PRECISIONS = {"fp64": 0, "fp32": 1}


#: cost of the most expensive slot, as in the kernels
MAX_SLOT_COST = 20
#: slots (of the most expensive kind) that a workgroup takes at least
MIN_SLOTS = 4


def workgroups(precision, cplx, order, cost, resident):
    """Workgroups that share slots of *cost* in all: those that the GPU holds at
    once (*resident*) with MIN_SLOTS each, since fewer leave the pipeline's start
    and the partial sums in the lead.

    In FP32 up to 6 times as many, of about 6 slots (orders up to 7: 8; complex: 2),
    in whole rounds: 1.5 rounds of 512 take 1165 us where 2 take 901.  A workgroup
    adds its products up in FP32, the workgroups' sums are added in FP64; with one
    range for each, locals were up to 2 times (order 3; 1.4 at order 10) as far from
    FP64 as the class matrices', whose tiles are split too.  This way they are nearer
    on all but single levels (0.3 to 1.04 times over orders 3-10 and 30000 to 700000
    uniform, clustered and sphere points; complex 0.4 to 1.00, order 12 up to 1.03).
    The M2L of 700000 uniform points took 473 us and takes 502 (order 6), 1067 and
    1118 (order 10), of 150000 on a sphere, complex, order 12 904 and 953."""
    g = min(resident, cost//(MIN_SLOTS*MAX_SLOT_COST))
    if precision == "fp32":
        slots = 2 if cplx else 8 if order <= 7 else 6
        more = cost//(slots*MAX_SLOT_COST)
        if more > resident:  # (a seventh of a round is not worth a whole one)
            more = min(6, max(1, math.ceil(more/resident - 1/7)))*resident
        g = max(g, more)
    return max(g, 1)


@lru_cache(maxsize=None)
def sizes(order):
    """(folded axes, row blocks, k pairs, row blocks and k pairs by parity)."""
    out = _sizes(order)
    return int(out[0]), int(out[1]), int(out[2]), out[3:11].tolist(), out[11:19].tolist()


def _sizes(order):
    out = np.zeros(41, np.int32)
    _capi.call("sumpyhip_m2l_fold_sizes", order, out.ctypes.data)
    return out


@lru_cache(maxsize=None)
def layout(order, precision):
    """(S0, S1, entries) of the class data in LDS, by precision."""
    i = 22 if precision == "fp64" else 19
    return tuple(int(v) for v in _sizes(order)[i:i + 3])


@lru_cache(maxsize=None)
def offsets(order, precision):
    """``off(m)`` of every padded row and column (0 for padding, whose
    products are multiplied by zero columns or dropped)."""
    from sumpy_amd.expansion.terms import get_terms_table
    ax = sizes(order)[0]
    s0, s1, _ = layout(order, precision)
    q = get_terms_table(order, 3, True).stored >> (np.arange(3) < ax)
    off = q @ np.array([s0, s1, 1])
    return [np.where(m >= 0, off[m], 0).astype(np.int32) for m in maps(order)[:2]]


def table_size(ax):
    """Entries of a level's class-matrix table (``table_index``)."""
    return 4**ax*7**(3 - ax)


def table_index(n, ax):
    """Table index of canonical vectors *n* (count, 3)."""
    r = np.zeros(len(n), np.int64)
    for d in range(3):
        r = 4*r + n[:, d] if d < ax else 7*r + n[:, d] + 3
    return r


def max_slots(ax):
    """Canonical list-2 vectors: not all components within 1."""
    return 4**ax*7**(3 - ax) - 2**ax*3**(3 - ax)


@lru_cache(maxsize=None)
def maps(order, compressed=True):
    """(row map, k map, parity of each stored multi-index): the stored
    coefficient of every padded row and column, -1 for padding, parity classes
    in order."""
    from sumpy_amd.expansion.terms import get_terms_table
    ax, _, _, nrb, nkp = sizes(order)
    st = get_terms_table(order, 3, compressed).stored
    par = (st[:, 0] & 1) | (st[:, 1] & 1) << 1 | (st[:, 2] & 1) << 2
    cls = par & ((1 << ax) - 1)
    out = []
    for blocks, size in ((nrb, 16), (nkp, 8)):
        parts = []
        for p in range(1 << ax):
            idx = np.nonzero(cls == p)[0]
            m = np.full(blocks[p]*size, -1, np.int64)
            m[:len(idx)] = idx
            parts.append(m)
        out.append(np.concatenate(parts).astype(np.int32))
    return out[0], out[1], par.astype(np.int32)


@lru_cache(maxsize=None)
def _device_maps(order, precision, device):
    return tuple(torch.from_numpy(a).to(device)
                 for a in (*maps(order)[:2], *offsets(order, precision)))


@lru_cache(maxsize=None)
def _max_workgroups(precision, cplx, order, device):
    out = np.zeros(1, np.int32)
    with torch.cuda.device(device):
        _capi.call("sumpyhip_m2l_fold_max_wg", precision, cplx, order, out.ctypes.data)
    return int(out[0])


def _class_vectors(wrangler):
    """Integer vectors (nclasses, 3) of the translation classes in box sizes of
    their level, or None where they are not such."""
    got = wrangler._memo.get("m2l_fold_vectors", False)
    if got is not False:
        return got
    ls = np.asarray(wrangler._class_level_starts).astype(np.int64)
    v = wrangler.translation_classes_data \
        .from_sep_siblings_translation_class_to_distance_vector.cpu().numpy()
    lev = np.repeat(np.arange(len(ls) - 1), np.diff(ls))
    x = (v[:, :len(lev)]/(wrangler.tree.root_extent*2.0**-lev)).T
    n = np.rint(x)
    ok = x.shape[1] == 3 and (np.abs(n) <= 3).all() and (np.abs(n) > 1).any(axis=1).all() \
        and (np.abs(x - n) < 1e-10).all()
    got = n.astype(np.int64) if ok else None
    wrangler._memo["m2l_fold_vectors"] = got
    return got


def usable(wrangler, order):
    """Whether the M2L of *order* on this wrangler's octree can be folded."""
    ti = wrangler.tree_indep
    prec = ti.m2l_translation.precision
    if not (1 <= order <= MAX_ORDER) or prec not in PRECISIONS:
        return False
    if (np.dtype(wrangler.dtype).kind == "c") != ti.get_base_kernel().is_complex_valued:
        return False  # the class data have the kernel's planes
    mpole, local = ti.multipole_expansion(order), ti.local_expansion(order)
    n = (order + 1)**2
    if len(local) != n or len(mpole) != n or not (mpole.compressed and local.compressed):
        return False
    planes = 2 if np.dtype(wrangler.dtype).kind == "c" else 1
    row = sizes(order)[2]*8*planes*(8 if prec == "fp64" else 4)
    return wrangler.tree.nboxes*row < 2**31


def takes(wrangler, mpole_exps):
    """Whether the kernels may read *mpole_exps* as the rows of all boxes: the
    wrangler's dtype, every value in place (no lazily conjugated or negated view,
    whose memory holds other values)."""
    m = mpole_exps
    dtype = torch.complex128 if np.dtype(wrangler.dtype).kind == "c" else torch.float64
    return (m.dtype == dtype and m.dim() == 1 and m.is_contiguous()
            and not (m.is_conj() or m.is_neg())
            and m.numel() == int(wrangler.multipole_expansions_level_starts()[-1]))


def runs(wrangler, starts, target_boxes, src_box_starts, src_box_lists):
    """[(order, levels)] of the folded M2L of a pass: the runs of consecutive
    levels of one order; None where the pass needs the general contraction
    (other lists than the traversal's own or a part of a level's target boxes,
    not an octree in 3D, other expansions)."""
    trav, tree = wrangler.traversal, wrangler.tree
    if not (wrangler.supports_translation_classes and tree.dimensions == 3
            and wrangler.tree_indep.m2l_translation.use_preprocessing
            and tree.nlevels <= MAX_LEVELS):
        return None
    for ary, name in ((target_boxes, "target_or_target_parent_boxes"),
                      (src_box_starts, "from_sep_siblings_starts"),
                      (src_box_lists, "from_sep_siblings_lists")):
        if ary is not getattr(trav, name, None):
            return None
    own = trav.host["level_start_target_or_target_parent_box_nrs"]
    classes = wrangler.m2l_translation_class_level_start_box_nrs()
    out, ok = [], set()
    for lev in range(tree.nlevels):
        if starts[lev] == starts[lev + 1] or classes[lev] == classes[lev + 1]:
            continue
        if starts is not own and (starts[lev] != own[lev] or starts[lev + 1] != own[lev + 1]):
            return None
        order = wrangler.level_orders[lev]
        if order not in ok and not usable(wrangler, order):
            return None
        ok.add(order)
        if out and out[-1][0] == order and out[-1][1][-1] == lev - 1:
            out[-1][1].append(lev)
        else:
            out.append((order, [lev]))
    return out if _class_vectors(wrangler) is not None else None


def _plan(actx, wrangler, levels, ax):
    trav, tree = wrangler.traversal, wrangler.tree
    tcd = wrangler.translation_classes_data
    plans = trav.__dict__.setdefault("_m2l_fold_plans", [])
    # the arrays that the plan is made from, as they are now: a plan does not
    # outlive their replacement or a change in place
    arrays = (trav.target_or_target_parent_boxes, trav.from_sep_siblings_starts,
              trav.from_sep_siblings_lists, tcd.from_sep_siblings_translation_classes,
              tree.box_centers, tree.box_levels)
    versions = [a._version for a in arrays]
    for p in plans:
        if p["tcd"] is tcd and p["key"] == (levels, ax):
            if p["versions"] == versions and all(map(is_, p["arrays"], arrays)):
                return p
            plans.remove(p)
            break
    dev = actx.device
    lst = np.asarray(trav.host["level_start_target_or_target_parent_box_nrs"]).astype(np.int64)
    lev_slot = np.full(tree.nlevels, -1, np.int32)
    lev_slot[list(levels)] = np.arange(len(levels))
    # tiles per level: at most one ragged tile per octant
    nt = np.diff(lst)[list(levels)]
    nblocks = (nt//TCOL + np.minimum(nt, 8) + WAVES - 1)//WAVES
    base = np.concatenate([[0], np.cumsum(nblocks)]).astype(np.int32)
    nb, ntiles = int(base[-1]), int(base[-1])*WAVES
    vecs = _class_vectors(wrangler)
    code = (vecs[:, 0] + 3)*49 + (vecs[:, 1] + 3)*7 + vecs[:, 2] + 3

    def i32(a):
        return torch.from_numpy(np.ascontiguousarray(a, np.int32)).to(dev)

    totp, starts, lists, classes, box_levels = map(as_i32, (*arrays[:4], arrays[5]))
    centers = tree.box_centers.contiguous()
    code_d = i32(code)
    n = int(totp.numel())
    keys = torch.empty(n, dtype=torch.int32, device=dev)
    geo = (ax, tree.nlevels, lev_slot.ctypes.data, len(levels), base.ctypes.data,
           float(tree.root_extent), tree.nboxes, _capi.ptr(box_levels), _capi.ptr(centers), n,
           _capi.ptr(totp), _capi.ptr(starts))
    _capi.call("sumpyhip_m2l_fold_keys", *geo, _capi.ptr(keys), actx.stream_handle)
    skeys, order = torch.sort(keys, stable=True)
    nkeys = 8*len(levels)
    key_start = torch.searchsorted(skeys, torch.arange(nkeys + 1, dtype=torch.int32, device=dev))
    tile_target = torch.full((ntiles*TCOL,), -1, dtype=torch.int32, device=dev)
    src = torch.full((ntiles*NVEC*TCOL,), -1, dtype=torch.int32, device=dev)
    present = torch.zeros(nb*NVEC, dtype=torch.int32, device=dev)
    tgt_pos = torch.empty(n, dtype=torch.int32, device=dev)
    ms = max_slots(ax)
    slots, costs = torch.empty((2, nb*ms), dtype=torch.int32, device=dev)
    type_end = torch.empty(nb*8, dtype=torch.int32, device=dev)
    bcost = torch.empty(nb, dtype=torch.int64, device=dev)
    _capi.call("sumpyhip_m2l_fold_plan", *geo, _capi.ptr(lists), _capi.ptr(classes),
               _capi.ptr(code_d), _capi.ptr(skeys), _capi.ptr(order), _capi.ptr(key_start),
               _capi.ptr(tile_target), _capi.ptr(tgt_pos), _capi.ptr(src), _capi.ptr(present),
               ms, _capi.ptr(slots), _capi.ptr(costs), _capi.ptr(type_end), _capi.ptr(bcost),
               actx.stream_handle)
    block_cost = torch.zeros(nb + 1, dtype=torch.int64, device=dev)
    torch.cumsum(bcost, 0, out=block_cost[1:])
    plan = dict(tcd=tcd, key=(levels, ax), arrays=arrays, versions=versions, nblocks=nb,
                maxslots=ms, tile_target=tile_target, src=src, slots=slots, costs=costs,
                type_end=type_end, block_cost=block_cost,
                block_level=i32(np.repeat(np.arange(len(levels)), nblocks)))
    # (waits for the plan: passes on other streams may use it at once)
    plan["cost"] = int(block_cost[-1])
    plans.append(plan)
    return plan


def _table(actx, wrangler, order, levels):
    """The class data of the canonical vectors of *levels* in the kernel's
    layout, from the wrangler's class data (once per wrangler)."""
    key = ("m2l_fold_table", order, levels)
    got = wrangler._memo.get(key)
    if got is not None:
        return got
    ti = wrangler.tree_indep
    prec = ti.m2l_translation.precision
    cplx = np.dtype(wrangler.dtype).kind == "c"
    ax = sizes(order)[0]
    nt = table_size(ax)
    m = m2l_device_tables(order, order, True, str(actx.device))
    ls = np.asarray(wrangler._class_level_starts).astype(np.int64)
    vecs = _class_vectors(wrangler)
    stride = nt*layout(order, prec)[2]*(2 if cplx else 1)
    shape = _capi.np_i32(m["shape"])
    table = torch.empty(len(levels)*stride, device=actx.device,
                        dtype=torch.float64 if prec == "fp64" else torch.float32)
    data = wrangler.multipole_to_local_precompute()
    rep = np.full((len(levels), nt), -1, np.int32)
    sgn = np.zeros((len(levels), nt), np.int32)
    for s, lev in enumerate(levels):
        v = vecs[ls[lev]:ls[lev + 1]]
        c = v.copy()
        c[:, :ax] = np.abs(c[:, :ax])
        idx = table_index(c, ax)
        rep[s, idx] = np.arange(len(v))
        neg = (v < 0) & (np.arange(3) < ax)
        sgn[s, idx] = neg @ np.array([1, 2, 4])
    reps = torch.from_numpy(np.stack([rep, sgn])).to(actx.device)
    for s, lev in enumerate(levels):
        _capi.call("sumpyhip_m2l_fold_table", PRECISIONS[prec], int(cplx), order, nt,
                   shape.ctypes.data, _capi.ptr(reps[0, s]), _capi.ptr(reps[1, s]), _capi.ptr(data[lev]),
                   _capi.ptr(table[s*stride:]), actx.stream_handle)
    torch.cuda.current_stream(actx.device).synchronize()
    got = (table, stride)
    wrangler._memo[key] = got
    return got


def apply(actx, wrangler, order, levels, mpole_exps, local_exps):
    """M2L of *levels* (all of *order*): overwrites the local rows of the
    target boxes with a list 2."""
    ti = wrangler.tree_indep
    prec = ti.m2l_translation.precision
    pid = PRECISIONS[prec]
    cplx = np.dtype(wrangler.dtype).kind == "c"
    planes = 2 if cplx else 1
    ax, nrb, nkp, _, _ = sizes(order)
    levels = tuple(levels)
    plan = _plan(actx, wrangler, levels, ax)
    table, stride = _table(actx, wrangler, order, levels)
    row, kmap, off_t, off_s = _device_maps(order, prec, str(actx.device))
    dt = torch.float64 if prec == "fp64" else torch.float32
    # expansions of one order everywhere are one row per tree box; otherwise
    # the levels' rows are addressed from their first box
    b0 = int(wrangler.tree_level_start_box_nrs[levels[0]])
    b1 = int(wrangler.tree_level_start_box_nrs[levels[-1] + 1])
    nboxes, n = b1 - b0, (order + 1)**2
    msrc = mpole_exps[int(wrangler.multipole_expansions_level_starts()[levels[0]]):]
    lout = local_exps[int(wrangler.local_expansions_level_starts()[levels[0]]):]
    packed = torch.empty(nboxes*nkp*8*planes, dtype=dt, device=actx.device)
    _capi.call("sumpyhip_m2l_fold_pack", pid, int(cplx), nboxes, n, nkp*8, _capi.ptr(msrc),
               _capi.ptr(kmap), _capi.ptr(packed), actx.stream_handle)
    wg = workgroups(prec, cplx, order, plan["cost"],
                    _max_workgroups(pid, int(cplx), order, str(actx.device)))
    partial = torch.empty(2*wg*WAVES*planes*nrb*256, dtype=dt, device=actx.device)
    # of the dense products that the fold replaces
    flops = 2.0*n*n*planes**2*int(wrangler.traversal.from_sep_siblings_lists.numel())
    with kernel_span(f"m2l_fold_{prec}", flops):
        _capi.call("sumpyhip_m2l_fold_apply", pid, int(cplx), order, plan["nblocks"],
                   plan["maxslots"], b0, nboxes, n,
                   _capi.ptr(plan["tile_target"]), _capi.ptr(plan["src"]),
                   _capi.ptr(plan["slots"]), _capi.ptr(plan["costs"]),
                   _capi.ptr(plan["type_end"]), _capi.ptr(plan["block_level"]),
                   _capi.ptr(plan["block_cost"]), _capi.ptr(row), _capi.ptr(off_t),
                   _capi.ptr(off_s), _capi.ptr(packed), _capi.ptr(table), stride, wg,
                   1, _capi.ptr(partial), _capi.ptr(lout), actx.stream_handle)


__all__ = ["apply", "runs"]
