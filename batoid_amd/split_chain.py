"""traceSplit's ray sets as chains, one launch for all that were turned back
equally often.

Between two turns back a set of traceSplit (batoid/optic.py:1184-1282) meets
Interface after Interface; the reflected part of each split starts another
set.  With constant coatings which sets exist is known before any ray is
traced: every set carries a flux bound (see CompoundOptic._flux_bound), and a
set whose bound is below the threshold holds no ray that is kept.  So the
work queue runs here first on names and bounds alone, in the reference's
order, and then each set runs through its whole chain of Interfaces in one
pass (bt_split_chains), its reflected parts going to their own buffers.

For 998,388 rays through the twelve-interface telescope with 2 % reflective
glass (44 paths out) three launches take the place of 279 of one Interface
each, 36 us apiece (132 B a ray and Interface of traffic): a call takes 7.3
instead of 12.0 ms, of which the chains are 4.7 (FP64 issue), the copies out
0.8; for 10,368 rays, where the launches' host side was the time, 2.2 instead
of 6.1 ms."""
import ctypes

from . import _lib, _device
from .coordTransform import CoordTransform
from .rayVector import RayVector


class _Set:
    """A ray set: the steps of its chain as (interface, reversed, reflected
    set or None), where it started (None: the caller's own set), and whether
    the filter applies to it before its first step."""
    __slots__ = ("steps", "rays", "start", "leaves", "first", "filtered")

    def __init__(self, start):
        self.steps, self.start = [], start
        self.rays, self.leaves, self.first = None, False, 0
        self.filtered = start is not None


class _Token:
    """A set at one point of its way: the set, its flux bound and its path."""
    __slots__ = ("set", "bound", "path")

    def __init__(self, set_, bound, path):
        self.set, self.bound, self.path = set_, bound, path


def supported(optic):
    """Whether every item is of a kind whose split is known here (the
    package's own classes, not subclasses that may change it)."""
    from .optic import (CompoundOptic, Lens, RefractiveInterface, Mirror, Detector, Baffle)
    if optic.skip:
        return type(optic) in (CompoundOptic, Lens, RefractiveInterface, Mirror, Detector, Baffle)
    if type(optic) in (CompoundOptic, Lens):
        return all(supported(item) for item in optic.items)
    return type(optic) in (RefractiveInterface, Mirror, Detector, Baffle)


def _leaf(item, token, reverse, minFlux, sets):
    """Interface.traceSplit on a token: (forward, back) tokens."""
    from .optic import Mirror, Baffle, Detector
    path = token.path + [item.name]
    chain = token.set
    if type(item) in (Mirror, Baffle):
        chain.steps.append((item, reverse, None))
        on = _Token(chain, token.bound, path)
        return ([], [on]) if reverse else ([on], [])
    if type(item) is Detector:
        assert not reverse
    ft, fr = item._split_fractions(reverse)
    back = None
    if token.bound * abs(fr) >= minFlux:
        split = _Set(item)
        sets.append(split)
        back = _Token(split, token.bound * abs(fr), path)
    chain.steps.append((item, reverse, back.set if back else None))
    on = [_Token(chain, token.bound * abs(ft), path)]
    backs = [back] if back else []
    return (backs, on) if reverse else (on, backs)


def _walk(optic, inputs, minFlux, sets):
    """CompoundOptic._split_deferred on tokens: per input, the tokens leaving
    forward and back, in the reference's order."""
    last = len(optic.items) - 1
    work = [(k, (), tok, rev, last if rev else 0) for k, (tok, rev) in enumerate(inputs)]
    outs = [([], []) for _ in inputs]
    while work:
        groups = {}
        for w in work:
            groups.setdefault(w[4], []).append(w)
        work = []
        for index in sorted(groups):
            entries = groups[index]
            item = optic.items[index]
            if item.skip:
                results = [([], [w[2]]) if w[3] else ([w[2]], []) for w in entries]
                for w in entries:            # the filter follows a skipped item too
                    w[2].set.filtered |= not w[2].set.steps
            elif hasattr(item, 'items'):
                results = _walk(item, [(w[2], w[3]) for w in entries], minFlux, sets)
            else:
                results = [_leaf(item, w[2], w[3], minFlux, sets) for w in entries]
            for (k, key, _, _, _), sides in zip(entries, results):
                pushed = seq = 0
                for side, toks in enumerate(sides):
                    leaves = index == (0 if side else last)
                    for tok in toks:
                        if not tok.bound >= minFlux:
                            continue
                        if leaves:
                            outs[k][side].append(((key, seq), tok))
                            seq += 1
                        else:
                            work.append((k, key + (-pushed,), tok, side == 1,
                                         index - 1 if side else index + 1))
                            pushed += 1
    return [tuple([t for _, t in sorted(lst, key=lambda e: e[0])] for lst in o) for o in outs]


def _record(item, reverse, frame):
    """bt_chain_step of one step (without its split buffer)."""
    from .optic import Mirror, Baffle
    st = _lib.BtChainStep()
    st.surface = item.surface._dev.ptr().value
    if item.obscuration is not None:
        dev = item.obscuration._dev
        st.obsc, st.obsc_len = dev.ptr().value, dev.count
    st.dr[:], st.drot[:] = frame
    if type(item) is Mirror:
        st.action = _lib.ACT_REFLECT
    elif type(item) is Baffle:
        st.action = _lib.ACT_INTERSECT
    else:
        st.action = _lib.ACT_SPLIT
        m2 = item.inMedium if reverse else item.outMedium
        st.medium = m2._dev.ptr().value
        st.transmissivity, st.reflectivity = (float(f) for f in item._split_fractions(reverse))
    return st


def _kinds(steps):
    surfaces = [item.surface for item, _, _ in steps]
    if all(s._analytic for s in surfaces):
        return _lib.PLAN_ANALYTIC
    from .plan import _has_nested_sum
    return 0 if any(_has_nested_sum(s._records()[0]) for s in surfaces) else _lib.PLAN_FLAT_SUMS


def trace_split(optic, rv, reverse, minFlux, bound):
    """CompoundOptic.traceSplit of ``rv`` (whose largest kept |flux| is
    ``bound``): (forward, back) lists of RayVectors.  ``rv`` is left as the
    set that was never turned back, its dropped rays where they were."""
    from .global_vars import _batoid_niter
    root = _Set(None)
    root.rays = rv
    sets = [root]
    path = list(getattr(rv, 'path', []))
    (forward, back), = _walk(optic, [(_Token(root, bound, path), reverse)], minFlux, sets)
    leaving = forward + back
    for tok in leaving:
        tok.set.leaves = True
    for s in sets[1:]:
        if not s.leaves:                 # a chain that ends unseen: up to its last split
            while s.steps and s.steps[-1][2] is None:
                s.steps.pop()
    # a set that nothing comes of is not written (a set's reflected parts stand
    # behind it in the list)
    live = set()
    for s in reversed(sets):
        ok = s.leaves
        for k, (item, rev, split) in enumerate(s.steps):
            if split in live:
                ok = True
            else:
                s.steps[k] = (item, rev, None)
        if ok:
            live.add(s)
    rv.path = path + [item.name for item, _, _ in root.steps]
    frames, records, kinds = {}, {}, {}
    n = len(rv)
    # sets by generation (how often they were turned back) and kernel: those of
    # one group are independent of each other
    recs, generations = [], [[root]]
    for generation in generations:
        nexts = []
        for s in generation:
            prev, cs = s.start, rv.coordSys if s.start is None else s.start.coordSys
            s.first = len(recs)
            for item, rev, split in s.steps:
                key = (id(prev), id(item))
                if key not in frames:
                    ct = CoordTransform(cs, item.coordSys)
                    frames[key] = (tuple(ct.dr.tolist()), tuple(ct.drot.ravel().tolist()))
                if (key, rev) not in records:
                    records[key, rev] = bytes(_record(item, rev, frames[key]))
                st = _lib.BtChainStep.from_buffer_copy(records[key, rev])
                if split is not None:
                    split.rays = RayVector._empty(n, item.coordSys)
                    st.split = split.rays._rays
                    nexts.append(split)
                recs.append(st)
                prev, cs = item, item.coordSys
        if nexts:
            generations.append(nexts)
    steps = _device.upload_bytes(_lib.struct_array_bytes(recs))
    groups, chains = [], []              # (first chain, count, kernel) of each launch
    for generation in generations:
        by_kinds = {}
        for s in generation:
            surfs = tuple(id(item.surface) for item, _, _ in s.steps)
            if surfs not in kinds:
                kinds[surfs] = _kinds(s.steps)
            by_kinds.setdefault(kinds[surfs], []).append(s)
        for k, group in by_kinds.items():
            for at in range(0, len(group), 65535):
                part = group[at:at + 65535]
                groups.append((len(chains), len(part), k))
                for s in part:
                    flags = _lib.CHAIN_FILTERED if s.filtered else 0
                    if s is root:
                        flags |= _lib.CHAIN_KEEP if s.filtered else 0
                    elif not s.leaves:
                        flags |= _lib.CHAIN_NO_OUTPUT
                    chains.append(_lib.BtChain(
                        steps.data_ptr() + s.first * ctypes.sizeof(_lib.BtChainStep),
                        len(s.steps), flags, s.rays._rays))
    table = _device.upload_bytes(_lib.struct_array_bytes(chains))
    size = ctypes.sizeof(_lib.BtChain)
    for at, count, k in groups:
        _lib.call("bt_split_chains", table.data_ptr() + at * size, count, n, float(minFlux),
                  _batoid_niter, k, _device.stream())
    for s in sum(generations, []):
        if s.steps:
            s.rays.coordSys = s.steps[-1][0].coordSys
    outs = ([], [])
    if leaving:
        sel = RayVector._count_select([t.set.rays for t in leaving], minFlux)
        counts = sel.counts.tolist()
        for j, (t, out) in enumerate(zip(leaving, sel.scatter_all(counts))):
            if counts[j]:
                out.path = t.path
                outs[0 if j < len(forward) else 1].append(out)
    return outs
