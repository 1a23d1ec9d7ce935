"""Argument and failure handling of the C ABI on a GPU: capacity changes that
would cut live records, allocations that fail, checkpoint blocks that do not
fit the context, and parameters the step does not implement.  Each case
checks that the call is refused with the right code and that the context
goes on exactly as a twin that never saw the call."""
import ctypes
import re

import numpy as np
import pytest

from godar_amd import _lib
from godar_amd import generators as g
from godar_amd.params import GodarParams
from workloads import config0_params, kick, packed_box, squeeze

pytestmark = pytest.mark.gpu

STATE = ["x", "y", "u", "v", "omega", "r", "h", "theta"]


def _ctx(n, members=1, precision="fp64"):
    from godar_amd.sim import Context
    return Context(n, members, precision, record_forces=True)


def _box():
    f = kick(squeeze(packed_box(64, 3)), 1)
    return f, config0_params(f, sigmanc_crit=1e5)


def _same(a, b, ma, mb):
    fa, fb = a.floes(ma), b.floes(mb)
    for k in STATE:
        assert np.array_equal(fa[k], fb[k]), k
    assert a.pairs(ma, "contact")[0].tolist() == b.pairs(mb, "contact")[0].tolist()


def test_reserve_refuses_to_cut_live_records():
    """godar_reserve may not shrink the history list below the records a
    floe holds (the kernels walk every record up to the floe's count); a
    shrink that keeps them is applied, and the run stays bitwise equal to
    one that never changed its capacities."""
    f, p = _box()
    a, b = _ctx(f.n), _ctx(f.n)
    ma, mb = a.add_field(p, f), b.add_field(p, f)
    a.step(30)
    b.step(30)
    with pytest.raises(_lib.GodarError) as e:
        a.reserve(hist=1)
    assert e.value.code == _lib.GODAR_ERR_ARG
    live = int(re.search(r"histories (\d+)", str(e.value)).group(1))
    assert live > 1
    a.reserve(hist=live)          # down to the longest list: allowed
    a.step(25)                    # later steps may need more; capacity grows on its own
    b.step(25)
    _same(a, b, ma, mb)
    a.close()
    b.close()


def test_failed_reserve_keeps_the_context():
    """An allocation that fails (an outer list of 65,534 entries for 2^21
    floe slots needs about a terabyte) returns GODAR_ERR_NOMEM and leaves the
    context with its lists: the next steps run and equal a twin's."""
    f, p = _box()
    a, b = _ctx(1 << 21), _ctx(f.n)
    ma, mb = a.add_field(p, f), b.add_field(p, f)
    a.step(5)
    b.step(5)
    with pytest.raises(_lib.GodarError) as e:
        a.reserve(outer=65534)
    assert e.value.code == _lib.GODAR_ERR_NOMEM
    a.step(20)
    b.step(20)
    _same(a, b, ma, mb)
    a.close()
    b.close()


def test_member_add_refuses_stale_tree_cadence():
    """ntree != 1 (a neighbour tree of positions older than the step,
    stepper.f90:44-50) is refused rather than run with current positions."""
    f, p = _box()
    p.ntree = 5
    a = _ctx(f.n)
    with pytest.raises(_lib.GodarError) as e:
        a.add_field(p, f)
    assert e.value.code == _lib.GODAR_ERR_ARG
    assert "ntree" in str(e.value)
    p.ntree = 1
    a.add_field(p, f)
    a.close()


def _hist_offset(block):
    """Byte offset of the first contact-history record of a checkpoint block
    (header 40 B, parameters, 12 + 4 doubles per floe, n history counts)."""
    n = int(np.frombuffer(block[12:16], dtype=np.int32)[0])
    base = 40 + ctypes.sizeof(GodarParams)
    return base + n * (12 + 4) * 8 + n * 4, n, base


def test_restore_refuses_foreign_blocks():
    """A checkpoint whose history names a partner outside (i, n), or that was
    saved in a context of the other precision, is refused; the intact block
    restores and continues exactly."""
    f, p = _box()
    a = _ctx(f.n)
    m = a.add_field(p, f)
    a.step(30)
    block = a.checkpoint(m, p)
    a.step(10)
    off, n, base = _hist_offset(block)
    hc = np.frombuffer(block[off - 4 * n:off], dtype=np.int32)
    assert hc.sum() > 0
    for bad_j in (0, n, -1):
        bad = bytearray(block)
        bad[off:off + 4] = np.int32(bad_j).tobytes()
        b = _ctx(f.n)
        with pytest.raises(_lib.GodarError) as e:
            b.restore(bytes(bad))
        assert e.value.code == _lib.GODAR_ERR_ARG, bad_j
        b.close()
    mixed = _ctx(f.n, 1, "mixed")
    with pytest.raises(_lib.GodarError) as e:
        mixed.restore(block)
    assert e.value.code == _lib.GODAR_ERR_ARG
    assert "precision" in str(e.value)
    mixed.close()
    b = _ctx(f.n)
    mb = b.restore(block)
    b.step(10)
    _same(a, b, m, mb)
    a.close()
    b.close()


@pytest.mark.parametrize("n", [64, 40, 200])
def test_lists_of_a_member_that_left_are_not_walked(n):
    """A member that was reshaping floes leaves and another takes its slot,
    in the same storage (64 and 40 floes fit the gap) or past the others' (200):
    before the next step the totals, pair lists and statistics are those of
    the member that stayed, and the new one has none; after a step every
    member's are those it has alone."""
    f, p = _box()
    mate = kick(squeeze(packed_box(64, 11)), 4)
    pm = config0_params(mate, sigmanc_crit=1e5)
    new = kick(squeeze(packed_box(n, 7, box=2.0e4 * np.sqrt(n / 64))), 2)
    pn = config0_params(new, sigmanc_crit=1e5)
    a = _ctx(f.n + mate.n + 200, 2)
    ma, mb = a.add_field(p, f), a.add_field(pm, mate)
    for _ in range(40):
        a.step(1)
        if a.stats(ma)["seeds"] > 0:
            break
    assert a.stats(ma)["seeds"] > 0
    steps = a.tstep(mb) - 1
    kinds = ("candidate", "contact", "bond")
    of_mate = {k: [x.tolist() for x in a.pairs(mb, k)] for k in kinds}
    a.remove(ma)
    mc = a.add_field(pn, new)
    assert mc == ma
    t = a.totals()
    assert (t["candidates"], t["contacts"], t["bonds"]) == tuple(len(of_mate[k][0]) for k in kinds)
    assert set(a.stats(mc).values()) == {0}
    assert t["ridging_seeds"] == a.stats(mb)["seeds"]
    for k in kinds:
        assert a.pairs(mc, k)[0].size == 0, k
        assert [x.tolist() for x in a.pairs(mb, k)] == of_mate[k], k
    a.step(1)
    t = a.totals()
    want = dict.fromkeys(kinds, 0)
    for m, fld, par, done in ((mb, mate, pm, steps + 1), (mc, new, pn, 1)):
        b = _ctx(fld.n)
        m1 = b.add_field(par, fld)
        b.step(done)
        for k in kinds:
            pair = [x.tolist() for x in b.pairs(m1, k)]
            assert [x.tolist() for x in a.pairs(m, k)] == pair, k
            want[k] += len(pair[0])
        b.close()
    assert (t["candidates"], t["contacts"], t["bonds"]) == tuple(want[k] for k in kinds)
    a.close()


def _copy_bonds(ctx, m, f):
    i, j = ctx.pairs(m, "bond")
    s = ctx.bond_state(m)
    ctx.set_bonds(m, i, j, np.stack([s[k] for k in s], axis=1))


UNSYNCED = {
    "floes": lambda c, m, f, p: c.floes(m),
    "forces": lambda c, m, f, p: c.forces(m),
    "walls": lambda c, m, f, p: c.walls(m),
    "pairs": lambda c, m, f, p: {str(k): v for k in ("candidate", "contact", "bond")
                                 for k, v in enumerate(c.pairs(m, k))},
    "totals": lambda c, m, f, p: c.totals(),
    "stats": lambda c, m, f, p: c.stats(m),
    "tstep": lambda c, m, f, p: {"t": c.tstep(m), "all": c.tsteps()},
    "checkpoint": lambda c, m, f, p: {"block": np.frombuffer(c.checkpoint(m, p), np.uint8)},
    "remove": lambda c, m, f, p: c.remove(m) or {},
    "add": lambda c, m, f, p: {"m": c.add_field(p, f)},
    "restore": lambda c, m, f, p: {"m": c.restore(c.checkpoint(m, p))},
    "run_until": lambda c, m, f, p: c.run_until(m, 12) or {},
    "set_forcing": lambda c, m, f, p: c.set_forcing(m, -9.0, 4.0, 0.1, -0.2) or {},
    "set_bonds": lambda c, m, f, p: _copy_bonds(c, m, f) or {},
    "reserve": lambda c, m, f, p: c.reserve(hist=48) or {},
    "search": lambda c, m, f, p: c.set_search(0.05, 2, 0) or {},
    "step": lambda c, m, f, p: c.step(3) or {},
}


@pytest.mark.parametrize("k", [2, 3, 8])
@pytest.mark.parametrize("call", list(UNSYNCED))
def test_calls_after_step_async_see_its_steps(call, k):
    """With no skin every step needs a build, so the launches behind the second
    step of a run do nothing (an odd or an even number of them) until
    they are run again: every call that reads or writes state in between gives
    and leaves what it does after godar_sync."""
    f, p = _box()
    mate = kick(squeeze(packed_box(50, 11)), 4)
    pm = config0_params(mate, sigmanc_crit=1e5)
    out = []
    for sync in (True, False):
        c = _ctx(2 * f.n + mate.n, 3)
        c.set_skin(0.0)
        m, mm = c.add_field(p, f), c.add_field(pm, mate)
        c.step(1)
        c.step_async(k)
        if sync:
            c.sync()
        got = UNSYNCED[call](c, m, f, p)
        c.sync()
        c.step(5)
        out.append([got, c.tsteps()] + [c.floes(x) for x in (m, mm) if c.tsteps()[x] > 0])
        c.close()
    for a, b in zip(*out):
        if isinstance(a, dict):
            assert a.keys() == b.keys()
            for key in a:
                assert np.array_equal(a[key], b[key]), key
        else:
            assert np.array_equal(a, b)


@pytest.mark.parametrize("k", [30, 31])
def test_state_after_an_unsynced_capacity_error(k):
    """An asynchronous run that ends at a full history list: the state read
    before godar_sync is that of its last complete step, and godar_sync still
    reports the error."""
    f = kick(packed_box(64, 3), 1)      # (gaps of half a metre: no contact in the first step)
    p = config0_params(f, sigmanc_crit=1e5)
    a, b = _ctx(f.n), _ctx(f.n)
    ma, mb = a.add_field(p, f), b.add_field(p, f)
    a.reserve(hist=1)
    a.step_async(k)
    got, t = a.floes(ma), a.tstep(ma)
    with pytest.raises(_lib.GodarError) as e:
        a.sync()
    assert e.value.code == _lib.GODAR_ERR_CAPACITY and 1 < t <= k
    b.step(t - 1)
    want = b.floes(mb)
    for key in STATE:
        assert np.array_equal(got[key], want[key]), key
    a.reserve(hist=16)
    a.step(k + 1 - t)
    b.step(k + 1 - t)
    _same(a, b, ma, mb)
    a.close()
    b.close()


def test_lists_after_a_step_that_failed():
    """A step that ends at a full superset pool (the context's first, before
    any lists are built) or history list (after steps that completed) leaves
    no candidates or contacts to read until a step completes; bonds are those
    of the last complete step; the run then goes on as a twin's."""
    f, p = _box()
    p.rtree = 1.0e5                     # every floe is a candidate of every other: 63 a floe, room for 8
    a, b = _ctx(f.n), _ctx(f.n)
    ma, mb = a.add_field(p, f), b.add_field(p, f)
    a.step_async(3)
    for _ in range(2):
        t = a.totals()
        assert (t["candidates"], t["contacts"], t["bonds"]) == (0, 0, 0)
        for k in ("candidate", "contact", "bond"):
            assert a.pairs(ma, k)[0].size == 0, k
        if _ == 0:
            with pytest.raises(_lib.GodarError) as e:
                a.sync()
            assert "superset" in str(e.value)
    a.step(3)
    b.step(3)
    assert a.totals() == b.totals() and a.totals()["candidates"] > 0
    _same(a, b, ma, mb)
    a.close()
    b.close()
    f = kick(packed_box(64, 3), 1)
    p = config0_params(f, sigmanc_crit=1e5, bond_lim=50.0, bond_frac=0.1)
    a, b = _ctx(f.n), _ctx(f.n)
    ma, mb = a.add_field(p, f), b.add_field(p, f)
    a.reserve(hist=1)
    a.step_async(200)
    with pytest.raises(_lib.GodarError):
        a.sync()
    done = a.tstep(ma) - 1
    assert 0 < done < 200
    b.step(done)
    t = a.totals()
    assert (t["candidates"], t["contacts"]) == (0, 0)
    assert a.stats(ma)["candidates"] == 0 and a.pairs(ma, "contact")[0].size == 0
    assert t["bonds"] == b.totals()["bonds"] > 0
    assert [x.tolist() for x in a.pairs(ma, "bond")] == [x.tolist() for x in b.pairs(mb, "bond")]
    a.step(5)                            # (the list grows)
    b.step(5)
    assert a.totals() == b.totals() and a.totals()["contacts"] > 0
    _same(a, b, ma, mb)
    a.close()
    b.close()


def test_pair_lists_after_the_last_storage_slots_are_freed():
    """A member whose floes came first in the cell order but last in storage
    leaves: the other's pair lists, totals and list capacities are what they
    were, though its positions are past the floe slots in use now."""
    f, p = _box()                                  # (first: 64 slots and cells enough for the guest)
    mate, guest = kick(squeeze(packed_box(64, 11)), 4), kick(squeeze(packed_box(70, 12)), 5)
    pm = config0_params(mate, sigmanc_crit=1e5)
    pg = config0_params(guest, sigmanc_crit=1e5, rtree=9000.0)       # (a few large cells)
    a, b = _ctx(f.n + mate.n + guest.n, 2), _ctx(mate.n)
    ma, mm = a.add_field(p, f), a.add_field(pm, mate)
    mb = b.add_field(pm, mate)
    a.remove(ma)
    mg = a.add_field(pg, guest)
    a.step(12)
    b.step(12)
    kinds = ("candidate", "contact", "bond")
    want = [[x.tolist() for x in b.pairs(mb, k)] for k in kinds]
    assert len(want[0][0]) > 0 and len(want[1][0]) > 0
    for gone in (False, True):
        if gone:
            a.remove(mg)
            assert a.totals()["candidates"] == len(want[0][0])
            assert a.totals()["contacts"] == len(want[1][0])
            with pytest.raises(_lib.GodarError) as e:
                a.reserve(outer=1)
            assert e.value.code == _lib.GODAR_ERR_ARG
        for k, w in zip(kinds, want):
            assert [x.tolist() for x in a.pairs(mm, k)] == w, (gone, k)
        s = a.stats(mm)
        assert (s["candidates"], s["contacts"]) == (len(want[0][0]), len(want[1][0]))
    a.step(5)
    b.step(5)
    _same(a, b, mm, mb)
    a.close()
    b.close()


def _peak_rss():
    with open("/proc/self/status") as f:
        return int(re.search(r"VmHWM:\s+(\d+) kB", f.read()).group(1)) * 1024


def test_long_pair_lists_in_parts():
    """Lists longer than the staging area (524,288 pairs, 43,690 bonds) come in
    parts: a lattice's candidates, and the bonds and contacts of its
    neighbours, are those a tree search gives, and the candidate list takes
    host memory for 8 bytes a pair, not for a bond's state."""
    from scipy.spatial import cKDTree
    n, side = 24000, 155
    rng = np.random.default_rng(8)
    f = g.config0_member(51, 100)
    at = rng.permutation(side * side)[:n]
    f.x, f.y = 2000.0 * (at % side) + 1000.0, 2000.0 * (at // side) + 1000.0
    f.r, f.h = 1001.0 + rng.uniform(-2, 2, n), rng.uniform(0.8, 1.2, n)
    f.theta, f.omega, f.u, f.v = np.zeros((4, n))
    f.box = 2000.0 * side
    p = config0_params(f, bond_lim=900.0, bond_frac=1.0, rtree=7500.0, ridging=0)
    ctx = _ctx(n)
    m = ctx.add_field(p, f)
    ctx.step(1)
    pq = cKDTree(np.stack([f.x, f.y], 1)).query_pairs(9000.0, output_type="ndarray")
    pq = np.sort(pq, axis=1)
    pq = pq[np.lexsort((pq[:, 1], pq[:, 0]))]
    dx, dy = f.x[pq[:, 0]] - f.x[pq[:, 1]], f.y[pq[:, 0]] - f.y[pq[:, 1]]
    d = np.sqrt(dx * dx + dy * dy)
    gap = d - (f.r[pq[:, 0]] + f.r[pq[:, 1]])
    want = {"candidate": pq[d <= f.r[pq[:, 0]] + p.rtree], "bond": pq[gap <= p.bond_lim], "contact": pq[gap < 0]}
    assert len(want["candidate"]) > 524288 and len(want["bond"]) > 43690 and len(want["contact"]) > 10000
    cnt = ctypes.c_int32()
    got = np.empty((2, len(want["candidate"])), np.int32)
    got[:] = 0
    i32 = ctypes.POINTER(ctypes.c_int32)
    before = _peak_rss()
    _lib.check(ctx.h, _lib.load().godar_get_pairs(ctx.h, m, _lib.PAIRS_CANDIDATE, got.shape[1], got[0].ctypes.data_as(i32),
                                                  got[1].ctypes.data_as(i32), ctypes.byref(cnt)))
    assert _peak_rss() - before < 24 * got.shape[1]
    assert cnt.value == got.shape[1]
    for k, w in want.items():
        assert np.array_equal(np.stack(ctx.pairs(m, k), 1), w), k
    assert np.array_equal(got.T, want["candidate"])
    assert ctx.bond_state(m)["bond"].size == len(want["bond"])
    ctx.close()


@pytest.mark.parametrize("trial", [1, 3])
def test_autotune_times_no_stage_that_steps_do_not_launch(trial):
    """The contact stage's block size is of the steps timed stage by stage
    alone: no trial steps are spent on it and it stays as set (six stages of
    three sizes each are timed, and six to eight search shapes: a skin or
    threshold that was left for a better one is priced again)."""
    f, p = _box()
    a = _ctx(f.n)
    m = a.add_field(p, f)
    a.set_stage_block(4, 128)
    a.profile(True)                      # (no launch mode to time)
    blocks = a.autotune(trial)
    assert blocks["contacts"] == 128
    shapes, rest = divmod(a.tstep(m) - 1 - (1 + 3 * trial * 6), 1 + max(4, 4 * trial))
    assert rest == 0 and 6 <= shapes <= 8
    a.close()


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
def test_block_sizes_change_between_builds(prec):
    """The work queues are laid out by the search's block size anew in every
    step, so a size that changes in the middle of a run, on steps with the
    supersets of an earlier build, changes nothing: the trajectory is that of
    the sizes left alone, for a dense member beside one that is not."""
    f, p = _box()
    dense = kick(squeeze(packed_box(300, 9, box=4.3e4)), 6)
    pd = config0_params(dense, sigmanc_crit=1e5, rtree=9000.0)
    out = []
    for sizes in ((), (128, 256, 64, 192)):
        a = _ctx(f.n + dense.n, 2, prec)
        ms = [a.add_field(p, f), a.add_field(pd, dense)]
        a.step(6)
        for k in range(4):
            if sizes:
                a.set_block(sizes[k])
            a.step(5)
        out.append([a.floes(m) for m in ms] + [a.totals()])
        a.close()
    for x, y in zip(*out):
        for k in x:
            assert np.array_equal(x[k], y[k]), k
    assert out[0][2]["contacts"] > 0


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("extra", [1, 2, 3])
def test_stopped_members_keep_their_pair_state(extra, prec):
    """A member that stops keeps the contact histories and bonds of its last
    step, however many steps the others take after it (the two buffers of the
    pair state change place every step) and whatever the lists grow to: its
    checkpoint and bonds stay what they are alone, and when it goes on it takes
    the steps it takes alone."""
    f, p = _box()
    p = config0_params(f, sigmanc_crit=1e5, bond_lim=50.0, bond_frac=0.3)
    mate = kick(squeeze(packed_box(64, 11)), 4)
    a, b = _ctx(f.n + mate.n, 2, prec), _ctx(f.n, 1, prec)
    ma, mb = a.add_field(p, f), b.add_field(p, f)
    a.add_field(config0_params(mate, sigmanc_crit=1e5), mate)
    a.run_until(ma, 10)
    a.step(10)
    b.step(10)
    block, bonds = b.checkpoint(mb, p), b.bond_state(mb)
    for step in range(3):
        assert a.checkpoint(ma, p) == block, step
        got = a.bond_state(ma)
        assert all(np.array_equal(got[k], bonds[k]) for k in bonds)
        if step == 1:
            a.reserve(hist=40, bonds=40)
        if step < 2:
            a.step(extra)
    a.run_until(ma, 0)
    a.step(7)
    b.step(7)
    assert a.tstep(ma) == 18
    _same(a, b, ma, mb)
    a.close()
    b.close()


@pytest.mark.parametrize("k", [1, 2, 5])
def test_held_up_steps_record_forces_as_launched(k):
    """Steps that a missed build held up run again with the force recording
    they were launched with, whatever it was set to since."""
    f, p = _box()
    out = []
    for sync in (True, False):
        c = _ctx(f.n)
        c.set_skin(0.0)
        m = c.add_field(p, f)
        c.step(1)
        for on, n in ((0, k), (1, 1), (0, 3), (1, k), (0, 2)):
            c.record_forces(bool(on))
            c.step_async(n)
            if sync:
                c.sync()
        out.append([c.forces(m), c.floes(m)])
        c.record_forces(True)
        c.step(1)
        out[-1] += [c.forces(m), {"t": c.tstep(m)}]
        c.close()
    for a, b in zip(*out):
        for key in a:
            assert np.array_equal(a[key], b[key]), key
