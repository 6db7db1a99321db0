"""Which dispatches may run side by side (te_plan_batches): never two of which
one writes a word that the other one reads or writes, wherever the words lie
(word 0 included), whatever the parameter is (field, profile, metric, flag) and
however long a merged copy is.  The operands that the rule knows of each kernel
are held against the reference's recorded signatures; on the GPU a tape of
dependent dispatches is held against the oracle, word for word."""
import json
import os

import numpy as np
import pytest

import oracle_lib as ol
import tapeplan
import te_host

NX, NY, NZ, SJ, SK = 9, 7, 12, 16, 14
FIELD = SJ * SK * (NZ + 1)
FLAGS = 40 * 2 * FIELD  # parameter words above the fields
DIMS = FLAGS
WORDS = FLAGS + 4096


def signatures():
    P = {}
    for preset in tapeplan.PRESETS:
        P.update(json.load(open(os.path.join(tapeplan.GOLDEN, preset, "kernel_params.json"))))
    return P


# kernels of the pointwise batches with a recorded signature, and the recorded
# parameters that the kernel here has no use for
POINTWISE = {
    "rayleigh_damping": (), "turb_rho_faces": (), "turb_def_centers": (), "turb_def_faces": (), "turb_def_assemble": (),
    "turb_nm": (), "turb_km_kh": (), "turb_km_kh_xy": (), "turb_dissipative_heating": (), "turb_gettau": (30,),
    "tke_sources": (), "turb_scalar_flux_h": (), "tke_flux_h": (), "turb_openbc_flux": (),
    "update_diagnostics_moist": (), "stage_tendency_reset": (), "stage_state_reset": (), "build_sadv": (),
    "ppx_finish_xy": (), "diabatic_rates": (), "pressure_tendency": (), "update_rho_prs": (), "tke_advance_xy": (),
    "rk_update_xy": (1,)}
# column sweeps: the elimination coefficients stay in registers, TKE's fluxes are read
SWEEPS = {"turb_u_tendency_lds": (12, 13), "turb_v_tendency_lds": (12, 13), "turb_w_tendency_lds": (11, 12),
          "turb_scalar_vert_implicit_lds": (11, 12), "tke_transport_lds": (9, 10)}


class Tape:
    """A program over slots of 2 fields' words each and single parameter words."""

    def __init__(self):
        self.M = np.zeros(WORDS, np.uint32)
        self.M[DIMS: DIMS + 5] = NX, NY, NZ, SJ, SK
        self.M[DIMS + 5: DIMS + 8] = np.float32(1e-3).view(np.uint32)
        self.names, self.args, self.top = [], [], DIMS + 64

    def words(self, *values):
        o = self.top
        self.M[o: o + len(values)] = np.array(values, np.int32).view(np.uint32)
        self.top += 8
        return o

    def op(self, name, bind, grid=(NX, NY, NZ)):
        a = np.zeros(64, np.uint32)
        a[:3] = grid
        a[4] = DIMS
        for q, off in bind.items():
            a[4 + q] = off
        self.names.append(name)
        self.args.append(a)

    def copy(self, src, dst, n=FIELD):
        self.op("copy_fields", {1: src, 5: dst, 9: self.words(1)}, (n, 1, 1))

    def batches(self):
        return te_host.plan_batches(self.M, self.names, np.array(self.args)).tolist()


def slot(n):
    return (n + 1) * 2 * FIELD


def recorded(name):
    base = name[:-3] if name.endswith("_xy") else name[:-4] if name.endswith("_lds") else name
    return [(q, kind, bool(w)) for q, kind, w in signatures()[base] if q > 0]


@pytest.mark.parametrize("at", [0, slot(35)], ids=["word0", "elsewhere"])
@pytest.mark.parametrize("name", sorted(POINTWISE))
def test_pointwise_operands_are_known(name, at):
    """A copy next to the kernel, into or out of each of its parameters."""
    params = [p for p in recorded(name) if p[0] not in POINTWISE[name]]
    for q, kind, written in params:
        def tape(order):
            t = Tape()
            bind = {i: (t.words(0) if k == "ref" else slot(i)) for i, k, _ in recorded(name)}
            bind[q] = at
            for o in order:
                if o == "k":
                    t.op(name, bind)
                else:
                    t.copy(*((slot(36), at) if o == "into" else (at, slot(36))))
            return t.batches()
        assert tape(("into", "k")) == [1, 1], (q, "copied into before")
        assert tape(("k", "into")) == [1, 1], (q, "copied into after")
        out = tape(("out", "k"))
        assert out == ([1, 1] if written else [2, 0]), (q, "copied from")


@pytest.mark.parametrize("at", [0, slot(35)], ids=["word0", "elsewhere"])
@pytest.mark.parametrize("name", sorted(SWEEPS))
def test_sweep_operands_are_known(name, at):
    """A scalar's sweep next to the kernel: its tendency, or the scalar, is one
    of the kernel's parameters."""
    scalar = {i: (slot(20) if k == "ptr" else 0) for i, k, _ in recorded("turb_scalar_vert_implicit_lds")}
    for q, kind, written in recorded(name):
        if q in SWEEPS[name]:
            continue
        written = written and not (name == "tke_transport_lds" and q in (11, 12))
        def tape(scalar_q):
            t = Tape()
            other = dict(scalar)
            for i, k, _ in recorded("turb_scalar_vert_implicit_lds"):
                other[i] = t.words(0) if k == "ref" else slot(20)
            other[13] = slot(21)
            other[scalar_q] = at
            bind = {i: (t.words(0) if k == "ref" else slot(i if i < 19 else 22)) for i, k, _ in recorded(name)}
            bind[q] = at
            t.op("turb_scalar_vert_implicit_lds", other, (NX, NY, 1))
            t.op(name, bind, (NX, NY, 1))
            return t.batches()
        assert tape(13) == [1, 1], q
        assert tape(1) == ([1, 1] if written else [2, 0]), q


@pytest.mark.parametrize("at", [0, slot(35)], ids=["word0", "elsewhere"])
def test_advections_of_one_field(at):
    """Two advections, of which the second advects what the first one writes
    (its tendency, or the field that its chain updates), in both orders."""
    def tape(first, chain, order=1):
        t = Tape()
        base = {2: slot(0), 4: slot(1), 6: slot(2), 13: slot(3), 14: slot(4), 1: t.words(1), 3: t.words(0),
                5: t.words(0), 12: t.words(0), 17: t.words(0, 0), 20: t.words(0), 21: t.words(0), 30: slot(5)}
        base.update({i: slot(6) for i in (7, 8, 9, 10, 15, 16)})
        one = dict(base)
        one.update({2: slot(7), 11: slot(8), 32: t.words(chain), 39: slot(9), 40: slot(10), 41: t.words(0)})
        one.update(first)
        two = dict(base)
        two.update({2: at, 11: slot(11), 32: t.words(0)})
        for b in (one, two)[::order]:
            t.op("adv_fused", b)
        return t.batches()
    assert tape({}, 0) == [2, 0]
    for order in (1, -1):
        assert tape({11: at}, 0, order) == [1, 1]
        assert tape({40: at}, 8, order) == [1, 1]
        assert tape({11: at}, 8, order) == [2, 0]  # a chained update leaves the tendency


def test_copies_reach_as_far_as_they_copy():
    """A copy of three slots and a read of the third; one of a field's tail."""
    t = Tape()
    t.copy(slot(0), slot(10), 3 * 2 * FIELD)
    t.op("build_sadv", {1: slot(20), 2: slot(12), 3: slot(21)}, (SJ, SK, NZ + 1))
    assert t.batches() == [1, 1]
    for off, together in ((FIELD - 1, False), (FIELD, True)):
        t = Tape()
        t.copy(slot(0), slot(10) + off, 8)
        t.op("build_sadv", {1: slot(20), 2: slot(10), 3: slot(21)}, (SJ, SK, NZ + 1))
        assert t.batches() == ([2, 0] if together else [1, 1])


def test_copies_into_a_profile():
    """theta's base profile is copied in before the dispatch that adds it: the
    words of its levels, not the one past them."""
    for off, together in ((NZ, False), (NZ + 1, True)):
        t = Tape()
        t.copy(slot(0), slot(20) + off, 4)
        t.op("build_sadv", {1: slot(20), 2: slot(12), 3: slot(21)}, (SJ, SK, NZ + 1))
        assert t.batches() == ([2, 0] if together else [1, 1])


@pytest.mark.parametrize("kw", [dict(tke=1, initial_tke=3), dict(species=7), dict(open_x=1, open_y=1)])
def test_the_step_still_groups_its_dispatches(kw):
    run = te_host.Run(te_host.config(nx=12, ny=10, nz=16, **kw), encode_only=True)
    names, A = run.program()
    b = te_host.plan_batches(run.read(0, run.mem_words), names, A)
    assert b.sum() == len(names) and (b > 1).sum() >= 8
    run.close()


def dependent_tape(at):
    """rf written (at word `at`) and read; a field copied with two others and
    read; a profile copied and read."""
    rng = np.random.default_rng(5)
    t = Tape()
    t.M[:FLAGS] = rng.uniform(0.5, 1.5, FLAGS).astype(np.float32).view(np.uint32)
    whole = (SJ, SK, NZ + 1)
    w = t.words(*np.array([0.9, 0.3, -0.2], np.float32).view(np.int32))
    t.op("turb_rho_faces", {1: slot(0), 2: slot(1), 3: slot(2), 4: slot(3), 5: at, 6: w, 7: w}, (NX + 4, NY + 4, NZ + 1))
    t.op("turb_def_faces", {1: slot(4), 2: slot(5), 3: slot(6), 4: at, 5: slot(7), 6: slot(8), 7: slot(9), 30: slot(10)},
         (NX + 2, NY + 2, NZ + 1))
    t.copy(slot(11), slot(14), 3 * 2 * FIELD)
    t.op("build_sadv", {1: slot(17), 2: slot(16), 3: slot(18)}, whole)
    t.copy(slot(19), slot(20), NZ + 1)
    t.op("build_sadv", {1: slot(20), 2: slot(21), 3: slot(22)}, whole)
    return t


@pytest.mark.gpu
@pytest.mark.parametrize("at", [0, slot(35)], ids=["word0", "elsewhere"])
def test_dependent_tape_bit_exact(gpu, at):
    t = dependent_tape(at)
    print("dependent tape", at, flush=True)
    A = np.array(t.args)
    r = te_host.Replayer(WORDS, t.names, A)
    r.upload(0, t.M)
    buf = np.zeros((1 << 16) + WORDS + FIELD + 4096, np.uint32)
    M = buf[1 << 16:]
    M[:WORDS] = t.M
    prog = ol.Program(t.names, A)
    for n in (1, 2):  # a single step, then two replays of the captured graph
        r.run(n)
        r.sync()
        for _ in range(n):
            prog.run(M)
        assert np.array_equal(r.read(0, WORDS), M[:WORDS])
    r.close()


def test_a_tape_that_writes_its_own_flags_is_not_planned_by_them():
    """A copy over the chain flags of the dispatches after it."""
    def tape(dst):
        t = Tape()
        chain = t.words(0)
        t.op("_copy", {0: slot(0), 1: dst(chain)}, (4, 1, 1))
        for f in (1, 3):
            t.op("turb_zero", {1: slot(f)}, (SJ, SK, NZ + 1))
        adv = {q: t.words(0) for q in (1, 3, 5, 12, 20, 21)}
        adv.update({2: slot(5), 4: slot(6), 6: slot(7), 13: slot(8), 14: slot(9), 17: t.words(0, 0), 30: slot(10)})
        adv.update({q: slot(11) for q in (7, 8, 9, 10, 15, 16)})
        t.M[adv[1]] = 1
        for f in (12, 13):
            t.op("adv_fused", {**adv, 11: slot(f), 32: chain})
        return t.batches()
    assert tape(lambda chain: slot(1)) == [1, 1, 1, 2, 0]
    assert tape(lambda chain: chain - 2) == [1, 1, 1, 1, 1]


def flagged_tape():
    """An advection that stores its tendency (chain 0) or updates a field (8,
    with its halo 40), one that advects that field, a merged copy and a reader
    of its second destination.  Returns the tape and its flags' words."""
    rng = np.random.default_rng(11)
    t = Tape()
    t.M[:FLAGS] = rng.uniform(0.5, 1.5, FLAGS).astype(np.float32).view(np.uint32)
    chain, sides, count = t.words(0), t.words(0, 0), t.words(1)
    one = {1: t.words(1), 3: t.words(0), 5: t.words(0), 12: t.words(0), 20: t.words(0), 21: t.words(0), 17: sides,
           4: slot(1), 6: slot(2), 13: slot(3), 14: slot(4), 30: slot(5)}
    one.update({q: slot(6) for q in (7, 8, 9, 10, 15, 16)})
    one.update({22: slot(18), 23: slot(19), 24: slot(20)})  # the fluxes of the separate dispatches
    dt = t.words(*np.array([0.01], np.float32).view(np.int32))
    t.op("adv_fused", {**one, 2: slot(7), 11: slot(8), 32: chain, 39: slot(9), 40: slot(10), 41: dt})
    t.op("adv_fused", {**one, 2: slot(10), 11: slot(11), 32: t.words(0)})
    t.op("copy_fields", {1: slot(12), 5: slot(13), 2: slot(14), 6: slot(15), 9: count}, (FIELD, 1, 1))
    t.op("build_sadv", {1: slot(16), 2: slot(15), 3: slot(17)}, (SJ, SK, NZ + 1))
    return t, chain, sides, count


@pytest.mark.gpu
def test_uploaded_flags_reach_the_plan(gpu):
    """Flags uploaded between runs: every run, alone and as a replayed graph, is
    the oracle's, and dispatches that the new flags make dependent no longer
    share a launch."""
    t, chain, sides, count = flagged_tape()
    A = np.array(t.args)
    r = te_host.Replayer(WORDS, t.names, A)
    r.upload(0, t.M)
    buf = np.zeros((1 << 16) + WORDS + FIELD + 4096, np.uint32)
    M = buf[1 << 16:]
    M[:WORDS] = t.M
    prog = ol.Program(t.names, A)
    for flags, groups in ((dict(), [2, 0, 2, 0]), ({chain: 8}, [1, 1, 2, 0]), ({count: 2}, [1, 1, 1, 1]),
                          ({chain: 40}, [1, 1, 1, 1]), ({sides: 1}, [1, 1, 1, 1]), ({sides + 1: 1}, [1, 1, 1, 1]),
                          ({chain: 0, sides: 0, sides + 1: 0, count: 1}, [2, 0, 2, 0])):
        print("flags", flags, flush=True)
        for at, v in flags.items():
            r.upload(at, np.array([v], np.uint32))
            M[at] = v
        assert r.launches()[:, 0].tolist() == groups
        for n in (2, 1):
            r.run(n)
            r.sync()
            for _ in range(n):
                prog.run(M)
            got, want = r.read(0, WORDS), M[:WORDS].copy()
            # not stored here: the oracle's fluxes and a chained update's tendency
            for w in (got, want):
                w[slot(18): slot(21)] = 0
                if M[chain] & 8:
                    w[slot(8): slot(8) + FIELD] = 0
            assert np.array_equal(got, want), (flags, n)
    r.close()


@pytest.mark.gpu
def test_uploaded_flags_reach_an_ensemble_member(gpu):
    """w's buoyancy switched off (chain flag 64) between steps of an ensemble:
    its next step is the oracle's of the changed program."""
    import ctypes

    import runs
    cfg = te_host.config(nx=18, ny=12, nz=14, tke=1, initial_tke=3)
    ens = te_host.Ensemble([cfg, te_host.config(nx=12, ny=10, nz=8)])
    member = te_host.lib().te_ensemble_member(ens.h, 0)
    ref = runs.OracleRun(cfg, fused=True)
    end = runs.arena_end(ref.enc)
    keep = runs.state_mask(ref.enc)
    chains = {int(A[4 + 32]) for n, A in zip(ref.names, ref.args) if n == "adv_fused" and ref.M[A[4 + 32]] & 64}
    assert chains
    for off in (False, True):
        if off:
            for at in chains:
                v = np.array([int(ref.M[at]) & ~64], np.uint32)
                ref.M[at] = v[0]
                assert te_host.lib().te_upload_words(member, at, v.ctypes.data_as(ctypes.POINTER(ctypes.c_uint32)),
                                                     1) == te_host.TE_OK
        ens.step(2)
        ens.sync()
        ref.step(2)
        got, want = ens.member_words(0, 0, end), ref.M[:end].copy()
        got[~keep] = 0
        want[~keep] = 0
        assert np.array_equal(got, want), (off, runs.first_difference(ref, got, want))
    ens.close()
