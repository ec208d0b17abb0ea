"""Host-side planning of the GPU engine (index maps, batch tables, S3 jobs) checked
against the oracle through the NumPy emulator of the C ABI (no GPU needed)."""
import ctypes

import numpy as np
import pytest

import abi_emulator
from oracle import rccsdt_tri as tri


@pytest.mark.parametrize("o,v", [(1, 2), (3, 4), (4, 5), (5, 3)])
def test_engine_residual_and_update_plan(monkeypatch, o, v):
    abi_emulator.install(monkeypatch)
    from distr_cc.synthetic import SyntheticSystem
    from distr_cc.t3_engine import TriplesEngine
    s = SyntheticSystem(o, v, naux=20, seed=11 + o)
    rng = np.random.default_rng(3)
    im = {k: x + 1e-3 * rng.normal(size=x.shape) for k, x in s.bare_intermediates().items()}
    t2, t3 = s.t2(), s.t3_tri()
    eng = TriplesEngine(o, v)
    eng.set_t3(t3)
    eng.set_intermediates(im, t2)
    eng.residual()
    Ro = tri.compute_r3_tri(o, v, im, t2, t3, batch_size=7)
    assert abs(eng.R.download() - Ro).max() <= 1e-12 * abs(Ro).max()
    n2, na = eng.finalize(s.mo_energy, level_shift=0.02, nvir_diis=max(1, v - 1))
    t3o, _, n2o, nao = tri.t3_update(o, Ro, t3, s.mo_energy, 0.02, max(1, v - 1))
    assert abs(eng.get_t3() - t3o).max() <= 1e-13 * abs(t3o).max()
    # (an i=j=k block is entirely abc-symmetric, so its projected update is round-off: absolute floor)
    assert abs(n2 - n2o) <= 1e-12 * n2o + 1e-26


@pytest.mark.parametrize("o,v,pairs,fused", [(4, 5, 3, True), (5, 3, 1, True), (4, 4, 4, False)])
def test_engine_ring_chunked(monkeypatch, o, v, pairs, fused):
    """The ring operator G computed for a few pairs at a time (the memory-bounded path of large
    systems), with and without the fused W_ovvo + Z GEMM."""
    abi_emulator.install(monkeypatch)
    from distr_cc.synthetic import SyntheticSystem
    from distr_cc.t3_engine import TriplesEngine
    s = SyntheticSystem(o, v, naux=20, seed=19 + o)
    rng = np.random.default_rng(4)
    im = {k: x + 1e-3 * rng.normal(size=x.shape) for k, x in s.bare_intermediates().items()}
    t2, t3 = s.t2(), s.t3_tri()
    eng = TriplesEngine(o, v, ring_fused=fused, ring_g_bytes=pairs * o * v ** 3 * 8)
    assert eng.Gs.shape[0] == pairs
    eng.set_t3(t3)
    eng.set_intermediates(im, t2)
    eng.residual()
    Ro = tri.compute_r3_tri(o, v, im, t2, t3, batch_size=7)
    assert abs(eng.R.download() - Ro).max() <= 1e-12 * abs(Ro).max()


def pair_symmetric_noise(im, rng, scale=1e-3):
    """Independent noise on every intermediate except W_vvvv, whose noise keeps its pair symmetry
    W[a,b,d,e] = W[b,a,e,d] (and nothing more: it is not symmetric in (a,b) or (d,e) alone)."""
    out = {k: x + scale * rng.normal(size=x.shape) for k, x in im.items()}
    n = scale * rng.normal(size=im['W_vvvv'].shape)
    out['W_vvvv'] = im['W_vvvv'] + n + n.transpose(1, 0, 3, 2)
    return out


@pytest.mark.parametrize("o,v,prec,chunk", [(3, 5, "fp64", None), (4, 4, "fp64", 7), (3, 6, "fp32", 5),
                                            (3, 7, "bf16x3", None), (2, 9, "bf16x3", 2)])
def test_engine_vvvv_pairs(monkeypatch, o, v, prec, chunk):
    """W_vvvv x T3 as symmetric / antisymmetric products over triangular pairs (split, one two-entry
    GEMM, unfold per term and chunk of blocks) against the oracle's plain einsums."""
    abi_emulator.install(monkeypatch)
    from distr_cc.synthetic import SyntheticSystem
    from distr_cc.t3_engine import GemmLaunch, TriplesEngine, pair_dims
    s = SyntheticSystem(o, v, naux=20, seed=41 + v)
    im = pair_symmetric_noise(s.bare_intermediates(), np.random.default_rng(6))
    t2, t3 = s.t2(), s.t3_tri()
    kw = {"fp64": {}, "fp32": dict(dtype=np.float32),
          "bf16x3": dict(dtype=np.float32, contract="bf16x3")}[prec]
    nS, nA, kp = pair_dims(v)
    assert (nS, nA) == (v * (v + 1) // 2, v * (v - 1) // 2) and kp % 64 == 0 and kp >= nS
    isz = 8 if prec == "fp64" else 4
    eng = TriplesEngine(o, v, vvvv_pairs=True,
                        pair_bytes=None if chunk is None else chunk * 2 * v * (kp + nS) * isz, **kw)
    # chunks of equal size within the bound (and within the T2 -> T3 / ring scratch they borrow)
    nbc = eng.Tp.shape[1]
    nchunk = -(-eng.n3 // nbc)
    assert nbc <= (chunk or eng.n3) and nbc == -(-eng.n3 // nchunk)
    assert eng.Tp.nbytes <= eng.Xt.nbytes and eng.Up.nbytes <= eng.Gs.nbytes
    pairs = [g for g in eng.launches if isinstance(g, GemmLaunch) and g.name.startswith("W_vvvv pairs")]
    assert len(pairs) == 3 * nchunk and not any(g.name.startswith("W_vvvv a") for g in eng.launches)
    if prec == "bf16x3":
        assert all(g.fn == "dcc_contract_packed_bf16x3" for g in pairs)
    eng.set_t3(t3)
    eng.set_intermediates(im, t2)
    eng.residual()
    Ro = tri.compute_r3_tri(o, v, im, t2, t3)
    tol = {"fp64": 1e-12, "fp32": 2e-5, "bf16x3": 3e-4}[prec]
    assert abs(eng.R.download().astype(np.float64) - Ro).max() <= tol * abs(Ro).max()


def test_engine_vvvv_pairs_rejects_asymmetric(monkeypatch):
    """An engine with pair-symmetric W_vvvv products refuses intermediates whose W_vvvv lacks the
    symmetry, instead of computing the symmetrised term."""
    abi_emulator.install(monkeypatch)
    from distr_cc.synthetic import SyntheticSystem
    from distr_cc.t3_engine import TriplesEngine
    s = SyntheticSystem(3, 4, naux=20, seed=5)
    rng = np.random.default_rng(8)
    im = {k: x + 1e-3 * rng.normal(size=x.shape) for k, x in s.bare_intermediates().items()}
    eng = TriplesEngine(3, 4, vvvv_pairs=True)
    with pytest.raises(ValueError, match="pair-symmetric"):
        eng.set_intermediates(im, s.t2())
    eng.set_intermediates(pair_symmetric_noise(s.bare_intermediates(), rng), s.t2())


def test_engine_oooo_chunk_rounding(monkeypatch):
    """W_oooo/F_oo target chunks: a bound of 52 targets is rounded up to one 64-row chunk (within
    5/4 of the bound), leaving a partial second chunk of 20 of the 84 targets."""
    abi_emulator.install(monkeypatch)
    from distr_cc.synthetic import SyntheticSystem
    from distr_cc.t3_engine import TriplesEngine
    o, v = 7, 3
    s = SyntheticSystem(o, v, naux=20, seed=23)
    rng = np.random.default_rng(5)
    im = {k: x + 1e-3 * rng.normal(size=x.shape) for k, x in s.bare_intermediates().items()}
    t2, t3 = s.t2(), s.t3_tri()
    eng = TriplesEngine(o, v, ring_g_bytes=52 * 5 * v ** 3 * 8)
    assert eng.n3 == 84 and eng.Xp.shape[1] == 64
    eng.set_t3(t3)
    eng.set_intermediates(im, t2)
    eng.residual()
    Ro = tri.compute_r3_tri(o, v, im, t2, t3, batch_size=11)
    assert abs(eng.R.download() - Ro).max() <= 1e-12 * abs(Ro).max()


@pytest.mark.parametrize("o,v", [(1, 3), (3, 4), (4, 3), (2, 5)])
def test_engine_t3_to_r1r2_and_w_plan(monkeypatch, o, v):
    _t3_to_r1r2_and_w(monkeypatch, o, v, None)


@pytest.mark.parametrize("o,v,qc", [(4, 3, 1), (5, 3, 2), (3, 4, 2)])
def test_engine_t3_to_r1r2_and_w_chunked(monkeypatch, o, v, qc):
    """Middle index q processed in chunks of qc (the memory-bounded path of large systems)."""
    _t3_to_r1r2_and_w(monkeypatch, o, v, qc)


def _t3_to_r1r2_and_w(monkeypatch, o, v, qc):
    abi_emulator.install(monkeypatch)
    from distr_cc.synthetic import SyntheticSystem
    from distr_cc.t3_engine import TriplesEngine
    s = SyntheticSystem(o, v, naux=20, seed=17 + v)
    im, t2, t3 = s.bare_intermediates(), s.t2(), s.t3_tri()
    nmo = o + v
    rng = np.random.default_rng(4)
    E = s.pppp() + 0.01 * rng.normal(size=(nmo,) * 4)
    E = 0.5 * (E + E.transpose(1, 0, 3, 2))
    F = s.fock + 0.01 * rng.normal(size=(nmo, nmo))
    eng = TriplesEngine(o, v)
    if qc is not None:
        eng._setup_lower(z_budget_bytes=qc * o * o * v ** 3 * 8)
        assert eng._lower['qc'] == qc and len(eng._lower['chunks']) == -(-o // qc)
    eng.set_t3(t3)
    eng.set_intermediates(im, t2)
    eng.set_t1_dressed(F[:o, o:], E[:o, :o, o:, o:], E[:o, :o, :o, o:], E[o:, :o, o:, o:])
    r1, r2 = eng.t3_to_r1r2()
    r1o, r2o = np.zeros((o, v)), np.zeros((o, o, v, v))
    tri.r1r2_add_t3_tri(o, v, F, E, t3, r1o, r2o)
    floor = 1e-12 * abs(t3).max() * abs(E).max()
    assert abs(r1 - r1o).max() <= 1e-12 * abs(r1o).max() + floor
    assert abs(r2 - r2o).max() <= 1e-12 * abs(r2o).max() + floor
    eng.t3_to_w()
    Wv, Wvv = eng.get_w_t3_adjusted()
    Wvo, Wvvo = im['W_vooo'].copy(), im['W_vvvo'].copy()
    tri.intermediates_t3_add_t3_tri(o, v, E, t3, Wvo, Wvvo)
    assert abs(Wv - Wvo).max() <= 1e-12 * abs(Wvo).max()
    assert abs(Wvv - Wvvo).max() <= 1e-12 * abs(Wvvo).max()


@pytest.mark.parametrize("o,v,bs", [(2, 5, 2), (3, 4, 3), (2, 5, 5), (1, 3, 2)])
@pytest.mark.parametrize("w_mode", ["dense", "task"])
def test_q_engine_plan(monkeypatch, o, v, bs, w_mode):
    """Both W_vvvvoo forms: dense, and per-chunk slots of the distinct ordered block triples (with a
    one-task chunk size, so that every chunk builds its own slots)."""
    abi_emulator.install(monkeypatch)
    from distr_cc.device import DeviceArray
    from distr_cc.q_engine import QEngine
    from distr_cc.synthetic import SyntheticSystem
    from oracle import q_energy as Q
    from oracle import t3_layout as TL
    s = SyntheticSystem(o, v, naux=20, seed=3 + o, sigma_t3=1e-3)
    pppp, t2, t3 = s.pppp(), s.t2(), s.t3_tri()
    ref = Q.kernel(o, v, pppp, t2, TL.full_t3_from_tri(t3, o), s.mo_energy, blksize=bs)
    chunk_bytes = bs ** 4 * o ** 4 * 8 if w_mode == "task" else 1 << 30
    eng = QEngine(o, v, blksize=bs, w_mode=w_mode, max_chunk_bytes=chunk_bytes)
    got = eng.kernel(pppp, t2, DeviceArray.from_host(t3), s.mo_energy)
    for g, r in zip(got, ref):
        assert abs(g - r) <= 1e-12 * abs(r) + 1e-25
    if w_mode == "task":
        from distr_cc.q_engine import create_full_task_list
        assert "Wv" not in eng.dev
        assert len(next(iter(eng.task_plans.values()))[-1]) == len(create_full_task_list(v, bs))


@pytest.mark.parametrize("o,v", [(3, 4), (4, 5)])
def test_engine_fp32_plan(monkeypatch, o, v):
    """FP32 storage path: same plan, FP32 rounding only (relative 1e-5 of the residual scale)."""
    abi_emulator.install(monkeypatch)
    from distr_cc.synthetic import SyntheticSystem
    from distr_cc.t3_engine import TriplesEngine
    s = SyntheticSystem(o, v, naux=20, seed=40 + o)
    im, t2, t3 = s.bare_intermediates(), s.t2(), s.t3_tri()
    eng = TriplesEngine(o, v, dtype=np.float32)
    eng.set_t3(t3)
    eng.set_intermediates(im, t2)
    eng.residual()
    Ro = tri.compute_r3_tri(o, v, im, t2, t3)
    assert abs(eng.R.download().astype(np.float64) - Ro).max() <= 1e-5 * abs(Ro).max()
    eng.finalize(s.mo_energy)
    t3o = tri.t3_update(o, Ro, t3, s.mo_energy)[0]
    assert abs(eng.get_t3() - t3o).max() <= 1e-5 * abs(t3o).max()


@pytest.mark.parametrize("split", [False, True])
@pytest.mark.parametrize("o,v,seed", [(2, 3, 1), (3, 4, 2), (1, 4, 3)])
def test_full_iteration_plan(monkeypatch, o, v, seed, split):
    """RCCSDTEngine.update_amps (dressing, lower order, T3, update) == oracle update_amps; ``split``
    lowers the split-K thresholds so every long-K lower-order contraction takes the partial-slice path."""
    abi_emulator.install(monkeypatch)
    from ccsdt_cases import molecule_like, random_amplitudes
    from distr_cc import rccsdt_engine as RE
    from distr_cc.rccsdt_engine import RCCSDTEngine
    from oracle import rccsdt_lower as lo
    if split:
        monkeypatch.setattr(RE, "SPLIT_K_MIN", 1)
        monkeypatch.setattr(RE, "SPLIT_MIN_SLICES", 2)
    F, g, e, _ = molecule_like(o, v, seed)
    t1, t2, t3 = random_amplitudes(o, v, seed + 100)
    eng = RCCSDTEngine(o, v, F, g, e, level_shift=0.05, nvir_diis=max(1, v - 1))
    eng.set_amplitudes(t1, t2, t3)
    assert abs(eng.energy() - tri.energy_rhf(o, F, g, t1, t2)) < 1e-14
    res = eng.update_amps()
    a1, a2, a3 = eng.get_amplitudes()
    b1, b2, b3, rres = lo.update_amps(o, F, g, e, t1, t2, t3, level_shift=0.05, nvir_diis=max(1, v - 1))
    assert np.allclose(res, rres, rtol=1e-12, atol=1e-15)
    for a, b in ((a1, b1), (a2, b2), (a3, b3)):
        assert abs(a - b).max() <= 1e-12 * max(abs(b).max(), 1e-30)


def test_diis_packing_round_trip_and_steps(monkeypatch):
    abi_emulator.install(monkeypatch)
    from ccsdt_cases import molecule_like, random_amplitudes
    from distr_cc.device import DeviceArray
    from distr_cc.diis import DeviceDIIS
    from distr_cc.rccsdt_engine import RCCSDTEngine
    from oracle.diis import DIIS
    o, v = 3, 4
    F, g, e, _ = molecule_like(o, v, 7)
    eng = RCCSDTEngine(o, v, F, g, e, nvir_diis=3)
    t1, t2, t3 = random_amplitudes(o, v, 8)
    eng.set_amplitudes(t1, t2, t3)
    x = DeviceArray((eng.diis_size(),))
    eng.pack(x)
    host = x.download()
    pairs = [(i, j) for i in range(o) for j in range(i, o)]
    ref = np.concatenate([t1.ravel(), np.concatenate([t2[i, j].ravel() for i, j in pairs]),
                          t3[:, :3, :3, :3].ravel()])
    assert np.array_equal(host, ref)
    eng.set_amplitudes(0 * t1, 0 * t2, t3)
    eng.unpack(x)
    a1, a2, a3 = eng.get_amplitudes()
    assert np.array_equal(a1, t1) and np.array_equal(a2, t2) and np.array_equal(a3, t3)
    rng = np.random.default_rng(9)
    dd, od = DeviceDIIS(ref.size, space=3), DIIS(space=3)
    vec = ref.copy()
    for step in range(6):
        vec = vec + 0.5 ** step * rng.standard_normal(vec.size)
        x.upload(vec)
        got = dd.update(x).download()
        want = od.update(vec)
        assert abs(got - want).max() <= 1e-12 * abs(want).max()


def test_kernel_converges_to_oracle_fixed_point(monkeypatch):
    abi_emulator.install(monkeypatch)
    from ccsdt_cases import DuckMF, molecule_like
    from distr_cc.distribute_t3 import SINGLE_RANK
    from distr_cc.rccsdt import RCCSDT, _PhysicistsERIs
    from oracle import rccsdt_lower as lo
    o, v = 2, 3
    F, g, e, _ = molecule_like(o, v, 22)
    cc = RCCSDT(DuckMF(o, v, e), SINGLE_RANK)
    cc.conv_tol, cc.conv_tol_normt, cc.verbose = 1e-12, 1e-10, 0
    e_cc, tamps = cc.kernel(eris=_PhysicistsERIs(F, e, g))
    assert cc.converged
    _, t1, t2 = tri.init_amps_rhf(o, F, e, g)
    t3 = np.zeros_like(tamps[2][1])
    for _ in range(200):
        t1, t2, t3, res = lo.update_amps(o, F, g, e, t1, t2, t3)
        if max(res) < 1e-12:
            break
    assert abs(e_cc - tri.energy_rhf(o, F, g, t1, t2)) < 1e-10
    assert abs(tamps[1] - t2).max() < 1e-8


def test_mixed_iteration_plan(monkeypatch):
    """FP32 triples inside the FP64 iteration: one step stays within FP32 rounding of the oracle."""
    abi_emulator.install(monkeypatch)
    from ccsdt_cases import molecule_like, random_amplitudes
    from distr_cc.rccsdt_engine import RCCSDTEngine
    from oracle import rccsdt_lower as lo
    o, v = 3, 4
    F, g, e, _ = molecule_like(o, v, 2)
    t1, t2, t3 = random_amplitudes(o, v, 102)
    eng = RCCSDTEngine(o, v, F, g, e, t3_dtype=np.float32)
    eng.set_amplitudes(t1, t2, t3)
    eng.update_amps()
    a1, a2, a3 = eng.get_amplitudes()
    b1, b2, b3, _ = lo.update_amps(o, F, g, e, t1, t2, t3)
    assert abs(a1 - b1).max() <= 1e-6 * abs(b1).max()
    assert abs(a2 - b2).max() <= 1e-6 * abs(b2).max()
    assert abs(a3 - b3).max() <= 1e-5 * abs(b3).max()


@pytest.mark.parametrize("o,v", [(3, 5), (3, 7), (3, 14)])
def test_bf16x3_residual_plan(monkeypatch, o, v):
    """Split-BF16x3 residual plan; at nvir=5 an FP32 GEMM (K = o v <= 16) reads Y/Z, which then get a
    packed copy, at nvir=7 and 14 Y/Z are written as packed words by the transform itself; at nvir=14
    the fused T2 -> T3 GEMM (K = v + o = 17) runs on operands its operand pass packs."""
    abi_emulator.install(monkeypatch)
    from distr_cc.synthetic import SyntheticSystem
    from distr_cc.t3_engine import TriplesEngine
    s = SyntheticSystem(o, v, naux=20, seed=31)
    im, t2, t3 = s.bare_intermediates(), s.t2(), s.t3_tri()
    eng = TriplesEngine(o, v, dtype=np.float32, contract="bf16x3")
    assert eng._yz_direct == (o * v > 16)
    # every residual GEMM with K > 16 reads packed (pre-split) operands, the others stay FP32
    gemms = [g for g in eng.launches if hasattr(g, "args")]
    assert all(g.fn == ("dcc_contract_packed_bf16x3" if g.args[2] > 16 else "dcc_contract_f32") for g in gemms)
    assert any(g.fn == "dcc_contract_f32" for g in gemms) and any(g.args[2] > 16 for g in gemms)
    eng.set_t3(t3)
    eng.set_intermediates(im, t2)
    eng.residual()
    Ro = tri.compute_r3_tri(o, v, im, t2, t3)
    assert abs(eng.R.download().astype(np.float64) - Ro).max() <= 3e-4 * abs(Ro).max()


def test_bf16x3_tile_transfer(monkeypatch):
    """Tiles transferred by launch name: a 256-wide split-BF16x3 tile falls back to 128x128 on a
    launch whose extent on that side is at most 128; other tiles are applied as given."""
    abi_emulator.install(monkeypatch)
    from distr_cc.t3_engine import GemmLaunch, TriplesEngine
    eng = TriplesEngine(3, 5, dtype=np.float32, contract="bf16x3")
    gemms = [g for g in eng.launches if isinstance(g, GemmLaunch) and g.fn.endswith("bf16x3")]
    assert gemms and all(g.max_rows <= 128 and g.args[1] <= 128 for g in gemms)
    for t, want in ((4, 3), (5, 3), (2, 2)):
        eng.set_tiles_by_name({g.name: t for g in gemms})
        assert all(g.tile == want for g in gemms)


def test_batched_ensemble_plan(monkeypatch):
    """Grouped launches + graph replay == per-system engines, for an uneven ensemble."""
    abi_emulator.install(monkeypatch)
    from distr_cc.batched import BatchedTriples
    from distr_cc.device import Stream
    from distr_cc.synthetic import SyntheticSystem
    from distr_cc.t3_engine import TriplesEngine
    systems = [(2, 4), (3, 5), (1, 3), (3, 3)]
    st = Stream.__new__(Stream)
    st.handle, st._own = ctypes.c_void_p(7), False
    bt = BatchedTriples(systems, st)
    refs = []
    for n, (o, v) in enumerate(systems):
        s = SyntheticSystem(o, v, naux=15, seed=50 + n)
        im, t2, t3 = s.bare_intermediates(), s.t2(), s.t3_tri()
        bt.set_system(n, t3, im, t2, s.mo_energy)
        e = TriplesEngine(o, v)
        e.set_t3(t3)
        e.set_intermediates(im, t2)
        e.residual()
        refs.append((e.finalize(s.mo_energy), e.get_t3()))
    bt.capture()
    bt.step()
    for e, (nrm, t3ref) in zip(bt.engines, refs):
        assert abs(e.get_t3() - t3ref).max() <= 1e-13 * abs(t3ref).max()
        assert abs(e.read_norms()[0] - nrm[0]) <= 1e-12 * nrm[0]


def test_init_amps_unshifted_with_level_shift(monkeypatch):
    """The MP2 guess divides by e_i - e_a without the level shift (rccsdt.py:212-214), also when the
    iteration's denominators carry one; t1 != 0 through a non-canonical f_ov."""
    abi_emulator.install(monkeypatch)
    from ccsdt_cases import DuckMF, molecule_like, with_fov
    from distr_cc.distribute_t3 import SINGLE_RANK
    from distr_cc.rccsdt import RCCSDT, _PhysicistsERIs
    o, v = 3, 4
    F, g, e, _ = molecule_like(o, v, 31)
    F = with_fov(F, o, 0.02, 32)
    cc = RCCSDT(DuckMF(o, v, e), SINGLE_RANK)
    cc.level_shift, cc.verbose = 0.05, 0
    emp2, tamps = cc.init_amps(_PhysicistsERIs(F, e, g))
    e_ref, t1, t2 = tri.init_amps_rhf(o, F, e, g)
    assert abs(t1).max() > 1e-4
    assert abs(tamps[0] - t1).max() <= 1e-14 * abs(t1).max()
    assert abs(tamps[1] - t2).max() <= 1e-14 * abs(t2).max()
    assert abs(emp2 - e_ref) <= 1e-14 * abs(e_ref) and not tamps[2][1].any()


@pytest.mark.parametrize("with_t3,nvir_diis,diis,shift", [(True, None, True, 0.0), (True, 2, True, 0.05),
                                                         (False, None, True, 0.0), (False, 2, True, 0.05),
                                                         (True, None, False, 0.0)])
def test_kernel_diis_trajectory(monkeypatch, with_t3, nvir_diis, diis, shift):
    """RCCSDT.kernel after 4 cycles == the oracle loop after 4 cycles: unified T1/T2/T3 DIIS
    (do_diis_max_t = True, with an nvir_diis subspace), standard T1/T2 DIIS (do_diis_max_t = False)
    and no DIIS, with and without a level shift (distr_cc/rccsdt.py:1026-1148)."""
    abi_emulator.install(monkeypatch)
    from ccsdt_cases import DuckMF, molecule_like, oracle_kernel, with_fov
    from distr_cc.distribute_t3 import SINGLE_RANK
    from distr_cc.rccsdt import RCCSDT, _PhysicistsERIs
    o, v = 2, 4
    F, g, e, _ = molecule_like(o, v, 41)
    F = with_fov(F, o, 0.01, 42)
    cc = RCCSDT(DuckMF(o, v, e), SINGLE_RANK)
    cc.do_diis_max_t, cc.nvir_diis, cc.diis, cc.level_shift = with_t3, nvir_diis, diis, shift
    cc.max_cycle, cc.verbose = 4, 0
    e_cc, tamps = cc.kernel(eris=_PhysicistsERIs(F, e, g))
    t1, t2, t3, energies = oracle_kernel(o, F, g, e, 4, level_shift=shift, nvir_diis=nvir_diis, diis=diis,
                                         with_t3=with_t3)
    assert cc.cycles == 4
    assert abs(e_cc - energies[-1]) <= 1e-13
    for a, b in ((tamps[0], t1), (tamps[1], t2), (tamps[2][1], t3)):
        assert abs(a - b).max() <= 1e-11 * abs(b).max()


def test_engine_cache_follows_attributes(monkeypatch):
    """A second kernel() on the same eris picks up changed level_shift / nvir_diis / triples_precision."""
    abi_emulator.install(monkeypatch)
    from ccsdt_cases import DuckMF, molecule_like
    from distr_cc.distribute_t3 import SINGLE_RANK
    from distr_cc.rccsdt import RCCSDT, _PhysicistsERIs
    o, v = 2, 3
    F, g, e, _ = molecule_like(o, v, 43)
    eris = _PhysicistsERIs(F, e, g)
    cc = RCCSDT(DuckMF(o, v, e), SINGLE_RANK)
    cc.max_cycle, cc.verbose = 2, 0
    cc.kernel(eris=eris)
    eng = cc.engine
    cc.level_shift, cc.nvir_diis = 0.1, 2
    cc.kernel(eris=eris)
    assert cc.engine is eng and eng.level_shift == 0.1 and eng.nvir_diis == 2
    ref = e[:o, None] - e[None, o:] - 0.1
    assert abs(eng.eia.download() - ref).max() < 1e-15
    cc.triples_precision = "fp32"
    cc.kernel(eris=eris)
    assert cc.engine is not eng and cc.engine.mixed


def test_batched_rccsdt_plan(monkeypatch):
    """Whole RCCSDT iterations of an uneven ensemble (grouped triples launches, one graph per step) ==
    each system's own RCCSDTEngine.update_amps, energies and amplitudes after two steps."""
    abi_emulator.install(monkeypatch)
    from ccsdt_cases import molecule_like, random_amplitudes
    from distr_cc.batched import BatchedRCCSDT
    from distr_cc.device import Stream
    from distr_cc.rccsdt_engine import RCCSDTEngine
    shapes = [(2, 3, 81), (3, 4, 82), (1, 4, 83), (3, 3, 84)]
    st = Stream.__new__(Stream)
    st.handle, st._own = ctypes.c_void_p(7), False
    syss = [(o, v) + molecule_like(o, v, seed)[:3] for o, v, seed in shapes]
    amps = [random_amplitudes(o, v, seed + 1) for o, v, seed in shapes]
    bt = BatchedRCCSDT(syss, st)
    # the lower-order contractions of the four systems run grouped, operation by operation
    assert len(bt.lower_phases) >= 50 and all(len(ph.launches) == 4 for ph in bt.lower_phases)
    for n, a in enumerate(amps):
        bt.set_amplitudes(n, *a)
    bt.capture()
    for _ in range(2):
        bt.step()
        got = bt.energies()
    for n, ((o, v, F, g, e), a) in enumerate(zip(syss, amps)):
        ref = RCCSDTEngine(o, v, F, g, e)
        ref.set_amplitudes(*a)
        for _ in range(2):
            ref.update_amps()
        assert abs(got[n] - ref.energy()) <= 1e-14
        for x, y in zip(bt.engines[n].get_amplitudes(), ref.get_amplitudes()):
            assert abs(x - y).max() <= 1e-13 * max(abs(y).max(), 1e-30)


@pytest.mark.parametrize("o,v,shift", [(1, 2, 0.0), (2, 5, 0.1), (5, 3, 0.0), (3, 4, 0.0)])
def test_lower_schedule_matches_programs(monkeypatch, o, v, shift):
    """The few-launch schedule of the lower-order part == the one-by-one programs, with a non-canonical Fock
    matrix (t1 != 0) and a level shift, over two iterations; the denominators follow configure()."""
    abi_emulator.install(monkeypatch)
    from ccsdt_cases import molecule_like, random_amplitudes, with_fov
    from distr_cc.rccsdt_engine import RCCSDTEngine
    F, g, e, _ = molecule_like(o, v, 70 + o)
    F = with_fov(F, o, 0.05, 5)
    engs = [RCCSDTEngine(o, v, F, g, e, level_shift=shift, schedule=s) for s in (True, False)]
    assert engs[0].sched is not None and engs[1].sched is None
    for eng in engs:
        eng.set_amplitudes(*random_amplitudes(o, v, 6))
    for shift2 in (shift, 0.2):
        res = []
        for eng in engs:
            eng.configure(level_shift=shift2)
            res.append(eng.update_amps() + [eng.energy()])
        assert np.allclose(res[0], res[1], rtol=1e-12, atol=1e-15)
        for x, y in zip(engs[0].get_amplitudes(), engs[1].get_amplitudes()):
            assert abs(x - y).max() <= 1e-13 * max(abs(y).max(), 1e-30)


def test_schedule_drops_kept_t3_terms(monkeypatch):
    """t3_to_w(reuse_z=True) after t3_to_r1r2 and then a scheduled iteration computes the T3 terms of W_vooo and
    W_vvvo from the new T3: the iteration has overwritten what t3_to_r1r2 kept."""
    abi_emulator.install(monkeypatch)
    from ccsdt_cases import molecule_like, random_amplitudes
    from distr_cc.rccsdt_engine import RCCSDTEngine
    o, v = 3, 4
    F, g, e, _ = molecule_like(o, v, 7)
    res = []
    for schedule in (True, False):
        eng = RCCSDTEngine(o, v, F, g, e, schedule=schedule)
        assert (eng.sched is not None) == schedule
        eng.set_amplitudes(*random_amplitudes(o, v, 6))
        eng.tr.set_t1_dressed_device(eng.G0, eng.F0, o + v)
        eng.tr.t3_to_r1r2()
        eng.update_amps()
        eng.tr.t3_to_w(reuse_z=True)
        res.append(eng.tr.get_w_t3_adjusted())
    for x, y in zip(*res):
        assert abs(x - y).max() <= 1e-13 * abs(y).max()


def test_diis_extrapolate_keeps_nothing(monkeypatch):
    """DeviceDIIS.extrapolate only forms the vector: the norm of the last update, the previous iterate and the
    vector that the next update returns are as without the call."""
    abi_emulator.install(monkeypatch)
    from distr_cc.device import DeviceArray
    from distr_cc.diis import DeviceDIIS
    from oracle.diis import DIIS
    n, steps = 9, 5
    xs = np.random.default_rng(2).standard_normal((steps, n))
    plain, asked, od = DeviceDIIS(n, space=4), DeviceDIIS(n, space=4), DIIS(space=4)
    for k, x in enumerate(xs):
        ref = od.update(x.copy())
        got = plain.update(DeviceArray.from_host(x)).download()
        assert np.array_equal(asked.update(DeviceArray.from_host(x)).download(), got)
        assert np.abs(got - ref).max() <= 1e-9 * np.abs(ref).max()
        nd = sum(v is not None for v in asked.xs)
        for m in range(1, nd + 1):
            y = asked.extrapolate(m).download()
            c = asked.coefficients(m)[1:]
            want = sum(ci * v.download() for ci, v in zip(c, asked.xs))
            assert np.abs(y - want).max() <= 1e-12 * np.abs(c).max() * np.abs(xs).max()
        assert asked.last_delta_norm_sq == plain.last_delta_norm_sq
        assert np.array_equal(asked._xprev.download(), plain._xprev.download())


def test_tile_8_of_split_bf16x3_and_plain_launches(monkeypatch):
    """Tile 8 is 256x256 with direct-to-LDS staging for a split-BF16x3 launch, packed or not, and the library's own
    choice for an FP64 or FP32 one."""
    abi_emulator.install(monkeypatch)
    from distr_cc import _lib as L
    from distr_cc.t3_engine import GemmLaunch, TriplesEngine
    eng = TriplesEngine(3, 6, dtype=np.float32, contract="bf16x3", ring_fused=True)
    eng._setup_lower()
    plain = TriplesEngine(3, 6, ring_fused=True)
    launches = [g for e in (eng, plain) for g in e._tunable() if isinstance(g, GemmLaunch)]
    seen, calls = set(), []
    monkeypatch.setattr(L, "call", lambda name, *a: calls.append((name, a)))
    for g in launches:
        g.tile = 8
        del calls[:]
        g.run(None)
        name, args = [c for c in calls if c[0].startswith("dcc_contract")][0]
        seen.add(g.fn)
        if g.fn.endswith("bf16x3"):
            assert name == {"dcc_contract_f32_bf16x3": "dcc_contract_tiled_f32_bf16x3"}.get(g.fn, g.fn), g.name
            assert args[-2] == 8
        else:
            assert name == g.fn, g.name
    assert {"dcc_contract_f32_bf16x3", "dcc_contract_packed_bf16x3", "dcc_contract_f64"} <= seen


def test_schedule_groups_unequal_engines(monkeypatch):
    """An ensemble whose systems have different numbers of contractions in a stage: every one is issued once, in a
    group with at most one of each system."""
    abi_emulator.install(monkeypatch)
    from ccsdt_cases import molecule_like
    from distr_cc.rccsdt_engine import RCCSDTEngine
    from distr_cc.schedule import LowerSchedule
    from distr_cc.t3_engine import GemmLaunch
    engines = []
    for o, v in ((2, 3), (1, 2), (2, 4)):
        F, g, e, _ = molecule_like(o, v, 5)
        engines.append(RCCSDTEngine(o, v, F, g, e, schedule=False))
    sched = LowerSchedule(engines, None)
    gemms = [(k, [s for s in e.prog["dress"].steps if isinstance(s, GemmLaunch)]) for k, e in enumerate(engines)]
    gemms = [(k, g) for k, gs in gemms for g in gs[:(4, 1, 2)[k]]]
    groups = [ph.launches for ph in sched._contractions(gemms)]
    assert sorted(map(len, groups)) == [1, 1, 2, 3]
    assert sorted(id(g) for gs in groups for g in gs) == sorted(id(g) for _, g in gemms)


def _with_op(monkeypatch, name, add):
    """Engines whose program ``name`` gets one more operation from add(engine, program)."""
    from distr_cc.rccsdt_engine import RCCSDTEngine
    build = RCCSDTEngine._build_program

    def changed(self):
        steps = build(self)
        add(self, steps[name])
        return steps

    monkeypatch.setattr(RCCSDTEngine, "_build_program", changed)


@pytest.mark.parametrize("case", ["read before complete", "set after read", "not set"])
def test_schedule_refuses_order_it_cannot_keep(monkeypatch, case):
    """A program that reads a tensor before its last contribution, or sets or accumulates out of order, runs one by
    one (no schedule) and gives what its order says."""
    abi_emulator.install(monkeypatch)
    from ccsdt_cases import molecule_like, random_amplitudes
    from distr_cc.rccsdt_engine import RCCSDTEngine
    from distr_cc.t3_engine import Operand
    o, v = 2, 3
    F, g, e, _ = molecule_like(o, v, 11)

    def add(eng, p):
        h, W = eng.nview(eng.h_ovvo, "ladi"), eng.nview(eng.imd["W_ovvo"], "ladi")
        if case == "read before complete":    # W_ovvo has been formed from h by now
            p.axpby(h, eng.gview(eng.G, "ladi"), "ladi", 0.5, 1.0)
        elif case == "set after read":        # t2 is read by every contraction before
            p.axpby(Operand(eng.t2, "ijab", (o, o, v, v)), eng.gview(eng.G, "ijab"), "ijab", 1.0, 0.0)
        else:                                 # accumulates into the result of another program
            p.axpby(eng.nview(eng.Foo1, "ki"), eng.gview(eng.Fd, "ki"), "ki", 1.0, 1.0)

    _with_op(monkeypatch, "imds3", add)
    engs = [RCCSDTEngine(o, v, F, g, e, schedule=s) for s in (True, False)]
    assert engs[0].sched is None
    for eng in engs:
        eng.set_amplitudes(*random_amplitudes(o, v, 6))
        eng.update_amps()
    for x, y in zip(engs[0].get_amplitudes(), engs[1].get_amplitudes()):
        assert np.array_equal(x, y)


def test_ensemble_schedule_leaves_room(monkeypatch):
    """The partial results of an ensemble's schedule are allocated only where they leave as much free memory as they
    take, over all systems; without room the ensemble and a single engine run operation by operation, to the same
    result."""
    emu = abi_emulator.install(monkeypatch)
    from ccsdt_cases import molecule_like, random_amplitudes
    from distr_cc.batched import BatchedRCCSDT
    from distr_cc.device import Stream
    from distr_cc.rccsdt_engine import RCCSDTEngine
    from distr_cc.schedule import LowerSchedule
    st = Stream.__new__(Stream)
    st.handle, st._own = None, False
    monkeypatch.setattr(Stream, "synchronize", lambda self: None)
    systems = []
    for o, v in ((2, 4), (3, 4), (2, 3)):
        F, g, e, _ = molecule_like(o, v, 21)
        systems.append((o, v, F, g, e))

    free = [288 << 30]

    def info(pfree, ptotal):
        pfree._obj.value, ptotal._obj.value = free[0], 288 << 30
        return 0

    monkeypatch.setattr(emu, "dcc_mem_get_info", info)
    one = RCCSDTEngine(*systems[0])
    used = [8 * (max(LowerSchedule._targets(e, n)[1].used for n in ("r1r2", "imds3")) + (e.nocc * e.nvir) ** 2)
            for e in (RCCSDTEngine(*s, schedule=False) for s in systems)]
    res = []
    # room for all; for each of them but not for all; for none
    for free[0], all_fit, one_fits in ((2 * sum(used), True, True), (2 * sum(used) - 1, False, True), (0, False, False)):
        bt = BatchedRCCSDT(systems, st)
        assert (bt.sched is not None) == all_fit
        for k, (o, v, *_) in enumerate(systems):
            bt.set_amplitudes(k, *random_amplitudes(o, v, 6 + k))
        bt.issue_step()
        res.append([bt.energies()] + [x for e in bt.engines for x in e.get_amplitudes()])
        one = RCCSDTEngine(*systems[1])
        assert (one.sched is not None) == one_fits
    for other in res[1:]:
        for x, y in zip(res[0], other):
            assert np.allclose(x, y, rtol=1e-12, atol=1e-15)


@pytest.mark.parametrize("nested", [1, 3])
def test_diis_iterates_freed_during_a_wait(monkeypatch, nested):
    """Iterates freed while another one waits for the device in its free(): each piece of memory is either kept as
    the one spare vector or released, once, and nothing is left when the DIIS goes."""
    emu = abi_emulator.install(monkeypatch)
    from distr_cc.device import DeviceArray
    from distr_cc.diis import DeviceDIIS
    n = 33
    dd = DeviceDIIS(n, space=3)
    rng = np.random.default_rng(1)
    its = [dd.update(DeviceArray.from_host(rng.standard_normal(n))) for _ in range(nested + 2)][1:]
    ptrs = [y.ptr for y in its]
    assert len(set(ptrs)) == nested + 1
    freed, waiting = [], its[1:]
    monkeypatch.setattr(emu, "dcc_free", lambda p: freed.append(p.value if p.value in ptrs else None) or 0)

    def wait():
        if waiting:
            waiting.pop().free()
        return 0

    monkeypatch.setattr(emu, "dcc_device_synchronize", wait, raising=False)
    its[0].free()
    assert not waiting
    assert sorted([p for p in freed if p] + [dd._spare]) == sorted(ptrs)
    for y in its:
        assert y.ptr == 0
        y.free()
    y = dd.update(DeviceArray.from_host(rng.standard_normal(n)))
    assert y.ptr in ptrs and dd._spare is None   # the spare is used again


@pytest.mark.parametrize("o,v,bs,fused", [(1, 18, 4, True), (1, 23, 4, True), (1, 24, 4, False), (1, 25, 3, True),
                                          (1, 26, 3, False), (1, 60, 2, True), (2, 33, 4, True), (2, 34, 6, False), (2, 30, 8, False),
                                          (2, 48, 3, True), (2, 60, 3, False), (2, 60, 1, True), (3, 60, 4, True),
                                          (9, 30, 4, True)])
def test_q_form_by_sizes(monkeypatch, o, v, bs, fused):
    """Which form of (Q) runs: the fused quadruples except for nocc <= 2 with many virtuals (both sides of the rule
    were timed at these sizes)."""
    abi_emulator.install(monkeypatch)
    from distr_cc.q_engine import QEngine
    assert QEngine(o, v, blksize=bs).fused == fused
    assert not QEngine(o, v, blksize=bs, finalize_ws=True).fused


@pytest.mark.parametrize("w_mode", ["dense", "task"])
@pytest.mark.parametrize("o,v,bs", [(1, 5, 4), (2, 5, 3)])
def test_q_engine_gemms_below_nocc_10(monkeypatch, o, v, bs, w_mode):
    """The batched GEMMs with the finalize that needs no workspace == the fused quadruples == the oracle."""
    emu = abi_emulator.install(monkeypatch)
    from distr_cc.device import DeviceArray
    from distr_cc.q_engine import QEngine
    from distr_cc.synthetic import SyntheticSystem
    from oracle import q_energy as Q
    from oracle import t3_layout as TL
    s = SyntheticSystem(o, v, naux=30, seed=500 + o * v, sigma_t3=1e-3)
    pppp, t2, t3 = s.pppp(), s.t2(), s.t3_tri()
    ref = Q.kernel(o, v, pppp, t2, TL.full_t3_from_tri(t3, o), s.mo_energy, blksize=bs)
    for fused in (True, False):
        eng = QEngine(o, v, blksize=bs, w_mode=w_mode)
        assert eng.fused
        eng.fused = fused
        for _ in range(2):
            got = eng.kernel(pppp, t2, DeviceArray.from_host(t3), s.mo_energy)
            for x, y in zip(got, ref):
                assert abs(x - y) <= 1e-12 * abs(y)
    assert "dcc_q_quads_f64" in emu.calls and "dcc_q_finalize_f64" in emu.calls


def test_canonical_cases_of_arrays():
    """canonical_cases == canonical_case and ijk_to_linear, triple by triple."""
    from distr_cc.distribute_t3 import canonical_case, canonical_cases, ijk_to_linear
    o = 5
    i, j, k = np.ogrid[:o, :o, :o]
    case, lin = canonical_cases(i, j, k, o)
    for x in np.ndindex(o, o, o):
        c, t = canonical_case(*x)
        assert (case[x], lin[x]) == (c, ijk_to_linear(*t, o))


@pytest.mark.parametrize("kw", [dict(ring_fused=True), dict(ring_fused=False),
                                dict(ring_fused=True, dtype=np.float32, contract="bf16x3")])
def test_planning_builds_tables_with_array_operations(monkeypatch, kw):
    """Planning an engine makes no Python call per source block or job (364 -> 1540 blocks, 936 -> 4200 Y blocks), only
    some per batch entry of a contraction."""
    import sys
    abi_emulator.install(monkeypatch)
    from distr_cc.t3_engine import TriplesEngine
    counts = []
    for o in (12, 20):
        TriplesEngine(2, 3, **kw)   # imports and caches
        n = [0]

        def count(frame, event, arg):
            n[0] += event in ("call", "c_call")

        sys.setprofile(count)
        try:
            eng = TriplesEngine(o, 3, **kw)
            eng._setup_lower()
        finally:
            sys.setprofile(None)
        launches = [g for g in eng._tunable() if hasattr(g, "nbatch")]
        counts.append((n[0], sum(g.nbatch for g in launches)))
    calls, entries = (y - x for x, y in zip(*counts))
    assert entries < 1200 and calls < 15 * entries, counts


@pytest.mark.parametrize("fused", [True, False])
def test_packed_operands_are_read(monkeypatch, fused):
    """Every tensor that a split-BF16x3 engine packs for a residual is read, to its end, by a product."""
    abi_emulator.install(monkeypatch)
    from distr_cc.t3_engine import GemmLaunch, TriplesEngine
    eng = TriplesEngine(4, 6, dtype=np.float32, contract="bf16x3", ring_fused=fused)
    assert eng._packs
    for src, dst, n in eng._packs:
        assert n == src.size == dst.size
        last = -1
        for g in eng.launches:
            if not isinstance(g, GemmLaunch) or g.fn != "dcc_contract_packed_bf16x3":
                continue
            M, N, K, _, _, A, am, ak, B, bk, bn = g.args[:11]
            for ptr, field, rows, k, nrow in ((A, "a_off", am, ak, None), (B, "b_off", bn, bk, N)):
                if not dst.ptr <= ptr.value < dst.ptr + dst.nbytes:
                    continue
                at = lambda m, x: (x // (m.e1 * m.e2) * m.s0 + x // m.e2 % m.e1 * m.s1 + x % m.e2 * m.s2).max()
                for b in g.table:
                    nr = int(b["m_end"]) if nrow is None else nrow
                    off = (ptr.value - dst.ptr) // 4 + int(b[field])
                    last = max(last, off + int(at(rows, np.arange(nr)) + at(k, np.arange(K))))
        assert last == n - 1, (src.shape, last)
