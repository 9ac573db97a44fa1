"""Batched uneven SPD factor + solve (mi_dposv_vbatched / mi_sposv_vbatched).

Each system is checked against the oracle's restatement of llt_inplace::blocked / unblocked
and LLT::_solve_impl (oracle/llt_oracle.c) on the same input: the factor within 1e-12
relative to ||L||, solve backward error <= 1e-14 (FP64); FP32 against the FP64 oracle within
FP32 bounds.  Failing pivots, argument errors, the upper triangle left untouched, the
longest-first schedule, graph replay and the autotuner are covered too."""
import ctypes
import json

import numpy as np
import pytest
import torch

import mi_llt
import oracle
from mi_llt import batched, workloads

pytestmark = pytest.mark.gpu


def fill(vb, seed=0, shift=0.1, upper_junk=True):
    rng = np.random.default_rng(seed)
    mats, rhss = [], []
    for i in range(vb.count):
        n, r = int(vb.ns[i]), int(vb.rs[i])
        a = workloads.gram_spd(n, seed=seed + i, shift=shift) if n else np.zeros((0, 0))
        if upper_junk and n > 1:
            a = a.copy()
            a[np.triu_indices(n, 1)] = 1e30  # must never be read
        b = rng.standard_normal((n, r))
        if n:
            vb.A(i).copy_(torch.from_numpy(a))
        if n * r:
            vb.B(i).copy_(torch.from_numpy(b))
        mats.append(a)
        rhss.append(b)
    return mats, rhss


def check_system(vb, i, a, b, ftol, stol):
    n, r = int(vb.ns[i]), int(vb.rs[i])
    if n == 0:
        return
    asym = np.tril(a) + np.tril(a, -1).T
    l = np.tril(vb.A(i).cpu().double().numpy())
    up = np.triu(vb.A(i).cpu().double().numpy(), 1)
    assert np.all(up == np.triu(a, 1).astype(up.dtype)), f"system {i}: upper triangle modified"
    m_ref, info = oracle.llt_blocked(np.asfortranarray(asym))
    assert info == -1
    l_ref = np.tril(m_ref)
    assert np.linalg.norm(l - l_ref) <= ftol * np.linalg.norm(l_ref), f"system {i} n={n}: factor"
    if r:
        x = vb.B(i).cpu().double().numpy()
        res = asym @ x - b
        be = (np.linalg.norm(res, axis=0) / (np.linalg.norm(asym) * np.linalg.norm(x, axis=0))).max()
        assert be <= stol, f"system {i} n={n} r={r}: solve berr {be:.2e}"


SIZES = [0, 1, 2, 3, 7, 8, 15, 16, 17, 31, 32, 33, 47, 64, 100, 127, 128, 129, 191, 200, 255, 256]


@pytest.mark.parametrize("group,lpt", [(4, True), (2, False)])
def test_vbatched_fp64_matches_oracle(dev, group, lpt):
    ns = SIZES + [5, 250, 96]
    rs = [(i * 5) % 9 for i in range(len(ns))]
    rs[-1] = 17  # two groups of right-hand sides
    print(f"[gpu] vbatched fp64 group={group} lpt={lpt} count={len(ns)}", flush=True)
    vb = batched.VBatch(ns, rs, device=dev)
    mats, rhss = fill(vb, seed=10)
    h = mi_llt.Handle()
    batched.set_config(h, 2, group, lpt)
    info = batched.posv_vbatched_(vb, h)
    assert torch.all(info == 0), info
    for i in range(vb.count):
        check_system(vb, i, mats[i], rhss[i], 1e-12, 1e-14)


def test_vbatched_fp32_within_fp32_bounds(dev):
    ns = SIZES
    rs = [1 + i % 8 for i in range(len(ns))]
    vb = batched.VBatch(ns, rs, dtype=torch.float32, device=dev)
    mats, rhss = fill(vb, seed=20)
    info = batched.posv_vbatched_(vb)
    assert torch.all(info == 0)
    for i in range(vb.count):
        n = int(vb.ns[i])
        # u_fp32 * n-ish bounds against the FP64 oracle
        check_system(vb, i, mats[i].astype(np.float32).astype(np.float64), rhss[i].astype(np.float32).astype(np.float64),
                     2e-5 * max(1.0, n / 16), 2e-6 * max(1.0, n / 16))


def test_vbatched_failing_pivots_and_arguments(dev):
    ns = [40, 100, 300, 50, 129, 64]
    rs = [2, 2, 1, 3, 1, 1]
    vb = batched.VBatch(ns, rs, device=dev)
    mats, rhss = fill(vb, seed=30)
    # system 0: indefinite at column 17; system 4: at column 128; system 2: n = 300 > 256
    for i, k in ((0, 17), (4, 128)):
        a = workloads.indefinite_at(int(ns[i]), k, seed=40 + i)
        vb.A(i).copy_(torch.from_numpy(a))
        mats[i] = a
    lda_bad = vb.d_lda.clone()
    lda_bad[3] = 10  # system 3: lda < n
    vb.d_lda.copy_(lda_bad)
    b_before = [vb.B(i).clone() for i in range(vb.count)]
    info = batched.posv_vbatched_(vb).cpu().tolist()
    assert info == [18, 0, -1, -2, 129, 0]
    for i in (0, 2, 3, 4):
        assert torch.equal(vb.B(i), b_before[i])  # B unchanged for failed / skipped systems
    for i in (1, 5):
        check_system(vb, i, mats[i], rhss[i], 1e-12, 1e-14)


def test_vbatched_graph_replay(dev):
    vb = batched.gram_batch(300, seed=3, device=dev)
    a0, b0 = vb.a_flat.clone(), vb.b_flat.clone()
    h = mi_llt.Handle()
    batched.posv_vbatched_(vb, h)  # eager: sizes the workspace
    torch.cuda.synchronize()
    ref_a, ref_b = vb.a_flat.clone(), vb.b_flat.clone()
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    g = torch.cuda.CUDAGraph()
    vb.a_flat.copy_(a0)
    vb.b_flat.copy_(b0)
    torch.cuda.synchronize()
    with torch.cuda.graph(g, stream=s):
        batched.posv_vbatched_(vb, h)
    for rep in range(3):
        vb.a_flat.copy_(a0)
        vb.b_flat.copy_(b0)
        _ = (vb.a_flat * 2.0).sum()  # unrelated eager work between replays
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(vb.a_flat, ref_a) and torch.equal(vb.b_flat, ref_b), f"replay {rep}"
        assert torch.all(vb.d_info == 0)


def test_vbatched_autotune_keeps_results(dev, tmp_path):
    vb = batched.gram_batch(200, seed=4, device=dev)
    a0, b0 = vb.a_flat.clone(), vb.b_flat.clone()
    h = mi_llt.Handle()
    batched.posv_vbatched_(vb, h)
    ref_a, ref_b = vb.a_flat.clone(), vb.b_flat.clone()
    vb.a_flat.copy_(a0)
    vb.b_flat.copy_(b0)
    out = batched.autotune(vb, h, candidates=[(1, 2, True), (2, 4, True), (2, 4, False)], reps=1,
                           cache=str(tmp_path / "tune.json"))
    assert tuple(out["config"]) == batched.get_config(h)
    batched.posv_vbatched_(vb, h)
    torch.cuda.synchronize()
    assert torch.equal(vb.a_flat, ref_a) and torch.equal(vb.b_flat, ref_b)  # deterministic per system
    again = batched.autotune(vb, h, cache=str(tmp_path / "tune.json"))  # from the cache
    assert again["config"] == out["config"]


def test_vbatched_full_workload_backward_error(dev):
    """20,000 systems, n ~ U{8..256}, 1..8 right-hand sides: every system's factor and solve
    backward errors (FP64, computed here with batched torch products per size class)."""
    vb = batched.gram_batch(20000, seed=0, device=dev)
    a0, b0 = vb.a_flat.clone(), vb.b_flat.clone()
    info = batched.posv_vbatched_(vb)
    assert int((info != 0).sum()) == 0
    worst_f, worst_s = 0.0, 0.0
    for n in np.unique(vb.ns):
        idx = np.nonzero(vb.ns == n)[0]
        n = int(n)
        ao = torch.from_numpy(vb.a_off[idx]).to(dev)
        pos = ao[:, None] + torch.arange(n * n, device=dev)[None, :]
        A = a0[pos].view(-1, n, n).transpose(1, 2)
        Lf = torch.tril(vb.a_flat[pos].view(-1, n, n).transpose(1, 2))
        rf = torch.linalg.matrix_norm(A - Lf @ Lf.transpose(1, 2).contiguous()) / torch.linalg.matrix_norm(A)
        worst_f = max(worst_f, float(rf.max()))
        for k in idx[:8]:  # solves: a sample of each size class
            r = int(vb.rs[k])
            o = int(vb.b_off[k])
            Ak = a0[int(vb.a_off[k]):int(vb.a_off[k]) + n * n].view(n, n).t()
            Bk = b0[o:o + n * r].view(r, n).t()
            Xk = vb.b_flat[o:o + n * r].view(r, n).t()
            be = float(((Ak @ Xk - Bk).norm(dim=0) / (torch.linalg.matrix_norm(Ak) * Xk.norm(dim=0))).max())
            worst_s = max(worst_s, be)
    assert worst_f <= 1e-14, worst_f
    assert worst_s <= 1e-14, worst_s


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_vbatched_group_edges(dev, dtype):
    """Orders around the group sizes (64, 128 and 256: one, two and four waves) and the 64-column
    blocks, leading dimensions larger than the order, 1, 16 and 17 right-hand sides, systems that
    fail in their last column in between; the bounds are those of the tests above."""
    ns = [48, 49, 63, 64, 65, 80, 112, 127, 128, 129, 144, 177, 192, 193, 240, 241, 255, 256] * 2
    pads = [(5 * i) % 4 for i in range(len(ns))]
    rs = [(1, 16, 17, 0, 3)[i % 5] for i in range(len(ns))]
    big = batched.VBatch([n + p for n, p in zip(ns, pads)], rs, dtype=dtype, device=dev)
    big.d_n.copy_(torch.tensor(ns, dtype=torch.int32))
    rng = np.random.default_rng(5)
    mats, rhss, before = [], [], []
    for i, n in enumerate(ns):
        bad = i % 9 == 4
        a = workloads.indefinite_at(n, n - 1, seed=60 + i) if bad else workloads.gram_spd(n, seed=60 + i)
        a = np.array(a)
        a[np.triu_indices(n, 1)] = 1e30  # must never be read
        b = rng.standard_normal((n, rs[i]))
        if dtype == torch.float32:
            a, b = a.astype(np.float32).astype(np.float64), b.astype(np.float32).astype(np.float64)
        big.A(i)[:n, :n].copy_(torch.from_numpy(a))
        if rs[i]:
            big.B(i)[:n].copy_(torch.from_numpy(b))
        mats.append(a)
        rhss.append(b)
        before.append(big.B(i).clone())
    info = batched.posv_vbatched_(big, mi_llt.Handle()).cpu().tolist()
    f32 = dtype == torch.float32
    for i, n in enumerate(ns):
        if i % 9 == 4:
            assert info[i] == n, (i, n, info[i])
            assert torch.equal(big.B(i), before[i])
            continue
        assert info[i] == 0, (i, n, info[i])
        a, b = mats[i], rhss[i]
        asym = np.tril(a) + np.tril(a, -1).T
        l = big.A(i)[:n, :n].cpu().double().numpy()
        assert np.all(np.triu(l, 1) == np.triu(a, 1).astype(l.dtype)) or f32, f"system {i}: upper triangle modified"
        lo = np.tril(oracle.llt_blocked(np.asfortranarray(asym))[0])
        assert np.linalg.norm(np.tril(l) - lo) <= (2e-5 * n / 16 if f32 else 1e-12) * np.linalg.norm(lo)
        if rs[i]:
            x = big.B(i)[:n].cpu().double().numpy()
            res = np.linalg.norm(asym @ x - b, axis=0) / (np.linalg.norm(asym) * np.linalg.norm(x, axis=0))
            assert res.max() <= (2e-6 * n / 16 if f32 else 1e-14), (i, n, rs[i], res.max())


def test_vbatched_schedule_round_trip(dev):
    """What a handle reports is what it launches by: saving a schedule and setting it again changes
    nothing, a new handle's included."""
    h = mi_llt.Handle()
    assert batched.get_config(h) == (3, 0, True)  # the default of both precisions
    batched.set_config(h, *batched.get_config(h))
    assert batched.get_config(h) == (3, 0, True)
    batched.set_config(h, 2, 4, False)
    assert batched.get_config(h) == (2, 4, False)


@pytest.mark.parametrize("batch", [1, 63, 1024, 1025, 5000])
@pytest.mark.parametrize("lpt", [0, 1])
def test_vbatched_queue_keeps_given_order(dev, batch, lpt):
    """The plan's queues (the last batch x 48 bytes of the plan, a system's index at byte 32): systems of
    one size class -- with longest first, of one tile count -- stand in the given order, and systems with
    bad arguments in none."""
    rng = np.random.default_rng(batch)
    ns = rng.integers(0, 257, size=batch)
    vb = batched.VBatch(ns, rng.integers(0, 3, size=batch))
    vb.a_flat.fill_(0.0)
    for i in range(batch):  # identity matrices
        vb.A(i).diagonal().fill_(1.0) if ns[i] else None
    bad = rng.random(batch) < 0.1
    n_arg = torch.from_numpy(np.where(bad, -1, ns).astype(np.int32)).to(dev)
    L = mi_llt.lib()
    plan_bytes = getattr(L, "_ZN2mi13vb_plan_bytesEl")  # mi::vb_plan_bytes, mi::launch_vbatched<double>
    plan_bytes.restype, plan_bytes.argtypes = ctypes.c_int64, [ctypes.c_int64]
    launch = getattr(L, "_ZN2mi15launch_vbatchedIdEEvlPKiPKPT_S2_S2_S6_S2_PiPviiP12ihipStream_t")
    vp = ctypes.c_void_p
    launch.restype, launch.argtypes = None, [ctypes.c_int64] + [vp] * 8 + [ctypes.c_int] * 2 + [vp]
    plan = torch.zeros(plan_bytes(batch), dtype=torch.uint8, device=dev)
    launch(batch, *(vp(t.data_ptr()) for t in (n_arg, vb.d_A, vb.d_lda, vb.d_nrhs, vb.d_B, vb.d_ldb, vb.d_info, plan)),
           min(batch, 256), lpt, vp(torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    nt = (ns + 15) // 16
    key = -nt if lpt else np.digitize(-nt, [-8, -4], right=False)  # orders up to 256, 128, 64
    good = np.nonzero(~bad)[0]
    want = good[np.argsort(key[good], kind="stable")]
    got = plan.cpu().numpy()[-48 * batch:].reshape(batch, 48)[:len(good), 32:36].copy().view(np.int32)[:, 0]
    np.testing.assert_array_equal(got, want)
    assert vb.d_info.tolist() == np.where(bad, -1, 0).tolist()


def test_vbatched_autotune_ignores_another_kernels_cache(dev, tmp_path):
    """A schedule cached under the batch's signature alone was timed for an earlier kernel: it is not
    applied, and the new one is kept under a key of its own."""
    vb = batched.gram_batch(16, nmin=8, nmax=64, seed=3)
    path = tmp_path / "tune.json"
    path.write_text(json.dumps({vb.signature(): {"config": [1, 4, False], "times_ms": {}}}))
    h = mi_llt.Handle()
    out = batched.autotune(vb, h, candidates=[(2, 0, True)], reps=1, cache=str(path))
    assert out["config"] == [2, 0, True] and batched.get_config(h) == (2, 0, True)
    assert len(json.loads(path.read_text())) == 2
    assert len(batched.CANDIDATES) == len({(w, o) for w, _, o in batched.CANDIDATES})  # group: no effect


def _fma32(a, b, c):
    """a b + c with one rounding to float32 (a product of two floats is exact in double)."""
    return (a.astype(np.float64) * b.astype(np.float64) + c.astype(np.float64)).astype(np.float32)


def _factor32(a):
    """Lower factors of a (m, n, n), n a multiple of 16, in float32 by tile columns of 16: A's column less
    the sum over all earlier columns, formed by itself; the tile's column loop with the reciprocal square
    root and one Newton step; the rows below by the tile's inverse."""
    f32 = np.float32
    m, n, _ = a.shape
    out = np.zeros_like(a)
    for k0 in range(0, n, 16):
        s = np.zeros((m, n - k0, 16), f32)
        for k in range(k0):
            s = _fma32(out[:, k0:, k, None], out[:, None, k0:k0 + 16, k], s)
        c = a[:, k0:, k0:k0 + 16] - s
        u, v = c[:, :16].copy(), np.broadcast_to(np.eye(16, dtype=f32), (m, 16, 16)).copy()
        for j in range(16):
            x = u[:, j, j].copy()
            r = (1 / np.sqrt(x.astype(np.float64))).astype(f32)
            r = r * _fma32(-(f32(0.5) * x * r), r, np.full_like(x, 1.5))
            u[:, :, j] *= r[:, None]
            v[:, :, j] *= r[:, None]
            for i in range(j + 1, 16):
                v[:, :, i] = _fma32(-u[:, i, j, None], v[:, :, j], v[:, :, i])
                u[:, :, i] = _fma32(-u[:, i, j, None], u[:, :, j], u[:, :, i])
        out[:, k0:k0 + 16, k0:k0 + 16] = np.tril(u)
        p = np.zeros((m, n - k0 - 16, 16), f32)
        for k in range(16):  # v[i][k] is the inverse's [k][i]
            p = _fma32(c[:, 16:, k, None], v[:, k, None, :], p)
        out[:, k0 + 16:, k0:k0 + 16] = p
    return out


@pytest.mark.parametrize("n,count", [(64, 200), (128, 60), (200, 30)])
def test_vbatched_float_sums_keep_their_own_rounding(dev, n, count):
    """The error of the single precision factor (one, two and four waves a system) against 64 bits is no
    more than 1.1 times that of the same arithmetic on the CPU with each column's sum formed by itself and
    subtracted from A once.  Products added to A one by one, within a block of 64 columns, would be
    rounded at A's magnitude: 1.5 times at n = 64 by the same emulation."""
    print(f"[gpu] float sums n={n}", flush=True)
    rng = np.random.default_rng(n)
    g = rng.standard_normal((count, n, n))
    a = (g @ g.swapaxes(1, 2) / n + 0.1 * np.eye(n)).astype(np.float32)
    a = np.tril(a) + np.tril(a, -1).swapaxes(1, 2)
    vb = batched.VBatch([n] * count, [0] * count, dtype=torch.float32, device=dev)
    for i in range(count):
        vb.A(i).copy_(torch.from_numpy(a[i]))
    assert int(batched.posv_vbatched_(vb, mi_llt.Handle()).abs().sum()) == 0
    got = np.stack([np.tril(vb.A(i).cpu().numpy()) for i in range(count)]).astype(np.float64)
    want = np.linalg.cholesky(a.astype(np.float64))
    pad = -n % 16
    ap = np.zeros((count, n + pad, n + pad), np.float32)
    ap[:, :n, :n] = a
    ap[:, range(n, n + pad), range(n, n + pad)] = 1
    emu = _factor32(ap)[:, :n, :n].astype(np.float64)
    assert np.linalg.norm(got - want) <= 1.1 * np.linalg.norm(emu - want)


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_vbatched_leaves_everything_else(dev, dtype):
    """Bytes outside the lower triangles and the right-hand sides -- the strictly upper triangles, the rows
    from n on of A and of B -- stay as they were, at the edges of tiles, blocks and groups."""
    ns = [1, 15, 16, 17, 48, 63, 64, 65, 127, 128, 129, 177, 193, 255, 256]
    pads = [(3 * i + 1) % 5 for i in range(len(ns))]
    rs = [(1, 16, 17)[i % 3] for i in range(len(ns))]
    vb = batched.VBatch([n + p for n, p in zip(ns, pads)], rs, dtype=dtype, device=dev)
    vb.d_n.copy_(torch.tensor(ns, dtype=torch.int32))
    gen = torch.Generator(device=dev).manual_seed(4)
    vb.a_flat.copy_(torch.randn(vb.a_flat.numel(), device=dev, generator=gen))
    vb.b_flat.copy_(torch.randn(vb.b_flat.numel(), device=dev, generator=gen))
    for i, n in enumerate(ns):
        spd = torch.from_numpy(workloads.gram_spd(n, seed=80 + i)).to(dev).to(dtype)
        vb.A(i)[:n, :n] = torch.where(torch.ones(n, n, device=dev).tril().bool(), spd, vb.A(i)[:n, :n])
    a0, b0 = [vb.A(i).clone() for i in range(len(ns))], [vb.B(i).clone() for i in range(len(ns))]
    assert int(batched.posv_vbatched_(vb, mi_llt.Handle()).abs().sum()) == 0
    for i, n in enumerate(ns):
        keep = torch.ones(n + pads[i], n + pads[i], device=dev).tril().bool()
        keep[n:], keep[:, n:] = False, False  # the system's lower triangle
        assert torch.equal(torch.where(keep, a0[i], vb.A(i)), a0[i]), n
        assert torch.equal(vb.B(i)[n:], b0[i][n:]), n
        assert bool((vb.B(i)[:n] != b0[i][:n]).any()), n
