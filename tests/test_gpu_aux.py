"""GPU parity of the kernels around the update loop (conversion, grouped storage, g-switching error,
RMSE, init, histogram/sort/reindex/shuffle) against the CPU checker, through the C ABI."""
import numpy as np
import pytest

import mfutil
from mfutil import to_dev, from_dev

pytestmark = pytest.mark.gpu


def _sync():
    import torch
    torch.cuda.synchronize()


def test_float2half_exhaustive_halves_and_midpoints(orc):
    """Bit-exact RN-even conversion: every binary16 value, every tie and its neighbours, random floats."""
    import torch
    h = mfutil.hip()
    hb = np.arange(65536, dtype=np.uint16)
    f = hb.view(np.float16).astype(np.float32)
    pos = np.arange(0, 0x7C00, dtype=np.uint16)
    lo = pos.view(np.float16).astype(np.float64)
    hi = (pos + 1).astype(np.uint16).view(np.float16).astype(np.float64)
    hi[-1] = 65536.0
    mid = ((lo + hi) / 2).astype(np.float32)
    rng = np.random.default_rng(1)
    rnd = rng.integers(0, 2 ** 32, 1_000_001, dtype=np.uint64).astype(np.uint32).view(np.float32)   # odd length: tail path
    x = np.concatenate([f[np.isfinite(f)], mid, np.nextafter(mid, np.float32(np.inf)), np.nextafter(mid, np.float32(-np.inf)), -mid, rnd])
    x = x[~np.isnan(x)]
    if x.size % 2 == 0:
        x = x[:-1]
    dx = to_dev(x)
    dout = torch.zeros(x.size + 1, dtype=torch.int16, device="cuda")
    h.mf_transform_float2half(dx.data_ptr(), dout.data_ptr(), x.size, mfutil.stream_ptr())
    _sync()
    got = dout.cpu().numpy().view(np.uint16)[:x.size]
    assert np.array_equal(got, orc.f2h(x))
    with np.errstate(over="ignore"):
        assert np.array_equal(got, x.astype(np.float16).view(np.uint16))


def test_float2half_golden_vectors():
    """The device conversion against tests/golden/half_vectors.npz (numpy float16, see make_half_vectors.py)."""
    import os
    import torch
    h = mfutil.hip()
    g = np.load(os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "half_vectors.npz"))
    x = g["f2h_in"]
    dx = to_dev(x)
    dout = torch.zeros(x.size, dtype=torch.int16, device="cuda")
    h.mf_transform_float2half(dx.data_ptr(), dout.data_ptr(), x.size, mfutil.stream_ptr())
    _sync()
    assert np.array_equal(dout.cpu().numpy().view(np.uint16), g["f2h_out"])


def test_half2float_exhaustive(orc):
    import torch
    h = mfutil.hip()
    hb = np.arange(65535, dtype=np.uint16)     # odd count on purpose
    dx = to_dev(hb)
    dout = torch.zeros(hb.size, dtype=torch.float32, device="cuda")
    h.mf_transform_half2float(dx.data_ptr(), dout.data_ptr(), hb.size, mfutil.stream_ptr())
    _sync()
    got = dout.cpu().numpy()
    want = orc.h2f(hb)
    nan = np.isnan(want)
    assert np.array_equal(got[~nan].view(np.uint32), want[~nan].view(np.uint32))
    assert np.all(np.isnan(got[nan]))


def test_empty_inputs_are_no_ops():
    h = mfutil.hip()
    assert h.mf_transform_float2half(None, None, 0, None) == 0
    assert h.mf_test_rmse(None, 0, None, None, 64, None, None) == 0
    assert h.mf_user_item_histogram(None, 0, None, None, None) == 0
    assert h.mf_sort_by_count(None, None, 0, None) == 0
    assert h.mf_shuffle_ratings(None, None, 0, 1, None) == 0


def test_a_failed_call_leaves_no_error_behind():
    """The runtime keeps the last error until it is asked for it.  A model that no card can hold is refused by hipMalloc, before
    anything is launched; the calls after it, of this library and of torch, must not find that error."""
    import ctypes as C
    import torch
    from importlib import import_module
    MfError = import_module("icdm-2021_mascot_amd.capi").MfError
    h = mfutil.hip()
    node, model, out = np.zeros(1, mfutil.NODE), np.zeros(128, np.float32), C.c_double(0)
    with pytest.raises(MfError, match=r"hipMalloc\(P\)"):
        h.mf_gpu_test_rmse(node.ctypes.data, 1, model.ctypes.data, model.ctypes.data, 0xffffffff, 1, 128, C.addressof(out))
    idx = torch.zeros(100, dtype=torch.int32, device="cuda")
    h.mf_init_idx_arr(idx.data_ptr(), 100, mfutil.stream_ptr())
    assert idx.sum().item() == 4950


def _preprocess_reference(orc, R, n_users, n_items, ug_req, ig_req):
    uc, ic = orc.histogram(R, n_users, n_items)
    suc, sui = orc.sort_by_count(uc)
    sic, sii = orc.sort_by_count(ic)
    uend, iend = orc.grouping(suc, ug_req), orc.grouping(sic, ig_req)
    u2s, u2g, usz = orc.reindex_tables(sui, uend)
    i2s, i2g, isz = orc.reindex_tables(sii, iend)
    return dict(uc=uc, ic=ic, suc=suc, sui=sui, sic=sic, sii=sii, uend=uend, iend=iend, u2s=u2s, u2g=u2g, i2s=i2s, i2g=i2g)


def test_histogram_sort_reindex(orc):
    import torch
    h = mfutil.hip()
    n_users, n_items = 3000, 700
    R = mfutil.make_ratings(5, n_users, n_items, 200_000, alpha=1.0)
    ref = _preprocess_reference(orc, R, n_users, n_items, 20, 10)
    dR = to_dev(R)
    ub = torch.zeros(n_users, dtype=torch.int32, device="cuda")
    ib = torch.zeros(n_items, dtype=torch.int32, device="cuda")
    st = mfutil.stream_ptr()
    h.mf_user_item_histogram(dR.data_ptr(), R.size, ub.data_ptr(), ib.data_ptr(), st)
    _sync()
    assert np.array_equal(ub.cpu().numpy().view(np.uint32), ref["uc"])
    assert np.array_equal(ib.cpu().numpy().view(np.uint32), ref["ic"])
    uidx = torch.zeros(n_users, dtype=torch.int32, device="cuda")
    iidx = torch.zeros(n_items, dtype=torch.int32, device="cuda")
    h.mf_init_idx_arr(uidx.data_ptr(), n_users, st)
    h.mf_init_idx_arr(iidx.data_ptr(), n_items, st)
    h.mf_sort_by_count(ub.data_ptr(), uidx.data_ptr(), n_users, st)
    h.mf_sort_by_count(ib.data_ptr(), iidx.data_ptr(), n_items, st)
    assert np.array_equal(ub.cpu().numpy().view(np.uint32), ref["suc"])
    assert np.array_equal(uidx.cpu().numpy().view(np.uint32), ref["sui"])      # stable: ties keep id order
    assert np.array_equal(iidx.cpu().numpy().view(np.uint32), ref["sii"])
    du2s, di2s = to_dev(ref["u2s"]), to_dev(ref["i2s"])
    h.mf_matrix_reconst_triplet(dR.data_ptr(), du2s.data_ptr(), di2s.data_ptr(), R.size, st)
    _sync()
    want = R.copy()
    orc.lib.orc_reindex(want.ctypes.data, want.size, ref["u2s"].ctypes.data, ref["i2s"].ctypes.data)
    assert np.array_equal(from_dev(dR, np.uint8), want.view(np.uint8).reshape(-1))


@pytest.mark.parametrize("n", [1, 2, 63, 3072, 3073, 4097, 6145, 393217, 786432, 786433, 1572865, 3000001])
def test_shuffle_sizes(orc, n):
    """No partition pass (up to 3072 ratings), one (up to 256 buckets of 3072) and two, at the sizes where the number of
    buckets changes and with tiles and chunks that end early; the permutation is unique, so it has to be the checker's."""
    import torch
    h = mfutil.hip()
    R = np.zeros(n, mfutil.NODE)
    R["r"], R["u"], R["i"] = np.arange(n) % 11, np.arange(n), np.arange(n)[::-1]
    dR, dOut = to_dev(R), torch.full((n * 12,), 0xee, dtype=torch.uint8, device="cuda")
    need = h.mf_shuffle_ratings_workspace_bytes(n)
    ws = torch.full((need,), 0xa5, dtype=torch.uint8, device="cuda")
    for seed in (5, 6):
        h.mf_shuffle_ratings_ws(dR.data_ptr(), dOut.data_ptr(), n, seed, ws.data_ptr(), need, mfutil.stream_ptr())
        torch.cuda.synchronize()
        assert np.array_equal(from_dev(dOut, mfutil.NODE).view(np.uint8), orc.shuffle(seed, R).view(np.uint8))


# 17, 18 and 19 bits of buckets of 3072 ratings: passes of 9 + 8, 9 + 9 and 10 + 9
@pytest.mark.parametrize("n", [(3072 << 16) + 77, (3072 << 17) + 77, (3072 << 18) + 77])
def test_shuffle_beyond_the_large_tiles(n):
    """From 2^16 buckets of 3072 ratings on a pass has more than 8 bits and takes smaller tiles; against torch's sort of the keys."""
    import torch
    h, seed = mfutil.hip(), 9
    R = torch.empty((n, 3), dtype=torch.int32, device="cuda")
    for word in range(3):
        R[:, word] = torch.arange(n, dtype=torch.int32, device="cuda") + word
    out = torch.zeros_like(R)
    need = h.mf_shuffle_ratings_workspace_bytes(n)
    ws = torch.empty(need, dtype=torch.uint8, device="cuda")
    h.mf_shuffle_ratings_ws(R.data_ptr(), out.data_ptr(), n, seed, ws.data_ptr(), need, mfutil.stream_ptr())
    del ws

    def signed(x):
        x &= (1 << 64) - 1
        return x - (1 << 64) if x >> 63 else x

    def shifted(x, by):           # logical shift of 64-bit words held as signed ones
        return (x >> by) & ((1 << (64 - by)) - 1)

    def mix64(x):
        x = x + signed(0x9E3779B97F4A7C15)
        x = (x ^ shifted(x, 30)) * signed(0xBF58476D1CE4E5B9)
        x = (x ^ shifted(x, 27)) * signed(0x94D049BB133111EB)
        return x ^ shifted(x, 31)
    base = mix64(torch.tensor([signed(seed ^ 0x53485546464C4521)], dtype=torch.int64, device="cuda"))
    key = mix64(base ^ torch.arange(n, dtype=torch.int64, device="cuda")) ^ signed(1 << 63)      # unsigned order
    order = torch.argsort(key).to(torch.int32)
    del key
    for word in range(3):
        assert torch.equal(out[:, word], order + word)


def test_shuffle_is_the_checkers_permutation(orc):
    import torch
    h = mfutil.hip()
    R = mfutil.make_ratings(6, 500, 300, 123_457)
    dR = to_dev(R)
    dOut = torch.zeros(R.size * 12, dtype=torch.uint8, device="cuda")
    h.mf_shuffle_ratings(dR.data_ptr(), dOut.data_ptr(), R.size, 77, mfutil.stream_ptr())
    got = from_dev(dOut, mfutil.NODE)
    want = orc.shuffle(77, R)
    assert np.array_equal(got.view(np.uint8), want.view(np.uint8))
    # a permutation of the input, and not the identity
    assert np.array_equal(np.sort(got.view(np.uint8).reshape(-1, 12).view("V12").ravel()), np.sort(R.view("V12").ravel()))
    assert not np.array_equal(got.view(np.uint8), R.view(np.uint8))


def test_init_normal_bit_exact_and_distribution(orc):
    import torch
    from scipy import stats
    h = mfutil.hip()
    n = 1_000_003
    d = torch.zeros(n, dtype=torch.float32, device="cuda")
    h.mf_init_rand_feature(d.data_ptr(), n, 42, 1, mfutil.stream_ptr())
    _sync()
    got = d.cpu().numpy()
    want = orc.init_normal(42, 1, n)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
    # model_init.cu:25: N(0,1) * 0.01
    assert abs(got.mean()) < 5e-5 and abs(got.std() - 0.01) < 5e-5
    assert stats.kstest(got[:200000] / 0.01, "norm").pvalue > 1e-3
    other = orc.init_normal(42, 0, 1000)
    assert not np.array_equal(other, want[:1000])


@pytest.mark.parametrize("k", [64, 128])
def test_scatter_gather_rmse_grouped(orc, k):
    import torch
    h = mfutil.hip()
    st = mfutil.stream_ptr()
    n_users, n_items = 900, 400
    R = mfutil.make_ratings(7 + k, n_users, n_items, 60_000)
    test = mfutil.make_ratings(8 + k, n_users, n_items, 10_001)
    ref = _preprocess_reference(orc, R, n_users, n_items, 12, 9)
    P = orc.init_normal(1, 0, n_users * k).reshape(n_users, k) * 10
    Q = orc.init_normal(1, 1, n_items * k).reshape(n_items, k) * 10
    # dense RMSE in original id space
    dT, dP, dQ = to_dev(test), to_dev(P), to_dev(Q)
    acc = torch.zeros(1, dtype=torch.float64, device="cuda")
    h.mf_test_rmse(dT.data_ptr(), test.size, dP.data_ptr(), dQ.data_ptr(), k, acc.data_ptr(), st)
    _sync()
    rm = float(np.sqrt(acc.cpu().numpy()[0] / test.size))
    assert abs(rm - orc.rmse(k, test, P, Q)) <= 1e-6 * rm
    # scatter rows into grouped binary16 storage (model_init.cu:30-56)
    sizes_u = np.diff(np.concatenate([[-1], ref["uend"].astype(np.int64)]))
    sizes_i = np.diff(np.concatenate([[-1], ref["iend"].astype(np.int64)]))
    gu = orc_grouped_zero(k, ref["uend"], sizes_u)
    gi = orc_grouped_zero(k, ref["iend"], sizes_i)
    du, di = mfutil.DeviceGrouped(gu), mfutil.DeviceGrouped(gi)
    d_u2g, d_u2s, d_i2g, d_i2s = to_dev(ref["u2g"]), to_dev(ref["u2s"]), to_dev(ref["i2g"]), to_dev(ref["i2s"])
    h.mf_cpyparams2grouped_params(dP.data_ptr(), du.ptrs.data_ptr(), du.end.data_ptr(), d_u2g.data_ptr(), d_u2s.data_ptr(), k, n_users, du.groups, st)
    h.mf_cpyparams2grouped_params(dQ.data_ptr(), di.ptrs.data_ptr(), di.end.data_ptr(), d_i2g.data_ptr(), d_i2s.data_ptr(), k, n_items, di.groups, st)
    _sync()
    Ps = np.empty_like(P); Ps[ref["u2s"]] = P          # rows in sorted order
    Qs = np.empty_like(Q); Qs[ref["i2s"]] = Q
    want_u = mfutil.host_grouped(orc, k, Ps, ref["uend"], np.zeros(du.groups, np.uint8))
    want_i = mfutil.host_grouped(orc, k, Qs, ref["iend"], np.zeros(di.groups, np.uint8))
    for got, want in zip(du.download() + di.download(), want_u.arrays + want_i.arrays):
        assert np.array_equal(got, want)
    # gather back to dense (sorted order), widening exactly
    dense = torch.zeros(n_users * k, dtype=torch.float32, device="cuda")
    h.mf_grouped_params2dense(du.ptrs.data_ptr(), du.end.data_ptr(), du.prec.data_ptr(), dense.data_ptr(), k, n_users, du.groups, st)
    _sync()
    assert np.array_equal(dense.cpu().numpy().reshape(n_users, k), orc.h2f(orc.f2h(Ps)))
    # RMSE straight from grouped storage on the re-indexed test set
    tr = test.copy()
    orc.lib.orc_reindex(tr.ctypes.data, tr.size, ref["u2s"].ctypes.data, ref["i2s"].ctypes.data)
    dTr = to_dev(tr)
    acc.zero_()
    h.mf_test_rmse_grouped(dTr.data_ptr(), tr.size, du.ptrs.data_ptr(), di.ptrs.data_ptr(), k, du.end.data_ptr(), di.end.data_ptr(),
                           du.prec.data_ptr(), di.prec.data_ptr(), du.groups, di.groups, acc.data_ptr(), st)
    _sync()
    rm_g = float(np.sqrt(acc.cpu().numpy()[0] / tr.size))
    want_g = orc.lib.orc_rmse_grouped(k, tr.ctypes.data, tr.size, want_u.ptrs, want_i.ptrs, want_u.end_idx.ctypes.data, want_i.end_idx.ctypes.data,
                                      want_u.prec.ctypes.data, want_i.prec.ctypes.data, want_u.groups, want_i.groups)
    assert abs(rm_g - want_g) <= 1e-6 * want_g
    assert abs(rm_g - rm) < 5e-3        # binary16 storage of the same model: close to the fp32 figure


def orc_grouped_zero(k, end_idx, sizes):
    from oracle import oracle as om
    arrays = [np.zeros(int(s) * k, np.uint16) for s in sizes]
    return om.GroupedModel(k, end_idx, np.zeros(len(sizes), np.uint8), arrays)


@pytest.mark.parametrize("k", [64, 128])
def test_group_error_matches_host_formula(orc, k):
    import torch
    h = mfutil.hip()
    rng = np.random.default_rng(9)
    G, nb = 37, 513
    gs = rng.standard_normal(G * k).astype(np.float32) * 3
    ns = rng.random(G * nb).astype(np.float32)
    prec = (rng.random(G) < 0.3).astype(np.uint8)
    init = (rng.random(G).astype(np.float32) + 0.5)
    want = np.zeros(G, np.float32)
    orc.lib.orc_group_error(k, G, gs.ctypes.data, ns.ctypes.data, nb, prec.ctypes.data, init.ctypes.data, want.ctypes.data)
    dgs, dns, dpr, din = to_dev(gs), to_dev(ns), to_dev(prec), to_dev(init)
    out = torch.zeros(G, dtype=torch.float32, device="cuda")
    h.mf_group_error(dgs.data_ptr(), dns.data_ptr(), nb, dpr.data_ptr(), din.data_ptr(), out.data_ptr(), k, G, mfutil.stream_ptr())
    _sync()
    got = out.cpu().numpy()
    assert np.array_equal(got[prec == 1], np.full(int(prec.sum()), -1, np.float32))
    assert np.allclose(got[prec == 0], want[prec == 0], rtol=1e-5)
    # the accumulators of binary16 groups are cleared for the next check epoch (mf_methods.cu:333)
    left = from_dev(dgs, np.float32).reshape(G, k)
    assert np.all(left[prec == 0] == 0)


@pytest.mark.parametrize("row_bytes", [128, 256, 512])
@pytest.mark.parametrize("coherent", [0, 1])
def test_row_traffic_probe_leaves_rows_unchanged(row_bytes, coherent):
    """The access-pattern probe reads the two rows of every rating and writes kept ones back as they are."""
    import torch
    h = mfutil.hip()
    rng = np.random.default_rng(row_bytes + coherent)
    n_users, n_items, n = 300, 70, 20_001
    R = np.zeros(n, mfutil.NODE)
    R["u"] = rng.integers(0, n_users, n); R["i"] = rng.integers(0, n_items, n); R["r"] = 1.0
    P = rng.integers(0, 256, n_users * row_bytes, dtype=np.uint8)
    Q = rng.integers(0, 256, n_items * row_bytes, dtype=np.uint8)
    ku = rng.choice(np.array([0, 100, 252, 253, 254, 255], np.uint8), n_users)
    kv = rng.choice(np.array([0, 100, 252, 253, 254, 255], np.uint8), n_items)
    dR, dP, dQ = to_dev(R), to_dev(P), to_dev(Q)
    k = row_bytes // 2
    plain = mfutil.HogwildOptions(k if k <= 128 else 128, cached_rows=1 - coherent)
    tables = mfutil.HogwildOptions(k if k <= 128 else 128, ku, kv, cached_rows=1 - coherent)
    for opt in (plain, tables):
        for workers in (1, 7, 4096):
            h.mf_row_traffic_probe(dR.data_ptr(), n, dP.data_ptr(), dQ.data_ptr(), row_bytes, workers, 5, mfutil.stream_ptr(), opt.ptr)
    h.mf_row_traffic_probe(dR.data_ptr(), n, dP.data_ptr(), dQ.data_ptr(), row_bytes, 64, 5, mfutil.stream_ptr(), None)
    torch.cuda.synchronize()
    assert np.array_equal(from_dev(dP, np.uint8), P) and np.array_equal(from_dev(dQ, np.uint8), Q)
    from importlib import import_module
    MfError = import_module("icdm-2021_mascot_amd.capi").MfError
    with pytest.raises(MfError, match="row_bytes must be"):
        h.mf_row_traffic_probe(dR.data_ptr(), n, dP.data_ptr(), dQ.data_ptr(), 64, 4, 5, mfutil.stream_ptr(), None)
    tables.o.item_keep = None
    with pytest.raises(MfError, match="both keep tables"):
        h.mf_row_traffic_probe(dR.data_ptr(), n, dP.data_ptr(), dQ.data_ptr(), row_bytes, 4, 5, mfutil.stream_ptr(), tables.ptr)
    h.mf_row_traffic_probe(None, 0, None, None, row_bytes, 4, 5, mfutil.stream_ptr(), None)      # nothing to do


@pytest.mark.parametrize("config", [1, 4, 5])
def test_generated_ratings_match_the_checker(orc, config):
    """mf_generate_ratings against its CPU twin, bit for bit, on scaled-down BASELINE configurations; any range of the
    stream can be generated on its own."""
    import torch
    from oracle import oracle as om
    h = mfutil.hip()
    c = h.synth_config(config)
    if config != 1:                      # keep the checker's tables small
        c.n_users, c.n_items = 30_000, 4_000
    n = 150_000
    want = orc.generate_ratings(c, 11, 0, n)
    out = torch.empty(n * 12, dtype=torch.uint8, device="cuda")
    import ctypes as C
    h.mf_generate_ratings(C.addressof(c), 11, 0, n, out.data_ptr(), mfutil.stream_ptr())
    got = from_dev(out, mfutil.NODE)
    assert np.array_equal(got.view(np.uint8), want.view(np.uint8))
    part = torch.empty(1000 * 12, dtype=torch.uint8, device="cuda")
    h.mf_generate_ratings(C.addressof(c), 11, 77_777, 1000, part.data_ptr(), mfutil.stream_ptr())
    assert np.array_equal(from_dev(part, mfutil.NODE).view(np.uint8), want[77_777:78_777].view(np.uint8))
    host = np.empty(500, mfutil.NODE)
    h.mf_generate_ratings_host(C.addressof(c), 11, 10, 500, host.ctypes.data)
    assert np.array_equal(host.view(np.uint8), want[10:510].view(np.uint8))


def test_workspace_forms_equal_the_allocating_forms(orc):
    """mf_sort_by_count_ws, mf_shuffle_ratings_ws and mf_generate_ratings_ws with caller-owned workspaces of exactly the
    size their queries return give what the forms that allocate for themselves give; a workspace that is too small or
    misaligned is refused before anything is launched."""
    import ctypes as C
    import torch
    from importlib import import_module
    MfError = import_module("icdm-2021_mascot_amd.capi").MfError
    h = mfutil.hip()
    st = mfutil.stream_ptr()
    rng = np.random.default_rng(5)
    for n in (1, 777, 300_001):
        cnt = rng.integers(0, 50, n).astype(np.uint32)
        a_cnt, b_cnt = to_dev(cnt), to_dev(cnt)
        a_idx, b_idx = torch.arange(n, dtype=torch.int32, device="cuda"), torch.arange(n, dtype=torch.int32, device="cuda")
        h.mf_sort_by_count(a_cnt.data_ptr(), a_idx.data_ptr(), n, st)
        need = h.mf_sort_by_count_workspace_bytes(n)
        assert need >= 8 * n
        ws = torch.full((need,), 0x5A, dtype=torch.uint8, device="cuda")
        h.mf_sort_by_count_ws(b_cnt.data_ptr(), b_idx.data_ptr(), n, ws.data_ptr(), need, st)
        torch.cuda.synchronize()
        assert torch.equal(a_cnt, b_cnt) and torch.equal(a_idx, b_idx)
        order = np.argsort(cnt, kind="stable")
        assert np.array_equal(from_dev(b_idx, np.uint32), order.astype(np.uint32))
        with pytest.raises(MfError, match="need"):
            h.mf_sort_by_count_ws(b_cnt.data_ptr(), b_idx.data_ptr(), n, ws.data_ptr(), need - 1, st)
        if need > 512:
            with pytest.raises(MfError, match="256-byte aligned"):
                h.mf_sort_by_count_ws(b_cnt.data_ptr(), b_idx.data_ptr(), n, ws.data_ptr() + 4, need - 256, st)
        # shuffle
        R = np.zeros(n, mfutil.NODE)
        R["u"], R["i"], R["r"] = np.arange(n), rng.integers(0, 1000, n), rng.integers(1, 6, n)
        dR = to_dev(R)
        o1, o2 = torch.empty_like(dR), torch.empty_like(dR)
        h.mf_shuffle_ratings(dR.data_ptr(), o1.data_ptr(), n, 42, st)
        need = h.mf_shuffle_ratings_workspace_bytes(n)
        ws = torch.full((need,), 0xA5, dtype=torch.uint8, device="cuda")
        h.mf_shuffle_ratings_ws(dR.data_ptr(), o2.data_ptr(), n, 42, ws.data_ptr(), need, st)
        torch.cuda.synchronize()
        assert torch.equal(o1, o2)
        assert np.array_equal(from_dev(o2, mfutil.NODE).view(np.uint8), orc.shuffle(42, R).view(np.uint8))
        with pytest.raises(MfError, match="need"):
            h.mf_shuffle_ratings_ws(dR.data_ptr(), o2.data_ptr(), n, 42, ws.data_ptr(), need - 1, st)
    # generator: tables once, any range afterwards without allocation or synchronisation
    for config in (1, 5):
        c = h.synth_config(config)
        c.n_users, c.n_items = 3000, 700
        need = h.mf_synth_tables_bytes(C.addressof(c))
        assert need >= 12 * 3700
        tables = torch.full((need,), 0x33, dtype=torch.uint8, device="cuda")
        h.mf_synth_build_tables(C.addressof(c), 9, tables.data_ptr(), need, st)
        want = orc.generate_ratings(c, 9, 0, 50_000)
        for first, count in ((0, 50_000), (12_345, 1_000), (49_999, 1)):
            out = torch.empty(count * 12, dtype=torch.uint8, device="cuda")
            h.mf_generate_ratings_ws(C.addressof(c), 9, tables.data_ptr(), first, count, out.data_ptr(), st)
            assert np.array_equal(from_dev(out, mfutil.NODE).view(np.uint8), want[first:first + count].view(np.uint8))
        with pytest.raises(MfError, match="need"):
            h.mf_synth_build_tables(C.addressof(c), 9, tables.data_ptr(), need - 1, st)


# up to 131072 ratings a table per workgroup; above, ids in several ranges of 80896 and (the last two of more than a million ids) in too many
@pytest.mark.parametrize("n,n_users,n_items,hot", [(1, 1, 1, False), (63, 80895, 1, False), (16385, 80896, 80897, False), (70_001, 3, 90_000, True),
                                                   (300_007, 161_793, 161_000, True), (900_001, 3_000_000, 700_000, True), (500_001, 1_000_000, 200_000, True), (400_003, 10, 5_000_000, False)])
def test_histogram_reindex_ranges(n, n_users, n_items, hot):
    import torch
    h = mfutil.hip()
    rng = np.random.default_rng(n)
    R = np.zeros(n, mfutil.NODE)
    R["u"], R["i"], R["r"] = rng.integers(0, n_users, n), rng.integers(0, n_items, n), rng.random(n)
    if hot:
        R["u"][rng.random(n) < 0.6] = n_users - 1
        R["i"][rng.random(n) < 0.3] = n_items // 2
    ub = torch.full((n_users,), 7, dtype=torch.int32, device="cuda")       # counts are added to what is there
    ib = torch.zeros(n_items, dtype=torch.int32, device="cuda")
    dR = to_dev(R)
    h.mf_user_item_histogram(dR.data_ptr(), n, ub.data_ptr(), ib.data_ptr(), mfutil.stream_ptr())
    u2s, i2s = rng.permutation(n_users).astype(np.uint32), rng.permutation(n_items).astype(np.uint32)
    d_u2s, d_i2s = to_dev(u2s), to_dev(i2s)
    h.mf_matrix_reconst_triplet(dR.data_ptr(), d_u2s.data_ptr(), d_i2s.data_ptr(), n, mfutil.stream_ptr())
    _sync()
    assert np.array_equal(ub.cpu().numpy(), np.bincount(R["u"], minlength=n_users) + 7)
    assert np.array_equal(ib.cpu().numpy(), np.bincount(R["i"], minlength=n_items))
    got = from_dev(dR, mfutil.NODE)
    assert np.array_equal(got["r"], R["r"]) and np.array_equal(got["u"], u2s[R["u"]]) and np.array_equal(got["i"], i2s[R["i"]])


# up to 786432 fours of words one per lane, then four; with the remainders of a four on both sides, and several rounds per lane
@pytest.mark.parametrize("n", [1_048_575, 1_048_576, 1_048_577, 1_048_578, 1_048_579, 22_369_622])
def test_reindex_sizes(n):
    import torch
    h = mfutil.hip()
    g = torch.Generator(device="cuda").manual_seed(n)
    n_users, n_items = 300_007, 5_003
    R = torch.randint(-2 ** 31, 2 ** 31 - 1, (n + 1, 3), generator=g, device="cuda", dtype=torch.int64).int()
    for word, ids in ((1, n_users), (2, n_items)):
        R[:, word] = torch.randint(0, ids, (n + 1,), generator=g, device="cuda")
    before = R.clone()
    to_user = torch.randperm(n_users, generator=g, device="cuda").int()
    to_item = torch.randperm(n_items, generator=g, device="cuda").int()
    h.mf_matrix_reconst_triplet(R.data_ptr(), to_user.data_ptr(), to_item.data_ptr(), n, mfutil.stream_ptr())
    assert torch.equal(R[n], before[n]) and torch.equal(R[:n, 0], before[:n, 0])
    assert torch.equal(R[:n, 1], to_user[before[:n, 1].long()]) and torch.equal(R[:n, 2], to_item[before[:n, 2].long()])


# Both sides of every line of the choice: table or ranges by the number of ratings; 21 and 32 ranges of which few ids make up most
# of the ratings or not; one range too many; users and items sharing a range (1 and 16 ranges) or not (2 and 17).
@pytest.mark.parametrize("n,n_users,n_items,share", [(131072, 480_000, 17_800, 0.0), (131073, 480_000, 17_800, 0.0), (131073, 480_000, 17_800, 0.9),
                                                     (524_287, 1_000_000, 625_000, 0.0), (524_288, 1_000_000, 625_000, 0.0), (524_288, 1_000_000, 625_000, 0.9), (600_001, 2_500_000, 80_896, 0.0),
                                                     (600_001, 2_500_000, 80_896, 0.9), (600_001, 2_588_672, 80_896, 0.0), (140_001, 70_000, 10_700, 0.3),
                                                     (140_001, 80_896, 10_700, 0.3), (140_001, 1_250_000, 44_000, 0.3), (600_001, 1_200_000, 161_000, 0.3)])
def test_histogram_choice(n, n_users, n_items, share):
    import torch
    h = mfutil.hip()
    g = torch.Generator(device="cuda").manual_seed(n + n_users)
    R = torch.zeros((n, 3), dtype=torch.int32, device="cuda")
    for word, ids in ((1, n_users), (2, n_items)):
        R[:, word] = torch.randint(0, ids, (n,), generator=g, device="cuda")
        popular = torch.rand(n, generator=g, device="cuda") < share
        R[:, word][popular] = torch.randint(ids - min(ids, 100), ids, (n,), generator=g, device="cuda", dtype=torch.int32)[popular]
        R[0, word] = ids - 1            # among the sampled ratings: the reach is known
    ub, ib = torch.full((n_users,), 7, dtype=torch.int32, device="cuda"), torch.zeros(n_items, dtype=torch.int32, device="cuda")
    h.mf_user_item_histogram(R.data_ptr(), n, ub.data_ptr(), ib.data_ptr(), mfutil.stream_ptr())
    assert torch.equal(ub.long(), torch.bincount(R[:, 1], minlength=n_users) + 7)
    assert torch.equal(ib.long(), torch.bincount(R[:, 2], minlength=n_items))


# A range's counters are 16 bits wide, ids x and x + 40448 of a range in one word: ids that pass 2^15 at least twice in every chunk of the
# ratings, in either half of a word, of users, of items, and of items that share a range with users
@pytest.mark.parametrize("n,chunks,n_users,n_items,user,item", [(3_000_001, 16, 1_000_000, 200_000, 5 * 80896 + 100, 80896 + 17),
                                                                (3_000_001, 16, 1_000_000, 200_000, 5 * 80896 + 40448 + 7, 80896 + 50_000),
                                                                (3_000_001, 16, 1_000_000, 200_000, 999_999, 199_999),
                                                                (25_000_003, 256, 70_000, 10_700, 5, 10_699), (25_000_003, 256, 70_000, 10_700, 69_999, 0)])
def test_histogram_counters_move_to_memory(n, chunks, n_users, n_items, user, item):
    import torch
    h = mfutil.hip()
    g = torch.Generator(device="cuda").manual_seed(n + user)
    R = torch.zeros((n, 3), dtype=torch.int32, device="cuda")
    for word, ids, hot in ((1, n_users, user), (2, n_items, item)):
        R[:, word] = torch.randint(0, ids, (n,), generator=g, device="cuda")
        R[:, word][torch.rand(n, generator=g, device="cuda") < 0.8] = hot
        per_chunk = (R[:, word] == hot).long().cumsum(0)[[n * (c + 1) // chunks - 1 for c in range(chunks)]].diff()
        assert int(per_chunk.min()) > 2 << 15
    ub, ib = torch.zeros(n_users, dtype=torch.int32, device="cuda"), torch.zeros(n_items, dtype=torch.int32, device="cuda")
    h.mf_user_item_histogram(R.data_ptr(), n, ub.data_ptr(), ib.data_ptr(), mfutil.stream_ptr())
    assert torch.equal(ub.long(), torch.bincount(R[:, 1], minlength=n_users))
    assert torch.equal(ib.long(), torch.bincount(R[:, 2], minlength=n_items))


# four rows of k = 128 per wavefront up to 24576, sixteen above, with remainders; groups of both precisions, and rows behind the last group
@pytest.mark.parametrize("k", [64, 128])
@pytest.mark.parametrize("rows", [3, 24575, 24576, 24577, 24593])
def test_gather_rows(k, rows):
    import torch
    h = mfutil.hip()
    g = torch.Generator(device="cuda").manual_seed(rows + k)
    end = sorted({min(rows - 1, x) for x in (0, 1, 6, 1000, 1001, 20_000, rows - 3, rows - 2)})      # the last row is in no group
    dense = (torch.randn((rows, k), generator=g, device="cuda") * 0.3).half().float()
    ptr, keep, first = [], [], 0
    for i, last in enumerate(end):
        part = dense[first:last + 1].half() if i % 2 else dense[first:last + 1].clone()
        keep.append(part)
        ptr.append(part.data_ptr())
        first = last + 1
    d_ptr, d_end = torch.tensor(ptr, dtype=torch.int64, device="cuda"), torch.tensor(end, dtype=torch.int32, device="cuda")
    prec = torch.tensor([1 - i % 2 for i in range(len(end))], dtype=torch.uint8, device="cuda")
    out = torch.full((rows + 1, k), 9.0, device="cuda")
    h.mf_grouped_params2dense(d_ptr.data_ptr(), d_end.data_ptr(), prec.data_ptr(), out.data_ptr(), k, rows, len(end), mfutil.stream_ptr())
    assert torch.equal(out[:end[-1] + 1], dense[:end[-1] + 1]) and bool((out[end[-1] + 1:] == 9.0).all())


# remainders of 64 ratings (and of a wavefront's four batches of 16) and of the 16 rows a wavefront moves, rows at odd alignments, both precisions in every combination,
# ratings of ids in no group; the sums in binary64 on the host from the same rows (a binary32 dot of k products is off by k / 2^24
# of the sum of their sizes at most)
@pytest.mark.parametrize("k", [64, 128])
@pytest.mark.parametrize("test_n", [1, 4, 5, 13, 17, 37, 63, 64, 65, 16 * 64 + 17, 40_003])
def test_rmse_gather_mixed_rows(k, test_n):
    import torch
    h = mfutil.hip()
    st = mfutil.stream_ptr()
    rng = np.random.default_rng(k + test_n)
    sides = []
    for end, prec in (([0, 4, 36, 100, 116], [1, 0, 1, 0, 0]), ([6, 7, 50], [0, 1, 0])):
        rows = end[-1] + 1
        dense = (rng.standard_normal((rows, k)) * 0.3).astype(np.float32)
        arena = torch.zeros(rows * k * 4 + 64 * len(end), dtype=torch.uint8, device="cuda")
        at, ptr, first = 0, [], 0
        for g, (last, single) in enumerate(zip(end, prec)):
            at = (at + 15) // 16 * 16 + (4 if single else 2 * (g % 3))      # aligned to elements only
            part = dense[first:last + 1] if single else dense[first:last + 1].astype(np.float16)
            dense[first:last + 1] = part
            raw = torch.from_numpy(part.reshape(-1).view(np.uint8).copy()).cuda()
            arena[at:at + raw.numel()] = raw
            ptr.append(arena.data_ptr() + at)
            at += raw.numel()
            first = last + 1
        d = dict(dense=dense, arena=arena, groups=len(end), ptr=torch.tensor(ptr, dtype=torch.int64, device="cuda"),
                 end=torch.tensor(end, dtype=torch.int32, device="cuda"), prec=torch.tensor(prec, dtype=torch.uint8, device="cuda"))
        out = torch.full(((rows + 1) * k,), 9.0, dtype=torch.float32, device="cuda")
        h.mf_grouped_params2dense(d["ptr"].data_ptr(), d["end"].data_ptr(), d["prec"].data_ptr(), out.data_ptr(), k, rows, len(end), st)
        _sync()
        assert np.array_equal(out[:rows * k].cpu().numpy().reshape(rows, k), dense) and bool((out[rows * k:] == 9.0).all())
        sides.append(d)
    U, I = sides
    T = np.zeros(test_n, mfutil.NODE)
    T["u"], T["i"], T["r"] = rng.integers(0, U["dense"].shape[0], test_n), rng.integers(0, I["dense"].shape[0], test_n), rng.random(test_n) * 4 + 1
    acc = torch.zeros(1, dtype=torch.float64, device="cuda")
    for outside in (False, True):
        if outside:
            T["u"][::3] = U["dense"].shape[0] + 5
        ok = T["u"] < U["dense"].shape[0]
        P, Q = U["dense"][np.where(ok, T["u"], 0)].astype(np.float64), I["dense"][T["i"]].astype(np.float64)
        err = np.where(ok, T["r"].astype(np.float64) - (P * Q).sum(1), 0.0)
        bound = (2 * np.abs(err) * (np.abs(P * Q).sum(1) * k + 8) * 2.0 ** -24).sum() + 1e-12
        dT = to_dev(T)
        acc.zero_()
        h.mf_test_rmse_grouped(dT.data_ptr(), test_n, U["ptr"].data_ptr(), I["ptr"].data_ptr(), k, U["end"].data_ptr(), I["end"].data_ptr(), U["prec"].data_ptr(), I["prec"].data_ptr(),
                               U["groups"], I["groups"], acc.data_ptr(), st)
        assert abs(float(acc) - (err ** 2).sum()) <= bound
        if not outside:
            dP, dQ = to_dev(U["dense"]), to_dev(I["dense"])
            acc.zero_()
            h.mf_test_rmse(dT.data_ptr(), test_n, dP.data_ptr(), dQ.data_ptr(), k, acc.data_ptr(), st)
            assert abs(float(acc) - (err ** 2).sum()) <= bound
