"""Gridding and degridding at the edges of tiles, batches and work items,
against the oracle's restatement of WStackingGridder<float> on the same
samples. Tolerances as for the other parity tests (relative L2: 1e-5 for the
reference precision, 3e-5 for the mixed one; the oracle's own float-double
spread is about 1e-6).

- Sizes that 16 does not divide take 16 x 16 uv tiles with a cut last tile
  where that holds K - 1 cells (12 at 60, 8 at 56, 72 and 120); 84 and 36 leave 4
  and keep a tile that divides them.
- A work item's records are gridded 64 at a time, a bin's in items of
  work_chunk, with the next batch loaded ahead: counts about both.
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

C_LIGHT = 299792458.0
TOL = {"reference": 1e-5, "mixed": 3e-5}


def rel(a, b):
    a, b = np.asarray(a, np.complex128).ravel(), np.asarray(b, np.complex128).ravel()
    return np.linalg.norm(a - b) / np.linalg.norm(b)


def both_ways(oracle, w, h, dl, uvw, wl, vis, nw, K, precision, chunk=0):
    """Invert and predict on the device and by the oracle; compared."""
    import wsclean_amd
    dev = torch.device("cuda:0")
    uvw_l = (uvw[:, None, :] / wl[None, :, None]).reshape(-1, 3)
    maxw = float(np.abs(uvw_l[:, 2]).max())
    ref = oracle.RefGridder(w, h, dl, dl, 1, K, 63, "float")
    ref.prepare_w_layers(nw, 1e12, 0.0, maxw)
    ref.start_inversion_pass(0)
    ref.add_samples(uvw_l, vis.reshape(-1))
    ref.finish_inversion_pass()
    ref.finalize_image(1.0)
    want = ref.image()
    model = np.random.default_rng(w + h).standard_normal((h, w)).astype(np.float32)
    pred = oracle.RefGridder(w, h, dl, dl, 1, K, 63, "float")
    pred.prepare_w_layers(nw, 1e12, 0.0, maxw)
    pred.initialize_prediction(model)
    pred.start_prediction_pass(0)
    want_v = pred.sample(uvw_l)

    g = wsclean_amd.DeviceGridder(w, h, dl, dl, K, 63, precision=precision, work_chunk=chunk)
    g.prepare_w_layers(nw, 0.0, maxw)
    d_vis = torch.from_numpy(vis).to(dev)
    g.plan(torch.from_numpy(uvw).to(dev), torch.from_numpy(wl).to(dev))
    img = torch.zeros((1, h, w), dtype=torch.float32, device=dev)
    g.invert(d_vis, 1.0, img)
    out = torch.empty_like(d_vis)
    g.predict(torch.from_numpy(model).to(dev)[None], None, out)
    g.synchronize()
    stats = g.stats()
    g.close()
    assert rel(img.cpu().numpy()[0], want) < TOL[precision]
    got = out.cpu().numpy().reshape(-1)
    ok = np.isfinite(want_v)
    assert np.array_equal(ok, np.isfinite(got)) and ok.any()
    assert rel(got[ok], want_v[ok]) < TOL[precision]
    return stats


@pytest.mark.parametrize("precision", ["reference", "mixed"])
@pytest.mark.parametrize("w,h,K,tiles", [(60, 60, 7, 16), (56, 72, 7, 20), (72, 56, 9, 20),
                                         (120, 60, 7, 32), (84, 84, 7, 49), (36, 60, 7, 15)])
def test_cut_tiles_match_oracle(oracle, w, h, K, tiles, precision):
    rng = np.random.default_rng(w * 7 + h)
    dl = 0.004
    wl = C_LIGHT / np.linspace(120e6, 150e6, 4)
    # the whole uv plane, so that footprints lie across every tile edge and
    # wrap round both axes
    umax = 0.499 / dl * wl.min()
    uvw = np.column_stack([rng.uniform(-umax, umax, 700), rng.uniform(-umax, umax, 700),
                           rng.uniform(-40, 40, 700)])
    vis = (rng.standard_normal((700, 4, 1)) + 1j * rng.standard_normal((700, 4, 1))
           ).astype(np.complex64)
    s = both_ways(oracle, w, h, dl, uvw, wl, vis, 3, K, precision)
    assert s["tiles_total"] == 3 * tiles
    # and with bins split into several items, summed from partial tiles
    s = both_ways(oracle, w, h, dl, uvw, wl, vis, 1, K, precision, chunk=16)
    assert s["chunks"] > s["bins_used"]


@pytest.mark.parametrize("precision", ["reference", "mixed"])
@pytest.mark.parametrize("n,chunk", [(1, 0), (63, 0), (64, 0), (65, 0), (129, 64), (257, 64),
                                     (1024, 0), (1025, 0), (4097, 100)])
def test_records_about_batches_and_items(oracle, n, chunk, precision):
    rng = np.random.default_rng(n)
    w, dl = 64, 0.004
    wl = C_LIGHT / np.array([140e6])
    # every sample in one uv cell (one bin, plus its neighbours' halves)
    uvw = np.column_stack([rng.uniform(-2, 2, n) + 30.0, rng.uniform(-2, 2, n) - 20.0,
                           rng.uniform(5, 30, n)])
    vis = (rng.standard_normal((n, 1, 1)) + 1j * rng.standard_normal((n, 1, 1))
           ).astype(np.complex64)
    both_ways(oracle, w, w, dl, uvw, wl, vis, 2, 7, precision, chunk)


@pytest.mark.parametrize("w,precision", [(60, "reference"), (60, "mixed"), (64, "reference"),
                                         (64, "mixed")])
def test_sums_of_dense_bins_keep_their_precision(oracle, w, precision):
    """Work items of 8192 records of noise about one uv cell in each of sixteen
    tiles, against the 64-bit oracle. The batches of 64 are summed on their own
    and then added, so that a cell's error is that of two short sums: with FP32
    roundings of at most u = 2^-24 / sqrt(3) rms and the partial sums of noise
    growing as sqrt(k), n additions leave u sqrt(n / 2), that is 5.7 u within a
    batch and 8 u over the 128 batches, and the kernel values and products 2 u:
    10 u = 3.4e-7, and half as much again for the scatter of sixteen sums
    (measured: 2.2e-7 to 3.1e-7; a running sum of the 2048 matrix products, 32 u
    and more: 1.5e-6 to 2.2e-6)."""
    import wsclean_amd
    rng = np.random.default_rng(w)
    n, dl = 8192, 0.004
    wl = C_LIGHT / np.array([140e6])
    # footprints of 7 cells about these lie inside one tile
    at = np.repeat(np.array([(x, y) for x in (8, 24, -20, -8) for y in (8, 24, -20, -8)]), n, 0)
    uvw = np.column_stack([(at + rng.uniform(-0.4, 0.4, at.shape)) * wl[0] / (w * dl),
                           rng.uniform(1, 2, len(at))])
    vis = (rng.standard_normal((len(at), 1, 1)) + 1j * rng.standard_normal((len(at), 1, 1))
           ).astype(np.complex64)
    uvw_l = (uvw[:, None, :] / wl[None, :, None]).reshape(-1, 3)
    maxw = float(uvw_l[:, 2].max())
    ref = oracle.RefGridder(w, w, dl, dl, 1, 7, 63, "double")
    ref.prepare_w_layers(1, 1e12, 0.0, maxw)
    ref.start_inversion_pass(0)
    ref.add_samples(uvw_l, vis.reshape(-1))
    g = wsclean_amd.WStackingGridder(w, w, dl, dl, 7, 63, precision=precision, work_chunk=n)
    g.prepare_w_layers(1, 0.0, 0.0, maxw)
    g.start_inversion_pass(0)
    g.add_data(uvw, wl, vis)
    e = rel(g.get_gridded_uv_layer(0, image=0), ref.layer(0))
    g.close()
    print(f"{w} {precision}: {e:.2e}")
    assert e < 15 * 2.0 ** -24 / np.sqrt(3.0)


@pytest.mark.parametrize("K", [1, 3, 5, 7, 9, 11, 13, 15])
@pytest.mark.parametrize("w,h", [(120, 60), (64, 96)])
def test_degridding_of_one_to_four_images(oracle, w, h, K):
    """The kernel sizes and image counts of the degridding kernel, footprints
    about every tile edge (120 x 60 has cut tiles up to K = 9)."""
    import wsclean_amd
    dev = torch.device("cuda:0")
    rng = np.random.default_rng(w + K)
    dl, nw = 0.003, 2
    wl = C_LIGHT / np.array([120e6, 150e6])
    umax = 0.45 / dl * wl.min()
    uvw = np.column_stack([rng.uniform(-umax, umax, 500), rng.uniform(-umax, umax, 500),
                           rng.uniform(-30, 30, 500)])
    uvw_l = (uvw[:, None, :] / wl[None, :, None]).reshape(-1, 3)
    maxw = float(np.abs(uvw_l[:, 2]).max())
    model = rng.standard_normal((4, h, w)).astype(np.float32)
    want = []
    for m in model:
        o = oracle.RefGridder(w, h, dl, dl, 1, K, 63, "float")
        o.prepare_w_layers(nw, 1e12, 0.0, maxw)
        o.initialize_prediction(m)
        o.start_prediction_pass(0)
        want.append(o.sample(uvw_l))
    d_uvw, d_wl = torch.from_numpy(uvw).to(dev), torch.from_numpy(wl).to(dev)
    for n in (1, 2, 3, 4):
        g = wsclean_amd.DeviceGridder(w, h, dl, dl, K, 63, precision="reference", n_images=n)
        g.prepare_w_layers(nw, 0.0, maxw)
        g.plan(d_uvw, d_wl)
        out = torch.empty((500, 2, n), dtype=torch.complex64, device=dev)
        g.predict(torch.from_numpy(model[:n]).to(dev), None, out)
        g.synchronize()
        g.close()
        got = out.cpu().numpy().reshape(-1, n)
        for k in range(n):
            ok = np.isfinite(want[k])
            assert np.array_equal(ok, np.isfinite(got[:, k])) and ok.any()
            assert rel(got[ok, k], want[k][ok]) < TOL["reference"], (n, k)


def test_degridding_four_images_takes_less_than_four_of_one():
    """Reading four images' cells must not cost more than four launches of one
    (with the images interleaved in LDS: 5.4 times one image; in planes: 2.1)."""
    import wsclean_amd
    dev = torch.device("cuda:0")
    rng = np.random.default_rng(3)
    w, K, nrow, nchan = 1000, 9, 100000, 32
    dl = 0.0005
    wl = C_LIGHT / np.linspace(120e6, 168e6, nchan)
    umax = 0.2 / dl * wl.min()
    uvw = np.column_stack([rng.uniform(-umax, umax, nrow), rng.uniform(-umax, umax, nrow),
                           rng.uniform(0, 30, nrow)])
    d_uvw, d_wl = torch.from_numpy(uvw).to(dev), torch.from_numpy(wl).to(dev)
    ms = {}
    for n in (1, 4):
        g = wsclean_amd.DeviceGridder(w, w, dl, dl, K, 63, n_images=n)
        g.prepare_w_layers(4, 0.0, float(uvw[:, 2].max() / wl.min()))
        g.plan(d_uvw, d_wl)
        model = torch.ones((n, w, w), dtype=torch.float32, device=dev)
        out = torch.empty((nrow, nchan, n), dtype=torch.complex64, device=dev)
        times = []
        for _ in range(9):
            g.predict(model, None, out)
            times.append(g.stats()["ms_grid"])
        g.close()
        ms[n] = sorted(times)[4]
    print(f"degridding: {ms}")
    assert ms[4] < 4 * ms[1]


@pytest.mark.parametrize("precision", ["reference", "mixed"])
@pytest.mark.parametrize("no_mfma", ["0", "1"])
def test_cut_tiles_with_images_rotation_batches_and_passes(oracle, monkeypatch, precision,
                                                           no_mfma):
    """A last tile of 8 by 12 cells with two real images and a complex one, a
    shifted and rotated phase centre and bins split into work items: two batches
    through the host protocol (the second adds to the tiles), then one pass and
    two on the device, by the matrix-core kernel and (HWS_NO_MFMA=1) the cell
    kernel."""
    import wsclean_amd
    dev = torch.device("cuda:0")
    monkeypatch.setenv("HWS_NO_MFMA", no_mfma)
    w, h, dl, nw, n = 120, 60, 0.003, 5, 700
    shift = (0.006, -0.004)
    rng = np.random.default_rng(120)
    wl = C_LIGHT / np.linspace(120e6, 150e6, 3)
    umax = 0.499 / dl * wl.min()
    uvw = np.column_stack([rng.uniform(-umax, umax, n), rng.uniform(-umax, umax, n),
                           rng.uniform(-40, 40, n)])
    # half of them about the edge of the cut tiles
    edge = wl.min() / dl * np.array([-9.0 / w, -13.0 / h])
    uvw[::2, :2] = edge + rng.uniform(-4, 4, (n // 2, 2)) * wl.min() / (dl * np.array([w, h]))
    vis = (rng.standard_normal((n, 3, 3)) + 1j * rng.standard_normal((n, 3, 3))
           ).astype(np.complex64)
    uvw_l = (uvw[:, None, :] / wl[None, :, None]).reshape(-1, 3)
    maxw = float(np.abs(uvw_l[:, 2]).max())
    ph = np.exp(-2j * np.pi * (uvw_l[:, 0] * shift[0] + uvw_l[:, 1] * shift[1]))
    model = rng.standard_normal((2, 3, h, w)).astype(np.float32)
    want, want_v = [], []
    for k in range(3):
        o = oracle.RefGridder(w, h, dl, dl, 1, 7, 63, "float")
        o.set_is_complex(k == 2)
        o.set_denormal_phase_centre(*shift)
        o.prepare_w_layers(nw, 1e12, 0.0, maxw)
        o.start_inversion_pass(0)
        o.add_samples(uvw_l, (vis[:, :, k].reshape(-1) * ph).astype(np.complex64))
        o.finish_inversion_pass()
        o.finalize_image(1.0)
        want += list(o.image(imag=True)) if k == 2 else [o.image()]
        o = oracle.RefGridder(w, h, dl, dl, 1, 7, 63, "float")
        o.set_is_complex(k == 2)
        o.set_denormal_phase_centre(*shift)
        o.prepare_w_layers(nw, 1e12, 0.0, maxw)
        o.initialize_prediction(model[0, k], model[1, k] if k == 2 else None)
        o.start_prediction_pass(0)
        want_v.append(o.sample(uvw_l) * np.conj(ph))
    kw = dict(precision=precision, n_images=3, complex_images=(2,), l_shift=shift[0],
              m_shift=shift[1], rotate_visibilities=True, work_chunk=37)

    def compare(re, im):
        for got, img in zip((re[0], re[1], re[2], im[2]), want):
            assert rel(got, img) < TOL[precision]

    g = wsclean_amd.WStackingGridder(w, h, dl, dl, 7, 63, **kw)
    g.prepare_w_layers(nw, 0.0, 0.0, maxw)
    g.start_inversion_pass(0)
    g.add_data(uvw[:300], wl, vis[:300])
    g.add_data(uvw[300:], wl, vis[300:])
    g.finish_inversion_pass()
    compare(*g.finalize_image(1.0))
    g.close()
    d_uvw, d_wl = torch.from_numpy(uvw).to(dev), torch.from_numpy(wl).to(dev)
    d_vis, d_model = torch.from_numpy(vis).to(dev), torch.from_numpy(model).to(dev)
    for passes, max_mem in ((1, 0.0), (2, w * h * 8.0 * 3 * 3)):
        g = wsclean_amd.DeviceGridder(w, h, dl, dl, 7, 63, **kw)
        assert g.prepare_w_layers(nw, 0.0, maxw, max_mem=max_mem) == passes
        g.plan(d_uvw, d_wl)
        re = torch.zeros((3, h, w), dtype=torch.float32, device=dev)
        im = torch.zeros_like(re)
        g.invert(d_vis, 1.0, re, im)
        out = torch.empty_like(d_vis)
        g.predict(d_model[0], d_model[1], out)
        stats = g.stats()
        assert stats["tiles_total"] == nw * 8 * 4 and stats["chunks"] > stats["bins_used"]
        compare(re.cpu().numpy(), im.cpu().numpy())
        for k in range(3):
            got, ok = out[:, :, k].cpu().numpy().reshape(-1), np.isfinite(want_v[k])
            assert np.array_equal(ok, np.isfinite(got)) and ok.any()
            assert rel(got[ok], want_v[k][ok]) < TOL[precision]
        g.close()


@pytest.mark.parametrize("oversampling,tiles", [(63, 16), (221, 16), (223, 9), (1023, 9)])
def test_cut_tiles_need_the_padded_table_in_lds(oversampling, tiles):
    """Tiles of 20 keep dividing 60 x 60 where the zero-padded kernel table does
    not fit the LDS (the oversampling is odd; 221 is the last that fits)."""
    import wsclean_amd
    dev = torch.device("cuda:0")
    g = wsclean_amd.DeviceGridder(60, 60, 0.004, 0.004, 7, oversampling)
    g.prepare_w_layers(2, 0.0, 1.0)
    g.plan(torch.zeros((4, 3), dtype=torch.float64, device=dev),
           torch.ones(1, dtype=torch.float64, device=dev))
    assert g.stats()["tiles_total"] == 2 * tiles
    g.close()
