"""Snowcover update from drift_mass (CHM snobal's drift consumer, src/modules/snobal.cpp:363-387,
third_party/snobal/sno.cpp _adj_snow / _adj_layers / _calc_layers / _layer_mass).

CPU: the oracle against values that follow from the rules themselves (layer splits at
the 0.1 m active layer and the 0.2 kg/m^2 mass threshold, removal at the pack density,
the 750 kg/m^3 cap, -9999 / NaN as no drift), the specific heat of ice at -15 C within
1 % of its measured value (Dorsey 1940: 2.0 kJ/kg/K), and mass conservation over random
deposition sequences.  GPU: the HIP kernels against the oracle bit for bit, and the
chain PBSM3D step -> snowcover update -> next step's swe / snowdepthavg."""
import math

import numpy as np
import pytest

from chm_amd import abi, meshgen

FREEZE = 273.16
F_ = {n: k for k, n in enumerate(abi.SNOW_FIELDS)}


def _cfg(**kw):
    c = abi.SnowConfig()
    c.drift_density, c.max_active_layer, c.ic_rho, c.max_h2o_vol, c.mass_threshold = 300.0, 0.1, 300.0, 1e-4, 0.2
    for k, v in kw.items():
        setattr(c, k, v)
    return c


def _face(st, i):
    return {n: st[k, i] for n, k in F_.items()}


# ---------------------------------------------------------------------------
# oracle (CPU)
# ---------------------------------------------------------------------------
def test_oracle_initial_snowcover(oracle):
    swe0 = np.array([0.0, 0.1, 20.0, 60.0, 30.06, -9999.0, np.nan])
    st = oracle.snow_init(len(swe0), swe0, _cfg())
    bare = _face(st, 0)
    assert bare["layer_count"] == 0 and bare["m_s"] == 0 and bare["z_s"] == 0 and bare["h2o_total"] == 0
    assert bare["T_s_0"] == pytest.approx(-75 + FREEZE) and bare["h2o_sat"] == 0
    # below the 0.2 kg/m^2 threshold the snow becomes liquid water, no layer
    thin = _face(st, 1)
    assert thin["layer_count"] == 0 and thin["m_s"] == 0 and thin["h2o_total"] == pytest.approx(0.1, abs=1e-15)
    # 20 kg/m^2 at 300 kg/m^3: one 0.0667 m layer
    one = _face(st, 2)
    assert one["layer_count"] == 1 and one["z_s"] == pytest.approx(20 / 300) and one["m_s_0"] == pytest.approx(20)
    assert one["m_s_l"] == 0 and one["T_s_l"] == pytest.approx(-75 + FREEZE) and one["cc_s_l"] == 0
    # 60 kg/m^2: 0.2 m = 0.1 m active layer + 0.1 m lower layer, 30 kg/m^2 each
    two = _face(st, 3)
    assert two["layer_count"] == 2 and two["z_s_0"] == pytest.approx(0.1) and two["z_s_l"] == pytest.approx(0.1)
    assert two["m_s_0"] == pytest.approx(30) and two["m_s_l"] == pytest.approx(30)
    # cold content = c_ice m dT with c_ice(-15 C) within 1 % of 2.0 kJ/kg/K, negative below freezing
    c_ice = two["cc_s_0"] / (two["m_s_0"] * -15.0)
    assert 1980 < c_ice < 2020
    assert two["cc_s_l"] == pytest.approx(two["cc_s_0"])
    # liquid water: 30 % of the holding capacity max_h2o_vol * z_s * rho_w (1 - rho_dry / rho_ice)
    assert two["h2o_vol"] == pytest.approx(0.3e-4)
    assert two["h2o"] == pytest.approx(0.3 * two["h2o_max"])
    assert two["h2o_max"] == pytest.approx(1e-4 * 0.2 * 999.87 * (1 - 300 / 917), rel=1e-4)
    # a 0.0002 m lower layer would hold 0.06 kg/m^2 < 0.2: one layer of 0.1002 m
    edge = _face(st, 4)
    assert edge["layer_count"] == 1 and edge["z_s_0"] == pytest.approx(0.1002)
    for i in (5, 6):  # no initial condition
        np.testing.assert_array_equal(st[:, i], st[:, 0])


def test_oracle_drift_rules(oracle):
    cfg = _cfg()
    st0 = oracle.snow_init(6, np.array([0.0, 20.0, 60.0, 20.0, 20.0, 60.0]), cfg)
    drift = np.array([10.0, 20.0, -15.0, -19.9, -30.0, -9999.0])
    st = oracle.snow_drift(st0, cfg, drift)
    # deposition on bare ground at 300 kg/m^3
    f = _face(st, 0)
    assert f["m_s"] == 10 and f["z_s"] == pytest.approx(10 / 300) and f["rho"] == pytest.approx(300)
    assert f["layer_count"] == 1 and f["m_s_0"] == pytest.approx(10)
    # 20 + 20 kg/m^2: 0.1333 m, a lower layer appears at the pack temperature
    f, f0 = _face(st, 1), _face(st0, 1)
    assert f["layer_count"] == 2 and f["z_s_l"] == pytest.approx(40 / 300 - 0.1) and f["m_s_l"] == pytest.approx(10)
    assert f["T_s_l"] == f0["T_s"] and f["cc_s_l"] < 0
    assert f["cc_s_0"] == f0["cc_s_0"]  # the surface layer's cold content is not recomputed
    # erosion of 15 kg/m^2 at the pack's own density keeps 300 kg/m^3
    f = _face(st, 2)
    assert f["m_s"] == 45 and f["z_s"] == pytest.approx(0.15) and f["rho"] == pytest.approx(300)
    assert f["m_s_l"] == pytest.approx(15)
    # erosion to 0.1 kg/m^2: below the threshold, the rest turns into liquid water
    f = _face(st, 3)
    assert f["layer_count"] == 0 and f["m_s"] == 0 and f["h2o_total"] == pytest.approx(0.1, abs=1e-12)
    assert f["T_s"] == pytest.approx(-75 + FREEZE) and f["h2o_sat"] == 0
    # erosion of more than the pack: nothing left, no water either
    f = _face(st, 4)
    assert f["layer_count"] == 0 and f["m_s"] == 0 and f["z_s"] == 0 and f["h2o_total"] == 0
    # -9999 (and NaN) is no drift: the consistent state is unchanged
    np.testing.assert_array_equal(st[:, 5], st0[:, 5])
    st_nan = oracle.snow_drift(st0, cfg, np.full(6, np.nan))
    np.testing.assert_array_equal(st_nan, st0)
    # the 750 kg/m^3 cap: a pack stored at 800 kg/m^3 is re-thickened to m_s / 750
    bad = st0[:, 2:3].copy()
    bad[F_["m_s"]], bad[F_["z_s"]], bad[F_["rho"]] = 80.0, 0.1, 800.0
    capped = _face(oracle.snow_drift(bad, cfg, np.array([0.0])), 0)
    assert capped["rho"] == 750 and capped["z_s"] == pytest.approx(80 / 750) and capped["layer_count"] == 2


def test_oracle_mass_conservation(oracle):
    """Deposition-only sequences conserve water: m_s + h2o_total = initial + sum of deposits."""
    rng = np.random.default_rng(4)
    n = 500
    cfg = _cfg()
    swe0 = rng.uniform(0, 80, n)
    st = oracle.snow_init(n, swe0, cfg)
    total0 = st[F_["m_s"]] + st[F_["h2o_total"]]
    added = np.zeros(n)
    for _ in range(6):
        d = rng.exponential(0.5, n)
        added += d
        st = oracle.snow_drift(st, cfg, d)
        assert np.all(st[F_["rho"]] <= 750)
        assert np.all((st[F_["m_s_0"]] + st[F_["m_s_l"]])[st[F_["layer_count"]] > 0] == pytest.approx(
            st[F_["m_s"]][st[F_["layer_count"]] > 0]))
    np.testing.assert_allclose(st[F_["m_s"]] + st[F_["h2o_total"]], total0 + added, rtol=1e-12, atol=1e-12)


# ---------------------------------------------------------------------------
# GPU
# ---------------------------------------------------------------------------
@pytest.fixture(scope="module")
def pb():
    from chm_amd import pbsm3d

    pbsm3d.lib()
    return pbsm3d


def _drifts(rng, n, steps):
    out = []
    for _ in range(steps):
        d = rng.normal(0, 8, n)
        d[::37] = -9999.0
        d[5::41] = np.nan
        d[7::53] = -500.0  # more than any pack holds
        out.append(d)
    return out


@pytest.mark.gpu
def test_gpu_snow_matches_oracle_bitwise(pb, oracle):
    print("[case] snow drift vs oracle", flush=True)
    rng = np.random.default_rng(9)
    n = 20011
    cfg = _cfg()
    swe0 = rng.uniform(0, 120, n)
    swe0[::11] = -9999.0
    swe0[3::17] = 0.05
    sn = pb.Snow(n, swe0, cfg)
    ref = oracle.snow_init(n, swe0, cfg)
    np.testing.assert_array_equal(sn.get_state(), ref)
    for d in _drifts(rng, n, 5):
        sn.drift(d)
        ref = oracle.snow_drift(ref, cfg, d)
        np.testing.assert_array_equal(sn.get_state(), ref)
    swe, sd = sn.outputs()
    np.testing.assert_array_equal(swe, ref[F_["m_s"]])
    np.testing.assert_array_equal(sd, ref[F_["z_s"]])
    # device pointers, and state round trip (checkpoint / restart)
    import torch

    d = torch.tensor(_drifts(rng, n, 1)[0], device="cuda:0")
    saved = sn.get_state()
    sn.drift(d)
    ref = oracle.snow_drift(ref, cfg, d.cpu().numpy())
    np.testing.assert_array_equal(sn.get_state(), ref)
    swe_d, sd_d = sn.outputs(device=True)
    np.testing.assert_array_equal(swe_d.cpu().numpy(), ref[F_["m_s"]])
    sn.set_state(saved)
    np.testing.assert_array_equal(sn.get_state(), saved)
    sn.close()
    # no initial condition anywhere
    bare = pb.Snow(64, None, cfg)
    np.testing.assert_array_equal(bare.get_state(), oracle.snow_init(64, None, cfg))
    bare.close()


@pytest.mark.gpu
def test_gpu_snow_any_state_matches_oracle_bitwise(pb, oracle):
    """States that the update itself never makes (a lower layer's mass, heat or water where no
    layer is): every member it does not renew is kept, as in the oracle."""
    print("[case] snow drift from arbitrary states", flush=True)
    rng = np.random.default_rng(31)
    n = 4099
    cfg = _cfg()
    sn = pb.Snow(n, rng.uniform(0, 120, n), cfg)
    st = sn.get_state() + rng.uniform(0.0, 1.0, (len(F_), n))
    st[F_["layer_count"]] = rng.integers(0, 3, n)
    st[F_["z_s"], ::5] = 0.0
    st[F_["m_s"], ::7] = 0.1
    sn.set_state(st)
    ref = st.copy()
    for d in _drifts(rng, n, 3):
        sn.drift(d)
        ref = oracle.snow_drift(ref, cfg, d)
        np.testing.assert_array_equal(sn.get_state(), ref)
    sn.close()


@pytest.mark.gpu
def test_gpu_chain_step_snow_step(pb, oracle, mesh_small):
    """PBSM3D step -> drift_mass -> snowcover update -> swe / snowdepthavg of the next step,
    on device arrays, against the same chain through the oracles."""
    import torch

    print("[case] PBSM3D -> snow -> PBSM3D", flush=True)
    F = mesh_small.n_faces
    g = pb.face_geometry(mesh_small)
    fo = meshgen.forcing_c1(F, seed=2)
    cfg = _cfg()
    swe0 = np.asarray(fo["swe"], dtype=np.float64)
    ctx = pb.Context(g, pb.default_config(nLayer=5, tol=1e-12))
    orc = oracle.Oracle(g, oracle.oracle_config(nLayer=5, tol=1e-13))
    sn = pb.Snow(F, swe0, cfg)
    ref = oracle.snow_init(F, swe0, cfg)
    d = {k: torch.tensor(v, device="cuda:0") for k, v in fo.items()}
    ofo = dict(fo)
    for step in range(3):
        outs = {k: torch.zeros(F, dtype=torch.float64, device="cuda:0") for k in abi.OUT_FIELDS}
        ctx.step(d, outs=outs, on_device=True)
        og, _ = orc.step(ofo)
        sn.drift(outs["drift_mass"])
        ref = oracle.snow_drift(ref, cfg, og["drift_mass"])
        swe, sd = sn.outputs(device=True)
        d["swe"], d["snowdepthavg"] = swe, sd
        ofo["swe"], ofo["snowdepthavg"] = ref[F_["m_s"]].copy(), ref[F_["z_s"]].copy()
        scale = max(1.0, float(np.abs(ofo["swe"]).max()))
        assert np.abs(swe.cpu().numpy() - ofo["swe"]).max() <= 1e-8 * scale, step
        assert np.abs(sd.cpu().numpy() - ofo["snowdepthavg"]).max() <= 1e-8 * scale / 100, step
    ctx.close()
    sn.close()
