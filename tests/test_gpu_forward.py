"""GPU parity of the forward time loop (HIP engine through the C ABI) against the CPU oracle."""

import numpy as np
import pytest

from oracle import fdtd_oracle as O
from oracle import scenes as S
from fdtdx_amd import scenarios as W

pytestmark = pytest.mark.gpu


def rel(a, b):
    a = np.asarray(a).astype(np.complex128 if np.iscomplexobj(a) else np.float64)
    b = np.asarray(b).astype(np.complex128 if np.iscomplexobj(b) else np.float64)
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300))


# Sweep schedules: the two in-place sweeps with four z cells per lane (the default but for small grids,
# which the setting overrides) and with one, the LDS-tiled fused kernel and the register-march kernel with 4
# and 2 rows per wavefront (short x chunks so chunk halos are exercised).
MODES = {
    "quad": {"FDTDX_SWEEP": "quad"},
    "two": {"FDTDX_SWEEP": "two"},
    "fused": {"FDTDX_SWEEP": "fused"},
    "march4": {"FDTDX_SWEEP": "march", "FDTDX_MARCH_TY": "4", "FDTDX_MARCH_XC": "5"},
    "march2": {"FDTDX_SWEEP": "march", "FDTDX_MARCH_TY": "2", "FDTDX_MARCH_XC": "3"},
}


def _set_mode(monkeypatch, mode):
    for k in ("FDTDX_SWEEP", "FDTDX_MARCH_TY", "FDTDX_MARCH_XC"):
        monkeypatch.delenv(k, raising=False)
    for k, v in MODES[mode].items():
        monkeypatch.setenv(k, v)


@pytest.fixture(params=list(MODES))
def sweep(request, monkeypatch):
    _set_mode(monkeypatch, request.param)
    return request.param


def _run(spec):
    import torch

    import fdtdx_amd as fx
    import scenarios

    objects, arrays, params, config = scenarios.build(spec)
    print(f"case shape={spec['shape']} T={spec['T']}", flush=True)
    _, arrays = fx.run_fdtd(arrays, objects, config)
    torch.cuda.synchronize()
    return objects, arrays


def test_dipole_cube_small_matches_oracle(sweep):
    spec = W.scenario_c1(T=200, n=32, pml=6, cube=8)
    objects, arrays = _run(spec)
    st, ds = O.run(S.build_scene(spec), spec["T"])
    E = arrays.fields.E.cpu().numpy()
    H = arrays.fields.H.cpu().numpy()
    print("E", rel(E, st.E), "H", rel(H, st.H))
    assert rel(E, st.E) < 1e-5
    assert rel(H, st.H) < 1e-5
    en = arrays.detector_states["energy"]["energy"].cpu().numpy()
    assert rel(en, ds[0]) < 1e-5
    ez = arrays.detector_states["ez"]["fields"].cpu().numpy()
    assert rel(ez, ds[1]) < 1e-5


def test_plane_wave_design_small_matches_oracle(sweep):
    spec = W.scenario_c2(T=151, shape=(60, 40, 30), pml=6, slab=(20, 20, 6))
    objects, arrays = _run(spec)
    st, ds = O.run(S.build_scene(spec), spec["T"])
    E = arrays.fields.E.cpu().numpy()
    print("E", rel(E, st.E))
    assert rel(E, st.E) < 1e-5
    assert rel(arrays.fields.H.cpu().numpy(), st.H) < 1e-5
    flux = arrays.detector_states["flux"]["poynting_flux"].cpu().numpy()
    assert rel(flux, ds[0]) < 1e-5
    ph = arrays.detector_states["phasor"]["phasor"].cpu().numpy()
    assert rel(ph, ds[1]) < 1e-5


def test_dispersive_anisotropic_small_matches_oracle(sweep):
    spec = W.scenario_c4(T=120, n=40, pml=6, slab=(16, 16, 6), cube=6)
    objects, arrays = _run(spec)
    st, ds = O.run(S.build_scene(spec), spec["T"])
    E = arrays.fields.E.cpu().numpy()
    print("E", rel(E, st.E))
    assert rel(E, st.E) < 1e-5
    assert rel(arrays.fields.H.cpu().numpy(), st.H) < 1e-5
    ph = arrays.detector_states["phasor"]["phasor"].cpu().numpy()
    assert rel(ph, ds[0]) < 1e-5


def test_quad_ade_tiles_match_the_one_cell_path(monkeypatch):
    """ADE tiles of the quad schedule (listed for the E half-step only; the H half-step sweeps
    them four cells per lane): fields, ADE state and phasors equal the one-cell schedule's bit for
    bit, and the oracle's within 1e-5."""
    import scenarios

    from fdtdx_amd import fdtd as F

    spec = W.scenario_c4(T=120, n=40, pml=6, slab=(16, 16, 8), cube=8)
    out = {}
    for mode in ("quad", "two"):
        _set_mode(monkeypatch, mode)
        objects, arrays, params, config = scenarios.build(spec)
        F.run_fdtd(arrays, objects, config)
        solve = F._solve_for(objects, config, arrays)
        out[mode] = (solve.plan.schedule, arrays.fields.E.cpu().numpy(), arrays.fields.H.cpu().numpy(),
                     arrays.ade_state.cpu().numpy(), arrays.detector_states["phasor"]["phasor"].cpu().numpy())
    assert out["quad"][0] != out["two"][0]
    for a, b in zip(out["quad"][1:], out["two"][1:]):
        np.testing.assert_array_equal(a, b)
    st, ds = O.run(S.build_scene(spec), spec["T"])
    assert rel(out["quad"][1], st.E) < 1e-5 and rel(out["quad"][4], ds[0]) < 1e-5


@pytest.mark.parametrize("nz,types", [(36, {}), (37, {}), (39, {}), (38, {"min_z": "periodic", "max_z": "periodic"})])
@pytest.mark.parametrize("sigma", [0.0, 2e4])
def test_quad_poles_equal_the_one_cell_poles_bitwise(nz, types, sigma, monkeypatch):
    """Poles inside the quad E sweep against one cell per lane: boxes with edges inside quads, one of
    them up to the row's last quad, isotropic and diagonal permittivity, one and two poles, with and
    without conductivity in the same cells. Fields, psi, poles and phasors agree bit for bit."""
    import scenarios

    from fdtdx_amd import fdtd as F

    spec = W.scenario_c4(T=41, n=36, pml=5, slab=(12, 12, 8), cube=6)
    spec["shape"] = (36, 34, nz)
    spec["pml"] = dict(spec["pml"], types=types)
    spec["detectors"] = [dict(d, slc=((26, 27), (0, 34), (0, nz))) for d in spec["detectors"]]
    poles = spec["boxes"][0]["poles"]
    spec["boxes"] = [dict(slc=((12, 25), (9, 22), (15, 26)), eps=(2.0, 4.0, 9.0), poles=poles, sigma_E=sigma),
                     dict(slc=((20, 29), (14, 23), (22, nz if types else nz - 5)), eps=4.0, poles=poles[:1],
                          sigma_E=sigma),
                     dict(slc=((9, 11), (9, 20), (18, 21)), eps=3.0, poles=[("drude", 2e15, 1e14)])]
    out = {}
    for mode in ("quad", "two"):
        _set_mode(monkeypatch, mode)
        objects, arrays, params, config = scenarios.build(spec)
        F.run_fdtd(arrays, objects, config)
        solve = F._solve_for(objects, config, arrays)
        assert solve.plan.quad == (mode == "quad" and not (sigma and nz % 4))
        out[mode] = [arrays.fields.E.cpu().numpy(), arrays.fields.H.cpu().numpy(), arrays.psi.cpu().numpy(),
                     arrays.ade_state.cpu().numpy()] + [t.cpu().numpy() for t in solve.det_tensors()]
    assert np.abs(out["two"][0]).max() > 0 and np.abs(out["two"][3]).max() > 0
    for a, b in zip(out["quad"], out["two"]):
        np.testing.assert_array_equal(a, b)


def test_single_pass_equals_two_sweep_bitwise(monkeypatch):
    """The single-pass kernels perform the two-sweep kernels' float operations in the same order:
    fields, psi, detector states and the interface record agree bit for bit (z split into two
    lane runs, partial y tiles and x chunks, an odd step count so the ping-pong copies back)."""
    import torch

    from fdtdx_amd import fdtd as F
    import scenarios

    spec = W.scenario_c2(T=37, shape=(50, 45, 70), pml=5, slab=(20, 16, 8))
    out = {}
    for mode in MODES:
        _set_mode(monkeypatch, mode)
        objects, arrays, params, config = scenarios.build(spec)
        s = F.Solve(objects, config, arrays, record_steps=spec["T"])
        arrays.reset()
        print(f"mode {mode}", flush=True)
        s.forward(0, spec["T"], record=True)
        torch.cuda.synchronize()
        out[mode] = [arrays.fields.E.cpu().numpy(), arrays.fields.H.cpu().numpy(), arrays.psi.cpu().numpy(),
                     s.record.cpu().numpy()] + [t.cpu().numpy() for t in s.det_tensors()]
    for mode in MODES:
        for a, b in zip(out[mode], out["two"]):
            assert np.array_equal(a, b), mode


@pytest.mark.parametrize("mode", ["two", "fused"])
def test_conductor_faces_match_oracle(mode, monkeypatch):
    """PEC / PMC faces (pec.py:70-77, pmc.py:62-75) on three faces, CPML on the others; a
    single-pass request falls back to the two sweeps, which apply the faces."""
    _set_mode(monkeypatch, mode)
    spec = W.scenario_c1(T=150, n=28, pml=5, cube=6)
    spec["pml"] = dict(spec["pml"], types={"max_x": "pec", "min_y": "pmc", "max_z": "pec"})
    spec["sources"][0]["profile"] = W.gaussian_profile(wavelength=0.4e-6, bandwidth=0.8)
    objects, arrays = _run(spec)
    st, ds = O.run(S.build_scene(spec), spec["T"])
    E = arrays.fields.E.cpu().numpy()
    H = arrays.fields.H.cpu().numpy()
    print("E", rel(E, st.E), "H", rel(H, st.H))
    assert rel(E, st.E) < 1e-5 and rel(H, st.H) < 1e-5
    assert not E[1:, -1].any() and not H[0, :, 0].any() and not H[2, :, 0].any() and not E[:2, :, :, -1].any()
    assert rel(arrays.detector_states["energy"]["energy"].cpu().numpy(), ds[0]) < 1e-5


@pytest.mark.parametrize("mode", ["two", "fused"])
def test_periodic_unit_cell_plane_wave_matches_oracle(mode, monkeypatch):
    """Periodic y and z (wrap padding, update.py:92-137) around an x-directed plane wave with a
    design slab: the classic unit cell. Flux and phasor planes span the periodic cross-section, so
    their interpolation stencils wrap too; a single-pass request falls back to the two sweeps."""
    _set_mode(monkeypatch, mode)
    spec = W.scenario_c2(T=151, shape=(60, 24, 20), pml=6, slab=(20, 12, 6))
    spec["pml"] = dict(spec["pml"], types={"min_y": "periodic", "max_y": "periodic", "min_z": "periodic",
                                           "max_z": "periodic"})
    objects, arrays = _run(spec)
    sc = S.build_scene(spec)
    assert sc.periodic == (False, True, True)
    st, ds = O.run(sc, spec["T"])
    E = arrays.fields.E.cpu().numpy()
    H = arrays.fields.H.cpu().numpy()
    print("E", rel(E, st.E), "H", rel(H, st.H), flush=True)
    assert rel(E, st.E) < 1e-5 and rel(H, st.H) < 1e-5
    assert rel(arrays.detector_states["flux"]["poynting_flux"].cpu().numpy(), ds[0]) < 1e-5
    assert rel(arrays.detector_states["phasor"]["phasor"].cpu().numpy(), ds[1]) < 1e-5


def test_periodic_dipole_matches_oracle():
    """Periodic x and y with CPML in z; a dipole radiates across the wrapped faces."""
    from scenarios import periodic_spec

    spec = periodic_spec(T=120)
    objects, arrays = _run(spec)
    st, ds = O.run(S.build_scene(spec), spec["T"])
    E = arrays.fields.E.cpu().numpy()
    print("E", rel(E, st.E), flush=True)
    assert rel(E, st.E) < 1e-5 and rel(arrays.fields.H.cpu().numpy(), st.H) < 1e-5
    # the field has crossed the wrapped faces: both edge planes of x carry it
    assert np.abs(E[:, 0]).max() > 1e-3 * np.abs(E).max() and np.abs(E[:, -1]).max() > 1e-3 * np.abs(E).max()
    assert rel(arrays.detector_states["flux"]["poynting_flux"].cpu().numpy(), ds[0]) < 1e-5


@pytest.mark.parametrize("mode", ["two", "march4"])
def test_conductivity_matches_oracle(mode, monkeypatch):
    """Electric (diagonal) and magnetic (isotropic) conductivity in two overlapping boxes, one
    reaching into the CPML (update.py:300-354, 741-750); a single-pass request falls back to the
    two sweeps, which apply the loss."""
    _set_mode(monkeypatch, mode)
    spec = W.scenario_c1(T=150, n=28, pml=5, cube=6)
    spec["boxes"] = spec["boxes"] + [
        dict(slc=((16, 26), (8, 20), (2, 12)), eps=2.0, sigma_E=(3e4, 1e4, 2e4), sigma_H=2e9),
        dict(slc=((4, 10), (4, 28), (15, 22)), eps=1.5, sigma_E=(5e3, 8e3, 6e3))]
    objects, arrays = _run(spec)
    sc = S.build_scene(spec)
    assert sc.sigma_E is not None and sc.sigma_H is not None
    st, ds = O.run(sc, spec["T"])
    E = arrays.fields.E.cpu().numpy()
    H = arrays.fields.H.cpu().numpy()
    print("E", rel(E, st.E), "H", rel(H, st.H), flush=True)
    assert rel(E, st.E) < 1e-5 and rel(H, st.H) < 1e-5
    assert rel(arrays.detector_states["energy"]["energy"].cpu().numpy(), ds[0]) < 1e-5


def test_conductivity_with_dispersion_matches_oracle():
    """Loss divides after the ADE correction (update.py:338-350): conductivity on the dispersive
    box of the anisotropic Lorentz/Drude case."""
    spec = W.scenario_c4(T=120, n=40, pml=6, slab=(16, 16, 6), cube=6)
    spec["boxes"] = [dict(b, sigma_E=(2e4, 1e4, 3e4)) if b.get("poles") else b for b in spec["boxes"]]
    objects, arrays = _run(spec)
    sc = S.build_scene(spec)
    assert sc.sigma_E is not None and sc.ade is not None
    st, ds = O.run(sc, spec["T"])
    E = arrays.fields.E.cpu().numpy()
    print("E", rel(E, st.E), flush=True)
    assert rel(E, st.E) < 1e-5 and rel(arrays.fields.H.cpu().numpy(), st.H) < 1e-5
    assert rel(arrays.detector_states["phasor"]["phasor"].cpu().numpy(), ds[0]) < 1e-5


def test_plane_source_in_dispersive_medium_matches_oracle():
    """A broadband plane wave launched inside a Lorentz medium (effective carrier permittivity and
    the filtered E-side table, linear_polarization.py:191-210, 330-351)."""
    spec = W.scenario_c2(T=151, shape=(60, 30, 24), pml=6, slab=(20, 12, 6))
    w = 2 * np.pi * 299792458.0 / 1.55e-6
    spec["boxes"] = [dict(slc=((0, 40), (0, 30), (0, 24)), eps=2.1, poles=[("lorentz", 1.4 * w, 0.1 * w, 0.8)])]
    objects, arrays = _run(spec)
    st, ds = O.run(S.build_scene(spec), spec["T"])
    E = arrays.fields.E.cpu().numpy()
    print("E", rel(E, st.E), flush=True)
    assert rel(E, st.E) < 1e-5 and rel(arrays.fields.H.cpu().numpy(), st.H) < 1e-5
    assert rel(arrays.detector_states["flux"]["poynting_flux"].cpu().numpy(), ds[0]) < 1e-5


def test_detector_options_match_oracle():
    """Reduced field and phasor detectors, apodized phasors (Tukey and Gaussian windows) and a flux
    plane keeping all three components, against the oracle."""
    from scenarios import detector_zoo_spec

    spec = detector_zoo_spec(T=120)
    objects, arrays = _run(spec)
    _, ds = O.run(S.build_scene(spec), spec["T"])
    keys = dict(flux="poynting_flux", ph="phasor", phr="phasor", fld="fields", en="energy", fl3="poynting_flux")
    for q, d in enumerate(spec["detectors"]):
        got = arrays.detector_states[d["name"]][keys[d["name"]]].cpu().numpy()
        print(d["name"], got.shape, "rel", rel(got, ds[q]), flush=True)
        assert got.shape == ds[q].shape
        assert rel(got, ds[q]) < 1e-5


def _surface_states(objects, arrays, spec):
    """Detector states of surface_zoo_spec in the oracle's (expanded) detector order."""
    out = []
    for d in spec["detectors"]:
        st = arrays.detector_states[d["name"]]
        if d["kind"] == "closed_phasor":
            for a in d["axes"]:
                for side in ("min", "max"):
                    out.append(st[f"phasor_axis{a}_{side}"])
        else:
            out.append(next(iter(st.values())))
    return [t.detach().cpu().numpy() for t in out]


def test_surface_detectors_match_oracle():
    """The net flux through the six faces of a box (one reduced flux detector per face, the later
    ones accumulating), the phasors of a phasor-flux plane and of the faces of a closed phasor
    surface against the oracle; the post-processed phasor flux and net phasor flux (computed on the
    device) against the oracle's post-processing of its own phasors."""
    import fdtdx_amd as fx
    from scenarios import surface_zoo_spec

    spec = surface_zoo_spec(T=120)
    objects, arrays = _run(spec)
    sc = S.build_scene(spec)
    _, ds = O.run(sc, spec["T"])
    got = _surface_states(objects, arrays, spec)
    for d, g, w in zip(sc.detectors, got, ds):
        print(d["name"], g.shape, "rel", rel(g, w), flush=True)
        assert g.shape == w.shape
        assert rel(g, w) < 1e-5
    dx2 = float(np.float32(spec["dx"] ** 2))
    pf = next(o for o in objects.detectors if isinstance(o, fx.PhasorPoyntingFluxDetector))
    by = {d["name"]: w for d, w in zip(sc.detectors, ds)}
    host = pf.compute_poynting_flux(arrays.detector_states["pf"]).cpu().numpy()
    want = O.phasor_poynting_flux(by["pf"][0], 0, 1, dx2)
    print("phasor flux", host, want, flush=True)
    assert rel(host, want) < 1e-5
    cp = next(o for o in objects.detectors if isinstance(o, fx.ClosedSurfacePhasorPoyntingFluxDetector))
    net = cp.compute_net_flux(arrays.detector_states["cp"]).cpu().numpy()
    faces = {(a, side): by[f"cp:phasor_axis{a}_{side}"] for a in (0, 2) for side in ("min", "max")}
    want = O.closed_phasor_net_flux(faces, dx2, inward=True)
    print("net phasor flux", net, want, flush=True)
    assert rel(net, want) < 1e-5


def test_batch_accumulating_detectors_equal_the_plain_solve():
    """A closed surface (face detectors accumulating into one state) advanced in a multi-instance
    batch equals the same solve run through fdtdx_forward, bit for bit; a plan whose accumulating
    detector follows no matching one is rejected."""
    import torch

    from fdtdx_amd import engine
    from fdtdx_amd.fdtd import Solve
    from scenarios import surface_zoo_spec

    spec = surface_zoo_spec(T=100)
    objects, arrays, params, config = W.build(spec)
    solve = Solve(objects, config, arrays)
    arrays.reset()
    solve.forward(0, spec["T"])
    torch.cuda.synchronize()
    plain = [t.clone() for t in solve.state_tensors()]
    arrays.reset()
    torch.cuda.synchronize()
    b = engine.Batch(solve.plan.spec["eps_comps"], solve.plan.spec["mu_comps"])
    try:
        buf = solve.buffers()
        b.attach(0, solve.plan, buf, solve._keep, 0, spec["T"])
        b.advance(spec["T"], engine.current_stream_handle(), graph=False)
        torch.cuda.synchronize()
        assert b.step_index(0) == spec["T"]
        for (name, key), x, y in zip(solve.state_keys, solve.state_tensors(), plain):
            print(name, key, "equal", bool(torch.equal(x, y)), flush=True)
            assert torch.equal(x, y), (name, key)
    finally:
        b.close()
    cf = [d for d in solve.spec["detectors"] if d["name"] == "cf"]
    with pytest.raises(engine.EngineError, match="accumulate"):
        engine.Plan(dict(solve.spec, detectors=[dict(cf[1])]))


@pytest.mark.parametrize("variant", ["cpml", "periodic_walls"])
def test_full_tensor_matches_oracle(variant):
    """Non-symmetric full-tensor permittivity and permeability (the curl sweep, then the tensor
    sweep with four-point means of the off-diagonal curl components) with a dipole injecting into
    all three components: CPML on every face, or periodic x and y with a PEC and a PMC face on z."""
    from scenarios import tensor_spec

    spec = tensor_spec(periodic=variant != "cpml", walls=None if variant == "cpml" else {"max_z": "pec", "min_z": "pmc"})
    objects, arrays = _run(spec)
    assert arrays.inv_permittivities.shape[0] == 9
    st, ds = O.run(S.build_scene(spec), spec["T"])
    E = arrays.fields.E.cpu().numpy()
    H = arrays.fields.H.cpu().numpy()
    print("E", rel(E, st.E), "H", rel(H, st.H), flush=True)
    assert rel(E, st.E) < 1e-5
    assert rel(H, st.H) < 1e-5
    for q, name in enumerate(("ez", "flux")):
        got = next(iter(arrays.detector_states[name].values())).cpu().numpy()
        print(name, rel(got, ds[q]), flush=True)
        assert rel(got, ds[q]) < 1e-5


@pytest.mark.parametrize("symmetry,e_pol", [((0, 1, -1), (0, 0, 1)), ((0, -1, 1), (0, 1, 0))])
def test_symmetry_reduced_run_matches_oracle(symmetry, e_pol):
    """A mirror-symmetry-reduced run (PEC face on the electric plane, CPML on the far faces only,
    detector stencils reading the electric plane's mirror halo) against the oracle's reduced run:
    fields, flux, x-plane snapshot and phasors."""
    from scenarios import symmetry_spec

    spec = symmetry_spec(symmetry=symmetry, e_pol=e_pol, T=120)
    objects, arrays = _run(spec)
    assert tuple(arrays.fields.E.shape) == (3, 36, 12, 10)
    st, ds = O.run(S.build_scene(spec), spec["T"])
    print("E", rel(arrays.fields.E.cpu().numpy(), st.E), flush=True)
    assert rel(arrays.fields.E.cpu().numpy(), st.E) < 1e-5
    assert rel(arrays.fields.H.cpu().numpy(), st.H) < 1e-5
    for q, name in enumerate(("flux", "snap", "ph")):
        got = next(iter(arrays.detector_states[name].values())).cpu().numpy()
        print(name, rel(got, ds[q]), flush=True)
        assert rel(got, ds[q]) < 1e-5


def test_energy_slices_match_oracle():
    """EnergyDetector(as_slices=True): collapsed-axis means (one thread per plane cell, float64
    sums) and planes at given cells, against the oracle."""
    from scenarios import energy_slices_spec

    spec = energy_slices_spec()
    objects, arrays = _run(spec)
    _, ds = O.run(S.build_scene(spec), spec["T"])
    q = 0
    for name in ("mean", "planes"):
        for key in ("XY Plane", "XZ Plane", "YZ Plane"):
            got = arrays.detector_states[name][key].cpu().numpy()
            want = ds[q].reshape(got.shape)
            print(name, key, rel(got, want), flush=True)
            assert rel(got, want) < 1e-5
            q += 1


def test_single_frequency_dipole_matches_oracle():
    """The reference's default temporal profile, SingleFrequencyProfile (profile.py:254-275), with
    a wave-character phase shift, driving the dipole of the cube case."""
    from fdtdx_amd import constants

    spec = W.scenario_c1(T=150, n=28, pml=6, cube=8)
    spec["sources"][0]["profile"] = dict(kind="single", frequency=constants.c / 1.55e-6, phase_shift=0.4)
    objects, arrays = _run(spec)
    st, ds = O.run(S.build_scene(spec), spec["T"])
    E = arrays.fields.E.cpu().numpy()
    print("single-frequency E", rel(E, st.E), flush=True)
    assert np.abs(st.E).max() > 0
    assert rel(E, st.E) < 1e-5
    assert rel(arrays.fields.H.cpu().numpy(), st.H) < 1e-5
    assert rel(arrays.detector_states["energy"]["energy"].cpu().numpy(), ds[0]) < 1e-5


def _quad_cases():
    c1 = W.scenario_c1(T=60, n=32, pml=8, cube=8)                                  # z slabs on quad edges
    c2 = W.scenario_c2(T=50, shape=(40, 36, 28), pml=5, slab=(12, 12, 8))          # z slabs inside quads
    c4 = W.scenario_c4(T=50, n=36, pml=8, slab=(12, 12, 8), cube=4)                # diagonal eps, ADE tiles
    lossy = W.scenario_c1(T=60, n=28, pml=4, cube=6)                               # conductivity, walls, mu
    lossy["pml"] = dict(lossy["pml"], types={"max_x": "pec", "min_y": "pmc"})
    lossy["boxes"] = lossy["boxes"] + [
        dict(slc=((14, 24), (8, 20), (4, 12)), eps=2.0, sigma_E=(3e4, 1e4, 2e4), sigma_H=2e9, mu=(1.5, 2.0, 2.5))]
    per = W.scenario_c2(T=50, shape=(48, 24, 20), pml=6, slab=(16, 12, 8))        # periodic y, z
    per["pml"] = dict(per["pml"], types={"min_y": "periodic", "max_y": "periodic", "min_z": "periodic",
                                         "max_z": "periodic"})
    return {"cube_aligned": c1, "plane_unaligned": c2, "dispersive": c4, "lossy_walls_mu": lossy, "periodic": per}


@pytest.mark.parametrize("case", ["cube_aligned", "plane_unaligned", "dispersive", "lossy_walls_mu", "periodic"])
def test_quad_sweeps_equal_one_cell_sweeps_bitwise(case, monkeypatch):
    """Four z cells per lane (dwordx4 loads and stores, z neighbours from the lane's registers,
    quad CPML) against one cell per lane: fields, psi, the interface record and every detector
    state agree bit for bit, with z slabs on and inside quad boundaries, ADE, conductivity, PEC /
    PMC faces, magnetic materials and periodic axes."""
    import torch

    from fdtdx_amd import fdtd as F
    import scenarios

    spec = _quad_cases()[case]
    assert spec["shape"][2] % 4 == 0
    out = {}
    for mode in ("two", "quad"):
        _set_mode(monkeypatch, mode)
        objects, arrays, params, config = scenarios.build(spec)
        rec = 0 if case == "dispersive" else spec["T"]
        s = F.Solve(objects, config, arrays, record_steps=rec)
        assert s.plan.quad == (mode == "quad")
        arrays.reset()
        print(f"case {case} mode {mode}", flush=True)
        s.forward(0, spec["T"], record=bool(rec))
        torch.cuda.synchronize()
        out[mode] = [arrays.fields.E.cpu().numpy(), arrays.fields.H.cpu().numpy(), arrays.psi.cpu().numpy()]
        out[mode] += [s.record.cpu().numpy()] if rec else []
        out[mode] += [t.cpu().numpy() for t in s.det_tensors()]
    assert np.abs(out["two"][0]).max() > 0
    for a, b in zip(out["quad"], out["two"]):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("T", [1, 15, 16, 17, 33])
@pytest.mark.parametrize("halo", [False, True])
def test_deferred_detector_sums_equal_a_launch_per_step(T, halo):
    """Sums finalized for 16 steps at a time (one call) against step by step calls (one step each):
    energy over the whole volume, flux with a switch, reduced field and phasor detectors and a closed
    surface's accumulating faces agree bit for bit, with zero and periodic halos."""
    import torch

    from fdtdx_amd import fdtd as F
    import scenarios

    n = 20
    full = ((0, n), (0, n), (0, n))
    spec = W.scenario_c1(T=T, n=n, pml=4, cube=4)
    spec["sources"][0]["profile"] = dict(kind="single", frequency=2e14, phase_shift=0.3)
    if halo:
        spec["pml"] = dict(spec["pml"], types={f: "periodic" for f in ("min_y", "max_y")})
    spec["detectors"] = [
        dict(name="energy", kind="energy", slc=full, reduce_volume=True),
        dict(name="flux", kind="flux", slc=((14, 15), (0, n), (4, 16)), axis=0, reduce_volume=True,
             switch={"interval": 3}),
        dict(name="field", kind="field", slc=((6, 9), (5, 12), (4, 9)), components=("Ez", "Hx"), reduce_volume=True),
        dict(name="phasor", kind="phasor", slc=((6, 9), (5, 12), (4, 9)), components=("Ez", "Hx"),
             frequencies=[2e14], reduce_volume=True),
        dict(name="box", kind="closed_flux", slc=((5, 15), (5, 15), (5, 15))),
    ]
    out = []
    for stepwise in (False, True):
        objects, arrays, params, config = scenarios.build(spec)
        s = F.Solve(objects, config, arrays)
        arrays.reset()
        print(f"T={T} halo={halo} stepwise={stepwise}", flush=True)
        for t in range(T if stepwise else 1):
            s.forward(t if stepwise else 0, t + 1 if stepwise else T)
        torch.cuda.synchronize()
        out.append([t.cpu().numpy() for t in s.state_tensors()])
    assert T == 1 or np.abs(out[0][0]).max() > 0  # the source's ramp starts from zero
    for a, b in zip(*out):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("nz", [28, 30, 31])
@pytest.mark.parametrize("axis", [0, 1, 2])
def test_sources_in_quads_equal_one_cell_sweeps_bitwise(nz, axis, monkeypatch):
    """Plane sources normal to each axis (one normal to z holds one cell of its quads) and dipoles in
    overlapping quads, one in the cells a ragged row's last quad repeats, over diagonal permittivity and
    permeability: fields, psi, the interface record and the flux equal one cell per lane bit for bit."""
    import torch

    from fdtdx_amd import fdtd as F
    import scenarios

    spec = W.scenario_c1(T=45, n=28, pml=4, cube=6)
    spec["shape"] = (26, 25, nz)
    spec["boxes"] = [dict(slc=((0, 26), (0, 25), (0, nz)), eps=(2.0, 3.0, 4.0), mu=(1.2, 1.5, 1.7))]
    prof = dict(kind="single", frequency=2e14, phase_shift=0.3)
    e_pol = [0, 0, 0]
    e_pol[(axis + 1) % 3] = 1
    spec["sources"] = [dict(kind="plane", axis=axis, index=6, direction="+", e_pol=tuple(e_pol), profile=prof),
                       dict(kind="dipole", cell=(12, 11, 13), polarization=axis, profile=prof),
                       dict(kind="dipole", cell=(13, 11, nz - 3), polarization=(axis + 1) % 3, profile=prof)]
    spec["detectors"] = [dict(name="flux", kind="flux", slc=((17, 18), (5, 20), (5, 20)), axis=0, reduce_volume=True)]
    out = {}
    for mode in ("two", "quad"):
        _set_mode(monkeypatch, mode)
        objects, arrays, params, config = scenarios.build(spec)
        s = F.Solve(objects, config, arrays, record_steps=spec["T"])
        assert s.plan.quad == (mode == "quad")
        arrays.reset()
        print(f"nz {nz} axis {axis} {mode}", flush=True)
        s.forward(0, spec["T"], record=True)
        torch.cuda.synchronize()
        out[mode] = [t.cpu().numpy() for t in (arrays.fields.E, arrays.fields.H, arrays.psi, s.record, *s.det_tensors())]
    assert np.abs(out["quad"][0]).max() > 0
    for a, b in zip(out["quad"], out["two"]):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("box", [((5, 8), (2, 22), (1, 22)), ((2, 22), (7, 11), (3, 22)), ((9, 10), (4, 13), (0, 24)),
                                 ((0, 24), (0, 24), (0, 24))])
def test_energy_slice_means_equal_the_means_of_per_cell_energies(box):
    """The collapsed-axis means of a box (one wavefront of a block where a plane has at most a quarter of
    the box's cells, whole blocks else) against the float64 sums, in order, of the per-cell energies."""
    import torch

    from fdtdx_amd import fdtd as F
    import scenarios

    spec = W.scenario_c1(T=30, n=24, pml=4, cube=6)
    on = {"fixed_on_time_steps": [11, 29]}
    spec["detectors"] = [dict(name="s", kind="energy", slc=box, as_slices=True, aggregate="mean", switch=on),
                         dict(name="c", kind="energy", slc=box, switch=on)]
    objects, arrays, params, config = scenarios.build(spec)
    F.run_fdtd(arrays, objects, config)
    torch.cuda.synchronize()
    cells = arrays.detector_states["c"]["energy"].cpu().numpy()
    assert cells.shape == (2, *(b - a for a, b in box)) and np.abs(cells[1]).max() > 0
    got = arrays.detector_states["s"]
    assert len(got) == 3
    for a, plane in enumerate(("YZ Plane", "XZ Plane", "XY Plane")):
        ref = np.zeros(np.delete(np.array(cells.shape), a + 1))
        for t in range(cells.shape[a + 1]):
            ref = ref + np.take(cells, t, a + 1).astype(np.float64)
        assert np.array_equal(got[plane].cpu().numpy(), (ref / cells.shape[a + 1]).astype(np.float32)), plane


@pytest.mark.parametrize("nz", [24, 25, 26, 27])
@pytest.mark.parametrize("kind", ["pec", "pmc"])
def test_conducting_faces_in_quads_equal_one_cell_sweeps_bitwise(nz, kind, monkeypatch):
    """Conducting faces on all three axes inside the quad sweeps against one cell per lane, with sources in the
    face cells: a plane wave that spans the cross-section (E and H sources up to the y and z faces) and a dipole
    tangential to the upper z face in its layer. Fields, psi, the interface record and the energy agree bit for
    bit, and the tangential field of a face stays zero."""
    import torch

    from fdtdx_amd import fdtd as F
    import scenarios

    spec = W.scenario_c1(T=45, n=24, pml=4, cube=6)
    spec["shape"] = (24, 22, nz)
    spec["boxes"] = [dict(slc=((8, 20), (5, 22), (9, nz)), eps=(2.0, 3.0, 4.0))]
    spec["pml"] = dict(spec["pml"], types={f: kind for f in ("max_x", "min_y", "max_y", "min_z", "max_z")})
    prof = dict(kind="single", frequency=2e14, phase_shift=0.3)
    spec["sources"] = [dict(kind="plane", axis=0, index=7, direction="+", e_pol=(0, 1, 0), profile=prof),
                       dict(kind="dipole", cell=(12, 11, nz - 1), polarization=0, profile=prof)]
    spec["detectors"] = [dict(name="energy", kind="energy", slc=((0, 24), (0, 22), (0, nz)), reduce_volume=True)]
    out = {}
    for mode in ("two", "quad"):
        _set_mode(monkeypatch, mode)
        objects, arrays, params, config = scenarios.build(spec)
        s = F.Solve(objects, config, arrays, record_steps=spec["T"])
        assert s.plan.quad == (mode == "quad")
        arrays.reset()
        print(f"nz {nz} {kind} {mode}", flush=True)
        s.forward(0, spec["T"], record=True)
        torch.cuda.synchronize()
        out[mode] = [t.cpu().numpy() for t in (arrays.fields.E, arrays.fields.H, arrays.psi, s.record, *s.det_tensors())]
    f = out["quad"][0 if kind == "pec" else 1]
    assert np.abs(f).max() > 0 and not f[:2, :, :, 0].any() and not f[:2, :, :, -1].any() and not f[0, :, 0].any()
    for a, b in zip(out["quad"], out["two"]):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("slots", ["last", "pairs", "wrapped"])
def test_detector_steps_that_share_a_slot_are_stored_in_order(slots):
    """Energy, flux, reduced field and a closed surface's accumulating faces whose time_to_idx maps several
    steps to one slot (keep the last value; two steps per slot; a ring of 7 slots, some steps off): one call and
    one batch leave what step by step calls leave, the last step's values of each slot."""
    import torch

    from fdtdx_amd import engine
    from fdtdx_amd import fdtd as F
    import scenarios

    n, T = 20, 41
    spec = W.scenario_c1(T=T, n=n, pml=4, cube=4)
    spec["sources"][0]["profile"] = dict(kind="single", frequency=2e14, phase_shift=0.3)
    spec["detectors"] = [
        dict(name="energy", kind="energy", slc=((0, n),) * 3, reduce_volume=True),
        dict(name="flux", kind="flux", slc=((14, 15), (0, n), (4, 16)), axis=0, reduce_volume=True),
        dict(name="box", kind="closed_flux", slc=((5, 15), (5, 15), (5, 15))),
        dict(name="field", kind="field", slc=((6, 9), (5, 12), (4, 9)), components=("Ez", "Hx"), reduce_volume=True),
    ]
    step = np.arange(T)
    tti = {"last": 0 * step, "pairs": step // 2, "wrapped": np.where(step % 5 == 3, -1, step % 7)}[slots]

    def solve(shared=True):
        objects, arrays, params, config = scenarios.build(spec)
        s = F.Solve(objects, config, arrays)
        if shared:
            low = F.lower(objects, config, arrays)
            for d in low["detectors"]:
                d["time_to_idx"] = tti.astype(np.int32)
            s.plan = engine.Plan(low)
        arrays.reset()
        return s

    def states(s):
        torch.cuda.synchronize()
        return [t.cpu().numpy() for t in s.state_tensors()]

    own, whole, stepwise, batched = solve(False), solve(), solve(), solve()
    print(f"slots {slots}", flush=True)
    own.forward(0, T)  # a slot per step
    whole.forward(0, T)
    for t in range(T):
        stepwise.forward(t, t + 1)
    stream = torch.cuda.Stream()
    torch.cuda.synchronize()
    batch = engine.Batch(1, 0)
    batch.attach(0, batched.plan, batched.buffers(), batched._keep, 0, T)
    for _ in range(2):
        batch.advance(21, engine.c_void_p(stream.cuda_stream))
    stream.synchronize()
    batch.close()
    last = {int(s): t for t, s in enumerate(tti) if s >= 0}  # the last step of each slot
    ref = states(own)
    assert np.abs(ref[0]).max() > 0 and np.abs(ref[2]).max() > 0
    for got in (stepwise, whole, batched):
        for a, r in zip(states(got), ref):
            for slot, t in last.items():
                assert np.array_equal(a[slot], r[t]), (slot, t)


@pytest.mark.parametrize("shape,kind,quad", [
    ((40, 40, 40), "", True), ((40, 40, 40), "poles", False), ((88, 88, 88), "poles", False),
    ((92, 92, 92), "poles", True), ((92, 92, 93), "poles", False), ((144, 144, 146), "poles", True),
    ((92, 92, 93), "poles open_z", True), ((40, 40, 41), "", False), ((73, 73, 74), "", False),
    ((74, 74, 74), "", True), ((300, 200, 7), "open_z", False), ((300, 200, 9), "open_z", True),
    ((40, 40, 8), "open_z", True), ((40, 40, 41), "bloch", True), ((40, 40, 41), "bloch poles", True)])
def test_schedule_of_grids_run_alone(shape, kind, quad, monkeypatch):
    """Small grids with poles (with rows of nz % 4 != 0 cells and CPML normal to z, larger ones too) or with
    such rows, and those with such rows of under 8 cells, run one cell per lane alone and in quads in a batch or under FDTDX_SWEEP=quad; larger ones,
    complex fields and other grids in quads."""
    import scenarios

    from fdtdx_amd import fdtd as F

    spec = W.scenario_c1(T=3, n=40, pml=5, cube=8)
    spec["shape"] = shape
    spec["detectors"] = []
    if shape[2] < 16:
        spec["boxes"] = []
        spec["sources"][0]["cell"] = (20, 20, 4)
    if "poles" in kind:
        spec["boxes"][0]["poles"] = [("drude", 2e15, 1e14)]
    if "open_z" in kind:
        spec["pml"] = dict(spec["pml"], types={"min_z": "pec", "max_z": "pec"})
    if "bloch" in kind:
        spec["pml"] = dict(spec["pml"], types={"min_x": "bloch", "max_x": "bloch"})
        spec["bloch_vector"] = (1e5, 0.0, 0.0)
    for mode in (None, "quad"):
        if mode:
            monkeypatch.setenv("FDTDX_SWEEP", mode)
        else:
            monkeypatch.delenv("FDTDX_SWEEP", raising=False)
        objects, arrays, params, config = scenarios.build(spec)
        plan = F.Solve(objects, config, arrays).plan
        assert plan.quad == (quad or mode == "quad") and plan.batch_quad


def _ragged_cases():
    """Rows of nz % 4 != 0 cells: the last quad of a row repeats cells of the quad before it."""
    c1 = W.scenario_c1(T=60, n=29, pml=5, cube=6)                                  # nz % 4 = 1
    c2 = W.scenario_c2(T=50, shape=(44, 36, 30), pml=6, slab=(12, 12, 8))          # nz % 4 = 2, H sources
    c4 = W.scenario_c4(T=50, n=35, pml=8, slab=(12, 12, 8), cube=4)                # nz % 4 = 3, ADE tiles
    lossy = W.scenario_c1(T=60, n=27, pml=4, cube=6)                               # conductivity, walls, mu
    lossy["pml"] = dict(lossy["pml"], types={"max_x": "pec", "max_z": "pec"})
    lossy["boxes"] = lossy["boxes"] + [
        dict(slc=((14, 24), (8, 20), (18, 27)), eps=2.0, sigma_E=(3e4, 1e4, 2e4), sigma_H=2e9, mu=(1.5, 2.0, 2.5))]
    per = W.scenario_c2(T=50, shape=(48, 24, 21), pml=6, slab=(16, 12, 8))        # periodic y, z
    per["pml"] = dict(per["pml"], types={"min_y": "periodic", "max_y": "periodic", "min_z": "periodic",
                                         "max_z": "periodic"})
    thin = W.scenario_c1(T=40, n=24, pml=4, cube=4)                                # two quads per row, no z CPML
    thin["shape"] = (24, 24, 5)
    thin["pml"] = dict(thin["pml"], types={"min_z": "pec", "max_z": "pec"})
    thin["boxes"] = [dict(slc=((8, 12), (8, 12), (1, 4)), eps=2.25)]
    thin["sources"][0]["cell"] = (12, 12, 2)
    thin["detectors"] = []
    return {"mod1": c1, "mod2": c2, "mod3_ade": c4, "lossy_walls_mu": lossy, "periodic": per, "thin": thin}


@pytest.mark.parametrize("case", ["mod1", "mod2", "mod3_ade", "lossy_walls_mu", "periodic", "thin"])
def test_ragged_quad_sweeps_equal_one_cell_sweeps_bitwise(case, monkeypatch):
    """The quad sweeps over rows whose length is no multiple of four against one cell per lane: the
    same operations in the same order, so every state agrees bit for bit."""
    import torch

    from fdtdx_amd import fdtd as F
    import scenarios

    spec = _ragged_cases()[case]
    assert spec["shape"][2] % 4 != 0
    out = {}
    for mode in ("two", "quad"):
        _set_mode(monkeypatch, mode)
        objects, arrays, params, config = scenarios.build(spec)
        rec = 0 if case == "mod3_ade" else spec["T"]
        s = F.Solve(objects, config, arrays, record_steps=rec)
        assert s.plan.quad == (mode == "quad")
        arrays.reset()
        print(f"case {case} mode {mode}", flush=True)
        s.forward(0, spec["T"], record=bool(rec))
        torch.cuda.synchronize()
        out[mode] = [arrays.fields.E.cpu().numpy(), arrays.fields.H.cpu().numpy(), arrays.psi.cpu().numpy()]
        out[mode] += [s.record.cpu().numpy()] if s.record is not None else []
        out[mode] += [t.cpu().numpy() for t in s.det_tensors()]
    assert np.abs(out["two"][0]).max() > 0
    for a, b in zip(out["quad"], out["two"]):
        assert np.array_equal(a, b)


def test_gaussian_mode_overlap_matches_oracle():
    """GaussianModeOverlapDetector (detectors/mode.py:666-798): the engine's 6-component phasor
    plane and the overlap with the diverging Gaussian reference at three frequencies against the
    oracle's phasors and its own overlap (mode_overlap, unit-flux gaussian_mode)."""
    from scenarios import mode_spec, oracle_modes

    spec = mode_spec()
    objects, arrays = _run(spec)
    det = next(o for o in objects.detectors if o.name == "mode")
    ov = det.compute_overlap(arrays.detector_states["mode"]).cpu().numpy()
    st, ds = O.run(S.build_scene(spec), spec["T"])
    ph = ds[2]
    assert rel(arrays.detector_states["mode"]["phasor"].cpu().numpy(), ph) < 1e-5
    ref = np.array([O.mode_overlap(ph[0, f], mE, mH, 0) for f, (mE, mH) in enumerate(oracle_modes(spec))])
    print("mode overlaps", ov, ref, flush=True)
    assert np.abs(ref).min() > 0
    assert rel(ov, ref) < 1e-5


def test_mode_source_and_mode_overlap_match_oracle():
    """ModePlaneSource (mode.py:21-306) and the solver-based ModeOverlapDetector
    (detectors/mode.py:448-597) in a strip waveguide: the engine launches the fundamental mode of
    its own solver; the oracle injects the same mode (solved on its own permittivity raster) through
    its TFSF plane tables. E, H, both flux traces, the phasor planes and the overlaps at three
    frequencies agree within 1e-5; the launch is one-way (backward flux below 1 % of forward) and
    the mode carries over 97 % of the phasor power at the overlap plane."""
    from scenarios import oracle_solver_modes, waveguide_spec, with_oracle_mode

    spec = waveguide_spec(T=600)
    objects, arrays = _run(spec)
    det = next(o for o in objects.detectors if o.name == "mode")
    ov = det.compute_overlap(arrays.detector_states["mode"]).cpu().numpy()
    ospec = with_oracle_mode(spec)
    st, ds = O.run(S.build_scene(ospec), spec["T"])
    assert rel(arrays.fields.E.cpu().numpy(), st.E) < 1e-5
    assert rel(arrays.fields.H.cpu().numpy(), st.H) < 1e-5
    back = arrays.detector_states["back"]["poynting_flux"].cpu().numpy()
    fwd = arrays.detector_states["flux"]["poynting_flux"].cpu().numpy()
    assert rel(back, ds[0]) < 1e-5 and rel(fwd, ds[1]) < 1e-5
    assert rel(arrays.detector_states["mode"]["phasor"].cpu().numpy(), ds[2]) < 1e-5
    ref = np.array([O.mode_overlap(ds[2][0, f], mE, mH, 0) for f, (mE, mH) in enumerate(oracle_solver_modes(spec))])
    print("mode overlaps", ov, ref, "back/fwd", back.sum() / fwd.sum(), flush=True)
    assert rel(ov, ref) < 1e-5
    assert abs(back.sum()) < 0.01 * fwd.sum()
    p = ds[3][0, 0]  # Ey, Ez, Hy, Hz phasors of the carrier frequency on the core's plane
    power = 0.5 * np.real(np.sum(p[0] * np.conj(p[3]) - p[1] * np.conj(p[2])))
    assert abs(ov[1]) ** 2 > 0.97 * power


def test_bloch_phases_match_oracle():
    """Complex fields with Bloch phases on x and y (bloch.py:61-97): the real and imaginary parts'
    sweeps couple across the periodic faces; every detector kind reads the complex fields,
    stencils crossing the faces included."""
    from scenarios import bloch_spec

    spec = bloch_spec()
    objects, arrays = _run(spec)
    assert arrays.fields.E.is_complex()
    sc = S.build_scene(spec)
    assert sc.complex_fields and sc.periodic == (True, True, False)
    st, ds = O.run(sc, spec["T"])
    E = arrays.fields.E.cpu().numpy()
    H = arrays.fields.H.cpu().numpy()
    print("E", rel(E, st.E), "H", rel(H, st.H), flush=True)
    assert np.abs(st.E.imag).max() > 1e-2 * np.abs(st.E).max()
    assert rel(E, st.E) < 1e-5 and rel(H, st.H) < 1e-5
    keys = [("flux", "poynting_flux"), ("ph", "phasor"), ("en", "energy"), ("phr", "phasor"), ("fld", "fields"),
            ("fl3", "poynting_flux")]
    for (name, key), ref in zip(keys, ds):
        got = arrays.detector_states[name][key].cpu().numpy()
        print(name, rel(got, ref), flush=True)
        assert got.shape == ref.shape and rel(got, ref) < 1e-5, name


@pytest.mark.parametrize("nz", [28, 29, 31])
@pytest.mark.parametrize("case", ["bloch", "all_axes", "lossy", "poles", "lossy_poles"])
def test_complex_quad_sweeps_equal_one_cell_sweeps_bitwise(nz, case, monkeypatch):
    """Both parts of complex fields four z cells per lane in one launch against a launch per part and
    one cell per lane: fields, psi, poles and detectors agree bit for bit, with Bloch phases on two and
    on all three axes, rows of any length, a magnetic box, conductivity and poles (both together run one
    cell per lane)."""
    from scenarios import bloch_spec
    import scenarios

    from fdtdx_amd import fdtd as F

    spec = bloch_spec(T=41, shape=(20, 16, nz))
    if case == "all_axes":
        spec["pml"] = dict(spec["pml"], types={f"{s}_{a}": "bloch" for s in ("min", "max") for a in "xyz"})
        spec["bloch_vector"] = spec["bloch_vector"][:2] + (0.6 / (nz * spec["dx"]),)
        spec["boxes"] = [dict(slc=((6, 13), (3, 11), (12, nz)), eps=(2.5, 3.0, 2.0), mu=1.5)]
    w = 2.5e15
    if "lossy" in case:
        spec["boxes"] += [dict(slc=((0, 5), (0, 16), (9, 15)), eps=2.0, sigma_H=1e9),
                          dict(slc=((8, 14), (4, 7), (9, 15)), eps=2.0, sigma_E=2e4)]
    if "poles" in case:
        spec["boxes"] += [dict(slc=((7, 13), (3, 11), (12, 19)), eps=(2.5, 3.0, 2.0),
                               poles=[("lorentz", w, 0.05 * w, 1.2)]),
                          dict(slc=((15, 19), (2, 7), (10, 19)), eps=2.0, poles=[("drude", w, 1e14)])]
    out = {}
    for mode in ("quad", "two"):
        _set_mode(monkeypatch, mode)
        objects, arrays, params, config = scenarios.build(spec)
        F.run_fdtd(arrays, objects, config)
        solve = F._solve_for(objects, config, arrays)
        assert solve.plan.quad == (mode == "quad" and case != "lossy_poles")
        out[mode] = [arrays.fields.E.cpu().numpy(), arrays.fields.H.cpu().numpy(), arrays.psi.cpu().numpy()]
        out[mode] += [arrays.ade_state.cpu().numpy()] if "poles" in case else []
        out[mode] += [t.cpu().numpy() for t in solve.det_tensors()]
    assert np.abs(out["two"][0].imag).max() > 0
    for a, b in zip(out["quad"], out["two"]):
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("magnetic", [False, True])
def test_full_conductivity_tensor_matches_oracle(magnetic):
    """Full electric (and magnetic) conductivity tensors on a full-tensor cube and on a diagonal-
    permittivity box (whose inverse permittivity the engine expands to nine components): per-cell
    A and B matrices, A avg(F) +- B avg(K) (update.py:356-492, 752-822)."""
    from scenarios import tensor_loss_spec

    spec = tensor_loss_spec(magnetic=magnetic)
    objects, arrays = _run(spec)
    assert arrays.electric_conductivity.shape[0] == 9
    st, ds = O.run(S.build_scene(spec), spec["T"])
    E = arrays.fields.E.cpu().numpy()
    H = arrays.fields.H.cpu().numpy()
    print("E", rel(E, st.E), "H", rel(H, st.H), flush=True)
    assert rel(E, st.E) < 1e-5 and rel(H, st.H) < 1e-5
    for q, name in enumerate(("ez", "flux")):
        got = next(iter(arrays.detector_states[name].values())).cpu().numpy()
        print(name, rel(got, ds[q]), flush=True)
        assert rel(got, ds[q]) < 1e-5


@pytest.mark.parametrize("sigma", [False, True])
def test_oriented_and_tensor_ade_match_oracle(sigma):
    """ADE poles in the full-tensor update (update.py:361-423): an oriented Lorentz pole (nine-
    component coupling with the symmetrized four-point means) in a diagonal-permittivity box that
    the engine expands to a full tensor, touching a full-tensor box with an isotropic Lorentz pole
    and an oriented Drude pole; optionally a full conductivity tensor on the second box."""
    from scenarios import oriented_ade_spec

    spec = oriented_ade_spec(sigma=sigma)
    objects, arrays = _run(spec)
    assert arrays.inv_permittivities.shape[0] == 9
    st, ds = O.run(S.build_scene(spec), spec["T"])
    E = arrays.fields.E.cpu().numpy()
    H = arrays.fields.H.cpu().numpy()
    print("E", rel(E, st.E), "H", rel(H, st.H), flush=True)
    assert rel(E, st.E) < 1e-5 and rel(H, st.H) < 1e-5
    for q, name in enumerate(("ez", "flux")):
        got = next(iter(arrays.detector_states[name].values())).cpu().numpy()
        print(name, rel(got, ds[q]), flush=True)
        assert rel(got, ds[q]) < 1e-5
