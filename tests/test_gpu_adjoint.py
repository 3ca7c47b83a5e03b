"""GPU parity of the reversible gradient (fdtdx_reverse_adjoint through torch.autograd) against the
oracle's reversible adjoint and FP64 central finite differences."""

import numpy as np
import pytest

from fdtdx_amd import scenarios as W
from oracle import fdtd_oracle as O
from oracle import scenes as S

pytestmark = pytest.mark.gpu


def _grad_gpu(spec, num_checkpoints=0, max_record_bytes=None):
    import torch

    import fdtdx_amd as fx

    objects, arrays, params, config = W.build(spec, gradient=True)
    config.gradient_config.num_checkpoints_reversible = num_checkpoints
    config.gradient_config.max_record_bytes = max_record_bytes
    rho = torch.tensor(np.asarray(spec["design"]["rho"], np.float32), device="cuda", requires_grad=True)
    arrays2, objects2, _ = fx.apply_params(arrays, objects, {"design": rho})
    _, arrays3 = fx.run_fdtd(arrays2, objects2, config)
    flux = arrays3.detector_states["flux"]["poynting_flux"]
    loss = flux.sum()
    loss.backward()
    torch.cuda.synchronize()
    return rho.grad.detach().cpu().numpy().astype(np.float64), flux.detach().cpu().numpy()


def _grad_oracle(spec, dtype=np.float32, num_checkpoints=0):
    sc = S.build_scene(spec, dtype)
    grad, ds, _ = O.reversible_gradient(sc, spec["T"], lambda ds: [np.ones_like(ds[0])], num_checkpoints,
                                        recorder_modules=spec.get("recorder"))
    d = spec["design"]
    slc = tuple(slice(*r) for r in d["slc"])
    rho = np.asarray(d["rho"], np.float64)
    eps = d["eps_a"] + rho * (d["eps_b"] - d["eps_a"])
    return grad[(0, *slc)].astype(np.float64) * (-(d["eps_b"] - d["eps_a"]) / eps**2), ds[0]


def test_reversible_gradient_matches_oracle_and_fd():
    spec = W.scenario_c3(T=160, shape=(34, 30, 28), pml=5, design=(8, 8, 6))
    print("case c3-small", spec["shape"], spec["T"], flush=True)
    g_gpu, flux = _grad_gpu(spec)
    g_or, flux_or = _grad_oracle(spec)
    rel_flux = np.linalg.norm(flux - flux_or) / np.linalg.norm(flux_or)
    rel_g = np.linalg.norm(g_gpu - g_or) / np.linalg.norm(g_or)
    print("flux rel", rel_flux, "grad rel vs oracle", rel_g, flush=True)
    assert rel_flux < 1e-5
    assert rel_g < 1e-4
    d = spec["design"]
    rho = np.asarray(d["rho"], np.float64)

    def scene_fn(r):
        s2 = dict(spec)
        s2["design"] = dict(d, rho=r)
        return S.build_scene(s2, np.float64)

    rng = np.random.default_rng(3)
    for _ in range(3):
        idx = tuple(int(rng.integers(0, n)) for n in rho.shape)
        fd = O.flux_loss_and_grad_fd(scene_fn, rho, idx, 1e-3, spec["T"])
        print("voxel", idx, "gpu", g_gpu[idx], "fd", fd, flush=True)
        assert abs(g_gpu[idx] - fd) <= 1e-3 * abs(fd)


def test_sliced_gradient_matches_oracle():
    """num_checkpoints_reversible = 3 (fdtd.py:106-121, 295-313): resets at the slice cuts."""
    spec = W.scenario_c3(T=120, shape=(30, 28, 24), pml=5, design=(8, 8, 6))
    print("case sliced", spec["shape"], spec["T"], flush=True)
    g_gpu, _ = _grad_gpu(spec, num_checkpoints=3)
    g_or, _ = _grad_oracle(spec, num_checkpoints=3)
    g_or1, _ = _grad_oracle(spec, num_checkpoints=0)
    rel = np.linalg.norm(g_gpu - g_or) / np.linalg.norm(g_or)
    print("sliced grad rel vs oracle", rel, "unsliced oracle differs by",
          np.linalg.norm(g_or1 - g_or) / np.linalg.norm(g_or), flush=True)
    assert rel < 1e-4


@pytest.mark.parametrize("num_checkpoints,recorder", [(0, None), (2, None),
                                                     (2, [("every_k", 4, 0), ("dtype", "bfloat16", ())])])
def test_record_regeneration_is_bit_identical(num_checkpoints, recorder):
    """A record budget of a few slots makes the backward regenerate the interface record chunk
    by chunk from state checkpoints; the gradient must not change by a single bit, also with a
    compressed, time-filtered record."""
    import fdtdx_amd as fx

    spec = W.scenario_c3(T=77, shape=(30, 26, 22), pml=5, design=(8, 8, 6))
    if recorder:
        spec["recorder"] = recorder
    objects, arrays, params, config = W.build(spec, gradient=True)
    from fdtdx_amd.fdtd import lower
    from fdtdx_amd import engine

    rec_bytes = engine.Plan(lower(objects, config, arrays)).record_slot_bytes
    print("case regen", spec["shape"], spec["T"], num_checkpoints, recorder, "record B/slot", rec_bytes, flush=True)
    g_stored, f_stored = _grad_gpu(spec, num_checkpoints)
    g_regen, f_regen = _grad_gpu(spec, num_checkpoints, max_record_bytes=9 * rec_bytes)
    assert np.array_equal(f_stored, f_regen)
    assert np.array_equal(g_stored, g_regen)


def test_gradient_with_conductor_faces_matches_oracle():
    """Transposes of the PEC / PMC zeroing in the adjoint (Z_H on lam_H, Z_E on mu_E)."""
    spec = W.scenario_c3(T=110, shape=(30, 28, 24), pml=5, design=(8, 8, 6))
    spec["pml"] = dict(spec["pml"], types={"max_x": "pec", "min_z": "pmc", "max_y": "pec"})
    print("case walls", spec["shape"], spec["T"], flush=True)
    g_gpu, flux = _grad_gpu(spec)
    g_or, flux_or = _grad_oracle(spec)
    rel_g = np.linalg.norm(g_gpu - g_or) / np.linalg.norm(g_or)
    print("grad rel vs oracle", rel_g, flush=True)
    assert np.linalg.norm(flux - flux_or) <= 1e-5 * np.linalg.norm(flux_or)
    assert rel_g < 1e-4


@pytest.mark.parametrize("num_checkpoints", [0, 2])
def test_gradient_periodic_matches_oracle(num_checkpoints):
    """Wrapped curls in the reverse sweeps and the adjoint, and the wrapped flux stencil."""
    from scenarios import periodic_spec

    spec = periodic_spec(T=90)
    print("case periodic", spec["shape"], spec["T"], num_checkpoints, flush=True)
    g_gpu, flux = _grad_gpu(spec, num_checkpoints)
    g_or, flux_or = _grad_oracle(spec, num_checkpoints=num_checkpoints)
    rel_g = np.linalg.norm(g_gpu - g_or) / np.linalg.norm(g_or)
    print("grad rel vs oracle", rel_g, flush=True)
    assert np.linalg.norm(flux - flux_or) <= 1e-5 * np.linalg.norm(flux_or)
    assert rel_g < 1e-4


def _reverse_cpml_cases():
    base = W.scenario_c3(T=90, shape=(30, 28, 24), pml=5, design=(8, 8, 6))
    (x0, x1), (y0, y1), (z0, z1) = base["design"]["slc"]
    kap = dict(base, pml=dict(base["pml"], params=dict(kappa_start=1.0, kappa_end=3.0), types={"max_x": "pec"}),
               boxes=[dict(slc=((x0 - 2, x1 - 3), (y0 + 1, y1 + 3), (z0 - 2, z1)), eps=1.0, mu=(1.4, 2.2, 1.8),
                           sigma_E=2000.0, sigma_H=2.0e8)])
    adj = W.scenario_c3(T=90, shape=(30, 28, 10), pml=5, design=(8, 8, 4))  # z slabs [0, 5) and [5, 10) touch
    (a, b), (c, e), _ = adj["detectors"][0]["slc"]
    adj["detectors"][0]["slc"] = ((a, b), (c, e), (2, 8))
    from scenarios import periodic_spec
    return {"c3": base, "kappa_mu_loss_pec": kap, "adjacent_z_slabs": adj, "periodic": periodic_spec(T=90)}


@pytest.mark.parametrize("case", ["c3", "kappa_mu_loss_pec", "adjacent_z_slabs", "periodic"])
def test_per_axis_reverse_cpml_equals_slab_loop_bitwise(case, monkeypatch):
    """The reverse H half-step and both adjoint passes with per-axis CPML (each axis's slab found
    from the cell's coordinate, every psi and lam_psi load issued up front) against the slab loop
    (FDTDX_REVERSE_CPML=loop): fluxes and design gradients agree bit for bit, with kappa > 1, a PEC
    face in place of a slab, magnetic and lossy boxes, two z slabs that touch and periodic axes."""
    spec = _reverse_cpml_cases()[case]
    out = {}
    for mode in ("loop", "axes"):
        if mode == "loop":
            monkeypatch.setenv("FDTDX_REVERSE_CPML", "loop")
        else:
            monkeypatch.delenv("FDTDX_REVERSE_CPML", raising=False)
        print("case", case, "reverse cpml", mode, spec["shape"], flush=True)
        out[mode] = _grad_gpu(spec)
    assert np.abs(out["loop"][0]).max() > 0
    assert np.array_equal(out["loop"][1], out["axes"][1])
    assert np.array_equal(out["loop"][0], out["axes"][0])


def _quad_adjoint_cases():
    def c3(shape, pml=5):
        return W.scenario_c3(T=70, shape=shape, pml=pml, design=(8, 8, 4))

    kap = c3((30, 28, 26))  # kappa > 1, diagonal permittivity and permeability
    kap["pml"] = dict(kap["pml"], params=dict(kappa_start=1.0, kappa_end=3.0))
    kap["boxes"] = [dict(slc=((4, 20), (6, 20), (3, 22)), eps=1.0, mu=(1.4, 2.2, 1.8))]
    del kap["design"]
    kap["boxes"].append(dict(slc=((12, 20), (8, 18), (9, 15)), eps=(2.0, 4.0, 3.0)))
    plane = W.scenario_c2(T=60, shape=(40, 30, 27), pml=5, slab=(10, 12, 8))  # E and H source hooks, phasors
    return {"aligned": c3((30, 28, 24), 4), "unaligned_slabs": c3((30, 28, 24)), "mod1": c3((30, 28, 25)),
            "mod2": c3((30, 28, 22)), "mod3": c3((28, 30, 23), 4), "kappa_mu_diag": kap, "plane": plane}


@pytest.mark.parametrize("case", ["aligned", "unaligned_slabs", "mod1", "mod2", "mod3", "kappa_mu_diag", "plane"])
def test_quad_adjoint_equals_one_cell_adjoint_bitwise(case, monkeypatch):
    """The reverse and adjoint sweeps with four z cells per lane against one (FDTDX_REVERSE_CPML=cell):
    the same operations in the same order, so the gradient of the whole permittivity array and the
    detector states agree bit for bit, with z slabs on and inside quads, rows of any length and
    kappa > 1."""
    import torch

    import fdtdx_amd as fx
    import scenarios
    from fdtdx_amd import fdtd

    spec = _quad_adjoint_cases()[case]
    out = {}
    for mode in ("cell", "quad"):
        if mode == "cell":
            monkeypatch.setenv("FDTDX_REVERSE_CPML", "cell")
        else:
            monkeypatch.delenv("FDTDX_REVERSE_CPML", raising=False)
        print("case", case, mode, spec["shape"], flush=True)
        objects, arrays, params, config = scenarios.build(spec, gradient=True)
        assert fdtd.Solve(objects, config, arrays).plan.reverse_quad == (mode == "quad")
        ie = arrays.inv_permittivities.detach().clone().requires_grad_(True)
        arrays.inv_permittivities = ie
        _, arrays = fx.run_fdtd(arrays, objects, config)
        states = [v for st in arrays.detector_states.values() for v in st.values()]
        sum((v.real.sum() + (0.5 * v.imag.sum() if v.is_complex() else 0.0)) for v in states).backward()
        torch.cuda.synchronize()
        out[mode] = [ie.grad.cpu().numpy()] + [v.detach().cpu().numpy() for v in states]
    assert np.abs(out["cell"][0]).max() > 0
    for a, b in zip(out["quad"], out["cell"]):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("num_checkpoints", [0, 2])
def test_gradient_with_conductivity_matches_oracle(num_checkpoints):
    """The lossy reverse update and the transposed loss factors (w_H, w_E, the pass-through of
    lam_H and lam_E, and the inv_eps derivative) with a conducting box over part of the design."""
    spec = W.scenario_c3(T=120, shape=(30, 28, 24), pml=5, design=(8, 8, 6))
    (x0, x1), (y0, y1), (z0, z1) = spec["design"]["slc"]
    spec["boxes"] = [dict(slc=((x0 - 2, x1 - 3), (y0 + 1, y1 + 3), (z0 - 2, z1)), eps=1.0, sigma_E=2000.0,
                          sigma_H=2.5e8)]
    print("case lossy", spec["shape"], spec["T"], num_checkpoints, flush=True)
    g_gpu, flux = _grad_gpu(spec, num_checkpoints)
    g_or, flux_or = _grad_oracle(spec, num_checkpoints=num_checkpoints)
    rel_g = np.linalg.norm(g_gpu - g_or) / np.linalg.norm(g_or)
    print("grad rel vs oracle", rel_g, flush=True)
    assert np.linalg.norm(flux - flux_or) <= 1e-5 * np.linalg.norm(flux_or)
    assert rel_g < 1e-4


@pytest.mark.parametrize("recorder", [
    [("dtype", "bfloat16", ())],
    [("every_k", 3, 0), ("dtype", "float8_e5m2fnuz", ("_H",))],
    [("dtype", "float16", ()), ("every_k", 4, 0)],
    [("every_k", 5, 2)],
])
def test_compressed_record_gradient_matches_oracle(recorder):
    """Recorder compression (modules.py:98-161, time_filter.py:140-257): narrow-float layers, an
    exclude filter, interpolation in float32 (filter first) and in the narrow type (cast first),
    a late recording start."""
    spec = W.scenario_c3(T=100, shape=(30, 28, 24), pml=5, design=(8, 8, 6))
    spec["recorder"] = recorder
    print("case recorder", recorder, flush=True)
    g_gpu, flux = _grad_gpu(spec)
    g_or, flux_or = _grad_oracle(spec)
    rel_g = np.linalg.norm(g_gpu - g_or) / np.linalg.norm(g_or)
    print("grad rel vs oracle", rel_g, flush=True)
    assert np.linalg.norm(flux - flux_or) <= 1e-5 * np.linalg.norm(flux_or)
    assert rel_g < 1e-4


def test_compressed_record_bytes_match_oracle_codes():
    """The record slots the forward writes hold, byte for byte, the oracle's codes of its own
    interface layers at the kept steps (E layers of every slab, then H layers, each 16-byte
    aligned)."""
    import torch

    from fdtdx_amd import fdtd as F
    from oracle import record_codec as R

    spec = W.scenario_c3(T=40, shape=(26, 24, 22), pml=5, design=(6, 6, 4))
    spec["recorder"] = [("every_k", 3, 1), ("dtype", "float8_e5m2fnuz", ("max_y",))]
    objects, arrays, params, config = W.build(spec, gradient=True)
    s = F.Solve(objects, config, arrays, record_steps=spec["T"])
    arrays.reset()
    s.forward(0, spec["T"], record=True)
    torch.cuda.synchronize()
    got = s.record.cpu().numpy()
    sc = S.build_scene(spec)
    rec = []
    O.run(sc, spec["T"], record=rec)
    keys = O.interface_keys(sc)
    save, tta = R.time_filter_tables(spec["T"], 3, 1)
    fmts = [("float32" if "max_y" in k else "float8_e5m2fnuz") for k in keys]
    slot_bytes = s.plan.record_slot_bytes
    assert s.plan.record_slots == len(save)
    for n in save:
        off = 0
        base = int(tta[n]) * slot_bytes
        for key, vals, fmt in zip(keys, rec[n], fmts):
            codes = R.encode(vals.reshape(-1), fmt)
            w = R.width(fmt) if fmt != "float32" else 4
            raw = got[base + off: base + off + codes.size * w].view(codes.dtype if fmt != "float32" else np.uint32)
            assert np.array_equal(raw, codes), (n, key)
            off = (off + codes.size * w + 15) // 16 * 16


@pytest.mark.parametrize("num_checkpoints,mu,sigma_H", [(0, (1.4, 2.2, 1.8), 0.0), (2, 1.7, 2.0e8)])
def test_gradient_with_kappa_and_permeability_matches_oracle(num_checkpoints, mu, sigma_H):
    """CPML with kappa > 1 (the (1/kappa - 1) d term of the correction) and a diagonal or
    isotropic permeability box (with magnetic loss) over part of the design."""
    spec = W.scenario_c3(T=110, shape=(30, 28, 24), pml=5, design=(8, 8, 6))
    (x0, x1), (y0, y1), (z0, z1) = spec["design"]["slc"]
    spec["pml"] = dict(spec["pml"], params=dict(kappa_start=1.0, kappa_end=3.0))
    spec["boxes"] = [dict(slc=((x0 - 2, x1 - 3), (y0 + 1, y1 + 3), (z0 - 2, z1)), eps=1.0, mu=mu, sigma_H=sigma_H)]
    print("case kappa/mu", mu, sigma_H, num_checkpoints, flush=True)
    g_gpu, flux = _grad_gpu(spec, num_checkpoints)
    g_or, flux_or = _grad_oracle(spec, num_checkpoints=num_checkpoints)
    rel_g = np.linalg.norm(g_gpu - g_or) / np.linalg.norm(g_or)
    print("grad rel vs oracle", rel_g, flush=True)
    assert np.linalg.norm(flux - flux_or) <= 1e-5 * np.linalg.norm(flux_or)
    assert rel_g < 1e-4


def test_gradient_through_every_detector_kind_matches_oracle():
    """One backward per detector of detector_zoo_spec, each with that detector's loss (|phasor|^2
    through torch's complex autograd, weighted field means, energy, unreduced three-component
    flux), against the oracle's reversible gradient with the same cotangent. The energy
    detector's gradient includes its direct inv_eps term."""
    import torch

    import fdtdx_amd as fx
    from scenarios import detector_zoo_losses, detector_zoo_spec

    spec = detector_zoo_spec(T=120)
    sc = S.build_scene(spec, np.float32)
    rng = np.random.default_rng(8)
    st = [O.init_detector_state(d, sc) for d in sc.detectors]
    weights = dict(fld=rng.standard_normal(st[3].shape), fl3=rng.standard_normal(st[5].shape))
    keys = dict(flux="poynting_flux", ph="phasor", phr="phasor", fld="fields", en="energy", fl3="poynting_flux")
    d = spec["design"]
    slc = tuple(slice(*r) for r in d["slc"])
    rho0 = np.asarray(d["rho"], np.float64)
    deps = -(d["eps_b"] - d["eps_a"]) / (d["eps_a"] + rho0 * (d["eps_b"] - d["eps_a"])) ** 2
    objects, arrays, params, config = W.build(spec, gradient=True)
    for q, det in enumerate(spec["detectors"]):
        print("case detector", det["name"], flush=True)
        rho = torch.tensor(np.asarray(d["rho"], np.float32), device="cuda", requires_grad=True)
        arrays2, objects2, _ = fx.apply_params(arrays, objects, {"design": rho})
        _, arrays3 = fx.run_fdtd(arrays2, objects2, config)
        ds = [arrays3.detector_states[x["name"]][keys[x["name"]]] for x in spec["detectors"]]
        w = {k: torch.tensor(v, dtype=torch.float32, device="cuda") for k, v in weights.items()}
        losses = [ds[0].sum(), (ds[1].abs() ** 2).sum(), (ds[2].abs() ** 2).sum(), (w["fld"] * ds[3]).sum(),
                  ds[4].sum(), (w["fl3"] * ds[5]).sum()]
        losses[q].backward()
        torch.cuda.synchronize()
        g_gpu = rho.grad.detach().cpu().numpy().astype(np.float64)

        def cot_fn(dso, q=q):
            _, cots = detector_zoo_losses(dso, weights)
            return [c if i == q else None for i, c in enumerate(cots)]

        g, _, _ = O.reversible_gradient(sc, spec["T"], cot_fn)
        g_or = g[(0, *slc)].astype(np.float64) * deps
        r = np.linalg.norm(g_gpu - g_or) / np.linalg.norm(g_or)
        print(det["name"], "grad rel vs oracle", r, flush=True)
        assert r < 1e-4


def test_gradient_through_surface_detectors_matches_oracle():
    """One backward per surface detector loss of surface_zoo_spec: the net flux through a closed
    box (the engine's accumulating face detectors share one cotangent), the phasor flux and the net
    phasor flux (post-processed on the device, differentiated by torch autograd into the phasor
    cotangents), against the oracle's reversible gradient with the same cotangents."""
    import torch

    import fdtdx_amd as fx
    from scenarios import surface_zoo_losses, surface_zoo_spec

    spec = surface_zoo_spec(T=120)
    sc = S.build_scene(spec, np.float32)
    names = [x["name"] for x in sc.detectors]
    d = spec["design"]
    slc = tuple(slice(*r) for r in d["slc"])
    rho0 = np.asarray(d["rho"], np.float64)
    deps = -(d["eps_b"] - d["eps_a"]) / (d["eps_a"] + rho0 * (d["eps_b"] - d["eps_a"])) ** 2
    objects, arrays, params, config = W.build(spec, gradient=True)
    pf = next(o for o in objects.detectors if isinstance(o, fx.PhasorPoyntingFluxDetector))
    cp = next(o for o in objects.detectors if isinstance(o, fx.ClosedSurfacePhasorPoyntingFluxDetector))
    for key in ("cf", "pf", "cp"):
        print("case detector", key, flush=True)
        rho = torch.tensor(np.asarray(d["rho"], np.float32), device="cuda", requires_grad=True)
        arrays2, objects2, _ = fx.apply_params(arrays, objects, {"design": rho})
        _, arrays3 = fx.run_fdtd(arrays2, objects2, config)
        st = arrays3.detector_states
        loss = {"cf": lambda: st["cf"]["poynting_flux"].sum(),
                "pf": lambda: pf.compute_poynting_flux(st["pf"]).sum(),
                "cp": lambda: cp.compute_net_flux(st["cp"]).sum()}[key]()
        loss.backward()
        torch.cuda.synchronize()
        g_gpu = rho.grad.detach().cpu().numpy().astype(np.float64)

        def cot_fn(dso, key=key):
            return [surface_zoo_losses(dso, names, spec, float(np.float32(spec["dx"])))[1][key].get(nm)
                    for nm in names]

        g, _, _ = O.reversible_gradient(sc, spec["T"], cot_fn)
        g_or = g[(0, *slc)].astype(np.float64) * deps
        r = np.linalg.norm(g_gpu - g_or) / np.linalg.norm(g_or)
        print(key, "grad rel vs oracle", r, flush=True)
        assert r < 1e-4


@pytest.mark.parametrize("periodic", [False, True])
def test_full_tensor_gradient_matches_oracle(periodic):
    """dL/d inv_eps of every one of the nine components (the flux-sum loss) through non-symmetric
    full-tensor permittivity and permeability, against the oracle's reversible adjoint over the
    whole grid; the curl buffers, transposed four-point means and off-diagonal gradient are all
    exercised."""
    import torch

    import fdtdx_amd as fx
    from scenarios import tensor_spec

    spec = tensor_spec(T=100, periodic=periodic)
    spec["detectors"] = spec["detectors"][1:]  # the flux plane
    objects, arrays, params, config = W.build(spec, gradient=True)
    ie = arrays.inv_permittivities.detach().clone().requires_grad_(True)
    arrays.inv_permittivities = ie
    _, arrays2 = fx.run_fdtd(arrays, objects, config)
    flux = arrays2.detector_states["flux"]["poynting_flux"]
    flux.sum().backward()
    torch.cuda.synchronize()
    g_gpu = ie.grad.detach().cpu().numpy().astype(np.float64)
    sc = S.build_scene(spec, np.float32)
    g_or, ds, _ = O.reversible_gradient(sc, spec["T"], lambda d: [np.ones_like(d[0])])
    g_or = g_or.astype(np.float64)
    fl = flux.detach().cpu().numpy().astype(np.float64)
    print("flux rel", np.linalg.norm(fl - ds[0]) / np.linalg.norm(ds[0].astype(np.float64)), flush=True)
    # outside the CPML, where the reconstruction is exact (inside it both use the frozen final psi
    # and the reconstruction error grows, so float32 rounding differences are amplified there)
    p = 6
    inner = (slice(None), slice(p, -p), slice(p, -p), slice(p, -p))
    for comp in range(9):
        a, b = g_gpu[comp][inner[1:]], g_or[comp][inner[1:]]
        r = np.linalg.norm(a - b) / np.linalg.norm(b)
        print("component", comp, "grad rel", r, "max", np.abs(b).max(), flush=True)
        assert r < 1e-4


@pytest.mark.parametrize("symmetry,e_pol", [((0, -1, 1), (0, 1, 0)), ((0, 1, -1), (0, 0, 1))])
def test_symmetry_reduced_gradient_matches_oracle(symmetry, e_pol):
    """The reversible gradient of a symmetry-reduced run (the flux plane's transposed stencils fold
    the electric plane's mirror halo back onto rows 0 and 1) against the oracle's reduced
    gradient."""
    from scenarios import symmetry_spec

    import torch

    import fdtdx_amd as fx

    spec = symmetry_spec(symmetry=symmetry, e_pol=e_pol, T=120)
    spec["detectors"] = spec["detectors"][:1]
    print("case symmetry", symmetry, flush=True)
    red = S.reduce_spec(spec)  # the kept part of the design
    objects, arrays, params, config = W.build(spec, gradient=True)
    rho = torch.tensor(np.asarray(red["design"]["rho"], np.float32), device="cuda", requires_grad=True)
    arrays2, objects2, _ = fx.apply_params(arrays, objects, {"design": rho})
    _, arrays3 = fx.run_fdtd(arrays2, objects2, config)
    flux_t = arrays3.detector_states["flux"]["poynting_flux"]
    flux_t.sum().backward()
    torch.cuda.synchronize()
    g_gpu = rho.grad.detach().cpu().numpy().astype(np.float64)
    flux = flux_t.detach().cpu().numpy()
    g_or, flux_or = _grad_oracle(red)
    r = np.linalg.norm(g_gpu - g_or) / np.linalg.norm(g_or)
    print("flux rel", np.linalg.norm(flux - flux_or) / np.linalg.norm(flux_or), "grad rel", r, flush=True)
    assert np.linalg.norm(flux - flux_or) / np.linalg.norm(flux_or) < 1e-5
    assert r < 1e-4


def test_energy_slices_gradient_matches_oracle():
    """dL/d inv_eps through the collapsed-axis energy means (each plane cell's cotangent spread
    along the axis, plus the direct inv_eps term) and through an indexed plane, against the
    oracle."""
    import torch

    import fdtdx_amd as fx
    from scenarios import energy_slices_spec

    spec = energy_slices_spec()
    objects, arrays, params, config = W.build(spec, gradient=True)
    ie = arrays.inv_permittivities.detach().clone().requires_grad_(True)
    arrays.inv_permittivities = ie
    _, arrays2 = fx.run_fdtd(arrays, objects, config)
    st = arrays2.detector_states
    rng = np.random.default_rng(5)
    w_mean = rng.standard_normal(tuple(st["mean"]["XZ Plane"].shape))
    w_plane = rng.standard_normal(tuple(st["planes"]["YZ Plane"].shape))
    loss = (torch.tensor(w_mean, dtype=torch.float32, device="cuda") * st["mean"]["XZ Plane"]).sum() + \
        (torch.tensor(w_plane, dtype=torch.float32, device="cuda") * st["planes"]["YZ Plane"]).sum()
    loss.backward()
    torch.cuda.synchronize()
    g_gpu = ie.grad.detach().cpu().numpy().astype(np.float64)
    sc = S.build_scene(spec, np.float32)

    def cot_fn(ds):
        out = [None] * len(ds)
        out[1] = w_mean.astype(np.float32)
        out[5] = w_plane.reshape(ds[5].shape).astype(np.float32)
        return out

    g_or, _, _ = O.reversible_gradient(sc, spec["T"], cot_fn)
    inner = (slice(None), slice(5, -5), slice(5, -5), slice(5, -5))
    r = np.linalg.norm(g_gpu[inner] - g_or[inner]) / np.linalg.norm(g_or[inner])
    print("grad rel", r, flush=True)
    assert r < 1e-4


@pytest.mark.parametrize("reset", [True, False])
def test_full_backward_matches_oracle(reset):
    """full_backward after a recorded forward (reversible_fdtd without a gradient keeps the
    interface record): the fields after reversing to step 30 and the inverse field, phasor and
    energy detectors match the oracle's time-reversed run."""
    import torch

    import fdtdx_amd as fx
    import scenarios as SC

    T, T0 = 80, 30
    spec = SC.backward_spec(T)
    objects, arrays, params, config = SC.build(spec, gradient=True)
    print(f"case full_backward reset={reset} shape={spec['shape']} T={T}", flush=True)
    t, arrays = fx.run_fdtd(arrays, objects, config)
    t, arrays = fx.full_backward((t, arrays), objects, config, reset_fields=reset, start_time_step=T0)
    torch.cuda.synchronize()
    assert t == T0
    sc = S.build_scene(spec)
    rec = []
    st, ds = O.run(sc, T, record=rec)
    O.full_backward(st, sc, T, T0, rec, ds, reset_fields=reset)
    names = [d["name"] for d in sc.detectors]

    def rel(a, b):
        a, b = np.asarray(a, np.complex128), np.asarray(b, np.complex128)
        return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300))

    assert rel(arrays.fields.E.cpu().numpy(), st.E) < 1e-5
    assert rel(arrays.fields.H.cpu().numpy(), st.H) < 1e-5
    got = arrays.detector_states
    assert rel(got["fwd"]["fields"].cpu().numpy(), ds[names.index("fwd")]) < 1e-5
    assert rel(got["ifld"]["fields"].cpu().numpy(), ds[names.index("ifld")]) < 1e-5
    assert rel(got["iph"]["phasor"].cpu().numpy(), ds[names.index("iph")]) < 1e-5
    assert rel(got["ien"]["energy"].cpu().numpy().reshape(-1), ds[names.index("ien")].reshape(-1)) < 1e-5
    # one more reversed step through backward()
    t, arrays = fx.backward((t, arrays), config, objects, reset_fields=reset)
    torch.cuda.synchronize()
    O.full_backward(st, sc, T0, T0 - 1, rec, ds, reset_fields=reset)
    assert t == T0 - 1
    assert rel(arrays.fields.E.cpu().numpy(), st.E) < 1e-5


def test_full_backward_with_conductivity_tensors_matches_oracle():
    """The time-reversed run through full-tensor media with full conductivity tensors: inside the
    conductivity boxes E = A_rev avg(E) - B_rev avg(K) and H = A_rev avg(H) + B_rev avg(K)
    (update.py:611-680, 930-1000). Undoing a lossy step amplifies rounding: over these 20 reversed
    steps the oracle's float32 and float64 runs differ by about 7e-6, hence the 5e-5 bound."""
    import torch

    import fdtdx_amd as fx
    import scenarios as SC

    T, T0 = 80, 60
    spec = SC.tensor_loss_spec(T=T)
    objects, arrays, params, config = SC.build(spec, gradient=True)
    print(f"case full_backward conductivity tensors shape={spec['shape']} T={T}", flush=True)
    t, arrays = fx.run_fdtd(arrays, objects, config)
    t, arrays = fx.full_backward((t, arrays), objects, config, reset_fields=False, start_time_step=T0)
    torch.cuda.synchronize()
    sc = S.build_scene(spec)
    rec = []
    st, ds = O.run(sc, T, record=rec)
    O.full_backward(st, sc, T, T0, rec, ds, reset_fields=False)

    def rel(a, b):
        return float(np.linalg.norm(np.asarray(a, np.float64) - b) / np.linalg.norm(np.asarray(b, np.float64)))

    rE, rH = rel(arrays.fields.E.cpu().numpy(), st.E), rel(arrays.fields.H.cpu().numpy(), st.H)
    print("E", rE, "H", rH, flush=True)
    assert rE < 5e-5 and rH < 5e-5
