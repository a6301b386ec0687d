"""The explicit stage inside the tile kernel (k_stage_tile) against the separate
gradient, flux, sum and update kernels of the same step (fused = 0): the same
operations in the same order, so the same bits, ghost rows included."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# a mesh of one tile, tiles of few cells, the automatic ones (a thread to a cell),
# and tiles whose rings and faces take the threads more than one turn
@pytest.mark.parametrize("ni,nj,tile", [(16, 4, 0), (31, 12, 16), (64, 40, 0), (64, 40, 224)])
@pytest.mark.parametrize("model,opts", [("inviscid", {}), ("laminar", {}), ("inviscid", {"second_order": False}),
                                        ("laminar", {"second_order": False}), ("inviscid", {"limiter": "michalak"}),
                                        ("laminar", {"gradient_scheme": "least-squares"})])
def test_steps_equal_the_separate_kernels(ni, nj, tile, model, opts):
    from aeroflex_amd import rans
    m = rans.Mesh.jittered(ni, nj, r_far=20.0 if nj > 10 else 3.0, first_h=2e-3 if nj > 10 else 0.3, seed=3,
                           quad_frac=0.3)
    far = rans.BoundaryVariables(mach=0.5, angle=0.03)
    out = []
    for fused in (True, False):
        s = rans.Solver(m, gas=rans.Gas(mu_L=1e-3), viscosity_model=model, tile_cells=tile, fused=fused, **opts)
        s.set_bcs({"farfield": rans.BoundaryCondition("farfield", far),
                   "wall": rans.BoundaryCondition("wall" if model == "laminar" else "slip-wall")})
        s.init()
        s.refill_bcs()
        s.set_cfl(0.4)
        q = s.get_q()
        q[:4 * s.n_real] *= 1.0 + 1e-2 * np.random.default_rng(5).standard_normal(4 * s.n_real)
        s.set_q(q)
        err = [s.explicit_solve(0.8) for _ in range(3)]
        out.append((s.get_q(), np.array(err)))
    (a, ea), (b, eb) = out
    assert np.isfinite(a).all()
    if opts.get("gradient_scheme") == "least-squares":
        # the tile kernel takes x_other - x_cell from the face offsets: three
        # steps of last-bit differences in the gradients
        assert np.max(np.abs(a - b)) <= 1e-11 * np.max(np.abs(b))
        assert np.max(np.abs(ea - eb)) <= 1e-9 * np.max(eb)
    else:
        assert np.array_equal(a, b)
        assert np.array_equal(ea, eb)
