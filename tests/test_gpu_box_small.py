"""Coarsest levels that one work-group holds in LDS or that take two sweeps per
launch: sweeps and early exit against the patch-wise passes and the
grid-parallel sweep, bit for bit."""
import numpy as np
import pytest

import hier_cases as hc

pytestmark = pytest.mark.gpu

KEYS = dict(max_cycles=2, residual_tol=1e-300, relative_residual_tol=1e-300, num_pre_sweeps=1,
            num_post_sweeps=1, coarse_solver_choice="redblack")


def one_level(*n):
    """A domain of n cells in two patches (the last one decides the early
    exit), cut at an even index in x (2-D colours are patch-relative)."""
    dim = len(n)
    hi = tuple(v - 1 for v in n)
    cut = n[0] // 2 // 2 * 2
    if cut == 0:
        boxes = [((0,) * dim, hi)]
    else:
        boxes = [((0,) * dim, (cut - 1,) + hi[1:]), ((cut,) + (0,) * (dim - 1), hi)]
    return dict(name="x".join(map(str, n)), dim=dim, levels=[boxes], ratio=2, dlo=(0,) * dim,
                dhi=hi)


def solve(case, data, spec, keys, fused, variant, bits):
    from samrai_amd import fac
    dim = case["dim"]
    n0 = np.array(case["dhi"]) + 1
    h = fac.PatchHierarchy(dim, case["dlo"], case["dhi"], [0.0] * 3,
                           list(n0 / n0.min()) + [1.0] * (3 - dim))
    h.add_level(1, case["levels"][0])
    h.finalize()
    u, f = fac.PatchData(h, 1), fac.PatchData(h, 0)
    D = fac.PatchData(h, 0, "side") if spec["dvar"] else None
    C = fac.PatchData(h, 0) if spec["cmode"] == 2 else None
    for p in range(len(case["levels"][0])):
        f.put(0, p, data["f"][0][p])
        if C is not None:
            C.put(0, p, data["C"][0][p])
        if D is not None:
            for a in range(dim):
                D.put(0, p, data["D"][0][p][a], axis=a)
    s = fac.CellPoissonFACSolver(h, **dict(KEYS, **keys))
    if D is not None:
        s.set_d_patch_data(D)
    if C is not None:
        s.set_c_patch_data(C)
    elif spec["cmode"] == 1:
        s.set_c_constant(-0.7)
    bc = hc.bc_robin(dim) if spec["robin"] else hc.BC_DIRICHLET
    s.set_boundaries(bc["a"][:2 * dim], bc["b"][:2 * dim], bc["g"][:2 * dim])
    s.initialize_solver_state(u, f)
    s.set_coarse_precision(bits)
    s.set_fused_coarsest(fused, variant)
    s.solve_system(u, f)
    out = [u.get(0, p) for p in range(len(case["levels"][0]))]
    e, r = s.internal_vector("e"), s.internal_vector("r")
    e.fill(0.0)
    count = s.smooth(e, r, 0, 9, tol=keys["coarse_solver_tolerance"])
    return out, np.array(s.history()), count


# slots per colour and thread 1, 2, 4 and (FP32 in 2-D) 8, the last sizes
# that one work-group takes and the first that go to pairs, which calls of fewer
# than 16 sweeps do from 4 slots on; odd rows, one-cell-wide and thin domains
SIZES = [(3, 2, 2), (1, 5, 7), (9, 10, 11), (13, 17, 15), (16, 16, 16), (17, 16, 16), (32, 16, 16),
         (34, 16, 16), (2, 40, 40), (5, 3), (31, 23), (64, 64), (65, 64), (90, 91), (128, 64),
         (130, 64), (300, 9),
         # two sweeps per launch: both 3-D tiles, ragged ends of each, a last
         # patch smaller than a tile's halo, and the first size past the rule
         (33, 31, 35), (37, 41, 29), (6, 70, 40), (54, 53, 53), (251, 130)]


@pytest.mark.parametrize("spec", [dict(dvar=False, cmode=0, robin=False),
                                  dict(dvar=False, cmode=1, robin=True),
                                  dict(dvar=True, cmode=2, robin=True)],
                         ids=["constD", "constD-constC-robin", "varD-varC-robin"])
@pytest.mark.parametrize("n", SIZES, ids=lambda n: "x".join(map(str, n)))
def test_lds_sweeps_are_bit_identical(gpu_lib, n, spec):
    """Solution, residual history, sweep count and maximum residual of the
    early exit equal those of the patch-wise passes; the FP32 coarse solve
    equals the grid-parallel sweep's.  Sweep counts odd and even, with a
    tolerance that stops the loop and one that does not."""
    case = one_level(*n)
    data = hc.make_data(case, seed=sum(n))
    # (13, 0.9) and (40, 0.5) stop after odd and even sweeps on different sizes
    for sweeps, tol in ((7, 1e-300), (40, 0.5), (13, 0.9), (8, 1e-300)):
        print("lds sweeps", case["name"], spec, sweeps, tol, flush=True)
        keys = dict(coarse_solver_max_iterations=sweeps, coarse_solver_tolerance=tol)
        for bits, fused, variant in ((64, False, 0), (32, True, 0)):
            ref = solve(case, data, spec, keys, fused, variant, bits)
            got = solve(case, data, spec, keys, True, -1, bits)
            assert got[2] == ref[2]
            np.testing.assert_array_equal(got[1], ref[1])
            for a, b in zip(got[0], ref[0]):
                np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("n,tiled", [((64, 64), False), ((53, 53, 53), False),
                                     ((56, 55, 54), True), ((512, 600), True)],
                         ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v))
def test_tile_shape_is_tuned_only_where_tiles_run(gpu_lib, n, tiled):
    """A level whose sweeps run in one work-group or two per launch reports no
    tile shape and times none at set-up; a larger one, or one with a shape of
    the caller's, does."""
    from samrai_amd import fac
    print("tile shape", n, flush=True)
    dim = len(n)
    h = fac.PatchHierarchy(dim, (0,) * dim, [v - 1 for v in n], [0.0] * 3, [1.0] * 3)
    cut = n[1] // 4 * 2  # a patch is at most 512 cells wide
    h.add_level(1, [((0,) * dim, (n[0] - 1, cut - 1) + tuple(v - 1 for v in n[2:])),
                    ((0, cut, 0)[:dim], tuple(v - 1 for v in n))])
    h.finalize()
    u, f = fac.PatchData(h, 1), fac.PatchData(h, 0)
    s = fac.CellPoissonFACSolver(h, max_cycles=1)
    s.set_dirichlet(0.0)
    s.initialize_solver_state(u, f)
    assert s.fused_coarsest_active()
    shapes = len(fac.fused_tile_shapes(dim))
    assert len(s.fused_tile_timings()) == (shapes if tiled else 0)
    assert 0 <= s.fused_tile_variant() < shapes if tiled else s.fused_tile_variant() == -1
    s.set_fused_coarsest(True, 2)
    assert s.fused_tile_variant() == 2 and s.fused_tile_timings() == []
    s.set_fused_coarsest(True)
    assert (s.fused_tile_variant() >= 0) == tiled


MG = dict(residual_tol=1e-300, relative_residual_tol=1e-300, num_pre_sweeps=1,
          num_post_sweeps=1, coarse_solver_choice="mg")
# lower parts of one to six levels, starting on the finest or a coarser level,
# first levels of one and of four cells a thread and of exactly 1024 cells,
# halving that stops at odd extents (the last grid's 64 sweeps) or at the
# smallest edge, a level too large for the lower part that cannot be halved
# (33^3: none)
MG_SIZES = [(4, 4, 4), (8, 8, 8), (12, 20, 8), (16, 16, 16), (24, 16, 18), (20, 20, 20),
            (32, 16, 16), (33, 33, 33), (40, 32, 48), (4, 6), (64, 64), (62, 46), (66, 62),
            (96, 40), (128, 32), (256, 128)]
MG_SPECS = [dict(dvar=False), dict(dvar=True, cmode=2, robin=True),
            dict(dvar=True, cmode=1, cconst=-0.3),
            dict(dvar=False, cmode=1, cconst=-0.7, robin=True)]
MG_IDS = ["constD", "varD-varC-robin", "varD-constC", "constD-constC-robin"]


def mg_pair(n, spec, cycles, tol, max_cycles=6):
    case = one_level(*n)
    spec = dict(spec)
    if spec.pop("robin", False):
        spec["bc"] = hc.bc_robin(case["dim"])
    data = hc.make_data(case, seed=sum(n))
    print("multigrid lower part", case["name"], spec, cycles, tol, flush=True)
    return hc.Pair(case, dict(MG, max_cycles=max_cycles, coarse_solver_max_iterations=cycles,
                              coarse_solver_tolerance=tol), data, **spec)


# the lower part in one work-group (at most three V-cycles a coarse solve, or a
# tolerance that one or two meet) and as a matrix
@pytest.mark.parametrize("cycles,tol", [(3, 1e-300), (10, 1e-300), (10, 0.05)],
                         ids=["three", "matrix", "loose"])
@pytest.mark.parametrize("spec", MG_SPECS, ids=MG_IDS)
@pytest.mark.parametrize("n", MG_SIZES, ids=lambda n: "x".join(map(str, n)))
def test_multigrid_lower_part_matches_oracle(gpu_lib, n, spec, cycles, tol):
    """Residual history and solution of a one-level FAC solve with the
    multigrid coarse solver against the oracle's multigrid: the values of every
    level operation are the same and only the norms' sums are ordered
    differently, so both agree to 1e-10 as the other multigrid solves do.

    After ten V-cycles a residual is soon all rounding.  A cell's is a sum of
    2 dim fluxes D (u - u') / dx^2, each rounded a few times in relation to
    D u / dx^2, and the matrix rounds in other places than the steps it stands
    for: 16 roundings of the stencil's 4 D sum(1 / dx^2) max |u|."""
    pr = mg_pair(n, spec, cycles, tol)
    pr.s.solve_system(pr.u, pr.f)
    _, it, _, hist = pr.o.solve()
    assert pr.s.number_of_iterations() == it
    atol = 1e-13 * max(hist)
    if cycles == 10 and tol < 1e-10:
        D = np.exp(0.8) if spec["dvar"] else 1.0
        u = max(np.abs(pr.o.get("u", 0, p)).max() for p in range(pr.npatch(0)))
        atol = max(atol, 16 * 2.0 ** -53 * 4 * D * sum(v * v for v in n) * u)
        assert atol <= 1e-9  # the first residual is of order 1
    np.testing.assert_allclose(pr.s.history(), hist, rtol=1e-10, atol=atol)
    pr.compare(pr.u, "u", interior_only=True, rtol=1e-10)


@pytest.mark.parametrize("spec", MG_SPECS, ids=MG_IDS)
@pytest.mark.parametrize("n", [n for n in MG_SIZES if np.prod(n) > 1024 and n != (33, 33, 33)],
                         ids=lambda n: "x".join(map(str, n)))
def test_multigrid_matrix_in_fp32(gpu_lib, n, spec):
    """The FP32 coarse solve with its lower levels as a matrix: every FAC cycle
    reduces the FP64 residual by a coarse solve to 1e-6 or by ten V-cycles (30
    times on 66 x 62, whose last grid 33 x 31 takes 64 sweeps), so ten of them
    reach the FP64 oracle's solution to 1e-8 of max |u|."""
    pr = mg_pair(n, spec, 10, 1e-300, max_cycles=10)
    pr.s.set_coarse_precision(32)
    pr.s.solve_system(pr.u, pr.f)
    pr.o.solve()
    hist = pr.s.history()
    assert hist[-1] <= 1e-9 * hist[0]
    pr.compare(pr.u, "u", interior_only=True, rtol=1e-8)
