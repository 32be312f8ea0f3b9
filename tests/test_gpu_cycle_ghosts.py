"""Ghost cells after a solve and between its cycles, edges and corners too.

The cycle of the library's own operators fills only the ghosts that they
read; what a caller sees, the solution and error after solveSystem and the
solution that an overridden postprocessOneCycle gets after every cycle
(solv/FACOperatorStrategy.h:82-364), has all of them filled."""
import ctypes
import subprocess

import numpy as np
import pytest

import hier_cases as hc

pytestmark = pytest.mark.gpu

KEYS = dict(max_cycles=3, residual_tol=1e-300, relative_residual_tol=1e-300, num_pre_sweeps=2,
            num_post_sweeps=1, coarse_solver_tolerance=1e-12, coarse_solver_max_iterations=30,
            prolongation_method="CONSERVATIVE_LINEAR_REFINE")


@pytest.mark.parametrize("coarse", ["redblack", "mg"])
@pytest.mark.parametrize("spec", [dict(), dict(dvar=True, cmode=2, robin=True)],
                         ids=["constD", "varD-varC-robin"])
@pytest.mark.parametrize("mk", hc.ALL + [hc.case_2d_c0], ids=lambda f: f.__name__)
def test_ghosts_after_a_solve_match_oracle(gpu_lib, mk, spec, coarse):
    """Every value of u and e, ghosts included, against the oracle's solve,
    which fills all ghosts in every operation; inhomogeneous Robin data, fine
    patches on coarse-fine and physical faces, edges and corners."""
    case = mk()
    spec = dict(spec)
    if spec.pop("robin", False):
        spec["bc"] = hc.bc_robin(case["dim"])
    print("ghosts after a solve", case["name"], spec, coarse, flush=True)
    pr = hc.Pair(case, dict(KEYS, coarse_solver_choice=coarse), hc.make_data(case, seed=11),
                 **spec)
    pr.s.solve_system(pr.u, pr.f)
    pr.o.solve()
    rtol = 1e-12 if coarse == "redblack" else 1e-10
    pr.compare(pr.u, "u", rtol=rtol)
    pr.compare(pr.s.internal_vector("e"), "e", rtol=rtol)


HOOK = r"""
#include "fac_solver.hpp"
using namespace samrai_amd;
using pdat::PatchDataSet;
using namespace samrai_amd::solv;

// counts the values of u that a full ghost fill would change after a cycle
struct Hook : CellPoissonFACOps {
  using CellPoissonFACOps::CellPoissonFACOps;
  int levels = 0, cycles = 0;
  long stale = 0;
  void postprocessOneCycle(int, const SAMRAIVectorReal& u, const SAMRAIVectorReal&) override {
    const hier::PatchHierarchy& h = u.data->hierarchy();
    PatchDataSet full(h, PatchDataSet::kCell, u.data->ghost());
    full.copyFrom(*u.data, 0, levels - 1, stream());
    for (int ln = 0; ln < levels; ++ln) ghostFill(full, ln, ln > 0, false, false);
    hip_check(hipStreamSynchronize(stream()), "hook");
    for (int ln = 0; ln < levels; ++ln)
      for (int p = 0; p < (int)h.level(ln).boxes.size(); ++p) {
        const long n = u.data->size(ln, p);
        std::vector<double> a(n), b(n);
        hip_check(hipMemcpy(a.data(), u.data->pointer(ln, p), 8 * n, hipMemcpyDeviceToHost), "a");
        hip_check(hipMemcpy(b.data(), full.pointer(ln, p), 8 * n, hipMemcpyDeviceToHost), "b");
        for (long k = 0; k < n; ++k) stale += !(a[k] == b[k]);
      }
    ++cycles;
  }
};

extern "C" int hook_solve(int dim, int nlevels, const int* nboxes, const int* boxes, int ratio,
                          const int* dlo, const int* dhi, const double* a, const double* b,
                          const double* g, int graphs, long* stale, int* cycles) {
  try {
    const double lo[3] = {0, 0, 0}, hi[3] = {1, 1, 1};
    hier::PatchHierarchy h(dim, dlo, dhi, lo, hi);
    for (int ln = 0; ln < nlevels; ++ln) {
      std::vector<Box> list;
      for (int p = 0; p < nboxes[ln]; ++p, boxes += 6) {
        Box x{};
        for (int d = 0; d < 3; ++d) {
          x.lo[d] = boxes[d];
          x.hi[d] = boxes[3 + d];
        }
        list.push_back(x);
      }
      h.addLevel(ratio, list);
    }
    h.finalize();
    hipStream_t s;
    hip_check(hipStreamCreate(&s), "stream");
    {
      Hook ops(h, s);
      ops.levels = nlevels;
      FACPreconditioner fac(ops, &ops);
      fac.setMaxCycles(3);
      fac.setResidualTolerance(1e-300);
      ops.setCoarsestLevelSolverChoice("redblack");
      ops.setCoarseFineDiscretization("Ewing");
      ops.setProlongationMethod("CONSERVATIVE_LINEAR_REFINE");
      ops.setUseGraphs(graphs != 0);
      PatchDataSet u(h, PatchDataSet::kCell, 1), f(h, PatchDataSet::kCell, 0),
          w(h, PatchDataSet::kCell, 0);
      u.fill(0.0, s);
      f.fill(1.0, s);
      ops.computeVectorWeights(w, 0, nlevels - 1);
      ops.setPoissonSpecifications(PoissonSpecifications());
      LocationIndexRobinBcCoefs bc;
      for (int k = 0; k < 2 * dim; ++k) {
        bc.a[k] = a[k];
        bc.b[k] = b[k];
        bc.g[k] = g[k];
      }
      ops.setPhysicalBcCoefObject(bc);
      SAMRAIVectorReal uv{&u, &w, 0, nlevels - 1}, fv{&f, &w, 0, nlevels - 1};
      fac.solveSystem(uv, fv);
      *stale = ops.stale;
      *cycles = ops.cycles;
    }
    (void)hipStreamDestroy(s);
    return 0;
  } catch (const Error& e) {
    std::fprintf(stderr, "%s\n", e.msg.c_str());
  } catch (...) {
  }
  return 1;
}
"""


@pytest.fixture(scope="module")
def hook(gpu_lib, tmp_path_factory):
    """A subclass of the operators that overrides postprocessOneCycle, built
    against the library."""
    from samrai_amd import build, fac
    d = tmp_path_factory.mktemp("hook")
    (d / "hook.cpp").write_text("#include <cstdio>\n" + HOOK)
    # compiled as the library's own host sources are
    cc = [build.HIPCC, "--offload-arch=" + build.ARCH] + build.COMMON
    subprocess.run(cc + ["-c", str(d / "hook.cpp"), "-o", str(d / "hook.o")], check=True)
    subprocess.run(cc + ["-shared", str(d / "hook.o"), fac.LIB_PATH, "-o", str(d / "hook.so")],
                   check=True)
    return ctypes.CDLL(str(d / "hook.so"))


@pytest.mark.parametrize("graphs", [0, 1], ids=["eager", "graphs"])
@pytest.mark.parametrize("mk", [hc.case_2d, hc.case_3d_boundary], ids=lambda f: f.__name__)
def test_an_overridden_hook_sees_filled_ghosts(hook, mk, graphs):
    case = mk()
    dim = case["dim"]
    print("hook", case["name"], graphs, flush=True)

    def ints(v):
        return np.array(list(v) + [0] * (3 - len(v)), np.int32)

    boxes = np.concatenate([np.concatenate([ints(lo), ints(hi)])
                            for level in case["levels"] for lo, hi in level])
    nboxes = np.array([len(level) for level in case["levels"]], np.int32)
    bc = hc.bc_robin(dim)
    coef = [np.array(bc[k], np.float64) for k in "abg"]
    stale, cycles = ctypes.c_long(-1), ctypes.c_int(-1)
    ip, dp = ctypes.POINTER(ctypes.c_int), ctypes.POINTER(ctypes.c_double)
    dlo, dhi = ints(case["dlo"]), ints(case["dhi"])
    st = hook.hook_solve(dim, len(nboxes), nboxes.ctypes.data_as(ip), boxes.ctypes.data_as(ip),
                         case["ratio"], dlo.ctypes.data_as(ip), dhi.ctypes.data_as(ip),
                         *[c.ctypes.data_as(dp) for c in coef], graphs, ctypes.byref(stale),
                         ctypes.byref(cycles))
    assert st == 0
    assert cycles.value == 3
    assert stale.value == 0
