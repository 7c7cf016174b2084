"""The launched iteration on systems small enough to iterate in one launch
(csrc/group.hip), which take the other form by themselves: the tests of the
batch narrowing, the replayed graphs, the poll period, the rows per partial
sum, the face orders and the FP32 forms once more, every context iterating by
launches.  It is the form of systems that do not fit on the chip, and the one
a solve goes on with when a wait gives up."""
import pytest

from mhfem_amd import capi
import _group
from test_gpu_batch import (test_autotune_keeps_results, test_batch_iterations_per_instance,  # noqa: F401
                            test_batch_matches_individual_runs, test_batch_narrowed_steps_equal_single_runs,
                            test_graph_step_after_coefficient_updates, test_graph_step_equals_eager_step)
from test_gpu_boundary_model import test_graph_steps_see_each_steps_time  # noqa: F401
from test_gpu_parity import (case, test_face_groups, test_fp32_refinement, test_fp32_reliable_iterations,  # noqa: F401
                             test_krylov_iteration_parity, test_solvers_on_zero_rhs_and_from_the_solution,
                             test_time_steps)
from test_zz_no_alloc import test_noalloc_equals_solve_rhs  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def by_launches(monkeypatch):
    made = []

    class Launched(capi.Solver):
        def setupLinearSystem(self):
            super().setupLinearSystem()
            _group.launched(self)
            made.append(self)

    monkeypatch.setattr(capi, "Solver", Launched)
    yield
    assert made
    for s in made:
        assert not s.ctx or _group.info(s)["launches"] == 0
