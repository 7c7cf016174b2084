"""The FP64 iteration's matrix copy with its blocks in planes (csrc/common.hpp,
ld_planes) is taken for n = 2 from 160 MiB of block values on: the smallest mesh
past that, in the grouped face order, against the natural order, which keeps the
blocks interleaved.  Both stop at 1e-12; the solutions of two such solves differ
by about 1e-10 on these systems, the bar is 2e-9."""
import numpy as np
import pytest

from mhfem_amd import capi, problems
import _group

pytestmark = pytest.mark.gpu


def test_planes_match_interleaved_blocks():
    pr = problems.adr_3d(s=42, n=2, preconditioner="diagonal")
    assert pr.num_faces * 5.9 * 32 > 160 << 20
    z = []
    for groups in (1, 0):
        print(f"\n[planes] groups {groups}", flush=True)
        s = capi.Solver(pr, preconditioner="diagonal", tol=1e-12, face_groups=groups)
        assert _group.info(s)["planes"] == groups
        for k in range(2):
            assert s.step(k * pr.dt, pr.dt).converged
        z.append(s.get_array("Z_iF"))
        s.close()
    assert np.linalg.norm(z[0] - z[1]) < 2e-9 * np.linalg.norm(z[1])
