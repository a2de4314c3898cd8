"""The reverse of the edge flux on clearly subcritical edges
(samoa_amd/csrc/swe_adjoint_clear.hpp) against the general one, compiled for
the host: equal bit for bit (a zero's sign aside)."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "samoa_amd", "csrc")
S = np.sqrt(0.5)
NORMALS = np.array([(1.0, 0.0), (S, S), (0.0, 1.0), (-S, S), (-1.0, -0.0), (-S, -S), (0.0, -1.0),
                    (S, -S)])


@pytest.fixture(scope="module")
def shim(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("shim") / "libclear_adjoint_shim.so")
    subprocess.run(["hipcc", "-O2", "-fPIC", "-shared", "-std=c++17", "-ffp-contract=off",
                    "--offload-arch=gfx950", "-Xclang", "-target-feature", "-Xclang",
                    "-packed-fp32-ops", f"-I{CSRC}",
                    os.path.join(HERE, "native", "clear_adjoint_shim.hip"), "-o", out],
                   check=True, capture_output=True)
    return C.CDLL(out)


# depth, speed scale, spread of the beds, least share of clear edges
SCENES = {"ocean": (4000.0, 0.3, 30.0, 0.99), "shelf": (50.0, 2.0, 3.0, 0.8),
          "basin": (5.0, 1.0, 0.0, 0.95), "still": (5.0, 0.0, 0.2, 0.95),
          "margin": (2.0, 3.0, 0.05, 0.2), "steep": (10.0, 0.5, 4.0, 0.0)}


@pytest.mark.parametrize("solver", [0, 1])
@pytest.mark.parametrize("scene", sorted(SCENES))
def test_equals_the_general_reverse(shim, solver, scene):
    h, du, db, share = SCENES[scene]
    rng = np.random.default_rng(len(scene))
    n = 50000
    q = []
    for _ in range(2):
        b = -h + db * rng.normal(0, 1, n)
        d = np.maximum(-b + 1e-3 * h * rng.normal(0, 1, n), 0.0)
        u = du * rng.normal(0, 1, (2, n))
        q.append(np.ascontiguousarray(np.stack([b + d, d * u[0], d * u[1], b], 1)))
    nrm = np.ascontiguousarray(NORMALS[rng.integers(0, 8, n)])
    # seeds on the depth as large as those on the momenta times a speed
    gf = rng.normal(0, 1, (2, n, 3)) * np.array([np.sqrt(9.81 * h), 1.0, 1.0])
    want, got = np.zeros((n, 8)), np.zeros((n, 8))
    clear = np.zeros(n, np.int8)
    p = lambda a: a.ctypes.data_as(C.c_void_p)  # noqa: E731
    shim.shim_clear_adjoint(solver, C.c_long(n), p(nrm), p(q[0]), p(q[1]), p(gf[0]), p(gf[1]),
                            C.c_double(1e-3), C.c_double(9.80665), p(want), p(got), p(clear))
    ok = clear != 0
    assert ok.mean() >= share
    assert np.array_equal(want[ok], got[ok])
