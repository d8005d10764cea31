"""The general hybrid kernel (csrc/rhs_hybrid.hip, k_hybrid) against the oracle.

Meshes just too large for the small-mesh kernel in 1-D and 2-D, and 3-D ones: every node count and two-point
flux, walls, outflow, inflow and Dirichlet ends, FP64 and FP32; and meshes whose metric or face frames are
not exactly axis-aligned, which take its full contraction.  Bounds as the hybrid form's other tests: 1e-12
in FP64, 2e-5 in FP32 of the largest value.
"""
import numpy as np
import pytest

import flouhip as F
import oracle_lib as O
from cases import GAMMA, random_euler_state
from test_gpu_hybrid import TP, surface

pytestmark = pytest.mark.gpu
pytest.importorskip("torch")

SURF = [(O.AVG_CHANDRASEKHAR, O.DISS_MATRIX), (O.AVG_STD, O.DISS_LXF), (O.AVG_CHANDRASEKHAR, O.DISS_SCALAR)]


def outer(x):
    """Dirichlet state at a point."""
    v = np.zeros(len(x) + 2)
    v[0] = 1.0 + 0.1 * np.sin(3.0 * np.sum(x))
    v[1] = 0.2
    v[-1] = 2.5 + 0.2 * np.cos(2.0 * np.sum(x))
    return v


def check(nd, n, nel, tp, savg, sdiss, ends, precision="fp64", tilt=None):
    finish = [1.0, 1.5, 2.0][:nd]
    b = F.LagrangeBasis("GLL", n)
    std = [None, F.StdSegment, F.StdQuad, F.StdHex][nd](b, F.DGSEMrec(b), nd + 2)
    mesh = F.CartesianMesh(nd, [0.0] * nd, finish, nel)
    mesh.apply_periodicBCs(*[(str(2 * k + 1), str(2 * k + 2)) for k in range(1 if ends else 0, nd)])
    state = np.array([1.1] + [0.3] * nd + [2.6])
    first = {"slip": (F.EulerSlipBC(), O.BC_SLIP), "inflow": (F.EulerInflowBC(state), O.BC_INFLOW),
             "dirichlet": (F.GenericBC(lambda _, x, *__: outer(x)), O.BC_DIRICHLET), None: (None, None)}[ends]
    if tilt:
        tilt(mesh, nd)
    eq = F.EulerEquation(nd, GAMMA)
    disc = F.MultielementDisc(mesh, std, eq, F.HybridDivOperator(TP[tp](), surface(savg, sdiss), 0.5),
                              {"1": first[0], "2": F.EulerOutflowBC()} if ends else {}, precision=precision)
    assert disc.kernel_name() == "k_hybrid"
    orc = O.OracleDisc(nd, n, nel, [0.0] * nd, finish, [0 if ends and k == 0 else 1 for k in range(nd)],
                       O.build_ops(n, "GLL"), O.EQ_EULER, [GAMMA], O.VOL_HYBRID, tp, savg, sdiss, 1.0)
    orc.set_blend(0.5)
    orc.set_option(0, 0)  # corrected 3-D surface fluxes on both sides
    disc.set_option(0, 0)
    if ends:
        data = state
        if ends == "dirichlet":
            fx = mesh.face_node_coords(std)
            data = np.array([[outer(x) for x in face] for face in fx])
        orc.set_bc(0, first[1], data)
        orc.set_bc(1, O.BC_OUTFLOW)
    Q = random_euler_state(orc.coords()[0], nd, seed=n, amp=0.3, smooth=False)
    if precision == "fp32":
        Q = Q.astype(np.float32).astype(np.float64)
    dQ = disc.new_state()
    F.rhs_(dQ, disc.to_device(Q), F.EquationConfig(disc, eq))
    disc.check()
    ref = orc.rhs(Q)
    err = np.max(np.abs(disc.to_host(dQ) - ref) / np.max(np.abs(ref), axis=0))
    assert err <= (1e-12 if precision == "fp64" else 2e-5), err


def above(nd, n, precision):
    """A mesh of one element (1-D) or one row of elements (2-D) more than the small-mesh kernel takes."""
    most = (768 if precision == "fp64" else 1024) * (128 // ((n if nd == 2 else 1) * (n + 1)))
    return [most + 1] if nd == 1 else [most // 32 + 1, 32]


@pytest.mark.parametrize("tp", sorted(TP))
@pytest.mark.parametrize("nd,n", [(nd, n) for nd in (1, 2) for n in range(2, 9)])
def test_meshes_above_the_limit(nd, n, tp):
    k = (n + tp) % 3
    check(nd, n, above(nd, n, "fp64"), tp, *SURF[k], [None, "slip", "dirichlet"][k])
    k = (k + 1) % 3
    check(nd, n, above(nd, n, "fp64"), tp, *SURF[k], ["inflow", "dirichlet", "slip"][k])


@pytest.mark.parametrize("nd,n", [(nd, n) for nd in (1, 2) for n in (2, 5, 6, 7, 8)])
def test_fp32(nd, n):
    tp = sorted(TP)[n % 3]
    check(nd, n, above(nd, n, "fp32"), tp, *SURF[n % 2], [None, "slip", "dirichlet"][n % 3], "fp32")


@pytest.mark.parametrize("ends", ["slip", "inflow", "dirichlet"])
@pytest.mark.parametrize("n", range(2, 9))
def test_3d_with_ends(n, ends):
    k = n + len(ends)
    check(3, n, [2, 3, 1], sorted(TP)[k % 3], *SURF[k % 3], ends)


def metric_not_exactly_diagonal(mesh, nd):
    """Off-diagonal metric terms of 1e-300: not zero, but nothing to any sum."""
    geometry = mesh.element_geometry

    def tilted(std):
        jac, metric, volume = geometry(std)
        m = np.array(metric).reshape(len(jac), nd, nd)
        m[:, ~np.eye(nd, dtype=bool)] = 1e-300
        return jac, m.reshape(np.shape(metric)), volume

    mesh.element_geometry = tilted


def rotated_tangents(mesh, nd):
    """3-D face frames whose tangents are turned about the normal: the same fluxes up to rounding."""
    geometry = mesh.face_geometry

    def turned():
        frames, jac = geometry()
        fr = np.array(frames).reshape(len(jac), 3, nd)
        c, s = 0.8, 0.6
        t, b = fr[:, 1].copy(), fr[:, 2].copy()
        fr[:, 1], fr[:, 2] = c * t + s * b, c * b - s * t
        return fr.reshape(np.shape(frames)), jac

    mesh.face_geometry = turned


@pytest.mark.parametrize("tp", sorted(TP))
@pytest.mark.parametrize("nd,n,tilt", [(2, 4, metric_not_exactly_diagonal), (2, 7, metric_not_exactly_diagonal),
                                       (3, 4, metric_not_exactly_diagonal), (3, 5, rotated_tangents)])
def test_not_axis_aligned(nd, n, tp, tilt):
    nel = [5, 4] if nd == 2 else [2, 3, 2]
    check(nd, n, nel, tp, *SURF[(n + tp) % 3], "slip", tilt=tilt)
    check(nd, n, nel, tp, *SURF[(n + tp + 1) % 3], None, "fp32", tilt=tilt)
