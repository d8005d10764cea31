"""Which kernel a discretisation runs (flou_hip_kernel_name): the forms, geometries and precisions
that have a kernel of their own, and what falls to the general one."""
import pytest

import flouhip as F
from cases import warp

pytestmark = pytest.mark.gpu
pytest.importorskip("torch")

LXF = F.LxF(F.StdAverage(), 1.0)
MATRIX = F.MatrixDissipation(F.ChandrasekharAverage(), 1.0)
CH, KG, STD = F.ChandrasekharAverage(), F.KennedyGruber(), F.StdAverage()


def disc(nd, n, nel, op, precision="fp64", curved=False, nodes="GLL", eq=None):
    b = F.LagrangeBasis(nodes, n)
    eq = eq or F.EulerEquation(nd, 1.4)
    std = [None, F.StdSegment, F.StdQuad, F.StdHex][nd](b, F.DGSEMrec(b), 1 if isinstance(eq, F.LinearAdvection) else nd + 2)
    mesh = F.CartesianMesh(nd, (0.0,) * nd, (1.0,) * nd, nel)
    mesh.apply_periodicBCs(*[(str(2 * k + 1), str(2 * k + 2)) for k in range(nd)])
    if curved:
        mesh.apply_mapping(warp)
    return F.MultielementDisc(mesh, std, eq, op, precision=precision)


@pytest.mark.parametrize("rhs,adjoint,args", [
    ("k_split", "k_svjp", (2, 4, [3, 3], F.SplitDivOperator(CH, LXF))),
    ("k_split", "k_svjp", (3, 5, [2, 2, 2], F.SplitDivOperator(KG, LXF))),
    ("k_split", "k_vjp", (2, 6, [3, 3], F.SplitDivOperator(CH, LXF))),
    ("k_split_1d", "k_vjp", (1, 3, [20], F.SplitDivOperator(CH, MATRIX))),
    ("k_split", "k_vjp", (1, 8, [4200], F.SplitDivOperator(CH, LXF))),
    ("k_plain", "k_vjp", (1, 8, [4200], F.SplitDivOperator(CH, MATRIX))),
    ("k_plain", "k_vjp", (2, 4, [3, 3], F.SplitDivOperator(CH, MATRIX))),
    ("k_split_curved", "k_svjp", (3, 5, [2, 2, 2], F.SplitDivOperator(CH, LXF), "fp64", True)),
    ("k_split_curved", "k_vjp", (2, 6, [3, 3], F.SplitDivOperator(STD, LXF), "fp64", True)),
    ("k_strong", "k_vjp", (3, 5, [2, 2, 2], F.StrongDivOperator(LXF))),
    ("k_strong", "k_vjp", (3, 5, [2, 2, 2], F.StrongDivOperator(LXF), "fp32")),
    ("k_plain", "k_vjp", (3, 5, [2, 2, 2], F.StrongDivOperator(LXF), "fp64", True)),
    ("k_hybrid_lines", "", (2, 6, [5, 3], F.HybridDivOperator(CH, MATRIX, 1.0))),
    ("k_hybrid_lines", "", (1, 4, [30], F.HybridDivOperator(CH, MATRIX, 1.0), "fp32")),
    ("k_hybrid", "", (2, 6, [60, 60], F.HybridDivOperator(CH, MATRIX, 1.0))),
    ("k_hybrid", "", (3, 4, [2, 2, 2], F.HybridDivOperator(CH, MATRIX, 1.0))),
    ("k_plain", "", (2, 4, [3, 3], F.SplitDivOperator(CH, LXF), "fp64", False, "GL")),
    ("k_fast", "k_fvjp", (3, 6, [2, 2, 2], F.SplitDivOperator(CH, LXF), "fp32")),
    ("k_fastc", "k_fvjp", (3, 7, [2, 2, 2], F.SplitDivOperator(CH, LXF), "fp32", True)),
], ids=lambda x: str(x) if isinstance(x, str) else "-".join(map(str, x[:3])).replace(" ", ""))
def test_kernel_names(rhs, adjoint, args):
    d = disc(*args)
    assert (d.kernel_name(), d.kernel_name(adjoint=True)) == (rhs, adjoint)


def test_plain_option():
    d = disc(3, 6, [2, 2, 2], F.SplitDivOperator(CH, LXF), "fp32")
    d.set_option(1, 1)
    assert (d.kernel_name(), d.kernel_name(adjoint=True)) == ("k_plain", "k_vjp")


SPLIT_CH, SPLIT_KG, SPLIT_STD = (F.SplitDivOperator(tp, LXF) for tp in (CH, KG, STD))
HYBRID = F.HybridDivOperator(CH, MATRIX, 1.0)


# the last mesh of each size rule's range, and the first beyond it
@pytest.mark.parametrize("inside,outside,args,nel_in,nel_out", [
    ("k_split_1d", "k_split", (1, 5, SPLIT_CH), [768 * 12], [768 * 12 + 1]),
    ("k_split_1d", "k_split", (1, 8, SPLIT_STD), [768 * 4], [768 * 4 + 1]),
    ("k_split_1d", "k_plain", (1, 8, F.SplitDivOperator(CH, MATRIX)), [1024 * 4], [1024 * 4 + 1]),
    ("k_split_1d", "k_plain", (1, 2, F.SplitDivOperator(KG, MATRIX)), [1024 * 64], [1024 * 64 + 1]),
    ("k_hybrid_lines", "k_hybrid", (2, 6, HYBRID), [48, 48], [48, 49]),
    ("k_hybrid_lines", "k_hybrid", (2, 6, HYBRID, "fp32"), [64, 48], [64, 49]),
    ("k_hybrid_lines", "k_hybrid", (1, 5, HYBRID), [256 * 21], [256 * 21 + 1]),
    ("k_hybrid_lines", "k_hybrid", (1, 5, HYBRID), [256 * 51 + 1], [256 * 51]),
    ("k_hybrid_lines", "k_hybrid", (1, 5, HYBRID), [768 * 21], [768 * 21 + 1]),
    ("k_hybrid_lines", "k_hybrid", (1, 5, HYBRID, "fp32"), [1024 * 21], [1024 * 21 + 1]),
], ids=lambda x: None if isinstance(x, tuple) else str(x).replace(" ", ""))
def test_size_rules_of_the_rhs(inside, outside, args, nel_in, nel_out):
    nd, n, op, *precision = args
    assert disc(nd, n, nel_in, op, *precision).kernel_name() == inside
    assert disc(nd, n, nel_out, op, *precision).kernel_name() == outside


# meshes that take the line adjoint, and ones too small for it (or None)
@pytest.mark.parametrize("args,nel,small", [
    ((2, 4, SPLIT_CH, False), [1, 2], None),
    ((2, 5, SPLIT_CH, False), [96, 80], [95, 80]),
    ((2, 5, SPLIT_KG, False), [80, 64], [79, 64]),
    ((2, 6, SPLIT_KG, False), [64, 56], [63, 56]),
    ((2, 8, SPLIT_CH, False), [88, 64], [87, 64]),
    ((2, 8, SPLIT_STD, False), [3, 3], None),
    ((3, 6, SPLIT_CH, False), [8, 8, 4], [17, 5, 3]),
    ((3, 5, SPLIT_CH, False), [12, 8, 8], [11, 8, 8]),
    ((3, 5, SPLIT_KG, False), [1, 2, 2], None),
    ((3, 7, SPLIT_CH, False), [1, 2, 2], None),
    ((2, 4, SPLIT_STD, True), [2, 2], None),
    ((2, 5, SPLIT_CH, True), [96, 80], [95, 80]),
    ((2, 5, SPLIT_STD, True), [80, 64], [79, 64]),
    ((2, 6, SPLIT_KG, True), [64, 56], [63, 56]),
    ((2, 7, SPLIT_STD, True), [64, 56], [63, 56]),
    ((3, 6, SPLIT_KG, True), [1, 2, 2], None),
], ids=lambda x: f"{x[0]}d-n{x[1]}" if isinstance(x, tuple) else str(x).replace(" ", ""))
def test_size_rules_of_the_adjoint(args, nel, small):
    nd, n, op, curved = args
    assert disc(nd, n, nel, op, curved=curved).kernel_name(adjoint=True) == "k_svjp"
    if small:
        assert disc(nd, n, small, op, curved=curved).kernel_name(adjoint=True) == "k_vjp"


@pytest.mark.parametrize("n,op", [(5, SPLIT_KG), (7, SPLIT_KG), (8, SPLIT_CH), (8, SPLIT_STD)])
def test_general_adjoint_on_large_curved_meshes(n, op):
    assert disc(2, n, [100, 80], op, curved=True).kernel_name(adjoint=True) == "k_vjp"
