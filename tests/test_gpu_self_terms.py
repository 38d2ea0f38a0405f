"""Self terms of needle triangles: their one-dimensional cubature goes past
the orders whose nodes are evaluated at once (one node per lane), to a single
node more and then to nodes kept in a scratch slab."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# the flatter the tetrahedron, the nearer the integrand's poles to the
# interval: order 4, 5, 6 and more
@pytest.mark.parametrize("material,eps", [("PEC", None), ("CONST_EPS_4", 4.0)])
@pytest.mark.parametrize("h", [0.8, 0.3, 0.1, 0.03])
def test_needle_tetrahedron(sx, O, h, material, eps):
    print(f"needle tetrahedron h={h} {material}", flush=True)
    V = np.array([[0, 0, 0], [1, 0, 0], [0.47, h, 0], [0.52, h / 3, 0.9 * h]], dtype=float)
    T = np.array([[0, 2, 1], [0, 1, 3], [1, 2, 3], [2, 0, 3]], dtype=np.int32)
    G = sx.RWGGeometry()
    G.AddMesh(V, T, material)
    Go = O.Geometry()
    if eps is None:
        Go.add_surface(V, T, kind=0)
    else:
        Go.add_surface(V, T, kind=1, eps=eps)
    M, Mo = G.AssembleBEMMatrix(1.0).numpy(), Go.assemble(1.0)
    # every integral stops at a relative 1e-10 (self) or 1e-5 (touching
    # pairs) by the same decisions on both sides: what differs is rounding
    err = np.linalg.norm(M - Mo) / np.linalg.norm(Mo)
    assert err <= 1e-11, err
