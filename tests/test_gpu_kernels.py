"""Edges of single kernels' ranges (tile remainders, smallest and largest
sizes of a dispatch rule) against the checker, bit for bit (GPU)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _states(sim, T):
    st, died = sim._read_agents(T)
    st = np.ascontiguousarray(st)
    return st.view(np.uint8).reshape(len(st), st.dtype.itemsize), died


# rows of 16 cells (the shortest of the row kernel) and below, row lengths
# around its 8-cell groups and 512-cell waves, one to four dimensions, reaches
# 1, 2 and 7 (the largest) and 8 (past it), extents smaller than the reach
ROWS = [((16, 5), 1, "chebyshev"), ((15, 6), 1, "chebyshev"), ((17, 3), 2, "euclidean"), ((23, 9), 7, "manhattan"),
        ((50,), 8, "manhattan"), ((40,), 3, "chebyshev"), ((512, 4), 1, "chebyshev"), ((513, 7), 1, "manhattan"),
        ((519, 1), 2, "manhattan"), ((33, 6, 5), 1.5, "euclidean"), ((16, 3, 2, 4), 1, "chebyshev")]


@pytest.mark.parametrize("periodic", [True, False])
@pytest.mark.parametrize("dims,dist,metric", ROWS, ids=lambda v: str(v).replace(" ", ""))
def test_diffuse_rows(vh, ora, gpu_ready, dims, dist, metric, periodic):
    """diffuse on a raster of one-byte cells; some active cells hold values
    other than 1 (any nonzero byte is true and becomes 1)."""
    n = int(np.prod(dims))
    rng = np.random.default_rng(n)
    raw = np.where(rng.random(n) < 2.0 / n, rng.choice([1, 2, 128, 255], n), 0).astype(np.uint8)
    raw[[0, n - 1]] = [255 if n % 2 else 0, 64]
    got = []
    for V in (vh, ora):
        Cell = V.struct("Cell", [("active", "?")])
        Adj = V.struct("Adj")
        model = (V.ModelTypes() | V.register_agenttype_(Cell, "Immortal")
                 | V.register_edgetype_(Adj, "Stateless", target=Cell) | V.create_model("rows"))
        sim = V.create_simulation(model)
        V.raster.add_raster_(sim, "r", dims, raw.view([("active", "?")]), T=Cell)
        V.raster.connect_raster_neighbors_(sim, "r", Adj(), distance=dist, metric=metric, periodic=periodic,
                                           device=None if V is vh else False)
        V.finish_init_(sim)
        out = []
        for _ in range(3):
            V.apply_(sim, V.transitions.diffuse(Adj, Cell), Cell, [Cell, Adj], Cell)
            out.append(_states(sim, Cell)[0].copy())
        got.append(out)
    for k, (a, b) in enumerate(zip(*got)):
        assert np.array_equal(a, b), k
