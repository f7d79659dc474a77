"""Plans at the largest LDS budgets (host only): a tile is cut to the budget with a front part
of its own size, and where the plan's largest front and largest back part do not fit one CU
together the tiles are cut again, so every budget up to the CU's LDS gives a valid plan."""
import pytest


@pytest.mark.parametrize("op", [0, 1])
@pytest.mark.parametrize("mesh", ["cube", "delaunay"])
@pytest.mark.parametrize("budget", [155000, 160000, 163000, 163840])
def test_largest_budgets(mf, op, mesh, budget):
    import bench
    from minifem.setup import plan_host_stats
    coord, e2n, code, nnz = (mf.generate_cube(40, 0.25, 3, 203) if mesh == "cube"
                             else bench.delaunay_arrays(6000, seed=3))
    m = mf.Mesh(coord, e2n, code, nnz, op)
    stats = plan_host_stats(m, tile_lds_bytes=budget)  # validates the plan
    assert stats["lds_bytes"] <= 163840
    assert stats["tiles"] <= plan_host_stats(m, tile_lds_bytes=120000)["tiles"]
