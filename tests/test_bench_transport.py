"""The figures bench.py prints of the transport sweeps: one launch, the bytes that it cannot do
without and the chain of its steps."""
import bench


def test_gs_launch():
    g = bench.gs_launch(256, 256, 64, 4, 5, 0.2)
    assert g["sweeps"] == 6 and g["avg_launch_us"] == 1200.0
    assert g["bytes"] == 258 * 258 * 66 * 15 * 8
    assert g["GBs"] == round(g["bytes"] / 1.2e-3 / 1e9, 1)
    assert g["frac"] == round(g["bytes"] / 1.2e-3 / 1e9 / bench.HBM_PEAK_GBS, 4)
    assert "chain of 594 steps" in g["bound"]  # 258 + 258 + 66 + 12


def test_gs_launch_of_many_sweeps():
    assert bench.gs_launch(8, 8, 8, 1, 0, 0.01)["sweeps"] == 1
    assert bench.gs_launch(8, 8, 8, 1, 6, 0.01)["sweeps"] == 4   # 4 + 3
    assert bench.gs_launch(8, 8, 8, 1, 11, 0.01)["sweeps"] == 6  # 6 + 6
    assert bench.gs_launch(8, 8, 8, 1, 12, 0.01)["sweeps"] == 5  # 5 + 4 + 4
