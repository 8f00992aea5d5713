"""bench.py's roofline objects: the fraction of the peak is that of the bytes of the
blocks that are launched, whatever the rate over all cells would be."""
import bench


def test_rate_of_the_launched_blocks():
    r = bench.roofline(9000.0, 0.4)
    assert r["peak"] == 8000.0 and r["achieved"] == 3600.0 and r["frac"] == 0.45
    assert r["block_share"] == 0.4 and r["all_cells"] == 9000.0
    assert bench.roofline(4000.0, 1.0)["frac"] == 0.5
