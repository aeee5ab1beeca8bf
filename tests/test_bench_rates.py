"""The benchmark's bandwidth of the gene-tree kernels is that of measured
traffic: without a counter summary of the workload there is none, rather than
one from bytes that the kernels only count."""
import os
import types

import bench


def test_rate_of_measured_traffic():
    r = bench.measured_rate("latency", 4.0e9, 2.0)
    assert r["achieved"] == 2000.0 and r["frac"] == 0.25 and r["bound"] == "latency"
    r = bench.measured_rate("hbm", None, 2.0)
    assert r["achieved"] is None and r["frac"] is None and r["traffic"] is None


def test_summaries_cover_the_default_gene_tree_workload():
    args = types.SimpleNamespace()
    for tail in ("", " height moves"):
        key = f"config=5 elements=20000 seed=3 precision=fp32{tail}"
        traffic, source = bench.measured_traffic(args, None, key)
        assert traffic > 1e8 and os.path.exists(os.path.join(bench.ROOT, source))
        assert bench.measured_traffic(args, None, key.replace("seed=3", "seed=4")) == (None, None)
