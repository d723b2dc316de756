"""The benchmark's printed line and its byte counts, from made-up statistics.  No
GPU calls."""
import json
from types import SimpleNamespace

import pytest

import bench
from clbool_amd import _capi

THIRD = 1e11 / 3


def _product(name):
    mode = {"ms_per_step": THIRD, "products_per_s": THIRD, "nnz_per_s": THIRD, "row_blocks": 18,
            "fallback_rate": 1 / 3, "bin_products": [10**11] * 32, "tuning": {f"knob_{k}": k for k in range(24)},
            "roofline": {"bound": "hbm", "achieved": 1234.5, "peak": 8000.0, "unit": "GB/s", "frac": 0.1234,
                         "traffic": 10**11, "kernel": "onepass_compact", "launches": 100, "avg_launch_ms": 12.3456,
                         "algorithmic_bytes_per_launch": 10**11}}
    config = {"workload": name, "scale": 22, "edge_factor": 16, "seed": 1, "rmat_abcd": [0.57, 0.19, 0.19, 0.05],
              "a_nnz": 10**8, "a_nzr": 10**7, "products": 10**12, "block_bound": 2**32 - 1}
    return {"config": config, "nnz_out": 10**11, "validated_rows": {"plain": 864, "learned": 864, "bound": 1584},
            "modes": {m: mode for m in ("plain", "learned", "bound")}, "learned_vs_plain": 4 / 3,
            "bound_vs_plain": 4 / 3, "learned_vs_bound": 4 / 3}


def test_line_is_short_and_whole():
    leg = {"seconds": 1 / 3, "products": 10**12, "step_pool": [[1, 2.5, 3, 4.5, 5.5]] * 12}
    details = {
        "device": {"arch": "gfx950:sramecc+:xnack-", "compute_units": 256},
        "workloads": {w: _product(f"{w}_ef16_AxA") for w in ("rmat22", "rmat20")},
        "closure": {"labels": 64, "per_triple_plain": leg, "batched_plain": leg, "batched_learned": leg,
                    "identical_results": True},
        "hypersparse": {"tests": [{"plain_ms": 1 / 3, "learned_ms": 1 / 3, "fallback_rows": 0, "identical": True}] * 4},
        "c5": {"kronecker": {"seconds": 1 / 3, "GB_per_s": 1e4 / 3},
               "kk_step": {"plain": {"seconds": 1 / 3}, "learned": {"seconds": 1 / 3}, "identical_results": True}},
        "cpu_baseline": {"value": 1e8 / 3, "unit": "products/s", "cores": 1, "kind": "port", "sample": "x" * 100},
        "cpu_gustavson": {"value": 1e9 / 3, "cores": 16, "sample": "x" * 100},
    }
    line = bench.report("rmat22", 20, 5, "learned", details)
    assert len(line) < 2500 and "\n" not in line
    out = json.loads(line)
    for k in ("metric", "value", "unit", "n_gpus", "steps", "warmup", "ms_per_step", "higher_is_better", "scaling",
              "vs_baseline", "dtype", "data", "config"):
        assert k in out
    assert out["steps"] == 20 and out["warmup"] == 5 and abs(out["value"] / THIRD - 1) < 1e-5
    assert out["rmat20"]["ms"]["plain"] == out["ms_per_step"]
    assert len(bench.report("rmat22", 20, 5, "learned", {k: details[k] for k in ("device", "workloads")})) < 2500


# one row in bin 5 (a table), two in 20 (bitmap), three in 13 (kept): A nonzeros,
# products, columns
A_NNZ, PRODUCTS, COLUMNS = {5: 10, 13: 300, 20: 200}, {5: 40, 13: 6000, 20: 4000}, {5: 30, 13: 500, 20: 700}


@pytest.mark.parametrize("family, nbytes", [
    ("sym_bitmap", 12 * 500 + 4 * 10000 + 8 * 5),                 # gathers the kept rows too
    ("num_bitmap", 12 * 200 + 4 * 4000 + 4 * 700 + 8 * 2 + 4 * 500),  # expands them
    ("onepass_bitmap", 12 * 200 + 4 * 4000 + 4 * 700 + 8 * 2),
    ("onepass_emit", 4 * 500),
    ("onepass_compact", 8 * (1230 - 500)),
    ("num_hash", 12 * 10 + 4 * 40 + 4 * 30 + 8),
])
def test_bytes_of_a_family(family, nbytes):
    agg = bench._new_agg()
    for b, rows in ((5, 1), (20, 2), (13, 3)):
        agg["bin_rows"][b], agg["bin_a_nnz"][b] = rows, A_NNZ[b]
        agg["bin_products"][b], agg["bin_out_nnz"][b] = PRODUCTS[b], COLUMNS[b]
    agg["nnz"] = sum(COLUMNS.values())
    f = _capi.KERNEL_FAMILIES.index(family)
    agg["ms_kernel"][f], agg["launches"][f] = 1.0, 1
    r = bench.roofline_of(SimpleNamespace(_capi=_capi), agg, "none")
    assert r["kernel"] == family and r["algorithmic_bytes_per_launch"] == nbytes
