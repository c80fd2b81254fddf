"""The rocprofv3 summary tool's traffic calibration (CPU only: synthetic counter CSVs).

FETCH_SIZE / WRITE_SIZE readings are scaled by what the same counters read for the
256 MiB calibration copy that `bench.py --profile` runs. An input recipe may launch
the copy's kernel on larger or smaller tensors too; the copy is told apart by its grid.
"""

import csv

from evograd_amd import profiling

FIELDS = ["Dispatch_Id", "Kernel_Name", "Grid_Size", "Counter_Name", "Counter_Value",
          "Start_Timestamp", "End_Timestamp"]
COPY = "void at::native::vectorized_elementwise_kernel<4, at::native::AUnaryFunctor<float, " \
       "float, float, at::native::binary_internal::MulFunctor<float> > >"


def _write(path, counter, rows):
    with open(path, "w", newline="") as f:
        w = csv.DictWriter(f, fieldnames=FIELDS)
        w.writeheader()
        for i, (name, grid, kib) in enumerate(rows):
            w.writerow({"Dispatch_Id": i + 1, "Kernel_Name": name, "Grid_Size": grid,
                        "Counter_Name": counter, "Counter_Value": kib,
                        "Start_Timestamp": 0, "End_Timestamp": 1000})


def test_traffic_calibrates_on_the_copy_grid_not_the_largest_reading(tmp_path):
    copy_kib = profiling.COPY_BYTES / 1024
    # FETCH_SIZE reads half the copy's bytes on this part (x2 calibration), WRITE_SIZE
    # all of them; a recipe scaling an 8x larger tensor with the same kernel comes first
    fetch = [(COPY, profiling.COPY_GRID * 8, 8 * copy_kib / 2),
             ("eg::my_kernel", 4096, 1000.0),
             ("eg::my_kernel", 4096, 1002.0),
             (COPY, profiling.COPY_GRID, copy_kib / 2)]
    write = [(COPY, profiling.COPY_GRID * 8, 8 * copy_kib),
             ("eg::my_kernel", 4096, 500.0),
             ("eg::my_kernel", 4096, 500.0),
             (COPY, profiling.COPY_GRID, copy_kib)]
    _write(tmp_path / "f.csv", "FETCH_SIZE", fetch)
    _write(tmp_path / "w.csv", "WRITE_SIZE", write)
    e = profiling.traffic(str(tmp_path / "f.csv"), str(tmp_path / "w.csv"), "my_kernel", "k")
    assert e["key"] == "k"
    assert abs(e["copy_calibration"]["fetch_scale"] - 2.0) < 1e-12
    assert abs(e["copy_calibration"]["write_scale"] - 1.0) < 1e-12
    # the kernel's median reading (1001 KiB fetched, 500 KiB written), scaled
    assert e["fetch_bytes_per_launch"] == round(1001.0 * 1024 * 2)
    assert e["write_bytes_per_launch"] == 500 * 1024
    assert e["hbm_bytes_per_launch"] == e["fetch_bytes_per_launch"] + e["write_bytes_per_launch"]


def test_bench_finds_a_layers_products_on_either_kernel():
    """The decoder layer reports its gate and up projections, the third product, whichever
    kernels the products before it run on."""
    import bench

    kt = {k: 1.0 for k in ("fwd:0:rmsnorm_fwd_row", "fwd:1:gemm_kernel",
                           "fwd:2:splitk_reduce_kernel", "fwd:3:attn_fwd_kernel",
                           "fwd:4:gemm_mid_kernel", "fwd:5:gemm_kernel", "fwd:6:silu_mul_kernel",
                           "fwd:7:gemm_kernel", "bwd:0:gemm_kernel")}
    phase, name, occurrence = bench.DOMINANT["llama3_decoder_layer@llama3_8b_T1024"]
    assert bench.find_kernel(kt, phase, name, occurrence) == "fwd:5:gemm_kernel"
    assert bench.find_kernel(kt, "fwd", "silu_mul_kernel", 0) == "fwd:6:silu_mul_kernel"


def test_bench_line_leaves_the_details_out():
    """The result line's share of one operator is its figures, whatever the number of
    kernels and saved tensors behind them, and an operator that failed keeps its error."""
    import json

    import bench

    r = {"config": {"dims": {"T": 1024}, "dtype": "bfloat16"}, "fwd_us": 555.0900001,
         "bwd_us": 1450.4, "full_us": 1947.8, "mfma_frac_full": 0.27951234,
         "saved": {"logical_saved_bytes": 462053376, "ratio_to_memory_inputs": 1.5},
         "saved_tensors": [{"kind": "tensor", "shape": [1024, 4096]}] * 40,
         "kernels_us": {f"bwd:{i}:gemm_kernel": 200.123456789 for i in range(60)},
         "dominant_kernel": {"name": "fwd:8:gemm_kernel", "phase": "fwd", "us": 209.891234,
                             "flops": 1, "frac": 0.45534}}
    out = bench.op_summary(r)
    assert out == {"fwd_us": 555.09, "bwd_us": 1450.4, "full_us": 1947.8,
                   "mfma_frac_full": 0.27951, "saved_bytes": 462053376,
                   "kernel": {"name": "fwd:8:gemm_kernel", "us": 209.89, "frac": 0.45534}}
    assert len(json.dumps(out)) < 400
    assert bench.op_summary({"error": "RuntimeError: x"}) == {"error": "RuntimeError: x"}
    sweep = {"256": {"full_us": 13.1, "hbm_frac_full": 0.1, "kernels_us": {"k": 4.0}}}
    assert bench.sweep_summary(sweep) == {"256": [13.1, 0.1]}
    assert bench.sweep_summary({"error": "e"}) == {"error": "e"}
