"""The harness's --counters join against the library's own kernels: every
kernel that a suite kernel launches is counted for it, and for it alone."""

import csv
import os
import subprocess

import pytest

from rajaperf_amd.suite import run_suite

pytestmark = pytest.mark.gpu

# Device kernels (names without their template arguments) of each suite kernel.
OWN = {
    "Algorithm_SCAN": ["scan_kernel"],
    "Algorithm_SORT": ["gather_kernel", "sample_kernel", "hist_kernel", "colscan_kernel", "scatter_kernel",
                       "second_level_kernel", "bucket_kernel", "overfull_kernel"],
    "Polybench_GEMM": ["gemm_mfma_f64_kernel", "gemm_naive_kernel"],
    "Polybench_JACOBI_2D": ["jacobi_block_kernel", "jacobi_wide_kernel", "jacobi_grid_kernel", "jacobi_fused_kernel",
                            "jacobi_stream_kernel", "jacobi_vec_kernel", "jacobi_scalar_kernel"],
    "Apps_MASS3DPA": ["mass3dpa_kernel", "mass3dpa_naive_kernel"],
    "Apps_DIFFUSION3DPA": ["diffusion3dpa_kernel"],
}
# The first template argument tells these apart.
BY_ARGUMENT = {
    "stream_vec_kernel": {"0": "Stream_COPY", "1": "Stream_MUL", "2": "Stream_ADD", "3": "Stream_TRIAD"},
    "reduce_kernel": {"true": "Stream_DOT", "false": "Algorithm_REDUCE_SUM"},
    "small_reduce_kernel": {"true": "Stream_DOT", "false": "Algorithm_REDUCE_SUM"},
}
# Input generation, table set-up, unaligned streams, and kernels of entry points outside the suite's own.
OTHER = {"fill_const_kernel", "fill_formula_kernel", "fill_grid_kernel", "fill_sym_tensor_kernel",
         "fill_uniform_kernel", "zero_kernel", "zero_u32_kernel", "boundary_copy_kernel", "seg_prep_kernel",
         "stream_scalar_kernel", "mass3dpa_batched_kernel", "mass3dpa_order_kernel", "mass3dpa_order_chunk_kernel",
         "mass3dpa_mixed_kernel", "diffusion3dpa_mixed_kernel", "kron_slices_kernel", "diff_kron_slices_kernel",
         "prepare_kernel", "split_cols_kernel", "ozaki_gemm_kernel", "crt_combine_kernel"}


def library_kernels(rpx):
    """Demangled signatures of the library's kernels, from the host stubs hipcc makes for them."""
    out = subprocess.run(["nm", "-C", rpx.lib().path], check=True, capture_output=True, text=True).stdout
    return sorted({line.split(" ", 2)[2].replace("__device_stub__", "") for line in out.splitlines()
                   if "__device_stub__" in line})


def owner(signature):
    name = signature.split("::", 1)[1]
    base, _, rest = name.partition("<") if "<" in name.split("(")[0] else (name.split("(")[0], "", "")
    if base in BY_ARGUMENT:
        return BY_ARGUMENT[base][rest.split(",")[0].split(">")[0]]
    for kernel, names in OWN.items():
        if base in names:
            return kernel
    assert base in OTHER, f"{base}: which suite kernel is it behind?"
    return None


def test_every_kernel_is_joined(rpx, tmp_path):
    signatures = library_kernels(rpx)
    assert len(signatures) > 100
    cnt = tmp_path / "counter_collection.csv"
    with open(cnt, "w", newline="") as f:
        w = csv.writer(f)
        w.writerow(["Dispatch_Id", "Kernel_Name", "Counter_Name", "Counter_Value"])
        for i, s in enumerate(signatures):
            w.writerow([i, s, f"c{i}", i + 1])
    res = run_suite(["--size", "20000", "--checkrun", "1", "--input-mode", "seeded", "-t", "default", "--counters",
                     str(cnt)])
    assert res["rc"] == 0, res.get("failures")
    rows = {r["Kernel"]: r for r in csv.DictReader(open(os.path.join(res["outdir"], "RAJAPerf-roofline.csv")))}
    assert len(rows) == 12
    for i, s in enumerate(signatures):
        column = f"c{i} per dispatch"
        joined = [k for k, r in rows.items() if r.get(column)]
        want = owner(s)
        assert joined == ([want] if want else []), s
        if want:
            assert float(rows[want][column]) == i + 1
