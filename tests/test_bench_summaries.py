"""The counter summaries of bench.py find a kernel that is a template by its plain name."""
import csv

import bench

COUNTERS = ("SQ_LDS_BANK_CONFLICT", "SQ_LDS_IDX_ACTIVE", "SQ_INSTS_LDS", "SQ_WAIT_INST_LDS", "SQ_BUSY_CYCLES",
            "SQ_INSTS_VALU", "SQ_INSTS_VMEM_RD", "SQ_WAIT_INST_ANY", "TA_TA_BUSY_sum", "TD_TD_BUSY_sum")
KERNELS = ("void vfd::k_density_factor<4u>(vfd::SceneParams const*)", "vfd::k_div_iter(vfd::SceneParams const*)",
           "void vfd::k_build_halo<4u, 1u>(vfd::SceneParams const*)")


def _run(tmp_path):
    with open(tmp_path / "run_counter_collection.csv", "w", newline="") as f:
        w = csv.DictWriter(f, ["Kernel_Name", "Counter_Name", "Counter_Value", "Start_Timestamp", "End_Timestamp"])
        w.writeheader()
        for k in KERNELS:
            for c in COUNTERS:
                w.writerow(dict(Kernel_Name=k, Counter_Name=c, Counter_Value=32e5, Start_Timestamp=0, End_Timestamp=10**6))
    return str(tmp_path)


def test_instantiations_are_found_by_the_kernel_name(tmp_path):
    run = _run(tmp_path)
    rows = [line.split("|")[1].strip() for line in bench.counter_summary(run, run).splitlines()[2:]]
    assert rows == ["div_iter", "density_factor", "build_halo"]
    rows = [line.split("|")[1].strip() for line in bench.memory_unit_summary(run).splitlines()[2:]]
    assert rows == ["div_iter", "build_halo"]
