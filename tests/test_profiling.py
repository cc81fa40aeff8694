"""The profiling summaries' arithmetic, on made-up counter rows (no GPU)."""
import argparse
import json
import subprocess

import pytest

from aieplace_amd import profiling


def run_mfma(monkeypatch, tmp_path, flops, bins):
    """profiling.mfma with a driver that reports `flops` per field solve; (result, commands)."""
    drv = dict(run={}, profile=[dict(name="field_transforms", launches=4, avg_us=100.0, bytes=1.0, flops=flops)])
    cmds = []

    def rocprof(pre, cmd, out_dir, timeout):
        cmds.append(cmd)
        return ["rocprofv3"] + pre + ["--"] + cmd, drv

    values = dict.fromkeys(profiling.MFMA_COUNTERS, 4.0)
    values["SQ_VALU_MFMA_BUSY_CYCLES"] = 8.0  # of 4 SIMDs x 4 cycles: half
    rows = [dict(Dispatch_Id=1, Kernel_Name="k_sym_f32<true, 0, 32>", Counter_Name=c, Counter_Value=v)
            for c, v in values.items()]
    monkeypatch.setattr(profiling, "_rocprof", rocprof)
    monkeypatch.setattr(profiling, "_csv", lambda out_dir, suffix: rows)
    monkeypatch.setattr(profiling, "PROFILES", str(tmp_path))
    monkeypatch.setattr(profiling.subprocess, "run",
                        lambda cmd, **kw: subprocess.CompletedProcess(cmd, 0, json.dumps(drv) + "\n", ""))
    args = argparse.Namespace(workload="stdcell_2m", precision=0, reps=5, scratch=str(tmp_path), timeout=10, bins=bins,
                              iters=0)
    return profiling.mfma(args), cmds


def test_mfma_takes_a_grid_of_products(monkeypatch, tmp_path):
    path, cmds = run_mfma(monkeypatch, tmp_path, 1e12, 0)
    assert cmds[0][cmds[0].index("--bins") + 1] == "4112"
    text = open(path).read()
    assert "mfma field_transforms busy 0.5000 tflops 10000.00" in text


def test_mfma_refuses_a_grid_of_ffts(monkeypatch, tmp_path):
    with pytest.raises(SystemExit, match="FFTs solve the field"):
        run_mfma(monkeypatch, tmp_path, 0.0, 1024)
    assert not list(tmp_path.glob("mfma_*"))


@pytest.mark.parametrize("precision", [0, 1, 2])
def test_dispatches_of_an_item(precision):
    item = dict(name="field_transforms", launches=4, flops=1.0)
    assert profiling._item_dispatches(item, precision) == (5 if precision == 2 else 4)  # and the cleared maxima
    assert profiling._item_dispatches(dict(item, launches=3, flops=0.0), precision) == 3
    assert profiling._item_dispatches(dict(item, name="overflow", launches=1, flops=0.0), precision) == 1
