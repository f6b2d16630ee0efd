"""bench.py's traffic bookkeeping names kernels that the library has: the
patterns of the headline path's kernel classes and the committed counter file
each match a built kernel, a counter run without one of the classes is refused,
and bytes measured for another kernel are not reported as the running one's."""
import json
import os
import shutil
import subprocess

import pytest

import bench
import gdhip


def _built_kernels():
    so = os.path.join(os.path.dirname(gdhip.__file__), "libgdhip.so")
    if not os.path.exists(so) or not shutil.which("nm"):
        pytest.skip("needs the built library and nm")
    out = subprocess.run(["nm", "-C", so], capture_output=True, text=True, check=True).stdout
    return [line.split("__device_stub__", 1)[1] for line in out.splitlines() if "__device_stub__" in line]


def _name(k):
    return k.split("(anonymous namespace)::")[-1].replace("void ", "").split("(")[0]


def test_patterns_and_counter_file_name_built_kernels():
    built = _built_kernels()
    for cls in bench.TANG_KERNELS:
        for fp64 in (False, True):
            assert any(bench.is_tang_kernel(cls, fp64, k) for k in built), (cls, fp64)
    with open(bench.TRAFFIC_JSON) as f:
        traffic = json.load(f)
    for prec in ("fp32", "fp64"):
        assert set(traffic[prec]) == set(bench.TANG_KERNELS)
        for cls, rec in traffic[prec].items():
            assert bench.is_tang_kernel(cls, prec == "fp64", rec["kernel"]), rec["kernel"]
            assert any(_name(rec["kernel"]) == _name(k) for k in built), rec["kernel"]


def _counter_run(path, drop=None):
    for cnt in ("fetch", "write"):
        os.makedirs(os.path.join(path, cnt))
        with open(os.path.join(path, cnt, "run_counter_collection.csv"), "w") as f:
            f.write('"Kernel_Name","Counter_Value"\n"copy_kernel(a)",1024\n')
            for cls, pats in bench.TANG_KERNELS.items():
                for T in ("float", "double"):
                    if (cls, T) != drop:
                        f.write('"void %s(X)",2048\n' % pats[-1].format(T=T))


def test_counter_run_without_a_class_is_refused(tmp_path, monkeypatch):
    monkeypatch.setattr(bench, "TRAFFIC_JSON", str(tmp_path / "traffic.json"))
    _counter_run(str(tmp_path / "whole"))
    out = bench.derive_traffic(str(tmp_path / "whole"))
    assert set(out["fp32"]) == set(out["fp64"]) == set(bench.TANG_KERNELS)
    _counter_run(str(tmp_path / "part"), drop=("analysis_vector", "float"))
    with pytest.raises(RuntimeError):
        bench.derive_traffic(str(tmp_path / "part"))


def test_bytes_of_another_kernel_are_not_reported(tmp_path, monkeypatch):
    path = tmp_path / "traffic.json"
    monkeypatch.setattr(bench, "TRAFFIC_JSON", str(path))
    times = {"synth_vector": 1.0, "ring_fft_products": 0.1}
    for kernel, expect in (("void synth_reg_kernel<float, true, 4, 0>(SynthArgs, int, int)", 7),
                           ("void older_synthesis<float>(SynthArgs)", None)):
        path.write_text(json.dumps({"fp32": {"synth_vector": {"kernel": kernel, "hbm_bytes_per_launch": 7}}}))
        assert bench.roofline(times, "fp32")[1]["traffic"] == expect
