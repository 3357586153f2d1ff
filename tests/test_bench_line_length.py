"""The default line keeps to a few KB, with the headline exact and every part of it still there; the rest goes to --details.
CPU only."""
import copy
import json
import os
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)
import bench  # noqa: E402

X = 12345678901.234567


def unsteady():
    roofline = dict(bound="hbm", kernel="k_grad", achieved=X / 1e7, peak=8000.0, unit="GB/s", frac=X / 3e10, traffic=X,
                    traffic_source="profiles/hbm_traffic_vortex2d.md", alg_bytes=X)
    kern = {f"k_{k}": dict(launches=12, avg_us=X / 1e8, total_ms=X / 1e10, alg_bytes=X, gbs=X / 1e7, timed_one_in=5)
            for k in ("grad", "flux", "update")}
    base = dict(value=X, unit="face-updates/s", cores=16, kind="port", sample="x" * 130, cpu_model="y" * 40, nproc=16,
                usable_cpus=16, threads8=dict(value=X, sample="x" * 130))
    return dict(metric="m" * 80, value=X, unit="face-updates/s", n_gpus=1, steps=20, warmup=5, ms_per_step=X / 1e9,
                higher_is_better=True, scaling="weak", vs_baseline=None, dtype="f64", data="synthetic",
                config=dict(workload="w" * 80, cells=2000000, faces=3002000, scheme="Roe", limiter="van Leer", rk=3, cfl=0.5,
                            strategy="fused", cell_order="hilbert", context_setup_s=X / 1e10),
                roofline=roofline, kernels=kern,
                strategies={s: dict(value=X, ms_per_step=X / 1e9, roofline=dict(roofline), kernels=copy.deepcopy(kern))
                            for s in ("face", "cell", "patch", "fused")},
                copy_probe=dict(bytes=268435456, ms=X / 1e10, gbs=X / 1e7),
                mixed=dict(value=X, ms_per_step=X / 1e9, speedup=X / 1e10, dtype="fp32 flux+limiter / fp64 gather+update",
                           strategy="fused", kernels=copy.deepcopy(kern), strategies={s: X / 1e9 for s in "abcd"},
                           compare_steps=200, rel_l2_per_field=[X / 1e18] * 5, rel_linf_per_field=[X / 1e16] * 5),
                fused_minimum=dict(bytes_per_stage=216048000, achieved_gbs=X / 1e7, frac=X / 3e10), state_finite=True,
                cpu_baseline=base)


def test_default_line():
    out = unsteady()
    case = {f"field_{k}": X / 1e9 for k in range(40)}
    out["configs"] = dict(pulse3d=unsteady(), ramp=dict(
        metric="m" * 60, config=dict(workload="w" * 200, cells=300000, faces=450850), unit="s",
        cold={k: X / 1e11 for k in ("explicit_s", "lusgs_s", "lusgs_speedup_vs_explicit")}, roofline=out["roofline"],
        kernels=out["kernels"], cpu_baseline=out["cpu_baseline"],
        warm_start=dict(value=X / 1e10, unit="u" * 130, summary={f"key_of_summary_{k}": X / 1e10 for k in range(16)},
                        training={f"k{k}": X for k in range(8)}, network={f"k{k}": X for k in range(8)}, held_out=8,
                        cases=[case] * 8)))
    full = copy.deepcopy(out)
    line = json.dumps(bench.short_line(out))
    assert out == full  # (what --details writes)
    assert len(json.dumps(full)) > 15000 and len(line) < 8000, len(line)
    d = json.loads(line)
    assert d["value"] == full["value"] and d["ms_per_step"] == full["ms_per_step"]
    assert set(d) == set(full) and set(d["configs"]["pulse3d"]) == set(full["configs"]["pulse3d"])
    assert abs(d["roofline"]["frac"] / full["roofline"]["frac"] - 1) < 1e-5
    assert abs(d["configs"]["pulse3d"]["strategies"]["patch"]["value"] / X - 1) < 1e-5
    assert "cases" not in d["configs"]["ramp"]["warm_start"] and d["configs"]["ramp"]["warm_start"]["held_out"] == 8
