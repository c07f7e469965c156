"""bench.py's roofline.traffic comes from the committed counter summary only
while the kernel sources are the ones it was measured on, and its CPU
baseline stays within the positions the model holds (no GPU)."""
import os
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)
import bench  # noqa: E402
import pytest  # noqa: E402


def test_traffic_summary_matches_the_sources():
    traffic, commit = bench.measured_traffic(16, "q4_k_m", 4096)
    if traffic is None:
        pytest.skip("the traffic summary was measured on other kernel sources (bench reports null)")
    assert commit
    # 1.0-1.1x the algorithmic bytes of a 4096-context pass (15.46 GB), per 16-pass launch
    assert 16 * 15.4e9 < traffic < 16 * 17.0e9


def test_traffic_is_null_for_other_sources_or_workloads(monkeypatch):
    assert bench.measured_traffic(16, "bf16", 4096) == (None, None)
    assert bench.measured_traffic(16, "q4_k_m", 8192) == (None, None)
    monkeypatch.setattr(bench, "kernel_source_digest", lambda: "0" * 64)
    assert bench.measured_traffic(16, "q4_k_m", 4096) == (None, None)


def test_cpu_baseline_stops_at_the_last_kv_row(monkeypatch):
    """A fast CPU decodes more steps in the time given than the context has
    rows left; a step past the last row writes past the mirrored KV cache."""
    import types
    import oracle
    seen = []

    class Mirror:
        def __init__(self, m):
            pass

        def step(self, tok, pos):
            seen.append(pos)
            return tok, None

    monkeypatch.setattr(oracle, "ModelMirror", Mirror)
    m = types.SimpleNamespace(cfg=types.SimpleNamespace(n_ctx=4157))
    r = bench.cpu_baseline(m, 4096, 1e9)
    assert seen == list(range(4096, 4157)) and r["value"] > 0


def test_traffic_depends_on_the_interpreters_own_sources_only():
    """The figure is for what interp.hip is compiled from: a change to the
    batched prefill's units or their header leaves it valid."""
    names = {os.path.basename(p) for p in bench.kernel_sources()}
    assert {"interp.hip", "internal.h", "isa.h", "dev_common.h", "gemv.h", "gdn.h", "attn.h", "synth.h"} == names
    csrc = os.path.join(ROOT, "sinter-qwen36-nomtp-tu102_amd", "csrc")
    others = [f for f in os.listdir(csrc) if f.endswith((".h", ".hip")) and f not in names]
    assert "batched.h" in others and "ubatch.hip" in others
    for f in names:
        with open(os.path.join(csrc, f)) as s:
            assert "batched.h" not in s.read(), f
