"""What bench.py says of its launches: every operation of a chunk counted, every kernel that it names in the sources (no GPU)."""
import os
import re
import sys
import types

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)


@pytest.mark.parametrize("path", ["exact", "bf16"])
def test_a_chunks_launches_add_up_to_its_products(monkeypatch, path):
    import bench
    from illatio_amd import ds4f, hip
    dev, n, ne, nu, d, ff, seen = hip.Device(0, hip.DeviceInfo(), 0), 40, 16, 3, 512, 256, []
    monkeypatch.setattr(hip, "launch", lambda dev, kernel, grid, block, args, shared=0: seen.append((kernel, args)))
    buf = lambda dev, nbytes, zero=True: hip.DBuf(0x1000, nbytes, dev)
    pool = types.SimpleNamespace(d=d, ff=ff, gate_bytes=ff * d // 256 * 66, grb=d // 256 * 66, drb=ff // 256 * 84, ptrs=buf(dev, 8 * ne))
    routed = ds4f.ffn_routed_chunk_bf16 if path == "bf16" else ds4f.ffn_routed_chunk
    x = buf(dev, 4 * n * d)
    routed(dev, pool, x, x, x, n, ne, nu, 1.5, 0.0, ws=types.SimpleNamespace(alloc=buf))
    assert sum(bench.chunk_work(kernel, args, n * nu) for kernel, args in seen) == 2.0 * n * nu * 3 * ff * d


def test_every_kernel_it_names_is_in_the_sources():
    src = os.path.join(ROOT, "illatio_amd", "csrc")
    text = "".join(open(os.path.join(src, f)).read() for f in sorted(os.listdir(src)) if f.endswith(".hip"))
    here = set(re.findall(r"__global__[^;{]*?\b([a-z0-9_]+_kernel)\(", text))
    named = {k for f in ("bench.py", os.path.join("profiles", "hbm_traffic_per_launch.md")) for k in re.findall(r"\b([a-z0-9]\w*_kernel)\b(?!_c\d)", open(os.path.join(ROOT, f)).read())}
    assert len(here) > 30 and len(named) > 5
    assert not named - here
