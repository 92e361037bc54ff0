"""The fp32 kernel's counted waits, read from the assembly that its source compiles to (CPU; no kernel runs).

`attend_f32` lets a tile's K, loaded straight into LDS, land by a count of the
loads still in flight. A load that the compiler drops because nothing reads it
is not there to be counted, so every wait that leaves N loads in flight is
checked against the loads that really stand before it.
"""

from __future__ import annotations

import re
import subprocess

import pytest

from liteinfer_amd import _build


def _assembly(tmp_path) -> str:
    try:
        compiler = _build.hipcc()
    except RuntimeError as e:
        pytest.skip(str(e))
    out = tmp_path / "attend_f32.s"
    subprocess.run([compiler, *_build.DEVICE_FLAGS, *_build.SOURCE_FLAGS.get("attend_f32.hip", []), "-w",
                    "--offload-device-only", "-S", str(_build.CSRC_DIR / "attend_f32.hip"), "-o", str(out)],
                   check=True, capture_output=True, timeout=300)
    return out.read_text()


def _counted_waits(body: str):
    """(N, loads before it in its basic block) of each hand-written ``s_waitcnt vmcnt(N)`` with N > 0."""
    loads, ours = 0, False
    for line in body.splitlines():
        text = line.strip()
        if re.match(r"\.LBB\d+_\d+:", text):
            loads = 0
        elif text.startswith(";APP") or text.startswith(";;#ASMSTART"):
            ours = True
        elif text.startswith(";NO_APP") or text.startswith(";;#ASMEND"):
            ours = False
        elif text.startswith("global_load"):
            loads += 1
        elif ours and (m := re.match(r"s_waitcnt vmcnt\((\d+)\)$", text)) and int(m[1]):
            yield int(m[1]), loads


def test_every_counted_wait_has_its_loads(tmp_path):
    kernels = re.findall(r"^_ZN\S*attend_f32ILi(\d+)\S*:(.*?)^\s*s_endpgm", _assembly(tmp_path), re.M | re.S)
    assert sorted(int(dim) for dim, _ in kernels) == [64, 128]
    for dim, body in kernels:
        waits = list(_counted_waits(body))
        assert waits  # (the loop's two steps)
        tile_v = 4 * int(dim) // 64  # the tile's own V loads, issued after its K in the step before
        for n, loads in waits:
            assert n == 2 * tile_v + 1
            # The tile's K is older than its V and the step's loads; with no
            # more than n in flight it has landed only if they are n or more.
            assert tile_v + loads >= n, f"head_dim {dim}: vmcnt({n}) after {loads} loads of the step"
