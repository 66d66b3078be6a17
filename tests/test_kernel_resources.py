"""What the compiler reports for kernels whose speed rests on their registers:
waves per SIMD that fit, and no spilled register."""
import os
import re
import subprocess

import pytest

from xyce_amd import build

pytestmark = pytest.mark.skipif(not os.path.exists(build.HIPCC), reason="no hipcc here")


def _report(src):
    """{mangled kernel name: {field: value}} of a source's device code, from
    the build's own flags."""
    r = subprocess.run([build.HIPCC] + build.COMMON + build.DEVICE +
                       ["-x", "hip", "--cuda-device-only", "-c",
                        os.path.join(build.CSRC, src), "-o", os.devnull,
                        "-Rpass-analysis=kernel-resource-usage"],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    out, name = {}, None
    for key, value in re.findall(r"remark:\s+([^:\n]+): (\S+)", r.stderr):
        if key == "Function Name":
            name = value
            out[name] = {}
        else:
            out[name][key] = int(value) if value.lstrip("-").isdigit() else value
    return out


def test_fold_keeps_full_occupancy():
    """The fold gathers at random: every circuit's short records need all
    eight waves per SIMD, beside the wide form (a lane per chunk) too.  With
    the wide form's 104 registers in every load (four waves), an RC ladder's
    load took 18.2 us instead of 16.7."""
    folds = {k: v for k, v in _report("xg_reduce.hip").items() if "fold_kernel" in k}
    assert folds
    for name, r in folds.items():
        assert r["Occupancy [waves/SIMD]"] == 8, (name, r)
        assert r["SGPRs Spill"] == 0 and r["VGPRs Spill"] == 0, (name, r)


def test_panels_spill_no_register():
    """A panel's row tiles are in registers (or its rows in memory, above 2048)
    so that a column step waits on its own chain only."""
    panels = {k: v for k, v in _report("xg_front.hip").items() if "panel_kernel" in k}
    assert len(panels) == 6
    for name, r in panels.items():
        assert r["VGPRs Spill"] == 0, (name, r)
        assert r["ScratchSize [bytes/lane]"] == 0, (name, r)
