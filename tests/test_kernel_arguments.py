"""Static check of the kernels' argument lists, on the metadata of the gfx950
code (CPU only: hipcc cross-compiles): every argument is a number to the
runtime (a pointer parameter would cost host time in each launch) and lies at
its natural alignment, which is how launch.hpp's enqueue packs the buffer it
launches with."""
import importlib.util
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "dinov3-loom_amd")
spec = importlib.util.spec_from_file_location("dinov3_build_flags", os.path.join(PKG, "build.py"))
build = importlib.util.module_from_spec(spec)
spec.loader.exec_module(build)


@pytest.mark.parametrize("src", [s for s in build.SOURCES if s.endswith(".hip")])
def test_arguments_are_numbers_at_their_natural_alignment(src, tmp_path):
    if not os.path.exists(build.HIPCC):
        pytest.skip("hipcc not found")
    out = str(tmp_path / "kernels.s")
    subprocess.check_call([build.HIPCC, *build.COMMON, *build.DEVICE_FLAGS, "--cuda-device-only", "-S",
                           os.path.join(PKG, "csrc", src), "-o", out], stderr=subprocess.DEVNULL)
    kernels = open(out).read().split("amdhsa.kernels:")[1].split("amdhsa.target:")[0].split(".args:")[1:]
    assert kernels
    for text in kernels:
        name = re.search(r"\.name: +(\S+)", text).group(1)
        args = re.findall(r"\.offset: +(\d+)\n +\.size: +(\d+)\n +\.value_kind: +(\S+)", text.split(".group_segment")[0])
        end = 0
        for offset, size, kind in args:
            if kind.startswith("hidden_"):
                continue
            offset, size = int(offset), int(size)
            assert kind == "by_value" and size in (4, 8), (name, kind, size)
            assert offset == (end + size - 1) // size * size, (name, offset)
            end = offset + size
        assert end > 0, name
