"""The host side of bulk transfers and kept device blocks (csrc/hostio.hip),
run without a device: hostio_harness.cpp stands in for the HIP calls.
no_memory: a transfer that cannot allocate still moves the data, with no
exception out of the C ABI.  kept_blocks: at most 4 GiB stay, those of the
latest calls, and all go with the last context."""
import shutil
import subprocess
from pathlib import Path

import pytest

from ramgpu.build import CSRC, HIPCC_FLAGS, INCLUDE, hipcc

HERE = Path(__file__).resolve().parent


@pytest.fixture(scope="module")
def harness(tmp_path_factory):
    try:
        cc = hipcc()
    except FileNotFoundError:
        pytest.skip("no hipcc")
    out = tmp_path_factory.mktemp("hostio")
    flags = [f for f in HIPCC_FLAGS if f != "-shared"] + ["--cuda-host-only", f"-I{INCLUDE}", f"-I{CSRC}"]
    objs = []
    for src, lang in ((CSRC / "hostio.hip", []), (HERE / "hostio_harness.cpp", ["-x", "hip"])):
        objs.append(str(out / (src.name + ".o")))
        subprocess.run([cc, *flags, *lang, "-c", str(src), "-o", objs[-1]], check=True, capture_output=True)
    exe = out / "harness"
    cxx = shutil.which("g++") or shutil.which("c++")
    subprocess.run([cxx, *objs, "-o", str(exe), "-lpthread"], check=True)
    return exe


@pytest.mark.parametrize("check", ["no_memory", "kept_blocks"])
def test_hostio(harness, check):
    r = subprocess.run([str(harness), check], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, f"{r.returncode}: {r.stdout}{r.stderr}"
