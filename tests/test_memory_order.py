"""Memory that outlives a handle is handed out behind its last use, also where a wait fails: the library's host code,
compiled for the host alone, on a stand-in for the HIP runtime (cases/fake_runtime.cpp)."""
import importlib.util
import re
import subprocess

import pytest

from conftest import ROOT

SCENARIOS = re.findall(r"^ +SCENARIO\((\w+)\)", (ROOT / "tests" / "cases" / "fake_runtime.cpp").read_text(), re.M)


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    spec = importlib.util.spec_from_file_location("_accel_build", ROOT / "iccad-accel-gcn_amd" / "build.py")
    build = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(build)
    out = tmp_path_factory.mktemp("fake_runtime")
    sources = [build.CSRC / s for s in build.SOURCES if s.endswith(".hip")] + [ROOT / "tests" / "cases" / "fake_runtime.cpp"]
    # the host half of each source alone: the kernels' device code is not compiled, their launches are calls
    flags = ["-x", "hip", "--offload-host-only", f"--offload-arch={build.ARCH}", "-O1", "-std=c++17",
             "-Wno-unused-command-line-argument", "-Wno-unused-result", f"-I{ROOT / 'include'}", f"-I{build.CSRC}"]
    objects = [out / (s.name + ".o") for s in sources]
    running = [subprocess.Popen([build.hipcc(), *flags, "-c", str(s), "-o", str(o)], stdout=subprocess.PIPE,
                                stderr=subprocess.STDOUT, text=True) for s, o in zip(sources, objects)]
    for p in running:
        text, _ = p.communicate()
        assert p.returncode == 0, text
    # the code objects that are not there
    names = subprocess.run(["nm", "-u", *map(str, objects)], check=True, capture_output=True, text=True).stdout
    absent = [f"-Wl,--defsym={n}=0" for n in sorted(set(re.findall(r"\b__hip_fatbin\w*", names)))]
    exe = out / "fake_runtime"
    subprocess.run(["g++", "-no-pie", "-pthread", *map(str, objects), *absent, "-o", str(exe)], check=True)
    return exe


@pytest.mark.parametrize("scenario", SCENARIOS)
def test_memory_is_handed_out_behind_its_last_use(program, scenario):
    r = subprocess.run([str(program), scenario], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
