"""The library's host code when the HIP runtime fails or a thread cannot be
had: C++ programs that compile it with the runtime's calls on host memory
(tests/cpp/hip_host.h), so every call can be made to fail without a device."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "quadray-engine_amd", "csrc")
PROGRAMS = {"upload_faults": ["engine", "image"],
            "batch_download": ["engine", "image", "capi", "batch"],
            "serve_faults": ["engine", "image", "capi", "serve"]}


@pytest.fixture(scope="module")
def programs(tmp_path_factory):
    """The programs, by name; every source is compiled once, side by side."""
    out = tmp_path_factory.mktemp("faults")
    flags = ["-std=c++17", "-O1", "-Wall", "-Wno-unused-function", "-D__HIP_PLATFORM_AMD__",
             "-I", "/opt/rocm/include", "-I", os.path.join(ROOT, "include"), "-I", CSRC]
    parts = sorted(set(sum(PROGRAMS.values(), [])))
    src = {p: os.path.join(CSRC, p + ".cpp") for p in parts}
    src.update({p: os.path.join(ROOT, "tests", "cpp", p + ".cpp") for p in PROGRAMS})
    jobs = [subprocess.Popen(["g++", *flags, "-c", s, "-o", str(out / (p + ".o"))])
            for p, s in src.items()]
    assert [j.wait() for j in jobs] == [0] * len(jobs)
    for p, need in PROGRAMS.items():
        subprocess.run(["g++", "-o", str(out / p)] + [str(out / (x + ".o")) for x in [p, *need]] +
                       ["-lpthread"], check=True)
    return {p: str(out / p) for p in PROGRAMS}


def run(exe, *args):
    res = subprocess.run([exe, *args], capture_output=True, text=True, timeout=120)
    assert res.returncode == 0, (res.returncode, res.stdout[-2000:], res.stderr[-2000:])
    return res.stdout


def test_tables_after_a_failed_upload(programs):
    """Whichever call of an upload or of a device update fails, the next
    upload leaves every device table current: none is taken for sent."""
    print(run(programs["upload_faults"]))


def test_batch_download_into_shared_buffers_and_after_faults(programs):
    """Frames whose requests name the same memory leave what downloads one
    after another would; a download whose allocations, threads or runtime
    calls fail returns an error or the frames, and the next one the frames."""
    run(programs["batch_download"], "shared")
    print(run(programs["batch_download"], "faults"))


def test_server_after_a_failed_request(programs):
    """Whichever call of a served request fails, the requests after it get
    their own scenes' frames."""
    print(run(programs["serve_faults"]))
