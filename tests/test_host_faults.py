"""The library's host code when the HIP runtime fails or a thread cannot be
had: C++ programs that compile it with the runtime's calls on host memory
(tests/cpp/hip_host.h), so every call can be made to fail without a device."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "quadray-engine_amd", "csrc")


def build(out, name, sources):
    exe = str(out / name)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Wno-unused-function",
                    "-D__HIP_PLATFORM_AMD__", "-I", "/opt/rocm/include",
                    "-I", os.path.join(ROOT, "include"), "-I", CSRC,
                    os.path.join(ROOT, "tests", "cpp", name + ".cpp")] +
                   [os.path.join(CSRC, s) for s in sources] + ["-lpthread", "-o", exe],
                   check=True)
    return exe


def run(exe, *args):
    res = subprocess.run([exe, *args], capture_output=True, text=True, timeout=120)
    assert res.returncode == 0, (res.returncode, res.stdout[-2000:], res.stderr[-2000:])
    return res.stdout


def test_tables_after_a_failed_upload(tmp_path):
    """Whichever call of an upload or of a device update fails, the next
    upload leaves every device table current: none is taken for sent."""
    print(run(build(tmp_path, "upload_faults", ["engine.cpp", "image.cpp"])))


def test_batch_download_into_shared_buffers_and_after_faults(tmp_path):
    """Frames whose requests name the same memory leave what downloads one
    after another would; a download whose allocations, threads or runtime
    calls fail returns an error or the frames, and the next one the frames."""
    exe = build(tmp_path, "batch_download",
                ["engine.cpp", "image.cpp", "capi.cpp", "batch.cpp"])
    run(exe, "shared")
    print(run(exe, "faults"))


def test_server_after_a_failed_request(tmp_path):
    """Whichever call of a served request fails, the requests after it get
    their own scenes' frames."""
    exe = build(tmp_path, "serve_faults",
                ["engine.cpp", "image.cpp", "capi.cpp", "serve.cpp"])
    print(run(exe))
