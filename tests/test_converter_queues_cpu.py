"""A blob converter given several command queues in turn, on the CPU: its buffers (page-locked slots, device staging,
scale and bias operands) must not be written again while a queue still has to read them.  The converter's own sources are
compiled with g++ against stand-ins of the C ABI whose queues run only when they are waited for."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HOST = os.path.join(ROOT, "tnn_amd", "host")
LIB = os.path.join(ROOT, "tnn_amd", "lib")


def test_buffers_are_not_rewritten_under_another_queue(tmp_path):
    exe = str(tmp_path / "converter_queues")
    sources = [os.path.join(ROOT, "tests", "cpu_harness", "converter_queues.cc")]
    sources += [os.path.join(HOST, n) for n in ("rocm_device.cc", "host_core.cc")]
    objects = [str(tmp_path / (os.path.basename(s) + ".o")) for s in sources]
    flags = ["-std=c++14", "-O0", "-w", "-fopenmp", "-I" + HOST, "-I" + os.path.join(ROOT, "include")]
    for p in [subprocess.Popen(["g++"] + flags + ["-c", s, "-o", o]) for s, o in zip(sources, objects)]:
        assert p.wait() == 0
    subprocess.check_call(["g++", "-fopenmp", "-o", exe] + objects + ["-L" + LIB, "-ltnn_rocm", "-Wl,-rpath," + LIB])
    out = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0, out.stdout + out.stderr
