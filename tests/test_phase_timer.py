"""The phase timers when memory runs out (cqbem_pool.hpp): the end of a timed scope allocates nothing (an exception there would
end the process), its beginning throws to the caller; every event is recorded in pairs and destroyed."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_out_of_memory(tmp_path):
    out = tmp_path / "check"
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    r = subprocess.run([hipcc, "-x", "hip", "--offload-host-only", "-O1", "-std=c++17", "-o", str(out),
                        os.path.join(HERE, "phase_timer_check.cpp")], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([str(out)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, (r.returncode, r.stderr)
    assert r.stdout.split() == ["1", "1", "0", "0"]
