"""The sub-steps in which the lanes of a wave add to shared slots (cqbem_kernels.hpp: in_sub_steps), on 64 host threads that
are ordered by the wave's synchronisation alone: no addition is lost, whatever the threads' timing."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_no_addition_is_lost(tmp_path):
    out = tmp_path / "check"
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    r = subprocess.run([hipcc, "-x", "hip", "--offload-host-only", "-O2", "-std=c++17", "-pthread", "-o", str(out),
                        os.path.join(HERE, "sub_steps_check.cpp")], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr
    for _ in range(3):
        r = subprocess.run([str(out)], capture_output=True, text=True, timeout=60)
        assert [int(t) for t in r.stdout.split()] == [sum(i + 1 for i in range(64) if i % 5 == k) for k in range(5)]
