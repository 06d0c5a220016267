"""The library's Makefile used from any folder."""
import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "laboetie_amd", "csrc")


def test_makefile_runs_from_any_folder(tmp_path):
    """Every prerequisite is found beside the Makefile, not in the working
    folder; and each header of the library is one."""
    r = subprocess.run(["make", "-n", "-B", "-f", os.path.join(CSRC, "Makefile")], cwd=tmp_path, capture_output=True,
                       text=True)
    assert r.returncode == 0, r.stderr
    db = subprocess.run(["make", "-n", "-p", "-f", os.path.join(CSRC, "Makefile")], cwd=tmp_path, capture_output=True,
                        text=True).stdout
    rule = next(line for line in db.splitlines() if "liblbx.so:" in line)
    for h in os.listdir(CSRC):
        if h.endswith(".h"):
            assert os.path.join(CSRC, h) in rule, h
