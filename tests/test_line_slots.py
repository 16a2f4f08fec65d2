"""The LDS slots of the sweep kernels' lines, by the layout's own functions on
the host: every one lies inside its line, for every row count and both widths
(the mirrored dummy slot of 5 rows a lane was one before it)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


def test_every_slot_is_inside_its_line(tmp_path):
    exe = str(tmp_path / "line_slots")
    subprocess.run([HIPCC, "-O1", "-std=c++17", "--offload-arch=gfx950", "--offload-host-only", "-w",
                    "-I" + os.path.join(ROOT, "nuc3d-cartisian_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "line_slots.hip"), "-o", exe], check=True, timeout=300)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
