"""What the dense f32 products refuse, on the host: no GPU is asked for anything before the refusal."""
import os
import subprocess

from burn_dragon_amd import build

HERE = os.path.dirname(os.path.abspath(__file__))


def test_a_product_added_to_a_c_in_pieces_is_refused(tmp_path):
    exe = str(tmp_path / "gemm_refusal_test")
    subprocess.run([build.HIPCC, *build.FLAGS, "-x", "hip", os.path.join(HERE, "gemm_refusal_test.cpp"), "-x", "none", "-o", exe, "-L" + build.PKG,
                    "-lbdh_mi355x", "-Wl,-rpath," + build.PKG], check=True, capture_output=True)
    done = subprocess.run([exe], capture_output=True, text=True)
    assert done.returncode == 0 and done.stdout == "ok\n", (done.returncode, done.stdout, done.stderr)
