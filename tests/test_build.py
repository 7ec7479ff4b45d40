"""The package's Makefile: a change of the flags rebuilds what they compile."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "-damn-low-level-fence-inference-version-1_amd")


def test_a_changed_makefile_rebuilds_every_object():
    # a dry run in which the Makefile counts as just changed
    out = subprocess.run(["make", "-n", "-C", PKG, "-W", os.path.join(PKG, "Makefile")], capture_output=True,
                         text=True, check=True).stdout
    for src in sorted(os.listdir(os.path.join(PKG, "csrc"))):
        if src.endswith((".hip", ".cpp")):
            assert f"csrc/{src} -o" in out, f"{src} keeps an object built with other flags"
