"""The traffic summary finds its kernels by name prefix: every prefix names a
kernel of the built library (a template parameter added to a kernel would leave
its rows out without a word)."""
import os
import shutil
import subprocess

import pytest

from mesoengine_amd import traffic

LIB = os.path.join(os.path.dirname(traffic.__file__), "_build", "libmeso_hip.so")


@pytest.mark.skipif(not os.path.exists(LIB) or not shutil.which("c++filt"),
                    reason="library not built")
def test_every_prefix_names_a_kernel():
    syms = subprocess.run(["nm", LIB], capture_output=True, text=True, check=True).stdout
    mangled = [line.split()[-1] for line in syms.splitlines() if "meso" in line]
    names = subprocess.run(["c++filt"], input="\n".join(mangled), capture_output=True,
                           text=True, check=True).stdout.splitlines()
    for prefix in traffic.KERNELS:
        if prefix.startswith("void meso::"):
            assert any(n.startswith(prefix) for n in names), prefix
