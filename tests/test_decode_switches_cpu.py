"""The environment switches of the decode kernels: of the attention, read in Python and by the launcher (both have to choose the same
kernel), and of the decode products."""
import ctypes
import os
import subprocess
import sys

import pytest

from generativeaiexamples_amd import ops


@pytest.mark.parametrize("nt", [None, "1", "0", "", "false", "true", "00", " 0", "2", "-1", "+0", "0x1", "1x"])
@pytest.mark.parametrize("variant", [None, "1", "0", "01", " 1", "", "one", "3"])
def test_default_kernel_as_the_launcher_reads_it(monkeypatch, nt, variant):
    for name, value in (("GAI_DECODE_NT", nt), ("GAI_DECODE_VARIANT", variant)):
        monkeypatch.delenv(name, raising=False)
        if value is not None:
            monkeypatch.setenv(name, value)
    atoi = ctypes.CDLL(None).atoi
    want = (nt is None or atoi(nt.encode()) != 0) and (variant is None or atoi(variant.encode()) == 1)
    assert ops._decode_default() == want


@pytest.mark.skipif(not ops.native_available(), reason="the kernels are not built")
@pytest.mark.parametrize("asked,want", [(None, [6, 8, 6]), ("8", [8, 8, 8]), ("4", [4, 4, 4]), ("6", [8, 8, 8])])
def test_split_k_waves_as_asked(asked, want):
    """GAI_SPLITK_WPG is what every shape gets, also where the rule would choose six waves. (Read once a process.)"""
    env = {k: v for k, v in os.environ.items() if k != "GAI_SPLITK_WPG"}
    if asked is not None:
        env["GAI_SPLITK_WPG"] = asked
    code = "from generativeaiexamples_amd import ops; print([ops.native().gemm_splitk_waves(*s) for s in ((6144, 4), (4096, 8), (128, 2))])"
    p = subprocess.run([sys.executable, "-c", code], env=env, cwd=os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                       capture_output=True, text=True, timeout=300)
    assert p.returncode == 0 and p.stdout.split("\n")[0] == str(want), p.stdout + p.stderr


@pytest.mark.skipif(not ops.native_available(), reason="the kernels are not built")
@pytest.mark.parametrize("switch,value,want", [(None, None, 1), ("GAI_DEC2", "0", 0), ("GAI_DEC2", "1", 1), ("GAI_DEC2_NT", "8", 0), ("GAI_DEC2_NT", "4", 1)])
def test_pair_of_products_as_asked(switch, value, want):
    """Two products in one launch of the LDS-staged kernel: off with it, and where column tiles of another width are asked for."""
    env = {k: v for k, v in os.environ.items() if not k.startswith("GAI_DEC2")}
    if switch is not None:
        env[switch] = value
    code = "from generativeaiexamples_amd import ops; print(int(ops.native().gemm_dec2_pair_ok(24, 11264, 3088, 2048)))"
    p = subprocess.run([sys.executable, "-c", code], env=env, cwd=os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                       capture_output=True, text=True, timeout=300)
    assert p.returncode == 0 and p.stdout.split("\n")[0] == str(want), p.stdout + p.stderr
