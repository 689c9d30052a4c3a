"""Device memory kept between problems, against a stand-in of the HIP runtime
(tests/drivers/fake_hip.c): which device a returned block waits for, and what
an upload and the next problem do after one that ran out of memory.  No GPU is
needed."""
import os
import shutil
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    cc = shutil.which("gcc") or shutil.which("cc")
    if not cc:
        pytest.skip("no C compiler")
    out = str(tmp_path_factory.mktemp("fake") / "libfake_hip.so")
    subprocess.check_call([cc, "-shared", "-fPIC", "-O1", "-w", "-o", out,
                           os.path.join(ROOT, "tests", "drivers", "fake_hip.c")])
    return out


def _run(fake, body):
    # its own process: the stand-in comes before the HIP runtime in the search
    code = f"""
import ctypes, sys
sys.path.insert(0, {ROOT!r})
fake = ctypes.CDLL({fake!r}, mode=ctypes.RTLD_GLOBAL)
import bddcml_amd
from bddcml_amd.cube import CubeProblem
p = CubeProblem(8, 2)  # 18,432 triplets a subdomain: assembled on the device
subs = list(p.subdomains())
def start():
    b = bddcml_amd.Bddcml()
    b.init(2, [p.nsub, 1], numbase=p.numbase)
    return b
""" + body
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr


def test_blocks_wait_for_their_own_device(fake):
    """The caller has gone on to another device when the problem ends."""
    _run(fake, """
fake.fake_device(1)
b = start()
for d in subs[:3]:
    b.upload_subdomain_data(d)
assert fake.fake_busy(1) == 1
fake.fake_device(0)
b.finalize()
assert fake.fake_busy(1) == 0, "blocks taken back while their device works"
assert fake.fake_current() == 0
# the blocks serve device 1 again, not device 0
before = fake.fake_copies()
b = start()
b.upload_subdomain_data(subs[0])
assert fake.fake_copies() > before and fake.fake_bad_copies() == 0
b.finalize()
""")


@pytest.mark.parametrize("nth", range(8))
def test_upload_after_out_of_memory(fake, nth):
    """The nth device allocation fails: that upload reports it, and the next
    ones copy into memory that is there."""
    _run(fake, f"""
b = start()
fake.fake_fail_at({nth})
failed = 0
for d in subs:
    for again in range(2):
        try:
            b.upload_subdomain_data(d)
            break
        except RuntimeError as e:
            assert "hipMalloc" in str(e), e
            failed += 1
assert fake.fake_bad_copies() == 0, fake.fake_bad_copies()
assert failed <= 1
assert failed == 1 or {nth} > 2
b.finalize()
""")


@pytest.mark.parametrize("what", ["fake_fail_at", "fake_fail_host_at"])
def test_next_problem_after_out_of_memory(fake, what):
    """An allocation that failed and was reported is not reported again by the
    error checks of the next problem."""
    _run(fake, f"""
p = CubeProblem(8, 3)  # 27 subdomains: several batches
subs = list(p.subdomains())
b = start()
fake.{what}(0)
try:
    b.upload_subdomain_data(subs[0])
    assert False, "taken without memory"
except RuntimeError as e:
    assert "Malloc" in str(e), e
b.finalize()
b = start()
for d in subs:
    b.upload_subdomain_data(d)
b.finalize()
""")
