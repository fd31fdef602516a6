"""What a box holds of the device and how it fails, on the CPU: the library on a
stand-in for the HIP runtime (fake_hip.c) that counts memory, streams and events
and runs no kernel.  Each check in a process of its own."""
import os
import pathlib
import subprocess
import sys

import pytest

HERE = pathlib.Path(__file__).resolve().parent

PRELUDE = """
import ctypes, sys
import numpy as np
fake = ctypes.CDLL({fake!r}, mode=ctypes.RTLD_GLOBAL)
fake.fake_device_bytes.restype = ctypes.c_size_t
sys.path.insert(0, {root!r})
import mcac_amd as m

def state(n):
    pos = np.random.default_rng(1).uniform(0, 1e-6, (n, 3))
    one = np.ones(n)
    return (dict(x=pos[:, 0], y=pos[:, 1], z=pos[:, 2], r=1e-8 * one, vol=4.2e-24 * one, surf=1.3e-15 * one, rx=0 * one,
                 ry=0 * one, rz=0 * one),
            dict(pos=pos, rcm=np.zeros((n, 3)), rmax=1e-8 * one, volume=4.2e-24 * one, surface=1.3e-15 * one,
                 count=np.ones(n, np.int64), members=np.arange(n)))
"""


@pytest.fixture(scope="module")
def run(tmp_path_factory):
    lib = tmp_path_factory.mktemp("fake") / "libfakehip.so"
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-o", str(lib), str(HERE / "fake_hip.c")], check=True)
    prelude = PRELUDE.format(fake=str(lib), root=str(HERE.parent))

    def go(code):
        env = {k: v for k, v in os.environ.items() if k != "MCAC_VERIFY_CELLS"}  # no cell list is built
        r = subprocess.run([sys.executable, "-c", prelude + code], capture_output=True, text=True, timeout=120, env=env)
        assert r.returncode == 0, r.stdout + r.stderr

    return go


@pytest.mark.parametrize("n,volsurf", [(1, 0), (64, 1), (5000, 2)])
def test_a_box_takes_what_the_estimate_says(run, n, volsurf):
    run(f"""
box = m.Box(1e-6, 4, {n}, {n}, volsurf={volsurf})
p = np.zeros(1, m.Box.PARAMS)
p["box_length"], p["n_div"], p["max_spheres"], p["max_aggregates"], p["volsurf"] = 1e-6, 4, {n}, {n}, {volsurf}
more = fake.fake_device_bytes() - m.load_gpu().mcac_box_device_bytes(p.ctypes.data)
assert 0 <= more <= 256 * 100, more  # some 80 buffers, each rounded up to 256 bytes
box.close()
assert fake.fake_device_bytes() == 0
""")


def test_a_compaction_gives_the_old_member_pool_back(run):
    run("""
n, pool = 64, 66
box = m.Box(1e-6, 4, n, n, member_pool=pool)
box.upload(*state(n))
before = fake.fake_device_bytes()
c = np.zeros(1, m.CONTACT_DTYPE)[0]
c["other_sphere"], c["other_agg"], c["contact"] = 1, 1, 1
try:  # the pair's segment of 4 is past the pool, four entries for each monomer past twice the pool
    box.merge(c)
    raise SystemExit("a merge without a kernel")
except m.MCACError:
    pass
assert box.stats()["pool_compactions"] == 1, box.stats()
assert fake.fake_device_bytes() - before == 4 * (4 * pool - pool), (fake.fake_device_bytes(), before)
box.close()
assert fake.fake_device_bytes() == 0
""")


def test_a_stream_that_cannot_be_made_fails_the_creation(run):
    run("""
fake.fake_fail_streams(1)
try:
    m.Box(1e-6, 4, 8, 8)
    raise SystemExit("created without a stream")
except m.MCACError as e:
    assert "status 32" in str(e)
assert fake.fake_device_bytes() == 0 and fake.fake_streams() == 0
fake.fake_fail_streams(0)
box = m.Box(1e-6, 4, 8, 8)
assert fake.fake_streams() == 1
L, group = m.load_gpu(), ctypes.c_void_p()
assert L.mcac_group_create(0, 2, ctypes.byref(group)) == 0 and fake.fake_streams() == 2
assert L.mcac_group_add(group, box.h) == 0 and fake.fake_streams() == 1
box.close()
assert fake.fake_streams() == 1
L.mcac_group_destroy(group)
assert fake.fake_streams() == 0
""")


def test_timing_events_belong_to_the_box_device(run):
    run("""
far = m.Box(1e-6, 4, 8, 8, device=1)
near = m.Box(1e-6, 4, 8, 8, device=0)
before = [fake.fake_events(d) for d in range(2)]
far.set_timing(1)
assert fake.fake_events(0) == before[0] and fake.fake_events(1) > before[1]
""")
