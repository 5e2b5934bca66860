"""Renders and loads when device memory is short, without a GPU: the library runs in a child process over
tests/fake_hip.cpp, a HIP runtime of limited memory that lists the launched kernels instead of running
them.

A megakernel render above 2^22 samples runs as queues, which take 249 bytes of path state a sample on
top of the radiance (12 bytes) and the film. The state is at most that of an automatic pass (2^28 / 12
samples); where it finds no memory the pass runs as whole paths, and a context gives its state back when
something else needs the memory. No render fails that whole paths have memory for.
"""
import ctypes as C
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
sys.path[:0] = [os.path.dirname(HERE)]  # the child process has no conftest

from lighttransportsimulation_amd import Context, LtsError, scenegen

W, H, SPP = 1536, 1024, 4   # 6.3M samples: above 2^22
SAMPLES = W * H * SPP
RADIANCE, FILM = 12 * SAMPLES, 28 * W * H
STATE_BYTES = 249            # of a path
STATE = STATE_BYTES * SAMPLES
SLACK = 1 << 20              # scene records, counters


# ------------------------------------------------------------------------------ in the child process
class Child:
    def __init__(self, folder):
        self.fake = C.CDLL(None)  # the preloaded runtime
        self.fake.fake_hip_used.restype = self.fake.fake_hip_peak.restype = C.c_size_t
        self.fake.fake_hip_limit.argtypes = [C.c_size_t]
        self.fake.fake_hip_fail.argtypes = [C.c_char_p, C.c_int]
        self.fake.fake_hip_launched.restype = C.c_char_p
        scenegen.write_bin(os.path.join(folder, "tri"), [[0, 0, 0], [1, 0, 0], [0, 1, 0]], [[0, 1, 2]])
        st = scenegen.SceneText(camera=(0, 0, -4, 0, 0, 0, 0, 1, 0, 40, 4))
        st.meshes, st.mats, st.infinite = ["tri"], [scenegen.mat_matte((0.5, 0.5, 0.5))], (1, 1, 1)
        st.write(folder, "one")
        self.folder, self.ctx = folder, Context(0)

    def load(self, w=W, h=H):
        self.ctx.load_scene(self.folder, "one", None, w, h)

    def room(self, nbytes):
        """Leaves this much memory free."""
        self.fake.fake_hip_limit(self.fake.fake_hip_used() + nbytes)

    def forms(self):
        """How the passes since the last call ran."""
        names = self.fake.fake_hip_launched().decode()
        return ("paths" if "k_paths" in names else "") + ("queues" if "k_wf_trace" in names or "graph" in names else "")

    def render(self, spp=SPP, **kw):
        self.forms()
        out = self.ctx.render(spp, 3, 2, 1, integrator=0, **kw)
        return self.forms(), out[2]


def path_state_does_not_fit(c):
    c.load()
    c.room(RADIANCE + FILM + STATE // 2)
    assert c.render()[0] == "paths"
    assert c.fake.fake_hip_used() <= c.fake.fake_hip_peak() and c.render()[0] == "paths"
    c.room(STATE + SLACK)
    assert c.render()[0] == "queues"


def path_state_fits_and_nothing_else(c):
    # radiance and film are allocated first, so they find room wherever whole paths do
    for extra in (SLACK, RADIANCE // 2, RADIANCE + FILM - SLACK):
        with Context(0) as c.ctx:
            c.load()
            c.room(STATE + extra)
            assert c.render()[0] == "paths", extra
    with Context(0) as c.ctx:
        c.load()
        c.room(STATE + RADIANCE + FILM + SLACK)
        assert c.render()[0] == "queues"


def no_memory_for_the_graph(c):
    c.load()
    c.fake.fake_hip_fail(b"hipGraphInstantiate", 2)
    assert c.render()[0] == "queues"
    # a film that continues: no sample is gathered twice
    assert c.render(spp=8, sample_end=4)[0] == "queues"
    c.ctx.render(8, 3, 2, 1, integrator=0, sample_begin=4)
    names = c.fake.fake_hip_launched().decode()
    assert names.count("k_film_gather") == 1 and "k_wf_trace" in names and "k_paths" not in names


def an_error_of_a_started_render_is_final(c):
    c.load()
    c.fake.fake_hip_fail(b"hipGraphLaunch", 2)
    c.forms()
    with pytest.raises(LtsError, match="-5"):
        c.ctx.render(SPP, 3, 2, 1, integrator=0)
    assert "k_paths" not in c.fake.fake_hip_launched().decode()
    c.fake.fake_hip_fail(b"", 0)
    assert c.render()[0] == "queues"  # nothing of the error is left


def the_state_is_bounded(c):
    c.load()
    used = c.fake.fake_hip_used()
    c.room(1 << 40)
    form, st = c.render(spp=64, spp_per_pass=64)  # 100M samples in passes of at most 2^28 / 12
    assert form == "queues" and st["launches"] == 5
    assert c.fake.fake_hip_peak() - used <= STATE_BYTES * (1 << 28) // 12 + (1 << 28) + FILM + SLACK
    form, st = c.render(spp=16, want_samples=True)  # 25M samples returned from one pass
    assert form == "paths" and st["launches"] == 1


def the_state_is_given_back(c):
    c.load()
    assert c.render()[0] == "queues"
    held = c.fake.fake_hip_used()
    c.room(RADIANCE // 2)  # not enough for twice the samples, nor for the larger film
    c.load(2 * W, 2 * H)
    assert c.render(spp=2)[0] == "paths" and c.fake.fake_hip_used() < held
    c.room(RADIANCE + STATE + SLACK)
    c.load()
    assert c.render()[0] == "queues"
    c.room(1 << 10)
    c.load(W // 2, H // 2)  # a scene load finds the memory too
    c.ctx.trace_rays([[0, 0, -4]] * 1000, [[0, 0, 1]] * 1000)


SCENARIOS = [path_state_does_not_fit, path_state_fits_and_nothing_else, no_memory_for_the_graph,
             an_error_of_a_started_render_is_final, the_state_is_bounded, the_state_is_given_back]


# ------------------------------------------------------------------------------------------ the tests
@pytest.fixture(scope="module")
def fake_hip(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("fake_hip") / "libfake_hip.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-o", so,
                    os.path.join(HERE, "fake_hip.cpp")], check=True)
    return so


def run_in_child(fake_hip, folder, file, scenario):
    env = dict(os.environ, LD_PRELOAD=" ".join(filter(None, [fake_hip, os.environ.get("LD_PRELOAD")])))
    p = subprocess.run([sys.executable, file, str(folder), scenario], env=env, capture_output=True, text=True, timeout=300)
    assert p.returncode == 0, p.stdout + p.stderr


@pytest.mark.parametrize("scenario", [s.__name__ for s in SCENARIOS])
def test_short_memory(fake_hip, tmp_path, scenario):
    run_in_child(fake_hip, tmp_path, __file__, scenario)


if __name__ == "__main__":
    globals()[sys.argv[2]](Child(sys.argv[1]))
