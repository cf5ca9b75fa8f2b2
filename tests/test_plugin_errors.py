"""The plugin's host code after a failed launch or allocation, on the CPU: its sources compiled for the
host alone run on a stand-in HIP runtime (tests/fake_hip/fake_hip.cpp) whose launches and allocations can
be made to fail and whose stream can be watched. What a failed call leaves must not reach the next one.
"""
import ctypes as C
import os
import shutil
import subprocess

import pytest

import prender_amd as pa

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
SRC = os.path.join(ROOT, "ar-renderer_amd", "csrc", "plugin")
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"

pytestmark = pytest.mark.skipif(not os.path.exists(HIPCC), reason="needs hipcc")


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    out = tmp_path_factory.mktemp("fake_hip")
    inc = ["-I" + os.path.join(ROOT, "include"), "-I" + SRC, "-I/opt/rocm/include"]
    jobs, objs = [], []
    for name in ("api.hip", "pt.hip", "v4.hip", "guide.hip"):
        objs.append(str(out / (name + ".o")))
        jobs.append([HIPCC, "-x", "hip", "--offload-host-only", "--offload-arch=gfx950", "-fuse-cuid=none", "-std=c++17",
                     "-O1", "-fPIC", "-ffp-contract=off", "-w", *inc, "-c", os.path.join(SRC, name), "-o", objs[-1]])
    for path in (os.path.join(SRC, "wbvh_build.cpp"), os.path.join(SRC, "sheen_table.cpp"),
                 os.path.join(HERE, "fake_hip", "fake_hip.cpp")):
        objs.append(str(out / (os.path.basename(path) + ".o")))
        jobs.append(["g++", "-std=c++17", "-O1", "-fPIC", "-w", "-D__HIP_PLATFORM_AMD__", *inc, "-c", path, "-o", objs[-1]])
    for p in [subprocess.Popen(j) for j in jobs]:
        assert p.wait() == 0
    so = str(out / "libplugin_on_fake_hip.so")
    subprocess.run(["g++", "-shared", "-Wl,-Bsymbolic", "-Wl,--allow-multiple-definition", *objs, "-o", so, "-lpthread"], check=True)
    return so


@pytest.fixture(scope="module")
def fake(lib):
    p = pa.Plugin(lib)
    f = p.lib
    for name in ("fake_pending", "fake_live", "fake_mallocs", "fake_launches", "fake_null_counters"):
        getattr(f, name).restype = C.c_long
    f.fake_fail_malloc.argtypes = [C.c_long]
    f.fake_fail_launch.argtypes = [C.c_char_p, C.c_long]
    assert len(p.devices()) == 1
    return p


@pytest.fixture
def plugin(fake):
    fake.lib.fake_rounds(3)
    fake.lib.fake_lazy(0)
    yield fake
    fake.lib.fake_lazy(0)
    fake.lib.fake_fail_malloc(0)
    fake.lib.fake_fail_launch(b"", 0)
    fake.profile(0)
    fake.release()


def params(**k):
    return pa.render_params(spp=1, first_sample=0, seed=1, max_depth=8, rr_start=3, **k)


def test_failed_round_leaves_nothing_queued(plugin, host):
    # The bounce loop queues a round ahead of the path count it waits for. When a launch of that round fails,
    # its traversal is queued and will publish a count, in the word and under the tag that the next call waits for.
    s = host.generate(1, 16, 16, 0.25)
    plugin.render_ex(s, params())
    plugin.lib.fake_lazy(1)
    plugin.lib.fake_fail_launch(b"k_surface", 2)
    with pytest.raises(RuntimeError):
        plugin.render_ex(s, params())
    assert plugin.lib.fake_pending() == 0


def grow_and_fail(plugin, small, large, call):
    """call(small), then call(large) with its k-th allocation failing, for every k; yields after each failure."""
    call(small)
    k = 0
    while True:
        k += 1
        before = plugin.lib.fake_mallocs()
        plugin.lib.fake_fail_malloc(k)
        try:
            call(large)
        except RuntimeError:
            assert plugin.lib.fake_mallocs() - before == k
            yield k
            continue
        plugin.lib.fake_fail_malloc(0)
        return


@pytest.mark.parametrize("flags", [0, pa.RENDER_GUIDE | pa.RENDER_GUIDE_TRAIN], ids=["plain", "guided"])
def test_failed_growth_leaves_no_missing_buffer(plugin, host, flags):
    # The batch's buffers are sized by the largest batch so far. A growth that fails half way has freed some of
    # them: a smaller batch must not run on what is left.
    s = host.generate(1, 16, 16, 0.25)

    def call(spp):
        plugin.render_ex(s, pa.render_params(spp=spp, first_sample=0, seed=1, max_depth=8, rr_start=3, flags=flags))

    call(1)
    whole = plugin.lib.fake_live()
    plugin.release()
    failures = 0
    for _ in grow_and_fail(plugin, 1, 4, call):
        failures += 1
        call(1)
        assert plugin.lib.fake_live() == whole
        plugin.release()
        call(1)
    assert failures > 15
    assert plugin.lib.fake_live() == whole


def test_failed_growth_of_the_training_ring(plugin, host):
    s = host.generate(1, 16, 16, 0.25)
    flags = pa.RENDER_GUIDE | pa.RENDER_GUIDE_TRAIN

    def call(replay):
        plugin.tune_set("guide_replay", replay)
        plugin.render_ex(s, params(flags=flags))

    try:
        plugin.tune_set("guide_batch", 256)
        call(1 << 12)
        whole = plugin.lib.fake_live()
        plugin.lib.fake_fail_malloc(1)  # the ring is all that grows
        with pytest.raises(RuntimeError):
            call(1 << 13)
        call(1 << 12)
        assert plugin.lib.fake_live() == whole
    finally:
        plugin.tune_set("guide_batch", 1 << 18)
        plugin.tune_set("guide_replay", 1 << 20)


@pytest.mark.parametrize("k", [1, 2])
def test_failed_film_reset_leaves_no_film(plugin, host, k):
    s = host.generate(1, 16, 16, 0.25)
    plugin.film_reset(16, 16)
    plugin.render_resident(s, params())
    plugin.lib.fake_fail_malloc(k)
    with pytest.raises(RuntimeError):
        plugin.film_reset(32, 32)
    with pytest.raises(RuntimeError, match="not reset"):
        plugin.render_resident(s, params())
    with pytest.raises(RuntimeError):
        plugin.film_read(16, 16)


def test_failed_model_setup_leaves_no_model(plugin):
    plugin.guide_params()
    whole = plugin.lib.fake_live()
    plugin.release()
    k = 0
    while True:
        k += 1
        plugin.lib.fake_fail_malloc(k)
        try:
            plugin.guide_params()
        except RuntimeError:
            plugin.lib.fake_fail_malloc(0)
            plugin.guide_params()
            assert plugin.lib.fake_live() == whole
            plugin.release()
            continue
        break
    assert k > 5


def test_failed_device_setup_is_done_again(lib, tmp_path, host):
    # (a copy of the library has a state of its own: no call has set its device up)
    fresh = pa.Plugin(shutil.copy(lib, tmp_path / "fresh.so"))
    fresh.lib.fake_fail_malloc.argtypes = [C.c_long]
    fresh.devices()
    s = host.generate(1, 16, 16, 0.25)
    fresh.lib.fake_fail_malloc(1)  # the flags that every traversal reports to
    with pytest.raises(RuntimeError):
        fresh.render_ex(s, params())
    fresh.render_ex(s, params())


def test_counting_traversal_without_counters(plugin, host):
    # prgpu_release frees the counters of profile mode 2, which stays on; and they may not be allocated.
    s = host.generate(1, 16, 16, 0.25)
    plugin.profile(2)
    plugin.render_ex(s, params())
    plugin.release()
    plugin.render_ex(s, params())
    plugin.profile(0)
    plugin.lib.fake_fail_malloc(1)
    with pytest.raises(RuntimeError):
        plugin.profile(2)
    plugin.render_ex(s, params())
    assert plugin.lib.fake_null_counters() == 0
