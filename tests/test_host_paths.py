"""The library's host side without a GPU: workspace sizes after failed allocations
and the order of launches, with tests/native/host_hip.cpp in the place of the HIP
runtime.  Kernels do nothing there but what the host reads back."""
import os
import shutil
import subprocess
import sys

import pytest

from prender_amd import prt

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PRELUDE = """
import ctypes as C, sys
sys.modules["torch"] = None  # it would bring the real runtime
host = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
host.hh_fail_above.argtypes = [C.c_size_t]
from prender_amd import generators as G, prt

def script(*children):
    host.hh_script((C.c_uint32 * len(children))(*children), len(children))

def launched():
    out = C.create_string_buffer(1 << 20)
    host.hh_launched(out, len(out))
    return out.value.decode().split()

def no_faults():
    out = C.create_string_buffer(1 << 16)
    assert host.hh_faults(out, len(out)) == 0, out.value.decode()
"""


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("needs the HIP headers and compiler")
    if not os.path.exists(prt.LIB_PATH):
        pytest.skip("libprt.so is not built (python -m prender_amd.build)")
    d = tmp_path_factory.mktemp("host_hip")
    obj, lib = str(d / "host_hip.o"), str(d / "libhost_hip.so")
    subprocess.run([hipcc, "-x", "hip", "--offload-host-only", "--offload-arch=gfx950", "-O1", "-std=c++17", "-fPIC",
                    "-I", os.path.join(ROOT, "prender_amd", "csrc"), "-c",
                    os.path.join(ROOT, "tests", "native", "host_hip.cpp"), "-o", obj], check=True)
    subprocess.run(["g++", "-shared", "-o", lib, obj], check=True)

    def run(body):
        r = subprocess.run([sys.executable, "-c", PRELUDE + body, lib], cwd=ROOT, stdout=subprocess.PIPE,
                           stderr=subprocess.STDOUT, text=True, timeout=300)
        assert r.returncode == 0, r.stdout[-3000:]
        return r.stdout

    return run


# A frame of the path kernel whose accumulators cannot be allocated has released
# the ones that the queued renders had: the next render allocates its own.
@pytest.mark.parametrize("after", ["box.render(engine=1)", "box.render(engine=1, samples=2)",
                                   "box.render_mlt(chains=64, mutations_per_chain=2)"])
def test_render_after_a_failed_allocation(host, after):
    host(f"""
box = prt.Scene(G.config2(width=32, height=24, samples=2, level=2))
big = prt.Scene(G.cornell_spheres(width=1024, height=1024, samples=1))
{after}
host.hh_fail_above(90 << 20)  # the big frame's 96 MiB of accumulators are not to be had
try:
    big.render()
    raise SystemExit("the allocation did not fail")
except prt.PrtError as e:
    assert "(-3)" in str(e), e
{after}
no_faults()
host.hh_fail_above(1 << 40)
big.render()
{after}
no_faults()
""")


# Two launches of any-hit rays share one stack area, so one must end before the
# other begins: also where the path kernel takes a batch's last rays while the
# shadow rays of the depth before are on the second stream.  script: rays that the
# shading of each depth leaves; the host looks at the first and every fourth.
@pytest.mark.parametrize("children,tail", [((200000, 200000, 200000, 200000, 1000), True), ((60000,), True),
                                           ((200000, 200000, 100, 0), False), ((0,), False)])
def test_shadow_launches_are_ordered(host, children, tail):
    host(f"""
box = prt.Scene(G.config2(width=400, height=400, samples=1, level=2))
script{tuple(children)!r}
_, _, st = box.render(variance=False)
assert any("k_pathILi2E" in k for k in launched()) == {tail}
assert st["extension_rays"] == {sum(children)} and st["shadow_rays"] == {3 * sum(children)}, st
no_faults()
""")


# the same over an adjoint's recording pass and its replay, and a batch
def test_other_overlapping_launches_are_ordered(host):
    host("""
d = G.config5(width=64, height=48, samples=2)
s = prt.Scene(d)
dimg, grad = C.c_void_p(), C.c_void_p()
host.hipMalloc(C.byref(dimg), C.c_size_t(64 * 48 * 12))
host.hipMalloc(C.byref(grad), C.c_size_t(d.entities[1].indices.shape[0] * 12))
script(*[3000] * 6)
s.adjoint_device(dimg.value, 1, grad.value, 2)
out = C.c_void_p()
host.hipMalloc(C.byref(out), C.c_size_t(64 * 48 * 12))
prt.render_batch_device([s], [out.value], None, prt.batch_opts())
names = launched()
assert sum("k_shadow" in k for k in names) >= 6 and any("k_stream_shadow" in k for k in names)
no_faults()
""")


# A render whose path kernel loses a sample fails its own check, as the batched
# form's does.
@pytest.mark.parametrize("call", ["box.render()", "spheres.render()", "box.render_mlt(chains=64, mutations_per_chain=3)",
                                  "box.render_erpt(mutation=2.0)",
                                  "prt.render_batch_device([spheres], [out.value], None, prt.batch_opts(persistent=1))"])
def test_a_lost_sample_is_an_error(host, call):
    host(f"""
box = prt.Scene(G.config2(width=32, height=24, samples=2, level=2))
spheres = prt.Scene(G.cornell_spheres(width=32, height=24, samples=2))
out = C.c_void_p()
host.hipMalloc(C.byref(out), C.c_size_t(32 * 24 * 12))
{call}
host.hh_lose(1)
try:
    {call}
    raise SystemExit("the lost sample went unnoticed")
except prt.PrtError as e:
    assert "(-6)" in str(e), e
no_faults()
""")


# What a sample costs differs over an image, so every wave of a path launch has
# many claims to take, or claims single chunks.
@pytest.mark.parametrize("nee", [0, 1])
def test_path_claims_leave_work_to_share(host, nee):
    host(f"""
for height in (1023, 1024, 1025, 2048, 4096):
    s = prt.Scene(G.cornell_spheres(width=1024, height=height, samples=2, supersamples=1, nee={nee}))
    s.render(engine=3, variance=False)
    got = (C.c_uint32 * 3)()
    host.hh_path(got)
    chunks, claim, waves = got
    assert chunks >= 1024 * height * 2 // 64 and waves >= 2048
    assert claim == 1 or chunks >= 64 * claim * waves, (height, chunks, claim, waves)
    s.close()
no_faults()
""")


# Records that cannot be allocated: the batch is replayed, its samples' radiance
# being known; nothing else of the call depends on them.
@pytest.mark.parametrize("limit,replayed", [(1 << 40, False), (3 << 20, True)])
def test_adjoint_without_memory_for_records(host, limit, replayed):
    host(f"""
d = G.config5(width=64, height=48, samples=8)
s = prt.Scene(d)
dimg, grad = C.c_void_p(), C.c_void_p()
host.hipMalloc(C.byref(dimg), C.c_size_t(64 * 48 * 12))
host.hipMalloc(C.byref(grad), C.c_size_t(d.entities[1].indices.shape[0] * 12))
script(*[2000] * 4)
s.adjoint_device(dimg.value, 1, None, 2)
host.hh_fail_above({limit})
launched()
script(*[2000] * 4, 0, *[2000] * 4)
_, st = s.adjoint_device(dimg.value, 1, grad.value, 2)
names = launched()
assert any("k_shadeILi2E" in k for k in names)
assert any("k_shadeILi1E" in k for k in names) == {replayed}
assert any("k_adjoint_resolve" in k for k in names) != {replayed}
assert st["primary_rays"] == 64 * 48 * 4 * {2 if replayed else 1}
no_faults()
""")


# The tuner times each form once per instance of the path kernel that there is
# (light sampling: two waves per SIMD; without: two and three), and reports one of
# them.  Every measured span here is shorter than the last, so the last trial wins.
@pytest.mark.parametrize("nees,instances,form,waves", [((0, 1), 3, 2, 3), ((1, 1), 1, 1, 2), ((0, 0), 2, 1, 3)])
def test_tuner_times_each_instance_once(host, nees, instances, form, waves):
    host(f"""
scenes = [prt.Scene(G.cornell_spheres(width=32 + 8 * i, height=24, samples=2, nee=n)) for i, n in enumerate({nees!r})]
outs = []
for s in scenes:
    p = C.c_void_p()
    host.hipMalloc(C.byref(p), C.c_size_t(s.width * s.height * 12))
    outs.append(p.value)
best, _ = prt.tune_batch(scenes, outs)
tried = [k for k in launched() if "k_pathILi0E" in k]
assert len(tried) == len(set(tried)) == {instances}, tried
assert best.persistent == {form}
assert (best.persist_waves or best.trav_blocks_per_cu) == {waves}, (best.persist_waves, best.trav_blocks_per_cu)
prt.render_batch_device(scenes, outs, None, best)
ran = [k for k in launched() if "k_pathILi0E" in k]
assert len(ran) == 1 and ran[0] == tried[-1] and ran[0].endswith("Li{waves}EEv7Persist6Params"), ran
no_faults()
""")


# The more analytic entities there are beside a block's LDS copy, the smaller the
# frames that the path kernel takes; the others go to the engine for their scene.
@pytest.mark.parametrize("entities,glass,samples,path", [
    (16, 1, 1 << 21, True), (17, 1, 1 << 21, True), (117, 1, 300000, True), (117, 1, 360000, False),
    (1016, 1, 33000, True), (1016, 1, 34000, False), (16, 0, 3 << 17, True), (80, 0, 3 << 17, True),
    (416, 0, 83000, True), (416, 0, 85000, False)])
def test_path_frames_by_entities(host, entities, glass, samples, path):
    host(f"""
d = G.cornell_spheres(width={samples} // 8, height=8, samples=1, supersamples=1, nee=1)
if not {glass}:
    for m in d.materials:
        m.reflection = "diffuse"
while len(d.entities) < {entities}:
    d.entities.append(G.Sphere((50.0, 40.0, 60.0 + 0.01 * len(d.entities)), 1.0, 2))
prt.Scene(d).render(variance=False)
names = launched()
assert any("k_path" in k for k in names) == {path}, names
assert any("k_stream" in k for k in names) == {bool(glass and not path)}
assert any("k_extend" in k for k in names) == {not glass and not path}
no_faults()
""")


# Without memory for queues those frames take the path kernel after all, as they did
# before the limit depended on the entities; frames above its own limits fail.
@pytest.mark.parametrize("glass,samples,ok", [(1, 1 << 20, True), (1, 3 << 20, False), (0, 3 << 17, True),
                                              (0, 1 << 19, False)])
def test_path_frames_without_memory_for_queues(host, glass, samples, ok):
    host(f"""
d = G.cornell_spheres(width={samples} // 8, height=8, samples=1, supersamples=1, nee=1)
if not {glass}:
    for m in d.materials:
        m.reflection = "diffuse"
while len(d.entities) < 1016:
    d.entities.append(G.Sphere((50.0, 40.0, 60.0 + 0.01 * len(d.entities)), 1.0, 2))
s = prt.Scene(d)
host.hh_fail_above({80 if glass else 25} << 20)
try:
    s.render(variance=False)
    assert {ok} and any("k_path" in k for k in launched())
except prt.PrtError as e:
    assert not {ok} and "(-3)" in str(e), e
no_faults()
""")
