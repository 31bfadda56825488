"""The library's host side on a HIP runtime of the host alone (hip_stub.hip):
what is launched and uploaded, no numbers. Each case runs in a process of its
own, where the stub's symbols come before the HIP runtime's."""
import os
import shutil
import subprocess
import sys
import textwrap

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = os.environ.get("HIPCC") or shutil.which("hipcc") or "/opt/rocm/bin/hipcc"

PREAMBLE = """
import ctypes as C, os, sys
import numpy as np
stub = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
stub.stub_listed.restype = C.c_char_p
for f in ("u", "out", "u2", "out2"):
    getattr(stub, "stub_" + f).restype = C.c_void_p
import profess_amd as pa
from profess_amd import calpot
L = pa.lib()

def system(grid, spin=False, **kw):
    s = pa.OFDSystem(np.diag(0.4 * np.array(grid)), grid, 21.0, **kw)
    if spin:
        s.set_spin(2)
    if kw.get("kinetic") == 5:
        s.set_wgc_table(*[np.linspace(0.01, 5.0, 50)] * 4)
    return s

def enqueue(s, rho, pot):   # device addresses: no kernel runs that would read them
    return L.ofd_calpot_enqueue(s._h, C.c_void_p(rho), 1, C.c_void_p(pot), None)

def passes(s):   # "family kernel" of each launch of one evaluation
    import re
    stub.stub_clear()
    assert enqueue(s, 4096, 8192) == 0
    return [" ".join(m) for m in re.findall(r"_ZN3ofd(?:\\d(fast|gen|yz))?\\d+(\\w+?)(?:I|E)", stub.stub_listed().decode())]

FAMILY = {"yz k_rows_fwd": "three", "fast k_plane_fwd": "plane", "gen k_rows_fwd": "general"}
OPTS = {"wt4": dict(alpha=0.9, beta=0.7), "spin4": dict(alpha=0.9, beta=0.7), "wgc": dict(kinetic=5)}

def family_of(s):   # the passes that an FP64 evaluation takes
    return next((FAMILY[x] for x in passes(s) if x in FAMILY), "staged")

def family(grid, kind):
    return family_of(system(grid, spin=kind.startswith("spin"), **OPTS.get(kind, {})))

def device(s, rho, pot):   # the synchronous call; nothing writes the sums, so it ends by its 50 ms
    return L.ofd_calpot_device(s._h, C.c_void_p(rho), 1, C.c_void_p(pot), None)
"""


@pytest.fixture(scope="module")
def run(tmp_path_factory):
    if not os.path.exists(os.path.join(ROOT, "profess_amd", "libprofess_amd.so")):
        pytest.skip("library not built")
    so = str(tmp_path_factory.mktemp("stub") / "hip_stub.so")
    subprocess.run([HIPCC, "-x", "hip", "--cuda-host-only", "-std=c++17", "-O1", "-fPIC", "-shared", "-o", so,
                    os.path.join(ROOT, "tests", "hip_stub.hip")], check=True)

    def go(code):
        r = subprocess.run([sys.executable, "-c", PREAMBLE + textwrap.dedent(code), so], cwd=ROOT,
                           capture_output=True, text=True, timeout=120)
        assert r.returncode == 0, r.stdout + r.stderr
        return r.stdout
    return go


@pytest.mark.parametrize("call", ["enqueue", "device"])
def test_failed_descriptor_upload_is_repeated(run, call):
    """A call whose descriptor did not reach the device fails, and the same
    call made again uploads it: the pass reads the second call's pointers."""
    run(f"""
    s = system((24, 24, 24))
    assert {call}(s, 4096, 8192) == 0 and stub.stub_u() == 4096
    stub.stub_fail(b"k_put_desc")
    assert {call}(s, 12288, 16384) != 0
    stub.stub_fail(b"")
    assert {call}(s, 12288, 16384) == 0
    assert (stub.stub_u(), stub.stub_out()) == (12288, 16384)
    """)


def test_failed_batch_upload_is_repeated(run):
    """As above for the descriptors of a batched call, which are copied."""
    run("""
    s = [system((24, 24, 24)) for _ in range(2)]
    def many(rho, pot):
        return calpot.CalculatePotentialPlusMany(s, [rho, rho + 4096], [pot, pot + 4096], eTable=False)
    many(4096, 65536)
    assert stub.stub_u() == 4096
    stub.stub_fail(b"hipMemcpyAsync")
    try:
        many(16384, 131072)
        assert False
    except calpot.OFDError:
        pass
    stub.stub_fail(b"")
    many(16384, 131072)
    assert (stub.stub_u(), stub.stub_out()) == (16384, 131072)
    """)


@pytest.mark.parametrize("call", ["enqueue", "device"])
def test_new_arguments_are_refused_under_capture(run, call):
    """A call that needs its descriptor uploaded is refused while the stream is
    captured and launches nothing; made again afterwards it is uploaded. The
    form for captures is not refused."""
    run(f"""
    s = system((24, 24, 24))
    assert {call}(s, 4096, 8192) == 0
    stub.stub_capture(1)
    stub.stub_clear()
    assert {call}(s, 12288, 16384) != 0 and stub.stub_listed() == b""
    assert L.ofd_calpot_noalloc(s._h, C.c_void_p(4096), 1, C.c_void_p(8192), None) == 0
    stub.stub_capture(0)
    assert {call}(s, 12288, 16384) == 0
    assert (stub.stub_u(), stub.stub_out()) == (12288, 16384)
    """)


@pytest.mark.parametrize("grid,kinetic", [((128, 128, 192), 4), ((128, 128, 24), 5)])
@pytest.mark.parametrize("lds", [65536, 131072, 163840])
def test_plane_passes_only_where_the_plane_fits(run, grid, kinetic, lds):
    """Every evaluation starts with a forward pass over x, also where a
    workgroup has less LDS than the 128 x 128 plane (157 KB whole) takes."""
    run(f"""
    stub.stub_lds({lds})
    p = passes(system({grid}, kinetic={kinetic}))
    assert p[0] == ("fast k_plane_fwd" if {lds} == 163840 else "gen k_rows_fwd"), p
    """)


def test_shapes_reach_the_passes_they_test(run):
    """The shapes of the tests of one family of FP64 passes against another
    take that family, so that no change of the dispatch empties a test."""
    run("""
    from tests import test_gpu_lengths as lengths, test_gpu_plane_fp64 as plane, test_gpu_three_pass as three
    from tests import test_gpu_forms as forms
    want = [(g, k, "plane") for g, k in plane.CASES]
    want += [(g, k, "general") for g in lengths.GRIDS for k in ("wt", "wt4", "spin", "wgc")
             if g != (100, 75, 81) or k == "wgc"]
    want += [(g, k, "three") for g in three.GRIDS for k in ("wt", "wt4", "spin") if (g, k) != ((162, 63, 27), "spin")]
    want += forms.CASES
    got = [(g, k, family(g, k)) for g, k, _ in want]
    assert got == want, [(a, b[2]) for a, b in zip(got, want) if a != b]
    """)


def test_descriptor_layout_of_the_form_tests(run):
    """The descriptor that the tests of single forms fill is the library's."""
    run("""
    from tests.eval_forms import PLAN_BYTES, ReqDesc
    stub.stub_desc.restype = C.POINTER(ReqDesc)
    assert C.sizeof(ReqDesc) == stub.stub_sizes(0) and PLAN_BYTES >= stub.stub_sizes(1)
    s = system((24, 24, 24), spin=True, alpha=0.9, beta=0.7)
    assert enqueue(s, 4096, 8192) == 0
    D = stub.stub_desc().contents
    n = 8 * 24 ** 3
    assert (D.u, D.out, D.u2, D.out2) == (4096, 8192, 4096 + n, 8192 + n)
    assert (D.alpha, D.beta, D.opt_sqrt, D.lsda, D.pad, D.newton_ch, D.cb2, D.hfin) == (0.9, 0.7, 1, 1, 0, 0, 0.0, None)
    assert abs(D.rb[0] - 2 * np.pi / 9.6) < 1e-12 and D.wtk and D.fin and D.work and D.sums and D.vion
    """)


def test_autotune_evaluates_both_channels(run):
    """The evaluations that the tuner times have the arrays of both channels."""
    run("""
    from tests.eval_forms import ReqDesc
    stub.stub_desc.restype = C.POINTER(ReqDesc)
    s = system((24, 24, 24), spin=True)
    s.autotune(reps=1)
    D = stub.stub_desc().contents
    n = 24 ** 3
    assert (D.u2, D.out2) == (D.u + 8 * n, D.out + 8 * n)
    rho = np.ctypeslib.as_array(C.cast(D.u, C.POINTER(C.c_double)), (2 * n,))
    assert np.all(np.abs(rho * 2 * s.vol / 21.0 - 1.0) < 1e-12)
    """)


@pytest.mark.parametrize("grid,kind", [((64, 64, 256), "spin"), ((64, 64, 256), "wt"), ((32, 32, 24), "wgc"),
                                       ((200, 27, 20), "wt"), ((24, 24, 24), "wt"), ((16, 16, 16), "wt")])
def test_tuning_keeps_the_passes(run, grid, kind):
    """A tuned system takes the passes it took before, also with one channel
    again after two, and so does the next system of its shape: another family
    would change a result's last bits."""
    run(f"""
    grid, kind = {grid}, "{kind}"
    one = family(grid, kind.replace("spin", "wt"))
    before = family(grid, kind)
    s = system(grid, spin=kind == "spin", **OPTS.get(kind, {{}}))
    s.autotune(reps=1)
    assert family_of(s) == before
    if kind == "spin":
        s.set_spin(1)
        assert family_of(s) == one, family_of(s)
    assert family(grid, kind) == before and family(grid, kind.replace("spin", "wt")) == one
    """)


@pytest.mark.parametrize("grid,kw", [((128, 128, 128), {}), ((128, 128, 192), {}), ((128, 128, 128), dict(precision=1)),
                                     ((120, 120, 120), dict(precision=1)), ((200, 27, 20), {}), ((16, 16, 16), {})])
def test_tuner_reports_the_plane_pass(run, grid, kw):
    run(f"""
    s = system({grid}, **{kw})
    p = passes(s)
    assert s.autotune(reps=1)["plane"] == int("fast k_plane_fwd" in p), p
    """)


def test_tiles_of_one_precision_stay_with_it(run):
    """A mixed-precision system tuned at a length where FP32 takes the staged
    passes: their z tile of one column is not the three-pass z tile of the
    solve's FP64 evaluations."""
    run("""
    def fp64_tile(s):
        try:
            pa.ProjNormRhoMinimization(s, np.full(s.shape, 21.0 / s.vol), max_iter=1, max_line=1)
        except calpot.OFDError:
            pass   # no kernel runs
        return stub.stub_grid(b"k_yz")
    grid = (72, 72, 72)
    before = fp64_tile(system(grid, precision=1))
    stub.stub_fastest(2)
    s = system(grid, precision=1)
    r = s.autotune(reps=1)
    assert before > 0 and (r["kb_z"], r["kb_y"]) == (1, 0), (before, r)
    assert fp64_tile(s) == before and fp64_tile(system(grid, precision=1)) == before
    t = system(grid)   # tuned in FP64: that tile, also in the FP64 evaluations of a mixed solve
    stub.stub_fastest(2)
    assert t.autotune(reps=1)["kb_z"] == 1 and fp64_tile(system(grid, precision=1)) > before
    """)


def test_polled_slots_are_coherent_and_portable(run):
    """The host polls a slot while the kernel that stores into it runs, and the
    slots serve the contexts of every device."""
    run("""
    s = system((24, 24, 24))
    portable, coherent = 0x1, 0x40000000
    assert stub.stub_host_flags() & (portable | coherent) == portable | coherent
    """)
