"""When the segment lists of the row-by-row forward walks are built, kept and
given up: the library's host side on a HIP runtime without a GPU (fake_hip.c),
which counts device memory and logs launches.  Each script runs in a process of
its own, since the stand-in's symbols are global."""
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))

PREAMBLE = """
import ctypes, sys
sys.path.insert(0, {root!r})
H = ctypes.CDLL({shim!r}, ctypes.RTLD_GLOBAL)
H.fake_log.restype = ctypes.c_char_p
H.fake_used.restype = ctypes.c_size_t
H.fake_budget.argtypes = [ctypes.c_size_t]
import kevernals_amd as K
from kevernals_amd import geometry as G
L = K.load_library()
drop = getattr(L, "_Z22kv_internal_drop_listsP10kv_context")
batch_drop = getattr(L, "_Z28kv_internal_batch_drop_listsP8kv_batch")
GIB = 1 << 30

def arc(nz=16, nv=128, views=7):
    return G.arc_geometry((64, 64, nz), (0.5, 0.5, 2.0), (128, nv), (0.6, 0.6), views, 15.0)

def context(g):
    return K.Context(0, g, follow_torch_stream=False)

def launches(f, *args):
    H.fake_log_clear()
    st = f(*args)
    assert st == 0, (st, L.kv_last_error())
    return H.fake_log().decode().split()

def forward(c, mode):
    return launches(L.kv_forward_project, c.handle, buf, buf, mode)

def ran(names, kernel):
    return any(str(len(kernel)) + kernel in n for n in names)

buf = ctypes.c_void_p()
assert L.kv_create(0, ctypes.byref(buf)) == 0
spare = buf
buf = ctypes.c_void_p()
assert L.kv_malloc(spare, 1 << 22, ctypes.byref(buf)) == 0
A, R = K.MODE_A, K.MODE_R
"""


@pytest.fixture(scope="module")
def run(tmp_path_factory):
    shim = str(tmp_path_factory.mktemp("hip") / "libfake_hip.so")
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1", "-o", shim, os.path.join(HERE, "fake_hip.c")], check=True)
    head = PREAMBLE.format(root=os.path.dirname(HERE), shim=shim)

    def go(script):
        r = subprocess.run([sys.executable, "-c", head + script], capture_output=True, text=True, timeout=300)
        assert r.returncode == 0, r.stderr[-3000:]

    return go


def test_built_on_a_modes_first_forward_pass(run):
    """Nothing for contexts that only backproject; one mode's lists for one
    mode's passes, complete (waited for) when the call returns."""
    run("""
c = context(arc())
none = H.fake_used()
names = launches(L.kv_back_project, c.handle, buf, buf, R) + launches(L.kv_back_project, c.handle, buf, buf, A)
assert not ran(names, "seg_a_kernel") and not ran(names, "seg_r_kernel")
tables = H.fake_used()
names = forward(c, A)
built = [i for i, n in enumerate(names) if "seg_a_kernel" in n][0]
assert "sync" in names[built:] and ran(names, "fp_a_row_kernel") and not ran(names, "seg_r_kernel")
lists = H.fake_used() - tables
assert lists > 0
names = forward(c, A)
assert len(names) == 1 and ran(names, "fp_a_row_kernel")
names = forward(c, R)
assert ran(names, "seg_r_kernel") and ran(names, "fp_r_row_kernel")
assert drop(c.handle) == 0 and H.fake_used() == tables
assert ran(forward(c, A), "fp_a_kernel") and ran(forward(c, R), "fp_r_kernel")
c.set_geometry(arc())
assert H.fake_used() == none
assert ran(forward(c, A), "fp_a_row_kernel")
""")


def test_each_modes_limit_counts_its_own_entries(run):
    """Mode A's entries are half the size of mode R's: up to 1 GiB of either."""
    run("""
g = G.arc_geometry((8, 60, 400), (0.5, 0.2, 0.2), (2, 4096), (0.6, 0.02), 60, 15.0, det_shift=(0.3, 0.0))
c = context(g)
none = H.fake_used()
names = forward(c, A)
assert ran(names, "fp_a_row_kernel") and GIB // 2 < H.fake_used() - none <= GIB + (1 << 23), H.fake_used() - none
assert ran(forward(c, R), "fp_r_kernel")
""")


def test_give_way_to_memory_that_calls_need(run):
    run("""
c = context(arc())
none = H.fake_used()
launches(L.kv_back_project, c.handle, buf, buf, A)
tables = H.fake_used() - none
c.set_geometry(arc())
forward(c, A)
have = H.fake_used()
p = ctypes.c_void_p()
assert L.kv_malloc(c.handle, 1 << 40, ctypes.byref(p)) == 3 and not p.value  # of no use here
assert H.fake_used() == have
H.fake_budget(have + tables - (have - none) // 2)  # enough without the lists
names = launches(L.kv_back_project, c.handle, buf, buf, A)
assert ran(names, "tables_a_kernel")
assert ran(forward(c, A), "fp_a_kernel")
assert L.kv_malloc(c.handle, 1 << 40, ctypes.byref(p)) == 3 and not p.value
assert launches(L.kv_memset, c.handle, buf, 0, 16) == []  # no error left behind
assert ran(forward(c, A), "fp_a_kernel")
""")


def test_not_taken_where_memory_is_short(run):
    """1 GiB is left free."""
    run("""
c = context(arc())
H.fake_budget(H.fake_used() + GIB)
have = H.fake_used()
assert ran(forward(c, A), "fp_a_kernel") and H.fake_used() == have
""")


@pytest.mark.parametrize("mode", ["R", "A"])
def test_batches_take_them_last(run, mode):
    """A batch that fits without lists can be made."""
    run("""
gs = [arc(16), arc(20, 100), arc(11, 64, 5)]
mode = %s
b = K.Batch(gs, mode=mode)
full = H.fake_used()
names = launches(L.kv_batch_mlem, b.handle, (ctypes.c_int32 * 3)(1, 1, 1), ctypes.c_float(1.0), 0, None)
assert ran(names, "fp_r_batch_kernel" if mode == R else "fp_a_batch_kernel")
assert batch_drop(b.handle) == 0
least = H.fake_used()
assert least < full
b.close()
H.fake_budget(least)
b = K.Batch(gs, mode=mode)
assert H.fake_used() == least
b.close()
""" % mode)


def test_graph_capture(run):
    """Nothing is allocated, waited for or built under capture, and lists
    whose addresses a graph holds are kept."""
    run("""
c = context(arc())
have = H.fake_used()
H.fake_capture(1)
names = forward(c, A)
assert len(names) == 1 and ran(names, "fp_a_kernel") and H.fake_used() == have
H.fake_capture(0)
assert ran(forward(c, A), "fp_a_row_kernel")
H.fake_capture(1)
names = forward(c, A)
assert len(names) == 1 and ran(names, "fp_a_row_kernel")
H.fake_capture(0)
have = H.fake_used()
H.fake_budget(have + 1000)
assert L.kv_back_project(c.handle, buf, buf, A) == 3  # no memory
assert H.fake_used() == have and ran(forward(c, A), "fp_a_row_kernel")
H.fake_budget(1 << 40)
c = context(arc())  # lists that no graph holds: kept too, since freeing them waits
forward(c, A)
have = H.fake_used()
H.fake_budget(have + 1000)
H.fake_capture(1)
assert L.kv_back_project(c.handle, buf, buf, A) == 3 and H.fake_used() == have
H.fake_capture(0)
assert ran(forward(c, A), "fp_a_row_kernel")
""")


def test_tuner_leaves_forward_layouts_of_row_by_row_passes(run, tmp_path):
    """Without a layout to choose none is timed, applied or written down; a
    batch that needs one times it, whatever the file says of brick depths."""
    run("""
path = %r
gs = [arc(16), arc(20, 100)]

def tuned(b, cache):
    n = sum("fp_a_batch_kernel" in k for k in launches(L.kv_batch_autotune, b.handle, cache))
    return n, [b.get_tiles(i) for i in range(len(gs))]

b = K.Batch(gs, mode=A)
before = [l for l, _ in (b.get_tiles(i) for i in range(len(gs)))]
n, tiles = tuned(b, path)
assert n == 2 * 2 and [l for l, _ in tiles] == before, (n, tiles)
assert [ln.split()[2] for ln in open(path)] == ["0"]
assert tuned(b, path) == (0, tiles)
assert batch_drop(b.handle) == 0
n, tiles = tuned(b, path)
assert n == 2 * 4 * 2
(line,) = open(path).readlines()
assert all((str(l), str(z)) == tuple(line.split()[2:4]) for l, z in tiles) and tiles[0][0] in (1, 2, 4, 8)
assert tuned(b, path) == (0, tiles)
b = K.Batch(gs, mode=A)  # with lists: the file's depth, its own layout
n, again = tuned(b, path)
assert n == 0 and [l for l, _ in again] == before and [z for _, z in again] == [z for _, z in tiles]
""" % str(tmp_path / "tiles").encode())


def test_backprojectors_without_a_caller_are_not_built(run):
    """Weights without their test (FW, the last parameter but one) are mode R's,
    and not of the pair count, which needs the test."""
    run("""
H.fake_kernel.restype = ctypes.c_char_p
names = [H.fake_kernel(i).decode() for i in range(H.fake_kernels())]
fw = [n for n in names if "bp_tiled_kernel" in n and ("Lb1ELb0EEEv" in n or "Lb1ELb1EEEv" in n)]
assert len(fw) == 6 and all("ILi0ELi%dE" % (i // 2) in n for i, n in enumerate(sorted(fw))), fw
""")
