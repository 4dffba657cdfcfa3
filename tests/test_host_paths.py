"""Host paths of the library without a GPU: libqpslice.so on a HIP runtime that
records kernels instead of running them (hip_stub.cpp).  Each test is a program of
its own, so that the stub is the only runtime of its process."""
import os
import subprocess
import sys
import textwrap

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
PKG = os.path.join(os.path.dirname(HERE), "quickpic-opensource_amd")
ROCM = "/opt/rocm/include"

pytestmark = pytest.mark.skipif(
    not (os.path.isdir(ROCM) and os.path.exists(os.path.join(PKG, "libqpslice.so"))),
    reason="needs the ROCm headers and the built library")

HEAD = """
import ctypes as C, os, sys, traceback
stub = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
sys.path.insert(0, sys.argv[2])
import qpslice as qps

def sims(n, ind=4):
    out = []
    for _ in range(n):
        ctx = qps.Ctx(ind, ind, 4)
        sim = qps.Sim(ctx, [qps.Species(ctx, ppc=(1, 1))], [])
        sim.begin_step()
        out.append(sim)
    return out

def refused(fn, *args):
    try:
        fn(*args)
    except qps.QPError as e:
        return e
    raise AssertionError("not refused")

def test():
"""

TAIL = """
try:
    test()
except BaseException:
    traceback.print_exc()
    os._exit(1)
os._exit(0)   # the stub's process ends without the runtime's tear-down
"""


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("stub") / "libhipstub.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-w", "-I" + ROCM,
                    os.path.join(HERE, "hip_stub.cpp"), "-o", so], check=True)
    return so


def run(stub, body):
    p = subprocess.run([sys.executable, "-c", HEAD + textwrap.indent(body, "    ") + TAIL, stub, PKG],
                       capture_output=True, text=True, timeout=120)
    assert p.returncode == 0, p.stdout + p.stderr


@pytest.mark.parametrize("tol,residual", [(0.0, 0.0), (1e-3, 0.0), (1e-3, 1.0)])
def test_scan_runs_whatever_device_is_current(stub, tol, residual):
    """A run by a thread that has another device current: the graphs that are made
    executable in it are the scan's device's, and the thread keeps its own."""
    run(stub, f"""
stub.stub_residual(C.c_size_t(8 * 64), C.c_double({residual}))
scan = qps.Scan(sims(2), iter_max=6, tol={tol})
stub.hipSetDevice(1)
scan.run(2)
assert stub.stub_graph_launches() >= 4
d = C.c_int(-1)
stub.hipGetDevice(C.byref(d))
assert d.value == 1
""")


@pytest.mark.parametrize("tol,at", [(0.0, 1), (0.0, 2), (0.0, 3), (1e-3, 3), (1e-3, 4)])
def test_scan_run_ended_by_an_error(stub, tol, at):
    """Graph launch `at` of a run fails.  The streams are waited for; every
    species's pointers are those of the slices that were launched; and the scan,
    whose simulations are at different slices, runs no further.  Launches in
    order, for two simulations: fixed passes 0 1 0 1 (slices); to a tolerance,
    converged in the first graph, starts 0 1, end and next start of 0, of 1."""
    run(stub, f"""
stub.stub_residual(C.c_size_t(8 * 64), C.c_double(0.0))
stub.stub_word.restype = C.c_ulonglong
s = sims(2)

def buffer(x):
    x.species[0].push(x.field(qps.F_FXY), x.field(qps.F_BXYZ), x.field(qps.F_PSIT), x.ctx.dex)
    return stub.stub_word(b"k_push")

at0 = [buffer(x) for x in s]
at1 = [buffer(x) for x in s]
assert at0 != at1
scan = qps.Scan(s, iter_max=3, tol={tol})   # the particles are at at0
syncs = [stub.stub_syncs(i) for i in range(2)]
stub.stub_fail_launch({at})
refused(scan.run, 2)
# one wait reads the slice word, one follows the error
assert all(stub.stub_syncs(i) >= n + 2 for i, n in enumerate(syncs))
e = refused(scan.run, 1)
assert e.code == -3, e.code   # QP_ERR_STATE
done = {{0.0: {{1: (0, 0), 2: (1, 0), 3: (1, 1)}}, 1e-3: {{3: (0, 0), 4: (1, 0)}}}}[{tol}][{at}]
assert [buffer(x) for x in s] == [(at0, at1)[n][i] for i, n in enumerate(done)]
""")


def test_polled_residuals_are_coherent(stub):
    """qp_scan_run reads the residuals while kernels run: the memory they are
    written to is asked for as coherent."""
    run(stub, """
ctx = qps.Ctx(4, 4, 4)
flags = C.c_uint(stub.stub_host_flags(C.c_size_t(8 * 64))).value
assert flags != 0xffffffff and flags & 0x40000000, hex(flags)   # hipHostMallocCoherent
""")


@pytest.mark.parametrize("ind", [4, 11])
def test_refused_pass_count_leaves_the_slice_prepared(stub, ind):
    """qp_slice_run refuses iter_max 0 after the slice's first part, on which
    qp_slice_finish goes on, with the fused field solves (16^2) as without (2048^2)."""
    run(stub, f"""
x = sims(1, {ind})[0]
e = refused(lambda: x.slice(1, iter_max=0, tol=1e-3))
assert "iter_max" in str(e)
assert x.finish(1, iter_max=2)[0] == 2
""")


NET = """
L = qps.lib()
P = [C.c_void_p(1 << 12 + i) for i in range(8)]   # addresses that only kernels would use
"""


def test_head_gradient_without_outputs(stub):
    """No output planes: no gradient to add up, and no error."""
    run(stub, NET + """
rc = L.qp_net_head_bwd(None, P[0], 32, 32, P[1], 0, C.c_size_t(64), P[2], P[3], 4, P[4], P[5])
assert rc == 0, L.qp_last_error()
""")


CONV = NET + """
def conv(H, W, cin, cout, mask=None):
    stub.stub_clear_launches()
    rc = L.qp_net_conv3x3(None, P[0], mask, H, W, cin, cin, P[1], None, P[2], cout, cout, 1, 0)
    assert rc == 0, L.qp_last_error()
    return stub.stub_launched(b"k_conv3x3_deep")

"""


@pytest.mark.parametrize("cin", [16, 32, 48, 64, 96, 128, 192])
def test_convolution_within_the_devices_lds(stub, cin):
    """A layer whose pixels and weights do not fit a workgroup's LDS is computed
    from memory; one that does keeps the kernel that stages them."""
    run(stub, CONV + f"""
stub.stub_limits(163840, 256)
assert conv(128, 128, {cin}, 32) == 0
need = stub.stub_lds(b"k_conv3x3")
stub.hipSetDevice(1)
stub.stub_limits(need, 256)
assert conv(128, 128, {cin}, 32) == 0
stub.hipSetDevice(2)
stub.stub_limits(need - 1, 256)
assert conv(128, 128, {cin}, 32) == 1
""")


def test_convolution_blocks_follow_the_compute_units(stub):
    """Blocks of four pixel groups (18 x 6 pixels) where four blocks fill the
    device, of one (18 x 3) where they leave most of it idle."""
    run(stub, CONV + """
stub.stub_limits(163840, 4)
conv(16, 16, 16, 16)
assert stub.stub_lds(b"k_conv3x3") == (18 * 6 + 144) * 48
stub.hipSetDevice(1)
stub.stub_limits(163840, 256)
conv(16, 16, 16, 16)
assert stub.stub_lds(b"k_conv3x3") == (18 * 3 + 144) * 48
""")


@pytest.mark.parametrize("precision", ["FP32", "FP64"])
def test_default_form_of_the_separate_transforms(stub, precision):
    """QP_TUNE_FFT 7: what the default's number names, a transpose between row
    passes (FP32) or column pairs (FP64), without the default's fused routes."""
    run(stub, f"""
ctx = qps.Ctx(5, 5, 4, precision=qps.{precision})
sim = qps.Sim(ctx, [qps.Species(ctx, ppc=(1, 1))], [])

def kernels(value):
    ctx.tune(qps.TUNE_FFT, value)
    stub.stub_clear_launches()
    f = qps.Field2d(ctx, 1)
    f.fftrk(1)
    f.fftkr(1)
    sim.begin_step()
    sim.slice(1)
    return [stub.stub_launched(k) > 0 for k in (b"k_mid", b"k_fft_xt", b"k_transpose")]

fp32 = {precision == "FP32"}
assert kernels(-1) == [True, True, False]
assert kernels(7) == [False, False, fp32]
assert kernels(1) == [not fp32, not fp32, False]
""")


@pytest.mark.parametrize("np_,runs,dense", [
    ((64, 64, 32), 1, True), ((64, 64, 32), 131072 // 28, True), ((64, 64, 32), 131072 // 24, False),
    ((64, 64, 32), 131072, False), ((16, 16, 16), 4096 // 200, True), ((16, 16, 16), 4096 // 100, False),
    ((16, 16, 16), 4096, False)])
def test_beam_deposit_by_the_runs_of_the_last_push(stub, np_, runs, dense):
    """Eight particles a thread where the push found long runs of one cell, one a
    thread where it found short ones, and where the order is not known: before the
    first push and after an upload."""
    run(stub, f"""
ctx = qps.Ctx(4, 4, 4)
bm = qps.Beam(ctx, np_={np_}, sigma=(1.0, 1.0, 1.0), center=(0.0, 0.0, 5.0), peak=1.0)
n = bm.np
blocks = (n + 255) // 256
every = max(1, blocks // 64)
samples = 8 if every > 1 else 1
counted = sum(max(0, min(64, n - j - m * every * 256 // samples))
              for j in range(0, n, every * 256) for m in range(samples))
stub.stub_key_changes(max(1, round({runs} * counted / n)))
e, b = qps.Field3d(ctx, 3), qps.Field3d(ctx, 3)

def eights():
    stub.stub_clear_launches()
    bm.qdp()
    one, eight = (stub.stub_launched(k) for k in (b"k_beam_depositILi1E", b"k_beam_depositILi8E"))
    assert one + eight == 1
    return eight == 1

assert not eights()
bm.push(e, b, ctx.dex, ctx.dxi)
assert eights() == {dense}
bm.upload(bm.download())
assert not eights()
""")


@pytest.mark.parametrize("H,W,cin,cout,wide", [
    (256, 256, 80, 48, True), (128, 128, 80, 48, False), (160, 160, 160, 96, True),
    (128, 128, 256, 48, True), (256, 256, 80, 16, False), (256, 256, 64, 64, False)])
def test_convolution_of_a_large_plane(stub, H, W, cin, cout, wide):
    """Channel counts without a kernel of their own: all output channels in a wave
    where the plane has waves enough, 16 in a wave elsewhere."""
    run(stub, CONV + f"""
conv({H}, {W}, {cin}, {cout})
assert stub.stub_launched(b"k_conv3x3_wide") == {int(wide)}
""")


@pytest.mark.parametrize("H,W,cin,cout,mask,wide", [
    (224, 224, 16, 32, True, True), (192, 192, 16, 32, True, False), (192, 192, 16, 48, True, True),
    (160, 160, 16, 64, True, True), (128, 128, 16, 96, True, False),
    (224, 224, 48, 128, True, True), (256, 256, 48, 96, True, True),
    (224, 224, 32, 192, True, False), (256, 256, 48, 64, True, False),
    (256, 256, 64, 192, True, False), (1024, 1024, 16, 192, False, False)])
def test_masked_convolution_of_a_large_plane(stub, H, W, cin, cout, mask, wide):
    """Few input and many output channels: pixels and mask are read once."""
    run(stub, CONV + f"""
conv({H}, {W}, {cin}, {cout}, P[3] if {mask} else None)
assert stub.stub_launched(b"k_conv3x3_wide") == {int(wide)}
""")


@pytest.mark.parametrize("indy,dim,columns", [(5, 1, False), (7, 3, False), (8, 1, False),
                                              (8, 2, True), (9, 1, True)])
def test_transforms_of_long_rows(stub, indy, dim, columns):
    """FP32 transforms at nx = 2048: through transposed planes with rows enough."""
    run(stub, f"""
ctx = qps.Ctx(11, {indy}, 4, precision=qps.FP32)
f = qps.Field2d(ctx, {dim})
f.fftrk(1)
f.fftkr(1)
assert stub.stub_launched(b"k_fft_xt") == {2 * columns}
assert stub.stub_launched(b"k_transpose") == {2 * (not columns)}
""")


WGRAD = NET + """
def wgrad(H, W, cin, cout, nchunk, db):
    stub.stub_clear_launches()
    rc = L.qp_net_conv3x3_wgrad(None, P[0], cin, cin, P[1], P[2], cout, cout, H, W, nchunk, P[3],
                                P[4], P[5] if db else None)
    assert rc == 0, L.qp_last_error()
    return stub.stub_blocks(b"k_wgrad")
"""


@pytest.mark.parametrize("H,W,cin,cout,nchunk,per_chunk", [
    (64, 64, 16, 16, 8, 1), (1024, 1024, 16, 16, 32, 1), (1024, 1024, 16, 16, 1, 1),
    (32, 190, 16, 16, 32, 0.25), (96, 64, 48, 48, 32, 1), (160, 160, 64, 96, 32, 1),
    (128, 128, 64, 96, 32, 0.25), (512, 512, 192, 192, 32, 0.25), (512, 512, 64, 48, 200, 0.25)])
def test_weight_gradient_of_few_chunks(stub, H, W, cin, cout, nchunk, per_chunk):
    """A chunk of many pixels takes four waves where the launch has few, one where it
    has many."""
    run(stub, WGRAD + f"""
assert wgrad({H}, {W}, {cin}, {cout}, {nchunk}, False) == {int(cout // 16 * cin // 16 * 3 * nchunk * per_chunk)}
""")


@pytest.mark.parametrize("nchunk,launches", [(144, 1), (145, 2), (400, 2), (1000, 1)])
def test_bias_gradient_of_many_chunks(stub, nchunk, launches):
    """More chunks than 9 cin: the bias's partial sums come in a launch of their
    own, and the weights' stay spread over the chunks.  Chunks small enough for a
    block stay there."""
    run(stub, WGRAD + f"""
blocks = wgrad(250, 200, 16, 16, {nchunk}, True)
assert stub.stub_launched(b"k_wgrad") == {launches}
assert blocks == {3 * nchunk if nchunk < 200 else 3 * nchunk // 4 if nchunk < 1000 else 3}
""")


def test_beam_push_reads_its_counts_into_pinned_memory(stub):
    """A copy to pageable memory goes through a staging buffer, with a wait of its own."""
    run(stub, """
ctx = qps.Ctx(4, 4, 4)
bm = qps.Beam(ctx, np_=(8, 8, 8), sigma=(1.0, 1.0, 1.0), center=(0.0, 0.0, 5.0), peak=1.0)
e, b = qps.Field3d(ctx, 3), qps.Field3d(ctx, 3)
was = stub.stub_pageable()
bm.push(e, b, ctx.dex, ctx.dxi)
assert stub.stub_pageable() == was
""")
