"""What the library does around its kernels - device memory, streams, waits, the order of its
launches - on a host model of the HIP runtime (hip_model.c), without a GPU.  Each test runs in a
process of its own, which loads the model in the runtime's place before the library; kernels do
nothing there, copies and fills are carried out as late as the streams' rules allow."""
import os
import shutil
import subprocess
import sys
import textwrap

import pytest

import ptn_hip

HERE = os.path.dirname(os.path.abspath(__file__))

PRELUDE = """
import ctypes, sys
model = ctypes.CDLL(%r, ctypes.RTLD_GLOBAL)
model.model_trace.restype = ctypes.c_char_p
for f in (model.model_in_use, model.model_peak):
    f.restype = ctypes.c_size_t
model.model_limit.argtypes = [ctypes.c_size_t]
for f in (model.model_mallocs, model.model_frees):
    f.restype = ctypes.c_long
model.model_fail_after.argtypes = [ctypes.c_long]
sys.path.insert(0, %r)
import numpy as np
import ptn_hip as P
MB = 1 << 20

def trace():
    return [model.model_trace(i).decode() for i in range(model.model_trace_size())]

def factors(dims, R):
    return [np.random.default_rng(I).random((I, R)) for I in dims]

def tensor(h, dims, storage=P.TENSOR_BOTH):
    # (the model's kernels do nothing: no values, only the memory)
    h.generate_tensor(list(dims), 3, seed=1, storage=storage)
"""


@pytest.fixture(scope="module")
def on_model(tmp_path_factory):
    cc = shutil.which("gcc") or shutil.which("cc")
    if cc is None:
        pytest.skip("no host C compiler")
    so = str(tmp_path_factory.mktemp("model") / "libhip_model.so")
    subprocess.run([cc, "-O1", "-Wall", "-Wextra", "-Werror", "-shared", "-fPIC", "-o", so,
                    os.path.join(HERE, "hip_model.c"), "-lpthread"], check=True)
    prelude = PRELUDE % (so, os.path.dirname(ptn_hip.LIB_PATH))

    def run(code):
        r = subprocess.run([sys.executable, "-c", prelude + textwrap.dedent(code)], capture_output=True, text=True,
                           timeout=300)
        assert r.returncode == 0, r.stdout[-4000:] + r.stderr[-4000:]
        return r.stdout

    return run


CALLS = """
def network_rows(n):
    return np.zeros((n, P.MLP_IN), np.float32), np.zeros((n, P.MLP_OUT), np.float32), np.full(n, 7, np.uint8)

def calls(h):
    d3, d4 = (60, 50, 40), (12, 11, 10, 9)
    kw = dict(max_iter=3, threshold_error=0.0, time_passes=1)    # (timed runs wait for events, not for kernels' stores)
    tree = dict(kw, mttkrp_form=P.MTTKRP_DIMTREE)
    return [
        lambda: h.set_tensor(np.ones(d3), storage=P.TENSOR_BOTH), lambda: h.set_tensor(np.ones(d3), storage=P.TENSOR_F32),
        lambda: tensor(h, d3), lambda: h.norm_sq(), lambda: h.mttkrp(factors(d3, 5), 0),
        lambda: h.mttkrp(factors(d3, 40), 1, arith=P.ARITH_BF16X3), lambda: h.mttkrp_dimtree(factors(d3, 20)),
        lambda: h.cost_explicit(factors(d3, 5)), lambda: h.cpd(5, factors(d3, 5), **kw),
        lambda: h.cpd(33, factors(d3, 33), constraints=[1, 2, 0], **tree),
        lambda: h.cpd(20, factors(d3, 20), arith=P.ARITH_F32, fuse_accel=1, **tree),
        lambda: tensor(h, d4), lambda: h.mttkrp_dimtree(factors(d4, 9), arith=P.ARITH_F32),
        lambda: h.cpd(9, factors(d4, 9), arith=P.ARITH_BF16X3, fuse_accel=1, **tree),
        lambda: h.cpd(9, factors(d4, 9), **kw),
        lambda: h.nesterov(np.eye(6), np.ones((30, 6)), np.ones((30, 6))), lambda: h.sym_extremes(np.eye(6)),
        lambda: h.mlp_init(1), lambda: h.mlp_set_params(np.zeros(P.MLP_PARAMS, np.float32)), lambda: h.mlp_params(),
        lambda: h.mlp_forward(np.zeros((3, P.MLP_IN), np.float32)), lambda: h.mlp_data_add(*network_rows(40)),
        lambda: h.mlp_data_add(*network_rows(90)), lambda: h.mlp_loss_grad(*network_rows(70)),
        lambda: h.mlp_train(1, batch=32, lr=1e-3, seed=7),
        lambda: h.cpd(9, factors(d4, 9), arith=P.ARITH_F32, fuse_accel=1, mlp_harvest=1, warm_start=1, **tree),
        lambda: h.batch_generate([(20, 19, 18), (17, 16, 21)], [4, 5], seed=1),
        lambda: h.batch_init_factors(seed=2), lambda: h.cpd_batch(h.batch_init_factors(seed=2), max_iter=2),
    ]
"""


FAILING = CALLS + """
# every call with its allocations failing from the k-th on, for every k: yields (call, (its index, k))
# after each failure
def failing_calls():
    for i in range(len(calls(None))):
        k, failed = 0, True
        while failed:
            with P.Handle(0) as h:
                cs = calls(h)
                for j in (2, 11, 17, 21, 26):                # what the later calls need
                    if j < i:
                        cs[j]()
                model.model_fail_after(k)
                failed = False
                try:
                    cs[i]()
                except P.PtnError as e:
                    assert e.code == 2, (i, k, e)
                    failed = True
                model.model_fail_after(-1)
                if failed:
                    yield cs[i], (i, k)
            k += 1
"""


def test_a_call_that_ran_out_of_memory_does_not_fail_the_next(on_model):
    """The runtime remembers an error until it is asked for; the next call on the thread must not
    take it for its own."""
    on_model(FAILING + textwrap.dedent("""
        n = 0
        for c, at in failing_calls():
            c()
            n += 1
        assert n > 200, n
        """))


def test_no_work_is_left_queued_when_a_call_returns(on_model):
    """A returned call's memory may go to another handle, so nothing that reads or writes it may
    still wait in a stream, the null stream included; nor after a call that ran out of memory."""
    on_model(FAILING + textwrap.dedent("""
        left = []
        with P.Handle(0) as h:
            for i, c in enumerate(calls(h)):
                c()
                if model.model_pending():
                    left.append((i, model.model_pending()))
        for c, at in failing_calls():
            if model.model_pending():
                left.append((at, model.model_pending()))
        assert not left, left
        """))


def test_a_tensor_that_did_not_fit_leaves_none(on_model):
    """Setting a tensor gives up the one before; when the memory for the new one is not there, the
    handle has none, and calls that need one say so instead of reading it."""
    on_model("""
        for storage in (P.TENSOR_F64, P.TENSOR_F32, P.TENSOR_BOTH):
            for k in (0, 1, 2):
                with P.Handle(0) as h:
                    tensor(h, (20, 10, 5), storage)
                    dims = h.dims
                    model.model_fail_after(k)
                    fits = False
                    try:
                        tensor(h, (60, 50, 40), storage)
                        fits = True
                    except P.PtnError as e:
                        assert e.code == 2, e
                    model.model_fail_after(-1)
                    if fits:
                        continue
                    h.dims = dims
                    for c in (h.norm_sq, lambda: h.cost_explicit(factors(dims, 3)),
                              lambda: h.mttkrp(factors(dims, 3), 0), lambda: h.cpd(3, factors(dims, 3), max_iter=1)):
                        try:
                            c()
                            raise AssertionError((storage, k))
                        except P.PtnError as e:
                            assert e.code == 5, (storage, k, e)
                    tensor(h, dims, storage)
                    h.norm_sq()
        """)


def test_activation_buffers_that_did_not_fit_are_taken_again(on_model):
    """The network's buffers grow by giving up the smaller ones.  When a larger one does not fit, a
    later call of the old size must not go on with the missing one (the model copies to the address
    it is given)."""
    on_model("""
        for k in range(40):
            with P.Handle(0) as h:
                h.mlp_init(1)
                h.mlp_forward(np.zeros((3, P.MLP_IN), np.float32))
                model.model_fail_after(k)
                failed = False
                try:
                    h.mlp_forward(np.zeros((3000, P.MLP_IN), np.float32))
                except P.PtnError as e:
                    assert e.code == 2, e
                    failed = True
                model.model_fail_after(-1)
                h.mlp_forward(np.zeros((3, P.MLP_IN), np.float32))
                if not failed:
                    assert k > 10
                    break
        """)


def test_a_tensor_given_up_is_given_back(on_model):
    """Setting another tensor, or another storage, returns the old one's memory to the device at once
    (tensors of up to 128 MB to the pool), a tensor of the same size takes it over, and the work buffers
    kept between calls stay."""
    on_model("""
        big, small = (1000, 800, 600), (30, 20, 10)
        nb, ns = 480000000, 6000
        with P.Handle(0) as h:
            tensor(h, small)
            none = model.model_in_use()
            tensor(h, big)
            full = model.model_in_use()
            assert full > none + 12 * (nb - ns)
            mallocs = model.model_mallocs()
            tensor(h, big)
            tensor(h, (800, 1000, 600))
            assert (model.model_mallocs(), model.model_in_use()) == (mallocs, full)
            tensor(h, big, P.TENSOR_F32)
            assert model.model_in_use() <= full - 8 * nb
            tensor(h, small)
            assert model.model_in_use() < none + MB, (model.model_in_use(), none)
            h.mttkrp(factors(small, 5), 0)                   # work buffers
            tensor(h, big)
            h.mttkrp(factors(big, 5), 0)
            tensor(h, small)
            mallocs, used = model.model_mallocs(), model.model_in_use()
            assert used < none + 6000 * MB, used
            h.mttkrp(factors(small, 5), 0)
            tensor(h, big)
            h.mttkrp(factors(big, 5), 0)
            assert model.model_mallocs() == mallocs + 2      # the two copies of the tensor
            # up to 128 MB: kept for the next handle's, and given back when asked for
            h.release_memory()
            tensor(h, small)
            h.release_memory()
            none = model.model_in_use()
            tensor(h, (100, 400, 400), P.TENSOR_F64)
            kept = model.model_in_use()
            tensor(h, small)
            with P.Handle(0) as g:
                tensor(g, (100, 400, 400), P.TENSOR_F64)
                assert model.model_in_use() < kept + MB, (model.model_in_use(), kept)
            h.release_memory()
            assert model.model_in_use() == none, (model.model_in_use(), none)
        assert model.model_in_use() == 0
        """)


def test_an_fp32_tensor_is_not_staged_whole(on_model):
    """FP64 host data for an FP32 tensor passes through a buffer of a bounded size, which is what stays
    in the pool of work buffers afterwards."""
    on_model("""
        with P.Handle(0) as h:
            before = model.model_in_use()
            X = np.zeros((300, 300, 333), order="F")         # 240 MB, 120 MB in FP32
            h.set_tensor(X, storage=P.TENSOR_F32)
            assert model.model_peak() <= before + X.size * 4 + 80 * MB, model.model_peak()
            copies = [int(t.split("bytes=")[1].split()[0]) for t in trace() if t.startswith("copy kind=1")]
            casts = [t for t in trace() if "k_cast" in t]
            assert sum(copies) == 8 * X.size and len(casts) == len(copies) > 1
        """)


def test_a_call_needs_no_memory_for_what_it_has_replaced(on_model):
    """A buffer that a call replaces by a larger one is kept until the call's work is done with it, but
    not when its memory is needed: with room for the larger buffers alone the call still runs.  The
    paired line search of order 4 takes its larger partial sums at once."""
    on_model("""
        def rows(n):
            return np.zeros((n, P.MLP_IN), np.float32)
        with P.Handle(0) as h:
            h.mlp_init(1)
            h.mlp_forward(rows(8000))
            need = model.model_in_use()
        with P.Handle(0) as h:
            h.mlp_init(1)
            h.mlp_forward(rows(6000))
            model.model_limit(need + MB)
            h.mlp_forward(rows(8000))
            model.model_limit(1 << 62)
            assert model.model_pending() == 0

        # partial sums of 64 splits of (I0 I1) rows of 64 (paired: 128) floats
        dims, R = (200, 200, 20, 20), 64
        kw = dict(max_iter=3, threshold_error=0.0, time_passes=1, mttkrp_form=P.MTTKRP_DIMTREE, arith=P.ARITH_F32)
        part = 64 * 200 * 200 * 64 * 4
        peak = []
        for fuse in (0, 1):
            with P.Handle(0) as h:
                tensor(h, dims, P.TENSOR_F32)
                model.model_reset_peak()
                h.cpd(R, factors(dims, R), fuse_accel=fuse, **kw)
                peak.append(model.model_peak())
        # paired: twice the partial sums, the pair of left nodes (as large as 2 of the 64 splits), the
        # pair of mode-0 results and the packed operand for both
        assert peak[1] - peak[0] < part + part // 32 + 40 * MB, [p // MB for p in peak]
        """)


def test_blocks_of_other_calls_do_not_crowd_out_a_call(on_model):
    """A call that fits the memory by itself fits after larger calls too: it does not hold their larger
    blocks in the place of its own."""
    on_model("""
        dims, R = (40, 1500, 1500), 20
        with P.Handle(0) as h:
            tensor(h, dims)
            h.mttkrp(factors(dims, R), 1)
            need = model.model_peak()
        larger = (40, 1600, 1800)
        with P.Handle(0) as h:
            tensor(h, larger)
            h.mttkrp(factors(larger, R), 1)
            tensor(h, dims)
            model.model_limit(need + MB)
            h.mttkrp(factors(dims, R), 1)
        """)


def test_freeing_blocks_does_not_stop_other_handles(on_model):
    """hipFree waits for the device.  While one handle's call frees blocks of the pool, another handle's
    calls go on (the model holds the hipFree until they have, or two seconds)."""
    on_model("""
        import threading
        dims = (30, 20, 10)
        a, b = P.Handle(0), P.Handle(0)
        tensor(a, dims)
        tensor(b, dims)
        b.mttkrp(factors(dims, 5), 0)
        big = (4000, 3000, 2)                                # work buffers beyond what the pool keeps
        tensor(a, big, P.TENSOR_F64)
        a.mttkrp(factors(big, 5), 0)
        model.model_limit(model.model_in_use() + 40 * MB)
        model.model_hold_free(1)
        t = threading.Thread(target=lambda: a.nesterov(np.eye(60), np.ones((3000, 60)), np.ones((3000, 60))))
        t.start()                                            # finds no memory: the pool is emptied
        while not model.model_free_held():
            assert t.is_alive() or model.model_free_timed_out()
        b.mttkrp(factors(dims, 5), 1)
        b.sym_extremes(np.eye(5))
        assert not model.model_free_timed_out()
        model.model_hold_free(0)
        t.join()
        """)


def test_the_kept_work_buffers_can_be_given_back(on_model):
    """Up to 8 GiB of work buffers stay on the device between calls; release_memory returns them, of
    every handle of the GPU, and leaves the tensors, the network and the calls alone."""
    on_model(CALLS + textwrap.dedent("""
        a, b = P.Handle(0), P.Handle(0)
        tensor(a, (60, 50, 40))
        tensor(b, (60, 50, 40))
        a.release_memory()
        before = model.model_in_use()
        for c in calls(a)[3:11]:
            c()
        b.mttkrp(factors((60, 50, 40), 5), 1)
        assert before + 4 * MB < model.model_in_use() < before + 8192 * MB
        b.release_memory()
        assert model.model_in_use() == before
        for c in calls(a)[3:11]:
            c()
        a.release_memory()
        assert model.model_in_use() == before
        a.close()
        b.close()
        assert model.model_in_use() == 0
        """))


def test_timed_passes_hold_the_contraction_alone(on_model):
    """t_pass_ms is the device time of the tensor passes: the NNLS set-up that rides along with an FP64
    contraction of rank <= 16 (the instances whose last template parameter is true) stays out of a
    timed one."""
    on_model("""
        dims, R = (60, 50, 40), 10
        with P.Handle(0) as h:
            tensor(h, dims)
            for arith in (P.ARITH_F64, P.ARITH_F32_F64):
                model.model_trace_clear()
                kw = dict(max_iter=3, threshold_error=0.0, mttkrp_form=P.MTTKRP_DIMTREE, arith=arith)
                try:
                    h.cpd(R, factors(dims, R), **kw)         # (ends in an error: no kernel publishes the sweep)
                except P.PtnError as e:
                    assert e.code == 3
                assert any("k_gemm" in t and "Lb1EEE" in t for t in trace())
                model.model_trace_clear()
                _, _, log = h.cpd(R, factors(dims, R), time_passes=1, **kw)
                assert all(t > 0 for l in log for t in l["t_pass_ms"])
                lines = [t for t in trace() if not t.startswith("copy")]
                timed = [t for a, t, b in zip(lines, lines[1:], lines[2:])
                         if a.startswith("record") and b.startswith("record")]
                assert len([t for t in timed if "k_gemm_cm_f64" in t]) == 3
                assert len([t for t in timed if "k_gemm_ck_f64" in t]) == 3
                assert not any("k_gemm" in t and "Lb1EEE" in t for t in lines)
                assert any("k_eig_extremes" in t for t in lines)
        """)


def test_a_set_up_that_a_contraction_does_not_take_is_not_lost(on_model):
    """The FP64 contractions take an NNLS set-up along in their rank-16 instances only, and say whether
    they did, so that the caller launches it where they did not; and without it they have no block
    for it."""
    on_model("""
        lib = P.lib()
        buf = ctypes.create_string_buffer(1 << 16)
        spec = (ctypes.c_int64 * 33)(1, 50)                  # KrSpec: one mode of 50
        setup = (ctypes.c_int64 * 16)()                      # NnlsSetup
        at = ctypes.addressof(buf)
        i64, vp = ctypes.c_int64, ctypes.c_void_p
        cm = lib["_ZN3ptn11gemm_cm_f64EP12ihipStream_tPKdPKfllRKNS_6KrSpecEiiPdPKNS_9NnlsSetupE"]
        ck = lib["_ZN3ptn11gemm_ck_f64EP12ihipStream_tPKdPKfllRKNS_6KrSpecEiPdPKNS_9NnlsSetupE"]
        cm.argtypes = [vp, vp, vp, i64, i64, vp, ctypes.c_int, ctypes.c_int, vp, vp]
        ck.argtypes = [vp, vp, vp, i64, i64, vp, ctypes.c_int, vp, vp]
        cm.restype = ck.restype = ctypes.c_bool
        for x64, x32 in ((at, None), (None, at)):
            for ldr in (16, 32, 48, 64):
                for s in (None, setup):
                    model.model_trace_clear()
                    took = (cm(None, x64, x32, 640, 50, spec, ldr, 1, at, s),
                            ck(None, x64, x32, 50, 640, spec, ldr, at, s))
                    lines = [t for t in trace() if "k_gemm" in t]
                    want = s is not None and ldr == 16
                    assert len(lines) == 2 and took == (want, want), (ldr, took)
                    for t, blocks in zip(lines, (10, 40)):
                        assert ("Lb1EEE" in t) == want and ("grid=%d," % (blocks + want)) in t, t
        """)


def test_schedules_of_a_sweep(on_model):
    """Which streams a sweep's set-ups and contractions take, on both sides of every limit (schedule_for):
    all on one, the contraction aside, or the set-up aside.  Whatever aside is, the update waits for
    both."""
    on_model("""
        def schedule(h, dims, R, form, arith, cons):
            model.model_trace_clear()
            kw = dict(max_iter=2, threshold_error=0.0, mttkrp_form=form, arith=arith, time_passes=1)
            h.cpd(R, factors(dims, R), constraints=cons, **kw)
            lines = trace()
            lines = lines[next(i for i, t in enumerate(lines) if "stream=0 blocking" in t):]    # the sweeps
            stream = lambda what: [t.split("stream=")[1].split()[0] for t in lines if what in t]
            update = set(stream("k_nnls_iterate"))
            assert len(update) == 1
            nnls = next(k for k, c in enumerate(cons) if c == 1)
            setup, gemm = set(stream("k_eig_extremes")), stream("k_gemm_c")
            if not stream("wait"):
                assert setup == update == set(gemm)
                return "one"
            if setup == update:
                assert set(gemm) - update
                return "contraction"
            assert update <= set(gemm) and not setup & set(gemm)
            return "set-up"

        def cubes(order, mb, size):
            d = round((mb * MB / size) ** (1.0 / order))
            return [d] * order

        std, tree = P.MTTKRP_STANDARD, P.MTTKRP_DIMTREE
        # order, rank, form, FP64?, limit of one stream, limit of the contraction aside (MB)
        rules = [(3, 16, std, 1, 600, 0), (3, 16, tree, 1, 600, 0), (4, 10, std, 1, 600, 0), (5, 8, std, 1, 150, 0),
                 (5, 9, std, 1, 20, 0), (6, 8, std, 1, 90, 0), (6, 16, std, 1, 5, 0), (6, 16, tree, 1, 600, 0),
                 (3, 16, std, 0, 10, 0), (3, 8, std, 0, 32, 0), (3, 5, std, 0, 96, 0), (4, 9, std, 0, 10, 0),
                 (4, 5, std, 0, 96, 0), (5, 5, std, 0, 32, 0), (5, 6, std, 0, 2, 0), (6, 5, std, 0, 32, 0),
                 (6, 6, std, 0, 1, 0), (4, 16, tree, 0, 96, 128),
                 (3, 17, std, 1, 8, 84), (3, 32, tree, 1, 8, 288), (3, 33, std, 1, 0, 276), (3, 64, tree, 1, 0, 640),
                 (3, 20, std, 0, 0, 63), (3, 64, std, 0, 0, 591), (4, 20, std, 1, 0, 63), (4, 20, std, 0, 0, 60),
                 (4, 24, tree, 0, 0, 288), (5, 24, std, 1, 0, 12), (5, 24, std, 0, 0, 4), (6, 25, std, 1, 0, 5),
                 (6, 24, std, 0, 0, 2), (7, 40, tree, 1, 0, 640)]
        for order, R, form, fp64, one, aside in rules:
            seen = []
            for lim in sorted({one, aside}):
                for mb in (lim * 0.75, lim * 1.3) if lim else (0.5,):
                    for arith, size in ((P.ARITH_F64, 8), (P.ARITH_F32_F64, 4)) if fp64 else \\
                            ((P.ARITH_F32, 4), (P.ARITH_BF16X3, 4)):
                        dims = cubes(order, mb, size)
                        got = np.prod([float(d) for d in dims]) * size / MB
                        if (got - lim) * (mb - lim) <= 0:      # (small orders jump past the limit)
                            continue
                        with P.Handle(0) as h:
                            tensor(h, dims, P.TENSOR_F64 if arith == P.ARITH_F64 else P.TENSOR_F32)
                            want = "one" if got <= one else "contraction" if got <= aside else "set-up"
                            got_s = schedule(h, dims, R, form, arith, [1] * order)
                            assert got_s == want, (order, R, form, arith, dims, got_s, want)
                            seen.append(want)
            assert len(set(seen)) == 1 + (one > 0) + (aside > one) or order >= 5, (order, R, seen)
        # the order-3 tree with FP32 products keeps its own (the right node on a third stream)
        with P.Handle(0) as h:
            tensor(h, (30, 30, 30), P.TENSOR_F32)
            assert schedule(h, (30, 30, 30), 5, tree, P.ARITH_F32, [1, 1, 1]) == "set-up"
        """)


def test_failing_calls_on_several_threads(on_model):
    """Handles on four threads, one of them running out of memory again and again with buffers taken:
    every other call runs, no block is given to two calls at once (the model's hipFree knows its
    blocks, and copies through them keep their values), and all memory returns at the end."""
    on_model("""
        import threading
        bad, done = [], []
        def rows(n):
            return np.full((n, P.MLP_IN), n, np.float32), np.zeros((n, P.MLP_OUT), np.float32), np.full(n, 7, np.uint8)
        def work(k):
            try:
                with P.Handle(0) as h:
                    for i in range(12):
                        tensor(h, (20 + k, 30, 40))
                        h.mttkrp(factors((20 + k, 30, 40), 5 + 9 * k), i % 3)
                        n = 30 + 17 * k + i
                        h.mlp_data_clear()
                        h.mlp_data_add(*rows(n))
                        h.mlp_data_add(*rows(n))             # grows: the rows before are copied
                        assert (h.mlp_data_get(0, 2 * n)[0] == n).all()
                        if k == 0:
                            try:
                                h.nesterov(np.eye(64), np.zeros((20000, 64)), np.zeros((20000, 64)))
                                bad.append("ran")
                            except P.PtnError as e:
                                assert e.code == 2
                    done.append(k)
            except BaseException as e:
                bad.append((k, repr(e)))
        model.model_limit(300 * MB)                          # (51 iterates of 20000 x 64: 522 MB)
        threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
        for t in threads: t.start()
        for t in threads: t.join()
        assert not bad and sorted(done) == [0, 1, 2, 3], (bad, done)
        assert model.model_in_use() == 0 and model.model_pending() == 0
        """)


def test_short_quotient_and_root_equal_the_operators(tmp_path):
    """The quotient and square root in the kernels' dependent chains (csrc/short_ops.inc) are correctly
    rounded over the operands their callers keep to: 24 million of each, random, next to powers of two
    and to the middles between doubles."""
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("no host C++ compiler")
    exe = str(tmp_path / "short_ops_check")
    subprocess.run([cxx, "-O2", "-ffp-contract=off", "-std=c++17", "-Wall", "-I",
                    os.path.join(os.path.dirname(ptn_hip.LIB_PATH), "csrc"), "-o", exe,
                    os.path.join(HERE, "short_ops_check.cpp")], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and r.stdout == "0\n", r.stdout


def test_fused_right_node_has_no_idle_waves(on_model):
    """The order-3 right node with its leaf contraction in one launch: chunks of 64 fibres of one index of
    the last mode, four to a block whatever that index is."""
    on_model("""
        for dims in ((13, 50, 79), (30, 1, 101), (32, 64, 7), (31, 65, 9), (40, 256, 3), (64, 257, 5), (33, 300, 1)):
            with P.Handle(0) as h:
                tensor(h, dims, P.TENSOR_F32)
                for arith in (P.ARITH_F32, P.ARITH_BF16X3):
                    for R in (5, 40):
                        model.model_trace_clear()
                        h.mttkrp_dimtree(factors(dims, R), arith=arith)
                        grid = [int(t.split("grid=")[1].split(",")[0]) for t in trace() if "k_gemm_ck_lds" in t]
                        assert grid == [((dims[1] + 63) // 64 * dims[2] + 3) // 4], (dims, grid)
        """)


def test_loads_of_the_fp64_column_contraction(on_model):
    """Non-temporal loads (the contraction's second-last template parameter) for FP64 tensors whose columns
    are whole cache lines and which the last-level cache does not hold; cached ones elsewhere."""
    on_model("""
        for dims, storage, want in (((512, 512, 128), P.TENSOR_F64, "00"), ((512, 512, 129), P.TENSOR_F64, "11"),
                                    ((496, 528, 140), P.TENSOR_F64, "01"), ((513, 521, 140), P.TENSOR_F64, "00"),
                                    ((640, 640, 640), P.TENSOR_F32, "00"), ((64, 10, 10), P.TENSOR_F64, "00")):
            with P.Handle(0) as h:
                tensor(h, dims, storage)
                arith = P.ARITH_F64 if storage == P.TENSOR_F64 else P.ARITH_F32_F64
                for R in (5, 20, 40, 64):
                    model.model_trace_clear()
                    h.mttkrp(factors(dims, R), 0, arith=arith)
                    h.time_contraction(0, factors(dims, R), arith=arith, iters=1)
                    kernels = [t for t in trace() if "k_gemm_cm_f64" in t]
                    got = [t[t.index("ELb0EEE") - 1] for t in kernels]      # mode 0, then the left node twice
                    assert got == [want[0], want[1], want[1]], (dims, kernels)
        """)
