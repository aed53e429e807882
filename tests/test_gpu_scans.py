"""GPU parity of the WKV-7 and ROSA scan kernels against the CPU oracle.

Tolerances: fp32 outputs and final states within
1e-4 relative / 1e-5 absolute of the float64 oracle.
"""

import os

import numpy as np
import pytest
import torch

from oracle import rosa as orosa
from oracle import wkv7 as owkv
from yufmusicgen_amd.synth import rosa_inputs, wkv_inputs

pytestmark = pytest.mark.gpu

RTOL, ATOL = 1e-4, 1e-5


def _dev(x):
    return torch.from_numpy(np.ascontiguousarray(x, dtype=np.float32)).cuda()


def _oracle_wkv(arrs, s0=None):
    t = [torch.from_numpy(np.asarray(x, dtype=np.float64)) for x in arrs]
    return owkv.wkv7_scan(*t, None if s0 is None else torch.from_numpy(np.asarray(s0, np.float64)))


KERNELS = ("serial", "chunked")


@pytest.mark.parametrize("wkv_kernel", KERNELS, indirect=True)
@pytest.mark.parametrize("size", [8, 16, 32, 40, 48, 64, 128])
@pytest.mark.parametrize("steps", [1, 16, 17, 50, 100])
def test_wkv7_matches_oracle(size, steps, wkv_kernel):
    from yufmusicgen_amd.ops import rwkv7_scan

    print(f"wkv7 parity N={size} T={steps} kernel={wkv_kernel}", flush=True)
    arrs = wkv_inputs(100 + size + steps, 2, steps, 3, size)
    s0 = np.random.default_rng(size).standard_normal((2, 3, size, size)).astype(np.float32) * 0.3
    y, s = rwkv7_scan(*(_dev(x) for x in arrs), state=_dev(s0))
    ye, se = _oracle_wkv(arrs, s0)
    torch.cuda.synchronize()
    np.testing.assert_allclose(y.cpu().numpy(), ye.numpy(), rtol=RTOL, atol=ATOL)
    np.testing.assert_allclose(s.cpu().numpy(), se.numpy(), rtol=RTOL, atol=ATOL)


@pytest.mark.parametrize("wkv_kernel", ["chunked"], indirect=True)
@pytest.mark.parametrize("size", [8, 40])
def test_wkv7_many_heads_one_workgroup_each(size, wkv_kernel):
    """More than 128 heads (here 9 x 16 = 144) run one workgroup per head
    instead of two; with N = 40 (and N = 8) the last 16-key tile is half
    padding and takes the permuted half-tile form."""
    from yufmusicgen_amd.ops import rwkv7_scan

    print(f"wkv7 unsplit N={size}", flush=True)
    arrs = wkv_inputs(300 + size, 9, 37, 16, size)
    s0 = np.random.default_rng(size + 1).standard_normal((9, 16, size, size)).astype(np.float32) * 0.3
    y, s = rwkv7_scan(*(_dev(x) for x in arrs), state=_dev(s0))
    ye, se = _oracle_wkv(arrs, s0)
    torch.cuda.synchronize()
    np.testing.assert_allclose(y.cpu().numpy(), ye.numpy(), rtol=RTOL, atol=ATOL)
    np.testing.assert_allclose(s.cpu().numpy(), se.numpy(), rtol=RTOL, atol=ATOL)


@pytest.mark.parametrize("split", ["1", "2", "4"])
@pytest.mark.parametrize("size", [32, 40, 48, 64])
@pytest.mark.parametrize("steps", [1, 15, 33, 80])
def test_wkv7_split_heads(size, steps, split, monkeypatch):
    """A head over two workgroups or one per 16 value rows, of two to
    four tiles with a half or whole last one: the oracle's outputs and states, for the
    fewest chunks a pipeline of five can meet (one, ragged) and for several."""
    from yufmusicgen_amd.ops import rwkv7_scan

    print(f"wkv7 split={split} N={size} T={steps}", flush=True)
    monkeypatch.setenv("YUF_WKV7_KERNEL", "chunked")
    monkeypatch.setenv("YUF_WKV7_SPLIT", split)
    arrs = wkv_inputs(500 + size + steps, 2, steps, 5, size)
    s0 = np.random.default_rng(size + 7).standard_normal((2, 5, size, size)).astype(np.float32) * 0.3
    y, s = rwkv7_scan(*(_dev(x) for x in arrs), state=_dev(s0))
    ye, se = _oracle_wkv(arrs, s0)
    torch.cuda.synchronize()
    np.testing.assert_allclose(y.cpu().numpy(), ye.numpy(), rtol=RTOL, atol=ATOL)
    np.testing.assert_allclose(s.cpu().numpy(), se.numpy(), rtol=RTOL, atol=ATOL)


@pytest.mark.parametrize("size", [32, 40, 48, 64])
@pytest.mark.parametrize("steps", [33, 80])
def test_wkv7_forms_are_bit_identical(size, steps, monkeypatch):
    """Whole heads, two workgroups per head and one per 16 value rows sum in one
    order: how many heads a call brings, which chooses the form, does not change
    the bits of a head's outputs and state."""
    from yufmusicgen_amd.ops import rwkv7_scan

    print(f"wkv7 forms N={size} T={steps}", flush=True)
    monkeypatch.setenv("YUF_WKV7_KERNEL", "chunked")
    arrs = wkv_inputs(900 + size + steps, 2, steps, 3, size)
    s0 = np.random.default_rng(size).standard_normal((2, 3, size, size)).astype(np.float32) * 0.3
    got = []
    for split in ("0", "2", "4"):
        monkeypatch.setenv("YUF_WKV7_SPLIT", split)
        got.append(rwkv7_scan(*(_dev(x) for x in arrs), state=_dev(s0)))
    torch.cuda.synchronize()
    for y, s in got[1:]:
        assert torch.equal(y, got[0][0]) and torch.equal(s, got[0][1])


def test_wkv7_reference_golden(golden_dir):
    from yufmusicgen_amd.ops import rwkv7_scan

    z = np.load(os.path.join(golden_dir, "wkv7_ref.npz"))
    y, s = rwkv7_scan(*(_dev(z[n]) for n in ("r", "w_raw", "k", "v", "a", "b")), state=_dev(z["s0"]))
    np.testing.assert_allclose(y.cpu().numpy(), z["y"], rtol=RTOL, atol=ATOL)
    np.testing.assert_allclose(s.cpu().numpy(), z["s"], rtol=RTOL, atol=ATOL)


def test_wkv7_zero_state_matches_reference_entry():
    """rwkv7_cuda (zero start) equals the stateful call with an explicit zero state."""
    from yufmusicgen_amd.ops import rwkv7_cuda, rwkv7_scan

    arrs = [_dev(x) for x in wkv_inputs(7, 2, 33, 2, 40)]
    y0, s0 = rwkv7_cuda(*arrs)
    y1, s1 = rwkv7_scan(*arrs, state=torch.zeros(2, 2, 40, 40, device="cuda"))
    assert torch.equal(y0, y1) and torch.equal(s0, s1)


@pytest.mark.parametrize("wkv_kernel", KERNELS, indirect=True)
def test_wkv7_c2_full_size_parity_and_linearity(wkv_kernel):
    """C2 at its full size (B=8, T=2048, H=16, N=40) against the float64 oracle,
    plus linearity in v (a size-independent property)."""
    from yufmusicgen_amd.ops import rwkv7_scan

    print(f"wkv7 C2 full size kernel={wkv_kernel}", flush=True)
    arrs = wkv_inputs(0, 8, 2048, 16, 40)
    dev = [_dev(x) for x in arrs]
    y, s = rwkv7_scan(*dev)
    ye, se = _oracle_wkv(arrs)
    np.testing.assert_allclose(y.cpu().numpy(), ye.numpy(), rtol=RTOL, atol=ATOL)
    np.testing.assert_allclose(s.cpu().numpy(), se.numpy(), rtol=RTOL, atol=ATOL)
    v2 = torch.randn_like(dev[3])
    y2, s2 = rwkv7_scan(dev[0], dev[1], dev[2], v2, dev[4], dev[5])
    y3, s3 = rwkv7_scan(dev[0], dev[1], dev[2], dev[3] + v2, dev[4], dev[5])
    torch.testing.assert_close(y3, y + y2, rtol=1e-4, atol=1e-4)
    torch.testing.assert_close(s3, s + s2, rtol=1e-4, atol=1e-4)


@pytest.mark.parametrize("wkv_kernel", KERNELS, indirect=True)
def test_wkv7_chunked_continuation_equals_one_pass(wkv_kernel):
    """Splitting T across calls that carry the state (stateful prefill) equals one pass."""
    from yufmusicgen_amd.ops import rwkv7_scan

    dev = [_dev(x) for x in wkv_inputs(3, 2, 100, 4, 40)]
    y, s = rwkv7_scan(*dev)
    ya, sa = rwkv7_scan(*(x[:, :37].contiguous() for x in dev))
    yb, sb = rwkv7_scan(*(x[:, 37:].contiguous() for x in dev), state=sa)
    torch.testing.assert_close(torch.cat([ya, yb], 1), y, rtol=RTOL, atol=ATOL)
    torch.testing.assert_close(sb, s, rtol=RTOL, atol=ATOL)


def test_wkv7_delta_rule_write_property():
    """Unit decay, a = -kappa, b = k = kappa: after each token S kappa = v."""
    from yufmusicgen_amd.ops import rwkv7_scan

    r, _, _, v, a, _ = wkv_inputs(9, 2, 12, 2, 40)
    kappa = -a
    w = np.full_like(r, -80.0)
    state = None
    for t in range(12):
        sl = slice(t, t + 1)
        args = [_dev(x[:, sl]) for x in (r, w, kappa, v, a, kappa)]
        _, state = rwkv7_scan(*args, state=state)
        mapped = torch.einsum("bhij,bhj->bhi", state, _dev(kappa[:, t]))
        torch.testing.assert_close(mapped, _dev(v[:, t]), rtol=1e-4, atol=1e-4)


@pytest.mark.parametrize("dim", [12, 32, 128, 256, 512, 1000])
@pytest.mark.parametrize("steps", [1, 19, 64])
@pytest.mark.parametrize("gated", [False, True])
def test_rosa_matches_oracle(dim, steps, gated):
    from yufmusicgen_amd.ops import rosa_householder_scan

    print(f"rosa parity D={dim} T={steps} gated={gated}", flush=True)
    cand, write, read_raw, decay, u = rosa_inputs(dim + steps, 3, steps, dim)
    m0 = np.random.default_rng(dim).standard_normal((3, dim)).astype(np.float32)
    read, m = rosa_householder_scan(*(_dev(x) for x in (cand, write, read_raw, decay, u, m0)), gated=gated)
    t64 = [torch.from_numpy(x.astype(np.float64)) for x in (cand, write, read_raw, decay, u, m0)]
    re, me = orosa.rosa_scan(*t64, gated=gated)
    np.testing.assert_allclose(read.cpu().numpy(), re.numpy(), rtol=RTOL, atol=ATOL)
    np.testing.assert_allclose(m.cpu().numpy(), me.numpy(), rtol=RTOL, atol=ATOL)


def test_rosa_reference_golden(golden_dir):
    from yufmusicgen_amd.ops import rosa_householder_scan

    z = np.load(os.path.join(golden_dir, "rosa_ref.npz"))
    args = [_dev(z[n]) for n in ("cand", "write", "read_raw", "decay", "direction", "m0")]
    read, m = rosa_householder_scan(*args, gated=True)
    np.testing.assert_allclose(read.cpu().numpy(), z["read"], rtol=RTOL, atol=ATOL)
    np.testing.assert_allclose(m.cpu().numpy(), z["m"], rtol=RTOL, atol=ATOL)


@pytest.mark.parametrize("decay_value", [None, 0.99, 0.05])
def test_rosa_full_size(decay_value):
    """C3 shape (B=8, T=2048, D=128, gated), with the drawn decays and with
    every decay pinned at 0.99 (slow memory) and 0.05 (fast memory).  At 0.999
    even an exact-order float32 recurrence leaves elements outside 1e-4/1e-5."""
    from yufmusicgen_amd.ops import rosa_householder_scan

    print(f"rosa full size decay={decay_value}", flush=True)
    cand, write, read_raw, decay, u = rosa_inputs(11, 8, 2048, 128)
    if decay_value is not None:
        decay = np.full_like(decay, decay_value)
    m0 = np.random.default_rng(5).standard_normal((8, 128)).astype(np.float32)
    arrs = (cand, write, read_raw, decay, u, m0)
    read, m = rosa_householder_scan(*(_dev(x) for x in arrs), gated=True)
    re, me = orosa.rosa_scan(*(torch.from_numpy(x.astype(np.float64)) for x in arrs), gated=True)
    np.testing.assert_allclose(read.cpu().numpy(), re.numpy(), rtol=RTOL, atol=ATOL)
    np.testing.assert_allclose(m.cpu().numpy(), me.numpy(), rtol=RTOL, atol=ATOL)


@pytest.mark.parametrize("dim,steps,gated", [(64, 128, True), (64, 320, True), (128, 640, False), (256, 256, True),
                                             (256, 1088, False), (128, 2048, True)])
def test_rosa_segmented_operator(dim, steps, gated, monkeypatch):
    """The operator's segment form (D in {64, 128, 256}: one segment up to 192
    tokens; above, A^64 or A^128 built on the device in double, segments from
    zero, then each from its start state) against the float64 oracle and
    against the sequential scan (YUF_ROSA_SEGMENTED=0), from a non-zero memory."""
    from yufmusicgen_amd.ops import rosa_householder_scan

    print(f"rosa segmented D={dim} T={steps} gated={gated}", flush=True)
    cand, write, read_raw, decay, u = rosa_inputs(12 + dim, 3, steps, dim)
    m0 = np.random.default_rng(6).standard_normal((3, dim)).astype(np.float32)
    arrs = (cand, write, read_raw, decay, u, m0)
    read, m = rosa_householder_scan(*(_dev(x) for x in arrs), gated=gated)
    re, me = orosa.rosa_scan(*(torch.from_numpy(x.astype(np.float64)) for x in arrs), gated=gated)
    np.testing.assert_allclose(read.cpu().numpy(), re.numpy(), rtol=RTOL, atol=ATOL)
    np.testing.assert_allclose(m.cpu().numpy(), me.numpy(), rtol=RTOL, atol=ATOL)
    monkeypatch.setenv("YUF_ROSA_SEGMENTED", "0")
    read_s, m_s = rosa_householder_scan(*(_dev(x) for x in arrs), gated=gated)
    np.testing.assert_allclose(read.cpu().numpy(), read_s.cpu().numpy(), rtol=RTOL, atol=ATOL)
    np.testing.assert_allclose(m.cpu().numpy(), m_s.cpu().numpy(), rtol=RTOL, atol=ATOL)


def test_rosa_chunked_continuation():
    """Scanning T tokens in ragged pieces, carrying the memory, equals one scan."""
    from yufmusicgen_amd.ops import rosa_householder_scan

    cand, write, read_raw, decay, u = rosa_inputs(4, 2, 100, 128)
    m = torch.zeros(2, 128, device="cuda")
    full, m_full = rosa_householder_scan(*(_dev(x) for x in (cand, write, read_raw, decay, u)), m, gated=True)
    outs = []
    for lo, hi in ((0, 7), (7, 40), (40, 41), (41, 100)):
        piece = [_dev(x[:, lo:hi]) for x in (cand, write, read_raw)]
        r, m = rosa_householder_scan(*piece, _dev(decay), _dev(u), m, gated=True)
        outs.append(r)
    torch.testing.assert_close(torch.cat(outs, dim=1), full, rtol=RTOL, atol=ATOL)
    torch.testing.assert_close(m, m_full, rtol=RTOL, atol=ATOL)


@pytest.mark.parametrize("dim", [64, 128, 256])
@pytest.mark.parametrize("steps", [2, 8, 9, 31, 33, 192, 193, 320, 641, 1111, 4161])
def test_rosa_segments(dim, steps):
    """The segment kernel at the edges of its range (above 8 tokens at D = 256), of
    its 32-token chunks and of its segment rule (one segment up to 192 tokens, 64- then 128-token segments with a ragged
    last one, the separate carry pass above 32 segments), gated and not, against
    the float64 oracle, with the memory updated in place."""
    from yufmusicgen_amd._lib import check, lib

    print(f"rosa segments D={dim} T={steps}", flush=True)
    batch = 2
    cand, write, read_raw, decay, u = (_dev(x) for x in rosa_inputs(31 + dim, batch, steps, dim))
    m0 = np.random.default_rng(8).standard_normal((batch, dim)).astype(np.float32)
    t64 = [x.cpu().double() for x in (cand, write, read_raw, decay, u)] + [torch.from_numpy(m0).double()]
    for gated in (True, False):
        mem, out = _dev(m0), torch.full((batch, steps, dim), float("nan"), device="cuda")
        check(lib().yuf_rosa_scan_f32(batch, steps, dim, cand.data_ptr(), write.data_ptr(),
                                      read_raw.data_ptr() if gated else None, decay.data_ptr(), u.data_ptr(),
                                      mem.data_ptr(), mem.data_ptr(), out.data_ptr(),
                                      torch.cuda.current_stream().cuda_stream))
        torch.cuda.synchronize()
        re, me = orosa.rosa_scan(*t64, gated=gated)
        np.testing.assert_allclose(out.cpu().numpy(), re.numpy(), rtol=RTOL, atol=ATOL)
        np.testing.assert_allclose(mem.cpu().numpy(), me.numpy(), rtol=RTOL, atol=ATOL)


@pytest.mark.parametrize("dim", [64, 128, 256])
@pytest.mark.parametrize("steps", [33, 705])
def test_rosa_nearly_closed_write_gates(dim, steps):
    """Write gates down to sigmoid(-80) (1e-35) with saturated candidates: the
    inputs stay what they are instead of vanishing, so reads and memory follow
    the float64 oracle to 3e-5 of their largest value (e^{-80} in fp32 is good to
    |w| 2^-23 = 1e-5; the state is a sum of such values, 1e3 and more above the
    smallest normal number)."""
    from yufmusicgen_amd.ops import rosa_householder_scan

    print(f"rosa closed gates D={dim} T={steps}", flush=True)
    cand, write, read_raw, decay, u = rosa_inputs(91 + dim, 2, steps, dim)
    cand = np.sign(cand + 0.01).astype(np.float32) * 12.0
    write = (-70.0 - 10.0 * np.random.default_rng(4).random(write.shape)).astype(np.float32)
    args = [cand, write, read_raw, decay, u, np.zeros((2, dim), dtype=np.float32)]
    out, mem = rosa_householder_scan(*(_dev(x) for x in args), gated=False)
    torch.cuda.synchronize()
    re, me = orosa.rosa_scan(*(torch.from_numpy(np.asarray(x)).double() for x in args), gated=False)
    for got, want in ((out, re), (mem, me)):
        assert float(want.abs().max()) > 1e-32
        assert float((got.cpu().double() - want).abs().max()) <= 3e-5 * float(want.abs().max())


def _rosa_call(args, mem, out, gated, stream):
    from yufmusicgen_amd._lib import check, lib

    cand, write, read_raw, decay, u = args
    batch, steps, dim = cand.shape
    check(lib().yuf_rosa_scan_f32(batch, steps, dim, cand.data_ptr(), write.data_ptr(),
                                  read_raw.data_ptr() if gated else None, decay.data_ptr(), u.data_ptr(),
                                  mem.data_ptr(), mem.data_ptr(), out.data_ptr(), stream))


@pytest.mark.parametrize("steps", [640, 1100])
def test_rosa_operator_under_capture(steps):
    """The operator captured into a graph, on a stream that has a scratch buffer
    and on one that has none, and replayed between eager calls on the capturing
    stream that outgrow every buffer (ragged and whole lengths): each replay
    gives the eager call's result -- bit for bit at a multiple of 64, where both
    run in segments, and to the tolerance of the scans at a ragged length, which
    a graph runs as one segment."""
    dim = 128
    args = [_dev(x) for x in rosa_inputs(77, 2, steps, dim)]
    m0 = _dev(np.random.default_rng(3).standard_normal((2, dim)).astype(np.float32))
    torch.cuda.synchronize()
    for warm in (True, False):
        print(f"rosa capture T={steps} warm={warm}", flush=True)
        st = torch.cuda.Stream()
        mem, out = m0.clone(), torch.full((2, steps, dim), float("nan"), device="cuda")
        torch.cuda.synchronize()
        with torch.cuda.stream(torch.cuda.current_stream() if not warm else st):
            _rosa_call(args, mem, out, True, torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        want, want_mem = out.clone(), mem.clone()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=st):
            _rosa_call(args, mem, out, True, st.cuda_stream)
        for i, (batch, length) in enumerate(((2, 1111), (4, 2048), (8, 4161))):
            big = [_dev(x) for x in rosa_inputs(i, batch, length, dim)]
            big_mem, big_out = torch.zeros(batch, dim, device="cuda"), torch.empty(batch, length, dim, device="cuda")
            mem.copy_(m0)
            out.fill_(float("nan"))
            torch.cuda.synchronize()
            _rosa_call(big, big_mem, big_out, True, st.cuda_stream)
            with torch.cuda.stream(st):
                graph.replay()
            torch.cuda.synchronize()
            if steps % 64 == 0:
                assert torch.equal(out, want) and torch.equal(mem, want_mem), i
            else:
                torch.testing.assert_close(out, want, rtol=RTOL, atol=ATOL)
                torch.testing.assert_close(mem, want_mem, rtol=RTOL, atol=ATOL)
            assert torch.isfinite(big_out).all()


@pytest.mark.parametrize("shared", ["stream", "per_thread_default"])
def test_rosa_operator_from_several_threads(shared):
    """Two host threads call the operator at lengths that need scratch, on one
    stream and on the per-thread default stream (one handle, a stream per
    thread): every call gives the result of the same call alone."""
    import threading

    print(f"rosa threads {shared}", flush=True)
    dim = 128
    jobs = []
    for seed, steps in ((5, 1100), (6, 705)):
        args = [_dev(x) for x in rosa_inputs(seed, 2, steps, dim)]
        mem, out = torch.zeros(2, dim, device="cuda"), torch.empty(2, steps, dim, device="cuda")
        torch.cuda.synchronize()
        _rosa_call(args, mem, out, True, torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        reps = [(torch.zeros(2, dim, device="cuda"), torch.empty(2, steps, dim, device="cuda")) for _ in range(40)]
        jobs.append((args, mem, out, reps))
    st = torch.cuda.Stream()
    handle = st.cuda_stream if shared == "stream" else 2  # hipStreamPerThread
    torch.cuda.synchronize()
    errors = []

    def work(args, reps):
        try:
            for mem, out in reps:
                _rosa_call(args, mem, out, True, handle)
        except Exception as exc:  # noqa: BLE001 - reported below
            errors.append(exc)

    threads = [threading.Thread(target=work, args=(args, reps)) for args, _, _, reps in jobs]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert not errors, errors
    for _, mem, out, reps in jobs:
        for i, (m, o) in enumerate(reps):
            assert torch.equal(m, mem) and torch.equal(o, out), i
