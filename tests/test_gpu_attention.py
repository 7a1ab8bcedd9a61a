"""GPU parity of the relative-position attention core
(mynah_asr_hip_relpos_attention_dev) against the oracle's float64 restatement
of src/encoder.c:315-410 (full) and :220-313 (chunked-limited).

Bar: |ctx - ref| <= 1e-4*|ref| + 1e-5*max|v| per element. The kernels compute
in f32 like the reference, with another summation order and base-2
exponentials (full attention forms its products from f16 hi + lo splits of
scaled operands, 22 bits of each row's, or V tile column's, maximum), so a
context element near zero (a cancelling weighted sum of v) carries an absolute
error of order 1e-6 * max|v| — the scale term covers that. A row of a chunked
window depends on the keys it sees alone: bit for bit.
Inputs: q, k, v, rk N(0, 1) and bias_u, bias_v N(0, 0.1), seeded.
"""
import sys

import numpy as np
import pytest

import mynah_hip as M
from attention import relpos_attention

pytestmark = pytest.mark.gpu
RTOL, VTOL = 1e-4, 1e-5


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def make(seed, T, d, nseq=1):
    r = np.random.default_rng(seed)
    f = lambda *s, sc=1.0: (r.standard_normal(s) * sc).astype(np.float32)
    return (f(nseq, T, d), f(nseq, T, d), f(nseq, T, d), f(2 * T - 1, d), f(d, sc=0.1), f(d, sc=0.1))


def run_gpu(gpu, arrs, T, d, H, left, right, nseq):
    import torch
    q, k, v, rk, bu, bv = (torch.from_numpy(a).cuda() for a in arrs)
    ctx = torch.full((nseq, T, d), float("nan"), dtype=torch.float32, device="cuda")
    torch.cuda.synchronize()
    M.relpos_attention_dev(gpu, q.data_ptr(), k.data_ptr(), v.data_ptr(), rk.data_ptr(), bu.data_ptr(),
                           bv.data_ptr(), ctx.data_ptr(), T, d, H, left, right, nseq)
    torch.cuda.synchronize()
    return ctx.cpu().numpy()


def check(out, arrs, H, left, right):
    q, k, v, rk, bu, bv = arrs
    for s in range(q.shape[0]):
        ref = relpos_attention(q[s], k[s], v[s], rk, bu, bv, H, left, right)
        err = np.abs(out[s] - ref)
        lim = RTOL * np.abs(ref) + VTOL * np.abs(v[s]).max()
        assert np.isfinite(out[s]).all()
        assert (err <= lim).all(), (f"seg {s}: {int((err > lim).sum())} outside, max err {err.max():.3g}, "
                                    f"worst ratio {(err / lim).max():.3g}")


@pytest.mark.parametrize("T,d,H,left,right,nseq", [
    (1, 128, 2, -1, 0, 1),        # one frame
    (37, 128, 2, -1, 0, 1),       # dk 64, ragged tiles
    (64, 256, 2, -1, 0, 1),       # dk 128, one exact row block
    (65, 256, 2, -1, 0, 2),       # one row past a block, two segments
    (130, 256, 2, 32, 7, 1),      # chunked: chunk 8, 4 chunks of left context
    (130, 256, 2, 4, 3, 3),       # chunked: chunk 4, one chunk of left context
    (200, 512, 4, 0, 0, 1),       # chunk 1, no left context: each row sees itself only
    (300, 256, 4, 70, 13, 1),     # chunk 14, lc 5, T not a multiple of the chunk
    (300, 512, 4, 1000, 299, 1),  # one chunk covering all rows: equals full attention
])
def test_relpos_attention_matches_oracle(gpu, T, d, H, left, right, nseq):
    say("attention", T, d, H, left, right, nseq)
    arrs = make(T * 7 + d, T, d, nseq)
    out = run_gpu(gpu, arrs, T, d, H, left, right, nseq)
    check(out, arrs, H, left, right)


def test_relpos_attention_fastconformer_segment(gpu):
    """FastConformer-0.6B: d_model 1024, 8 heads (dk 128), one 750-frame
    segment, full attention and the streaming chunked-limited window."""
    T, d, H = 750, 1024, 8
    arrs = make(11, T, d, 2)
    for left, right in ((-1, 0), (70, 13)):
        say("attention fastconformer", T, left, right)
        out = run_gpu(gpu, arrs, T, d, H, left, right, 2)
        check(out, arrs, H, left, right)


@pytest.mark.parametrize("d", [256, 128])
def test_relpos_attention_many_segments(gpu, d):
    """More (query block, head, segment) workgroups than the chip holds at once, dk 128 and 64."""
    T, H, nseq = 200, 2, 128
    say("attention many segments", T, d, H, nseq)
    arrs = make(21 + d, T, d, nseq)
    out = run_gpu(gpu, arrs, T, d, H, -1, 0, nseq)
    check(out, arrs, H, -1, 0)


@pytest.mark.parametrize("left,right", [(-1, 0), (1000, 299)])
def test_relpos_attention_wide_row_scales(gpu, left, right):
    """Rows of q, k and rk scaled by 2^-30 .. 2^30, rows of zeros, and rows
    with one feature 1e4 times the rest; V's features scaled by 2^-20 .. 2^20
    with a zero key tile: the split operands carry each row's (V: each key
    tile and feature's) own scale, so the bar holds as for N(0, 1) inputs
    (full attention on the split path, and the one-chunk window, the same
    products on the f32 path)."""
    T, d, H = 150, 256, 2
    r = np.random.default_rng(77)
    q, k, v, rk, bu, bv = make(41, T, d, 1)
    for a, n in ((q[0], T), (k[0], T), (rk, 2 * T - 1)):
        a *= np.exp2(r.integers(-30, 31, size=(n, 1))).astype(np.float32)
        a[r.integers(0, n, size=5)] = 0.0
        a[r.integers(0, n, size=5), r.integers(0, d, size=5)] *= 1e4
    # V: features scaled by 2^-20 .. 2^20 (its split carries one exponent per
    # key tile and feature), a zero tile of keys, zero rows
    v[0] *= np.exp2(r.integers(-20, 21, size=(1, d))).astype(np.float32)
    v[0, 32:64] = 0.0
    v[0, r.integers(0, T, size=5)] = 0.0
    bu[:] = 0.0
    bv[:] = 0.0
    say("attention wide row scales", left, right)
    arrs = (q, k, v, rk, bu, bv)
    out = run_gpu(gpu, arrs, T, d, H, left, right, 1)
    # the bar per feature: a context column's error scales with that column of V
    ref = relpos_attention(q[0], k[0], v[0], rk, bu, bv, H, left, right)
    err = np.abs(out[0] - ref)
    lim = RTOL * np.abs(ref) + VTOL * np.abs(v[0]).max(axis=0, keepdims=True)
    assert np.isfinite(out[0]).all()
    assert (err <= lim).all(), f"{int((err > lim).sum())} outside, worst ratio {(err / lim).max():.3g}"


@pytest.mark.parametrize("left,right", [(-1, 0), (20, 6)])
def test_relpos_attention_segments_independent(gpu, left, right):
    """A segment's context does not depend on the other segments of the call
    (bit-identical to running it alone)."""
    T, d, H = 97, 256, 2
    for nseq in (3, 256):   # fewer and more workgroups than the chip holds at once
        arrs = make(5, T, d, nseq)
        many = run_gpu(gpu, arrs, T, d, H, left, right, nseq)
        one = run_gpu(gpu, tuple(a[1:2] if a.ndim == 3 else a for a in arrs), T, d, H, left, right, 1)
        assert np.array_equal(many[1].view(np.uint32), one[0].view(np.uint32))


@pytest.mark.parametrize("d,H", [(128, 2), (256, 2)], ids=["dk64", "dk128"])
@pytest.mark.parametrize("left,right", [(0, 0), (4, 3), (70, 13), (0, 31)])
def test_relpos_attention_hidden_keys(gpu, d, H, left, right):
    """Keys outside a row's window, 2^20 (v) and 2^4 (k) times the visible ones,
    in the same key tiles: the row's context keeps its bits, and its bar is
    that of the values it sees."""
    T, chunk = 150, right + 1
    say("attention hidden keys", d, H, left, right)
    arrs = make(91, T, d, 1)
    plain = run_gpu(gpu, arrs, T, d, H, left, right, 1)[0]
    for c in (0, (T // chunk) // 2, (T - 1) // chunk):
        j0, j1 = max((c - left // chunk) * chunk, 0), min((c + 1) * chunk, T)
        rows = slice(c * chunk, j1)
        q, k, v, rk, bu, bv = (a.copy() for a in arrs)
        hidden = np.ones(T, bool)
        hidden[j0:j1] = False
        v[0, hidden] *= np.float32(2.0 ** 20)
        k[0, hidden] *= np.float32(16.0)
        got = run_gpu(gpu, (q, k, v, rk, bu, bv), T, d, H, left, right, 1)[0]
        assert np.array_equal(got[rows].view(np.uint32), plain[rows].view(np.uint32)), f"chunk {c}"
        ref = relpos_attention(q[0], k[0], v[0], rk, bu, bv, H, left, right)[rows]
        lim = RTOL * np.abs(ref) + VTOL * np.abs(v[0, j0:j1]).max()
        assert (np.abs(got[rows] - ref) <= lim).all(), f"chunk {c}"


def _window_calls(gpu, torch, n, T, d, H, nseq):
    """n sets of inputs on the GPU, and the call of set i on a stream."""
    sets, out = [], []
    for i in range(n):
        sets.append([torch.from_numpy(a).cuda() for a in make(200 + i, T, d, nseq)])
        out.append(torch.zeros((nseq, T, d), dtype=torch.float32, device="cuda"))

    def call(i, stream):
        M.relpos_attention_dev(gpu, *(a.data_ptr() for a in sets[i]), out[i].data_ptr(), T, d, H, 70, 13, nseq,
                               stream=stream.cuda_stream)
    return call, out, sets


def test_relpos_attention_window_on_two_streams(gpu):
    """Chunked-window calls of one thread on two streams, not ordered with each
    other, give the bits of the calls alone."""
    import torch
    say("attention windows on two streams")
    call, out, _sets = _window_calls(gpu, torch, 2, 750, 1024, 8, 4)
    ss = [torch.cuda.Stream(), torch.cuda.Stream()]
    torch.cuda.synchronize()
    alone = []
    for i in range(2):
        call(i, ss[0])
        torch.cuda.synchronize()
        alone.append(out[i].clone())
        out[i].zero_()
    torch.cuda.synchronize()
    for rep in range(10):
        for i in range(2):
            call(i, ss[i])
    torch.cuda.synchronize()
    for i in range(2):
        assert torch.equal(out[i].view(torch.int32), alone[i].view(torch.int32))


def test_relpos_attention_window_captured(gpu):
    """Chunked-window calls larger than any before them in their thread are
    captured (nothing is allocated), and two such graphs replayed at once on two
    streams give the eager calls' bits, replay after replay."""
    import threading
    import torch
    say("attention windows captured")
    call, out, _sets = _window_calls(gpu, torch, 2, 600, 512, 4, 4)
    small, _o, _s = _window_calls(gpu, torch, 1, 1, 256, 2, 1)
    graphs, errs = [], []
    ss = [torch.cuda.Stream(), torch.cuda.Stream()]
    torch.cuda.synchronize()

    def capture():
        try:
            small(0, ss[0])   # (the thread's first call)
            torch.cuda.synchronize()
            for i in range(2):
                g = torch.cuda.CUDAGraph()
                with torch.cuda.graph(g, stream=ss[i]):
                    call(i, torch.cuda.current_stream())
                graphs.append(g)
        except Exception as e:   # (reported by the test's own thread)
            errs.append(e)

    t = threading.Thread(target=capture)
    t.start()
    t.join()
    assert not errs, errs
    eager = []
    for i in range(2):
        call(i, ss[0])
        torch.cuda.synchronize()
        eager.append(out[i].clone())
    for rep in range(3):
        for o in out:
            o.zero_()
        torch.cuda.synchronize()
        for i in range(2):
            with torch.cuda.stream(ss[i]):
                graphs[i].replay()
        torch.cuda.synchronize()
        for i in range(2):
            assert torch.equal(out[i].view(torch.int32), eager[i].view(torch.int32)), f"replay {rep}, graph {i}"


def test_relpos_attention_host_entry(gpu):
    """The host-pointer entry point gives the device entry point's bits."""
    T, d, H = 150, 256, 2
    arrs = make(31, T, d, 1)
    for left, right in ((-1, 0), (20, 4)):
        dev = run_gpu(gpu, arrs, T, d, H, left, right, 1)[0]
        q, k, v, rk, bu, bv = arrs
        host = M.host_relpos_attention(gpu, q[0], k[0], v[0], rk, bu, bv, H, left, right)
        assert np.array_equal(host.view(np.uint32), dev.view(np.uint32))


def test_relpos_attention_rejects_bad_arguments(gpu):
    import torch
    x = torch.zeros((4, 192), dtype=torch.float32, device="cuda")
    p = x.data_ptr()
    with pytest.raises(RuntimeError, match="head size"):
        M.relpos_attention_dev(gpu, p, p, p, p, p, p, x[1:].data_ptr(), 1, 192, 2)   # dk 96
    with pytest.raises(RuntimeError, match="right"):
        M.relpos_attention_dev(gpu, p, p, p, p, p, p, x[1:].data_ptr(), 1, 128, 2, 4, -1)
    with pytest.raises(RuntimeError, match="alias"):
        M.relpos_attention_dev(gpu, p, p, p, p, p, p, p, 1, 128, 2)


@pytest.mark.parametrize("T", [1, 31, 32, 33, 64, 65, 129, 257])
@pytest.mark.parametrize("d,H", [(128, 2), (256, 2)], ids=["dk64", "dk128"])
@pytest.mark.parametrize("left,right", [(-1, 0), (0, 0), (3, 1), (64, 31), (70, 13), (100000, 0)])
def test_relpos_attention_tile_edges(gpu, T, d, H, left, right):
    """Lengths around the 32-row tiles; windows narrower than a tile, as wide as
    one, and wider than the segment (fewer key tiles than waves, one wave's
    tiles, waves with none)."""
    say("attention tile edges", T, d, H, left, right)
    arrs = make(1000 + T, T, d, 2)
    check(run_gpu(gpu, arrs, T, d, H, left, right, 2), arrs, H, left, right)
