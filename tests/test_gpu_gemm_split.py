"""fp32 products of more than 8 rows through `automatic`, where it splits both
operands into bf16 terms (csrc/gemm_split.hip), against 64-bit products.

Bound per element: every MFMA adds its 32 products to an fp32 accumulator
with at most two roundings of 2^-24 each at the size of the sums so far, and
six terms a chunk in two accumulators of which only hi * hi is full size; the
slices' sum and the prior C add one each, the left-out terms at most one. So
(k / 16 + 24) * 2^-24 * sum |a||b| holds with room (the sums are rarely at
their largest throughout)."""
import ctypes
import threading

import numpy as np
import pytest
import torch

from tests import engine, inputs

em = engine.load()
pytestmark = pytest.mark.gpu


def dev(x):
    return torch.from_numpy(x).cuda()


def check(got, A, B, C0=None):
    k = A.shape[1]
    want = A.astype(np.float64) @ B.astype(np.float64)
    scale = np.abs(A).astype(np.float64) @ np.abs(B).astype(np.float64)
    if C0 is not None:
        want, scale = want + C0, scale + np.abs(C0)
    err = np.abs(got.astype(np.float64) - want)
    assert (err <= (k / 16 + 24) * 2.0 ** -24 * scale + 2.0 ** -149).all(), (err / scale).max()


# Rows around every tile height, k whole and ragged chunks (the last one
# overlapping the one before), columns off a tile, off a float4 and narrow.
SHAPES = [(9, 1000, 1100), (32, 1028, 1500), (33, 1156, 1000), (64, 4096, 300), (65, 36, 40000),
          (97, 2000, 700), (128, 1060, 1027), (129, 1000, 1153), (161, 1124, 1000),
          (193, 1500, 1001), (257, 2048, 1030), (320, 1100, 1000), (321, 1092, 2049),
          (513, 1028, 2000), (40, 44, 30001), (1100, 32, 40000)]


@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_tile_edges(shape):
    m, k, n = shape
    A = inputs.uniform((m, k), -1.0, 1.0, 71)
    B = inputs.uniform((k, n), -1.0, 1.0, 72)
    C0 = inputs.uniform((m, n), -4.0, 4.0, 73)
    first = em.matmul(dev(A), dev(B))
    check(first.cpu().numpy(), A, B)
    assert torch.equal(first, em.matmul(dev(A), dev(B)))
    C = dev(C0.copy())
    em.matmul(dev(A), dev(B), C, accumulate=True)
    check(C.cpu().numpy(), A, B, C0)
    # C off a 16-byte boundary: scalar stores of the same sums.
    flat = torch.empty(m * n + 1, device="cuda")
    off = flat[1:].view(m, n)
    em.matmul(dev(A), dev(B), off)
    assert torch.equal(off, first)


# A few narrow tiles of a deep k: tens of k slices, the last ones short.
@pytest.mark.parametrize("shape", [(9, 13000, 200), (12, 10912, 128), (33, 12004, 97), (64, 9000, 520)],
                         ids=str)
def test_many_slices(shape):
    m, k, n = shape
    A, B = inputs.uniform((m, k), -1.0, 1.0, 87), inputs.uniform((k, n), -1.0, 1.0, 88)
    C0 = inputs.uniform((m, n), -4.0, 4.0, 89)
    first = em.matmul(dev(A), dev(B))
    check(first.cpu().numpy(), A, B)
    assert torch.equal(first, em.matmul(dev(A), dev(B)))
    C = dev(C0.copy())
    em.matmul(dev(A), dev(B), C, accumulate=True)
    check(C.cpu().numpy(), A, B, C0)


@pytest.mark.parametrize("exponent", [-100, -115, -126, 40])
def test_magnitudes(exponent):
    # Below 2^-109 a lo term drops bits; the product must not. With B scaled
    # the other way the sums stay normal numbers.
    m, k, n = 70, 1100, 1200
    A = (inputs.uniform((m, k), 1.0, 2.0, 74) * 2.0 ** exponent).astype(np.float32)
    A[::2] = inputs.uniform((m, k), -1.0, 1.0, 75)[::2]
    B = (inputs.uniform((k, n), -1.0, 1.0, 76) * 2.0 ** (20 if exponent < 0 else -100)).astype(np.float32)
    check(em.matmul(dev(A), dev(B)).cpu().numpy(), A, B)
    check(em.matmul(dev(np.ascontiguousarray(B.T)), dev(np.ascontiguousarray(A.T))).cpu().numpy(),
          B.T, A.T)


@pytest.mark.parametrize("exponent", [-112, -126])
@pytest.mark.parametrize("shape", [(70, 1100, 1200), (300, 1028, 1001)], ids=str)
def test_dropped_bits_times_large_values(shape, exponent):
    # The bits a lo term drops below 2^-109 times values near 2^100 would show
    # in sums far above the smallest.
    m, k, n = shape
    A = inputs.uniform((m, k), 1.0, 2.0, 81) * np.float32(2.0 ** exponent)
    B = inputs.uniform((k, n), 1.0, 2.0, 82) * np.float32(2.0 ** 100)
    check(em.matmul(dev(A), dev(B)).cpu().numpy(), A, B)
    Bt, At = np.ascontiguousarray(B.T), np.ascontiguousarray(A.T)
    check(em.matmul(dev(Bt), dev(At)).cpu().numpy(), Bt, At)


def test_non_finite_values():
    m, k, n = 130, 1100, 1200
    A = inputs.uniform((m, k), 0.5, 1.0, 77)
    B = inputs.uniform((k, n), 0.5, 1.0, 78)
    A[3, 5], A[70, 1099], B[7, 11], B[1098, 1199] = np.inf, -np.inf, np.inf, np.nan
    A[5, 9] = np.float32(3.4e38)  # rounds up to infinity as a bf16
    with np.errstate(invalid="ignore"):
        want = A.astype(np.float64) @ B.astype(np.float64)
    got = em.matmul(dev(A), dev(B)).cpu().numpy()
    over = np.abs(want) > np.finfo(np.float32).max  # past fp32: +inf
    want[over & np.isfinite(want)] = np.inf
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(got[np.isinf(want)], want[np.isinf(want)].astype(np.float32))
    fine = np.isfinite(want)
    assert np.allclose(got[fine], want[fine], rtol=1e-5)


def test_threads_on_one_stream():
    # A product's slices and their sum are two launches over the stream's
    # buffer: no other thread's product comes between them.
    m, k, n = 200, 4096, 1024
    A, B = dev(inputs.uniform((m, k), -1, 1, 83)), dev(inputs.uniform((k, n), -1, 1, 84))
    As = [A * (i + 1) for i in range(4)]
    want = [em.matmul(a, B) for a in As]
    outs = [[torch.empty_like(want[i]) for _ in range(100)] for i in range(4)]
    torch.cuda.synchronize()

    def work(i):
        for out in outs[i]:
            em.matmul(As[i], B, out)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    [t.start() for t in threads]
    [t.join() for t in threads]
    torch.cuda.synchronize()
    assert all(torch.equal(out, want[i]) for i in range(4) for out in outs[i])


def test_streams_and_threads_share_nothing():
    # Sliced products on four threads with a stream each, and a graph captured
    # without a call before it: every result equals the first stream's.
    m, k, n = 200, 4096, 1024
    A, B = dev(inputs.uniform((m, k), -1, 1, 79)), dev(inputs.uniform((k, n), -1, 1, 80))
    As = [A * (i + 1) for i in range(4)]
    want = [em.matmul(a, B).clone() for a in As]
    torch.cuda.synchronize()
    bad = []

    def work(i):
        s = torch.cuda.Stream()
        with torch.cuda.stream(s):
            for _ in range(40):
                if not torch.equal(em.matmul(As[i], B), want[i]):
                    bad.append(i)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    [t.start() for t in threads]
    [t.join() for t in threads]
    assert not bad
    out = [torch.zeros((m, n), device="cuda") for _ in range(2)]
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        em.matmul(As[0], B, out[0])
        em.matmul(As[1], B, out[1])
    for _ in range(3):
        out[0].zero_(), out[1].zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out[0], want[0]) and torch.equal(out[1], want[1])
        em.matmul(As[2], B)


def test_left_out_terms_of_one_sign():
    # 0x1.00ff8p+0 = 1 + 2^-8 - 2^-17: mid and lo at their largest, and every
    # left-out sum 2^-24 of its product and of one sign.
    for m, k, n in [(9, 32, 40000), (300, 1028, 1001), (200, 4096, 1024)]:
        A = np.full((m, k), float.fromhex("0x1.00ff8p+0"), np.float32)
        B = np.full((k, n), float.fromhex("0x1.00ff8p+0"), np.float32)
        check(em.matmul(dev(A), dev(B)).cpu().numpy(), A, B)
        check(em.matmul(dev(A), dev(-B)).cpu().numpy(), A, -B)


def test_captures_threads_and_streams_give_their_slices_back():
    # Graphs captured and destroyed, threads that ran on their own default
    # stream and ended, and more streams than keep a buffer: none changes what
    # any product gives, and the memory stays bounded.
    m, k, n = 200, 4096, 1024
    A, B = dev(inputs.uniform((m, k), -1, 1, 85)), dev(inputs.uniform((k, n), -1, 1, 86))
    A2 = A * 2
    want, want2 = em.matmul(A, B), em.matmul(A2, B)
    out, out2 = torch.empty_like(want), torch.empty_like(want)
    torch.cuda.synchronize()

    def capture(a, o):
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            em.matmul(a, B, o)
        return g

    def replay(g, o, w):
        o.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(o, w)

    def captures(count):
        kept = capture(A2, out2)
        for _ in range(count):
            replay(capture(A, out), out, want)
        replay(kept, out2, want2)

    def product(stream, mine):
        em.matmul_f32_raw(m, n, k, A.data_ptr(), B.data_ptr(), mine.data_ptr(), "automatic",
                          False, None, stream)
        em.synchronize()

    def threads(count):
        for _ in range(count):
            mine = torch.zeros_like(want)
            torch.cuda.synchronize()
            t = threading.Thread(target=product, args=(em.STREAM_PER_THREAD, mine))
            t.start()
            t.join()
            assert torch.equal(mine, want)

    def streams(count):
        cudart, handles = torch.cuda.cudart(), []
        mine = torch.zeros_like(want)
        for _ in range(count):
            h = ctypes.c_void_p()
            assert int(cudart.cudaStreamCreate(ctypes.addressof(h))) == 0
            handles.append(h)
            mine.zero_()
            torch.cuda.synchronize()
            product(h.value, mine)
            assert torch.equal(mine, want)
        for h in handles:
            assert int(cudart.cudaStreamDestroy(h.value)) == 0

    captures(20), threads(4)
    free = torch.cuda.mem_get_info()[0]
    captures(70), threads(70)
    # A buffer is 4 MiB, so 140 kept ones would be 560; the rest is a graph's
    # end being noticed late, and the runtime's own.
    assert free - torch.cuda.mem_get_info()[0] < 140 << 20
    streams(70)
    captures(4), threads(4)
    replay(capture(A2, out2), out2, want2)
    assert torch.equal(em.matmul(A, B), want)
    assert free - torch.cuda.mem_get_info()[0] < 2 << 30
