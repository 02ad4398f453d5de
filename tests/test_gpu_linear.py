"""hip_linear against the oracle, bit for bit, on every tile shape of its dispatch (llmgen_amd/csrc/linear.hip): edges of
the tiles, K remainders, unaligned outputs, and values outside the windows in which products are exact."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle as O
from llmgen_amd._lib import lib

pytestmark = pytest.mark.gpu


def run(x, w, y_f32, offset=0):
    """hip_linear on bf16 bits; ``offset`` shifts the output by that many values from its aligned start."""
    M, N, K = x.shape[0], w.shape[0], x.shape[1]
    xd, wd = (torch.from_numpy(a.view(np.int16)).cuda() for a in (x, w))
    out = torch.full((M * N + offset + 8,), 77, dtype=torch.float32 if y_f32 else torch.int16, device="cuda")
    lib().hip_linear(out.data_ptr() + offset * out.element_size(), int(y_f32), xd.data_ptr(), wd.data_ptr(), M, N, K)
    torch.cuda.synchronize()
    assert lib().hip_last_error() == 0
    got = out.cpu().numpy()
    assert (got[:offset] == 77).all() and (got[offset + M * N:] == 77).all(), "wrote outside y"
    got = got[offset:offset + M * N].reshape(M, N)
    return got if y_f32 else got.view(np.uint16)


def check(x, w, y_f32, offset=0):
    got, ref = run(x, w, y_f32, offset), O.linear(x, w, out_bf16=not y_f32)
    if y_f32:
        nan = np.isnan(ref)
        got, ref, isnan = got.view(np.uint32), ref.view(np.uint32), np.isnan(got)
    else:
        nan, isnan = ((a & 0x7FFF) > 0x7F80 for a in (ref, got))
    np.testing.assert_array_equal(isnan, nan)
    np.testing.assert_array_equal(got[~nan], ref[~nan])


def draw(rng, *shape, std=1.0):
    return O.f32_to_bf16((std * rng.standard_normal(shape)).astype(np.float32))


# (M, N, K): one 16 x 16 block a workgroup, two blocks, up to 16 and up to 8 rows of many columns, then 32 x 32, 64 x 64, 64 x 192,
# 32 x 96 and 128 x 128 tiles
@pytest.mark.parametrize("M,N,K", [(1, 1, 8), (1, 16, 128), (17, 100, 24), (16, 1024, 1000), (3, 2049, 264),
                                   (33, 1700, 72), (40, 2000, 320), (16, 8200, 40), (5, 9001, 200),
                                   (8, 8196, 8), (1, 8321, 64), (8, 8200, 328), (50, 3000, 200),
                                   (129, 1031, 64), (512, 2048, 72), (1000, 3060, 40), (2051, 2048, 24), (200, 3001, 104),
                                   (2048, 6144, 16)])
def test_linear_tiles_bit_exact(gpu, M, N, K):
    rng = np.random.default_rng(M + 3 * N + K)
    check(draw(rng, M, K), draw(rng, N, K, std=0.05), y_f32=M % 2 == 1)


@pytest.mark.parametrize("N,offset", [(64, 0), (64, 1), (64, 2), (62, 0), (63, 3)])
@pytest.mark.parametrize("y_f32", [False, True])
def test_linear_any_output_alignment(gpu, N, offset, y_f32):
    rng = np.random.default_rng(N + offset)
    check(draw(rng, 19, 48), draw(rng, N, 48), y_f32, offset)


@pytest.mark.parametrize("M,N,K", [(9, 70, 136), (40, 2000, 72), (12, 8300, 72), (7, 8300, 136), (200, 1100, 200), (512, 2048, 40),
                                   (200, 3001, 104), (1000, 3060, 40), (2048, 6144, 16)])
@pytest.mark.parametrize("what", ["zeros", "tiny", "huge", "nonfinite", "edges"])
def test_linear_values_outside_the_exact_window(gpu, M, N, K, what):
    """Zeros stay on the fast path; values whose products leave f32's exact range (or are not finite) must take the
    separate multiply and add.  Only some tiles hold such values, so both paths run in one launch."""
    rng = np.random.default_rng(M * 5 + len(what))
    x, w = draw(rng, M, K), draw(rng, N, K, std=0.1)
    special = {"zeros": [0x0000, 0x8000], "tiny": [0x0001, 0x8001, 0x0080, 0x1000, 0x9A00],
               "huge": [0x7F00, 0xFF7F, 0x7E80, 0xF000], "nonfinite": [0x7F80, 0xFF80, 0x7FC0],
               # the first and last exponents inside and outside the windows of x (64..191) and w (60..187)
               "edges": [e << 7 for e in (59, 60, 63, 64, 187, 188, 191, 192)]}[what]
    for a in (x, w):
        n = max(1, a.size // 50) if what == "zeros" else 6
        at = rng.integers(0, a.size, n)
        a.reshape(-1)[at] = rng.choice(np.array(special, np.uint16), n)
    if what == "zeros":
        x[0], w[-1] = 0, 0
    if what in ("tiny", "edges"):  # whole rows of them, so that the sums are tiny too
        x[M // 2] = rng.choice(np.array(special, np.uint16), K)
        w[N // 2] = rng.choice(np.array(special, np.uint16), K)
    check(x, w, y_f32=True)
    check(x, w, y_f32=False)


@pytest.mark.parametrize("M", [1, 8, 9, 33, 300])
@pytest.mark.parametrize("Ns", [(2048, 1024, 1024), (3000, 3001, 0), (40, 24, 7), (0, 100, 33)])
def test_linear3_equals_single_products(gpu, M, Ns):
    """Column tiles of the three products share a grid: each must stay within its own matrix and output."""
    K, rng = 72, np.random.default_rng(M + sum(Ns))
    x, ws = draw(rng, M, K), [draw(rng, max(n, 1), K, std=0.1) for n in Ns]
    ws[1][0, 0] = 0x7F80  # only tiles of the second product take the separate operations
    xd, wd = torch.from_numpy(x.view(np.int16)).cuda(), [torch.from_numpy(w.view(np.int16)).cuda() for w in ws]
    ys = [torch.full((M * n + 8,), 77, dtype=torch.int16, device="cuda") for n in Ns]
    args = [a for y, w, n in zip(ys, wd, Ns) for a in ((y.data_ptr(), w.data_ptr(), n) if n else (None, None, 0))]
    lib().hip_linear3(*args, xd.data_ptr(), M, K)
    torch.cuda.synchronize()
    assert lib().hip_last_error() == 0
    for y, w, n in zip(ys, ws, Ns):
        got, ref = y.cpu().numpy(), run(x, w, False)[:, :n] if n else np.zeros((M, 0), np.uint16)
        assert (got[M * n:] == 77).all()
        np.testing.assert_array_equal(got[:M * n].view(np.uint16).reshape(M, n), ref)


@pytest.mark.parametrize("M,N", [(1, 1024), (8, 8300), (12, 8300), (33, 1701), (300, 1024)])
@pytest.mark.parametrize("what", ["in_place", "unaligned", "outside"])
def test_linear_add_equals_linear_then_add(gpu, M, N, what):
    K, rng = 136, np.random.default_rng(M + N)
    x, w, res = draw(rng, M, K), draw(rng, N, K, std=0.1), draw(rng, M, N)
    if what == "outside":
        x[0, 3] = 0x0001
    shift = 1 if what == "unaligned" else 0
    xd, wd = (torch.from_numpy(a.view(np.int16)).cuda() for a in (x, w))
    rd = torch.zeros(M * N + 1, dtype=torch.int16, device="cuda")
    rd[shift:shift + M * N] = torch.from_numpy(res.view(np.int16).reshape(-1)).cuda()
    yd = rd if what == "in_place" else torch.zeros(M * N, dtype=torch.int16, device="cuda")
    lib().hip_linear_add(yd.data_ptr(), rd.data_ptr() + 2 * shift, xd.data_ptr(), wd.data_ptr(), M, N, K)
    torch.cuda.synchronize()
    assert lib().hip_last_error() == 0
    got = yd.cpu().numpy()[:M * N].view(np.uint16).reshape(M, N)
    np.testing.assert_array_equal(got, O.add(res.reshape(-1), O.linear(x, w).reshape(-1)).reshape(M, N))


# Per kernel of the dispatch (at 256 CUs) a K of at least two trips of its pipelined loop and a remainder: (M, N, K) and the
# chunk of k, whole chunks
LOOPS = [(17, 900, 968, 128),    # one block a workgroup: 7
         (40, 2000, 712, 64),    # two blocks, loop of four chunks: 11
         (5, 8200, 712, 64),     # stream, loop of three stages: 11
         (12, 8300, 424, 64),    # 9 to 16 rows: 6
         (17, 4104, 424, 64),    # 32 x 32: 6
         (65, 5482, 248, 32),    # 32 x 96: 7
         (97, 6171, 248, 32),    # 64 x 64: 7
         (353, 6171, 200, 32),   # 64 x 192: 6
         (517, 5800, 248, 32)]   # 128 x 128: 7


@pytest.mark.parametrize("M,N,K,chunk", LOOPS)
def test_linear_main_loops_bit_exact(gpu, M, N, K, chunk):
    rng = np.random.default_rng(M + N + K)
    check(draw(rng, M, K), draw(rng, N, K, std=0.05), y_f32=M % 2 == 1)


@pytest.mark.parametrize("M,N,K,chunk", LOOPS)
@pytest.mark.parametrize("operand", ["x", "w"])
@pytest.mark.parametrize("what", ["tiny", "huge"])
def test_linear_one_chunk_outside_the_exact_window(gpu, M, N, K, chunk, operand, what):
    """One output of the last tile is the sum of two products from one chunk of k, all its other terms are zeros, and
    fused additions would give another sum: 2^-149 + 2^-150 (2^-149 as separate operations, 2^-148 fused), or
    -1.5 * 2^127 + 2^128 (+inf, 2^126 fused).  The chunk is the first, one in the middle, the last whole one, the
    remainder."""
    far, near = {"tiny": ((2.0**-90, 2.0**-90), (2.0**-59, 2.0**-60)),
                 "huge": ((-1.5 * 2.0**100, 2.0**100), (2.0**27, 2.0**28))}[what]
    rng = np.random.default_rng(M + N)
    whole = K // chunk
    x0, w0 = draw(rng, M, K), draw(rng, N, K, std=0.05)
    clean = O.linear(x0, w0, out_bf16=False)
    for at in (0, whole // 2, whole - 1, whole):
        x, w, k = x0.copy(), w0.copy(), at * chunk + 3
        row, col = (x, w) if operand == "x" else (w, x)
        row[-1], col[-1, k:k + 2] = 0, O.f32_to_bf16(np.array(near, np.float32))
        row[-1, k:k + 2] = O.f32_to_bf16(np.array(far, np.float32))
        ref = clean.copy()  # the special row and column anew, the rest is as it was
        ref[-1:], ref[:, -1:] = O.linear(x[-1:], w, out_bf16=False), O.linear(x, w[-1:], out_bf16=False)
        assert ref[-1, -1] == (np.float32(2.0**-149) if what == "tiny" else np.inf)
        got = run(x, w, y_f32=True)
        np.testing.assert_array_equal(got.view(np.uint32), ref.view(np.uint32))


# the products' column tiles in the streaming, 9..16-row, 32 x 96, 64 x 64, 64 x 192 and 128 x 128 kernels, main loops included
@pytest.mark.parametrize("M,Ns", [(1, (6144, 6144, 0)), (8, (5000, 3001, 1030)), (9, (6144, 6144, 0)),
                                  (16, (5000, 3001, 1030)), (300, (6144, 6144, 0)), (700, (5000, 3001, 1030)),
                                  (300, (5000, 3001, 1030)), (600, (6144, 6151, 0))])
def test_linear3_wide_equals_single_products(gpu, M, Ns):
    K, rng = 456, np.random.default_rng(M + sum(Ns))
    x, ws = draw(rng, M, K), [draw(rng, max(n, 1), K, std=0.1) for n in Ns]
    ws[1][0, 200] = 0x0001  # only tiles of the second product hold a value outside the window
    xd, wd = torch.from_numpy(x.view(np.int16)).cuda(), [torch.from_numpy(w.view(np.int16)).cuda() for w in ws]
    ys = [torch.full((M * n + 8,), 77, dtype=torch.int16, device="cuda") for n in Ns]
    args = [a for y, w, n in zip(ys, wd, Ns) for a in ((y.data_ptr(), w.data_ptr(), n) if n else (None, None, 0))]
    lib().hip_linear3(*args, xd.data_ptr(), M, K)
    torch.cuda.synchronize()
    assert lib().hip_last_error() == 0
    for y, w, n in zip(ys, ws, Ns):
        got, ref = y.cpu().numpy(), run(x, w, False)[:, :n] if n else np.zeros((M, 0), np.uint16)
        assert (got[M * n:] == 77).all()
        np.testing.assert_array_equal(got[:M * n].view(np.uint16).reshape(M, n), ref)


@pytest.mark.parametrize("M,N,K,chunk", LOOPS)
@pytest.mark.parametrize("chunks", [3, 4])
def test_linear_few_chunks_outside_the_exact_window(gpu, M, N, K, chunk, chunks):
    """Too short a K for the pipelined loop, and in every tile a value outside the window from the third chunk on: the waves
    of a workgroup learn of it in the last steps, and only there."""
    rng = np.random.default_rng(M + chunks)
    K = (chunks - 1) * chunk + 24
    x, w = draw(rng, M, K), draw(rng, N, K, std=0.05)
    x[::16, 2 * chunk + 5] = O.f32_to_bf16(np.array([2.0**-70], np.float32))[0]
    check(x, w, y_f32=True)


# the kernel of K = 8 and 16: eight rows and 256 columns a workgroup, an edge on either side; K = 24 is the first on tiles
@pytest.mark.parametrize("M,N", [(1, 1), (7, 255), (8, 256), (9, 257), (17, 1030), (2051, 4096)])
@pytest.mark.parametrize("K", [8, 16, 24])
@pytest.mark.parametrize("special", [False, True])
def test_linear_short_k(gpu, M, N, K, special):
    rng = np.random.default_rng(M + N + K)
    x, w = draw(rng, M, K), draw(rng, N, K)
    if special:
        for a in (x, w):
            at = rng.integers(0, a.size, 1 + a.size // 50)
            a.reshape(-1)[at] = rng.choice(np.array([0, 0x8000, 1, 0x8001, 0x1000, 0x7F00, 0xFF7F, 0x7F80, 0x7FC0], np.uint16),
                                           at.size)
    check(x, w, y_f32=True, offset=1)
    check(x, w, y_f32=False, offset=M % 2)


@pytest.mark.parametrize("K", [8, 16])
@pytest.mark.parametrize("M,Ns", [(1, (300, 1, 0)), (13, (256, 257, 33)), (300, (0, 2000, 600))])
def test_linear3_and_add_of_short_k(gpu, K, M, Ns):
    rng = np.random.default_rng(K + M)
    x, ws = draw(rng, M, K), [draw(rng, max(n, 1), K) for n in Ns]
    xd, wd = torch.from_numpy(x.view(np.int16)).cuda(), [torch.from_numpy(w.view(np.int16)).cuda() for w in ws]
    ys = [torch.full((M * n + 8,), 77, dtype=torch.int16, device="cuda") for n in Ns]
    args = [a for y, w, n in zip(ys, wd, Ns) for a in ((y.data_ptr(), w.data_ptr(), n) if n else (None, None, 0))]
    lib().hip_linear3(*args, xd.data_ptr(), M, K)
    refs = [O.linear(x, w)[:, :n].reshape(-1) for w, n in zip(ws, Ns)]
    sums = []
    for w, n, ref in zip(wd, Ns, refs):
        res = draw(rng, M * n)
        rd = torch.from_numpy(res.view(np.int16)).cuda()
        if n:
            lib().hip_linear_add(rd.data_ptr(), rd.data_ptr(), xd.data_ptr(), w.data_ptr(), M, n, K)
        sums.append((rd, O.add(res, ref) if n else res))
    torch.cuda.synchronize()
    assert lib().hip_last_error() == 0
    for y, ref, (rd, total) in zip(ys, refs, sums):
        got = y.cpu().numpy()
        assert (got[ref.size:] == 77).all()
        np.testing.assert_array_equal(got[:ref.size].view(np.uint16), ref)
        np.testing.assert_array_equal(rd.cpu().numpy().view(np.uint16), total)
