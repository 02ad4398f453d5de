"""The row and element ops of llmgen_amd/csrc/model_ops.hip at the edges of their launch rules, bit for bit against the
oracle: rows per wave of RMSNorm, vector and scalar parts of the elementwise ops, slices of a sampled row."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle as O
from llmgen_amd._lib import lib

pytestmark = pytest.mark.gpu


def up(a):
    a = np.ascontiguousarray(a)
    return torch.from_numpy(a.view(np.int16) if a.dtype == np.uint16 else a).cuda()


def down(t):
    torch.cuda.synchronize()
    assert lib().hip_last_error() == 0
    return t.cpu().numpy().view(np.uint16)


def draw(rng, *shape, std=1.0):
    return O.f32_to_bf16((std * rng.standard_normal(shape)).astype(np.float32))


# one, two, four and eight rows a wave, the last wave partly empty; D below, at and off the chain's step of 64
@pytest.mark.parametrize("rows,D", [(1, 8), (3, 72), (5, 8192), (2049, 136), (2051, 4096), (4099, 1000), (4097, 1024),
                                    (8195, 128), (8193, 512), (8193, 520)])
@pytest.mark.parametrize("offset", [0, 1])
def test_rmsnorm_rows_per_wave(gpu, rows, D, offset):
    rng = np.random.default_rng(rows + D)
    x, g = draw(rng, rows, D, std=2.0), (1 + 0.1 * rng.standard_normal(D)).astype(np.float32)
    out = torch.zeros(rows * D + offset + 8, dtype=torch.int16, device="cuda")
    xd, gd = up(x), up(g)
    lib().hip_rmsnorm(out.data_ptr() + 2 * offset, xd.data_ptr(), gd.data_ptr(), rows, D, 1e-6)
    got = down(out)
    np.testing.assert_array_equal(got[offset:offset + rows * D].reshape(rows, D), O.rmsnorm(x, g, 1e-6))
    assert not got[:offset].any() and not got[offset + rows * D:].any()


@pytest.mark.parametrize("n", [1, 7, 8, 9, 2047, 2048, 2049, 4101])
@pytest.mark.parametrize("offset", [0, 1, 4])
def test_elementwise_tails_and_alignment(gpu, n, offset):
    rng = np.random.default_rng(n)
    a, b = draw(rng, n, std=4.0), draw(rng, n, std=2.0)
    ad, bd = (torch.cat([torch.zeros(offset, dtype=torch.int16, device="cuda"), up(t)]) for t in (a, b))
    for name, ref in (("add", O.add(a, b)), ("mul", O.mul(a, b))):
        out = torch.zeros(n + 16, dtype=torch.int16, device="cuda")
        getattr(lib(), "hip_" + name)(out.data_ptr(), ad.data_ptr() + 2 * offset, bd.data_ptr() + 2 * offset, n)
        got = down(out)
        np.testing.assert_array_equal(got[:n], ref)
        assert not got[n:].any()


def test_silu_mul_equals_silu_then_mul(gpu):
    rng = np.random.default_rng(3)
    a, b = up(draw(rng, 3077, std=4.0)), up(draw(rng, 3077))
    ref, out = torch.empty_like(a), a.clone()
    lib().hip_silu(ref.data_ptr(), a.data_ptr(), a.numel())
    lib().hip_mul(ref.data_ptr(), ref.data_ptr(), b.data_ptr(), a.numel())
    lib().hip_silu_mul(out.data_ptr(), out.data_ptr(), b.data_ptr(), a.numel())
    np.testing.assert_array_equal(down(out), down(ref))


def test_silu_every_value(gpu):
    """All 65536 inputs against x / (1 + exp(-x)) with exp rounded once to f32, as a correctly rounded expf gives it."""
    bits = np.arange(65536, dtype=np.uint32).astype(np.uint16)
    out = torch.zeros(65536, dtype=torch.int16, device="cuda")
    lib().hip_silu(out.data_ptr(), up(bits).data_ptr(), 65536)
    got, v = down(out), O.bf16_to_f32(bits)
    with np.errstate(all="ignore"):
        e = np.exp(-v.astype(np.float64)).astype(np.float32)
        ref = O.f32_to_bf16(v / (np.float32(1) + e))
    nan = (ref & 0x7FFF) > 0x7F80
    np.testing.assert_array_equal((got & 0x7FFF) > 0x7F80, nan)
    np.testing.assert_array_equal(got[~nan], ref[~nan])


# one slice, several; rows that start unaligned (odd V); rows shorter than a vector
@pytest.mark.parametrize("S,V", [(1, 1), (3, 7), (2, 8191), (5, 16384), (3, 16391), (4, 65549), (1, 300007)])
def test_sample_slices(gpu, S, V):
    rng = np.random.default_rng(S + V)
    lg = draw(rng, S, V)
    lg[0, [V // 3, V - 1]] = O.f32_to_bf16(np.array([9.0], np.float32))[0]  # a tie, the second in the last slice
    if S > 2:
        lg[1] = 0xFF80  # no candidate: index 0
        lg[2, 0] = 0x7FC0  # NaN at the scan's starting index
    temps = np.array([0.0, 0.0, 0.9, 1.7, 0.4][:S], np.float32)
    seed = torch.tensor([1234567], dtype=torch.int64, device="cuda")
    out = torch.full((S,), -5, dtype=torch.int32, device="cuda")
    ld, td = up(lg), up(temps)
    for t, tdev in ((temps, td), (np.zeros_like(temps), torch.zeros_like(td))):
        for _ in range(3):
            lib().hip_sample(out.data_ptr(), ld.data_ptr(), tdev.data_ptr(), seed.data_ptr(), S, V, None)
            torch.cuda.synchronize()
            np.testing.assert_array_equal(out.cpu().numpy(), O.sample(lg, t, seed=1234567))


def test_sample_into_pinned_host_memory(gpu):
    """Ids written straight to the host: no device-side read-modify-write of that memory (it would need PCIe atomics)."""
    S, V = 3, 60007
    rng = np.random.default_rng(8)
    lg, temps = draw(rng, S, V), np.array([0.0, 0.8, 1.3], np.float32)
    seed = torch.tensor([99], dtype=torch.int64, device="cuda")
    ld, td = up(lg), up(temps)
    out = torch.full((S,), -5, dtype=torch.int32, pin_memory=True)
    lib().hip_sample(out.data_ptr(), ld.data_ptr(), td.data_ptr(), seed.data_ptr(), S, V, None)
    torch.cuda.synchronize()
    assert lib().hip_last_error() == 0
    np.testing.assert_array_equal(out.numpy(), O.sample(lg, temps, seed=99))


def test_mlp_and_sampling_captured(gpu):
    """The products, norms and sampling of a step recorded into a graph: replayed on new inputs, with eager work in
    between, each replay equals the eager launches."""
    T, D, F, V = 20, 256, 520, 40960
    L, rng = lib(), np.random.default_rng(4)
    g = up((1 + 0.1 * rng.standard_normal(D)).astype(np.float32))
    wg, wu, wd, wh = (up(draw(rng, n, k, std=0.05)) for n, k in ((F, D), (F, D), (D, F), (V, D)))
    temps, seed = up(np.where(np.arange(T) % 3 == 1, 0.8, 0).astype(np.float32)), torch.tensor([7], device="cuda")
    x, xn, gate, upp = (torch.zeros(T * n, dtype=torch.int16, device="cuda") for n in (D, D, F, F))
    logits = torch.zeros(T * V, dtype=torch.int16, device="cuda")
    ids = torch.zeros(T, dtype=torch.int32, device="cuda")

    def step():
        p = torch.Tensor.data_ptr
        L.hip_rmsnorm(p(xn), p(x), p(g), T, D, 1e-6)
        L.hip_linear3(p(gate), p(wg), F, p(upp), p(wu), F, None, None, 0, p(xn), T, D)
        L.hip_silu_mul(p(gate), p(gate), p(upp), T * F)
        L.hip_linear_add(p(x), p(x), p(gate), p(wd), T, D, F)
        L.hip_linear(p(logits), 0, p(x), p(wh), T, V, D)
        L.hip_sample(p(ids), p(logits), p(temps), p(seed), T, V, None)

    inputs = [up(draw(rng, T * D)) for _ in range(4)]
    refs = []
    for v in inputs:
        x.copy_(v)
        step()
        torch.cuda.synchronize()
        refs.append((x.clone(), logits.clone(), ids.clone()))
    assert L.hip_graph_begin() == 0
    step()
    graph = L.hip_graph_end()
    assert graph, "capture failed"
    try:
        for v, ref in zip(inputs, refs):
            x.copy_(v)
            logits.zero_()
            ids.fill_(-1)
            torch.cuda.synchronize()
            L.hip_graph_launch(graph)
            torch.cuda.synchronize()
            assert L.hip_last_error() == 0
            for got, want in zip((x, logits, ids), ref):
                assert torch.equal(got, want)
    finally:
        L.hip_graph_destroy(graph)


# (S, V) at the edges of the launch rule (256 CUs): 256, 512 and 1024 lanes for whole rows, cut rows with and without cut
# greedy ones, the most slices, and a row for every other CU and beyond
@pytest.mark.parametrize("S,V", [(2, 2048), (3, 2049), (257, 8190), (5, 4097), (40, 16384), (2, 70001), (1, 131072),
                                 (128, 16390), (129, 49151), (129, 49152), (200, 65537)])
def test_sample_any_previous_ids(gpu, S, V):
    """Cut rows meet in out_ids, whatever it holds before the call: rubbish, the answer, another index, an index whose
    logit is no candidate."""
    rng = np.random.default_rng(S * 3 + V)
    lg = draw(rng, S, V)
    lg[0] = 0xFF80  # no candidate: index 0
    lg[-1, 5] = 0x7FC0
    temps = np.where(np.arange(S) % 2 == 1, 0.9, 0.0).astype(np.float32)
    seed = torch.tensor([31], dtype=torch.int64, device="cuda")
    ref = O.sample(lg, temps, seed=31)
    ld, td = up(lg), up(temps)
    for before in (-1, 2**31 - 1, V, V - 1, 5, ref):
        out = torch.tensor(np.broadcast_to(before, S).astype(np.int32), device="cuda")
        lib().hip_sample(out.data_ptr(), ld.data_ptr(), td.data_ptr(), seed.data_ptr(), S, V, None)
        torch.cuda.synchronize()
        np.testing.assert_array_equal(out.cpu().numpy(), ref)
    assert lib().hip_last_error() == 0


@pytest.mark.parametrize("rows,D", [(3, 1000), (5, 8192), (2051, 264), (4099, 136), (8195, 128)])
@pytest.mark.parametrize("gains,offset", [(1, 0), (2, 3), (3, 1)])
def test_rmsnorm_gains_and_output_at_any_address(gpu, rows, D, gains, offset):
    rng = np.random.default_rng(rows * gains)
    x, g = draw(rng, rows, D, std=2.0), (1 + 0.1 * rng.standard_normal(D)).astype(np.float32)
    out = torch.zeros(rows * D + offset + 8, dtype=torch.int16, device="cuda")
    xd, gd = up(x), torch.cat([torch.zeros(gains, device="cuda"), up(g)])
    lib().hip_rmsnorm(out.data_ptr() + 2 * offset, xd.data_ptr(), gd.data_ptr() + 4 * gains, rows, D, 1e-6)
    got = down(out)
    np.testing.assert_array_equal(got[offset:offset + rows * D].reshape(rows, D), O.rmsnorm(x, g, 1e-6))
    assert not got[:offset].any() and not got[offset + rows * D:].any()


# the edges of the rule for slices (256 CUs): cut from 8193 values, beyond 128 rows from 16384 on; 32 slices for up to 32
# rows; four greedy slices for up to 160 rows from 65536 values on, else two; whole rows again beyond 1024 and 4096 rows
@pytest.mark.parametrize("S,V", [(1, 8192), (3, 8193), (128, 8193), (129, 16383), (129, 16384), (32, 65536), (33, 65535), (1, 131071),
                                 (160, 65536), (161, 65536), (300, 24575), (300, 24576), (1025, 16384), (1025, 24576), (4097, 8200)])
def test_sample_slices_rule_edges(gpu, S, V):
    """Every row holds its largest value twice, in two slices; a row without a candidate and one with NaN among them."""
    rng = np.random.default_rng(S + 2 * V)
    lg = np.broadcast_to(draw(rng, 1, V + 4096), (S, V + 4096))  # rows: one stream from another start each
    lg = np.stack([row[i % 4096:i % 4096 + V] for i, row in enumerate(lg)])
    for i, at in enumerate(rng.integers(0, V // 2, S)):
        lg[i, [at, V - 1 - at % 7]] = 0x4110  # 9.0
    lg[-1] = 0xFF80
    lg[S // 2, 0] = 0x7FC0
    temps = np.where(np.arange(S) % 5 == 1, 0.9, 0.0).astype(np.float32)
    seed = torch.tensor([3], dtype=torch.int64, device="cuda")
    ref = O.sample(lg, temps, seed=3)
    ld, td, out = up(lg), up(temps), torch.full((S,), -5, dtype=torch.int32, device="cuda")
    for _ in range(2):
        lib().hip_sample(out.data_ptr(), ld.data_ptr(), td.data_ptr(), seed.data_ptr(), S, V, None)
        torch.cuda.synchronize()
        np.testing.assert_array_equal(out.cpu().numpy(), ref)
    assert lib().hip_last_error() == 0


# a value per lane up to 2^17 values, vectors of eight beyond, where all three addresses allow them (offset 8 does)
@pytest.mark.parametrize("n", [65537, 131071, 131072, 131073, 131080, 140007, 300001])
@pytest.mark.parametrize("offset", [0, 1, 8])
def test_elementwise_long_streams(gpu, n, offset):
    rng = np.random.default_rng(n)
    a, b = draw(rng, n, std=4.0), draw(rng, n, std=2.0)
    ad, bd = (torch.cat([torch.zeros(offset, dtype=torch.int16, device="cuda"), up(t)]) for t in (a, b))
    for name, ref in (("add", O.add(a, b)), ("mul", O.mul(a, b)), ("silu_mul", None), ("silu", None)):
        out = torch.zeros(n + offset + 16, dtype=torch.int16, device="cuda")
        args = [t.data_ptr() + 2 * offset for t in ((out, ad) if name == "silu" else (out, ad, bd))]
        getattr(lib(), "hip_" + name)(*args, n)
        got = down(out)
        assert not got[:offset].any() and not got[offset + n:].any()
        np.testing.assert_array_equal(got[offset:offset + n], silu(a, b if name == "silu_mul" else None) if ref is None else ref)


def silu(bits, up_bits=None):
    """x / (1 + exp(-x)) with exp rounded once to f32, rounded to bf16; times ``up_bits``, rounded again."""
    v = O.bf16_to_f32(bits)
    with np.errstate(all="ignore"):
        s = O.f32_to_bf16(v / (np.float32(1) + np.exp(-v.astype(np.float64)).astype(np.float32)))
        return s if up_bits is None else O.f32_to_bf16(O.bf16_to_f32(s) * O.bf16_to_f32(up_bits))


@pytest.mark.parametrize("copies", [1, 3])  # a value per lane, vectors
def test_silu_and_silu_mul_every_gate(gpu, copies):
    """All 65536 gates, in both kernels of both ops, against the form with a double exp rounded once."""
    gates = np.tile(np.arange(65536, dtype=np.uint32).astype(np.uint16), copies)
    gd, out = up(gates), torch.zeros(gates.size, dtype=torch.int16, device="cuda")
    for factor in (None, 1.0, -0.7109375, 3.0e38, 2.0**-130):
        ud = None if factor is None else O.f32_to_bf16(np.full(gates.size, factor, np.float32))
        if ud is None:
            lib().hip_silu(out.data_ptr(), gd.data_ptr(), gates.size)
        else:
            lib().hip_silu_mul(out.data_ptr(), gd.data_ptr(), up(ud).data_ptr(), gates.size)
        got, ref = down(out), silu(gates, ud)
        nan = (ref & 0x7FFF) > 0x7F80
        np.testing.assert_array_equal((got & 0x7FFF) > 0x7F80, nan)
        np.testing.assert_array_equal(got[~nan], ref[~nan])


@pytest.mark.parametrize("rows,D", [(2047, 2560), (2048, 2560), (2049, 2560), (2049, 2568)])
def test_rmsnorm_two_rows_a_wave_up_to_2560(gpu, rows, D):
    rng = np.random.default_rng(rows + D)
    x, g = draw(rng, rows, D, std=2.0), (1 + 0.1 * rng.standard_normal(D)).astype(np.float32)
    out, xd, gd = torch.zeros(rows * D + 8, dtype=torch.int16, device="cuda"), up(x), up(g)
    lib().hip_rmsnorm(out.data_ptr(), xd.data_ptr(), gd.data_ptr(), rows, D, 1e-6)
    got = down(out)
    np.testing.assert_array_equal(got[:rows * D].reshape(rows, D), O.rmsnorm(x, g, 1e-6))
    assert not got[rows * D:].any()
