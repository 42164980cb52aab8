"""int4 format kernels vs the oracle, bit for bit: pack/unpack, RTN quantize, dequantize.

unpacked and dequantized weights match the reference bit-exactly."""

import numpy as np
import pytest
import torch

from _util import bits16, dev, to_np
from kernels.bench import cases
from kernels.quant import dequantize, pack_int4, quantize_rtn, unpack_int4, weight_bytes
from oracle import quant as oq
from oracle.reference import dequantize_ref

pytestmark = pytest.mark.gpu


def test_pack_unpack_bit_exact():
    rng = np.random.default_rng(0)
    q = rng.integers(0, 16, (1536, 2048)).astype(np.int32)
    packed = pack_int4(dev(q))
    assert np.array_equal(to_np(packed), oq.pack_int4(q))
    assert np.array_equal(to_np(unpack_int4(packed)), q)


def test_pack_extremes():
    q = torch.full((16, 3), 15, dtype=torch.int32, device="cuda")
    assert torch.equal(pack_int4(q).cpu(), torch.full((2, 3), -1, dtype=torch.int32))


def test_pack_out_of_range_wraps_like_reference():
    """quant.py:24-28 sums q << 4i in int64 and wraps to int32; so does the kernel."""
    rng = np.random.default_rng(1)
    q = rng.integers(-40, 40, (64, 8)).astype(np.int32)
    assert np.array_equal(to_np(pack_int4(dev(q))), oq.pack_int4(q))


@pytest.mark.parametrize("name,N,K", [("gate_up", 17920, 1536), ("down", 1536, 8960),
                                      ("k", 256, 1536)])
def test_quantize_rtn_bit_exact_config_shapes(name, N, K):
    w, _ = cases.w4a16_case(1, N, K, seed=0)
    qw, s, z = quantize_rtn(w.cuda(), 128)
    oqw, os_, oz = oq.quantize_rtn(w.numpy(), 128)
    assert qw.dtype == torch.int32 and s.dtype == torch.float16
    assert np.array_equal(to_np(qw), oqw)
    assert np.array_equal(bits16(s), bits16(os_))
    assert np.array_equal(bits16(z), bits16(oz))


@pytest.mark.parametrize("gs", [32, 64, 256])
def test_quantize_rtn_group_sizes(gs):
    w, _ = cases.w4a16_case(1, 96, 512, seed=5)
    qw, s, z = quantize_rtn(w.cuda(), gs)
    oqw, os_, oz = oq.quantize_rtn(w.numpy(), gs)
    assert np.array_equal(to_np(qw), oqw)
    assert np.array_equal(bits16(s), bits16(os_)) and np.array_equal(bits16(z), bits16(oz))


def test_quantize_rtn_fp32_weight_keeps_fp32_scales():
    w = torch.randn(64, 384, generator=cases.gen(6)) * 0.05
    qw, s, z = quantize_rtn(w.cuda(), 128)
    oqw, os_, oz = oq.quantize_rtn(w.numpy(), 128)
    assert s.dtype == torch.float32
    assert np.array_equal(to_np(qw), oqw)
    assert np.array_equal(to_np(s).view(np.uint32), os_.view(np.uint32))
    assert np.array_equal(to_np(z), oz)


def test_quantize_rtn_bf16_weight():
    """bf16 weights: the oracle runs on the (exact) fp32 values; scales are rounded to bf16 with
    torch's own RNE cast."""
    w = (torch.randn(32, 256, generator=cases.gen(7)) * 0.02).bfloat16()
    qw, s, z = quantize_rtn(w.cuda(), 128)
    oqw, os_, oz = oq.quantize_rtn(w.float().numpy(), 128)
    assert s.dtype == torch.bfloat16
    assert np.array_equal(to_np(qw), oqw)
    assert torch.equal(s.cpu().view(torch.int16), torch.from_numpy(os_).bfloat16().view(torch.int16))
    assert torch.equal(z.cpu().float(), torch.from_numpy(oz))


def test_quantize_rtn_edge_groups():
    """Constant groups (scale clamp), exact grids and ties, with known answers from the oracle
    tests."""
    w = np.zeros((4, 128), dtype=np.float32)
    w[0] = 0.5
    w[1] = -3e-6
    w[2] = (np.arange(128) % 16 - 3) * 0.25
    w[3, 0], w[3, 1] = 0.0, 15.0
    w[3, 2:6] = [2.5, 3.5, 0.5, 14.5]
    qw, s, z = quantize_rtn(dev(w), 128)
    oqw, os_, oz = oq.quantize_rtn(w, 128)
    assert np.array_equal(to_np(qw), oqw)
    assert np.array_equal(to_np(s).view(np.uint32), os_.view(np.uint32))
    assert np.array_equal(to_np(z), oz)


@pytest.mark.parametrize("N,K", [(17920, 1536), (1536, 8960), (40, 384)])
def test_dequantize_bit_exact(N, K):
    w, _ = cases.w4a16_case(1, N, K, seed=0)
    oqw, os_, oz = oq.quantize_rtn(w.numpy(), 128)
    out = dequantize(dev(oqw), dev(os_), dev(oz), 128)
    assert out.shape == (N, K) and out.dtype == torch.float16
    assert np.array_equal(bits16(out), bits16(dequantize_ref(oqw, os_, oz, 128)))


def test_weight_bytes_matches_buffers():
    qw, s, z = quantize_rtn(torch.zeros(17920, 1536, dtype=torch.float16, device="cuda"))
    nbytes = sum(t.numel() * t.element_size() for t in (qw, s, z))
    assert nbytes == weight_bytes(17920, 1536) == 14_622_720


# ------------------------------------------------ CPU tensors in, CPU tensors out (reference
# quant.py:20-49 and fp8.py:25-35 are device-agnostic torch code; its tests call them on the CPU)
def test_cpu_inputs_bit_exact_and_returned_on_cpu():
    from kernels.fp8 import dequantize_fp8, quantize_fp8
    from oracle import fp8 as of

    w, _ = cases.w4a16_case(1, 256, 1536, seed=0)  # fp16 [N, K] on the CPU
    qw, s, z = quantize_rtn(w, 128)
    oqw, os_, oz = oq.quantize_rtn(w.numpy(), 128)
    assert qw.device.type == s.device.type == z.device.type == "cpu"
    assert np.array_equal(qw.numpy(), oqw)
    assert np.array_equal(bits16(s), bits16(os_)) and np.array_equal(bits16(z), bits16(oz))
    deq = dequantize(qw, s, z, 128)
    assert deq.device.type == "cpu"
    assert np.array_equal(bits16(deq), bits16(dequantize_ref(oqw, os_, oz, 128)))
    q = torch.from_numpy(np.random.default_rng(3).integers(0, 16, (64, 40)).astype(np.int32))
    packed = pack_int4(q)
    assert packed.device.type == "cpu" and np.array_equal(packed.numpy(), oq.pack_int4(q.numpy()))
    assert torch.equal(unpack_int4(packed), q)
    wq, sc = quantize_fp8(w)
    owq, osc = of.quantize_fp8(w.numpy())
    assert wq.device.type == sc.device.type == "cpu"
    assert np.array_equal(wq.view(torch.uint8).numpy(), owq) and np.array_equal(bits16(sc), bits16(osc))
    back = dequantize_fp8(wq, sc)
    assert back.device.type == "cpu"
    assert np.array_equal(bits16(back), bits16(of.dequantize_fp8(owq, osc)))


def test_mixed_devices_rejected():
    q = torch.zeros((8, 4), dtype=torch.int32)  # K = 64: one group of 64
    with pytest.raises(RuntimeError, match="different devices"):
        dequantize(q.cuda(), torch.zeros((1, 4), dtype=torch.float16),
                   torch.zeros((1, 4), dtype=torch.float16, device="cuda"), 64)


def test_dequantize_column_sliced_scales_and_zeros():
    """Non-contiguous scales/zeros (column slices of a wider tensor) are copied to temporaries
    that must both stay alive until the launch is enqueued."""
    N, K = 96, 512
    w, _ = cases.w4a16_case(1, 2 * N, K, seed=8)
    oqw, os_, oz = oq.quantize_rtn(w.numpy(), 128)
    qw_t, s_t, z_t = dev(oqw), dev(os_), dev(oz)
    qs, ss, zs = qw_t[:, N:], s_t[:, N:], z_t[:, N:]
    assert not ss.is_contiguous() and not zs.is_contiguous()
    out = dequantize(qs, ss, zs, 128)
    ref = dequantize_ref(np.ascontiguousarray(oqw[:, N:]), np.ascontiguousarray(os_[:, N:]),
                         np.ascontiguousarray(oz[:, N:]), 128)
    assert np.array_equal(bits16(out), bits16(ref))


@pytest.mark.parametrize("N", [1, 63, 64, 65])
@pytest.mark.parametrize("gs,K", [(32, 96), (64, 192), (128, 384), (256, 512), (512, 1024), (24, 48)])
def test_quantize_rtn_column_tiles(N, gs, K):
    """The tiled quantizer (groups of 32 .. 512, 64 columns per workgroup) at the edges of its
    column tiles, and a group size that takes the general kernel; the last column's groups hold
    infinities and a NaN, whose quotients divide, and ties of w / scale."""
    w = (torch.randn(N, K, generator=cases.gen(N + gs)) * 0.05).half().numpy()
    w[0] = (np.arange(K) % 31 - 15) * 0.25
    if N > 1:
        w[-1, 0], w[-1, gs], w[-1, gs + 1] = np.inf, -np.inf, np.nan
    qw, s, z = quantize_rtn(dev(w), gs)
    oqw, os_, oz = oq.quantize_rtn(w[:max(1, N - 1)], gs)
    keep = slice(0, max(1, N - 1))
    assert np.array_equal(to_np(qw)[:, keep], oqw)
    assert np.array_equal(bits16(s)[:, keep], bits16(os_)) and np.array_equal(bits16(z)[:, keep], bits16(oz))
    if N > 1:  # scale = inf: finite weights and inf / inf give 0 (a -inf makes the zero NaN)
        assert to_np(qw)[: gs // 4, -1].max() == 0 and to_np(qw)[: gs // 4, -1].min() == 0


def test_quantize_rtn_unaligned_weight():
    """A weight whose base is not 16-byte aligned takes the general kernel; same bits."""
    base = (torch.randn(70 * 256 + 3, generator=cases.gen(4)) * 0.05).half().cuda()
    w = base[3:].view(70, 256)
    for a, b in zip(quantize_rtn(w, 128), quantize_rtn(w.clone(), 128)):
        assert torch.equal(a, b)


@pytest.mark.parametrize("N,K", [(1, 8), (63, 120), (64, 128), (65, 136), (130, 1032)])
def test_dequantize_tiles(N, K):
    """16 packed rows x 64 columns per workgroup, at the edges of both."""
    g = cases.gen(N)
    q = torch.randint(0, 16, (K, N), generator=g).int().numpy()
    s = (torch.rand(K // 8, N, generator=g) * 0.1).half().numpy()
    z = torch.randint(0, 16, (K // 8, N), generator=g).half().numpy()
    out = dequantize(dev(oq.pack_int4(q)), dev(s), dev(z), 8)
    assert np.array_equal(bits16(out), bits16(dequantize_ref(oq.pack_int4(q), s, z, 8)))


@pytest.mark.parametrize("N", [1, 63, 64, 128, 132, 257])
@pytest.mark.parametrize("K", [3, 64, 72, 129, 2056])
def test_fp8_convert_tiles(N, K):
    """quantize_fp8 (128 channels x 64 k per workgroup) and dequantize_fp8 (64 x 64) at the edges
    of their tiles, with and without 4-byte aligned k rows and 16-byte aligned weight rows."""
    from kernels.fp8 import dequantize_fp8, quantize_fp8
    from oracle import fp8 as of

    w = (torch.randn(N, K, generator=cases.gen(N + K)) * 0.05).half().numpy()
    w[0, 0] = -0.0
    wq, s = quantize_fp8(dev(w))
    owq, os_ = of.quantize_fp8(w)
    assert np.array_equal(wq.view(torch.uint8).cpu().numpy(), owq) and np.array_equal(bits16(s), bits16(os_))
    assert np.array_equal(bits16(dequantize_fp8(wq, s)), bits16(of.dequantize_fp8(owq, os_)))
    w32 = torch.from_numpy(w).float()
    wq, s = quantize_fp8(w32.cuda())
    owq, os_ = of.quantize_fp8(w32.numpy())
    assert np.array_equal(wq.view(torch.uint8).cpu().numpy(), owq) and np.array_equal(to_np(s), os_)
    assert np.array_equal(to_np(dequantize_fp8(wq, s)), of.dequantize_fp8(owq, os_))


@pytest.mark.parametrize("N", [(1 << 20) + 1, (1 << 24) + 133])
def test_fp8_quantize_many_channels(N):
    """More channels than the absmax launch has workgroups, and than it could have at one each."""
    from kernels.fp8 import quantize_fp8
    from oracle import fp8 as of

    g = torch.Generator(device="cuda").manual_seed(N)
    w = (torch.randn(N, 8, generator=g, device="cuda") * torch.rand(N, 1, generator=g, device="cuda")).half()
    wq, s = quantize_fp8(w)
    rows = torch.cat([torch.arange(300), torch.arange((1 << 20) - 150, (1 << 20) + 1), torch.arange(N - 300, N)])
    owq, os_ = of.quantize_fp8(w[rows].cpu().numpy())
    assert np.array_equal(bits16(s[rows]), bits16(os_))
    assert np.array_equal(to_np(wq.view(torch.uint8)[:, rows]), owq.view(np.uint8))


@pytest.mark.parametrize("N,K", [(1, (1 << 30) + 72), ((1 << 30) + 130, 1)])
def test_fp8_more_tiles_than_one_grid_dimension(N, K):
    """One row or one column of more than 2^24 tiles (2^32 threads in all): codes, scales and the
    values back, in windows at both ends and around the first tile of the grid's second row."""
    from kernels.fp8 import FP8, dequantize_fp8, quantize_fp8
    from oracle import fp8 as of

    w = torch.empty(N, K, dtype=torch.float16, device="cuda").normal_(std=0.05)
    wq, s = quantize_fp8(w)
    back = dequantize_fp8(wq, s)
    n = max(N, K)
    for at in (0, (64 << 20) - 70, (128 << 20) - 70, n - 140):
        win = slice(at, at + 140)
        if K == 1:
            owq, os_ = of.quantize_fp8(w[win].cpu().numpy())
            got, sc, ref = wq[:, win], s[win], of.dequantize_fp8(owq, os_)
        else:
            top = float(w.abs().max())
            row = np.append(w[:, win].cpu().numpy(), np.float16([[top]]), 1)  # the row's absmax with the window
            owq, os_ = of.quantize_fp8(row)
            owq, got, sc = owq[:-1], wq[win], s
            ref = of.dequantize_fp8(owq, os_)
        assert np.array_equal(to_np(got.contiguous().view(torch.uint8)), owq) and np.array_equal(bits16(sc), bits16(os_))
        b = back[win] if K == 1 else back[:, win]
        assert np.array_equal(bits16(b.contiguous()), bits16(ref))


def test_dequantize_more_tiles_than_one_grid_dimension():
    """One column of more than 2^24 tiles of 16 packed rows."""
    R, G = (1 << 28) + 16, 1 << 7
    g = torch.Generator(device="cuda").manual_seed(1)
    qw = torch.randint(-(2 ** 31), 2 ** 31 - 1, (R, 1), generator=g, device="cuda", dtype=torch.int64).int()
    s = torch.rand(R * 8 // G, 1, generator=g, device="cuda").half()
    z = torch.randint(0, 16, (R * 8 // G, 1), generator=g, device="cuda").half()
    out = dequantize(qw, s, z, G)
    for r in (0, (1 << 24) - 32, R - 64):  # windows of 64 packed rows, whole groups
        win, grp = slice(r, r + 64), slice(r * 8 // G, (r + 64) * 8 // G)
        ref = dequantize_ref(to_np(qw[win]), to_np(s[grp]), to_np(z[grp]), G)
        assert np.array_equal(bits16(out[:, r * 8:(r + 64) * 8].contiguous()), bits16(ref))


@pytest.mark.parametrize("N", [1, 5, 64])
def test_fp8_dequantize_every_code(N):
    """The conversion instruction against the format's table: every code times scales of both signs,
    to zero, to fp16's subnormals and past its range."""
    from kernels.fp8 import FP8, dequantize_fp8
    from oracle import fp8 as of

    codes = np.repeat(np.arange(256, dtype=np.uint8)[:, None], N, 1)
    scales = np.resize(np.array([1.0, -0.37, 6e-8, 146.0, -3e-5, 0.0, -0.0, 1e-3], dtype=np.float32), N)
    nan = (np.arange(256) & 0x7F) == 0x7F
    for dt in (np.float32, np.float16):
        s = scales.astype(dt)
        got = to_np(dequantize_fp8(dev(codes).view(FP8), dev(s)))
        with np.errstate(over="ignore", invalid="ignore"):
            ref = (of.e4m3_decode(codes) * s.astype(np.float32)).astype(dt).T
        assert np.isnan(got[:, nan]).all() and np.array_equal(np.signbit(got[:, nan]), codes.T[:, nan] > 127)
        bits = [np.ascontiguousarray(a[:, ~nan]).view(np.uint8) for a in (got, ref)]
        assert np.array_equal(*bits)
