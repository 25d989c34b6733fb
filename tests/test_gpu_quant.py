"""GPU parity of the decoders, quantizers and epilogues against the oracle: bit-exact.

Dequantization must match ref/kernel.py bit for bit (ref/kernel.py:89-90, :98-101), so every
e4m3 and e2m1 code is decoded under a spread of scales, including the E8M0 edge codes 0 and 255.
"""

import numpy as np
import pytest
import torch

import oracle
from stblarge_amd import data, ops
from util import bits_equal, np_

pytestmark = pytest.mark.gpu


def test_dequant_fp4_every_code_every_scale(gpu):
    # 256 rows: row r uses scale byte r for all its groups; each row holds every code byte twice
    k = 1024
    codes = np.tile(np.arange(256, dtype=np.uint8), (256, 2))
    scales = np.repeat(np.arange(256, dtype=np.uint8)[:, None], k // 32, axis=1)
    got = ops.dequant_fp4(torch.from_numpy(codes).to(gpu), torch.from_numpy(scales).to(gpu))
    want = oracle.dequant_fp4(codes, scales)
    assert bits_equal(np_(got), want)


def test_dequant_fp8_every_code(gpu):
    rng = np.random.default_rng(0)
    codes = np.tile(np.arange(256, dtype=np.uint8), (256, 2))  # includes the NaN codes 0x7f, 0xff
    scales = (rng.random((2, 4)) * 0.01).astype(np.float32)
    scales[0, 0] = 1.0
    got = ops.dequant_fp8(torch.from_numpy(codes).to(gpu), torch.from_numpy(scales).to(gpu))
    assert bits_equal(np_(got), oracle.dequant_fp8_b128(codes, scales))
    e8 = rng.integers(0, 256, (8, 16), dtype=np.uint8)
    got = ops.dequant_fp8(torch.from_numpy(codes).to(gpu), torch.from_numpy(e8).to(gpu), e8m0=True)
    assert bits_equal(np_(got), oracle.dequant_fp8_e8m0_b32(codes, e8))


def test_dequant_gguf17(gpu):
    rng = np.random.default_rng(1)
    rows, k = 37, 512
    codes = rng.integers(0, 256, (rows, k // 2), dtype=np.uint8)
    scales = rng.integers(0, 256, (rows, k // 32), dtype=np.uint8)
    blocks = oracle.ocp_to_gguf17(codes, scales)
    got = ops.dequant_gguf17(torch.from_numpy(blocks).to(gpu), rows, k)
    assert bits_equal(np_(got), oracle.dequant_fp4(codes, scales))


@pytest.mark.parametrize("rows,k", [(8, 64), (33, 96), (2048, 7168), (7168, 2048)])
def test_quant_fp4_matches_oracle(gpu, rows, k):
    w = data.weight(rows, k, seed=rows + k)
    if rows == 33:  # edge groups: all zero, tiny, signed zeros, huge
        w[0, :32] = 0.0
        w[1, :32] = -1e-30
        w[2, 5] = -0.0
        w[3, :32] = 3.0e38
        w[4, 40] = 1e-39
    codes, scales = ops.quant_fp4(w.to(gpu))
    oc, os_ = oracle.quant_fp4(w.numpy())
    assert np.array_equal(np_(codes), oc)
    assert np.array_equal(np_(scales), os_)


def test_quant_fp4_ties_and_neighbours(gpu):
    # every multiple of 1/64 of the scale up to 6 with both signs, each next to its fp32 neighbours (so
    # all ties and both sides of them), under scales 2^-20 .. 2^20, with NaN and infinities
    grid = np.arange(-384, 385, dtype=np.float32) / 64
    vals = np.concatenate([grid, np.nextafter(grid, np.float32(9)), np.nextafter(grid, np.float32(-9)), [-0.0, 0.0]])
    vals = np.resize(vals.astype(np.float32), (75, 31))
    rows = np.concatenate([np.full((75, 1), 6, np.float32), vals], 1)  # the group's maximum is 6: its scale 1
    w = np.concatenate([rows * np.float32(2.0 ** e) for e in range(-20, 21, 5)], 0)
    w[0, 3], w[1, 4], w[2, 5] = np.nan, np.inf, -np.inf
    codes, scales = ops.quant_fp4(torch.from_numpy(w).to(gpu))
    with np.errstate(invalid="ignore"):
        oc, os_ = oracle.quant_fp4(w)
    assert np.array_equal(np_(scales), os_)
    assert np.array_equal(np_(codes), oc)


@pytest.mark.parametrize("rows,k", [(130, 260), (2048, 7168), (7168, 2048)])
def test_quant_fp8_b128_matches_oracle(gpu, rows, k):
    w = data.weight(rows, k, seed=3 * rows + k)
    if rows == 130:
        w[129, 259] = 0.5
        w[0:128, 128:256] = 0.0  # an all-zero block: amax clamps to 1e-4
    codes, scales = ops.quant_fp8_b128(w.to(gpu))
    oc, os_ = oracle.quant_fp8_b128(w.numpy())
    assert np.array_equal(np_(scales), os_)
    assert np.array_equal(np_(codes), oc)

@pytest.mark.parametrize("rows,k", [(70, 96), (33, 32), (2304, 5120), (5120, 2304)])
def test_quant_fp8_e8m0_matches_oracle(gpu, rows, k):
    w = data.weight(rows, k, seed=rows + k)
    w[0, :32] = 0  # a block row with a zero part
    codes, scales = ops.quant_fp8_e8m0(w.to(gpu))
    oc, os_ = oracle.quant_fp8_e8m0_b32(w.numpy())
    assert np.array_equal(np_(codes), oc) and np.array_equal(np_(scales), os_)
    deq = ops.dequant_fp8(codes, scales, e8m0=True)
    assert bits_equal(np_(deq), oracle.dequant_fp8_e8m0_b32(oc, os_))



@pytest.mark.parametrize("rows,k,shift", [(1, 128, 0), (129, 132, 0), (127, 1412, 0), (200, 130, 0), (130, 260, 1),
                                          (256, 384, 2)])
def test_quant_fp8_b128_edges_and_alignment(gpu, rows, k, shift):
    # whole and partial blocks read 16 bytes at a time, and the k and the unaligned w that are read value
    # by value; an infinity gives its block the scale +Inf, a NaN is skipped by the maximum
    w = data.weight(rows, k, seed=rows + k) * torch.logspace(-6, 6, k)
    w[0, 0], w[-1, -1] = float("nan"), float("inf")
    buf = torch.zeros(rows * k + 4, device=gpu)
    wg = buf[shift:shift + rows * k].view(rows, k)
    wg.copy_(w)
    codes, scales = ops.quant_fp8_b128(wg)
    oc, os_ = oracle.quant_fp8_b128(w.numpy())
    assert np.array_equal(np_(scales), os_)
    assert np.array_equal(np_(codes), oc)


@pytest.mark.parametrize("rows,k,shift", [(1, 32, 0), (33, 160, 0), (95, 2304, 0), (64, 128, 1)])
def test_quant_fp8_e8m0_edges_and_alignment(gpu, rows, k, shift):
    w = data.weight(rows, k, seed=rows + k) * torch.logspace(-6, 6, k)
    w[0, 0], w[-1, -1] = float("nan"), float("-inf")
    buf = torch.zeros(rows * k + 4, device=gpu)
    wg = buf[shift:shift + rows * k].view(rows, k)
    wg.copy_(w)
    codes, scales = ops.quant_fp8_e8m0(wg)
    oc, os_ = oracle.quant_fp8_e8m0_b32(w.numpy())
    assert np.array_equal(np_(codes), oc) and np.array_equal(np_(scales), os_)


@pytest.mark.parametrize("fmt,dim,inter", [(0, 96, 32), (0, 7168, 2048), (1, 260, 132), (1, 7168, 2048), (1, 130, 66),
                                           (2, 160, 96), (2, 5120, 2304)])
@pytest.mark.parametrize("where", ["new", "given", "host", "shared"])
def test_quant_expert_equals_its_matrices(gpu, fmt, dim, inter, where):
    # the one-launch form and the one that copies matrix by matrix (dims the launch does not take, a slot
    # in host memory, a slot sharing the weights' memory) write what the quantizers give for each matrix,
    # and nothing between the parts
    ws = [data.weight(r, k, seed=r + k + i, device=gpu) for i, (r, k) in enumerate(((inter, dim), (inter, dim), (dim, inter)))]
    q = {0: ops.quant_fp4, 1: ops.quant_fp8_b128, 2: ops.quant_fp8_e8m0}[fmt]
    parts = [t for w in ws for t in q(w)]
    n, _ = ops.expert_layout(fmt, dim, inter)
    fill = 0 if where == "new" else 77
    want = ops.pack_slot(parts, fmt, dim, inter, out=torch.full((n,), fill, dtype=torch.uint8, device=gpu))
    out = None
    if where == "given":
        out = torch.full((n + 256,), fill, dtype=torch.uint8, device=gpu)[256:]
    elif where == "host":
        out = torch.full((n,), fill, dtype=torch.uint8)
    elif where == "shared":
        buf = torch.empty(n + ws[2].numel() * 4, dtype=torch.uint8, device=gpu)  # n is a multiple of 256
        ws[2] = buf[n:].view(torch.float32).view(ws[2].shape).copy_(ws[2])
        out = buf[:n].fill_(fill)
    got = ops.quant_expert(*ws, fmt, out=out)
    assert out is None or got is out
    assert np.array_equal(np_(got), np_(want))


@pytest.mark.parametrize("block,pow2", [(32, True), (128, True), (128, False)])
def test_act_quant_matches_oracle(gpu, block, pow2):
    x = (data.normal((5, 1024), 1.0, seed=block) * torch.logspace(-3, 3, 1024)).to(torch.bfloat16)
    x[0, :block] = 0
    # non-finite values (the engine's rules, stbl/kernels.cu:56-63): a block holding an infinity has
    # scale +Inf, codes x / Inf and a NaN in-place form; a NaN is skipped by its block's maximum
    x[1, 3], x[2, block + 5], x[3, 2 * block] = float("inf"), float("-inf"), float("nan")
    codes, scales, deq = ops.act_quant(x.to(gpu), block, pow2, want_deq=True)
    oc, os_, od = oracle.act_quant(x.float().numpy(), block, pow2)
    assert np.array_equal(np_(scales), os_)
    assert np.array_equal(np_(codes), oc)
    assert bits_equal(np_(deq), od)


@pytest.mark.parametrize("rows,n,block,shift", [(1, 8, 8, 0), (3, 48, 16, 0), (7, 192, 64, 0), (33, 512, 256, 0),
                                                (2, 1024, 512, 0), (300, 896, 128, 0), (5, 96, 24, 0), (3, 64, 4, 0),
                                                (3, 1024, 1024, 0), (4, 256, 32, 1)])
@pytest.mark.parametrize("pow2", [True, False])
def test_act_quant_block_lengths_and_alignment(gpu, rows, n, block, shift, pow2):
    # blocks of 1, 2, 4, ... 64 lanes of 8 values (partial workgroups among them), and the block lengths
    # and the unaligned x that take one thread per block: all as the oracle, bit for bit
    x = (data.normal((rows, n), 1.0, seed=rows + n) * torch.logspace(-4, 4, n)).to(torch.bfloat16)
    x[-1, -1] = float("inf")
    x[0, 0] = float("nan")
    buf = torch.zeros(rows * n + 8, dtype=torch.bfloat16, device=gpu)
    xg = buf[shift:shift + rows * n].view(rows, n)
    xg.copy_(x)
    codes, scales, deq = ops.act_quant(xg, block, pow2, want_deq=True)
    oc, os_, od = oracle.act_quant(x.float().numpy(), block, pow2)
    assert np.array_equal(np_(scales), os_)
    assert np.array_equal(np_(codes), oc)
    assert bits_equal(np_(deq), od)


def test_stbl_act_quant_fp8_inplace(gpu):
    # the reference engine's form (stbl/kernels.cu:54-63): fp32 buffer of bf16 values, block 32
    x = (data.normal((4, 256), 3.0, seed=7)).to(torch.bfloat16).float()
    x[1, 40], x[2, 70], x[3, 100] = float("inf"), float("-inf"), float("nan")  # NaN blocks, NaN skipped
    got = ops.stbl_act_quant_fp8(x.clone().to(gpu))
    want = oracle.act_quant(x.numpy(), 32, True)[2]
    assert bits_equal(np_(got), want)


@pytest.mark.parametrize("n", [13824, 13824 + 96, 32])
def test_stbl_act_quant_fp8_inplace_fp32_scales(gpu, n):
    # any fp32 values (not only bf16 ones), blocks spread over 2^-30 .. 2^40, an all-zero block and a
    # block below the 1e-4 floor, at the engine's SwiGLU-output size and with a partial workgroup
    rng = np.random.default_rng(n)
    x = (rng.standard_normal(n) * np.repeat(2.0 ** rng.integers(-30, 41, n // 32), 32)).astype(np.float32)
    if n >= 96:
        x[32:64] = 0
        x[64:96] *= 1e-12
    got = ops.stbl_act_quant_fp8(torch.from_numpy(x.copy()).to(gpu))
    want = oracle.act_quant(x[None], 32, True)[2][0]
    assert bits_equal(np_(got), want)


def test_round_bf16_axpy(gpu):
    x = data.normal((5000,), 10.0, seed=8)
    got = ops.stbl_round_bf16(x.clone().to(gpu))
    assert bits_equal(np_(got), oracle.bf16_round(x.numpy()))
    y = data.normal((5000,), 1.0, seed=9)
    got = ops.stbl_axpy(y.clone().to(gpu), x.to(gpu), 1.0, 5000)
    assert bits_equal(np_(got), (y.numpy() + x.numpy()).astype(np.float32))
    got = ops.stbl_axpy(y.clone().to(gpu), x.to(gpu), 0.3, 5000)
    want = (y.double() + 0.3 * x.double()).float().numpy()  # one rounding: a fused multiply-add
    assert np.max(np.abs(np_(got) - want)) <= 1e-6 * np.max(np.abs(want))


def test_swiglu_batch(gpu):
    n, count = 2304, 3
    g = (data.normal((count * n,), 4.0, seed=10)).to(torch.bfloat16).float()
    u = (data.normal((count * n,), 4.0, seed=11)).to(torch.bfloat16).float()
    ws = [0.37, 1.0, 0.05]
    for limit in (0.0, 10.0):
        out = torch.empty(count * n, device=gpu)
        ops.stbl_swiglu_batch(out, g.to(gpu), u.to(gpu), ws, limit, n)
        want = np.concatenate([oracle.swiglu(g[j * n:(j + 1) * n].numpy(), u[j * n:(j + 1) * n].numpy(), ws[j], limit)
                               for j in range(count)])
        got = np_(out)
        # exp differs from libm's by at most an ulp, so a rare bf16 rounding may flip
        assert np.mean(got != want) < 0.01
        assert np.max(np.abs(got - want)) <= 2.0 ** -7 * np.max(np.abs(want))
