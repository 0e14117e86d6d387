"""Rows far from one: the quantized products keep rows at a power of two of their own (mf_device.h), and none of it may show --
a bf16 number of any size gives what it gives as an fp32 product."""
import numpy as np
import pytest
import torch

from mference_amd import operators as ops
from helpers import ROOT_SEED, errors, make_moe, to_device_layer

pytestmark = pytest.mark.gpu


def _scaled_x(oracle, seed, t, d, powers):
    """N(0, 1) rows, row i times 2^powers[i]"""
    x = oracle.bf16_to_float(oracle.synth_x(ROOT_SEED + seed, t, d)).astype(np.float64)
    return oracle.bf16_bits((x * 2.0 ** np.asarray(powers, np.float64)[:, None]).astype(np.float32))


def _rows_close(oracle, got_bits, ref_bits, what):
    """row by row: a row of large numbers must not speak for the others.  An activation or a result that lands on the other side of a
    bf16 rounding boundary moves by 2^-8 of itself at most, so all of them together move a row by 2^-8 of its norm at most."""
    got, ref = oracle.bf16_to_float(got_bits).astype(np.float64), oracle.bf16_to_float(ref_bits).astype(np.float64)
    assert np.isfinite(ref).all() and (np.abs(ref).max(axis=1) > 0).all(), what
    for i, (g, r) in enumerate(zip(got, ref)):
        top = np.abs(r).max()
        _, rel = errors(g / top, r / top)
        assert np.isfinite(g).all() and rel <= 2.0 ** -8, (what, i, rel)


# x of 2^-50 gives activations of 2^-100; of 2^50, of 2^100
_POWERS = [0, 50, -50, 23, -24, 12, 58, -30]


@pytest.mark.parametrize("bits,d,f,e,k,t,form", [
    (4, 256, 128, 16, 4, 8, "fused"), (4, 2048, 512, 16, 8, 5, "fused"), (4, 704, 448, 12, 4, 1, "fused"), (2, 1024, 320, 16, 6, 8, "fused"),
    (2, 4096, 128, 16, 2, 1, "fused"), (1, 512, 256, 32, 8, 3, "fused"), (2, 128, 64, 16, 3, 7, "fused"), (4, 8192, 128, 4, 2, 8, "fused"),
    (4, 2816, 128, 8, 2, 3, "fused"), (4, 1600, 128, 8, 2, 4, "fused"),
    (4, 256, 128, 16, 4, 8, "phases"), (2, 640, 320, 16, 3, 8, "phases"), (1, 512, 256, 32, 8, 5, "phases"),
])
def test_decode_layer_of_rows_far_from_one(gpu, oracle, bits, d, f, e, k, t, form):
    layer = oracle.synth_layer(ROOT_SEED + 0x9500 + bits + d, d, f, e, k, bits=bits, fs=0)
    moe, wts = make_moe(gpu, layer), to_device_layer(layer)
    moe.set_fused(form == "fused")
    rng = np.random.default_rng(d + f)
    idx = np.stack([rng.permutation(e)[:k] for _ in range(t)]).astype(np.int32)
    w = rng.random((t, k), dtype=np.float32)
    for first in range(0, len(_POWERS), t):  # every power in some call, for any number of rows
        powers = (_POWERS[first:] + _POWERS)[:t]
        xb = _scaled_x(oracle, d + first, t, d, powers)
        y = torch.zeros((t, d), dtype=torch.bfloat16, device="cuda")
        wts.router_w = None
        moe.encode_decode_layer(wts, ops.bf16_tensor(xb), y, t=t, out_indices=torch.from_numpy(idx).cuda(), out_weights=torch.from_numpy(w).cuda())
        moe.status()
        ref = np.zeros((t, d), np.float32)
        for i in range(t):
            for j in range(k):
                blob = layer.experts[idx[i, j]]
                acts = oracle.expert_phase1(blob, layer.off, bits, d, f, xb[i])
                ref[i] += w[i, j] * oracle.expert_down(blob, layer.off, bits, d, f, acts).astype(np.float32)
        _rows_close(oracle, ops.bf16_bits(y), oracle.bf16_bits(ref), f"{form} bits={bits} d={d} f={f} 2^{powers}")


@pytest.mark.parametrize("bits", [4, 2, 1])
@pytest.mark.parametrize("power", [59, 100, -75, -110])
def test_routed_rows_of_one_sign(gpu, oracle, bits, power):
    """activations of one sign near 2^power through the down projection: a power of two on them is one on the result"""
    d, f, e, k, t = 192, 320, 8, 3, 2
    layer = oracle.synth_layer(ROOT_SEED + 0x9600 + bits, d, f, e, k, bits=bits, fs=0)
    moe, wts = make_moe(gpu, layer), to_device_layer(layer)
    acts = (1.0 + torch.rand((t, k, f), generator=torch.Generator().manual_seed(3))).to(torch.bfloat16)
    idx = torch.tensor([[0, 3, 5], [1, 2, 7]], dtype=torch.int32).cuda()
    w = torch.ones((t, k), device="cuda")
    out = []
    for p in (0, power):
        y = torch.zeros((t, d), dtype=torch.bfloat16, device="cuda")
        moe.encode_routed_phase2_reduce(wts.experts, wts.offsets, idx, w, (acts.double() * 2.0 ** p).to(torch.bfloat16).cuda(), None, y, t=t)
        torch.cuda.synchronize()
        out.append(y.double().cpu() * 2.0 ** -p)
    assert torch.equal(*out) and (out[0] != 0).double().mean() > 0.99


def _weights(oracle, rng, rows, cols, bits):
    if bits != 1:
        return oracle.quantize(rng.normal(0.0, 0.02, rows * cols).reshape(rows, cols), bits)
    codes = np.digitize(rng.uniform_fill(0.0, 1.0, rows * cols), (0.25, 0.75)).astype(np.uint8).reshape(rows, cols)
    scales = oracle.bf16_bits((np.abs(rng.normal(0.0, 0.02, rows * cols // 64)) + 1e-3).astype(np.float32).reshape(rows, cols // 64))
    return oracle.QTensor(oracle.pack_codes(codes, 1), scales, None, 1, rows, cols)


@pytest.mark.parametrize("bits,d,f,e,k,fs,t,tiled", [
    (4, 256, 256, 16, 4, 256, 40, False),    # tiles of 32, the resident kernel
    (4, 256, 512, 4, 2, 512, 150, True),     # tiles of 64
    (4, 192, 320, 8, 2, 128, 70, False),     # widths of odd numbers of groups
    (2, 512, 1024, 8, 2, 256, 33, True),     # the ring in both products, a 4-bit shared expert beside
    (2, 256, 128, 4, 2, 0, 260, False),
    (1, 384, 704, 8, 3, 0, 60, False),
])
def test_prefill_layer_of_rows_far_from_one(gpu, oracle, bits, d, f, e, k, fs, t, tiled):
    layer = oracle.synth_layer(ROOT_SEED + 0x9700 + bits + d, d, f, e, k, bits=bits, fs=fs, with_w_sg=False)
    moe, wts = make_moe(gpu, layer), to_device_layer(layer)
    wts.router_w = None
    if tiled:
        wts.experts_tiled = moe.tile_experts(wts.experts, wts.offsets)
    rng = np.random.default_rng(d + f)
    idx = np.stack([rng.permutation(e)[:k] for _ in range(t)]).astype(np.int32)
    w = rng.random((t, k), dtype=np.float32)
    for powers in (np.resize(_POWERS, t), np.zeros(t)):  # (the second: tiles whose rows are all ordinary)
        xb = _scaled_x(oracle, d + f, t, d, powers)
        y = torch.zeros((t, d), dtype=torch.bfloat16, device="cuda")
        moe.encode_prefill_layer(wts, ops.bf16_tensor(xb), y, t, out_indices=torch.from_numpy(idx).cuda(), out_weights=torch.from_numpy(w).cuda())
        torch.cuda.synchronize()
        ref = np.zeros((t, d), np.float32)
        for i in range(t):
            if fs:
                ref[i] = oracle.bf16_to_float(oracle.shared_expert(*layer.shared, xb[i]))
            for j in range(k):
                blob = layer.experts[idx[i, j]]
                acts = oracle.expert_phase1(blob, layer.off, bits, d, f, xb[i])
                ref[i] += w[i, j] * oracle.expert_down(blob, layer.off, bits, d, f, acts)
        _rows_close(oracle, ops.bf16_bits(y), oracle.bf16_bits(ref), f"prompt bits={bits} d={d} f={f}")


# (d = 7680: the gate / up pair in two windows)
@pytest.mark.parametrize("bits", [4, 2, 1])
@pytest.mark.parametrize("d,f,t", [(256, 192, 40), (1152, 640, 20), (192, 3200, 70), (7680, 256, 66)])
def test_mlp_block_of_rows_far_from_one(gpu, oracle, bits, d, f, t):
    rng = oracle.Rng.key(0xF1E, f"mlp-far-{bits}-{d}-{f}")
    qs = [_weights(oracle, rng, r, c, bits) for r, c in ((f, d), (f, d), (d, f))]
    op = ops.SharedExpertInt4(gpu)
    dev = [ops.QuantizedTensor.from_host(q.packed, q.scales, q.biases, q.bits, q.rows, q.n, "cuda") for q in qs]
    xb = _scaled_x(oracle, d + f, t, d, np.resize(_POWERS, t))
    y = torch.zeros((t, d), dtype=torch.bfloat16, device="cuda")
    op.encode(ops.bf16_tensor(xb), *dev, y, torch.zeros(op.scratch_bytes(d, f, t), dtype=torch.uint8, device="cuda"), t=t)
    torch.cuda.synchronize()
    _rows_close(oracle, ops.bf16_bits(y), np.stack([oracle.shared_expert(*qs, xb[i]) for i in range(t)]), f"mlp bits={bits} d={d} f={f} t={t}")


@pytest.mark.parametrize("bits", [4, 2, 1])
@pytest.mark.parametrize("m,n,k", [(40, 256, 256), (9, 128, 4096), (150, 384, 8192)])
def test_qmm_of_rows_far_from_one(gpu, bits, m, n, k):
    """a power of two on a row is one on its results, bit for bit, whatever the rows beside it hold; values of one sign"""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(m + n + k + bits)
    packed = torch.randint(0, 256, (n, k * (4 if bits == 4 else 2) // 8), generator=gen, device="cuda", dtype=torch.uint8)
    if bits == 1:
        packed &= 0x55  # codes 0 and 1
    scales = (0.01 + 0.01 * torch.rand(n, k // 64, generator=gen, device="cuda")).to(torch.bfloat16)
    biases = -scales if bits == 1 else (-0.1 * torch.rand(n, k // 64, generator=gen, device="cuda")).to(torch.bfloat16)
    q = ops.QuantizedTensor(packed, scales, biases, bits, n, k)
    x = (1.0 + torch.rand(m, k, generator=gen, device="cuda")).to(torch.bfloat16)
    op = ops.MPPPrefillInt4QMM(gpu)
    out = []
    for shifts in (torch.zeros(m), torch.arange(m) % 2 * 59.0, torch.arange(m) % 3 * 50.0, torch.arange(m) % 4 * -33.0):
        factor = (2.0 ** shifts.double()).cuda()[:, None]
        y = torch.zeros((m, n), dtype=torch.float32, device="cuda")
        assert op.encode(q, (x.double() * factor).to(torch.bfloat16), y, m, n, k) == "affine-matrix-core-bf16"
        out.append(y.double() / factor)
    assert all(torch.equal(out[0], o) for o in out[1:])


@pytest.mark.parametrize("bits", [4, 2, 1])
@pytest.mark.parametrize("m,n,t", [(2048, 4096, 8), (1088, 4992, 4), (4672, 11392, 1), (6656, 2048, 3), (64, 256, 5), (130, 320, 2)])
def test_few_rows_far_from_one(gpu, bits, m, n, t):
    """as test_qmm_of_rows_far_from_one, through the kernels of one to eight rows (the larger sizes: quad matrix instructions)"""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(m + n + t + bits)
    packed = torch.randint(0, 256, (m, n * (4 if bits == 4 else 2) // 8), generator=gen, device="cuda", dtype=torch.uint8)
    if bits == 1:
        packed &= 0x55
    scales = (0.01 + 0.01 * torch.rand(m, n // 64, generator=gen, device="cuda")).to(torch.bfloat16)
    biases = -scales if bits == 1 else (-0.1 * torch.rand(m, n // 64, generator=gen, device="cuda")).to(torch.bfloat16)
    q = ops.QuantizedTensor(packed, scales, None if bits == 1 else biases, bits, m, n)
    x = (1.0 + torch.rand(t, n, generator=gen, device="cuda")).to(torch.bfloat16)
    op = ops.DequantInt4GEMVMultiX(gpu)
    out = []
    for shifts in (torch.zeros(t), 59.0 - torch.arange(t) % 2, 100.0 - torch.arange(t) % 3 * 90, -80.0 + torch.arange(t) % 4 * 20):
        factor = (2.0 ** shifts.double()).cuda()[:, None]
        y = torch.zeros((t, m), dtype=torch.float32, device="cuda")
        op.encode(q, (x.double() * factor).to(torch.bfloat16), y, m, n, t, output_float32=True)
        out.append(y.double() / factor)
    assert all(torch.equal(out[0], o) for o in out[1:]) and (out[0] != 0).all()


@pytest.mark.parametrize("bits", [4, 2, 1])
@pytest.mark.parametrize("m,n,t", [(4096, 3072, 4), (4096, 2688, 7), (6144, 6144, 3), (4096, 11136, 5)])
def test_few_rows_far_from_one_in_six_chunks_a_lane(gpu, bits, m, n, t):
    """as above where a lane of the quad kernel takes six chunks of a row: their operands are made in the place of x"""
    test_few_rows_far_from_one(gpu, bits, m, n, t)


@pytest.mark.parametrize("bits", [4, 2])
@pytest.mark.parametrize("m,n,t", [(4096, 4096, 4), (4096, 3136, 3), (5120, 17408, 7)])
def test_few_rows_of_zeros_and_numbers_too_small_for_a_product(gpu, bits, m, n, t):
    """rows of zeros, single zeros and bf16 subnormals beside ordinary rows, whose lanes take the power of two by an addition to the
    exponent fields: a zero has no product and no part in a sum, a row has the bits it has alone"""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(m + n + t + bits)
    q = ops.Quantization(gpu).quantize_affine(torch.randn((m, n), generator=gen, device="cuda") * 0.02 + 0.01, bits)
    x = torch.randn((t, n), generator=gen, device="cuda").to(torch.bfloat16)
    x[0] = 0.0
    x[1, ::3] = 0.0
    x[1, 1::3] = -0.0
    x[2, 5:200] = 2.0 ** -130
    op = ops.DequantInt4GEMVMultiX(gpu)
    y, one = torch.full((t, m), 9.0, device="cuda"), torch.full((1, m), 9.0, device="cuda")
    op.encode(q, x, y, m, n, t, output_float32=True)
    for r in range(t):
        op.encode(q, x[r:r + 1].contiguous(), one, m, n, 1, output_float32=True)
        torch.cuda.synchronize()
        assert torch.equal(one[0], y[r]), r
    assert (y[0] == 0).all()
    without = x.clone()
    without[2, 5:200] = 0.0
    z = torch.zeros_like(y)
    op.encode(q, without, z, m, n, t, output_float32=True)
    torch.cuda.synchronize()
    # 195 numbers of 2^-130 against weights below 1 are under 2^-122: none of it is left in a sum of ordinary ones, which may only be
    # rounded elsewhere on its way (each of the up to 9 sums a lane makes per group, 2^-24 of what it has: under 1e-6 of the whole)
    assert torch.linalg.norm(z[2].double() - y[2].double()) <= 1e-6 * torch.linalg.norm(z[2].double())


@pytest.mark.parametrize("d,f,t,apart", [(128, 64, 16, 1), (576, 128, 70, 1), (192, 2112, 530, 3)])
def test_int8_matmul_of_small_codes_beside_large_values(gpu, d, f, t, apart):
    """every group holds A and -A against the same code and, elsewhere, numbers from 1 to 2 against codes of 1 to 3: gate is
    the sum of the latter, to the last bit of an fp32 sum whose largest term is A = 2^13 (24 bits of it: 2^-10 a term, of 64
    terms of at least 1).  up is one and down picks its row, so y is gate in bf16 (two roundings, 2^-8 of it)."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(d + f + t)
    x = (1.0 + torch.rand(t, d, generator=gen, device="cuda")).to(torch.bfloat16)
    x[:, ::64], x[:, apart::64], x[:, 5] = 2.0 ** 13, -2.0 ** 13, 1.0
    gate = torch.randint(1, 4, (f, d), generator=gen, device="cuda", dtype=torch.uint8)
    gate[:, ::64] = gate[:, apart::64] = 1
    up = torch.zeros((f, d), dtype=torch.uint8, device="cuda")
    up[:, 5] = 1
    down = torch.zeros((d, f), dtype=torch.uint8, device="cuda")
    pick = torch.arange(d, device="cuda") % f
    down[torch.arange(d, device="cuda"), pick] = 1
    one = lambda r, c: torch.ones((r, c // 64), dtype=torch.bfloat16, device="cuda")
    q = [ops.QuantizedTensor(c, one(*c.shape), torch.zeros_like(one(*c.shape)), 8, *c.shape) for c in (gate, up, down)]
    y = torch.zeros((t, d), dtype=torch.bfloat16, device="cuda")
    ops.SharedExpertInt8(gpu, silu_activation=True).encode(x, *q, y, torch.zeros((t, f), dtype=torch.bfloat16, device="cuda"), t=t)
    want = (x.double() @ gate.double().T)[:, pick]
    assert ((y.double() - want).abs() <= want * (2.0 ** -8 + 2.0 ** -10)).all()


@pytest.mark.parametrize("t", [16, 70])
def test_int8_matmul_of_rows_far_from_one(gpu, t):
    """the values the row kernels give, for rows of any magnitude"""
    d, f = 192, 320
    gen = torch.Generator(device="cuda")
    gen.manual_seed(t)
    def q(rows, n):
        table = lambda s: (s * (0.0005 + 0.0005 * torch.rand(rows, n // 64, generator=gen, device="cuda"))).to(torch.bfloat16)
        return ops.QuantizedTensor(torch.randint(0, 256, (rows, n), dtype=torch.uint8, generator=gen, device="cuda"), table(1), table(-128), 8, rows, n)
    qs = [q(f, d), q(f, d), q(d, f)]
    powers = torch.tensor(_POWERS, dtype=torch.float64, device="cuda").repeat(t)[:t, None]
    x = (torch.randn(t, d, generator=gen, device="cuda").double() * 2.0 ** powers).to(torch.bfloat16)
    op = ops.SharedExpertInt8(gpu, silu_activation=True)
    y, rows = torch.zeros((2, t, d), dtype=torch.bfloat16, device="cuda")
    scratch = torch.zeros((t, f), dtype=torch.bfloat16, device="cuda")
    op.encode(x, *qs, y, scratch, t=t)
    for i in range(0, t, 8):
        n = min(8, t - i)
        op.encode(x[i:i + n], *qs, rows[i:i + n], scratch, t=n)
    top = rows.double().abs().amax(dim=1, keepdim=True)
    assert torch.isfinite(rows).all() and (top > 0).all()
    assert (((y.double() - rows.double()) / top).norm(dim=1) <= 2.0 ** -8 * (rows.double() / top).norm(dim=1)).all()  # (_rows_close)
