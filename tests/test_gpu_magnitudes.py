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
    """row by row: a row of large numbers must not speak for the others"""
    got, ref = oracle.bf16_to_float(got_bits).astype(np.float64), oracle.bf16_to_float(ref_bits).astype(np.float64)
    assert np.isfinite(ref).all() and (np.abs(ref).max(axis=1) > 0).all(), what
    for i, (g, r) in enumerate(zip(got, ref)):
        top = np.abs(r).max()
        _, rel = errors(g / top, r / top)
        assert np.isfinite(g).all() and rel <= 1e-3, (what, i, rel)


# x of 2^-50 gives activations of 2^-100; of 2^50, of 2^100
_POWERS = [0, 50, -50, 23, -24, 12, 58, -30]


@pytest.mark.parametrize("bits,d,f,e,k,t,form", [
    (4, 256, 128, 16, 4, 8, "fused"), (4, 2048, 512, 16, 8, 5, "fused"), (4, 704, 448, 12, 4, 1, "fused"), (2, 1024, 320, 16, 6, 8, "fused"),
    (2, 4096, 128, 16, 2, 1, "fused"), (1, 512, 256, 32, 8, 3, "fused"), (2, 128, 64, 16, 3, 7, "fused"), (4, 8192, 128, 4, 2, 8, "fused"),
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
