"""GPU parity of the fused QKV projection (one launch over the Q, K and V
matrices' column tiles at decode and mid sizes) against the fp32 reference built from
the bit-exact dequant, plus the oracle on a small ragged case."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from gpu_helpers import TOL, announce, max_abs_rel, to_dev, to_np
from oracle import fp4 as ofp4

pytestmark = pytest.mark.gpu


def _weights(gen, K, N, g):
    import mmfp4
    w = (torch.randn((N, K), generator=gen, device="cuda") * 0.02).half()
    p, s = mmfp4.quantize_fp4(w, group_size=g)
    return p, s, mmfp4.dequant_fp4(p, s, K, N, g).float()


@pytest.mark.parametrize("M,K,Ns,g", [(1, 4096, (4096, 1024, 1024), 128),
                                      (8, 4096, (4096, 1024, 1024), 128),
                                      (16, 14336, (512, 256, 256), 128),
                                      (17, 4096, (4096, 1024, 1024), 128),
                                      (64, 4096, (4096, 1024, 1024), 128),
                                      (3, 1024, (260, 132, 68), 32),
                                      (1, 512, (258, 130, 64), 64)])
def test_fused_qkv_vs_fp32_reference(M, K, Ns, g):
    import mmfp4
    gen = torch.Generator(device="cuda").manual_seed(M + K)
    mats = [_weights(gen, K, n, g) for n in Ns]
    x = torch.randn((M, K), generator=gen, device="cuda").half()
    announce(f"fused qkv M={M} K={K} Ns={Ns}")
    outs = mmfp4.mmfp4_fused_qkv(x, mats[0][0], mats[0][1], mats[1][0], mats[1][1], mats[2][0],
                                 mats[2][1], g)
    for o, (_, _, w), n in zip(outs, mats, Ns):
        assert tuple(o.shape) == (M, n)
        assert max_abs_rel(to_np(o), to_np(x.float() @ w)) <= TOL
    again = mmfp4.mmfp4_fused_qkv(x, mats[0][0], mats[0][1], mats[1][0], mats[1][1], mats[2][0],
                                  mats[2][1], g)
    for o, o2 in zip(outs, again):
        assert torch.equal(o, o2)


def test_fused_qkv_1d_input_vs_oracle(rng):
    import mmfp4
    K, Ns, g = 256, (64, 32, 32), 64
    ws = [ofp4.quantize_fp4(rng.normal(0, 0.02, (n, K)).astype(np.float16), g) for n in Ns]
    x = rng.normal(0, 1, (K,)).astype(np.float16)
    announce("fused qkv 1-D input vs oracle")
    outs = mmfp4.mmfp4_fused_qkv(to_dev(x), *[to_dev(t) for pair in ws for t in pair], g)
    for o, (p, s), n in zip(outs, ws, Ns):
        assert tuple(o.shape) == (1, n)
        ref = x.astype(np.float32)[None] @ ofp4.dequant_fp4_f32(p, s, g)
        assert max_abs_rel(to_np(o), ref) <= TOL


def test_fused_qkv_more_columns_than_one_launch_takes():
    """17..32 rows, over a million columns together but not each: as three products."""
    import mmfp4
    M, K, N, g = 20, 64, 400_000, 64
    gen = torch.Generator("cuda").manual_seed(5)
    mats = [(torch.randint(-2**31, 2**31 - 1, (K // 8, N), device="cuda", dtype=torch.int32,
                           generator=gen),
             (torch.rand(1, N, device="cuda", generator=gen) * 0.01).half()) for _ in range(3)]
    x = torch.randn(M, K, device="cuda", generator=gen).half()
    announce(f"fused qkv M={M} N=3 x {N}")
    outs = mmfp4.mmfp4_fused_qkv(x, *[t for m in mats for t in m], g)
    for o, m in zip(outs, mats):
        assert torch.equal(o, mmfp4.marlin_gemm_fp4(x, *m, g))


def test_fused_qkv_errors():
    import mmfp4
    x = torch.zeros((1, 64), dtype=torch.float16, device="cuda")
    p = torch.zeros((8, 16), dtype=torch.int32, device="cuda")
    s = torch.zeros((1, 16), dtype=torch.float16, device="cuda")
    with pytest.raises(ValueError, match="K weights: K mismatch"):
        mmfp4.mmfp4_fused_qkv(x, p, s, p[:4], s, p, s, 64)


@pytest.mark.parametrize("M", [1, 40])
def test_binding_and_ctypes_agree(monkeypatch, M):
    """The fused projections and the row-packed product through the per-call
    binding and through ctypes: same results, and operands that are not in the
    binding's plain form (strided, other types) give them too."""
    import mmfp4
    from mmfp4 import kernels
    K, N, g = 256, 72, 64
    gen = torch.Generator("cuda").manual_seed(3)
    w = torch.randn(3, N, K, device="cuda", generator=gen) * 0.02
    marlin = [t for i in range(3) for t in mmfp4.quantize_fp4(w[i], g)]
    rows = [t.t().contiguous() if i % 2 == 0 else t for i, t in enumerate(marlin)]
    x = torch.randn(M, K, device="cuda", generator=gen).half()
    odd = [marlin[0].t().contiguous().t(), marlin[1].float()] + marlin[2:]

    def calls():
        yield from mmfp4.mmfp4_fused_qkv(x, *marlin, g)
        yield from mmfp4.mmfp4_fused_qkv(x.float(), *odd, g)
        yield mmfp4.mmfp4_fused_gate_up_marlin(x, *marlin[:4], g)
        yield mmfp4.fused_gate_up_gemm(x, *odd[:4], g)
        yield mmfp4.mmfp4_fused_gate_up(x, *rows[:4], g)
        yield mmfp4.mmfp4_gemm_rowpacked(x, rows[0], rows[1], g)
        yield mmfp4.mmfp4_gemm_rowpacked(x, rows[0], rows[1].t().contiguous(), g)

    announce(f"binding against ctypes M={M}")
    # the binding is there, takes the plain operands and leaves the others
    assert kernels._binding()
    bad = (x.float(), x.t().contiguous().t()) if M > 1 else (x.float(),)
    for args, plain in [((x, *odd[:4]), False), ((x, *marlin[:4]), True)] + \
            [((b, *marlin[:4]), False) for b in bad]:
        b, w0, s0, w1, s1 = args
        r0, r1 = w0.t().contiguous(), w1.t().contiguous()
        took = [kernels._fast("qkv", b, (w0, w1, w0), (s0, s1, s0), g),
                kernels._fast("gate_up", b, w0, s0, w1, s1, g, False, True),
                kernels._fast("gate_up", b, r0, s0, r1, s1, g, True, True),
                kernels._fast("rowpacked", b, r0, s0, g)]
        assert [t is not None for t in took] == [plain] * 4
    fast = list(calls())
    monkeypatch.setattr(kernels, "_BINDING", False)
    for a, b in zip(fast, calls(), strict=True):
        assert a.shape == b.shape and torch.equal(a, b)
