"""GPU parity: projections with FP8 block-scaled weights (ria_dequant_fp8, ria_linear_fp8[_group]).

The reference dequantises its float8_e4m3fn checkpoint weights once to fp16
(qwen36_dequant.py:35-58, qwen36_cached_loop.py:537-542) and runs fp16
F.linear.  The oracle (oracle.qwen36_cpu.projection_fp8, pinned against
fp64, torch's e4m3fn decoding and transformers' Fp8Dequantize) restates
that; the kernels must give the same dequantised weights bit for bit and
the same fp16 projection up to the order of the fp32 accumulation.
"""

from __future__ import annotations

import pytest
import torch

from conftest import announce
from helpers import assert_act_close
from oracle import qwen36_cpu as O
from router_ia import kernels as K
from router_ia import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("out_dtype", [torch.float16, torch.bfloat16, torch.float32])
def test_dequant_all_byte_values_bit_exact(gpu, out_dtype):
    announce(f"dequant_fp8: all 256 e4m3 bytes x 4 scale blocks -> {out_dtype}")
    w8 = torch.arange(256, dtype=torch.uint8).repeat(130, 1)  # [130, 256]: every byte in every block
    w8[:, :128] = w8[:, :128].roll(7, dims=1)
    s = torch.tensor([[1.0, 0.5], [3.0e-3, 117.25]])
    got = K.dequant_fp8(w8.to(gpu), s.to(gpu), out_dtype).cpu()
    want = O.dequantize_fp8_blockwise(w8.view(torch.float8_e4m3fn), s).to(out_dtype)
    torch.testing.assert_close(got, want, rtol=0, atol=0, equal_nan=True)


CASES = [  # (m, n, k, x dtype): decode batches, one and two 128-row blocks, 16- and 32-wide tiles
    (1, 8192, 2048, torch.bfloat16),   # up to 16 rows and K a multiple of 512: the one-pass decode kernel
    (7, 4096, 2048, torch.float16),
    (16, 2048, 4096, torch.float32),
    (9, 256, 512, torch.bfloat16),     # one wave of K
    (17, 512, 2048, torch.float16),    # one row past the decode kernel: the K-split kernel (fp16 x)
    (32, 2048, 4096, torch.float32),
    (128, 2048, 4096, torch.float16),  # 64-row workgroups: two per 16 features
    (70, 2048, 4096, torch.bfloat16),  # .. the second one with 6 rows
    (128, 512, 2048, torch.bfloat16),
    (128, 8192, 2048, torch.float16),
    (200, 32, 2048, torch.float16),
    (5, 1024, 1408, torch.bfloat16),   # 11 chunks: one ring group and a 3-chunk tail
    (3, 512, 384, torch.float16),      # 3 chunks: the tail alone
    (1, 64, 128, torch.bfloat16),      # one chunk
]


@pytest.mark.parametrize("m,n,k,xdt", CASES)
def test_linear_fp8_matches_oracle(gpu, m, n, k, xdt):
    announce(f"linear_fp8: M={m} N={n} K={k} x {xdt}")
    w8, s = W.fp8_block_weight(200 + m, n, k)
    g = torch.Generator().manual_seed(300 + m)
    # x rows inside a wider buffer (a strided view, as a fused projection output would be)
    wide = torch.randn((m, k + 64), generator=g).to(xdt)
    x = wide[:, :k]
    got = K.linear_fp8(x.to(gpu), w8.to(gpu), s.to(gpu)).cpu()
    want = O.projection_fp8(x, w8, s)
    assert got.dtype == torch.float16
    assert_act_close(got, want, f"M={m} N={n} K={k}")
    # Against the exact product of the same fp16 operands, the kernel is as
    # accurate as the oracle's fp32-accumulated F.linear: both err by the fp16
    # rounding of the result plus an fp32 summation error that depends on the
    # order (about 1e-4 here, where the K terms sum to ~26 in magnitude).
    w16 = O.dequantize_fp8_blockwise(w8, s).to(torch.float16)
    exact = x.to(torch.float16).double() @ w16.double().T
    e_got = (got.double() - exact).abs().max().item()
    e_ref = (want.double() - exact).abs().max().item()
    assert e_got <= 1.5 * e_ref + 1e-6, (e_got, e_ref)


KSPLIT_F16 = [  # fp16 x past 16 rows (the forward loop's projections): the K-split kernel's
    (96, 12288, 2048),   # tile shapes, with whole and partial row blocks and column tiles
    (128, 8192, 2048),
    (100, 20480, 2048),
    (64, 8192, 512),
    (128, 2048, 4096),   # the output projections' shape
    (128, 8192, 4096),   # K = 4096 with a wide N: 64-row x 64-feature tiles
    (70, 2048, 4096),
    (17, 512, 512),
    (33, 96, 128),       # one chunk of K, a partial last column tile
]


@pytest.mark.parametrize("m,n,k", KSPLIT_F16)
def test_ksplit_kernel_fp16_x_matches_oracle(gpu, m, n, k):
    announce(f"linear_fp8 K-split: M={m} N={n} K={k} x fp16")
    w8, s = W.fp8_block_weight(250 + m, n, k)
    g = torch.Generator().manual_seed(350 + m)
    wide = torch.randn((m, k + 64), generator=g).to(torch.float16)
    x = wide[:, :k]
    got = K.linear_fp8(x.to(gpu), w8.to(gpu), s.to(gpu)).cpu()
    want = O.projection_fp8(x, w8, s)
    assert_act_close(got, want, f"M={m} N={n} K={k}")
    w16 = O.dequantize_fp8_blockwise(w8, s).to(torch.float16)
    exact = x.double() @ w16.double().T
    e_got = (got.double() - exact).abs().max().item()
    e_ref = (want.double() - exact).abs().max().item()
    assert e_got <= 1.5 * e_ref + 1e-6, (e_got, e_ref)


@pytest.mark.parametrize("m", [9, 100])
def test_linear_fp8_output_dtypes_round_through_fp16(gpu, m):
    announce(f"linear_fp8: M={m} fp32 and bf16 outputs carry the fp16 result")
    w8, s = W.fp8_block_weight(400, 512, 2048)
    x = torch.randn((m, 2048), generator=torch.Generator().manual_seed(401)).to(torch.bfloat16).to(gpu)
    w8, s = w8.to(gpu), s.to(gpu)
    y16 = K.linear_fp8(x, w8, s)
    y32 = K.linear_fp8(x, w8, s, out_dtype=torch.float32)
    yb = K.linear_fp8(x, w8, s, out_dtype=torch.bfloat16)
    torch.cuda.synchronize()
    assert torch.equal(y32.cpu(), y16.cpu().float())
    assert torch.equal(yb.cpu(), y16.cpu().to(torch.bfloat16))


GROUPS = [  # (m, [n_j], k): a DeltaNet layer's input projections, attention q/k/v, 16-wide tiles
    (1, [8192, 4096, 32, 32], 2048),
    (128, [8192, 4096, 32, 32], 2048),
    (37, [8192, 512, 512], 2048),
    (130, [48, 256], 1408),
    (40, [8192, 48], 2048),   # 64-wide tiles: the 48-wide projection fills part of one
]


@pytest.mark.parametrize("xdt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m,ns,k", GROUPS)
def test_linear_fp8_group_equals_separate_calls(gpu, m, ns, k, xdt):
    announce(f"linear_fp8_group: M={m} N={ns} K={k} x {xdt}")
    proj = [W.fp8_block_weight(500 + j, n, k) for j, n in enumerate(ns)]
    x = torch.randn((m, k), generator=torch.Generator().manual_seed(510 + m)).to(xdt).to(gpu)
    proj_d = [(w.to(gpu), s.to(gpu)) for w, s in proj]
    dts = [torch.bfloat16, torch.float32, torch.float16, torch.float32][:len(ns)]  # each projection its own dtype
    ys = K.linear_fp8_group(x, proj_d, out_dtype=dts)
    for j, (w, s) in enumerate(proj_d):
        sep = K.linear_fp8(x, w, s, out_dtype=dts[j])
        torch.cuda.synchronize()
        assert ys[j].dtype == dts[j] and torch.equal(ys[j].cpu(), sep.cpu()), f"projection {j}"
    # and each against the oracle
    for j, (w, s) in enumerate(proj):
        want = O.projection_fp8(x.cpu(), w, s).to(dts[j])
        assert_act_close(ys[j].cpu(), want, f"projection {j}")


@pytest.mark.parametrize("m,n,k", [(100, 8192, 2048), (128, 2048, 4096), (37, 96, 128)])
def test_bf16_x_equals_its_fp16_conversion(gpu, m, n, k):
    """F.linear takes h.to(float16): bf16 x past 16 rows is converted inside the
    K-split kernel, which must give the bits of the same call on x.to(float16)
    (values spanning fp16's normal range, small ones included)."""
    announce(f"linear_fp8 bf16 x: M={m} N={n} K={k}")
    w8, s = W.fp8_block_weight(700 + m, n, k)
    g = torch.Generator().manual_seed(710 + m)
    x = torch.randn((m, k), generator=g) * torch.exp2(torch.randint(-12, 8, (m, k), generator=g).float())
    xb = x.to(torch.bfloat16).to(gpu)
    wd, sd = w8.to(gpu), s.to(gpu)
    got = K.linear_fp8(xb, wd, sd)
    ref = K.linear_fp8(xb.to(torch.float16), wd, sd)
    torch.cuda.synchronize()
    assert torch.equal(got.cpu(), ref.cpu())


@pytest.mark.parametrize("m", [3, 100, 128])  # one-pass kernel; past 16 rows with partial and with whole row blocks
def test_linear_fp8_group_accumulates_into_fp32(gpu, m):
    announce(f"linear_fp8_group: M={m} y += fp16 result (residual add)")
    w8, s = W.fp8_block_weight(600, 2048, 4096)
    g = torch.Generator().manual_seed(601)
    x = torch.randn((m, 4096), generator=g).to(torch.float16).to(gpu)
    base = torch.randn((m, 2048), generator=g).to(gpu)
    y = base.clone()
    K.linear_fp8_group(x, [(w8.to(gpu), s.to(gpu))], out=[y], accumulate=[True])
    sep = K.linear_fp8(x, w8.to(gpu), s.to(gpu), out_dtype=torch.float32)
    torch.cuda.synchronize()
    assert torch.equal(y.cpu(), base.cpu() + sep.cpu())


@pytest.mark.parametrize("m,k,hdt", [(1, 2048, torch.bfloat16), (3, 2048, torch.float16), (4, 4096, torch.bfloat16)])
def test_linear_fp8_group_with_fused_input_norm(gpu, m, k, hdt):
    announce(f"linear_fp8_group_normed: M={m} K={k} h {hdt}")
    ns = [8192, 4096, 32, 32] if k == 2048 else [2048]
    proj = [W.fp8_block_weight(700 + j, n, k) for j, n in enumerate(ns)]
    g = torch.Generator().manual_seed(710 + m)
    x = (torch.randn((m, k), generator=g) * 3.0).to(gpu)
    wn = (torch.randn((k,), generator=g) * 0.1).to(torch.bfloat16).float().to(gpu)
    proj_d = [(w.to(gpu), s.to(gpu)) for w, s in proj]
    fused = K.linear_fp8_group(x, proj_d, norm_weight=wn, norm_dtype=hdt)
    h = K.rmsnorm(x, wn, out=torch.empty((m, k), dtype=hdt, device=gpu))
    separate = K.linear_fp8_group(h, proj_d)
    for j, (w, s) in enumerate(proj):
        # both against the oracle's rmsnorm -> dtype -> fp16 projection
        want = O.projection_fp8(O.rmsnorm(x.cpu(), wn.cpu()).to(hdt), w, s)
        assert_act_close(fused[j].cpu(), want, f"fused projection {j}")
        assert_act_close(separate[j].cpu(), want, f"separate projection {j}")


def test_linear_fp8_group_normed_host_checks(gpu):
    w8, s = W.fp8_block_weight(720, 64, 2048)
    x = torch.randn((5, 2048)).to(gpu)
    wn = torch.zeros((2048,), device=gpu)
    with pytest.raises(RuntimeError, match="up to 4 rows"):
        K.linear_fp8_group(x, [(w8.to(gpu), s.to(gpu))], norm_weight=wn)


@pytest.mark.parametrize("xdt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m,ns,k", [
    (193, [8192, 32], 2048),            # fewest rows, 128 x 128 tiles, a 32-wide projection
    (255, [48, 272], 128),              # few features: the K-split kernel, fewer chunks of K than its waves
    (777, [8192, 4096, 32, 32], 2048),  # 128 x 128 tiles, two to a CU, 9 rows past a tile
    (4097, [272, 1040], 384),           # 256 x 128 tiles, one row past a tile, three scale blocks of K
    (1345, [512], 4096),                # few tiles at K = 4096: the K-split kernel
    (16400, [2064], 384),               # 256 x 256 tiles, 16 rows and 16 features past a tile
    (131089, [272, 16], 128),           # 256 x 256 tiles of two steps of K, and 16 features in the other launch
])
def test_many_row_kernel(gpu, m, ns, k, xdt):
    """Prompt-sized calls against the exact product of the same fp16 operands
    (error within 1.5x of an fp32-accumulated product's own), grouped calls
    equal to separate ones, the fp32 / bf16 outputs and the residual add equal
    to the fp16 result, and nothing written past the result's columns."""
    announce(f"linear_fp8 many rows: M={m} N={ns} K={k} x {xdt}")
    proj = [tuple(t.to(gpu) for t in W.fp8_block_weight(800 + j, n, k)) for j, n in enumerate(ns)]
    g = torch.Generator().manual_seed(810 + m)
    x = torch.randn((m, k + 8), generator=g).to(xdt).to(gpu)[:, :k]
    ys = K.linear_fp8_group(x, proj)
    for j, (w, s) in enumerate(proj):
        w16 = K.dequant_fp8(w, s, torch.float16)
        exact = x.to(torch.float16).double() @ w16.double().t()
        ref = (x.to(torch.float16).float() @ w16.float().t()).to(torch.float16)
        e_got, e_ref = ((t.double() - exact).abs().max().item() for t in (ys[j], ref))
        assert e_got <= 1.5 * e_ref + 1e-6, (j, e_got, e_ref)
        wide = torch.full((m, ns[j] + 3), 7.0, device=gpu)  # rows that are not 16-byte aligned
        K.linear_fp8(x, w, s, out=wide[:, :ns[j]])
        assert torch.equal(wide[:, :ns[j]], ys[j].float()) and bool((wide[:, ns[j]:] == 7.0).all())
        assert torch.equal(K.linear_fp8(x, w, s, out_dtype=torch.float32), ys[j].float())
        assert torch.equal(K.linear_fp8(x, w, s, out_dtype=torch.bfloat16), ys[j].to(torch.bfloat16))
        base = torch.randn((m, ns[j]), generator=g).to(gpu)
        y = base.clone()
        K.linear_fp8_group(x, [(w, s)], out=[y], accumulate=[True])
        assert torch.equal(y, base + ys[j].float())


@pytest.mark.parametrize("xdt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m,n,k", [
    (193, 512, 2048), (256, 2048, 4096),  # few tiles: the K-split kernel
    (257, 8192, 128), (321, 8208, 4224),  # 128 x 128 tiles, fewer chunks of K than sums, a feature tile of 16
    (450, 12352, 384), (513, 9216, 2048),  # 256 x 128 tiles, a ragged last chunk of the sums, one row past a tile
])
def test_rows_do_not_depend_on_the_call(gpu, m, n, k, xdt):
    """A prompt's projection against the same rows in calls of 96 to 160 rows:
    whatever kernel and tile a call takes below 2^25 results, the same bits."""
    announce(f"linear_fp8 rows of a call: M={m} N={n} K={k} x {xdt}")
    w, s = (t.to(gpu) for t in W.fp8_block_weight(900 + k, n, k))
    x = torch.randn((m, k), generator=torch.Generator().manual_seed(910 + m)).to(xdt).to(gpu)
    whole = K.linear_fp8(x, w, s)
    assert torch.equal(whole, torch.cat([K.linear_fp8(part, w, s) for part in x.chunk((m + 159) // 160)]))


@pytest.mark.parametrize("xdt", [torch.bfloat16, torch.float16])
def test_group_of_two_launches(gpu, xdt):
    """A group whose projections take different kernels (2048 features of 16400
    rows are more than 2^25 results): the bits of separate calls, each within
    1.5x of the fp32-accumulated product's error."""
    m, ns, k = 16400, [512, 2048, 32], 256
    announce(f"linear_fp8_group in two launches: M={m} N={ns} K={k} x {xdt}")
    proj = [tuple(t.to(gpu) for t in W.fp8_block_weight(930 + j, n, k)) for j, n in enumerate(ns)]
    x = torch.randn((m, k), generator=torch.Generator().manual_seed(940)).to(xdt).to(gpu)
    for y, (w, s) in zip(K.linear_fp8_group(x, proj), proj):
        assert torch.equal(y, K.linear_fp8(x, w, s))
        w16, x16 = K.dequant_fp8(w, s, torch.float16), x.to(torch.float16)
        exact = x16.double() @ w16.double().t()
        e_got, e_ref = ((t.double() - exact).abs().max().item() for t in (y, (x16.float() @ w16.float().t()).half()))
        assert e_got <= 1.5 * e_ref + 1e-6, (e_got, e_ref)
