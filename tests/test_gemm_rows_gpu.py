"""A8 over many rows (prefill): the large-tile projection kernels against Int8Linear in fp32.

Sizes reach each tile (128 x 128, 128 x 256, 256 x 256) with row counts one below, at and one
past its edges; every case pins the kernel that serves it.  Bars: 2.5e-3 relative for a plain product, whose only rounding beside fp32
sums is the bf16 output (2^-9, 1.1e-3 rms); 5e-3 for SwiGLU, which rounds gate, up, silu and
the product (four such, 2.3e-3).
"""

from __future__ import annotations

import pytest
import torch

from helpers import rel_err
from nanoengine_amd import _native, kernels
from nanoengine_amd._native import EPILOGUE_SWIGLU

pytestmark = pytest.mark.gpu


def weight(n, k, device, scale_dtype=torch.bfloat16, seed=0):
    g = torch.Generator(device=device).manual_seed(seed + n + k)
    codes = torch.randint(-127, 128, (n, k), dtype=torch.int8, device=device, generator=g)
    scales = torch.rand(n, device=device, generator=g) * 3e-4 + 1e-4
    return codes, scales.to(scale_dtype)


def product(x, w, s):
    return (x.float() @ w.float().t()) * s.float()


STAGED, FEW_ROWS, TILE_128X128, TILE_128X256, TILE_256X256 = range(5)


def kernel_of(m, n, k, splits=0, epilogue=0):
    return _native.load().ne_w8a16_kernel(m, n, k, splits, epilogue)


@pytest.mark.parametrize("tile,m,n,k", [
    (TILE_128X128, 897, 4096, 1024), (TILE_128X128, 1024, 4096, 128), (TILE_128X128, 1023, 4096, 256),
    (TILE_128X128, 1000, 4096, 384), (TILE_128X128, 641, 4096, 1024), (TILE_128X128, 2561, 1024, 2048),
    (TILE_128X256, 2047, 4096, 1024), (TILE_128X256, 2048, 4096, 128), (TILE_128X256, 2000, 4096, 384),
    (TILE_128X256, 4321, 1024, 2048), (TILE_128X256, 8191, 1024, 3072),
    (TILE_256X256, 3841, 4096, 1024), (TILE_256X256, 4096, 4096, 128), (TILE_256X256, 4095, 4096, 256),
    (STAGED, 4097, 1024, 2048), (TILE_128X256, 17, 65536, 1024),
])
def test_product(device, tile, m, n, k):
    assert kernel_of(m, n, k) == tile
    w, s = weight(n, k, device)
    x = torch.randn(m, k, device=device, generator=torch.Generator(device=device).manual_seed(m)).to(torch.bfloat16)
    out = kernels.w8a16_gemm(x, w, s)
    assert rel_err(out, product(x, w, s)) < 2.5e-3


@pytest.mark.parametrize("scale_dtype", [torch.float16, torch.float32])
def test_scale_types_and_strides(device, scale_dtype):
    w, s = weight(4096, 512, device, scale_dtype)
    wide = torch.randn(1001, 640, device=device).to(torch.bfloat16)
    x = wide[:, 64:576]
    out = torch.zeros(1002, 4096, dtype=torch.bfloat16, device=device)
    kernels.w8a16_gemm(x, w, s, out=out[:1001])
    assert rel_err(out[:1001], product(x, w, s)) < 2.5e-3
    assert not out[1001].any()  # the row after the last


# the two-k-group tile at its first and last rows, one row past and one before the others' edges
@pytest.mark.parametrize("tile,m", [
    (TILE_128X128, 561), (TILE_128X128, 600), (TILE_128X128, 639), (TILE_128X128, 640), (STAGED, 641),
    (TILE_128X256, 881), (TILE_128X256, 1025), (TILE_128X256, 1280), (STAGED, 1537), (TILE_256X256, 1601),
    (TILE_256X256, 2049), (TILE_256X256, 2560),
])
def test_swiglu(device, tile, m):
    assert kernel_of(m, 6144, 1024, epilogue=EPILOGUE_SWIGLU) == tile
    gate, gs = weight(3072, 1024, device, seed=1)
    up, us = weight(3072, 1024, device, seed=2)
    pair = lambda a, b: torch.stack([a.view(-1, 16, *a.shape[1:]), b.view(-1, 16, *b.shape[1:])], 1).flatten(0, 2)
    x = torch.randn(m, 1024, device=device).to(torch.bfloat16)
    out = kernels.w8a16_gemm(x, pair(gate, up).contiguous(), pair(gs, us).contiguous(), epilogue=EPILOGUE_SWIGLU)
    ref = torch.nn.functional.silu(product(x, gate, gs)) * product(x, up, us)
    assert out.shape == (m, 3072) and rel_err(out, ref) < 5e-3


@pytest.mark.parametrize("kv", ["int8-bf16-scales", "int8-fp16-scales", "bf16"])
@pytest.mark.parametrize("tile,m", [(TILE_128X128, 1000), (TILE_128X256, 2047), (TILE_256X256, 3900)])
def test_fused_qkv_equals_gemm_then_row_kernel(device, kv, tile, m):
    """The tiles' QK-norm + RoPE + KV-write epilogue gives the bits of the plain product
    followed by the row kernel, rows past the last written nowhere."""
    hq, hkv, k, slots_n = 16, 8, 1024, 5000
    assert kernel_of(m, 4096, k) == tile
    g = torch.Generator(device=device).manual_seed(m)
    w, s = weight(4096, k, device)
    x = torch.randn(m, k, device=device, generator=g).to(torch.bfloat16)
    x[5] = 0  # a zero row: zero vectors, the smallest scale
    q_norm, k_norm = ((1 + 0.1 * torch.randn(128, device=device, generator=g)).to(torch.bfloat16) for _ in range(2))
    positions = torch.randint(0, 6000, (m,), generator=g, dtype=torch.int32, device=device)
    rope = kernels.rope_table(6000, 1e6).to(device)
    slots = torch.randperm(slots_n, generator=g, device=device)[:m].to(torch.int32)

    def pool():
        if kv == "bf16":
            return [torch.zeros(slots_n, hkv, 128, dtype=torch.bfloat16, device=device) for _ in range(2)] + [None, None]
        sdt = torch.bfloat16 if kv == "int8-bf16-scales" else torch.float16
        return ([torch.zeros(slots_n, hkv, 128, dtype=torch.int8, device=device) for _ in range(2)]
                + [torch.zeros(slots_n, hkv, dtype=sdt, device=device) for _ in range(2)])

    a, b = pool(), pool()
    q_ref = kernels.qk_norm_rope_kv_write(kernels.w8a16_gemm(x, w, s), hq, hkv, q_norm, k_norm, 1e-6, positions, rope,
                                          slots, *a)
    q_out = torch.zeros(m + 1, hq, 128, dtype=torch.bfloat16, device=device)
    kernels.w8a16_qkv_norm_rope_kv(x, w, s, hq, hkv, q_norm, k_norm, 1e-6, positions, rope, slots, *b, q_out=q_out[:m])
    assert torch.equal(q_out[:m].view(torch.int16), q_ref.view(torch.int16)) and not q_out[m].any()
    for ta, tb in zip(a, b):
        if ta is not None:
            assert torch.equal(ta.view(torch.uint8), tb.view(torch.uint8))
    assert int(a[0].view(torch.uint8).ne(0).sum()) > 0


def test_unaligned_cache_takes_the_other_kernel(device):
    """A pool that starts at an odd byte (the row kernel stores single codes) is still written."""
    hq, hkv, k, m, n_slots = 16, 8, 256, 1000, 1100
    w, s = weight(4096, k, device)
    x = torch.randn(m, k, device=device).to(torch.bfloat16)
    ones = torch.ones(128, dtype=torch.bfloat16, device=device)
    pos = torch.arange(m, dtype=torch.int32, device=device)
    rope = kernels.rope_table(1024, 1e6).to(device)
    size = n_slots * hkv * 128
    raw = [torch.zeros(size + 1, dtype=torch.int8, device=device) for _ in range(2)]
    odd = [t[1:].view(n_slots, hkv, 128) for t in raw]
    even = [torch.zeros(n_slots, hkv, 128, dtype=torch.int8, device=device) for _ in range(2)]
    for caches in (odd, even):
        scales = [torch.zeros(n_slots, hkv, dtype=torch.bfloat16, device=device) for _ in range(2)]
        kernels.w8a16_qkv_norm_rope_kv(x, w, s, hq, hkv, ones, ones, 1e-6, pos, rope, pos, *caches, *scales,
                                       q_out=torch.empty(m, hq, 128, dtype=torch.bfloat16, device=device))
    # another summation order: a code may differ by the rounding of a tie
    for o, e in zip(odd, even):
        assert int((o.int() - e.int()).abs().max()) <= 2 and float((o != e).float().mean()) < 0.02


@pytest.mark.parametrize("m,pad,first", [(321, 4, 0), (330, 8, 4), (320, 8, 0), (640, 8, 0)])
def test_outputs_of_every_row_alignment(device, m, pad, first):
    """Rows that do not start on 16 bytes leave in 8-byte stores: the same bits, and nothing
    beyond the columns, from the projection tiles and the LM head (full and short blocks)."""
    g = torch.Generator(device=device).manual_seed(m)
    w, s = weight(4096, 256, device)
    embed = (torch.randn(65664, 256, device=device, generator=g) * 0.02).to(torch.bfloat16)
    for rows, n, call in ((1000, 4096, lambda x, out: kernels.w8a16_gemm(x, w, s, out=out)),
                          (m, 65664, lambda x, out: kernels.lm_head(x, embed, logits=out))):
        x = torch.randn(rows, 256, device=device, generator=g).to(torch.bfloat16)
        plain = torch.empty(rows, n, dtype=torch.bfloat16, device=device)
        call(x, plain)
        assert rel_err(plain, product(x, w, s) if n == 4096 else x.float() @ embed.float().t()) < 2.5e-3
        ld = n + pad
        flat = torch.zeros(rows * ld + 16, dtype=torch.bfloat16, device=device)
        view = flat[first:first + rows * ld].view(rows, ld)
        call(x, view[:, :n])
        assert torch.equal(view[:, :n], plain)
        assert not view[:, n:].any() and not flat[:first].any() and not flat[first + rows * ld:].any()


@pytest.mark.parametrize("m", [1, 5, 16, 17])
def test_few_rows_give_the_bits_of_many(device, m):
    """Up to 16 rows run their own kernel; it adds every output in the order of the kernel
    that 320 rows run, so a row's results do not depend on how many there are: plain,
    SwiGLU, split-K (K 512, 768 and 1,024 a split) and, with the cache, the fused QKV."""
    g = torch.Generator(device=device).manual_seed(m)
    for n, k, splits in ((4096, 1024, 0), (1024, 2048, 4), (1024, 3072, 4), (1024, 2048, 2)):
        for scale_dtype in (torch.bfloat16, torch.float16, torch.float32):
            w, s = weight(n, k, device, scale_dtype)
            x = torch.randn(320, k, device=device, generator=g).to(torch.bfloat16)
            if splits:
                few = kernels.w8a16_gemm_splitk(x[:m], w, s, splits)
                many = kernels.w8a16_gemm_splitk(x, w, s, splits)
                assert torch.equal(few.view(splits, m, n), many.view(splits, 320, n)[:, :m])
            else:
                assert torch.equal(kernels.w8a16_gemm(x[:m], w, s), kernels.w8a16_gemm(x, w, s)[:m])
    w, s = weight(6144, 1024, device)
    x = torch.randn(320, 1024, device=device, generator=g).to(torch.bfloat16)
    assert torch.equal(kernels.w8a16_gemm(x[:m], w, s, epilogue=EPILOGUE_SWIGLU),
                       kernels.w8a16_gemm(x, w, s, epilogue=EPILOGUE_SWIGLU)[:m])
    w, s = weight(4096, 1024, device)
    norms = [(1 + 0.1 * torch.randn(128, device=device, generator=g)).to(torch.bfloat16) for _ in range(2)]
    positions = torch.randint(0, 3000, (320,), generator=g, dtype=torch.int32, device=device)
    rope = kernels.rope_table(3000, 1e6).to(device)
    slots = torch.randperm(400, generator=g, device=device)[:320].to(torch.int32)
    for dtype in (torch.int8, torch.bfloat16):
        results = []
        for rows in (m, 320):
            caches = [torch.zeros(400, 8, 128, dtype=dtype, device=device) for _ in range(2)]
            scales = [torch.zeros(400, 8, dtype=torch.bfloat16, device=device) for _ in range(2)]
            q = torch.zeros(rows + 1, 16, 128, dtype=torch.bfloat16, device=device)
            kernels.w8a16_qkv_norm_rope_kv(x[:rows], w, s, 16, 8, *norms, 1e-6, positions[:rows], rope, slots[:rows],
                                           *caches, *(scales if dtype == torch.int8 else (None, None)), q_out=q[:rows])
            assert not q[rows].any()
            mine = slots[:m].long()
            results.append([q[:m]] + [c[mine] for c in caches] + [t[mine] for t in scales])
            if rows == m:
                other = torch.ones(400, dtype=torch.bool, device=device)
                other[mine] = False
                assert not any(c[other].any() for c in caches)
        for a, b in zip(*results):
            assert torch.equal(a, b)


@pytest.mark.parametrize("m", [1, 16])
def test_few_rows_of_a_wide_product_run_the_few_rows_kernel(device, m):
    """One split of the split-K product is the plain product's sum, in fp32."""
    w, s = weight(65536, 1024, device)
    x = torch.randn(m, 1024, device=device, generator=torch.Generator(device=device).manual_seed(m)).to(torch.bfloat16)
    assert torch.equal(kernels.w8a16_gemm(x, w, s),
                       kernels.w8a16_gemm_splitk(x, w, s, 1).view(m, 65536).to(torch.bfloat16))


# stage counts other than the benchmark model's 8 (K = 1,024) and 4, 6, 8 of a split product
@pytest.mark.parametrize("k", [128, 256, 384, 512, 640, 768, 896, 1024])
def test_few_rows_over_any_k(device, k):
    """Every K (per split) of up to 1,024 runs the few-rows kernel and gives a row the bits it
    has among 320, plain, paired, split and through the fused QKV epilogue."""
    m, g = 5, torch.Generator(device=device).manual_seed(k)
    x = torch.randn(320, 4 * k, device=device, generator=g).to(torch.bfloat16)
    for n, epilogue in ((4096, 0), (6144, EPILOGUE_SWIGLU)):
        assert kernel_of(m, n, k, 0, epilogue) == FEW_ROWS and kernel_of(320, n, k, 0, epilogue) == STAGED
        w, s = weight(n, k, device)
        few = kernels.w8a16_gemm(x[:m, :k], w, s, epilogue=epilogue)
        assert torch.equal(few, kernels.w8a16_gemm(x[:, :k], w, s, epilogue=epilogue)[:m])
        if epilogue == 0:
            assert rel_err(few, product(x[:m, :k], w, s)) < 2.5e-3
    assert kernel_of(m, 1024, 4 * k, 4) == FEW_ROWS and kernel_of(320, 1024, 4 * k, 4) == STAGED
    w, s = weight(1024, 4 * k, device)
    few, many = kernels.w8a16_gemm_splitk(x[:m], w, s, 4), kernels.w8a16_gemm_splitk(x, w, s, 4)
    assert torch.equal(few.view(4, m, 1024), many.view(4, 320, 1024)[:, :m])
    w, s = weight(4096, k, device)
    norms = [(1 + 0.1 * torch.randn(128, device=device, generator=g)).to(torch.bfloat16) for _ in range(2)]
    positions = torch.randint(0, 3000, (m,), generator=g, dtype=torch.int32, device=device)
    rope = kernels.rope_table(3000, 1e6).to(device)
    slots = torch.randperm(40, generator=g, device=device)[:m].to(torch.int32)
    pools = [[torch.zeros(40, 8, 128, dtype=torch.int8, device=device) for _ in range(2)]
             + [torch.zeros(40, 8, dtype=torch.bfloat16, device=device) for _ in range(2)] for _ in range(2)]
    q_ref = kernels.qk_norm_rope_kv_write(kernels.w8a16_gemm(x[:m, :k], w, s), 16, 8, *norms, 1e-6, positions, rope,
                                          slots, *pools[0])
    q = torch.zeros(m + 1, 16, 128, dtype=torch.bfloat16, device=device)
    kernels.w8a16_qkv_norm_rope_kv(x[:m, :k], w, s, 16, 8, *norms, 1e-6, positions, rope, slots, *pools[1], q_out=q[:m])
    assert torch.equal(q[:m], q_ref) and not q[m].any()
    for a, b in zip(*pools):
        assert torch.equal(a, b)
