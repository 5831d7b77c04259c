"""plm_gemm_wide: every output is one MFMA chain over K in ascending order, so it equals the packed
row-split kernel without K splits, as a one-link chain runs it (its own parity against the oracle:
tests/test_chain_gpu.py), bit for bit, at the edges of its tiles (16 to 160 rows of X by 64 to 256 of W)
and of its 64-wide K stages; and with K splits, which single linears on row-split tiles run with. Each
compiled tile and epilogue runs at least once, on shapes that pick it (TILE_SHAPES). The
activation epilogue equals torch's silu and multiply on the rounded projection up to one output step
where the two exponentials' last bits part."""

from __future__ import annotations

import pytest
import torch
import torch.nn.functional as F

from plm_amd import _lib, fast_gemm
from plm_amd.chain import Link, LinearChain
from plm_amd.fast_gemm import hip_linear, hip_linear_f32, pack_weight, release, released_linear
from plm_amd.gated_lora import gated_linear
from plm_amd.tiles import CU_COUNT, WIDE_TILES
from test_gemm_gpu import _inputs_on_gpu

pytestmark = pytest.mark.gpu

ROW_SPLIT = {"wave_frags": 2, "k_waves": 1, "split_k": 1, "unroll": 2}


def _wide(x, wp, N, kind, y):
    status = _lib.lib().plm_gemm_wide(_lib.DTYPE_CODES[x.dtype], x.data_ptr(), x.stride(0), wp.data_ptr(), y.data_ptr(),
                                      y.stride(0), x.shape[0], N, x.shape[1], kind, _lib.stream_handle(x.device))
    assert status == 0
    return y


def _chain(x, w, split=1):
    """fp32 ``x @ w^T`` on the packed row-split kernel, 128 rows of X at a time."""
    parts = []
    for m in range(0, x.shape[0], 128):
        rows = x[m:m + 128]
        parts.append(torch.empty(rows.shape[0], w.shape[0], device=x.device))
        LinearChain([Link(rows, w, parts[-1], split_k=split)], dict(ROW_SPLIT, split_k=1)).run()
    return torch.cat(parts)


# (M, N, K): below and past one tile of each height and width, a ragged N, K of one chunk, of an odd
# number of 32-wide steps and past a stage's end.
SHAPES = [(1, 1, 8), (33, 64, 64), (129, 257, 40), (160, 1003, 96), (161, 2048, 1416), (200, 11264, 72),
          (640, 2050, 1000), (500, 8192, 2048), (1281, 16384, 136)]


@pytest.mark.parametrize("M,N,K", SHAPES)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
def test_matches_the_row_split_chain_bit_for_bit(device, M, N, K, dtype):
    print(f"wide M={M} N={N} K={K} {dtype}", flush=True)
    x, w = (t.to(dtype) for t in _inputs_on_gpu(M, N, K, 3 * M + N, device))
    wp = pack_weight(w)
    ref = _chain(x, w)
    pad = torch.full((M, N + 5), float("nan"), device=device, dtype=dtype)   # rows that no 16-byte store fits
    assert torch.equal(_wide(x, wp, N, _lib.PLM_OUT_F32, torch.empty(M, N, device=device)), ref)
    assert torch.equal(_wide(x, wp, N, _lib.PLM_OUT_MODEL, torch.empty(M, N, device=device, dtype=dtype)), ref.to(dtype))
    assert torch.equal(_wide(x, wp, N, _lib.PLM_OUT_MODEL, pad[:, 1:N + 1]), ref.to(dtype))
    assert bool(pad[:, 0].isnan().all()) and bool(pad[:, N + 1:].isnan().all())


@pytest.mark.parametrize("M,N,K", [(129, 32, 8), (150, 1024, 1000), (640, 11264, 2048), (200, 2816, 512)])
def test_silu_mul_of_a_released_gate_up_weight(device, M, N, K):
    x, w = _inputs_on_gpu(M, N, K, N + K, device)
    y = _chain(x, w).to(x.dtype)
    want = F.silu(y[:, : N // 2]) * y[:, N // 2:]
    release(w)
    out = torch.empty(M, N // 2, device=device, dtype=x.dtype)
    got = fast_gemm.gate_up_silu(x, w)
    assert fast_gemm.gate_up_silu(x, w, out=out) is out and torch.equal(out, got)
    # expf of the two sides may round apart: one step of the silu (2^-8 relative) and one of the product.
    assert int((got != want).sum()) <= max(1, got.numel() // 1000)
    torch.testing.assert_close(got.float(), want.float(), rtol=2 * 2.0 ** -7, atol=1e-30)


def _picked(M, N, split=1, act=False):
    """``wide_pick`` of csrc/wide_gemm.hip: the tile of the least rounds over the CUs times bytes per K step."""
    def cost(tile):
        nf, mt = tile
        columns = 64 * nf // (2 if act else 1)
        items = -(-(N // 2 if act else N) // columns) * -(-M // (16 * mt)) * split
        return -(-items // CU_COUNT) * (4 * nf + mt)

    return min((t for t in WIDE_TILES if not (act and t[0] % 2)), key=cost)


# (M, N, split) that pick every compiled tile once, with M and N off its edges: past 128 rows and in the
# whole-weight form (plm_gemm_wide), on row-split tiles with K splits, and the gated-LoRA launch, whose
# 160-row and 256-column tiles are not compiled.
TILE_SHAPES = {
    "plain": [(m, n, 1) for m, n in ((1, 40), (17, 8296), (33, 8296), (49, 8296), (65, 8296), (97, 10944))] +
             [(m, 16571, 1) for m in (1, 17, 33, 49, 65, 81, 97, 129)] + [(65, 32790, 1)],
    "split": [(1, 40, 2)] + [(m, 1351, 6) for m in (17, 33, 49, 65)] + [(97, 1807, 6)] +
             [(m, 2719, 6) for m in (1, 17, 33, 49, 65, 81, 97)] + [(65, 5648, 6)],
    "act": [(1, 32, 1)] + [(m, 16544, 1) for m in (17, 33, 49, 65, 81, 97, 129)] + [(65, 33120, 1)],
    "act split": [(1, 32, 2)] + [(m, 5632, 3) for m in (17, 33, 49, 65, 81, 97)] + [(65, 10944, 3)],
    "lora": [(1, 40, 1)] + [(m, 2719, 3) for m in (17, 33, 49, 65)] + [(97, 3662, 3)] +
            [(m, 5648, 3) for m in (1, 17, 33, 49, 65, 81, 97)],
}


def test_the_shapes_pick_every_tile():
    for kind, shapes in TILE_SHAPES.items():
        act = kind.startswith("act")
        left_out = {"split": {(2, 10)}, "act split": {(2, 10)}, "lora": {(2, 10), (4, 8)}}.get(kind, set())
        want = {t for t in WIDE_TILES if not (act and t[0] % 2)} - left_out
        assert {_picked(*shape, act) for shape in shapes} == want, kind


@pytest.mark.parametrize("M,N,split", TILE_SHAPES["plain"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
def test_every_tile(device, M, N, split, dtype):
    test_matches_the_row_split_chain_bit_for_bit(device, M, N, 136, dtype)


@pytest.mark.parametrize("M,N,split", TILE_SHAPES["split"])
@pytest.mark.parametrize("K", [1000, 1536])   # ranges of K steps off the packed groups, and on them
def test_every_tile_with_k_splits(device, M, N, split, K):
    test_row_split_tiles_with_k_splits(device, M, N, K, split)


@pytest.mark.parametrize("M,N,split", TILE_SHAPES["act"] + TILE_SHAPES["act split"])
def test_every_tile_with_the_activation(device, M, N, split):
    x, w = _inputs_on_gpu(M, N, 1000, M + N, device)
    if M <= 128:
        test_silu_mul_on_row_split_tiles(device, M, N, 1000, split)
        y = torch.empty(M, N // 2, device=device, dtype=x.dtype)
        LinearChain([Link(x, w, y, act=True)], ROW_SPLIT).run()
    else:
        y = _chain(x, w).to(x.dtype)
        y = F.silu(y[:, : N // 2]) * y[:, N // 2:]
    if split == 1:   # the whole-weight form; past 128 rows up to a step of each rounding, as above
        got = _wide(x, pack_weight(w), N, _lib.PLM_OUT_SILU_MUL, torch.empty_like(y))
        assert int((got != y).sum()) <= (0 if M <= 128 else got.numel() // 1000)
        torch.testing.assert_close(got.float(), y.float(), rtol=2 * 2.0 ** -7, atol=1e-30)


@pytest.mark.parametrize("M,N,split", TILE_SHAPES["lora"])
def test_every_tile_with_gated_lora(device, M, N, split):
    """Two shards that meet inside a fragment, a rank past one MFMA's 32 elements."""
    test_gated_lora_on_row_split_tiles(device, M, (N // 2 | 1, N - (N // 2 | 1)), 1000, 40, M // 3, split)


# Rounds on row-split tiles: one row, a tile's edge and past it, the widest; ranges of K steps that
# start inside a group of packed steps, of odd length, and shorter than the loads in flight; a weight of
# 128 MiB, whose widest splits stay on the row-split kernel.
@pytest.mark.parametrize("M,N,K", [(1, 64, 96), (17, 1003, 1416), (56, 2048, 8192), (65, 4608, 3072), (128, 777, 1000),
                                   (30, 16384, 4096)])
@pytest.mark.parametrize("split", [1, 2, 3, 6])
def test_row_split_tiles_with_k_splits(device, M, N, K, split):
    print(f"row split M={M} N={N} K={K} split={split}", flush=True)
    x, w = _inputs_on_gpu(M, N, K, M + N + split, device)
    cfg = dict(ROW_SPLIT, split_k=split)
    ref = _chain(x, w, split)
    for _ in range(2):   # the second launch finds the first one's counters and partials
        assert torch.equal(hip_linear_f32(x, w, cfg), ref)
    assert torch.equal(hip_linear(x, w, cfg), ref.bfloat16())


@pytest.mark.parametrize("M,N,K", [(1, 32, 64), (42, 2816, 512), (110, 11264, 2048)])
@pytest.mark.parametrize("split", [1, 2])
def test_silu_mul_on_row_split_tiles(device, M, N, K, split):
    x, w = _inputs_on_gpu(M, N, K, M + K, device)
    want = torch.empty(M, N // 2, device=device, dtype=x.dtype)
    LinearChain([Link(x, w, want, split_k=split, act=True)], dict(ROW_SPLIT, split_k=1)).run()
    assert torch.equal(fast_gemm.gate_up_silu(x, w, dict(ROW_SPLIT, split_k=split)), want)


# One row, a tile's edge and past it, the widest; links that read the first columns of an earlier output, two
# that read the same one, an activation link in between, an fp32 last link and one that reads none.
@pytest.mark.parametrize("M", [1, 16, 49, 128])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
def test_row_split_chains_equal_their_links_alone(device, M, dtype):
    print(f"row split chain M={M} {dtype}", flush=True)
    g = torch.Generator(device=device).manual_seed(M)
    # (N, K, the link it reads, split, activation, fp32)
    shapes = [(1003, 264, -1, 1, False, False), (704, 1000, 0, 3, True, False), (520, 352, 1, 1, False, False),
              (136, 344, 1, 2, False, False), (777, 96, -1, 2, False, True), (2050, 520, 2, 1, False, True)]
    outs = [torch.full((M, -(-n // 64) * 64), float("nan"), device=device, dtype=torch.float32 if f32 else dtype)
            [:, :n // 2 if act else n] for n, _, _, _, act, f32 in shapes]
    x = torch.randn(M, 264, generator=g, device=device).to(dtype)
    links = []
    for (n, k, dep, split, act, _), y in zip(shapes, outs):
        w = (torch.randn(n, k, generator=g, device=device) / k ** 0.5).to(dtype)
        links.append(Link(x[:, :k] if dep < 0 else outs[dep][:, :k], w, y, dep, split, act))
    chain = LinearChain(links, ROW_SPLIT)
    for _ in range(2):
        x.copy_(torch.randn(M, 264, generator=g, device=device))
        chain.run()
        for i, ln in enumerate(links):
            alone = torch.empty_like(ln.y)
            LinearChain([Link(ln.x, ln.w, alone, split_k=ln.split_k, act=ln.act)], ROW_SPLIT).run()
            assert torch.equal(ln.y, alone), i
    chain.check()


# Shards that end inside a 16-column fragment, ranks past one MFMA's 32 elements and below them, gates at the
# first and last row, with and without K splits of the base linear (h: one range up to K = 1024, else four).
@pytest.mark.parametrize("M,shards,K,rank,gate,split", [
    (1, (24,), 64, 8, 0, 1), (56, (2048, 512, 512), 2048, 16, 7, 1), (42, (520, 136, 100), 1000, 40, 41, 2),
    (110, (1000, 1048), 3072, 72, 10, 3), (65, (7, 8, 9), 1416, 32, 3, 1)])
def test_gated_lora_on_row_split_tiles(device, M, shards, K, rank, gate, split):
    g = torch.Generator(device=device).manual_seed(M + K)
    N, cfg = sum(shards), dict(ROW_SPLIT, split_k=split)
    x, w = _inputs_on_gpu(M, N, K, M + N, device)
    a = (torch.randn(len(shards) * rank, K, generator=g, device=device) / K ** 0.5).bfloat16()
    bs = [torch.randn(n, rank, generator=g, device=device).bfloat16() for n in shards]
    got = [gated_linear(x, w, a, bs, gate, cfg=cfg) for _ in range(3)]
    assert torch.equal(got[0], got[1]) and torch.equal(got[0], got[2])
    base = hip_linear(x, w, cfg)
    assert torch.equal(got[0][:gate], base[:gate])
    h = x[gate:].double() @ a.double().t()
    delta = torch.cat([h[:, i * rank:(i + 1) * rank] @ b.double().t() for i, b in enumerate(bs)], dim=1)
    want = x[gate:].double() @ w.double().t() + delta
    # Roundings to bf16: the base (2^-9 of it), h (2^-9 of each of its products with B), the sum.
    hb = torch.cat([h[:, i * rank:(i + 1) * rank].abs() @ b.double().abs().t() for i, b in enumerate(bs)], dim=1)
    bound = 2.0 ** -8 * ((want - delta).abs() + hb + want.abs()) + 1e-4
    assert bool(((got[0][gate:].double() - want).abs() <= bound).all())


@pytest.mark.parametrize("M,shards,K,rank,split", [
    (7, (24, 30, 42), 64, 8, 1), (56, (520, 136, 100), 1000, 40, 2), (110, (5640, 5624), 256, 72, 1)])
@pytest.mark.parametrize("over", [0, 1])
def test_gated_lora_overflow_stays_in_its_shard(device, M, shards, K, rank, split, over):
    """One shard's h past fp16's largest value: the other shards' columns, those of the fragments it shares
    with them included, equal the run without the overflow."""
    g = torch.Generator(device=device).manual_seed(M)
    cfg = dict(ROW_SPLIT, split_k=split)
    x = torch.rand(M, K, generator=g, device=device).half()
    w = (torch.randn(sum(shards), K, generator=g, device=device) / K ** 0.5).half()
    a = (torch.randn(len(shards) * rank, K, generator=g, device=device) / K ** 0.5).half()
    bs = [torch.randn(n, rank, generator=g, device=device).half() for n in shards]
    want = gated_linear(x, w, a, bs, 3, cfg=cfg)
    a[over * rank:(over + 1) * rank] = 60000.0
    got = gated_linear(x, w, a, bs, 3, cfg=cfg)
    lo = sum(shards[:over])
    hi = lo + shards[over]
    assert torch.equal(got[:, :lo], want[:, :lo]) and torch.equal(got[:, hi:], want[:, hi:])
    assert torch.equal(got[:3], want[:3]) and not bool(got[3:, lo:hi].isfinite().any())


def test_calls_that_need_more_than_a_product_go_to_f_linear(device):
    """A bias, autograd, autocast and vmap of a released weight's wide calls act as F.linear's own."""
    x, w = _inputs_on_gpu(130, 256, 64, 9, device)
    ref_w = w.clone()
    release(w)
    bias = torch.randn(256, device=device).bfloat16()
    assert torch.equal(released_linear(x, w, bias), F.linear(x, ref_w, bias))
    leaf = x.clone().requires_grad_()
    released_linear(leaf, w).sum().backward()
    want = x.clone().requires_grad_()
    F.linear(want, ref_w).sum().backward()
    assert torch.equal(leaf.grad, want.grad)
    with torch.autocast("cuda", dtype=torch.float16):
        assert released_linear(x, w).dtype == torch.float16
    stack = torch.stack([x, -x])
    assert torch.func.vmap(lambda t: released_linear(t, w))(stack).shape == (2, 130, 256)
    with torch.no_grad():
        assert torch.equal(released_linear(leaf, w), F.linear(x, ref_w))


def test_rows_off_16_bytes_go_to_f_linear(device):
    """A contiguous X that starts off a 16-byte boundary, which no 16-byte load reads."""
    _, w = _inputs_on_gpu(130, 256, 64, 11, device)
    ref_w = w.clone()
    release(w)
    x = torch.randn(130 * 64 + 8, device=device).bfloat16()[1:130 * 64 + 1].view(130, 64)
    assert x.is_contiguous() and x.data_ptr() % 16
    y = F.linear(x, ref_w)
    assert torch.equal(released_linear(x, w), y)
    assert torch.equal(fast_gemm.gate_up_silu(x, w), F.silu(y[:, :128]) * y[:, 128:])


@pytest.mark.parametrize("M,N,K", [(2049, 64, 64), (1600, 8192, 64), (130, 64, 7176)])
def test_calls_the_library_is_faster_at(device, M, N, K):
    """Past the wide kernel's range the released calls are F.linear's, with the activation torch's."""
    x, w = _inputs_on_gpu(M, N, K, M + K, device)
    y = F.linear(x, w)
    release(w)
    assert torch.equal(released_linear(x, w), y)
    got, want = fast_gemm.gate_up_silu(x, w), F.silu(y[:, :N // 2]) * y[:, N // 2:]
    if M == 1600:   # the activation's own line is 2048 rows: the wide kernel, one step of each rounding
        torch.testing.assert_close(got.float(), want.float(), rtol=2 * 2.0 ** -7, atol=1e-30)
    else:
        assert torch.equal(got, want)
