"""Grid rules of the row-major block GEMVs (Q4_128, Q4_K, Q4_S256, preq, packed
Q4): a row's result does not depend on how many workgroups walk the tiles.  A
call with many tiles per compute unit is compared with two calls on its halves,
which take another grid and the same lanes per row.  Tolerance: none, the same
operations in the same order."""

import pytest

pytestmark = pytest.mark.gpu

HALF = 30016


# rows of one unit per lane (tiles of 5 and 9 KB), of two (15 KB) and of three
# and four, read straight from memory (30 and 40 KB)
@pytest.mark.parametrize("kind,K", [
    ("q4_128", 256), ("q4_128", 512), ("q4k", 512), ("s256", 256), ("preq", 512), ("preq", 1536), ("preq", 2048),
    ("preq_q8", 256), ("preq_q8", 768), ("preq_q8", 1280), ("q4_128_q8", 256), ("s256_q8", 2048), ("s256", 4096),
    ("packed", 256), ("packed", 768), ("packed", 2048)])
def test_rows_do_not_depend_on_the_grid(gpu, kind, K):
    import torch
    from asdsl.kernels import _native_gemv as ng

    M = 3 * HALF if kind in ("preq", "preq_q8", "s256", "s256_q8", "packed") and K > 512 else 2 * HALF
    name, q8 = kind.removesuffix("_q8"), kind.endswith("_q8")
    unit, size, head = {"q4_128": (128, 66, 1), "q4k": (256, 144, 2), "s256": (256, 144, 8), "preq": (32, 20, 2),
                        "packed": (32, 16, 0)}[name]
    g = torch.Generator(device="cuda").manual_seed(K)
    w = torch.randint(0, 256, (M * (K // unit), size), generator=g, device="cuda", dtype=torch.uint8)
    scale = torch.rand((len(w), max(head, 1)), generator=g, device="cuda") * 0.01 + 0.001
    if head:
        w[:, :2 * head] = scale.half().view(torch.uint8)
    x = torch.randn(K, generator=g, device="cuda")
    gs = 128 if name == "q4_128" else 32
    xq, xs = torch.empty(K, dtype=torch.int8, device="cuda"), torch.empty(K // gs, device="cuda")
    ng.quantize_activation_avx2(x, xq, xs, K, gs)
    side = scale.reshape(-1) if name == "packed" else None

    def run(a, b):
        y = torch.full((b - a,), float("nan"), device="cuda")
        blocks = w[a * (K // unit):b * (K // unit)].reshape(-1)
        if q8:
            fn = {"q4_128": ng.gemv_q4_128_preq_avx2, "s256": ng.gemv_q4_s256_preq_avx2, "preq": ng.gemv_q4_32_preq_avx2}
            fn[name](blocks, xq, xs, y, b - a, K, gs)
        elif name == "packed":
            ng.gemv_q4_q8_avx2(blocks, side[a * (K // 32):b * (K // 32)], x, y, b - a, K, 32)
        elif name == "q4_128":
            ng.gemv_q4_128_fused(blocks, x, y, b - a, K, 128)
        elif name == "q4k":
            ng.gemv_q4km_q8_avx2(blocks, x, y, b - a, K)
        elif name == "s256":
            ng.gemv_q4_s256_fused(blocks, x, y, b - a, K)
        else:
            ng.gemv_q4_32_preq_fused_avx2(blocks, x, y, b - a, K, 32)
        return y

    whole = run(0, M)
    assert torch.isfinite(whole).all()
    assert torch.equal(whole, torch.cat([run(a, a + HALF) for a in range(0, M, HALF)]))
