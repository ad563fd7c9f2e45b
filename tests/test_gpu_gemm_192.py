"""The 16-bit tiles of 256 x 192 and 192 x 64: edges in both directions, layouts, contractions that end inside a k tile, split
contractions, and the row sums that ride along with a weight gradient of theirs."""
import pytest

from dfdx_amd.rocm import KERNEL_AUTO, KERNEL_MFMA
from gpu_util import device
from test_gpu_gemm import run_case
from test_gpu_gemm_ring import test_bias_gradient_rides_along as bias_gradient_rides_along
from test_gpu_gemm_tail import tiles

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("tile", ["_dma_256x192x64", "_ring_192x64x64"])
@pytest.mark.parametrize("layout", ["nt", "nn", "tn", "tt"])
@pytest.mark.parametrize("m,k,n,splits", [(256, 64, 192, 1), (192, 192, 64, 1), (200, 128, 392, 1), (264, 320, 184, 2), (8, 256, 8, 1), (776, 192, 200, 3)])
def test_edges_of_tiles(dtype, tile, layout, m, k, n, splits):
    (variant,) = tiles(device(), dtype, tile)
    for accumulate in (False, True):
        assert tile in run_case(dtype, m, k, n, layout, accumulate, KERNEL_MFMA, variant, bias=not accumulate and splits == 1, split_k=splits, seed=m + n)


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("layout,m,k,n", [("nt", 200, 72, 136), ("nn", 384, 456, 72), ("tn", 136, 65, 200), ("nt", 193, 72, 67)])
def test_any_contraction(dtype, layout, m, k, n):
    (variant,) = tiles(device(), dtype, "_ring_192x64x64")
    run_case(dtype, m, k, n, layout, True, KERNEL_MFMA, variant, seed=k)


@pytest.mark.parametrize("accumulate", [False, True])
@pytest.mark.parametrize("layout,m,k,n,splits", [
    ("nt", 6144, 64, 4224, 1), ("nn", 6100, 192, 4224, 1), ("nn", 6144, 64, 4232, 1), ("tn", 6144, 192, 4168, 1),   # (the last two off the 128-byte lines)
    ("tn", 3584, 192, 2688, 3), ("nt", 3600, 512, 2624, 4),
])
def test_several_items_a_workgroup(layout, m, k, n, splits, accumulate):
    """More than two rounds of items, of one k tile and more each: a tile's stores leave under the next one's loads."""
    (variant,) = tiles(device(), "f16", "_dma_256x192x64")
    assert -(-m // 256) * -(-n // 192) * splits > 512
    assert "_dma_256x192x64" in run_case("f16", m, k, n, layout, accumulate, KERNEL_MFMA, variant, split_k=splits, seed=m + n)


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("layout,m,k,n,want", [
    ("nt", 3152, 768, 3072, "_dma_256x192"), ("tn", 2168, 1472, 4840, "_dma_256x192"), ("nt", 3152, 3072, 768, "_ring_192x64"),
    ("nn", 4096, 512, 4103, "_realigned"), ("nt", 7640, 64, 9536, "_dma_256x256"),   # (half lines: not behind one k tile)
])
def test_where_they_are_taken(dtype, layout, m, k, n, want):
    assert want in run_case(dtype, m, k, n, layout, False, KERNEL_AUTO, 0, bias=True, seed=m)


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("rows,i,o", [(1792, 2496, 1080), (4608, 1152, 5056)])
def test_row_sums(dtype, rows, i, o):
    bias_gradient_rides_along(dtype, rows, i, o)


@pytest.mark.parametrize("dtype,layout,m,k,n,accumulate,never", [
    ("bf16", "nn", 3778, 7038, 256, False, "_128x128x64_w2x2"), ("f16", "tn", 896, 7076, 512, False, "_128x128x64_w2x2"),
    ("f16", "nt", 2304, 576, 8188, True, "_256x256x64_w2x4"), ("f16", "tn", 1216, 2165, 1664, False, "_192x64x64"),
    ("f16", "nt", 1998, 4096, 1024, False, "_ring_128x64x64"),   # (slower in a chain of launches)
])
def test_where_another_tile_is_left(dtype, layout, m, k, n, accumulate, never):
    """Products that were faster on the tile before: by up to 2.4 times than in pieces on the large register-staged tiles."""
    name = run_case(dtype, m, k, n, layout, accumulate, KERNEL_AUTO, 0, seed=m)
    assert never not in name or "_dma_" in name, name
