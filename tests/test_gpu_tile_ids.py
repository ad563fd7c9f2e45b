"""A tile that a caller asks for by its id stays the same tile: new ones go behind, in front of the small-product kernel."""
import pytest

from dfdx_amd.rocm import KERNEL_MFMA
from gpu_util import device

pytestmark = pytest.mark.gpu

F32 = ("256x256x32_w2x4", "256x256x32_w2x2", "256x128x32_w2x2", "128x128x32_w2x2", "128x64x32_w4x1", "64x64x32_w2x2", "dma_256x256x32_w2x4",
       "dma_128x128x32_w2x2")
HALF = ("256x256x64_w2x4", "256x256x64_w2x2", "256x128x64_w2x2", "128x128x64_w2x2", "128x64x64_w4x1", "64x64x64_w2x2", "256x256x32_w2x4", "256x128x32_w2x2",
        "128x128x32_w2x2", "128x256x32_w2x2", "dma_256x256x64_w2x4", "dma_256x128x64_w4x2", "dma_128x128x64_w2x4", "dma_256x64x64_w4x2", "dma_128x64x64_w2x4",
        "ring_64x64x64_w2x2_s4", "ring_64x64x64_w2x2_s3", "ring_128x64x64_w2x2_s3", "ring_128x128x64_w2x4_s4")


def name(dtype, variant):
    dev = device()
    return dev.gemm_plan(dev.gemm_desc(dtype, 512, 512, 512, 256, (512, 1), 512, (512, 1), 1024, (512, 1), kernel=KERNEL_MFMA, variant=variant, no_split_k=True))[2]


@pytest.mark.parametrize("dtype,tiles", [("f32", F32), ("f16", HALF), ("bf16", HALF)])
def test_ids(dtype, tiles):
    for variant, tile in enumerate(tiles, 1):
        assert name(dtype, variant).endswith("_" + tile), (variant, name(dtype, variant))
    assert name(dtype, device().mfma_variant_count(dtype)).endswith("_small_16x16_ksliced")
