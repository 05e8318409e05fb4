"""How engines of unequal dofs are laid out (no GPU needed): both dofs padded to
the larger one only where that was measured faster than computing them as they are;
equal dofs and few columns as before."""
import pytest

import shaw_amd
from tests.test_gpu_rom_split import SIZES

# kv, ks, columns, padded modes (0: the dofs keep their own sizes)
FP64 = [(100, 64, 2048, 128), (100, 64, 2064, 0), (64, 100, 4096, 0), (128, 128, 4096, 128),
        (190, 60, 1024, 192), (190, 60, 1040, 0), (150, 128, 2048, 192), (150, 128, 2064, 0), (192, 192, 4096, 192),
        (256, 64, 257, 0), (64, 256, 1024, 0), (256, 128, 1024, 256), (256, 128, 1025, 0), (256, 192, 2048, 0),
        (256, 256, 4096, 256),
        (384, 64, 321, 0), (64, 300, 1024, 0), (320, 192, 1024, 384), (320, 192, 1040, 0), (320, 320, 1040, 0),
        (384, 320, 1040, 0), (384, 384, 2048, 384), (384, 384, 2064, 0),
        (512, 64, 257, 0), (448, 1, 1024, 0), (448, 128, 1024, 512), (512, 512, 1024, 512), (512, 512, 1040, 0),
        # few columns are shared among workgroups, whatever the smaller dof
        (256, 64, 256, 256), (64, 384, 320, 384), (512, 64, 256, 512)]


@pytest.mark.parametrize("kv,ks,cols,modes", FP64)
def test_fp64_pads(kv, ks, cols, modes):
    got, split, sets = shaw_amd.debug_rom_shape(shaw_amd.ROM_FP64, kv, ks, cols)
    assert got == modes
    assert (split > 1) == (modes >= 256 and cols <= {256: 256, 384: 320, 512: 256}[modes])
    assert shaw_amd.debug_rom_shape(shaw_amd.ROM_FP64, ks, kv, cols) == (got, split, sets)


def test_no_cooperative_launches_no_sharing():
    for precision in (shaw_amd.ROM_FP64, shaw_amd.ROM_BF16X3, shaw_amd.ROM_BF16X4):
        assert shaw_amd.debug_rom_shape(precision, 512, 512, 16, cus=0)[1] == 1


@pytest.mark.parametrize("kv,ks,cols,modes", [(512, 128, 896, 512), (512, 128, 897, 0), (64, 400, 1024, 0),
                                              (512, 129, 1024, 512), (512, 512, 4096, 512), (384, 64, 1280, 384)])
def test_bf16x3_pads(kv, ks, cols, modes):
    got, split, sets = shaw_amd.debug_rom_shape(shaw_amd.ROM_BF16X3, kv, ks, cols)
    assert got == modes
    assert (split > 1) == (0 < modes and cols <= {384: 1280, 512: 1024}[modes])


@pytest.mark.parametrize("precision", [shaw_amd.ROM_BF16X3, shaw_amd.ROM_BF16X4])
@pytest.mark.parametrize("kv,ks,m", SIZES)
def test_few_bf16_columns_are_shared(kv, ks, m, precision):
    """What the GPU tests of shared tiles compare is shared on one side only."""
    modes, split, _ = shaw_amd.debug_rom_shape(precision, kv, ks, m)
    most = modes // 64
    assert modes == (384 if max(kv, ks) <= 384 else 512)
    assert split == (most if (m + 15) // 16 <= {384: 40, 512: 32}[modes] else most // 2)
    assert shaw_amd.debug_rom_shape(precision, kv, ks, 2048)[1] == 1
