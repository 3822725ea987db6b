"""Window lists on a compressed y axis (lists.hip) against the kernels that scan the access arrays."""
import numpy as np
import pytest
import torch

import apr_cases
from pyapr import APR, _native
from pyapr.aprnet import _ops, utils

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def blocks(shape, seed, share):
    """Fine only in a few short runs along y, anywhere in a volume that is coarse elsewhere: most positions are not kept."""
    rng = np.random.default_rng(seed)
    field = np.zeros(tuple((s + 1) // 2 for s in shape), np.uint8)
    lmax = int(np.ceil(np.log2(max(max(shape), 2))))
    mask = rng.random(field.shape) < share
    field[mask] = rng.integers(max(lmax - 2, 1), lmax + 1, size=int(mask.sum()), dtype=np.uint8)
    return APR.from_level_field(shape, field)


# rows that end within, at and behind a 64-bit word of the bit maps; odd lengths, whose last position has no partner; single rows and
# positions; runs of several row groups in one window and several windows of one group; rows too long for a bit map each (16.6 k positions)
CASES = [((20, 21, 63), 0.02), ((20, 21, 64), 0.02), ((9, 18, 65), 0.05), ((33, 30, 127), 0.004), ((10, 12, 257), 0.3), ((5, 7, 1), 0.5), ((3, 1, 2), 1.0),
         ((40, 44, 300), 0.0005), ((1, 40, 130), 0.02), ((1, 3, 17001), 0.002), ((1, 1, 129), 0.1), ((2, 2, 9000), 0.002)]


@pytest.mark.parametrize("shape,share", CASES, ids=["x".join(map(str, s)) for s, _ in CASES])
@pytest.mark.parametrize("ksize", [(3, 3, 3), (1, 3, 3), (1, 5, 5)], ids=["333", "133", "155"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
def test_lists_give_what_a_scan_gives(shape, share, ksize, dtype):
    """Forward and both gradients of small whole numbers.  Level deltas, 1, 4 and 16 input channels (the pipelined kernel of first layers,
    groups of four channels, products of pieces)."""
    apr = blocks(shape, 11, share)
    gen = torch.Generator().manual_seed(3)
    lib = _native.hip()
    for delta in (0, 1):
        if delta > apr.level_max() - apr.level_min() or utils.number_particles(apr, delta) == 0:
            continue
        n, ld = utils.number_particles(apr, delta), torch.tensor([delta], dtype=torch.int32)
        for cin in (1, 4, 16):
            x = torch.randint(-3, 4, (1, cin, n), generator=gen).to(dtype).to(DEV)
            gy = torch.randint(-3, 4, (1, 18, n), generator=gen).to(dtype).to(DEV)
            w = torch.randint(-2, 3, (apr.level_max() - apr.level_min() + 1, 18, cin) + ksize, generator=gen).float().to(DEV)
            run = lambda: (_ops.conv_forward([apr], x, w, ld), *_ops.conv_backward([apr], x, w, gy, ld))
            for p in (20, 23):
                assert lib.aprnet_set_conv_path(p) == 0
            try:
                got = run()
                assert lib.aprnet_set_conv_path(5) == 0
                ref = run()
            finally:
                for p in (4, 18, 21):
                    lib.aprnet_set_conv_path(p)
            for k, (g, r) in enumerate(zip(got, ref)):
                # means down the tree carry fractions of 8^-depth, so that sums round in their last bits; bfloat16 results by one step of 2^-8
                scale = float(r.float().abs().max())
                assert float((g.float() - r.float()).abs().max()) <= (1e-5 if dtype == torch.float32 or k == 2 else 1e-2) * scale, (k, delta, cin)


def test_outputs_do_not_depend_on_their_window():
    """A sparse volume, whose windows hold pieces of many row groups: the fp32 instructions give the bits of the scanning kernel."""
    apr = blocks((64, 64, 500), 5, 0.0005)
    n, ld = apr.total_number_particles(), torch.zeros(1, dtype=torch.int32)
    x = torch.randn(1, 16, n, generator=torch.Generator().manual_seed(1)).to(DEV)
    w = torch.randn(apr.level_max() - apr.level_min() + 1, 16, 16, 3, 3, 3, generator=torch.Generator().manual_seed(2)).to(DEV)
    lib = _native.hip()
    lib.aprnet_set_conv_path(19)
    try:
        got = _ops.conv_forward([apr], x, w, ld)
        lib.aprnet_set_conv_path(5)
        ref = _ops.conv_forward([apr], x, w, ld)
    finally:
        for p in (4, 18):
            lib.aprnet_set_conv_path(p)
    assert torch.equal(got, ref)                   # same products in the same order, whatever window an output lies in
