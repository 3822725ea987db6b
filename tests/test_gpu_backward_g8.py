"""The backward pass of the stencil convolutions on copies grouped by eight channels (bfloat16 features): sizes at the
edges of the kernels' blocks (16 input / 16 or 32 output channels, 32 columns per product, 256 columns per staged group)."""
import ctypes as C

import pytest
import torch

import apr_cases
from oracle import oracle
from pyapr import _native
from pyapr.aprnet import _ops, utils
from pyapr.synthetic import make_config
from test_gpu_parity import _conv_case

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

# full windows of a uniformly fine image (more than one staged group of columns), sparse 3-D and 2-D ones, level deltas
CASES = [([("3d_dense", 0)], (3, 3, 3)), ([("3d_t", 0), ("3d_a", 1)], (3, 3, 3)), ([("2d_t", 0), ("2d_s", 1)], (1, 5, 5)),
         ([("2d_t", 0)], (1, 3, 3)), ([("3d_s", 1)], (1, 3, 3))]


@pytest.fixture(autouse=True)
def dense_case(monkeypatch):
    get = apr_cases.get
    monkeypatch.setattr(apr_cases, "get", lambda n: apr_cases.random_apr((12, 13, 150), 21, 0.6, 1) if n == "3d_dense" else get(n))


@pytest.mark.parametrize("cin,cout", [(1, 16), (8, 17), (16, 16), (24, 48), (40, 33)])
@pytest.mark.parametrize("bt,ksize", CASES, ids=["333-dense", "333", "155-2d", "133-2d", "133-3d"])
def test_weight_gradient_blocks(bt, ksize, cin, cout):
    """Against the oracle on the same bfloat16-representable values (the tree means it reads are rounded to bfloat16 on the
    GPU: 2^-9 per value, 1e-2 of the largest element as in the other bfloat16 tests), against the kernel on channel planes,
    which multiplies the same bfloat16 values exactly (fp32 sums in another order: 1e-5), and bit for bit on a second run."""
    x, aprs, ld, w_exp = _conv_case(bt, ksize, 2, cin, cout, torch.float32)
    xb = x.to(torch.bfloat16)
    gob = torch.randn(x.size(0), cout, x.size(2), generator=torch.Generator().manual_seed(5)).to(torch.bfloat16)
    _, gw_ref = oracle.conv_backward(aprs, xb.float(), w_exp, gob.float(), ld)
    wd = w_exp.permute(1, 2, 0, 3, 4, 5).contiguous().to(DEV)
    xd, gd = xb.to(DEV), gob.to(DEV)
    gw = _ops.conv_backward(aprs, xd, wd, gd, ld)[1]
    again = _ops.conv_backward(aprs, xd, wd, gd, ld)[1]
    lib = _native.hip()
    assert lib.aprnet_set_conv_path(9) == 0
    try:
        planes = _ops.conv_backward(aprs, xd, wd, gd, ld)[1]
    finally:
        lib.aprnet_set_conv_path(8)
    assert torch.equal(gw, again)
    scale = float(planes.abs().max())
    assert float((gw - planes).abs().max()) <= 1e-5 * scale
    assert float((gw.permute(2, 0, 1, 3, 4, 5).cpu() - gw_ref).abs().max()) <= 1e-2 * float(gw_ref.abs().max())


@pytest.mark.parametrize("shape", [(1, 1, 2), (1, 1, 3), (1, 2, 3), (2, 3, 3), (1, 1, 1030), (3, 5, 137)])
def test_grouped_copy_of_any_length(shape):
    """The grouped copy the kernels stage from: fewer particles than one thread takes (four), remainders of four and of a
    block's 1024.  Same products in the same order as the kernel that gathers from the planes: bit-identical."""
    apr = apr_cases.random_apr(shape, 3, 0.5, 1)
    n = apr.total_number_particles()
    x = torch.randn(1, 9, n, generator=torch.Generator().manual_seed(n)).to(torch.bfloat16).to(DEV)
    w = torch.randn(apr.level_max() - apr.level_min() + 1, 5, 9, 1, 3, 3, generator=torch.Generator().manual_seed(1)).to(DEV)
    ld = torch.zeros(1, dtype=torch.int32)
    y = _ops.conv_forward([apr], x, w, ld)
    lib = _native.hip()
    assert lib.aprnet_set_conv_path(9) == 0
    try:
        planes = _ops.conv_forward([apr], x, w, ld)
    finally:
        lib.aprnet_set_conv_path(8)
    assert torch.equal(y, planes)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("shape,drop,ksize,deltas", [((70, 90, 110), 4, (3, 3, 3), (0, 2)), ((1, 500, 611), 6, (1, 5, 5), (0, 1)),
                                                     ((9, 12, 1), 2, (1, 3, 3), (0,))])
def test_tree_gradient_of_the_nodes_with_outputs(shape, drop, ksize, deltas, dtype):
    """Handing the tree's gradient down from the nodes the forward lists name against handing it down from every node
    (levels walked in one launch, level by level from a list, whole), and the stored lists (plain stores where one column
    writes a place) against the kernel that scans and adds every column atomically.  Small whole numbers, so that the sums
    of the convolution do not depend on their order, hence bit-identical."""
    apr = apr_cases.random_apr(shape, 5, 0.01 if drop > 2 else 0.1, drop)
    gen = torch.Generator().manual_seed(3)
    lib = _native.hip()
    for delta in deltas:
        n = utils.number_particles(apr, delta)
        ld = torch.tensor([delta], dtype=torch.int32)
        x = torch.randint(-3, 4, (1, 5, n), generator=gen).to(dtype).to(DEV)
        gy = torch.randint(-3, 4, (1, 18, n), generator=gen).to(dtype).to(DEV)
        w = torch.randint(-2, 3, (apr.level_max() - apr.level_min() + 1, 18, 5) + ksize, generator=gen).float().to(DEV)
        got = _ops.conv_backward([apr], x, w, gy, ld)
        for off, on in ((17, 16), (5, 4)):
            assert lib.aprnet_set_conv_path(off) == 0
            try:
                ref = _ops.conv_backward([apr], x, w, gy, ld)
            finally:
                lib.aprnet_set_conv_path(on)
            assert float(ref[0].float().abs().max()) > 0
            assert torch.equal(got[0], ref[0])
            assert float((got[1] - ref[1]).abs().max()) <= 1e-5 * float(ref[1].abs().max())


@pytest.mark.parametrize("cin", [4, 8, 20, 36])
@pytest.mark.parametrize("shape,drop,ksize,deltas", [((70, 90, 110), 4, (3, 3, 3), (0, 2)), ((1, 500, 611), 6, (1, 5, 5), (0, 1)), ((31, 33, 35), 3, (1, 3, 3), (0, 1)),
                                                     ((9, 12, 1), 2, (1, 3, 3), (0,)), ((128, 128, 130), 6, (3, 3, 3), (0,))])
def test_input_gradient_in_groups_of_four_channels(monkeypatch, shape, drop, ksize, deltas, cin):
    """Work spaces in groups of four channels (whole groups only), cleared where something is added and finished by one pass, against
    the kernels that scan, on planes that are cleared whole; work spaces hold NaN before the call.  Small whole numbers, as above:
    bit-identical.  One to several groups per thread, levels of the tree walked in one launch, from a list and whole."""
    apr = apr_cases.random_apr(shape, 5, 0.01 if drop > 2 else 0.1, drop)
    gen = torch.Generator().manual_seed(3)
    lib, empty = _native.hip(), torch.empty
    monkeypatch.setattr(torch, "empty", lambda *a, **k: (lambda t: t.fill_(float("nan")) if t.is_floating_point() else t)(empty(*a, **k)))
    for delta in deltas:
        n = utils.number_particles(apr, delta)
        ld = torch.tensor([delta], dtype=torch.int32)
        x = torch.randint(-3, 4, (1, cin, n), generator=gen).to(torch.bfloat16).to(DEV)
        gy = torch.randint(-3, 4, (1, 18, n), generator=gen).to(torch.bfloat16).to(DEV)
        w = torch.randint(-2, 3, (apr.level_max() - apr.level_min() + 1, 18, cin) + ksize, generator=gen).float().to(DEV)
        got = _ops.conv_backward([apr], x, w, gy, ld)[0]
        for off, on in ((17, 16), (5, 4)):
            assert lib.aprnet_set_conv_path(off) == 0
            try:
                ref = _ops.conv_backward([apr], x, w, gy, ld)[0]
            finally:
                lib.aprnet_set_conv_path(on)
            assert float(ref.float().abs().max()) > 0
            assert torch.equal(got, ref)


def test_weight_gradient_without_room_for_the_copies():
    """A capture must not grow the plan's scratch buffer: when the copies do not fit what is there, the kernel on channel planes
    runs as it did for the eager call that sized the buffer (same kernel, same order of summation: bit-identical)."""
    apr = apr_cases.random_apr((70, 90, 110), 5, 0.01, 4)
    gen = torch.Generator().manual_seed(7)
    n, ld = apr.total_number_particles(), torch.zeros(1, dtype=torch.int32)
    x = torch.randn(1, 5, n, generator=gen).to(torch.bfloat16).to(DEV)
    gy = torch.randn(1, 18, n, generator=gen).to(torch.bfloat16).to(DEV)
    w = torch.randn(apr.level_max() - apr.level_min() + 1, 18, 5, 3, 3, 3, generator=gen).to(DEV)
    lib = _native.hip()
    assert lib.aprnet_set_conv_path(9) == 0
    try:
        planes = _ops.conv_backward([apr], x, w, gy, ld, need_input_grad=False)[1]
    finally:
        lib.aprnet_set_conv_path(8)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        captured = _ops.conv_backward([apr], x, w, gy, ld, need_input_grad=False)[1]
    for _ in range(3):
        captured.fill_(-1)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(captured, planes)


@pytest.mark.parametrize("cin,cout", [(5, 18), (32, 32)])
def test_grouped_weight_gradient_next_to_an_input_gradient_without_lists(cin, cout):
    """Forward lists there, input-gradient lists not: the weight gradient reads its grouped copies on the side stream while the
    input gradient packs fp32 weights, twice the size of the bfloat16 image, at the front of the same scratch buffer.  Reached
    by a capture: the 1x3x3 backward has built the row groups that 1x5x5 shares, the 1x5x5 lists of the input gradient would
    have to be built.  Weight gradient: same kernel, lists and order as the eager call without an input gradient, hence
    bit-identical.  Input gradient: fp32 products in place of bfloat16 ones on weights rounded to bfloat16 (2^-9 each)."""
    apr = apr_cases.random_apr((1, 300, 411), 5, 0.02, 5)
    gen = torch.Generator().manual_seed(11)
    n, ld = apr.total_number_particles(), torch.zeros(1, dtype=torch.int32)
    levels = apr.level_max() - apr.level_min() + 1
    x = torch.randn(1, cin, n, generator=gen).to(torch.bfloat16).to(DEV)
    gy = torch.randn(1, cout, n, generator=gen).to(torch.bfloat16).to(DEV)
    w3 = torch.randn(levels, cout, cin, 1, 3, 3, generator=gen).to(DEV)
    w5 = torch.randn(levels, cout, cin, 1, 5, 5, generator=gen).to(DEV)
    lib = _native.hip()
    assert lib.aprnet_plan_reserve(apr.plan(0), 256 << 20, None) == 0
    _ops.conv_backward([apr], x, w3, gy, ld)
    gw = _ops.conv_backward([apr], x, w5, gy, ld, need_input_grad=False)[1]
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        captured = _ops.conv_backward([apr], x, w5, gy, ld)
    eager = _ops.conv_backward([apr], x, w5, gy, ld)
    assert torch.equal(eager[1], gw)
    for _ in range(5):
        for t in captured:
            t.fill_(-1)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(captured[1], gw)
        assert float((captured[0].float() - eager[0].float()).abs().max()) <= 1e-2 * float(eager[0].float().abs().max())


def _memory_outside_torch():
    torch.cuda.synchronize()
    free, total = torch.cuda.mem_get_info()
    return total - free - torch.cuda.memory_reserved()


def test_partial_sums_of_a_wide_layer_stay_within_512_mib():
    """3x3x3 512 -> 512: a slot of the partial sums holds 28 MB, and one per workgroup of a narrow layer's grid would be
    2.2 GB.  What the call keeps besides them: the copies of 2 x 512 channels and the plan's lists."""
    apr = apr_cases.random_apr((40, 36, 44), 9, 0.02)
    apr.init_cuda()
    gen = torch.Generator().manual_seed(2)
    n, ld = apr.total_number_particles(), torch.zeros(1, dtype=torch.int32)
    x = torch.randn(1, 512, n, generator=gen).to(torch.bfloat16).to(DEV)
    gy = torch.randn(1, 512, n, generator=gen).to(torch.bfloat16).to(DEV)
    w = torch.randn(2, 512, 512, 3, 3, 3, device=DEV)
    before = _memory_outside_torch()
    gw = _ops.conv_backward([apr], x, w, gy, ld, need_input_grad=False)[1]
    grown = _memory_outside_torch() - before
    copies = 2 * 512 * (2 * n + apr.total_number_tree_particles())
    assert grown <= (512 << 20) + copies + (32 << 20)
    lib = _native.hip()
    assert lib.aprnet_set_conv_path(9) == 0
    try:
        planes = _ops.conv_backward([apr], x, w, gy, ld, need_input_grad=False)[1]
    finally:
        lib.aprnet_set_conv_path(8)
    assert float((gw - planes).abs().max()) <= 1e-5 * float(planes.abs().max())


@pytest.mark.parametrize("cin,cout", [(40, 33), (80, 32)])
def test_copies_of_a_large_layer_are_made_in_parts(cin, cout):
    """Features and tree of 7 M particles are copied 16, 16 and 8 channels at a time (40 -> 33), 48 and 32 (80 -> 32, where the
    smaller part has more slots of partial sums in all), so that the scratch buffer holds the copies of the output gradient
    and of one part (at most 256 MiB more than the forward pass needs).  Against the kernel on channel planes (the same
    products; fp32 sums of 7 M terms in another order) and a second run."""
    apr, _ = make_config("blobs512", scale=0.68)
    gen = torch.Generator(device=DEV).manual_seed(3)
    n, nt, ld = apr.total_number_particles(), _ops.tree_parts(apr, 0), torch.zeros(1, dtype=torch.int32)
    x = torch.randn(1, cin, n, device=DEV, generator=gen).to(torch.bfloat16)
    gy = torch.randn(1, cout, n, device=DEV, generator=gen).to(torch.bfloat16)
    w = torch.randn(2, cout, cin, 3, 3, 3, device=DEV, generator=gen)
    _ops.conv_backward([apr], x[:, :1].contiguous(), w[:, :1, :1].contiguous(), gy[:, :1].contiguous(), ld)      # the plan's lists
    torch.cuda.empty_cache()
    before = _memory_outside_torch()
    gw = _ops.conv_backward([apr], x, w, gy, ld)[1]
    grown = _memory_outside_torch() - before
    gi, go = (cin + 7) // 8, (cout + 7) // 8
    assert 16 * go * n <= grown <= 16 * max(gi * (n + nt), go * n) + (256 << 20) + (128 << 20)    # ... and the sums' slots
    assert torch.equal(gw, _ops.conv_backward([apr], x, w, gy, ld)[1])
    lib = _native.hip()
    assert lib.aprnet_set_conv_path(9) == 0
    try:
        planes = _ops.conv_backward([apr], x, w, gy, ld, need_input_grad=False)[1]
    finally:
        lib.aprnet_set_conv_path(8)
    assert float((gw - planes).abs().max()) <= 1e-4 * float(planes.abs().max())


@pytest.mark.parametrize("fill", [16, 17], ids=["needed-nodes", "whole-tree"])
@pytest.mark.parametrize("d", [0, 1, 2])
@pytest.mark.parametrize("ksize,c1,c2", [((3, 3, 3), 8, 0), ((1, 3, 3), 12, 12), ((1, 5, 5), 40, 0), ((3, 3, 3), 16, 24)])
def test_tree_made_of_the_regrouped_features(ksize, c1, c2, d, fill):
    """A 16-byte aligned tree work space takes the tree in groups of eight channels, made of the regrouped features; any other one the planes'
    tree, regrouped.  Same bits in the output and in the weight gradient, also where the rows of the work space are longer than the tree, and
    at the level deltas at which downsampled particles come first in a node's sum."""
    lib, st, cin, cout = _native.hip(), torch.cuda.current_stream().cuda_stream, c1 + c2, 16
    apr = apr_cases.get("3d_t" if ksize[0] == 3 else "2d_t")
    n, nt = _ops.number_particles(apr, d), _ops.tree_parts(apr, d)
    g = torch.Generator().manual_seed(cin)
    x = torch.randn(cin, n, generator=g).to(torch.bfloat16).to(DEV)
    gy = torch.randn(cout, n, generator=g).to(torch.bfloat16).to(DEV)
    S = apr.level_max() - apr.level_min() + 1
    w = (torch.randn(S, cout, cin, *ksize, generator=g) * 0.1).to(DEV)
    results = []
    try:
        assert lib.aprnet_set_conv_path(fill) == 0
        for shift in (0, 1):                                       # elements, 2 bytes each
            ldt = nt + 3
            tree = torch.full((cin * ldt + 8,), float("nan"), dtype=torch.bfloat16, device=DEV)[shift:]
            assert (tree.data_ptr() % 16 == 0) == (shift == 0)
            y, gx = torch.zeros(cout, n, dtype=torch.bfloat16, device=DEV), torch.zeros_like(x)
            gw = torch.zeros_like(w)
            gx32, gt = torch.zeros(cin, n, device=DEV), torch.zeros(cin, nt, device=DEV)
            fu = _ops._Fusion(x[c1:].data_ptr() if c2 else None, n, c2, 0)
            assert lib.aprnet_conv_fwd_fused_bf16(apr.plan(0), d, *ksize, x.data_ptr(), n, c1, w.data_ptr(), S, cout, None, y.data_ptr(), n,
                                                  tree.data_ptr(), ldt, C.byref(fu), st) == 0, lib.aprnet_last_error()
            assert lib.aprnet_conv_bwd_bf16(apr.plan(0), d, *ksize, x.data_ptr(), n, cin, w.data_ptr(), S, cout, gy.data_ptr(), n, gx.data_ptr(), n,
                                            gw.data_ptr(), tree.data_ptr(), ldt, gx32.data_ptr(), n, gt.data_ptr(), nt, st) == 0, lib.aprnet_last_error()
            results.append([t.float().cpu() for t in (y, gw)])        # (the input gradient does not read the tree)
    finally:
        lib.aprnet_set_conv_path(16)
    for name, a, b in zip(("output", "weight gradient"), *results):
        assert torch.isfinite(a).all() and torch.equal(a, b), name
