"""Plan housekeeping around HIP graphs: the scratch buffer of a plan never moves under a captured graph, and what
would have to allocate during a capture is an error code instead of a failed capture."""
import numpy as np
import pytest
import torch

import apr_cases
from pyapr import APR
from pyapr.aprnet import _ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _weights(levels, cout, cin, seed):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(levels, cout, cin, 3, 3, 3, generator=g) * 0.2).to(DEV)


def test_graph_replays_correctly_after_the_scratch_buffer_grew():
    """capture a small layer -> run a wider layer eagerly (its packed weights need a larger scratch buffer) -> the
    graph still replays into memory it owns and reproduces the eager result bit for bit."""
    apr = apr_cases.random_apr((33, 29, 37), 21, density=0.02)
    n = apr.total_number_particles()
    levels = apr.level_max() - apr.level_min() + 1
    ld = torch.zeros(1, dtype=torch.int32)
    g = torch.Generator().manual_seed(0)
    x_static = torch.randn(1, 4, n, generator=g).to(DEV)
    w_small = _weights(levels, 4, 4, 1)
    with torch.no_grad():
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            _ops.conv_forward([apr], x_static, w_small, ld)          # builds the lists, sizes the scratch for 4 -> 4
        torch.cuda.current_stream().wait_stream(side)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            y_static = _ops.conv_forward([apr], x_static, w_small, ld)
        # a much wider layer on the same plan: the scratch buffer has to grow
        x_wide = torch.randn(1, 48, n, generator=g).to(DEV)
        w_wide = _weights(levels, 64, 48, 2)
        y_wide = _ops.conv_forward([apr], x_wide, w_wide, ld)
        torch.cuda.synchronize()
        assert torch.isfinite(y_wide).all()
        for k in range(3):
            x_new = torch.randn(1, 4, n, generator=g).to(DEV)
            eager = _ops.conv_forward([apr], x_new, w_small, ld)
            torch.cuda.synchronize()
            x_static.copy_(x_new)
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(y_static, eager), f"replay {k}"
            _ops.conv_forward([apr], x_wide, w_wide, ld)             # the wide layer keeps using the new buffer
            torch.cuda.synchronize()


def test_growth_and_first_use_during_capture_are_refused():
    """Under capture the first convolution of a plan (tile and window lists) and a layer that needs a larger scratch
    buffer return APRNET_ERR_UNSUPPORTED (RuntimeError here) before anything is launched; after
    aprnet_plan_reserve the same layer captures."""
    from pyapr import _native
    apr = apr_cases.random_apr((33, 29, 37), 22, density=0.02)
    apr.init_cuda()
    n = apr.total_number_particles()
    levels = apr.level_max() - apr.level_min() + 1
    ld = torch.zeros(1, dtype=torch.int32)
    g = torch.Generator().manual_seed(0)
    x4 = torch.randn(1, 4, n, generator=g).to(DEV)
    x48 = torch.randn(1, 48, n, generator=g).to(DEV)
    w_small, w_wide = _weights(levels, 4, 4, 1), _weights(levels, 64, 48, 2)
    with torch.no_grad():
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            with pytest.raises(RuntimeError, match="captur"):
                _ops.conv_forward([apr], x4, w_small, ld)            # nothing built yet
        eager_small = _ops.conv_forward([apr], x4, w_small, ld)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            with pytest.raises(RuntimeError, match="captur"):
                _ops.conv_forward([apr], x48, w_wide, ld)            # lists are there, the scratch is too small
        lib = _native.hip()
        assert lib.aprnet_plan_reserve(apr.plan(0), 64 << 20, None) == 0
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            y_wide = _ops.conv_forward([apr], x48, w_wide, ld)
        graph.replay()
        torch.cuda.synchronize()
        eager_wide = _ops.conv_forward([apr], x48, w_wide, ld)
        assert torch.equal(y_wide, eager_wide)
        assert torch.equal(_ops.conv_forward([apr], x4, w_small, ld), eager_small)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
def test_aprs_built_beside_plans_that_come_and_go(dtype):
    """Plans dropped after a backward pass (its side stream and events with them) while further APRs are built: the arrays of
    the new APRs are those of the same APR built before any plan was destroyed, and stay so while their own plans run."""
    shapes = [(21 + k, 19, 25 + 7 * k) for k in range(5)]
    want = [[a.copy() for a in apr_cases.random_apr(s, 31 + k, density=0.03).get_state()[4:]] for k, s in enumerate(shapes)]
    ld, g = torch.zeros(1, dtype=torch.int32), torch.Generator().manual_seed(0)
    side = torch.cuda.Stream()
    for turn in range(4):
        for k, s in enumerate(shapes):
            apr = apr_cases.random_apr(s, 31 + k, density=0.03)
            n, levels = apr.total_number_particles(), apr.level_max() - apr.level_min() + 1
            x, gy = torch.randn(1, 8, n, generator=g).to(dtype).to(DEV), torch.randn(1, 20, n, generator=g).to(dtype).to(DEV)
            side.wait_stream(torch.cuda.current_stream())
            with torch.cuda.stream(side if turn % 2 else torch.cuda.current_stream()):
                gx, gw = _ops.conv_backward([apr], x, _weights(levels, 20, 8, k), gy, ld)
            torch.cuda.synchronize()
            assert torch.isfinite(gx.float()).all() and torch.isfinite(gw).all()
            for a, b in zip(apr.get_state()[4:], want[k]):
                assert (a == b).all()
            del apr


def test_partial_sums_of_a_very_wide_layer_stay_within_their_limit():
    """3x3x3 512 -> 512: the gradient of one stencil is 28 MB, and the weight gradient's partial sums take 32 of them at most, however
    many stencils (levels) have windows.  Scratch memory is the plan's own, outside torch's allocator."""
    c, shape = 512, (2, 8, 8192)
    field = np.zeros((1, 4, 4096), np.uint8)
    field[:, :, :550] = 13                                           # fine at one end, a few particles on each of eleven coarser levels
    ld, used = torch.zeros(1, dtype=torch.int32), []
    for _ in range(2):                                               # (the first turn: torch's own allocations)
        apr = APR.from_level_field(shape, field)
        it = apr.iterator()
        assert sum(it.particles_level_end(lv) > it.particles_level_begin(lv) for lv in range(apr.level_min(), 14)) == 12
        n = apr.total_number_particles()
        x, w = torch.randn(1, c, n, device=DEV), torch.randn(apr.level_max() - apr.level_min() + 1, c, c, 3, 3, 3, device=DEV) * 0.01
        apr.init_cuda()
        torch.cuda.synchronize()
        free = torch.cuda.mem_get_info()[0]
        _ops.conv_backward([apr], x, w, x, ld, need_input_grad=False)
        torch.cuda.synchronize()
        used.append(free - torch.cuda.mem_get_info()[0])
    assert used[1] <= 32 * c * c * 27 * 4 + (64 << 20)               # (lists and tables of 18 k particles, in whole pages)


def test_input_gradient_captured_before_the_table_of_parents_is_there():
    """bfloat16 features, eight channels: the first eager backward pass builds the plan's table of parents, a capture must not.  The pass it
    records instead works on channel planes; small whole numbers, so that every replay gives the eager pass's bits, whichever way that goes."""
    from pyapr import _native
    apr = apr_cases.random_apr((33, 29, 37), 23, density=0.02)
    apr.init_cuda()
    n, levels = apr.total_number_particles(), apr.level_max() - apr.level_min() + 1
    ld, g = torch.zeros(1, dtype=torch.int32), torch.Generator().manual_seed(0)
    rand = lambda c: torch.randint(-3, 4, (1, c, n), generator=g).to(torch.bfloat16).to(DEV)
    w = torch.randint(-2, 3, (levels, 16, 8, 3, 3, 3), generator=g).float().to(DEV)
    x, gy = rand(8), rand(16)
    _ops.conv_backward([apr], rand(5), w[:, :, :5].contiguous(), gy, ld)          # tiles, lists and nodes; five channels need no table
    assert _native.hip().aprnet_plan_reserve(apr.plan(0), 64 << 20, None) == 0
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        gx, gw = _ops.conv_backward([apr], x, w, gy, ld)
    assert b"table of parents" in _native.hip().aprnet_last_error()               # asked for and refused
    for k in range(3):
        x.copy_(rand(8)); gy.copy_(rand(16))
        want = _ops.conv_backward([apr], x, w, gy, ld) if k else None             # from the second replay on the table is there
        graph.replay()
        torch.cuda.synchronize()
        if want is None: want = _ops.conv_backward([apr], x, w, gy, ld)
        assert torch.equal(gx, want[0]) and torch.equal(gw, want[1]) and float(gx.float().abs().max()) > 0
