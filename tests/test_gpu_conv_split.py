"""Stencil convolution of fp32 features on products of bfloat16 pieces, against the oracle in float64, the fp32 matrix
instructions and the scanning kernels."""
import ctypes as C

import pytest
import torch

import apr_cases
from oracle import oracle
from pyapr import _native
from pyapr.aprnet import _ops
from test_gpu_parity import DEV, _conv_case, close

pytestmark = pytest.mark.gpu


@pytest.fixture
def path():
    lib = _native.hip()
    yield lambda p: lib.aprnet_set_conv_path(p)
    for p in (18, 4, 0):
        lib.aprnet_set_conv_path(p)


def layer(w_exp):
    return w_exp.permute(1, 2, 0, 3, 4, 5).contiguous().to(DEV)          # -> [S, Cout, Cin, k]


def error(got, ref):
    return float((got.cpu().double() - ref).norm() / ref.norm())


# 16 and 17 outputs: either side of a block of output channels; 18 and 19 inputs: incomplete groups of four
@pytest.mark.parametrize("cin,cout", [(16, 1), (18, 16), (19, 17), (32, 33), (64, 64)])
@pytest.mark.parametrize("ksize", [(3, 3, 3), (1, 5, 5)], ids=["k333", "k155"])
@pytest.mark.parametrize("bt", [[("3d_s", 0), ("3d_t", 1)], [("3d_c", 2)], [("2d_a", 1), ("2d_s", 0)]], ids=["3d", "3d_coarse", "2d"])
def test_against_float64(path, bt, ksize, cin, cout):
    x, aprs, ld, w_exp = _conv_case(bt, ksize, 2, cin, cout, torch.float32)
    ref = oracle.conv_forward(aprs, x.double(), w_exp.double(), ld)
    xd, wd = x.to(DEV), layer(w_exp)
    path(19)
    fp32 = _ops.conv_forward(aprs, xd, wd, ld)
    path(20)
    got = _ops.conv_forward(aprs, xd, wd, ld)
    assert not torch.equal(got, fp32)                                    # the other kernel ran
    close(got, ref.float(), torch.float32)
    # six products of pieces leave out less than 2^-25 of |x w| and the large sum is rounded once per 32 products, not once per
    # product: no larger an error than that of the fp32 products
    assert error(got, ref) <= error(fp32, ref)
    assert torch.equal(got, _ops.conv_forward(aprs, xd, wd, ld))         # no atomics
    # the input in two tensors, bias and ReLU
    b = torch.linspace(-1, 1, cout)
    c1 = cin - 5
    y = _ops.conv_forward(aprs, xd[:, :c1].contiguous(), wd, ld, b.to(DEV), relu=True, x2=xd[:, c1:].contiguous())
    for i, a in enumerate(aprs):
        n = oracle.number_parts(a, int(ld[i]))
        assert torch.equal(y[i, :, :n], (got[i, :, :n] + b.to(DEV)[:, None]).relu())


@pytest.mark.parametrize("cout", [3, 32, 40])
@pytest.mark.parametrize("where", ["features", "weights"])
def test_infinities_and_nan(path, where, cout):
    """A result that is not finite is computed again from the fp32 values: infinities and NaN where IEEE arithmetic has
    them, and nowhere else; values whose first bfloat16 piece is infinite give the finite result."""
    x, aprs, ld, w_exp = _conv_case([("3d_s", 0)], (3, 3, 3), 2, 16, cout, torch.float32)
    w_exp = w_exp * 1e-3
    inf = float("inf")
    if where == "features":
        n = oracle.number_parts(aprs[0], 0)
        for i, v in enumerate((inf, -inf, float("nan"), 3.4e38, -3.4e38)):
            x[0, 3 * i, (n * (i + 1)) // 7] = v
        w_exp[0] = 0.0                                                   # infinity times zero
    else:
        w_exp[2, 0, 1, 0, 1, 2], w_exp[5, -1, 0, 1, 1, 1], w_exp[7, 0, 2, 2, 2, 2] = inf, float("nan"), 3.4e38
        x[:, 7] *= 1e-6
    ref = oracle.conv_forward(aprs, x.double(), w_exp.double(), ld)
    path(20)
    got = _ops.conv_forward(aprs, x.to(DEV), layer(w_exp), ld).cpu()
    assert torch.equal(got.isnan(), ref.isnan())
    assert torch.equal(got[ref.isinf()].double(), ref[ref.isinf()])
    fin = ref.isfinite()
    assert fin.any() and not fin.all()
    assert bool(got[fin].isfinite().all())
    # 432 products and as many sums, each rounded to 2^-24 of at most the sum of the magnitudes at that place
    terms = oracle.conv_forward(aprs, x.double().abs(), w_exp.double().abs(), ld)
    bounded = fin & terms.isfinite()
    assert bool(((got.double() - ref).abs() <= 2 * 432 * 2.0 ** -24 * terms)[bounded].all())


@pytest.mark.parametrize("x_scale,w_scale", [(1e-33, 1), (1e-36, 1), (1e-38, 1), (1e-41, 1), (1, 1e-35), (1, 1e-38), (1e-36, 1e30), (1e-18, 1e-18), (1e-22, 1e-22)])
@pytest.mark.parametrize("ksize", [(3, 3, 3), (1, 5, 5)], ids=["k333", "k155"])
def test_small_operands_keep_their_bits(path, ksize, x_scale, w_scale):
    """Features, output gradients and weights down to the end of the exponent range: no larger an error than that of the fp32
    instructions, forward and input gradient.  (The tail of a softmax, or the gradient of a saturated one, lies there.)"""
    bt = [("3d_s", 0)] if ksize[0] == 3 else [("2d_t", 0)]
    x, aprs, ld, w_exp = _conv_case(bt, ksize, 2, 16, 16, torch.float32)
    x, w_exp = x * x_scale, w_exp * w_scale
    ref = oracle.conv_forward(aprs, x.double(), w_exp.double(), ld)
    gref = oracle.conv_backward(aprs, x.double(), w_exp.double(), x.double(), ld)[0]
    xd, wd, err = x.to(DEV), layer(w_exp), {}
    for p in (19, 20):
        path(p)
        err[p] = error(_ops.conv_forward(aprs, xd, wd, ld), ref), error(_ops.conv_backward(aprs, xd, wd, xd, ld)[0], gref)
    assert err[20][0] <= err[19][0] and err[20][1] <= err[19][1]


def nan_places(aprs, ld, x, every):
    x = x.clone()
    for i, a in enumerate(aprs):
        n = oracle.number_parts(a, int(ld[i]))
        x[i, (3 * i) % x.size(1), n // 3:n:every] = float("nan")
    return x


# many places of one tile, several tiles, and (96 outputs of a 64^3 volume) more tiles and blocks than there are words for their marks
@pytest.mark.parametrize("cin,cout,second,every", [(16, 16, 0, 997), (19, 33, 0, 499), (24, 40, 7, 997), (16, 3, 8, 499), (16, 96, 0, 9973)])
@pytest.mark.parametrize("bt,ksize", [([("3d_s", 0), ("3d_t", 1)], (3, 3, 3)), ([("3d_c", 2)], (3, 3, 3)), ([("2d_t", 0), ("2d_s", 1)], (1, 5, 5)), (None, (3, 3, 3))],
                         ids=["333", "333_coarse", "155", "333_many"])
def test_tiles_computed_again_are_those_of_the_fp32_instructions(path, bt, ksize, cin, cout, second, every):
    """Every result of a pass over features with NaN is the fp32 instructions' or, in tiles that none reaches, the pieces', bit for
    bit, with bias, ReLU and an input in two tensors; NaN is where the fp32 instructions have it."""
    if bt is None:
        apr = apr_cases.random_apr((96, 96, 128), 41, 0.4)
        aprs, ld, n = [apr], torch.zeros(1, dtype=torch.int32), apr.total_number_particles()
        x = torch.randn(1, cin, n, generator=torch.Generator().manual_seed(1))
        w_exp = torch.randn(cin, apr.level_max() - apr.level_min() + 1, cout, *ksize, generator=torch.Generator().manual_seed(2))
    else:
        x, aprs, ld, w_exp = _conv_case(bt, ksize, 2, cin, cout, torch.float32)
    wd, b = layer(w_exp), torch.linspace(-1, 1, cout).to(DEV)

    def run(p, xs):
        path(p)
        xs = xs.to(DEV)
        if second:
            return _ops.conv_forward(aprs, xs[:, :cin - second].contiguous(), wd, ld, b, relu=True, x2=xs[:, cin - second:].contiguous())
        return _ops.conv_forward(aprs, xs, wd, ld, b)
    xn = nan_places(aprs, ld, x, every)
    fp32, pieces, got = run(19, xn), run(20, x), run(20, xn)
    nan = fp32.isnan()
    assert bool(nan.any()) and not bool(nan.all()) and torch.equal(got.isnan(), nan)
    again = got == fp32
    assert bool((again | (got == pieces) | nan).all())
    assert bool((again & ~nan & (fp32 != pieces)).any())


def test_results_that_are_not_finite_cost_little(path):
    """A NaN in every window: all tiles are computed a second time, on the matrix cores as well.  (One thread per output: 33 times the
    finite pass.  The two passes and the copies come to less than four; eight leaves room for a busy machine.)"""
    apr = apr_cases.random_apr((96, 96, 128), 41, 0.4)
    apr.init_cuda()
    n, ld = apr.total_number_particles(), torch.zeros(1, dtype=torch.int32)
    g = torch.Generator().manual_seed(2)
    w = torch.randn(apr.level_max() - apr.level_min() + 1, 32, 32, 3, 3, 3, generator=g).to(DEV)
    x = torch.randn(1, 32, n, generator=g).to(DEV)
    xn = x.clone()
    xn[0, :, ::7] = float("nan")
    path(20)

    def ms(xs):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        times = []
        for _ in range(5):
            a.record()
            _ops.conv_forward([apr], xs, w, ld)
            b.record()
            b.synchronize()
            times.append(a.elapsed_time(b))
        return min(times)
    assert ms(xn) <= 8 * ms(x)


def test_route_by_work_space(path):
    """Little work, the 1x3x3 stencil and few channels ask for no work space; with too small a one, none, or lists switched off the
    call is the fp32 kernel's, bit for bit."""
    lib = _native.hip()
    x, aprs, ld, w_exp = _conv_case([("3d_s", 0)], (3, 3, 3), 2, 16, 32, torch.float32)
    xd, wd, a = x.to(DEV), layer(w_exp), aprs[0]
    a.init_cuda()
    S, n = wd.size(0), x.size(2)
    need = lambda kz, k, cin, cout: lib.aprnet_conv_ws_bytes_f32(a.plan(0), 0, kz, k, k, cin, S, cout)
    assert need(3, 3, 16, 16) == 0 and need(3, 3, 64, 32) == 0 and need(3, 3, 64, 4096) > 0
    path(20)
    assert need(1, 3, 64, 64) == 0 and need(5, 5, 64, 64) == 0 and need(3, 3, 15, 64) == 0
    nb = need(3, 3, 16, 32)
    assert nb > 0
    ldt = max(_ops.tree_parts(a, 0), 1)

    def run(nbytes):
        ws = torch.empty(max(nbytes, 1) + 16, dtype=torch.uint8, device=DEV)
        tree, y = torch.empty(16, ldt, device=DEV), torch.empty(32, n, device=DEV)
        rc = lib.aprnet_conv_fwd_ws_f32(a.plan(0), 0, 3, 3, 3, xd.data_ptr(), n, 16, wd.data_ptr(), S, 32, None, y.data_ptr(), n, tree.data_ptr(), ldt,
                                        None, ws.data_ptr() if nbytes else None, nbytes, torch.cuda.current_stream().cuda_stream)
        assert rc == 0, lib.aprnet_last_error()
        return y
    split = run(nb)
    path(19)
    fp32 = run(nb)
    path(20)
    assert not torch.equal(split, fp32)
    assert torch.equal(run(nb - 1), fp32) and torch.equal(run(0), fp32)
    path(5)
    assert torch.equal(run(nb), fp32)


def test_under_capture(path):
    """Recorded into a graph and replayed on new features, with eager calls in between."""
    x, aprs, ld, w_exp = _conv_case([("3d_s", 0)], (3, 3, 3), 2, 16, 32, torch.float32)
    xs, wd = x.to(DEV), layer(w_exp)
    path(20)
    _ops.conv_forward(aprs, xs, wd, ld)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = _ops.conv_forward(aprs, xs, wd, ld)
    for i in range(4):
        xs.copy_(x.to(DEV) * (i + 1))
        if i == 2:
            xs[0, 0, 5] = float("inf")
        want = _ops.conv_forward(aprs, xs, wd, ld)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(torch.nan_to_num(y), torch.nan_to_num(want)) and torch.equal(y.isnan(), want.isnan())


def gradients(path, p, aprs, xd, wd, gy, ld):
    path(p)
    return _ops.conv_backward(aprs, xd, wd, gy, ld)


@pytest.mark.parametrize("cin,cout", [(1, 16), (16, 18), (17, 19), (33, 32)])
@pytest.mark.parametrize("ksize", [(3, 3, 3), (1, 5, 5)], ids=["k333", "k155"])
@pytest.mark.parametrize("bt", [[("3d_s", 0), ("3d_t", 1)], [("3d_a", 0)], [("3d_c", 2)], [("2d_a", 1), ("2d_s", 0)]], ids=["3d", "3d_odd", "3d_coarse", "2d"])
def test_input_gradient_against_float64(path, bt, ksize, cin, cout):
    x, aprs, ld, w_exp = _conv_case(bt, ksize, 2, cin, cout, torch.float32)
    gy = torch.randn(x.size(0), cout, x.size(2), generator=torch.Generator().manual_seed(3))
    for i, a in enumerate(aprs):
        gy[i, :, oracle.number_parts(a, int(ld[i])):] = 0
    xd, wd, gd = x.to(DEV), layer(w_exp), gy.to(DEV)
    ref = _ops.conv_backward(aprs, xd.double(), wd.double(), gd.double(), ld)[0].cpu()
    fp32, fp32_w = gradients(path, 19, aprs, xd, wd, gd, ld)
    got, got_w = gradients(path, 20, aprs, xd, wd, gd, ld)
    assert not torch.equal(got, fp32) and torch.equal(got_w, fp32_w)
    close(got, ref.float(), torch.float32)
    assert error(got, ref) <= error(fp32, ref)
    # repeats bit for bit, far faces included; a flat stencil in a volume adds three sums to a coarser particle, from two slices and
    # its own level, in any order (on the fp32 path as well)
    if ksize[0] == 3 or bt[0][0].startswith("2d"):
        assert torch.equal(got, gradients(path, 20, aprs, xd, wd, gd, ld)[0])


@pytest.mark.parametrize("value", [float("inf"), float("nan"), 3.4e38])
def test_input_gradient_that_is_not_finite(path, value):
    """Then all of it is the fp32 instructions', bit for bit; 3.4e38 has an infinite first piece but finite results."""
    x, aprs, ld, w_exp = _conv_case([("3d_a", 0)], (3, 3, 3), 2, 8, 16, torch.float32)
    gy = torch.randn(1, 16, x.size(2), generator=torch.Generator().manual_seed(3))
    gy[0, 3, 11] = value
    xd, wd, gd = x.to(DEV), layer(w_exp) * 1e-3, gy.to(DEV)
    fp32 = gradients(path, 19, aprs, xd, wd, gd, ld)[0]
    got = gradients(path, 20, aprs, xd, wd, gd, ld)[0]
    assert torch.equal(got.nan_to_num(nan=7.0), fp32.nan_to_num(nan=7.0)) and bool(fp32.isfinite().all()) == (value == 3.4e38)

@pytest.mark.parametrize("cin,cout", [(8, 18), (33, 16), (17, 64)])
@pytest.mark.parametrize("bt,ksize", [([("3d_c", 2)], (3, 3, 3)), ([("3d_s", 0), ("3d_a", 0)], (3, 3, 3)), ([("2d_a", 1), ("2d_s", 0)], (1, 5, 5))], ids=["333_coarse", "333_two", "155"])
def test_input_gradient_made_again(path, bt, ksize, cin, cout):
    """As above for other stencils, level deltas, blocks of channels and batches of which one item is finite: the item with a NaN is
    the fp32 instructions', the other one the pieces'."""
    x, aprs, ld, w_exp = _conv_case(bt, ksize, 2, cin, cout, torch.float32)
    gy = torch.randn(x.size(0), cout, x.size(2), generator=torch.Generator().manual_seed(3))
    for i, a in enumerate(aprs):
        gy[i, :, oracle.number_parts(a, int(ld[i])):] = 0
    xd, wd = x.to(DEV), layer(w_exp)
    pieces = gradients(path, 20, aprs, xd, wd, gy.to(DEV), ld)[0]
    gy[0, cout // 2, oracle.number_parts(aprs[0], int(ld[0])) // 2] = float("nan")
    fp32 = gradients(path, 19, aprs, xd, wd, gy.to(DEV), ld)[0]
    got = gradients(path, 20, aprs, xd, wd, gy.to(DEV), ld)[0]
    assert bool(fp32[0].isnan().any()) and torch.equal(got[0].isnan(), fp32[0].isnan())
    assert torch.equal(got[0].nan_to_num(nan=7.0), fp32[0].nan_to_num(nan=7.0))
    assert torch.equal(got[1:], pieces[1:])



def test_recorded_pass_keeps_the_fp32_products(path):
    """A forward pass that a backward pass may follow is the fp32 instructions', as is the weight gradient."""
    from pyapr import aprnet
    x, aprs, ld, _ = _conv_case([("3d_s", 0)], (3, 3, 3), 2, 16, 32, torch.float32)
    conv, xd = aprnet.cuda.APRConv(16, 32, nstencils=2).to(DEV), x.to(DEV)
    out = {}
    for p in (19, 20):
        path(p)
        with torch.no_grad():
            out[p, "inference"] = conv(xd, aprs, ld)
        xg = xd.clone().requires_grad_(True)
        out[p, "training"] = conv(xg, aprs, ld)
        out[p, "grads"] = torch.autograd.grad(out[p, "training"].square().sum(), (conv.weight, conv.bias))
    assert torch.equal(out[19, "training"], out[20, "training"]) and torch.equal(out[19, "inference"], out[19, "training"])
    assert all(torch.equal(a, b) for a, b in zip(out[19, "grads"], out[20, "grads"]))
    assert not torch.equal(out[20, "inference"], out[20, "training"])


@pytest.mark.parametrize("products", [1, 2, 3, 9, 27])
@pytest.mark.parametrize("zeros", ["weights", "features"])
@pytest.mark.parametrize("ksize,cout", [((3, 3, 3), 16), ((3, 3, 3), 32), ((1, 5, 5), 16), ((1, 5, 5), 32)], ids=["k333_16", "k333_32", "k155_16", "k155_32"])
def test_few_products(path, ksize, cout, zeros, products):
    """Stencils or features with hardly a value that is not zero: a chain of fp32 multiply-adds is then rounded only a few times, and the
    error of the pieces is no larger.  (But for one product: what is left out of it, at most 2^-26 of it twice, has a quarter of
    the spread of one rounding at the most, so the error is at most sqrt(1 + 1/16) = 1.03 of one rounding's; 0.03 for the sample.)"""
    apr = apr_cases.random_apr((48, 64, 64), 43, 0.4)
    apr.init_cuda()
    n, ld, S, cin = apr.total_number_particles(), torch.zeros(1, dtype=torch.int32), apr.level_max() - apr.level_min() + 1, 16
    g = torch.Generator().manual_seed(5)
    x, w = torch.randn(1, cin, n, generator=g), torch.randn(S, cout, cin, *ksize, generator=g)
    taps = cin * w[0, 0, 0].numel()
    if zeros == "weights":
        flat = w.view(S, cout, taps)
        flat *= torch.zeros_like(flat).scatter_(2, torch.rand(flat.shape, generator=g).topk(products, 2)[1], 1.0)
    else:
        x *= torch.rand(x.shape, generator=g) < products / taps
    xd, wd, err = x.to(DEV), w.to(DEV), {}
    gd = torch.randn(1, cout, n, generator=g).to(DEV)
    if zeros == "features":
        gd *= (torch.rand(gd.shape, generator=g) < products / (taps * cout // cin)).to(DEV)
    ref, gref = (t.cpu() for t in (_ops.conv_forward([apr], xd.double(), wd.double(), ld), _ops.conv_backward([apr], xd.double(), wd.double(), gd.double(), ld)[0]))
    for p in (19, 20):
        path(p)
        err[p] = error(_ops.conv_forward([apr], xd, wd, ld), ref), error(_ops.conv_backward([apr], xd, wd, gd, ld)[0], gref)
    most = 1.06 if products == 1 else 1.0
    assert err[20][0] <= most * err[19][0]
    assert err[20][1] <= most * err[19][1]


def test_no_memory_for_the_work_space(path, monkeypatch):
    """The call runs on the fp32 instructions then, and says so."""
    x, aprs, ld, w_exp = _conv_case([("3d_s", 0)], (3, 3, 3), 2, 16, 32, torch.float32)
    xd, wd = x.to(DEV), layer(w_exp)
    gd = torch.randn(1, 32, x.size(2), generator=torch.Generator().manual_seed(3)).to(DEV)
    path(19)
    fp32, fp32_g = _ops.conv_forward(aprs, xd, wd, ld), _ops.conv_backward(aprs, xd, wd, gd, ld)[0]
    path(20)
    empty, refused = torch.empty, []

    def full(*size, **kw):
        if kw.get("dtype") is torch.uint8 and not refused:
            refused.append(size)
            raise torch.cuda.OutOfMemoryError("full")
        return empty(*size, **kw)
    for call, want in ((lambda: _ops.conv_forward(aprs, xd, wd, ld), fp32), (lambda: _ops.conv_backward(aprs, xd, wd, gd, ld)[0], fp32_g)):
        refused.clear()
        with monkeypatch.context() as m, pytest.warns(RuntimeWarning, match="work space"):
            m.setattr(torch, "empty", full)
            got = call()
        assert refused and torch.equal(got, want)


def test_what_counts_as_recorded(path):
    """Grad mode on with nothing that requires a gradient: no backward pass can follow, so the pass is inference's."""
    from pyapr import aprnet
    x, aprs, ld, _ = _conv_case([("3d_s", 0)], (3, 3, 3), 2, 16, 32, torch.float32)
    conv, xd = aprnet.cuda.APRConv(16, 32, nstencils=2).to(DEV), x.to(DEV)
    path(20)
    recorded = conv(xd, aprs, ld).detach()
    with torch.no_grad():
        inference = conv(xd, aprs, ld)
    conv.requires_grad_(False)
    assert torch.equal(conv(xd, aprs, ld), inference) and not torch.equal(inference, recorded)
    assert torch.equal(conv(xd.clone().requires_grad_(True), aprs, ld).detach(), recorded)


def test_pieces_switched_off_on_modules(path):
    """Re-entrant checkpointing runs its first forward pass without a record and repeats it with one: with ``pieces = False`` both
    give the same bits, those of the fp32 instructions, and so does the input gradient."""
    from pyapr import aprnet
    from torch.utils.checkpoint import checkpoint
    x, aprs, ld, _ = _conv_case([("3d_s", 0)], (3, 3, 3), 2, 16, 32, torch.float32)
    net = torch.nn.ModuleList([aprnet.cuda.APRConv(16, 32, nstencils=2), aprnet.cuda.APRConv(32, 16, nstencils=2)]).to(DEV)
    seen = []

    def region(t):
        for conv in net:
            t = conv(t, aprs, ld)
            seen.append(t.detach().clone())
        return t

    def step(p):
        path(p)
        seen.clear()
        xg = x.to(DEV).requires_grad_(True)
        y = checkpoint(region, xg, use_reentrant=True)
        net.zero_grad()
        y.square().sum().backward()
        return [xg.grad, *(w.grad.clone() for w in net.parameters())]
    with_pieces = step(20)
    assert len(seen) == 4 and not torch.equal(seen[0], seen[2])
    for conv in net:
        conv.pieces = False
    want = step(19)
    got = step(20)
    assert torch.equal(seen[0], seen[2]) and torch.equal(seen[1], seen[3])
    assert all(torch.equal(a, b) for a, b in zip(got, want)) and not torch.equal(got[0], with_pieces[0])
    with torch.no_grad():                                                # the fused form of inference
        fused = net[0].forward_fused(x.to(DEV), aprs, ld, relu=True)
        path(19)
        assert torch.equal(fused, net[0].forward_fused(x.to(DEV), aprs, ld, relu=True))


@pytest.mark.parametrize("cout", [3, 16])
@pytest.mark.parametrize("density,drop", [(0.01, 1), (0.95, 0)], ids=["sparse", "dense"])
def test_sparse_and_dense_windows(path, density, drop, cout):
    """At most 16 outputs run three workgroups per CU where windows hold few columns and two where they hold many: against 64 bits, and
    the tiles of a NaN are the fp32 instructions' either way."""
    apr = apr_cases.random_apr((40, 48, 100), 47, density, drop)
    apr.init_cuda()
    n, ld, S, cin = apr.total_number_particles(), torch.zeros(1, dtype=torch.int32), apr.level_max() - apr.level_min() + 1, 18
    g = torch.Generator().manual_seed(6)
    x, w, b = torch.randn(1, cin, n, generator=g).to(DEV), torch.randn(S, cout, cin, 3, 3, 3, generator=g).to(DEV), torch.linspace(-1, 1, cout).to(DEV)
    ref = (_ops.conv_forward([apr], x.double(), w.double(), ld) + b.double()[:, None]).cpu()
    out = {}
    for p in (19, 20):
        path(p)
        out[p] = _ops.conv_forward([apr], x, w, ld, b)
    assert not torch.equal(out[20], out[19]) and error(out[20], ref) <= error(out[19], ref)
    assert torch.equal(out[20], _ops.conv_forward([apr], x[:, :7].contiguous(), w, ld, b, x2=x[:, 7:].contiguous()))
    x[0, 3, n // 2] = float("nan")
    got = _ops.conv_forward([apr], x, w, ld, b)
    path(19)
    fp32 = _ops.conv_forward([apr], x, w, ld, b)
    assert bool(fp32.isnan().any()) and torch.equal(got.isnan(), fp32.isnan())
    assert bool(((got == fp32) | (got == out[20]) | fp32.isnan()).all())


# ---- weight gradient
@pytest.fixture
def dw_path():
    lib = _native.hip()
    lib.aprnet_set_conv_path(20)
    yield lambda p: lib.aprnet_set_conv_path(p)
    for p in (18, 21, 0):
        lib.aprnet_set_conv_path(p)


def weight_gradients(dw_path, p, aprs, xd, wd, gy, ld):
    dw_path(p)
    return _ops.conv_backward(aprs, xd, wd, gy, ld)[1]


def _dw_case(bt, ksize, cin, cout):
    x, aprs, ld, w_exp = _conv_case(bt, ksize, 2, cin, cout, torch.float32)
    gy = torch.randn(x.size(0), cout, x.size(2), generator=torch.Generator().manual_seed(3))
    for i, a in enumerate(aprs):
        gy[i, :, oracle.number_parts(a, int(ld[i])):] = 0
    return x, aprs, ld, w_exp, gy


# one and several blocks of eight input and of 16 or 32 output channels, incomplete groups of four on either side; windows of one to
# several groups of columns
@pytest.mark.parametrize("cin,cout", [(1, 16), (7, 17), (8, 32), (9, 33), (18, 16), (30, 70)])
@pytest.mark.parametrize("ksize", [(3, 3, 3), (1, 5, 5)], ids=["k333", "k155"])
@pytest.mark.parametrize("bt", [[("3d_s", 0), ("3d_t", 1)], [("3d_a", 0)], [("3d_c", 2)], [("2d_a", 1), ("2d_s", 0)]], ids=["3d", "3d_odd", "3d_coarse", "2d"])
def test_weight_gradient_against_float64(dw_path, bt, ksize, cin, cout):
    x, aprs, ld, w_exp, gy = _dw_case(bt, ksize, cin, cout)
    xd, wd, gd = x.to(DEV), layer(w_exp), gy.to(DEV)
    ref = _ops.conv_backward(aprs, xd.double(), wd.double(), gd.double(), ld)[1].cpu()
    fp32 = weight_gradients(dw_path, 22, aprs, xd, wd, gd, ld)
    got = weight_gradients(dw_path, 23, aprs, xd, wd, gd, ld)
    assert not torch.equal(got, fp32)
    close(got, ref.float(), torch.float32)
    # sums of a handful of products are rounded too few times for the mean to tell: no larger an error over the sample, one per cent of play
    assert error(got, ref) <= 1.01 * error(fp32, ref)
    assert torch.equal(got, weight_gradients(dw_path, 23, aprs, xd, wd, gd, ld))


@pytest.mark.parametrize("where", ["features", "gradient"])
@pytest.mark.parametrize("value", [float("inf"), float("nan"), 3.4e38])
@pytest.mark.parametrize("cin,cout", [(16, 16), (9, 40)])
def test_weight_gradient_that_is_not_finite(dw_path, cin, cout, value, where):
    """Then all of it is the fp32 instructions', bit for bit, of the batch item that holds the value (3.4e38 has an infinite first
    piece, the sums are finite)."""
    x, aprs, ld, w_exp, gy = _dw_case([("3d_s", 0), ("3d_a", 0)], (3, 3, 3), cin, cout)
    (x if where == "features" else gy)[0, 3, 11] = value
    (gy if where == "features" else x).mul_(1e-3)
    xd, wd, gd = x.to(DEV), layer(w_exp), gy.to(DEV)
    fp32 = weight_gradients(dw_path, 22, aprs[:1], xd[:1], wd, gd[:1], ld[:1])
    got = weight_gradients(dw_path, 23, aprs[:1], xd[:1], wd, gd[:1], ld[:1])
    assert torch.equal(got.nan_to_num(nan=7.0), fp32.nan_to_num(nan=7.0)) and bool(fp32.isfinite().all()) == (value == 3.4e38)
    both, item = (weight_gradients(dw_path, 23, aprs[k:], xd[k:], wd, gd[k:], ld[k:]) for k in (0, 1))
    assert torch.equal(both.isnan(), fp32.isnan()) and bool(item.isfinite().all())
    fin = fp32.isfinite() & (fp32.abs() < 1e30)
    assert torch.equal(both[fin], (got + item)[fin]) or error(both[fin], (got + item)[fin].cpu().double()) < 1e-6


@pytest.mark.parametrize("x_scale,g_scale", [(1e-36, 1), (1e-41, 1), (1, 1e-38), (1e-36, 1e30), (1e-18, 1e-18)])
def test_weight_gradient_of_small_operands(dw_path, x_scale, g_scale):
    x, aprs, ld, w_exp, gy = _dw_case([("3d_s", 0)], (3, 3, 3), 16, 16)
    xd, wd, gd = (x * x_scale).to(DEV), layer(w_exp), (gy * g_scale).to(DEV)
    ref = _ops.conv_backward(aprs, xd.double(), wd.double(), gd.double(), ld)[1].cpu()
    err = [error(weight_gradients(dw_path, p, aprs, xd, wd, gd, ld), ref) for p in (22, 23)]
    assert err[1] <= err[0]


@pytest.mark.parametrize("products", [1, 2, 3, 9, 27])
def test_weight_gradient_of_few_products(dw_path, products):
    """An output gradient that is zero but at a few places.  They lie in different windows, whose products go to sums of their own: each of
    these is a single product, whose error is at most 1.03 of one rounding's (see test_few_products), and adding them up rounds
    alike; 0.03 for the sample."""
    apr = apr_cases.random_apr((48, 64, 64), 43, 0.4)
    apr.init_cuda()
    n, ld, S = apr.total_number_particles(), torch.zeros(1, dtype=torch.int32), apr.level_max() - apr.level_min() + 1
    g = torch.Generator().manual_seed(5)
    x, w = torch.randn(1, 32, n, generator=g).to(DEV), torch.randn(S, 32, 32, 3, 3, 3, generator=g).to(DEV)
    gd = torch.zeros(1, 32, n)
    at = torch.randint(n // 2, n, (32, products), generator=g)
    gd[0].scatter_(1, at, torch.randn(32, products, generator=g))
    gd = gd.to(DEV)
    ref = _ops.conv_backward([apr], x.double(), w.double(), gd.double(), ld)[1].cpu()
    err = [error(weight_gradients(dw_path, p, [apr], x, w, gd, ld), ref) for p in (22, 23)]
    assert err[1] <= 1.06 * err[0]


def test_weight_gradient_under_capture(dw_path):
    """Recorded into a graph and replayed on new features, finite ones and others, with eager calls in between."""
    x, aprs, ld, w_exp, gy = _dw_case([("3d_s", 0)], (3, 3, 3), 16, 32)
    xs, wd, gd = x.to(DEV), layer(w_exp), gy.to(DEV)
    weight_gradients(dw_path, 23, aprs, xs, wd, gd, ld)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = _ops.conv_backward(aprs, xs, wd, gd, ld)[1]
    for i in range(4):
        xs.copy_(x.to(DEV) * (i + 1))
        if i == 2:
            xs[0, 0, 5] = float("nan")
        want = _ops.conv_backward(aprs, xs, wd, gd, ld)[1]
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out.nan_to_num(), want.nan_to_num()) and torch.equal(out.isnan(), want.isnan())


# ---- rows of many values: the planes of a group of channels are reached from the first one with unsigned 32-bit offsets
def planes(x, ld):
    """[C, n] -> the same values in rows of ``ld``, with 4 GiB of memory in front of them: an offset that wraps lands in there."""
    t = torch.empty((1 << 30) + x.shape[0] * ld, device=DEV)[1 << 30:].as_strided(x.shape, (ld, 1))
    return t.copy_(x)


@pytest.mark.parametrize("c2", [0, 8, 6], ids=["one-tensor", "two-tensors", "a-group-of-both"])
@pytest.mark.parametrize("ld", [200_000_000, (1 << 28) - 1, 1 << 28])
def test_forward_of_long_rows(path, ld, c2):
    """Offsets past 2^31 bytes and, from rows of 2^28 values on, a descriptor per plane: the bits that compact rows give."""
    path(20)
    lib, st, cin, cout = _native.hip(), torch.cuda.current_stream().cuda_stream, 16, 16
    x, aprs, _, w_exp = _conv_case([("3d_s", 0)], (3, 3, 3), 2, cin, cout, torch.float32)
    apr, xd, w = aprs[0], x[0].to(DEV), layer(w_exp)
    n, nt, c1 = _ops.number_particles(apr, 0), _ops.tree_parts(apr, 0), cin - c2
    xd = xd[:, :n].contiguous()
    out = []
    try:
        for lx, lt in ((n, nt), (ld, ld)):
            tree = planes(torch.zeros(cin, nt, device=DEV), lt)
            a, b = planes(xd[:c1], lx), planes(xd[c1:], lx) if c2 else None
            y = torch.empty(cout, n, device=DEV)
            ws_bytes = lib.aprnet_conv_ws_bytes_f32(apr.plan(0), 0, 3, 3, 3, cin, w.shape[0], cout)
            assert ws_bytes > 0
            ws = torch.empty(ws_bytes, dtype=torch.uint8, device=DEV)
            fu = _ops._Fusion(b.data_ptr() if c2 else None, lx, c2, 0)
            assert lib.aprnet_conv_fwd_ws_f32(apr.plan(0), 0, 3, 3, 3, a.data_ptr(), lx, c1, w.data_ptr(), w.shape[0], cout, None, y.data_ptr(), n,
                                              tree.data_ptr(), lt, C.byref(fu), ws.data_ptr(), ws_bytes, st) == 0, lib.aprnet_last_error()
            out.append(y)
            del tree, a, b
        assert torch.equal(*out)
    finally:
        torch.cuda.empty_cache()


@pytest.mark.parametrize("ld", [100_000_000, (1 << 27) - 1, 1 << 27])
def test_weight_gradient_of_long_rows(dw_path, ld):
    """The same with eight planes per workgroup; rows of 2^27 values and more are left to the fp32 instructions."""
    lib, st, cin, cout = _native.hip(), torch.cuda.current_stream().cuda_stream, 16, 16
    x, aprs, _, w_exp, gy = _dw_case([("3d_s", 0)], (3, 3, 3), cin, cout)
    apr, w = aprs[0], layer(w_exp)
    n, nt = _ops.number_particles(apr, 0), _ops.tree_parts(apr, 0)
    xd, gd = x[0, :, :n].contiguous().to(DEV), gy[0, :, :n].contiguous().to(DEV)
    out = []
    try:
        for lx, lt, p in ((n, nt, 23 if ld < 1 << 27 else 22), (ld, ld, 23)):
            dw_path(p)
            a, tree = planes(xd, lx), planes(torch.zeros(cin, nt, device=DEV), lt)
            gx, gw, gt = torch.empty(cin, n, device=DEV), torch.zeros_like(w), torch.empty(cin, nt, device=DEV)
            ws_bytes = lib.aprnet_conv_bwd_ws_bytes_f32(apr.plan(0), 0, 3, 3, 3, cin, w.shape[0], cout)
            assert ws_bytes > 0
            ws = torch.empty(ws_bytes, dtype=torch.uint8, device=DEV)
            assert lib.aprnet_conv_bwd_ws_f32(apr.plan(0), 0, 3, 3, 3, a.data_ptr(), lx, cin, w.data_ptr(), w.shape[0], cout, gd.data_ptr(), n,
                                              gx.data_ptr(), n, gw.data_ptr(), tree.data_ptr(), lt, gt.data_ptr(), nt, ws.data_ptr(), ws_bytes, st) == 0, \
                lib.aprnet_last_error()
            out.append(gw)
            del a, tree
        assert torch.equal(*out)
    finally:
        torch.cuda.empty_cache()
