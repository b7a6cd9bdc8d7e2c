"""GPU parity: every kernel family, called through the C ABI, against the CPU oracle on the same
seeded inputs.  Integer/selection work (addresses, gathered values, table lookups, eval outputs,
thermometer bits, argmax) must be bit-exact; floating-point sums are held to rtol 1e-5 with an
absolute floor of a few fp32 ulps of the operand scale (stated per test)."""
import numpy as np
import pytest
import torch

from oracle import c_oracle
from oracle import difflut_oracle as orc

pytestmark = pytest.mark.gpu

DEV = "cuda"


def _ops():
    from difflut_amd import ops
    return ops


def dev(a, dtype=torch.float32):
    return torch.as_tensor(np.ascontiguousarray(a)).to(DEV, dtype)


def make_case(seed, B, I, N, k, O, lo=-1.0, hi=1.0, binary=False):
    rng = np.random.default_rng(seed)
    x = rng.integers(0, 2, (B, I)).astype(np.float32) if binary else rng.random((B, I)).astype(np.float32)
    idx = orc.random_mapping(I, N, k, seed=seed + 1).numpy().astype(np.int64)
    tab = rng.uniform(lo, hi, (N, O, 1 << k)).astype(np.float32)
    gy = rng.standard_normal((B, N, O)).astype(np.float32)
    return x, idx, tab, gy


DWN_SHAPES = [  # (B, I, N, k, O)
    (100, 25, 36, 6, 1),   # reference tests/test_layers/test_fused_kernels.py:26-36
    (10, 16, 25, 4, 1),    # test_fused_kernels.py:62-72
    (8, 256, 128, 4, 1),   # tests/test_layers/test_layer_functionality.py:37-55
    (70, 40, 33, 3, 2),
    (64, 128, 256, 6, 1),
    (130, 300, 77, 5, 3),
    (1, 7, 5, 1, 1),
    (322, 52, 80, 1, 1),   # k = 1: the S-form table (2 floats per node) is larger than the D form (1 float)
    (65, 9, 300, 2, 1),
    (200, 1030, 515, 6, 2),
    (9, 30, 11, 7, 2),     # k > 6: generic kernels
    (5, 64, 6, 9, 1),
    (21, 1031, 1100, 7, 1),  # k > 6 from 1024 columns on: the row of x through the LDS (odd width: scalar staging)
    (6, 512, 520, 8, 2),     # the same with two outputs per node
]


@pytest.mark.parametrize("shape", DWN_SHAPES)
def test_dwn_layer_forward_backward(shape):
    B, I, N, k, O = shape
    ops = _ops()
    x, idx, luts, gy = make_case(sum(shape), *shape)
    plan = ops.MappingPlan(dev(idx, torch.int32), I)
    xt = dev(x).requires_grad_()
    lt = dev(luts).requires_grad_()
    alpha, beta = 0.5 * 0.75 ** (k - 1), 1.0 / 3.0
    y = ops.DWNLayerFunction.apply(xt, lt, plan, alpha, beta)
    want = orc.dwn_layer_forward(x, idx, luts).reshape(B, N * O)
    assert np.array_equal(y.detach().cpu().numpy(), want)  # bit exact
    y.backward(dev(gy.reshape(B, N * O)))
    gx, gl = orc.dwn_layer_backward(x, idx, luts, gy, np.float32(alpha), np.float32(beta))
    # gx sums <= fan-in terms of size alpha*|gy|*|D| ~ 0.1..1: rtol 1e-5, floor 2e-6
    np.testing.assert_allclose(xt.grad.cpu().numpy(), gx, rtol=1e-5, atol=2e-6)
    # table gradients are plain sums of gy over the rows that hit an entry
    np.testing.assert_allclose(lt.grad.cpu().numpy(), gl, rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("shape", [(1, 1, 1, 1, 2), (64, 17, 40, 6, 2), (65, 130, 61, 5, 2), (130, 9, 33, 3, 2), (66, 64, 30, 8, 2),
                                   (66, 64, 30, 7, 2), (70, 33, 20, 4, 3)])
@pytest.mark.parametrize("beta", [1.0 / 3.0, 0.75])  # both forms of the coefficient table
def test_dwn_backward_several_outputs_per_node(shape, beta):
    """Two outputs per node are requested with a step's entries, three and more are walked: both forms, lists shorter and
    longer than a step of eight."""
    B, I, N, k, O = shape
    ops = _ops()
    x, idx, luts, gy = make_case(sum(shape) + 5, *shape)
    plan = ops.MappingPlan(dev(idx, torch.int32), I)
    xt, lt = dev(x).requires_grad_(), dev(luts).requires_grad_()
    alpha = 0.5 * 0.75 ** (k - 1)
    ops.DWNLayerFunction.apply(xt, lt, plan, alpha, beta).backward(dev(gy.reshape(B, N * O)))
    gx, gl = orc.dwn_layer_backward(x, idx, luts, gy, np.float32(alpha), np.float32(beta))
    # a term is alpha |gy| |D| with |D| <= 2 (1 + beta)^(k-1) |lut|, at most 11.3 |gy| here (k = 8, beta = 0.75), and a sum has
    # O N k / I of them: 64 roundings of 6e-8 of terms of that size, as an absolute floor
    size = alpha * 2.0 * (1.0 + beta) ** (k - 1)
    np.testing.assert_allclose(xt.grad.cpu().numpy(), gx, rtol=1e-5, atol=max(2e-6, 64 * 6e-8 * size))
    np.testing.assert_allclose(lt.grad.cpu().numpy(), gl, rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("shape", [(33000, 50, 300, 6, 1), (40000, 7, 40, 2, 1)])
def test_dwn_backward_few_inputs_many_rows(shape):
    """Few inputs read by many nodes over many rows (the shape of the first level of a convolutional layer:
    CSR lists of ~36 entries per input, hundreds of batch tiles) against the C restatement on all rows."""
    B, I, N, k, O = shape
    ops = _ops()
    x, idx, luts, gy = make_case(sum(shape) % 1000, *shape)
    plan = ops.MappingPlan(dev(idx, torch.int32), I)
    alpha, beta = 0.5 * 0.75 ** (k - 1), 1.0 / 3.0
    xt = dev(x).requires_grad_()
    lt = dev(luts).requires_grad_()
    y = ops.DWNLayerFunction.apply(xt, lt, plan, alpha, beta)
    y.backward(dev(gy.reshape(B, N * O)))
    assert np.array_equal(y.detach().cpu().numpy(), c_oracle.dwn_layer_forward(x, idx, luts).reshape(B, N * O))
    wx, wl = c_oracle.dwn_layer_backward(x, idx, luts, gy, alpha, beta)
    # up to N*k/I (~36) terms of size alpha*|gy|*|D| per input: rtol 1e-5, floor 5e-6
    np.testing.assert_allclose(xt.grad.cpu().numpy(), wx, rtol=1e-5, atol=5e-6)
    np.testing.assert_allclose(lt.grad.cpu().numpy(), wl, rtol=1e-5, atol=2e-4)  # ~B/2^k terms per bin


@pytest.mark.parametrize("shape", [(700, 20, 200, 6, 1), (130, 50, 64, 5, 1), (260, 9, 40, 6, 1), (65, 100, 50, 6, 1)])
def test_dwn_backward_tile_major_output_all_list_lengths(shape):
    """The tile-major form of the input gradient (what a chained layer or the fold of a convolutional layer
    reads) through the C entry point, for average CSR list lengths of 60, 6.4, 27 and 3: the gather runs with
    1, 4, 4 and 16 inputs per wavefront.  Every tile against the row-major result of the same call sequence
    and against the oracle."""
    from difflut_amd import _native as nat
    B, I, N, k, O = shape
    ops = _ops()
    lib = nat.lib()
    x, idx, luts, gy = make_case(sum(shape) % 997, *shape)
    plan = ops.MappingPlan(dev(idx, torch.int32), I)
    alpha, beta = 0.5 * 0.75 ** (k - 1), 1.0 / 3.0
    dims = (B, I, N, k, O)
    xd, ld, gd = dev(x), dev(luts), dev(gy.reshape(B, N * O))
    y = torch.empty(B, N * O, device=DEV)
    saved = torch.empty(lib.dl_dwn_saved_bytes(*dims), dtype=torch.uint8, device=DEV)
    wf = torch.empty(lib.dl_dwn_fwd_workspace_bytes(*dims), dtype=torch.uint8, device=DEV)
    wb = torch.empty(lib.dl_dwn_bwd_workspace_bytes(*dims), dtype=torch.uint8, device=DEV)
    nat.check(lib.dl_dwn_layer_fwd(xd.data_ptr(), plan.idx32.data_ptr(), ld.data_ptr(), y.data_ptr(), saved.data_ptr(),
                                   wf.data_ptr(), wf.numel(), *dims, nat.stream()))
    BT = (B + 63) // 64
    results = []
    for tiled in (0, 1):
        gx = torch.zeros(BT * I * 64 if tiled else B * I, device=DEV)
        gl = torch.empty_like(ld)
        nat.check(lib.dl_dwn_layer_bwd_tiled(saved.data_ptr(), plan.inv_ptr.data_ptr(), plan.inv_pos.data_ptr(), ld.data_ptr(),
                                             gd.data_ptr(), 0, alpha, beta, gx.data_ptr(), tiled, gl.data_ptr(), wb.data_ptr(),
                                             wb.numel(), *dims, nat.stream()))
        results.append((gx, gl))
    row_major = results[0][0].view(B, I)
    tile_major = results[1][0].view(BT, I, 64).permute(0, 2, 1).reshape(BT * 64, I)[:B]
    assert torch.equal(tile_major, row_major)  # same sums in the same order, another layout
    wx, wl = orc.dwn_layer_backward(x, idx, luts, gy, np.float32(alpha), np.float32(beta))
    np.testing.assert_allclose(row_major.cpu().numpy(), wx, rtol=1e-5, atol=1e-5)
    np.testing.assert_allclose(results[1][1].cpu().numpy(), wl, rtol=1e-5, atol=2e-4)


FUSED_CHAIN_SHAPES = [  # (B, I0, k_front, I = nodes of the front layer, N, k)
    (200, 40, 6, 128, 64, 6),    # every input read three times: the unrolled path; fewer batch tiles than XCDs
    (1100, 64, 4, 256, 128, 6),  # 18 batch tiles: XCDs with three and with two; 16 bins per column
    (333, 30, 5, 100, 45, 5),    # lists of two and three entries, a last slab of 36 inputs
    (130, 16, 3, 20, 40, 6),     # twelve entries per input: four inputs per wavefront
    (64, 12, 6, 70, 35, 2),      # every input read once
    (150, 20, 4, 96, 32, 6),     # every input read twice
    (300, 16, 6, 48, 48, 6),     # every input read six times: four inputs per wavefront, unrolled
    (150, 16, 4, 24, 48, 6),     # twelve times
    (200, 24, 5, 64, 32, 6),     # three reads per input on average only (see the test)
]


@pytest.mark.parametrize("shape", FUSED_CHAIN_SHAPES)
def test_dwn_chained_backward_fills_the_table_gradient_of_the_layer_in_front(shape):
    """dl_dwn_layer_bwd_chain_fused against the two calls it replaces (the layer's own backward with a tile-major
    input gradient, then the front layer's histogram over that gradient) and against the oracle.  The input
    gradient and the layer's own table gradient keep their order of additions: bit-equal.  The front layer's
    bins are summed per block and then over blocks: rtol 1e-5 with a floor of 2e-5 of the largest bin."""
    from difflut_amd import _native as nat
    B, I0, kf, I, N, k = shape
    ops = _ops()
    lib = nat.lib()
    x0, idx_f, luts_f, _ = make_case(sum(shape) % 991, B, I0, I, kf, 1, lo=0.0)
    _, idx, luts, gy = make_case(sum(shape) % 983, B, I, N, k, 1)
    if shape == FUSED_CHAIN_SHAPES[-1]:
        # N k = 3 I, but drawn independently: the lists are uneven although the host sees a whole fan-in
        idx = np.random.default_rng(5).integers(0, I, (N, k)).astype(np.int64)
    plan_f = ops.MappingPlan(dev(idx_f, torch.int32), I0)
    plan = ops.MappingPlan(dev(idx, torch.int32), I)
    front, dims = (B, I0, I, kf, 1), (B, I, N, k, 1)
    rng = np.random.default_rng(7)
    alpha_n = dev(rng.uniform(0.1, 0.6, N).astype(np.float32))
    beta_n = dev(rng.uniform(-0.4, 0.45, N).astype(np.float32))
    beta_max = float(beta_n.abs().max())

    def forward(xin, pl, tab, d):
        y = torch.empty(d[0], d[2], device=DEV)
        saved = torch.empty(lib.dl_dwn_saved_bytes(*d), dtype=torch.uint8, device=DEV)
        ws = torch.empty(lib.dl_dwn_fwd_workspace_bytes(*d), dtype=torch.uint8, device=DEV)
        nat.check(lib.dl_dwn_layer_fwd(xin.data_ptr(), pl.idx32.data_ptr(), tab.data_ptr(), y.data_ptr(), saved.data_ptr(),
                                       ws.data_ptr(), ws.numel(), *d, nat.stream()))
        return y, saved

    lf, ld, gd = dev(luts_f), dev(luts), dev(gy.reshape(B, N))
    h, saved_f = forward(dev(x0), plan_f, lf, front)
    _, saved = forward(h, plan, ld, dims)
    BT = (B + 63) // 64
    assert lib.dl_dwn_chain_fusable(*dims, kf, beta_max) == 1
    # the two calls
    ws = torch.empty(lib.dl_dwn_bwd_workspace_bytes(*dims), dtype=torch.uint8, device=DEV)
    gx_ref = torch.zeros(BT * I * 64, device=DEV)
    gl_ref = torch.empty_like(ld)
    nat.check(lib.dl_dwn_layer_bwd_chain_nodes(saved.data_ptr(), plan.inv_ptr.data_ptr(), plan.inv_pos.data_ptr(), ld.data_ptr(),
                                               gd.data_ptr(), 0, 1, 1.0, alpha_n.data_ptr(), beta_n.data_ptr(), beta_max,
                                               gx_ref.data_ptr(), 1, gl_ref.data_ptr(), ws.data_ptr(), ws.numel(), *dims,
                                               nat.stream()))
    wsf = torch.empty(lib.dl_dwn_bwd_workspace_bytes(*front), dtype=torch.uint8, device=DEV)
    glf_ref = torch.empty_like(lf)
    nat.check(lib.dl_dwn_layer_bwd_tiled(saved_f.data_ptr(), None, None, lf.data_ptr(), gx_ref.data_ptr(), 1, 0.3, 0.3, None, 0,
                                         glf_ref.data_ptr(), wsf.data_ptr(), wsf.numel(), *front, nat.stream()))
    # the one call
    wsx = torch.empty(lib.dl_dwn_bwd_fused_workspace_bytes(*dims, kf), dtype=torch.uint8, device=DEV)
    gx = torch.zeros(BT * I * 64, device=DEV)
    gl = torch.empty_like(ld)
    glf = torch.full_like(lf, 7.0)
    nat.check(lib.dl_dwn_layer_bwd_chain_fused(saved.data_ptr(), plan.inv_ptr.data_ptr(), plan.inv_pos.data_ptr(), ld.data_ptr(),
                                               gd.data_ptr(), 0, 1, 1.0, alpha_n.data_ptr(), beta_n.data_ptr(), beta_max,
                                               gx.data_ptr(), 1, gl.data_ptr(), saved_f.data_ptr(), kf, glf.data_ptr(),
                                               wsx.data_ptr(), wsx.numel(), *dims, nat.stream()))
    assert torch.equal(gx, gx_ref)
    assert torch.equal(gl, gl_ref)
    floor = 2e-5 * float(glf_ref.abs().max())
    np.testing.assert_allclose(glf.cpu().numpy(), glf_ref.cpu().numpy(), rtol=1e-5, atol=floor)
    # the oracle on the front layer, fed with the input gradient just computed (rows past B carry zeros)
    rows = gx.view(BT, I, 64).permute(0, 2, 1).reshape(BT * 64, I)[:B].cpu().numpy()
    _, want = orc.dwn_layer_backward(x0, idx_f, luts_f, rows.reshape(B, I, 1), np.float32(0.3), np.float32(0.3))
    np.testing.assert_allclose(glf.cpu().numpy(), want, rtol=1e-5, atol=floor)
    # the layer's own table gradient already there: gy tile-major, no gluts
    gyT = torch.zeros(BT * 64, N, device=DEV)
    gyT[:B] = gd
    gyT = gyT.view(BT, 64, N).permute(0, 2, 1).contiguous()
    gx2 = torch.zeros_like(gx)
    glf2 = torch.empty_like(lf)
    nat.check(lib.dl_dwn_layer_bwd_chain_fused(saved.data_ptr(), plan.inv_ptr.data_ptr(), plan.inv_pos.data_ptr(), ld.data_ptr(),
                                               gyT.data_ptr(), 1, 1, 1.0, alpha_n.data_ptr(), beta_n.data_ptr(), beta_max,
                                               gx2.data_ptr(), 1, None, saved_f.data_ptr(), kf, glf2.data_ptr(),
                                               wsx.data_ptr(), wsx.numel(), *dims, nat.stream()))
    assert torch.equal(gx2, gx_ref)
    assert torch.equal(glf2, glf)  # fixed order of additions: the same bits on every call
    # no buffer for the input gradient (nobody behind the front layer reads it): the same bins, the same bits, and the
    # layer's own table gradient as before
    glf4, gl4 = torch.empty_like(lf), torch.empty_like(ld)
    nat.check(lib.dl_dwn_layer_bwd_chain_fused(saved.data_ptr(), plan.inv_ptr.data_ptr(), plan.inv_pos.data_ptr(), ld.data_ptr(),
                                               gd.data_ptr(), 0, 1, 1.0, alpha_n.data_ptr(), beta_n.data_ptr(), beta_max,
                                               None, 1, gl4.data_ptr(), saved_f.data_ptr(), kf, glf4.data_ptr(),
                                               wsx.data_ptr(), wsx.numel(), *dims, nat.stream()))
    assert torch.equal(glf4, glf) and torch.equal(gl4, gl_ref)
    # and without a front layer it is the plain chained backward
    gx3 = torch.zeros_like(gx)
    nat.check(lib.dl_dwn_layer_bwd_chain_fused(saved.data_ptr(), plan.inv_ptr.data_ptr(), plan.inv_pos.data_ptr(), ld.data_ptr(),
                                               gyT.data_ptr(), 1, 1, 1.0, alpha_n.data_ptr(), beta_n.data_ptr(), beta_max,
                                               gx3.data_ptr(), 1, None, None, 0, None, ws.data_ptr(), ws.numel(), *dims,
                                               nat.stream()))
    assert torch.equal(gx3, gx_ref)


def test_dwn_chained_backward_refuses_what_it_cannot_fuse():
    from difflut_amd import _native as nat
    lib = nat.lib()
    assert lib.dl_dwn_chain_fusable(64, 9, 64, 6, 1, 6, 0.3) == 0    # 42 entries per input: the one-input gather
    assert lib.dl_dwn_chain_fusable(64, 128, 64, 6, 1, 6, 0.75) == 0  # |beta| > 1/2: the other coefficient form
    assert lib.dl_dwn_chain_fusable(64, 128, 64, 6, 2, 6, 0.3) == 0   # two outputs per node
    assert lib.dl_dwn_chain_fusable(64, 128, 64, 6, 1, 7, 0.3) == 0   # front layer on the generic path
    assert lib.dl_dwn_chain_fusable(64, 128, 64, 6, 1, 4, 0.3) == 1
    buf = torch.zeros(1 << 16, device=DEV)
    rc = lib.dl_dwn_layer_bwd_chain_fused(buf.data_ptr(), buf.data_ptr(), buf.data_ptr(), buf.data_ptr(), buf.data_ptr(), 0, 1,
                                          1.0, buf.data_ptr(), buf.data_ptr(), 0.75, buf.data_ptr(), 1, buf.data_ptr(),
                                          buf.data_ptr(), 6, buf.data_ptr(), buf.data_ptr(), buf.numel() * 4, 64, 128, 64, 6, 1,
                                          nat.stream())
    assert rc == -3  # DL_ERR_UNSUPPORTED


@pytest.mark.parametrize("shape", [(300, 12, 128, 6, 1), (1300, 7, 80, 6, 1), (90, 5, 64, 5, 1)])
def test_dwn_backward_tile_major_output_uneven_long_lists(shape):
    """Inputs read by 40 to 90 nodes each, drawn independently (lists of very different lengths, some beyond what the
    gather for long lists keeps in registers): the tile-major input gradient against the row-major one of the same
    entry point (same terms in the same order: bit-equal) and against the oracle."""
    from difflut_amd import _native as nat
    B, I, N, k, O = shape
    ops = _ops()
    lib = nat.lib()
    rng = np.random.default_rng(sum(shape))
    x = rng.random((B, I)).astype(np.float32)
    idx = rng.integers(0, I, (N, k)).astype(np.int64)
    idx[:, 0] = np.where(rng.random(N) < 0.5, 0, idx[:, 0])  # input 0 is read far more often than the others
    luts = rng.uniform(-1, 1, (N, O, 1 << k)).astype(np.float32)
    gy = rng.standard_normal((B, N, O)).astype(np.float32)
    plan = ops.MappingPlan(dev(idx, torch.int32), I)
    alpha, beta = 0.5 * 0.75 ** (k - 1), 1.0 / 3.0
    dims = (B, I, N, k, O)
    xd, ld, gd = dev(x), dev(luts), dev(gy.reshape(B, N * O))
    y = torch.empty(B, N * O, device=DEV)
    saved = torch.empty(lib.dl_dwn_saved_bytes(*dims), dtype=torch.uint8, device=DEV)
    wf = torch.empty(lib.dl_dwn_fwd_workspace_bytes(*dims), dtype=torch.uint8, device=DEV)
    wb = torch.empty(lib.dl_dwn_bwd_workspace_bytes(*dims), dtype=torch.uint8, device=DEV)
    nat.check(lib.dl_dwn_layer_fwd(xd.data_ptr(), plan.idx32.data_ptr(), ld.data_ptr(), y.data_ptr(), saved.data_ptr(),
                                   wf.data_ptr(), wf.numel(), *dims, nat.stream()))
    BT = (B + 63) // 64
    results = []
    for tiled in (0, 1):
        gx = torch.zeros(BT * I * 64 if tiled else B * I, device=DEV)
        gl = torch.empty_like(ld)
        nat.check(lib.dl_dwn_layer_bwd_tiled(saved.data_ptr(), plan.inv_ptr.data_ptr(), plan.inv_pos.data_ptr(), ld.data_ptr(),
                                             gd.data_ptr(), 0, alpha, beta, gx.data_ptr(), tiled, gl.data_ptr(), wb.data_ptr(),
                                             wb.numel(), *dims, nat.stream()))
        results.append((gx, gl))
    row_major = results[0][0].view(B, I)
    tile_major = results[1][0].view(BT, I, 64).permute(0, 2, 1).reshape(BT * 64, I)[:B]
    assert torch.equal(tile_major, row_major)
    assert torch.equal(results[0][1], results[1][1])
    wx, wl = orc.dwn_layer_backward(x, idx, luts, gy, np.float32(alpha), np.float32(beta))
    # up to ~100 terms of size alpha*|gy|*|D| per input: rtol 1e-5, floor 2e-5
    np.testing.assert_allclose(row_major.cpu().numpy(), wx, rtol=1e-5, atol=2e-5)
    np.testing.assert_allclose(results[1][1].cpu().numpy(), wl, rtol=1e-5, atol=2e-4)


def test_dwn_threshold_is_inclusive_and_exact_at_half():
    ops = _ops()
    x = np.array([[0.5, 0.49999997, 0.50000006, 0.0, 1.0, -3.0]], dtype=np.float32)
    idx = np.arange(6)[None]
    luts = np.arange(64, dtype=np.float32)[None, None]
    plan = ops.MappingPlan(dev(idx, torch.int32), 6)
    y = ops.DWNLayerFunction.apply(dev(x), dev(luts), plan, 0.1, 0.3)
    assert y.item() == float(0b010101)


@pytest.mark.parametrize("beta", [0.0, 1.0, 0.9])
def test_dwn_backward_other_alpha_beta(beta):
    ops = _ops()
    shape = (33, 20, 17, 4, 2)
    x, idx, luts, gy = make_case(5, *shape)
    B, I, N, k, O = shape
    plan = ops.MappingPlan(dev(idx, torch.int32), I)
    xt = dev(x).requires_grad_(); lt = dev(luts).requires_grad_()
    ops.DWNLayerFunction.apply(xt, lt, plan, 0.7, beta).backward(dev(gy.reshape(B, -1)))
    gx, gl = orc.dwn_layer_backward(x, idx, luts, gy, np.float32(0.7), np.float32(beta))
    np.testing.assert_allclose(xt.grad.cpu().numpy(), gx, rtol=1e-5, atol=1e-5)
    np.testing.assert_allclose(lt.grad.cpu().numpy(), gl, rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("beta", [1.0 / 3.0, -0.5, 0.9])
@pytest.mark.parametrize("shape", [(70, 40, 25, 8, 1), (33, 24, 9, 7, 2), (20, 64, 5, 10, 1)])
def test_dwn_backward_more_than_six_inputs(shape, beta):
    """k > 6: the input gradient from tables smoothed once per call (|beta| <= 1/2) and from the 2^k-term sum
    (beta = 0.9), both against the oracle; the smoothed form amplifies rounding by (1 + |beta|)^k / (1 - beta) <= 52,
    hence rtol 1e-5 with a floor of 2e-5."""
    ops = _ops()
    B, I, N, k, O = shape
    x, idx, luts, gy = make_case(sum(shape), *shape)
    plan = ops.MappingPlan(dev(idx, torch.int32), I)
    xt = dev(x).requires_grad_(); lt = dev(luts).requires_grad_()
    y = ops.DWNLayerFunction.apply(xt, lt, plan, 0.3, beta)
    assert np.array_equal(y.detach().cpu().numpy().reshape(B, N, O), orc.dwn_layer_forward(x, idx, luts))
    y.backward(dev(gy.reshape(B, -1)))
    gx, gl = orc.dwn_layer_backward(x, idx, luts, gy, np.float32(0.3), np.float32(beta))
    np.testing.assert_allclose(xt.grad.cpu().numpy(), gx, rtol=1e-5, atol=2e-5 * max(1.0, float(np.abs(gx).max())))
    np.testing.assert_allclose(lt.grad.cpu().numpy(), gl, rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("k", [7, 8])
@pytest.mark.parametrize("B,I,N,O", [(64, 128, 64, 1),    # whole tiles
                                     (65, 131, 65, 2),    # one past a batch tile and a column tile
                                     (1000, 48, 140, 1),  # lists of about 20 entries per input; several chunks of tiles
                                     (130, 700, 129, 1)])
def test_dwn_tables_of_more_than_one_register(B, I, N, O, k):
    """k = 7 and 8: EFD with small and large |beta| (two ways to build the coefficient rows) and the gradient-stabilised
    node, against the oracle; and the forward without a workspace leaves the same addresses.  Coefficients are built in double
    and rounded once: rtol 1e-5 with a floor of 1e-6 of the largest gradient."""
    ops = _ops()
    from difflut_amd import _native as nat
    x, idx, luts, gy = make_case(B + I + N + k, B, I, N, k, O)
    plan = ops.MappingPlan(dev(idx, torch.int32), I)
    want = orc.dwn_layer_forward(x, idx, luts)
    for beta in (1.0 / 3.0, 0.9):
        xt = dev(x).requires_grad_(); lt = dev(luts).requires_grad_()
        y = ops.DWNLayerFunction.apply(xt, lt, plan, 0.3, beta)
        assert np.array_equal(y.detach().cpu().numpy().reshape(B, N, O), want)
        y.backward(dev(gy.reshape(B, -1)))
        gx, gl = orc.dwn_layer_backward(x, idx, luts, gy, np.float32(0.3), np.float32(beta))
        np.testing.assert_allclose(xt.grad.cpu().numpy(), gx, rtol=1e-5, atol=1e-6 * float(np.abs(gx).max()))
        np.testing.assert_allclose(lt.grad.cpu().numpy(), gl, rtol=1e-5, atol=1e-5)
    scale = np.linspace(0.5, 1.5, N).astype(np.float32)
    xt = dev(x).requires_grad_(); lt = dev(luts).requires_grad_()
    ops.DWNStableLayerFunction.apply(xt, ops.table_sigmoid(lt), dev(scale), plan).backward(dev(gy.reshape(B, -1)))
    gx, gl = orc.stable_layer_backward(x, idx, luts, gy, scale)  # luts as the raw tables
    np.testing.assert_allclose(xt.grad.cpu().numpy(), gx, rtol=1e-5, atol=1e-6 * float(np.abs(gx).max()))
    np.testing.assert_allclose(lt.grad.cpu().numpy(), gl, rtol=1e-5, atol=1e-5)
    lib, dims = nat.lib(), (B, I, N, k, O)
    xd, ld, bt = dev(x), dev(luts), (B + 63) // 64
    saved = torch.empty(2, lib.dl_dwn_saved_bytes(*dims), dtype=torch.uint8, device="cuda")
    ws = torch.empty(lib.dl_dwn_fwd_workspace_bytes(*dims), dtype=torch.uint8, device="cuda")
    y = torch.empty(B, N * O, device="cuda")
    for q, w in enumerate((ws, None)):
        nat.check(lib.dl_dwn_layer_fwd(nat.ptr(xd), nat.ptr(plan.idx32), nat.ptr(ld), nat.ptr(y), nat.ptr(saved[q]), nat.ptr(w),
                                       0 if w is None else w.numel(), *dims, nat.stream()))
        assert np.array_equal(y.cpu().numpy().reshape(B, N, O), want)
    got = saved[:, :bt * N * 64].view(2, bt, N, 64).permute(0, 1, 3, 2).reshape(2, bt * 64, N)[:, :B]
    assert torch.equal(got[0], got[1])


@pytest.mark.parametrize("k", [6, 7, 8])
@pytest.mark.parametrize("stable", [False, True])
def test_dwn_forward_keeps_addresses_instead_of_x(k, stable):
    """Between forward and backward a layer whose backward reads the saved addresses does not hold x."""
    ops = _ops()
    B, I, N = 256, 4096, 32
    g = torch.Generator("cuda").manual_seed(k)
    plan = ops.MappingPlan(torch.randint(0, I, (N, k), device="cuda", generator=g), I)
    luts = torch.rand(N, 1, 1 << k, device="cuda", generator=g).requires_grad_()
    leaf = torch.rand(B, I, device="cuda", generator=g).requires_grad_()
    scale = torch.ones(N, device="cuda")
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    x = leaf * 1.0
    y = ops.dwn_stable_layer(x, luts, scale, plan) if stable else ops.DWNLayerFunction.apply(x, luts, plan, 0.3, 1.0 / 3.0)
    del x
    assert torch.cuda.memory_allocated() - before < 2 * B * I
    y.sum().backward()
    assert torch.isfinite(leaf.grad).all() and leaf.grad.abs().max() > 0


def test_dwn_layer_of_more_nodes_than_the_lane_kernels_number():
    """2^23 nodes: the general kernels, whose backward reads x.  Sums of 2048 fp32 terms of either sign."""
    ops = _ops()
    B, I, N = 2, 4096, 1 << 23
    g = torch.Generator("cuda").manual_seed(8)
    idx = torch.randint(0, I, (N, 1), device="cuda", generator=g, dtype=torch.int32)
    x = torch.rand(B, I, device="cuda", generator=g).requires_grad_()
    luts = (torch.rand(N, 1, 2, device="cuda", generator=g) * 2 - 1).requires_grad_()
    gy = torch.randn(B, N, device="cuda", generator=g)
    y = ops.DWNLayerFunction.apply(x, luts, ops.MappingPlan(idx, I), 0.3, 0.25)
    y.backward(gy)
    col = idx[:, 0].long()
    addr = (x.detach()[:, col] >= 0.5).long()
    table = luts.detach()[:, 0]
    assert torch.equal(y, torch.gather(table.expand(B, N, 2), 2, addr[..., None])[..., 0])
    assert torch.equal(luts.grad[:, 0], sum(torch.nn.functional.one_hot(addr[b], 2) * gy[b][:, None] for b in range(B)))
    terms = 0.3 * gy.double() * (table[:, 1] - table[:, 0]).double()
    want, size = (torch.zeros(B, I, dtype=torch.float64, device="cuda").index_add_(1, col, t) for t in (terms, terms.abs()))
    assert float(((x.grad.double() - want).abs() / size).max()) <= 64 * 2.0 ** -24


def test_dwn_no_input_grad_and_unused_inputs():
    ops = _ops()
    B, I, N, k, O = 40, 50, 3, 2, 1  # 44 of the 50 inputs feed no node: their gradient must be 0
    x, idx, luts, gy = make_case(11, B, I, N, k, O)
    plan = ops.MappingPlan(dev(idx, torch.int32), I)
    lt = dev(luts).requires_grad_()
    ops.DWNLayerFunction.apply(dev(x), lt, plan, 0.2, 0.3).backward(dev(gy.reshape(B, -1)))
    _, gl = orc.dwn_layer_backward(x, idx, luts, gy, np.float32(0.2), np.float32(0.3))
    np.testing.assert_allclose(lt.grad.cpu().numpy(), gl, rtol=1e-5, atol=1e-5)
    xt = dev(x).requires_grad_()
    ops.DWNLayerFunction.apply(xt, dev(luts), plan, 0.2, 0.3).backward(dev(gy.reshape(B, -1)))
    unused = np.setdiff1d(np.arange(I), idx.reshape(-1))
    assert np.all(xt.grad.cpu().numpy()[:, unused] == 0.0)


@pytest.mark.parametrize("shape", [(12, 20, 9, 6, 2), (70, 33, 140, 3, 1), (4, 30, 5, 8, 1)])
def test_dwn_eval_forward(shape):
    ops = _ops()
    B, I, N, k, O = shape
    x, idx, luts, _ = make_case(3, *shape, lo=0.0, hi=1.0, binary=True)
    plan = ops.MappingPlan(dev(idx, torch.int32), I)
    y = ops.dwn_layer_eval(dev(x), dev(luts), plan).cpu().numpy().reshape(B, N, O)
    m = orc.gather_forward(x, idx)
    for n in range(N):
        assert np.array_equal(y[:, n], orc.dwn_eval_forward(m[:, n], luts[n]))


@pytest.mark.parametrize("shape", [(130, 40, 150, 6, 1), (64, 36, 70, 4, 2), (257, 33, 129, 5, 1),
                                   # from 1024 columns on the literal-address kernel stages the row of x in the LDS:
                                   # odd widths, two outputs per node, two windows of columns
                                   (37, 1031, 1100, 5, 1), (5, 300, 600, 3, 2), (9, 4096, 9000, 6, 1)])
def test_dwn_eval_forward_any_input_values(shape):
    """The eval entry point with a workspace answers through the bit-plane kernels when every input is 0 or 1 and
    through the literal float address otherwise; both against the oracle, including inputs where the two
    addresses differ (0.7 counts as 0.7 * 2^j, not as a set bit) and a single odd value in a binary batch."""
    ops = _ops()
    B, I, N, k, O = shape
    xb, idx, luts, _ = make_case(11, *shape, lo=0.0, hi=1.0, binary=True)
    rng = np.random.default_rng(5)
    xf = rng.random((B, I)).astype(np.float32) * 1.2          # arbitrary values, some above 1
    xo = xb.copy()
    xo[B // 2, idx[N // 2, 0]] = 0.25                          # one value that is neither 0 nor 1
    plan = ops.MappingPlan(dev(idx, torch.int32), I)
    for x in (xb, xf, xo, xb):                                 # the flag is reset on every call
        y = ops.dwn_layer_eval(dev(x), dev(luts), plan).cpu().numpy().reshape(B, N, O)
        m = orc.gather_forward(x, idx)
        L = 1 << k
        for n in range(N):
            addr = (m[:, n] * (2.0 ** np.arange(k)).astype(np.float32)).sum(-1, dtype=np.float32).astype(np.int64)
            want = (luts[n][:, np.clip(addr, 0, L - 1)].T >= np.float32(0.5)).astype(np.float32)  # clamped like the kernel
            assert np.array_equal(y[:, n], want)
            if x is not xf:
                assert np.array_equal(want, orc.dwn_eval_forward(m[:, n], luts[n]))


@pytest.mark.parametrize("shape", [(130, 40, 150, 4, 1), (64, 36, 70, 6, 2), (200, 33, 90, 3, 1),
                                   # from 1024 columns on both literal-address kernels stage the row of x in the LDS
                                   (33, 1031, 1100, 4, 1), (7, 300, 520, 6, 2)])
def test_prob_eval_forward_any_input_values(shape):
    """Probabilistic eval through the workspace entry point (binarised sigmoid table looked up by the DWN eval
    path) against the oracle, for 0/1 inputs (bit-plane kernels), arbitrary inputs and a single odd value
    (generic kernel), and against the entry point without a workspace."""
    from difflut_amd import _native as nat
    ops = _ops()
    B, I, N, k, O = shape
    rng = np.random.default_rng(21)
    idx = orc.random_mapping(I, N, k, seed=4).numpy().astype(np.int64)
    raw = rng.standard_normal((N, 1 << k, O)).astype(np.float32)
    raw[0, 0, 0] = 0.0                                         # sigmoid(0) = 0.5 counts as 1
    xb = rng.integers(0, 2, (B, I)).astype(np.float32)
    xf = rng.random((B, I)).astype(np.float32)
    xo = xb.copy()
    xo[3, idx[1, 0]] = 0.5
    plan = ops.MappingPlan(dev(idx, torch.int32), I)
    lib = nat.lib()
    rawd = dev(raw)
    for x in (xb, xf, xo):
        xd = dev(x)
        y = ops.prob_layer_eval(xd, rawd, plan, 0.7)
        plain = torch.empty_like(y)
        nat.check(lib.dl_prob_layer_eval(xd.data_ptr(), plan.idx32.data_ptr(), rawd.data_ptr(), 0.7, plain.data_ptr(),
                                         B, I, N, k, O, nat.stream()))
        assert torch.equal(y, plain)
        m = orc.gather_forward(x, idx)
        got = y.cpu().numpy().reshape(B, N, O)
        for n in range(N):
            assert np.array_equal(got[:, n], orc.prob_eval_forward(m[:, n], raw[n], 0.7))


@pytest.mark.parametrize("tag", ["k6o2", "k4o1", "k2o3"])
def test_dwn_node_against_reference_vectors(golden, tag):
    """Same inputs the reference's own CPU path was run on (tests/golden)."""
    from difflut_amd.nodes.dwn_node import efd_forward

    g = golden
    a, b = (float(v) for v in g[f"dwn_{tag}_ab"])
    xt = dev(g[f"dwn_{tag}_x"]).requires_grad_()
    lt = dev(g[f"dwn_{tag}_luts"]).requires_grad_()
    y = efd_forward(xt, lt, a, b)
    assert np.array_equal(y.detach().cpu().numpy(), g[f"dwn_{tag}_y"])
    y.backward(dev(g[f"dwn_{tag}_gy"]))
    np.testing.assert_allclose(xt.grad.cpu().numpy(), g[f"dwn_{tag}_gx"], rtol=1e-5, atol=2e-6)
    np.testing.assert_allclose(lt.grad.cpu().numpy(), g[f"dwn_{tag}_gl"], rtol=1e-5, atol=1e-6)


# ------------------------------------------------------------------------------ gather
@pytest.mark.parametrize("dtype", [torch.int16, torch.int32])
def test_gather_forward_backward(dtype):
    ops = _ops()
    B, I, N, k = 37, 211, 90, 5
    rng = np.random.default_rng(0)
    x = rng.standard_normal((B, I)).astype(np.float32)
    idx = orc.random_mapping(I, N, k, seed=9).numpy().astype(np.int64)
    it = dev(idx, dtype)
    xt = dev(x).requires_grad_()
    m = ops.GatherFunction.apply(xt, it, ops.MappingPlan(it, I))
    assert np.array_equal(m.detach().cpu().numpy(), orc.gather_forward(x, idx))
    gm = rng.standard_normal((B, N, k)).astype(np.float32)
    m.backward(dev(gm))
    np.testing.assert_allclose(xt.grad.cpu().numpy(), orc.gather_backward(gm, idx, I), rtol=1e-6, atol=1e-6)


@pytest.mark.parametrize("shape", [(70, 1031, 700, 6, torch.int16),      # 4200 connections: one piece, odd widths (scalar staging)
                                   (33, 3136, 2000, 6, torch.int16),     # cfg 1's layer: lists of three and four
                                   (25, 4096, 4096, 4, torch.int32),     # whole permutations, four inputs per thread
                                   (9, 16384, 8192, 6, torch.int32),     # two pieces per row, sixteen inputs per thread
                                   (5, 20001, 9000, 5, torch.int32),     # two windows of inputs, pieces of odd length
                                   (3, 300, 48000, 1, torch.int32)])     # hard selection's shape: long lists, one input each
def test_gather_through_the_lds(shape):
    """From 4096 connections on the row that is read at random (x forward, gm backward) is staged in the LDS.  The
    forward is a copy: exact.  The backward adds a list in its order, like the oracle's loop: exact as well."""
    ops = _ops()
    B, I, N, k, dtype = shape
    rng = np.random.default_rng(I + N)
    x = rng.standard_normal((B, I)).astype(np.float32)
    idx = orc.random_mapping(I, N, k, seed=5).numpy().astype(np.int64)
    it = dev(idx, dtype)
    xt = dev(x).requires_grad_()
    m = ops.GatherFunction.apply(xt, it, ops.MappingPlan(it, I))
    assert np.array_equal(m.detach().cpu().numpy(), x[:, idx])
    gm = rng.standard_normal((B, N, k)).astype(np.float32)
    m.backward(dev(gm))
    want = np.zeros((B, I), np.float32)
    flat = gm.reshape(B, -1)
    for p, i in enumerate(idx.reshape(-1)):  # ascending position within every input: the order of the CSR lists
        want[:, i] += flat[:, p]
    assert np.array_equal(xt.grad.cpu().numpy(), want)


@pytest.mark.parametrize("B", [1, 7, 8, 9, 63, 64, 65, 200])
@pytest.mark.parametrize("source", ["code", "x", "planes"])
@pytest.mark.parametrize("width,N,k,O,groups", [(40, 192, 6, 1, 3),    # groups of one wavefront
                                                (33, 65, 1, 1, 1),     # a group one column longer
                                                (96, 330, 4, 2, 9),    # groups of 74 columns, the last of 68, two outputs
                                                (2100, 1300, 5, 1, 1)])  # more columns than a block's threads
def test_eval_of_few_rows(B, source, width, N, k, O, groups):
    """One launch per layer against the bit-plane kernels: the same bits, as planes and as group sums; and the group sums from
    planes against the sums of the layer's output.  Sums of zeros and ones: exact."""
    from difflut_amd import _native as nat

    lib = nat.lib()
    g = torch.Generator("cuda").manual_seed(B + width)
    nbits = 3 if source == "code" else 1
    I, F = width * nbits, N * O
    idx = torch.randint(0, I, (N, k), device=DEV, generator=g, dtype=torch.int32)
    luts = torch.randn(N, O, 1 << k, device=DEV, generator=g)
    luts[0] = 0.5
    x = torch.rand(B, width, device=DEV, generator=g)
    thr = torch.rand(width, nbits, device=DEV, generator=g)
    x[0, 0] = thr[0, 0]  # not greater
    if source != "code":
        x = (x < 0.5).float()
    planes = torch.empty(lib.dl_dwn_planes_bytes(B, I), dtype=torch.uint8, device=DEV)
    if source == "code":
        nat.check(lib.dl_thermometer_planes(x.data_ptr(), thr.data_ptr(), planes.data_ptr(), B, width, nbits, nat.stream()))
    else:
        nat.check(lib.dl_dwn_pack_planes(x.data_ptr(), planes.data_ptr(), B, I, nat.stream()))
    dims = (B, I, N, k, O)
    y = torch.empty(B, F, device=DEV)
    used = (B + 63) // 64 * F * 8
    want, got = (torch.full((max(used, 256),), 7, dtype=torch.uint8, device=DEV) for _ in range(2))
    nat.check(lib.dl_dwn_layer_eval_planes(planes.data_ptr(), idx.data_ptr(), luts.data_ptr(), y.data_ptr(), want.data_ptr(), *dims, nat.stream()))
    given = (None, None, 1, planes.data_ptr()) if source == "planes" else (x.data_ptr(), thr.data_ptr() if source == "code" else None, nbits, None)
    nat.check(lib.dl_dwn_layer_rows(*given, idx.data_ptr(), luts.data_ptr(), got.data_ptr(), None, None, *dims, 0, 1.0, nat.stream()))
    assert torch.equal(want[:used], got[:used])
    gs = -(-F // groups)
    sums = torch.stack([y[:, q * gs:(q + 1) * gs].sum(1) for q in range(groups)], 1) * (1.0 / 0.5)
    logits = torch.full((2, B, groups), -1.0, device=DEV)
    nat.check(lib.dl_dwn_layer_rows(*given, idx.data_ptr(), luts.data_ptr(), None, logits[0].data_ptr(), None, *dims, groups, 0.5, nat.stream()))
    ws = torch.empty(lib.dl_dwn_groups_workspace_bytes(B, N, O, groups), dtype=torch.uint8, device=DEV)
    nat.check(lib.dl_dwn_layer_eval_planes_groups(planes.data_ptr(), idx.data_ptr(), luts.data_ptr(), logits[1].data_ptr(), ws.data_ptr(),
                                                  ws.numel(), *dims, groups, 0.5, nat.stream()))
    assert torch.equal(logits[0], sums) and torch.equal(logits[1], sums)
    # the training forward: planes and addresses the same (rows that the batch does not have are zeros); sums of up to 1300 values
    # of size 1 in another order
    saved = torch.full((2, lib.dl_dwn_saved_bytes(*dims)), 7, dtype=torch.uint8, device=DEV)
    nat.check(lib.dl_dwn_layer_fwd_planes(planes.data_ptr(), idx.data_ptr(), luts.data_ptr(), None, want.data_ptr(), saved[0].data_ptr(), *dims, nat.stream()))
    nat.check(lib.dl_dwn_layer_rows(*given, idx.data_ptr(), luts.data_ptr(), got.data_ptr(), None, saved[1].data_ptr(), *dims, 0, 1.0, nat.stream()))
    held = (B + 63) // 64 * N * 64
    assert torch.equal(want[:used], got[:used]) and torch.equal(saved[0][:held], saved[1][:held])
    nat.check(lib.dl_dwn_layer_fwd_planes_groups(planes.data_ptr(), idx.data_ptr(), luts.data_ptr(), logits[0].data_ptr(), saved[0].data_ptr(),
                                                 ws.data_ptr(), ws.numel(), *dims, groups, 0.5, nat.stream()))
    saved[1] = 7
    nat.check(lib.dl_dwn_layer_rows(*given, idx.data_ptr(), luts.data_ptr(), None, logits[1].data_ptr(), saved[1].data_ptr(), *dims, groups, 0.5, nat.stream()))
    assert torch.equal(saved[0][:held], saved[1][:held])
    torch.testing.assert_close(logits[0], logits[1], rtol=1e-5, atol=1e-4)


def _kernels_of(call):
    """The library kernels that `call` launches, from the library's record."""
    from difflut_amd import _native as nat

    nat.profile_read()
    nat.profile_enable(True)
    try:
        call()
        return [name for name, _ in nat.profile_read()]
    finally:
        nat.profile_enable(False)


@pytest.mark.parametrize("B,N,k,O,groups,kernel", [
    (300, 2560, 6, 1, 10, "dwn_eval_groups"),    # 256 columns a group
    (100, 2570, 6, 1, 10, "dwn_lookup_eval"),    # 257: a pass of more wavefronts
    (4000, 2570, 4, 1, 10, "dwn_eval_groups"),
    (1100, 4000, 3, 1, 1, "dwn_lookup_eval"),    # eight passes of one block per tile
    (9000, 2000, 2, 2, 2, "dwn_eval_groups"),    # four passes, many tiles
    (1024, 1500, 5, 2, 2, "dwn_lookup_eval")])
def test_eval_heads_of_wide_groups(B, N, k, O, groups, kernel):
    """Bit-sliced, or by the lookup where a wide group would keep few blocks busy for many passes: whole numbers, exact."""
    from difflut_amd import _native as nat

    lib = nat.lib()
    g = torch.Generator("cuda").manual_seed(B + N)
    I, F = 500, N * O
    idx = torch.randint(0, I, (N, k), device=DEV, generator=g, dtype=torch.int32)
    luts = torch.randn(N, O, 1 << k, device=DEV, generator=g)
    x = (torch.rand(B, I, device=DEV, generator=g) < 0.5).float()
    planes = torch.empty(lib.dl_dwn_planes_bytes(B, I), dtype=torch.uint8, device=DEV)
    nat.check(lib.dl_dwn_pack_planes(x.data_ptr(), planes.data_ptr(), B, I, nat.stream()))
    y = torch.empty(B, F, device=DEV)
    nat.check(lib.dl_dwn_layer_eval_planes(planes.data_ptr(), idx.data_ptr(), luts.data_ptr(), y.data_ptr(), None, B, I, N, k, O, nat.stream()))
    logits = torch.full((B, groups), -1.0, device=DEV)
    need = lib.dl_dwn_eval_groups_workspace_bytes(B, N, O, groups)
    assert (need == 0) == (kernel == "dwn_eval_groups")  # which writes the logits itself
    ws = torch.empty(need, dtype=torch.uint8, device=DEV) if need else None
    ran = _kernels_of(lambda: nat.check(lib.dl_dwn_layer_eval_planes_groups(
        planes.data_ptr(), idx.data_ptr(), luts.data_ptr(), logits.data_ptr(), nat.ptr(ws), need, B, I, N, k, O, groups, 0.5, nat.stream())))
    assert ran == ([kernel] if kernel == "dwn_eval_groups" else [kernel, "dwn_group_finish"])
    assert torch.equal(logits, y.view(B, groups, F // groups).sum(2) * 2.0)


@pytest.mark.parametrize("train", [False, True])
@pytest.mark.parametrize("B,features,bits,widths,groups,first,launches", [
    (100, 784, 4, (2000,), 10, "dwn_rows", 1),
    (768, 6000, 1, (1000,), 10, "dwn_pack_planes", 1),       # every group's blocks would turn the whole input
    (64, 6000, 8, (1000,), 10, "thermometer_planes", 1),     # 48 000 inputs
    (64, 300, 1, (4000,), 1, "dwn_rows", 1),                 # four passes of a block
    (5, 83, 3, (4779,), 3, "dwn_rows", 1),                   # two, in inference a row at a time
    (768, 3000, 1, (8000,), 10, "dwn_pack_planes", 0),       # 960 blocks that read 23 million values, 6 million outputs
    (200, 784, 4, (3000, 2000, 1000), 10, "dwn_rows", 2),    # not the hidden layer
    (200, 784, 4, (3000, 380, 1000), 10, "dwn_rows", 3),
    (77, 6000, 8, (300, 200, 100), 0, "thermometer_planes", 2),
    (200, 784, 4, (3000, 2000), 0, "dwn_rows", 1),
    (520, 3000, 1, (4000, 3000), 2, "dwn_pack_planes", 0)])  # 260 blocks
def test_few_rows_of_a_chain_layer_by_layer(B, features, bits, widths, groups, first, launches, train):
    """A launch per layer (dwn_rows) where that is the better one, layer by layer, and the results of the plane kernels: exact in
    inference; in training a group's sum has up to 4000 values of size 1, added in another order."""
    from difflut_amd import _native as nat
    from difflut_amd import ops

    g = torch.Generator("cuda").manual_seed(B + features)
    x = torch.rand(B, features, device=DEV, generator=g)
    thr = torch.rand(features, bits, device=DEV, generator=g).sort(1)[0].contiguous() if bits > 1 else None
    plans, luts, width = [], [], features * bits
    for n in widths:
        plans.append(ops.MappingPlan(torch.randint(0, width, (n, 6), device=DEV, generator=g), width))
        luts.append(torch.rand(n, 1, 64, device=DEV, generator=g) * 2 - 1)
        width = n
    got, hosts = [], [p.host for p in plans]
    if train:
        scalars = [(None, None, 0.1, 1 / 3)] * len(luts)
        ran = _kernels_of(lambda: got.append(nat.host().dwn_stack(x, luts, hosts, scalars, thr, [], None, groups, 1.0)))
    else:
        ran = _kernels_of(lambda: got.append(nat.host().dwn_stack_eval(x, thr, luts, hosts, groups, 1.0)))
    assert ran[0] == first and ran.count("dwn_rows") == launches
    bits_in = (x[:, :, None] > thr[None] if thr is not None else x >= 0.5).view(B, -1)
    for l, (plan, table) in enumerate(zip(plans, luts)):
        addr = (bits_in[:, plan.idx32.long()].long() << torch.arange(6, device=DEV)).sum(2)
        y = torch.gather(table[:, 0].expand(B, -1, -1), 2, addr[:, :, None])[:, :, 0]
        bits_in = y >= 0.5
    out = y if train else bits_in.float()
    if groups:
        out = out.double().view(B, groups, -1).sum(2).float()
    if train and groups:
        torch.testing.assert_close(got[0], out, rtol=1e-5, atol=1e-3)
    else:
        assert torch.equal(got[0], out)


@pytest.mark.parametrize("B", [1, 8, 65, 130])
@pytest.mark.parametrize("I,N,k,O", [(64, 64, 6, 1), (100, 33, 3, 2), (8192, 1100, 4, 1), (8193, 40, 5, 1)])  # the last: planes
def test_layer_forward_of_few_rows(B, I, N, k, O):
    """A single layer on few rows, one launch: output and addresses those of the bit-plane kernels."""
    from difflut_amd import _native as nat

    lib = nat.lib()
    g = torch.Generator("cuda").manual_seed(B + I)
    idx = torch.randint(0, I, (N, k), device=DEV, generator=g, dtype=torch.int32)
    luts = torch.randn(N, O, 1 << k, device=DEV, generator=g)
    x = torch.rand(B, I, device=DEV, generator=g)
    x[0, :4] = torch.tensor([0.5, float("nan"), float("inf"), -0.0], device=DEV)
    dims = (B, I, N, k, O)
    planes = torch.empty(lib.dl_dwn_planes_bytes(B, I), dtype=torch.uint8, device=DEV)
    y = torch.full((2, B, N * O), -7.0, device=DEV)
    saved = torch.full((2, lib.dl_dwn_saved_bytes(*dims)), 7, dtype=torch.uint8, device=DEV)
    nat.check(lib.dl_dwn_pack_planes(x.data_ptr(), planes.data_ptr(), B, I, nat.stream()))
    nat.check(lib.dl_dwn_layer_fwd_planes(planes.data_ptr(), idx.data_ptr(), luts.data_ptr(), y[0].data_ptr(), None, saved[0].data_ptr(), *dims, nat.stream()))
    ws = torch.empty(lib.dl_dwn_fwd_workspace_bytes(*dims), dtype=torch.uint8, device=DEV)
    nat.check(lib.dl_dwn_layer_fwd(x.data_ptr(), idx.data_ptr(), luts.data_ptr(), y[1].data_ptr(), saved[1].data_ptr(), ws.data_ptr(), ws.numel(),
                                   *dims, nat.stream()))
    held = (B + 63) // 64 * N * 64
    assert torch.equal(y[0], y[1]) and torch.equal(saved[0][:held], saved[1][:held])


@pytest.mark.parametrize("k", [7, 8])
@pytest.mark.parametrize("beta", [1 / 3, -0.5, 0.8])  # the compact form of the tables, its edge, the other one
@pytest.mark.parametrize("B,N,O", [(65, 5, 1), (130, 67, 2)])
def test_wide_coefficient_tables(B, N, O, beta, k):
    """Tables of 128 and 256 entries are built by a wavefront each, beside the histogram.  Floors as for the other gradients: a
    connection's term is a difference of two fp32 roundings of sums of up to 2^(k-1) products of size 1."""
    ops = _ops()
    I = 50
    rng = np.random.default_rng(B + k)
    x = rng.uniform(0, 1, (B, I)).astype(np.float32)
    idx = orc.random_mapping(I, N, k, seed=4).numpy().astype(np.int64)
    luts = rng.uniform(-1, 1, (N, O, 1 << k)).astype(np.float32)
    gy = rng.standard_normal((B, N, O)).astype(np.float32)
    xt, lt = dev(x).requires_grad_(), dev(luts).requires_grad_()
    alpha = 0.4 * 0.75 ** (k - 1)
    y = ops.DWNLayerFunction.apply(xt, lt, ops.MappingPlan(dev(idx, torch.int32), I), alpha, beta)
    y.backward(dev(gy.reshape(B, -1)))
    gx, gl = orc.dwn_layer_backward(x, idx, luts, gy, np.float32(alpha), np.float32(beta))
    scale = float(np.abs(gx).max())
    np.testing.assert_allclose(xt.grad.cpu().numpy(), gx, rtol=1e-5, atol=1e-6 * scale)
    np.testing.assert_allclose(lt.grad.cpu().numpy(), gl, rtol=1e-5, atol=1e-5)


# ------------------------------------------------------------------------------ probabilistic
PROB_SHAPES = [(32, 40, 24, 4, 2), (64, 128, 300, 4, 1), (17, 30, 9, 6, 1), (20, 9, 5, 1, 1), (10, 50, 7, 2, 3),
               (6, 40, 5, 7, 2), (200, 300, 260, 4, 1), (130, 70, 33, 5, 2), (65, 1000, 515, 3, 1),
               (300, 20, 3, 4, 1)]   # last: few nodes, many batch tiles -> several table-gradient chunks


@pytest.mark.parametrize("shape", PROB_SHAPES)
@pytest.mark.parametrize("T", [1.0, 0.5])
def test_prob_layer_forward_backward(shape, T):
    ops = _ops()
    B, I, N, k, O = shape
    rng = np.random.default_rng(sum(shape))
    x = (1 / (1 + np.exp(-rng.standard_normal((B, I))))).astype(np.float32)
    idx = orc.random_mapping(I, N, k, seed=4).numpy().astype(np.int64)
    raw = rng.uniform(0, 1, (N, 1 << k, O)).astype(np.float32)
    gy = rng.standard_normal((B, N, O)).astype(np.float32)
    plan = ops.MappingPlan(dev(idx, torch.int32), I)
    xt = dev(x).requires_grad_(); wt = dev(raw).requires_grad_()
    y = ops.ProbLayerFunction.apply(xt, wt, plan, T)
    want = orc.prob_layer_forward(x, idx, raw, T, dtype=torch.float64).reshape(B, N * O)
    np.testing.assert_allclose(y.detach().cpu().numpy(), want, rtol=1e-5, atol=1e-6)  # outputs lie in (0,1)
    y.backward(dev(gy.reshape(B, -1)))
    gx, gw = orc.prob_layer_backward(x, idx, raw, gy, T)
    np.testing.assert_allclose(xt.grad.cpu().numpy(), gx, rtol=1e-5, atol=2e-6)
    np.testing.assert_allclose(wt.grad.cpu().numpy(), gw, rtol=1e-5, atol=2e-6)


@pytest.mark.parametrize("k", [1, 2, 3, 4, 5, 6])
@pytest.mark.parametrize("B,N,O,T", [(64, 16, 1, 1.0),     # one block of sixteen columns, one batch tile
                                     (321, 17, 1, 0.5),    # a column and a row past that; several chunks of tiles
                                     (1025, 250, 2, 1.0),  # more blocks than fit one per chunk
                                     (130, 4100, 1, 1.0)]) # one chunk
def test_prob_backward_factored_weights(B, N, O, T, k):
    """The product weights factor into those of the lower k / 2 and of the upper inputs, sixteen columns to a block.  The
    gradient of an input with 2^k terms of size |gy| <= 4 rounds to a few 1e-7 of that: rtol 1e-5, floor 5e-6; table
    gradients sum up to 1025 rows: floor 1e-5."""
    ops = _ops()
    I = 37 + N // 3
    rng = np.random.default_rng(B + N + k)
    x = rng.uniform(0, 1, (B, I)).astype(np.float32)
    x[:, 0] = (x[:, 0] > 0.5)  # exact zeros and ones among the inputs
    idx = orc.random_mapping(I, N, k, seed=4).numpy().astype(np.int64)
    raw = rng.uniform(-1, 1, (N, 1 << k, O)).astype(np.float32)
    gy = rng.uniform(-4, 4, (B, N, O)).astype(np.float32)
    plan = ops.MappingPlan(dev(idx, torch.int32), I)
    xt = dev(x).requires_grad_(); wt = dev(raw).requires_grad_()
    ops.ProbLayerFunction.apply(xt, wt, plan, T).backward(dev(gy.reshape(B, -1)))
    gx, gw = orc.prob_layer_backward(x, idx, raw, gy, T)
    np.testing.assert_allclose(xt.grad.cpu().numpy(), gx, rtol=1e-5, atol=5e-6)
    np.testing.assert_allclose(wt.grad.cpu().numpy(), gw, rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("hybrid", [False, True])
def test_prob_input_gradient_rounds_by_what_the_table_varies(hybrid):
    """k = 6, uniform x, tables sigmoid(N(0, 1)): values of 0.5 +- 0.2.  Against float64 in the 2-norm: each weight is a product
    of three factors (3 roundings of 2^-25 rms, 9e-8), sums of eight terms of 0.2 are taken differences of (1e-7), the output
    is a product and a sum (4e-8): 1.4e-7, limit 2.1e-7.  Sums of the table itself, of 0.5, give 3.0e-7 (hybrid 2.2e-7)."""
    ops = _ops()
    B, I, N, k = 1000, 400, 300, 6
    g = torch.Generator("cuda").manual_seed(k)
    idx = torch.stack([torch.randperm(I, device="cuda", generator=g)[:k] for _ in range(N)])
    plan = ops.MappingPlan(idx, I)
    x = torch.rand(B, I, device="cuda", generator=g)
    gy = torch.randn(B, N, device="cuda", generator=g)
    raw = torch.randn(N, 1 << k, device="cuda", generator=g)
    xt = x.clone().requires_grad_()
    table = ops.table_sigmoid(raw) if hybrid else raw
    if hybrid:
        ops.hybrid_layer(xt, table.view(N, 1, 1 << k).clone().requires_grad_(), plan).backward(gy)
    else:
        ops.ProbLayerFunction.apply(xt, raw.view(N, 1 << k, 1).clone().requires_grad_(), plan, 1.0).backward(gy)
    cols = [x.double()[:, idx[:, j]].requires_grad_() for j in range(k)]
    v = (table if hybrid else torch.sigmoid(raw.double())).double().expand(B, N, 1 << k)
    for c in cols:
        v = v[..., 0::2] * (1 - c.unsqueeze(-1)) + v[..., 1::2] * c.unsqueeze(-1)
    v.squeeze(-1).backward(gy.double())
    want = torch.zeros(B, I, dtype=torch.float64, device="cuda")
    for j, c in enumerate(cols):
        q = c.detach() * (1 - c.detach())
        want.index_add_(1, idx[:, j], c.grad * q / (q + 1e-8) if hybrid else c.grad)
    assert float((xt.grad.double() - want).norm()) <= 2.1e-7 * float(want.norm())


@pytest.mark.parametrize("k", [1, 4, 6])
@pytest.mark.parametrize("hybrid", [False, True])
@pytest.mark.parametrize("B,N,O", [(63, 1, 1), (5000, 1, 1),    # one column
                                   (700, 3, 2), (700, 6, 2),   # blocks of four columns, the last half empty; their largest
                                   (700, 13, 1),               # one column more: blocks of sixteen
                                   (4160, 32, 1), (4161, 5, 1)])  # many chunks, a tile each and with a last one
def test_prob_backward_of_few_columns(B, N, O, hybrid, k):
    """Few columns over many rows: blocks of four columns, chunks down to one batch tile.  Floors as in
    test_prob_backward_factored_weights; table gradients sum up to 5000 rows of size 4, about sqrt(5000) * 4 * 6e-8: floor 2e-5."""
    ops = _ops()
    I = 11
    rng = np.random.default_rng(B + N + k)
    x = rng.uniform(0, 1, (B, I)).astype(np.float32)
    idx = orc.random_mapping(I, N, k, seed=4).numpy().astype(np.int64)
    gy = rng.uniform(-4, 4, (B, N, O)).astype(np.float32)
    plan = ops.MappingPlan(dev(idx, torch.int32), I)
    xt = dev(x).requires_grad_()
    if hybrid:
        raw = rng.uniform(-1, 1, (N, O, 1 << k)).astype(np.float32)
        wt = dev(raw).requires_grad_()
        ops.hybrid_layer(xt, ops.table_sigmoid(wt), plan).backward(dev(gy.reshape(B, -1)))
        gx, gw = orc.hybrid_layer_backward(x, idx, raw, gy)
    else:
        raw = rng.uniform(-1, 1, (N, 1 << k, O)).astype(np.float32)
        wt = dev(raw).requires_grad_()
        ops.ProbLayerFunction.apply(xt, wt, plan, 1.0).backward(dev(gy.reshape(B, -1)))
        gx, gw = orc.prob_layer_backward(x, idx, raw, gy, 1.0)
    np.testing.assert_allclose(xt.grad.cpu().numpy(), gx, rtol=1e-5, atol=5e-6)
    np.testing.assert_allclose(wt.grad.cpu().numpy(), gw, rtol=1e-5, atol=2e-5)


@pytest.mark.parametrize("k", [1, 2, 3, 4, 5, 6])
@pytest.mark.parametrize("B,N,offset", [(64, 16, 0),     # one block, one batch tile
                                        (1, 13, 0),      # one row, a block that is not full
                                        (65, 17, 0), (65, 18, 2), (200, 20, 1),  # a row and columns past that; x off 16 and off 8 bytes
                                        (129, 4112, 0),  # one chunk of tiles: no partial sums
                                        (1500, 33, 0)])  # several chunks
def test_prob_nodes_in_order(B, N, offset, k):
    """Nodes that take their inputs in order: the same sums in the same order as through an index table that says so, which the
    oracle checks in the tests above, so the tolerance is that of a differently contracted multiply-add: a few units of the last place."""
    ops = _ops()
    g = torch.Generator("cuda").manual_seed(B + N + k)
    M = N * k
    x = torch.rand(B * M + offset, device="cuda", generator=g)[offset:].view(B, M)
    x[:, 0] = (x[:, 0] > 0.5).float()
    raw = torch.randn(N, 1 << k, 1, device="cuda", generator=g)
    gy = torch.randn(B, N, device="cuda", generator=g)
    T = torch.rand(N, device="cuda", generator=g) + 0.5
    general = ops.MappingPlan(torch.arange(M, device="cuda", dtype=torch.int32).view(N, k), M)
    ordered = ops.MappingPlan.in_order(N, k, x.device)
    for name in ("idx32", "inv_ptr", "inv_pos"):
        assert torch.equal(getattr(general, name), getattr(ordered, name)) and getattr(general, name).dtype == getattr(ordered, name).dtype
    assert ordered.ordered and not general.ordered and general.I == ordered.I
    for temperature in (T, 0.7):
        got = []
        for plan in (general, ordered):
            xt, wt = x.detach().requires_grad_(), raw.clone().requires_grad_()
            y = ops.ProbLayerFunction.apply(xt, wt, plan, temperature)
            y.backward(gy)
            w2 = raw.clone().requires_grad_()  # the tables alone
            ops.ProbLayerFunction.apply(x, w2, plan, temperature).backward(gy)
            assert torch.equal(w2.grad, wt.grad)
            got.append((y.detach(), xt.grad, wt.grad))
        for a, b, floor in zip(*got, (5e-7, 2e-6, 2e-6 * B ** 0.5)):
            torch.testing.assert_close(a, b, rtol=1e-6, atol=floor)


@pytest.mark.parametrize("tag", ["k4o2", "k6o1"])
def test_prob_node_against_reference_vectors(golden, tag):
    from difflut_amd.nodes.probabilistic_node import probabilistic_forward
    ops = _ops()

    g = golden
    T = float(g[f"prob_{tag}_T"][0])
    xt = dev(g[f"prob_{tag}_x"]).requires_grad_()
    wt = dev(g[f"prob_{tag}_w"]).requires_grad_()
    y = probabilistic_forward(xt, wt, T)
    np.testing.assert_allclose(y.detach().cpu().numpy(), g[f"prob_{tag}_y"], rtol=1e-5, atol=1e-6)
    y.backward(dev(g[f"prob_{tag}_gy"]))
    np.testing.assert_allclose(xt.grad.cpu().numpy(), g[f"prob_{tag}_gx"], rtol=1e-5, atol=2e-6)
    np.testing.assert_allclose(wt.grad.cpu().numpy(), g[f"prob_{tag}_gw"], rtol=1e-5, atol=2e-6)
    k = g[f"prob_{tag}_x"].shape[1]
    plan = ops.MappingPlan.identity(k, DEV)
    ye = ops.prob_layer_eval(dev(g[f"prob_{tag}_eval_x"]), wt.detach().unsqueeze(0), plan, T)
    assert np.array_equal(ye.cpu().numpy(), g[f"prob_{tag}_eval_y"])


# ------------------------------------------------------------------------------ learnable mapping
@pytest.mark.parametrize("shape,tau", [((5, 20, 21), 1.0), ((70, 130, 200), 0.3), ((64, 64, 64), 1.0),
                                       ((33, 257, 18), 0.05), ((256, 384, 1000), 1.0),
                                       ((130, 260, 516), 0.5), ((129, 132, 4100), 2.0)])
def test_soft_mapping_forward_backward_fp32(shape, tau):
    ops = _ops()
    B, I, M = shape
    rng = np.random.default_rng(sum(shape))
    x = rng.random((B, I)).astype(np.float32)
    W = (rng.standard_normal((M, I)) * 0.5).astype(np.float32)
    gm = rng.standard_normal((B, M)).astype(np.float32)
    xt = dev(x).requires_grad_(); Wt = dev(W).requires_grad_()
    m = ops.SoftMapFunction.apply(xt, Wt, tau, 0)
    np.testing.assert_allclose(m.detach().cpu().numpy(), orc.soft_mapping_forward(x, W, tau, torch.float64),
                               rtol=1e-5, atol=1e-6)  # m is a convex mix of inputs in [0,1)
    m.backward(dev(gm))
    gx, gW = orc.soft_mapping_backward(x, W, gm, tau)
    np.testing.assert_allclose(xt.grad.cpu().numpy(), gx, rtol=1e-4, atol=1e-5)
    np.testing.assert_allclose(Wt.grad.cpu().numpy(), gW, rtol=1e-4, atol=1e-5 / tau)


@pytest.mark.parametrize("shape,tau", [((5, 20, 21), 1.0), ((256, 384, 1000), 1.0), ((130, 260, 516), 0.5),
                                       ((129, 132, 4100), 2.0), ((128, 256, 384), 1.0)])
def test_soft_mapping_bf16_operands(shape, tau):
    """precision=1 rounds x, S and gm to bf16 (8 significant bits, relative step 2^-8) before the
    MFMA and accumulates in fp32.  Tolerance: 1e-2 of the largest reference magnitude per tensor
    (rounding errors of the summands are independent, so the sums do better than 2^-8)."""
    ops = _ops()
    B, I, M = shape
    rng = np.random.default_rng(sum(shape) + 1)
    x = rng.random((B, I)).astype(np.float32)
    W = (rng.standard_normal((M, I)) * 0.5).astype(np.float32)
    gm = rng.standard_normal((B, M)).astype(np.float32)
    xt = dev(x).requires_grad_(); Wt = dev(W).requires_grad_()
    m = ops.SoftMapFunction.apply(xt, Wt, tau, 1)
    want_m = orc.soft_mapping_forward(x, W, tau, torch.float64)
    got_m = m.detach().cpu().numpy()
    assert np.abs(got_m - want_m).max() <= 1e-2 * np.abs(want_m).max()
    assert np.abs(got_m - want_m).max() > 0  # the bf16 path ran, not the fp32 one
    m.backward(dev(gm))
    gx, gW = orc.soft_mapping_backward(x, W, gm, tau)
    assert np.abs(xt.grad.cpu().numpy() - gx).max() <= 1e-2 * np.abs(gx).max()
    assert np.abs(Wt.grad.cpu().numpy() - gW).max() <= 1e-2 * np.abs(gW).max()


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("shape", [
    (1, 1, 1), (64, 31, 127), (128, 128, 256),   # one tile and its edges; rows of W that are no multiple of 8
    (129, 129, 257), (256, 1030, 300),           # 256-row tiles begin; every dimension one past a tile; widths of no 16-byte rows
    (257, 2050, 70), (300, 4100, 1050),          # row statistics with 512 and 1024 threads per block; ragged batches
    (40, 8200, 33),                              # rows too wide for the registers: read three times
    (70, 200, 70000),                            # gW in tiles of 256 rows of W; the last of them ragged
])
def test_soft_mapping_tile_edges(shape, precision):
    """Every padded edge of the matrix products against float64, in the 2-norm.  fp32 operands: a softmax entry carries
    |w - max| / tau * 2^-23 from its exponent (here below 5 * 2^-23) and two roundings, a sum of n products sqrt(n) * 2^-24
    for n <= 70000: below 1e-5 together.  bf16 operands: three factors rounded to 2^-9 each, 1e-2.  gW = S (G - r) / tau is a
    difference: its error is that of its two terms (with one input it is exactly zero, and they are not)."""
    ops = _ops()
    B, I, M = shape
    g = torch.Generator("cuda").manual_seed(B + I + M)
    x = torch.rand(B, I, device="cuda", generator=g)
    W = torch.randn(M, I, device="cuda", generator=g) * 0.5
    gm = torch.randn(B, M, device="cuda", generator=g)
    xt, Wt = x.clone().requires_grad_(), W.clone().requires_grad_()
    m = ops.SoftMapFunction.apply(xt, Wt, 1.0, precision)
    m.backward(gm)
    xd, Wd = x.double().requires_grad_(), W.double().requires_grad_()
    md = xd @ torch.softmax(Wd, dim=-1).t()
    md.backward(gm.double())
    limit = 1e-5 if precision == 0 else 1e-2
    S, G, r = torch.softmax(Wd.detach(), dim=-1), gm.double().t() @ x.double(), (gm.double() * md.detach()).sum(0)
    terms = (S * G).norm() + (S * r[:, None]).norm()
    for got, want, size in ((m.detach(), md.detach(), md.norm()), (xt.grad, xd.grad, xd.grad.norm()), (Wt.grad, Wd.grad, terms)):
        assert torch.isfinite(got).all()
        assert float((got.double() - want).norm()) <= limit * float(size)


def test_soft_mapping_bf16_gradient_of_w_takes_gm_itself():
    """With bf16 operands gW's products are of gm and x rounded once each; 1 / row sum comes in fp32 afterwards.  The same
    arithmetic in float64 leaves fp32 roundings, and an exponential that falls on the other side of a bf16 rounding boundary
    (one in 2^15 entries by 2^-8, in the 2-norm 2e-5): 1e-4.  Rounding gm / row sum instead differs by 5e-3."""
    ops = _ops()
    B, I, M, tau = 200, 300, 70, 0.7
    g = torch.Generator("cuda").manual_seed(9)
    x = torch.rand(B, I, device="cuda", generator=g)
    W = torch.randn(M, I, device="cuda", generator=g)
    gm = torch.randn(B, M, device="cuda", generator=g)
    xt, Wt = x.clone().requires_grad_(), W.clone().requires_grad_()
    m = ops.SoftMapFunction.apply(xt, Wt, tau, 1)
    m.backward(gm)
    E = torch.exp((W - W.max(dim=1, keepdim=True).values) / tau).bfloat16().double()
    S = E / E.sum(dim=1, keepdim=True)
    G = gm.bfloat16().double().t() @ x.bfloat16().double()
    r = (gm.double() * m.detach().double()).sum(0)
    want = S * (G - r[:, None]) / tau
    assert float((Wt.grad.double() - want).norm()) <= 1e-4 * float(want.norm())


@pytest.mark.parametrize("value", [float(np.finfo(np.float32).min), 3.3999999e38, 3.38e38])
def test_soft_mapping_of_values_beyond_bf16(value):
    """Finite float32 values up to the largest stay finite through the bf16 planes (3.39e38 and above would round to an
    infinity, and the lowest value's two upper planes could add up to one).  Each output is one dominant product, or a sum
    of terms of one sign: 1e-5 of it, as above."""
    ops = _ops()
    g = torch.Generator("cuda").manual_seed(5)
    x = torch.rand(70, 200, device="cuda", generator=g)
    x[::3, 17] = value
    W = torch.randn(130, 200, device="cuda", generator=g) * 0.5
    W[::2, 17] = 4.0  # the largest of its row: the value itself is summed
    m = ops.SoftMapFunction.apply(x, W, 1.0, 0)
    want = x.double() @ torch.softmax(W.double(), dim=-1).t()
    assert torch.isfinite(m).all()
    assert float(((m.double() - want).abs() / want.abs()).max()) <= 1e-5


def test_soft_mapping_fp32_input_gradient_does_not_drift():
    """The long reduction of gx (24000 selections) stays an fp32 sum.  Independent roundings of 2^-25 (rms): of S two and its
    exponent's (|w - max| about 2), 1.2e-7 together; of the running sum one per 16 products, 75 in a chunk, sqrt(75 / 2) of them
    in the 2-norm, 1.8e-7: 2.2e-7, limit 3e-7.  One running sum for all plane products, rounded downwards, has 6.2e-7."""
    ops = _ops()
    B, I, M = 64, 3136, 24000
    g = torch.Generator("cuda").manual_seed(3)
    x = torch.rand(B, I, device="cuda", generator=g).requires_grad_()
    W = torch.randn(M, I, device="cuda", generator=g) * 0.5
    gm = torch.randn(B, M, device="cuda", generator=g)
    ops.SoftMapFunction.apply(x, W.requires_grad_(), 1.0, 0).backward(gm)
    want = gm.double() @ torch.softmax(W.detach().double(), dim=-1)
    assert float((x.grad.double() - want).norm()) <= 3e-7 * float(want.norm())


LOWEST = float(np.finfo(np.float32).min)


@pytest.mark.parametrize("case", ["two_lowest", "all_lowest", "largest", "infinite", "nan", "huge", "tiny", "denormal"])
@pytest.mark.parametrize("side", ["x", "gm"])
@pytest.mark.parametrize("shape", [(70, 200, 130), (130, 300, 17), (200, 3000, 2000)])
def test_soft_mapping_fp32_range(shape, side, case):
    """fp32 operands of any magnitude give what fp32 sums give: against float64, infinities and NaN in the same places, finite
    results within 1e-5 in the 2-norm (as test_soft_mapping_tile_edges derives it).
    Magnitudes are mixed with ordinary values in two rows, or are those of the whole operand (huge, tiny, denormal)."""
    ops = _ops()
    B, I, M = shape
    g = torch.Generator("cuda").manual_seed(B + len(case))
    x = torch.rand(B, I, device="cuda", generator=g) + 0.1
    W = torch.randn(M, I, device="cuda", generator=g) * 0.5
    W[:3] = 0.0  # equal weights
    gm = torch.rand(B, M, device="cuda", generator=g) + 0.1
    v, other = (x, gm) if side == "x" else (gm, x)
    if case in ("two_lowest", "all_lowest", "largest"):
        other *= 1e-3  # products of the two stay within float32
    if case == "two_lowest":
        v[3, 5] = v[3, 11] = v[40, 2] = v[40, 9] = LOWEST
    elif case == "all_lowest":
        v[3], v[40] = LOWEST, LOWEST
    elif case == "largest":
        v[3, 5], v[40, 2] = -LOWEST, LOWEST
    elif case == "infinite":
        v[3, 5], v[40, 2], v[41, 1] = float("inf"), float("-inf"), float("inf")
    elif case == "nan":
        v[3, 5] = float("nan")
    else:
        v *= {"huge": 1e30, "tiny": 1e-33, "denormal": 1e-38}[case]
    xt, Wt = x.clone().requires_grad_(), W.clone().requires_grad_()
    m = ops.SoftMapFunction.apply(xt, Wt, 1.0, 0)
    m.backward(gm)
    xd, Wd = x.double().requires_grad_(), W.double().requires_grad_()
    S = torch.softmax(Wd, dim=-1)
    md = xd @ S.t()
    md.backward(gm.double())
    Sd, G, r = S.detach(), gm.double().t() @ x.double(), (gm.double() * md.detach()).sum(0)
    # gW = S (G - r) is a difference: its error is that of its terms, and where G and r are infinite alike it is NaN
    terms = Sd * (G.abs() + r.abs()[:, None])
    for got, want, size in ((m.detach(), md.detach(), x.double().abs() @ Sd.t()), (xt.grad, xd.grad, gm.double().abs() @ Sd),
                            (Wt.grad, Wd.grad, terms)):
        got = got.double()
        assert torch.equal(torch.isnan(got), torch.isnan(want))
        assert torch.equal(torch.isinf(got), torch.isinf(want)) and torch.equal(got[torch.isinf(want)], want[torch.isinf(want)])
        finite = torch.isfinite(want)
        scale = float(size[finite].norm()) if finite.any() else 0.0
        err = float((got[finite] - want[finite]).norm())
        assert err <= 1e-5 * scale + 1e-43 * finite.sum().sqrt(), (err, scale)
    # the forward is a mean: no larger than the values it is of, whatever the rounding of the weights
    if side == "x" and case in ("two_lowest", "all_lowest", "largest"):
        assert torch.isfinite(m).all()
        rel = (m.detach().double() - md.detach()).abs() / md.detach().abs()
        assert float(rel.max()) <= 1e-5


@pytest.mark.parametrize("case", ["ordinary", "two_orders", "wide_e", "wide_x", "scaled_gradients", "tiny", "huge", "infinite_x", "nan_gm"])
@pytest.mark.parametrize("shape", [(100, 1030, 60100), (257, 515, 50001)])  # 128- and 256-row tiles, ragged on every side
def test_soft_mapping_fp32_pairs(shape, case):
    """Products large enough for pairs of fp16 halves, and what sends them back to three planes or to fp32 sums.  A pair holds 23
    of 24 bits, so every output stays within 1e-5 (in the 2-norm, as test_soft_mapping_tile_edges derives it) of the sum of its
    terms' magnitudes; gx row by row, however far apart the rows' magnitudes are."""
    ops = _ops()
    B, I, M = shape
    g = torch.Generator("cuda").manual_seed(B + len(case))
    x = torch.rand(B, I, device="cuda", generator=g) + 0.01
    W = torch.randn(M, I, device="cuda", generator=g)
    gm = torch.randn(B, M, device="cuda", generator=g)
    if case == "two_orders":
        x[:, ::2] *= 0.01
        x[x < 0.002] = 0.0
    elif case == "wide_e":  # in the last of the rows: everything else has been written as pairs by then
        W[M - 1, 5] = 40.0
    elif case == "wide_x":
        x[B - 1] *= 1e-20
    elif case == "scaled_gradients":
        gm[::3] *= 1e-25
        gm[1::3] *= 1e10
        gm[:, ::7] *= 1e-6
        gm[5] = 0.0
    elif case == "tiny":
        x *= 1e-33
        gm *= 1e-5
    elif case == "huge":
        x *= 1e25
    elif case == "infinite_x":
        x[3, 7] = float("inf")
    elif case == "nan_gm":
        gm[4, 9] = float("nan")
    xt, Wt = x.clone().requires_grad_(), W.clone().requires_grad_()
    m = ops.SoftMapFunction.apply(xt, Wt, 1.0, 0)
    m.backward(gm)
    xd, gd = x.double(), gm.double()
    S = torch.softmax(W.double(), dim=-1)
    md = xd @ S.t()
    G, r = gd.t() @ xd, (gd * md).sum(0)
    for name, got, want, size in (("m", m.detach(), md, xd.abs() @ S.t()), ("gx", xt.grad, gd @ S, gd.abs() @ S),
                                  ("gW", Wt.grad, S * (G - r[:, None]), S * (G.abs() + (gd * md).abs().sum(0)[:, None]))):
        got = got.double()
        assert torch.equal(torch.isnan(got), torch.isnan(want)), name
        assert torch.equal(torch.isinf(got), torch.isinf(want)), name
        finite = torch.isfinite(want) & torch.isfinite(size)
        diff, size = (got - want).where(finite, 0.0), size.where(finite, 0.0)
        rows = (diff.norm(dim=1) <= 1e-5 * size.norm(dim=1) + 1e-43 * got.shape[1] ** 0.5)
        assert rows.all(), (name, float((diff.norm(dim=1) / size.norm(dim=1)).nan_to_num().max()))


@pytest.mark.parametrize("case", ["blank_sample", "blank_sample_512", "blank_sample_513", "masked_weights", "masked_weights_few",
                                  "any_magnitude", "few_of_any_magnitude", "wide_e_any_magnitude", "wide_x_any_magnitude"])
@pytest.mark.parametrize("shape", [(257, 515, 50001), (100, 1030, 60100)])
def test_soft_mapping_fp32_pairs_gradients_of_any_span(shape, case):
    """Gradients whose smallest values lie below what a pair holds beside the largest, where only they make a result: exact zeros
    in x or in the softmax take the large ones out of it.  Every element of m, gx and gW against float64, relative to the sum of
    its own terms' magnitudes: a product is good to 2^-22, a sum of n fp32 terms, in whatever order, on average to sqrt(n) 2^-24,
    60100 terms 1.5e-5 if they rounded one by one; they go in groups of 16 and more, so a quarter of it."""
    ops = _ops()
    B, I, M = shape
    g = torch.Generator("cuda").manual_seed(B + len(case))
    x = torch.rand(B, I, device="cuda", generator=g) + 0.01
    W = torch.randn(M, I, device="cuda", generator=g)
    gm = torch.randn(B, M, device="cuda", generator=g)
    small = torch.randn(B, M, device="cuda", generator=g) * 2.0 ** -45
    if case == "blank_sample":  # the largest gradients belong to a sample without input
        x[0] = 0.0
        gm[1:] = small[1:]
    elif case.startswith("blank_sample_"):  # in a few columns: as many values as are summed one by one, and one more
        x[0] = 0.0
        gm = torch.where(gm < 0, gm - 0.01, gm + 0.01)  # no small values but those
        gm[0] = gm[0].abs() + 1.0
        first = int(case.rsplit("_", 1)[1])
        cols = torch.arange(1, 1 + first // (B - 1), device="cuda")
        gm[1:, cols] = small[1:, cols].abs() + 2.0 ** -46
        rest = first % (B - 1)
        gm[1 : 1 + rest, M - 1] = 2.0 ** -46
        gm[1 + rest :, M - 1] = 0.0
    elif case.startswith("masked_weights"):  # no row of W with large gradients reads the first inputs
        few = case.endswith("few")
        rows = torch.tensor([3, 700, M - 2] if few else [7], device="cuda")
        if few:
            W[:, :9] = -float("inf")
            W[rows, :9] = 0.0
            gm[:, rows] = small[:, rows]
        else:
            W[rows, : I // 2] = -float("inf")
            gm = small
            gm[:, rows] = 1.0
    else:
        powers = torch.rand(B, M, device="cuda", generator=g) * 100.0 - 90.0
        spread = gm * torch.exp2(powers)
        if case == "few_of_any_magnitude":
            gm[5, 100:150], gm[90, 41:300] = spread[5, 100:150], spread[90, 41:300]
        else:
            gm = spread
        x[:, ::3] = 0.0
        W[:, 1::4] = -float("inf")
        W[::2, 2::4] = -float("inf")
        if case.startswith("wide_e"):
            W[M - 1, 0] = 25.0
        elif case.startswith("wide_x"):
            x[B - 1] *= 1e-12
    xt, Wt = x.clone().requires_grad_(), W.clone().requires_grad_()
    m = ops.SoftMapFunction.apply(xt, Wt, 1.0, 0)
    again = torch.autograd.grad(m, (xt, Wt), gm, retain_graph=True)
    m.backward(gm)
    assert torch.equal(xt.grad, again[0]) and torch.equal(Wt.grad, again[1])
    xd, gd = x.double(), gm.double()
    S = torch.softmax(W.double(), dim=-1)
    md = xd @ S.t()
    G, r = gd.t() @ xd, (gd * md).sum(0)
    for name, got, want, size in (("m", m.detach(), md, md), ("gx", xt.grad, gd @ S, gd.abs() @ S),
                                  ("gW", Wt.grad, S * (G - r[:, None]), S * (gd.abs().t() @ xd + (gd * md).abs().sum(0)[:, None]))):
        error = (got.double() - want).abs()
        worst = float((error / (size + 1e-37)).max())
        assert worst <= 4e-6, (name, worst)


@pytest.mark.parametrize("shape,limit", [((512, 512, 24000), 1.35e-7), ((512, 3136, 4000), 1.30e-7), ((512, 1000, 14000), 1.40e-7)])
def test_soft_mapping_fp32_input_gradient_of_short_reductions(shape, limit):
    """gx summed in short chunks is as close to float64 as with operands of 24 bits: measured 1.28e-7, 1.23e-7 and 1.35e-7 in the
    2-norm (1.42e-7, 1.38e-7 and 1.44e-7 with operands of 23)."""
    B, I, M = shape
    g = torch.Generator("cuda").manual_seed(B + I + M)
    x = torch.rand(B, I, device="cuda", generator=g).requires_grad_()
    W = torch.randn(M, I, device="cuda", generator=g) * 1.5
    gm = torch.randn(B, M, device="cuda", generator=g)
    _ops().SoftMapFunction.apply(x, W.requires_grad_(), 1.0, 0).backward(gm)
    want = gm.double() @ torch.softmax(W.detach().double(), dim=-1)
    assert float((x.grad.double() - want).norm() / want.norm()) <= limit


@pytest.mark.parametrize("precision", [0, 1])
def test_soft_mapping_of_more_rows_than_a_grid_dimension(precision):
    """4.19 million rows are 65536 blocks of 64 rows; limits as in test_soft_mapping_tile_edges."""
    ops = _ops()
    B, I, M = 4_194_400, 3, 2
    g = torch.Generator("cuda").manual_seed(1)
    x = torch.rand(B, I, device="cuda", generator=g).requires_grad_()
    W = torch.randn(M, I, device="cuda", generator=g)
    gm = torch.randn(B, M, device="cuda", generator=g)
    m = ops.SoftMapFunction.apply(x, W, 1.0, precision)
    m.backward(gm)
    S = torch.softmax(W.double(), dim=-1)
    limit = 1e-5 if precision == 0 else 1e-2
    for got, want in ((m.detach(), x.detach().double() @ S.t()), (x.grad, gm.double() @ S)):
        assert float((got.double() - want).abs().max()) <= limit * float(want.abs().max())


def test_soft_and_hard_mapping_against_reference_vectors(golden):
    ops = _ops()
    g = golden
    for tau_key, mk, gxk, gWk in [("soft_tau", "soft_m", "soft_gx", "soft_gW"),
                                  ("soft_tau_500", "soft500_m", "soft500_gx", "soft500_gW")]:
        tau = float(g[tau_key][0])
        xt = dev(g["soft_x"]).requires_grad_(); Wt = dev(g["soft_W"]).requires_grad_()
        m = ops.SoftMapFunction.apply(xt, Wt, tau, 0)
        np.testing.assert_allclose(m.detach().cpu().numpy(), g[mk].reshape(5, -1), rtol=1e-5, atol=1e-6)
        m.backward(dev(g["soft_gm"].reshape(5, -1)))
        np.testing.assert_allclose(xt.grad.cpu().numpy(), g[gxk], rtol=1e-4, atol=1e-5)
        np.testing.assert_allclose(Wt.grad.cpu().numpy(), g[gWk], rtol=1e-4, atol=1e-5)
    sel = ops.row_argmax(dev(g["soft_W"]))
    assert np.array_equal(sel.cpu().numpy().reshape(7, 3), g["hard_idx"])
    plan = ops.MappingPlan(sel.view(-1, 1), 20)
    xt = dev(g["soft_x"]).requires_grad_()
    hm = ops.HardSelectFunction.apply(xt, sel, plan)
    assert np.array_equal(hm.detach().cpu().numpy(), g["hard_m"].reshape(5, -1))
    gm = np.random.default_rng(1).standard_normal(hm.shape).astype(np.float32)
    hm.backward(dev(gm))
    want = orc.gather_backward(gm[:, :, None], sel.cpu().numpy().reshape(-1, 1), 20)
    np.testing.assert_allclose(xt.grad.cpu().numpy(), want, rtol=1e-6, atol=1e-6)


def test_row_argmax_ties_and_sizes():
    ops = _ops()
    rng = np.random.default_rng(2)
    W = rng.standard_normal((300, 1000)).astype(np.float32)
    W[5, 17] = W[5, 900] = 9.0   # tie: lowest index wins
    W[6, :] = -1.0
    sel = ops.row_argmax(dev(W)).cpu().numpy()
    assert np.array_equal(sel, W.argmax(1)) and sel[5] == 17 and sel[6] == 0
    # widths that are no multiple of four (one value per lane and load), of four but not of 1024 (a tail of 16-byte
    # loads), and a tie that straddles two lanes' pieces
    for M, I in ((9, 1031), (5, 2052), (7, 4096), (3, 12)):
        W = rng.standard_normal((M, I)).astype(np.float32)
        W[1, I - 1] = W[1, 2] = 7.0
        W[2, :] = 0.5
        sel = ops.row_argmax(dev(W)).cpu().numpy()
        assert np.array_equal(sel, W.argmax(1)) and sel[1] == 2 and sel[2] == 0


# ------------------------------------------------------------------------------ encoder / head
def test_thermometer_and_group_sum(golden):
    ops = _ops()
    g = golden
    bits = ops.thermometer_encode(dev(g["thermo_x"]), dev(g["thermo_thr"]))
    assert np.array_equal(bits.cpu().numpy().reshape(9, -1), g["thermo_bits"])
    xt = dev(g["groupsum_x"]).requires_grad_()
    y = ops.GroupSumFunction.apply(xt, 5, 2.0)
    np.testing.assert_allclose(y.detach().cpu().numpy(), g["groupsum_y"], rtol=1e-6, atol=1e-6)
    gy = np.random.default_rng(0).standard_normal((6, 5)).astype(np.float32)
    y.backward(dev(gy))
    np.testing.assert_allclose(xt.grad.cpu().numpy(), np.repeat(gy, 4, 1) / 2.0, rtol=1e-6)
    # rows of bits that are and are not a multiple of four values (16-byte stores or one value at a time), strict compare
    for B, F, nb in ((7, 5, 3), (64, 12, 4), (3, 6, 2), (130, 784, 4), (5, 1, 1)):
        rs = np.random.default_rng(B * F + nb)
        xs = rs.random((B, F)).astype(np.float32)
        th = np.sort(rs.random((F, nb)).astype(np.float32), axis=1)
        xs[0, 0] = th[0, 0]  # equal to a threshold: not above it
        got = ops.thermometer_encode(dev(xs), dev(th)).cpu().numpy().reshape(B, F, nb)
        assert np.array_equal(got, (xs[:, :, None] > th[None]).astype(np.float32))
    x = np.random.default_rng(1).standard_normal((3, 10)).astype(np.float32)  # 10 features, 4 groups: padded
    y = ops.GroupSumFunction.apply(dev(x), 4, 1.0)
    np.testing.assert_allclose(y.cpu().numpy(), orc.group_sum(x, 4, 1.0), rtol=1e-6, atol=1e-6)


@pytest.mark.parametrize("shape", [(8192, 10), (1, 3), (257, 1), (1000, 64), (33, 300)])
def test_cross_entropy_against_torch(shape):
    """Fused mean cross-entropy and its gradient against torch's own (float64 on the CPU): loss to rtol 1e-6,
    gradient to rtol 1e-5 with a floor of 1e-9 (entries are (softmax - onehot) / B); large logits do not overflow;
    a row with a label outside the classes adds nothing."""
    from difflut_amd.utils import cross_entropy
    B, C = shape
    rng = np.random.default_rng(B + C)
    z = (rng.standard_normal((B, C)) * 4).astype(np.float32)
    z[0, 0] = 90.0                                        # exp(90) overflows fp32 without the max shift
    y = rng.integers(0, C, (B,))
    zt = dev(z).requires_grad_()
    loss = cross_entropy(zt, torch.as_tensor(y, device=DEV))
    (loss * 3.0).backward()
    zr = torch.tensor(z, dtype=torch.float64, requires_grad=True)
    want = torch.nn.functional.cross_entropy(zr, torch.as_tensor(y))
    (want * 3.0).backward()
    np.testing.assert_allclose(loss.item(), want.item(), rtol=1e-6)
    np.testing.assert_allclose(zt.grad.cpu().numpy(), zr.grad.numpy(), rtol=1e-5, atol=1e-9)
    if B > 1:
        y2 = y.copy()
        y2[1] = C + 5
        l2 = cross_entropy(dev(z), torch.as_tensor(y2, device=DEV))
        keep = np.ones(B, bool); keep[1] = False
        ref = torch.nn.functional.cross_entropy(torch.tensor(z[keep], dtype=torch.float64), torch.as_tensor(y[keep]), reduction="sum") / B
        np.testing.assert_allclose(l2.item(), ref.item(), rtol=1e-6)


@pytest.mark.parametrize("B,C,blocks", [(256, 100, 1), (257, 19, 1), (512, 10, 1), (1024, 5, 1),
                                        (257, 20, 2), (512, 8, 2), (1024, 10, 4), (1024, 100, 4), (1000, 64, 4)])
def test_cross_entropy_of_many_classes(B, C, blocks):
    """One block only where its rows' logits stay in the L1 of a CU, and the same loss and gradient on either side of the line.  A row's
    loss is within 2e-6 of its size, its gradient within 2e-7 / B of an exponential, a sum of C and a reciprocal."""
    from difflut_amd import ops

    g = torch.Generator("cuda").manual_seed(B + C)
    z = torch.randn(B, C, device=DEV, generator=g)
    labels = torch.randint(0, C, (B,), device=DEV, generator=g)
    zt = z.clone().requires_grad_()
    ran = _kernels_of(lambda: ops.CrossEntropyFunction.apply(zt, labels).backward())
    assert ran.count("cross_entropy_rows") == 1 and ran.count("cross_entropy_mean") == (blocks > 1)
    zr = z.double().cpu().requires_grad_()
    want = torch.nn.functional.cross_entropy(zr, labels.cpu())
    want.backward()
    torch.testing.assert_close(ops.CrossEntropyFunction.apply(z, labels).double().cpu(), want.detach(), rtol=2e-6, atol=0)
    torch.testing.assert_close(zt.grad.double().cpu(), zr.grad, rtol=1e-5, atol=1e-6 / B)


@pytest.mark.parametrize("B,C", [(64, 2), (65, 3), (1024, 10), (1025, 10), (70000, 2)])
def test_cross_entropy_blocks(B, C):
    """One block, or sums of blocks; the last has more blocks than the kernel that adds them has threads.  A
    row's gradient is (p - 1) / B or p / B, p within 2e-7 (an exponential, a sum of C, a reciprocal); the loss a sum of B values of
    size up to 20 by halves: rtol 2e-6."""
    from difflut_amd.utils import cross_entropy

    g = torch.Generator("cuda").manual_seed(B + C)
    z = torch.randn(B, C, device=DEV, generator=g) * 5
    y = torch.randint(0, C, (B,), device=DEV, generator=g)
    zt = z.clone().requires_grad_()
    loss = cross_entropy(zt, y)
    loss.backward()
    zr = z.double().requires_grad_()
    want = torch.nn.functional.cross_entropy(zr, y)
    want.backward()
    torch.testing.assert_close(loss.double(), want.detach(), rtol=2e-6, atol=0.0)
    torch.testing.assert_close(zt.grad.double(), zr.grad, rtol=1e-5, atol=2e-7 / B)



# ------------------------------------------------------------------------------ error paths
def test_argument_errors_are_reported_not_launched():
    from difflut_amd import _native as nat
    lib = nat.lib()
    assert lib.dl_dwn_layer_fwd(None, None, None, None, None, None, 0, 1, 1, 1, 1, 1, None) == -1
    t = torch.zeros(64, device=DEV)
    p = t.data_ptr()
    assert lib.dl_dwn_layer_fwd(p, p, p, p, p, p, 0, 4, 4, 4, 2, 1, None) == -4   # workspace too small
    assert lib.dl_dwn_layer_fwd(p, p, p, p, p, p, 1 << 20, 4, 4, 4, 17, 1, None) == -3  # k beyond DL_MAX_K
    assert lib.dl_gather_fwd(p, p, 8, p, 1, 1, 1, 1, None) == -3
    assert lib.dl_prob_layer_fwd(p, p, p, 1.0, p, p, 256, 0, 1, 1, 1, 1, None) == -2
    with pytest.raises(RuntimeError, match="ROCm devices only"):
        _ops().DWNLayerFunction.apply(torch.zeros(2, 2), torch.zeros(1, 1, 4), None, 0.1, 0.1)
    with pytest.raises(IndexError):
        _ops().MappingPlan(torch.tensor([[0, 7]], device=DEV, dtype=torch.int32), 4)


def test_row_counts_beyond_one_grid_dimension():
    """B > 65535 rows for the gathers (RandomLayer.get_mapping, LearnableLayer eval) and more than 2^20 rows for the
    bit-plane packing (patch matrices of large image batches): the kernels walk the rows a grid dimension cannot hold."""
    from difflut_amd import _native as nat
    lib = nat.lib()
    rng = np.random.default_rng(5)
    B, I, N, k = 70001, 9, 5, 2
    x = rng.random((B, I)).astype(np.float32)
    idx = rng.integers(0, I, (N, k)).astype(np.int16)
    xd, idd = dev(x), torch.as_tensor(idx).to(DEV)
    m = torch.empty(B, N * k, device=DEV)
    nat.check(lib.dl_gather_fwd(xd.data_ptr(), idd.data_ptr(), 16, m.data_ptr(), B, I, N, k, nat.stream()))
    assert np.array_equal(m.cpu().numpy(), x[:, idx.reshape(-1).astype(np.int64)])
    plan = _ops().MappingPlan(idd.to(torch.int32), I)
    gm = rng.standard_normal((B, N * k)).astype(np.float32)
    gx = torch.empty(B, I, device=DEV)
    nat.check(lib.dl_gather_bwd(dev(gm).data_ptr(), plan.inv_ptr.data_ptr(), plan.inv_pos.data_ptr(), gx.data_ptr(), B, I, N, k,
                                nat.stream()))
    want = np.zeros((B, I), np.float32)
    for p, i in enumerate(idx.reshape(-1)):
        want[:, i] += gm[:, p]
    np.testing.assert_allclose(gx.cpu().numpy(), want, rtol=1e-6, atol=1e-6)
    # bit-planes of 1 050 000 rows x 8 columns: 65 625 pieces of 16 rows
    R, C = 1050000, 8
    v = torch.rand(R, C, device=DEV)
    planes = torch.zeros(lib.dl_dwn_planes_bytes(R, C) // 8, dtype=torch.int64, device=DEV)
    nat.check(lib.dl_dwn_pack_planes(v.data_ptr(), planes.data_ptr(), R, C, nat.stream()))
    BT = (R + 63) // 64
    bits = torch.zeros(BT * 64, C, dtype=torch.int64, device=DEV)
    bits[:R] = (v >= 0.5).long()
    want_planes = (bits.view(BT, 64, C) << torch.arange(64, device=DEV).view(1, 64, 1)).sum(1)  # wraps into the sign bit
    assert torch.equal(planes[:BT * C].view(BT, C), want_planes)


@pytest.mark.parametrize("opts", [dict(lr=0.01), dict(lr=0.003, betas=(0.8, 0.95), eps=1e-6, weight_decay=0.05),
                                  dict(lr=0.01, maximize=True)])
def test_bank_adam_against_torch_adam(opts):
    """`dl_adam_step`: several tensors of ragged sizes (one of them not 16-byte aligned) in one launch, five steps,
    against torch.optim.Adam on the same gradients."""
    from difflut_amd.utils import BankAdam

    torch.manual_seed(11)
    base = torch.randn(5000 + 1, device=DEV)
    ours = [torch.randn(300, 1, 64, device=DEV).requires_grad_(), torch.randn(2049, device=DEV).requires_grad_(),
            None, torch.randn(3, device=DEV).requires_grad_()]
    ours[2] = base[1:].detach().requires_grad_()  # a view that starts 4 bytes into its allocation
    ref = [t.detach().clone().requires_grad_() for t in ours]
    opt, ropt = BankAdam(ours, **opts), torch.optim.Adam(ref, **opts)
    for _ in range(5):
        for x, y in zip(ours, ref):
            g = torch.randn_like(x)
            x.grad, y.grad = g.clone(), g.clone()
        opt.step()
        ropt.step()
    for x, y in zip(ours, ref):
        np.testing.assert_allclose(x.detach().cpu().numpy(), y.detach().cpu().numpy(), rtol=2e-6, atol=1e-7)
    from difflut_amd import _native
    assert _native.lib().dl_adam_step(None, None, None, None, None, 1, 0.1, 0.9, 0.999, 1e-8, 0.0, 1, 0, None) == -1


@pytest.mark.parametrize("per_row", [False, True])
@pytest.mark.parametrize("subtract_mean", [False, True])
def test_grad_stabilize_against_the_reference_formula(per_row, subtract_mean):
    """`dl_grad_stabilize` against the torch operations of base_layer.py:266-339 evaluated in float64."""
    torch.manual_seed(3)
    rows, cols = 37, 5003
    g = (torch.randn(rows, cols, device=DEV) * 0.3 + 0.05)
    out = _ops().grad_stabilize(g, per_row, 0.7, subtract_mean, 1e-8)
    w = g.double()
    if subtract_mean:
        w = w - (w.mean(dim=1, keepdim=True) if per_row else w.mean())
    var = w.pow(2).mean(dim=1, keepdim=True) if per_row else w.pow(2).mean()
    want = w * torch.sqrt(0.7 / (var + 1e-8))
    np.testing.assert_allclose(out.cpu().numpy(), want.cpu().numpy(), rtol=1e-5, atol=1e-6)
    again = _ops().grad_stabilize(g, per_row, 0.7, subtract_mean, 1e-8)
    assert torch.equal(out, again)  # fixed order of additions


@pytest.mark.parametrize("k", [1, 2, 3, 4, 5, 6])
@pytest.mark.parametrize("B,N,O", [(63, 64, 1), (200, 301, 1), (129, 70, 3)])  # ragged rows, ragged wavefronts, stores by a node each
def test_address_bytes_of_hidden_layers(k, B, N, O):
    """The address of every node and row that a hidden layer of a chain keeps for its backward, against the inputs' bits."""
    from difflut_amd import _native as nat

    lib = nat.lib()
    g = torch.Generator("cuda").manual_seed(B + k)
    I = 90
    idx = torch.randint(0, I, (N, k), device=DEV, generator=g, dtype=torch.int32)
    luts = torch.randn(N, O, 1 << k, device=DEV, generator=g)
    x = (torch.rand(B, I, device=DEV, generator=g) < 0.5).float()
    tiles = (B + 63) // 64
    planes, out = (torch.empty(lib.dl_dwn_planes_bytes(B, c), dtype=torch.uint8, device=DEV) for c in (I, N * O))
    saved = torch.full((lib.dl_dwn_saved_bytes(B, I, N, k, O),), 77, dtype=torch.uint8, device=DEV)
    nat.check(lib.dl_dwn_pack_planes(x.data_ptr(), planes.data_ptr(), B, I, nat.stream()))
    nat.check(lib.dl_dwn_layer_fwd_planes(planes.data_ptr(), idx.data_ptr(), luts.data_ptr(), None, out.data_ptr(), saved.data_ptr(),
                                          B, I, N, k, O, nat.stream()))
    bits = torch.zeros(tiles * 64, I, dtype=torch.int64, device=DEV)
    bits[:B] = x.long()
    want = (bits[:, idx.long()] << torch.arange(k, device=DEV)).sum(-1).view(tiles, 64, N).transpose(1, 2)
    assert torch.equal(saved[:tiles * N * 64].view(tiles, N, 64).long(), want)


def test_forward_of_a_narrow_layer_on_very_many_rows():
    """A few columns on more rows than eight grid rows each could cover: y and the addresses against the bits."""
    ops = _ops()
    B, I, N, k = 8 * 65536 + 3, 3, 2, 2
    g = torch.Generator("cuda").manual_seed(3)
    x = (torch.rand(B, I, device=DEV, generator=g) < 0.5).float()
    idx = torch.tensor([[0, 2], [1, 0]], dtype=torch.int32, device=DEV)
    luts = torch.randn(N, 1, 1 << k, device=DEV, generator=g).requires_grad_()
    y = ops.dwn_layer(x, luts, ops.MappingPlan(idx, I), 0.1, 0.1)
    at = (x.long()[:, idx.long()] << torch.arange(k, device=DEV)).sum(-1)  # [B, N]
    assert torch.equal(y, luts.detach()[:, 0].gather(1, at.t()).t())
    y.backward(torch.ones_like(y))
    # ones, added in single precision by quads of rows: whole numbers below 2^24, so exact
    assert torch.equal(luts.grad[:, 0], torch.stack([torch.bincount(at[:, n], minlength=1 << k) for n in range(N)]).float())
