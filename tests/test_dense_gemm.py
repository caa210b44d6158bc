"""Large-M bf16 GEMM (csrc/dense_gemm.hip, the bf16 projections at prefill
sizes: acorninfer/models/qwen3.py:21-47's F.linear; the planner's default
from 256 rows, DENSE_M_MIN).

Oracle: the float64 product of the same bf16 operands. fp32 output must
match it to fp32 accumulation drift (a dropped k step, a wrong row or column,
a transposed tile all fail by orders of magnitude); the bf16 output must be
exactly the fp32 output rounded once (the same sums, rounded in the
epilogue).
Shapes: ragged M and N (tile edges inside the launch), every (BM, depth)
variant, configuration 3's projections at M = 2048 against an fp32 matmul;
plus the planner's routing (CPU), determinism, graph replay and no writes
outside [M, N].
"""
import pytest
import torch

from gpu_utils import graph_replays_match

DENSE_RT = -2
SMALL = [(512, 256, 128), (513, 260, 256), (1000, 1028, 512), (1100, 4096, 1024),
         (777, 1536, 384)]
CONFIG3 = {"qkv": (6144, 4096), "o": (4096, 4096), "gate_up": (24576, 4096),
           "down": (4096, 12288)}


def _operands(M, N, K, seed):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(M, K, generator=g).bfloat16()
    w = (0.02 * torch.randn(N, K, generator=g)).bfloat16()
    return x, w


def _planes(x, w, tiling):
    """fp32 split-K planes [ksplit, M, N] of the planned launch."""
    from acorninfer_amd._lib import WFMT_BF16
    from acorninfer_amd.ops.quant_gemm import gemm_partials, plan
    t, _ = plan(x.shape[0], w.shape[0], x.shape[1], WFMT_BF16, tiling)
    part = torch.full((t.ksplit, x.shape[0], w.shape[0]), float("nan"), device="cuda")
    gemm_partials(x, w, None, None, WFMT_BF16, part, t)
    return part


def _run(x, w, tiling, fp32):
    from acorninfer_amd.ops.quant_gemm import bf16_gemm
    if fp32:
        planes = _planes(x, w, tiling)
        total = planes[0].clone()
        for p in planes[1:]:              # in split order, as the consumers sum them
            total += p
        return total
    return bf16_gemm(x, w, cfg=tiling)


def test_planner_routes_prefill_sizes_to_the_dense_kernel():
    from acorninfer_amd._lib import WFMT_BF16, WFMT_W8
    from acorninfer_amd.ops.quant_gemm import Tiling, plan
    # from 256 rows: 256 x 256 tiles, both operands by direct-to-LDS loads,
    # split K while the tiles (16 x 2 here) leave CUs idle
    t, tiles = plan(512, 4096, 4096, WFMT_BF16)
    assert t == Tiling(DENSE_RT, 256, 128, 8, 4) and tiles == 16 * 2
    # ... but not into a second round of workgroups: 24 x 2 tiles take 4 splits,
    # 24 x 8 and 96 x 2 none
    assert plan(512, 6144, 4096, WFMT_BF16)[0] == Tiling(DENSE_RT, 256, 128, 4, 4)
    assert plan(2048, 6144, 4096, WFMT_BF16)[0] == Tiling(DENSE_RT, 256, 128, 1, 4)
    assert plan(512, 24576, 4096, WFMT_BF16)[0] == Tiling(DENSE_RT, 256, 128, 1, 4)
    assert plan(2048, 4096, 4096, WFMT_BF16)[0] == Tiling(DENSE_RT, 256, 128, 2, 4)
    assert plan(8192, 4096, 4096, WFMT_BF16)[0] == Tiling(DENSE_RT, 256, 128, 1, 4)
    assert plan(512, 4096, 4096, WFMT_BF16, Tiling(DENSE_RT, 128))[0] == \
        Tiling(DENSE_RT, 128, 64, 4, 4)                              # the 128-row form
    assert plan(8192, 4096, 4096, WFMT_BF16, Tiling(DENSE_RT, 256, 64))[0] == \
        Tiling(DENSE_RT, 256, 64, 1, 2)                              # register-staged form
    assert plan(255, 4096, 4096, WFMT_BF16)[0].rt != DENSE_RT       # tiled kernel below 256
    assert plan(256, 6144, 4096, WFMT_BF16)[0] == Tiling(DENSE_RT, 256, 128, 8, 4)
    assert plan(256, 4096, 12288, WFMT_BF16)[0] == Tiling(DENSE_RT, 256, 128, 16, 4)
    assert plan(4096, 4096, 192, WFMT_BF16)[0] == Tiling(DENSE_RT, 256, 128, 1, 4)  # 6 stages of 32
    assert plan(4096, 4096, 4096, WFMT_W8)[0].rt != DENSE_RT        # bf16 weights only
    assert plan(64, 4096, 4096, WFMT_BF16, Tiling(DENSE_RT, 64, 0, 1, 4))[0] == \
        Tiling(DENSE_RT, 64, 64, 1, 4)                               # on request at any M
    with pytest.raises(NotImplementedError):
        plan(4096, 4096, 4096, WFMT_BF16, Tiling(DENSE_RT, 32, 0, 0, 2))


@pytest.mark.gpu
@pytest.mark.parametrize("wn,bm,depth", [(64, 128, 2), (64, 128, 4), (64, 64, 2), (64, 64, 4),
                                         (128, 64, 2), (64, 256, 2), (128, 256, 4)])
def test_dense_gemm_matches_float64(wn, bm, depth):
    from acorninfer_amd.ops.quant_gemm import Tiling
    for i, (M, N, K) in enumerate(SMALL):
        # the direct-to-LDS form (256, 128) runs 32-k stages in pairs
        if ((K // 32) % 2 if (bm, wn) == (256, 128) else (K // 64) % depth):
            continue
        print(f"\n[dense GEMM M={M} N={N} K={K} wn={wn} bm={bm} depth={depth}]", flush=True)
        x, w = _operands(M, N, K, 100 + i)
        ref = x.double() @ w.double().T
        t = Tiling(DENSE_RT, bm, wn, 0, depth)
        got32 = _run(x.cuda(), w.cuda(), t, True).cpu()
        torch.testing.assert_close(got32.double(), ref, rtol=1e-5, atol=1e-5)
        # the bf16 output is the same fp32 sums rounded once (same tiles, same order)
        got16 = _run(x.cuda(), w.cuda(), t, False).cpu()
        assert torch.equal(got16, got32.to(torch.bfloat16))


@pytest.mark.gpu
@pytest.mark.parametrize("M", [2048, 256, 300])
@pytest.mark.parametrize("cls", list(CONFIG3))
def test_dense_gemm_config3_at_prefill_m(cls, M):
    """The default plan at M = 2048 (a 2048-token prompt) and at 256 / 300
    rows (the smallest that take the 256 x 256 form, up to 16 K splits, a
    ragged last tile) on configuration 3's shapes, fp32 partials against the
    fp32 matmul of the same operands."""
    from acorninfer_amd._lib import WFMT_BF16
    from acorninfer_amd.ops.quant_gemm import plan
    N, K = CONFIG3[cls]
    assert plan(M, N, K, WFMT_BF16)[0][:3] == (DENSE_RT, 256, 128)
    x, w = _operands(M, N, K, 7)
    xd, wd = x.cuda(), w.cuda()
    got = _run(xd, wd, None, True)
    ref = xd.float() @ wd.float().T
    rel = ((got - ref).norm() / ref.norm()).item()
    print(f"\n[dense GEMM {cls} M={M}: rel err vs fp32 matmul {rel:.3g}]", flush=True)
    assert rel < 1e-5


@pytest.mark.gpu
@pytest.mark.parametrize("bm,wn,depth", [(128, 0, 2), (256, 0, 2), (256, 128, 4)])
def test_dense_gemm_deterministic_graph_and_bounds(bm, wn, depth):
    from acorninfer_amd._lib import WFMT_BF16
    from acorninfer_amd.ops.quant_gemm import Tiling, gemm_partials
    M, N, K = 600, 516, 256
    x, w = _operands(M, N, K, 3)
    xd, wd = x.cuda(), w.cuda()
    t = Tiling(DENSE_RT, bm, wn, 1, depth)
    big = torch.full((M + 7, N), 9.0, device="cuda")       # 7 guard rows after the output
    part = big[:M].view(1, M, N)
    gemm_partials(xd, wd, None, None, WFMT_BF16, part, t)
    first = big.clone()
    gemm_partials(xd, wd, None, None, WFMT_BF16, part, t)
    assert torch.equal(big, first)
    assert bool((big[M:] == 9.0).all())

    def fn():
        gemm_partials(xd, wd, None, None, WFMT_BF16, part, t)

    assert graph_replays_match(fn, lambda: part)


@pytest.mark.gpu
@pytest.mark.parametrize("ks", [2, 4])
def test_dense_gemm_split_planes_are_k_range_products(ks):
    """Split s writes the product over its own K range: each plane against the
    float64 product of the matching column slices of x and w."""
    from acorninfer_amd.ops.quant_gemm import Tiling
    M, N, K = 300, 520, 1024
    x, w = _operands(M, N, K, 17)
    planes = _planes(x.cuda(), w.cuda(), Tiling(DENSE_RT, 64, 64, ks, 2)).cpu()
    assert planes.shape[0] == ks
    kr = K // ks
    for s in range(ks):
        ref = x[:, s * kr:(s + 1) * kr].double() @ w[:, s * kr:(s + 1) * kr].double().T
        torch.testing.assert_close(planes[s].double(), ref, rtol=1e-5, atol=1e-5)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(513, 272, 256), (1000, 1040, 512), (777, 1536, 384),
                                   (300, 4096, 1024)])
@pytest.mark.parametrize("tiling", [(DENSE_RT, 256, 128, 1, 4), (DENSE_RT, 256, 128, 2, 4),
                                    (DENSE_RT, 128, 64, 1, 2), (DENSE_RT, 128, 64, 2, 4),
                                    (DENSE_RT, 64, 64, 1, 4), (DENSE_RT, 64, 128, 1, 2)])
def test_dense_gemm_blocked_weights_bitwise(M, N, K, tiling):
    """The decode model's bf16 weights in 1 KB blocks (BF16B) on every form of
    the large-M kernel that reads them (direct-to-LDS 256 x 256; the
    register-direct 64 / 128 forms): the same operands in the same order as
    the natural rows, so the fp32 planes are bit for bit those of the natural
    layout. Ragged N (272, 1040: a last 256-row tile cut inside) and M, K
    splits, 6 and 12 k-pairs."""
    from acorninfer_amd._lib import WFMT_BF16, WFMT_BF16B
    from acorninfer_amd.ops.quant_gemm import Tiling, gemm_partials, plan
    from acorninfer_amd.quant.quantize import to_bf16b
    x, w = _operands(M, N, K, 29)
    xd, wd = x.cuda(), w.cuda()
    wb = to_bf16b(wd)
    t = Tiling(*tiling)
    try:
        tb, _ = plan(M, N, K, WFMT_BF16B, t)
    except NotImplementedError:
        pytest.skip(f"{tiling} not built for K={K}")
    assert tb == plan(M, N, K, WFMT_BF16, t)[0]
    outs = []
    for wf, ww in ((WFMT_BF16B, wb), (WFMT_BF16, wd)):
        part = torch.full((tb.ksplit, M, N), float("nan"), device="cuda")
        gemm_partials(xd, ww, None, None, wf, part, tb)
        outs.append(part)
    torch.cuda.synchronize()
    assert torch.equal(outs[0], outs[1]), tiling
    ref = xd.float() @ wd.float().T
    rel = ((outs[0].sum(0) - ref).norm() / ref.norm()).item()
    assert rel < 1e-5


def test_planner_refuses_blocked_weights_on_the_staged_form():
    """BF16B is read by the direct-to-LDS and register-direct forms only."""
    from acorninfer_amd._lib import WFMT_BF16B
    from acorninfer_amd.ops.quant_gemm import Tiling, plan
    with pytest.raises(NotImplementedError):
        plan(4096, 4096, 4096, WFMT_BF16B, Tiling(DENSE_RT, 256, 64, 1, 2))
    assert plan(4096, 4096, 4096, WFMT_BF16B)[0] == Tiling(DENSE_RT, 256, 128, 1, 4)


# (M, N, K): ragged rows and weight tiles (N a multiple of 16 only), the fewest
# k, one more than a tile, several splits
W8_SHAPES = [(256, 256, 128), (257, 272, 256), (700, 1040, 512), (513, 4096, 1024),
             (1025, 768, 384), (257, 512, 512), (900, 256, 1024)]


def _w8b(N, K, seed):
    from acorninfer_amd.models.qwen3 import WFMT_W8, QLinear
    g = torch.Generator().manual_seed(seed)
    q = torch.randint(-127, 128, (N, K), generator=g, dtype=torch.int8)
    q[0, :] = -127                                     # the range's ends in whole rows
    q[1, :] = 127
    scale = (0.001 + 0.01 * torch.rand(N, generator=g)).half()
    return QLinear(WFMT_W8, q.cuda(), N, K, scale.cuda()).blocked(), q, scale


def _launch8(lin, x, tiling, fp32):
    t, _ = lin.plan(x.shape[0], tiling)
    M = x.shape[0]
    st = torch.cuda.current_stream().cuda_stream
    part = torch.full((t.ksplit, M, lin.N), float("nan"), device="cuda")
    out = None if fp32 else torch.empty(M, lin.N, dtype=torch.bfloat16, device="cuda")
    lin.launch(x, M, t, out=out, part=part, stream=st)
    return part if fp32 else out


@pytest.mark.gpu
@pytest.mark.parametrize("shape", W8_SHAPES)
def test_w8b_large_m_matches_float64(shape):
    """int8 weights on the large-M kernel: the integers enter the MFMAs exactly,
    so fp32 sums differ from float64 by accumulation drift only; the bf16 output
    is the fp32 output rounded once; a split's planes add up to the whole."""
    from acorninfer_amd.ops.quant_gemm import Tiling
    M, N, K = shape
    lin, q, scale = _w8b(N, K, 7 * M + N)
    g = torch.Generator().manual_seed(M)
    x = torch.randn(M, K, generator=g).bfloat16().cuda()
    want = x.double() @ (q.cuda().double() * scale.cuda().double()[:, None]).t()
    rms = want.square().mean().sqrt()
    one = _launch8(lin, x, Tiling(DENSE_RT, 0, 0, 1, 0), True)
    # K terms of relative size up to 127 * 4 / (73 * 1): each add rounds at 2^-24 of the sum
    assert ((one[0].double() - want).abs().max() / rms) < K * 2.0 ** -24 * 8
    out = _launch8(lin, x, Tiling(DENSE_RT, 0, 0, 1, 0), False)
    assert torch.equal(out, one[0].bfloat16())
    for ks in (2, 4, 8):
        if (K // 32) % (2 * ks):
            continue
        planes = _launch8(lin, x, Tiling(DENSE_RT, 0, 0, ks, 0), True)
        assert planes.shape[0] == ks and bool(planes.isfinite().all())
        assert ((planes.double().sum(0) - want).abs().max() / rms) < K * 2.0 ** -24 * 8
    if N % 128:                                        # no form by default, as before
        with pytest.raises(NotImplementedError):
            lin.plan(M)
        return
    # the first rows on this kernel, the rest on the mid-M kernel
    if N % 256 == 0 and K % 512 == 0 and M > 256:
        tail = _launch8(lin, x, Tiling(DENSE_RT, 0, 0, 1, 1), False)
        assert torch.equal(tail[:256], out[:256])
        assert ((tail.double() - want).norm() / want.norm()) < 4e-3
        planes = _launch8(lin, x, Tiling(DENSE_RT, 0, 0, 1, 1), True)
        assert torch.equal(planes[0].bfloat16(), tail)
    # the planner's own choice at this size
    auto = _launch8(lin, x, None, False)
    assert ((auto.double() - want).norm() / want.norm()) < 4e-3       # one bf16 rounding


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(512, 512, 256), (600, 1056, 512)])
def test_w8b_large_m_swiglu_is_silu_mul_of_the_output(M, N, K):
    from acorninfer_amd._lib import BF16, check, lib, ptr, stream_ptr
    from acorninfer_amd.ops.quant_gemm import Tiling
    lin, _, _ = _w8b(N, K, N)
    lin.il16 = True                                    # rows read as gate / up blocks of 16
    x = torch.randn(M, K, generator=torch.Generator().manual_seed(3)).bfloat16().cuda()
    act = torch.empty(M, N // 2, dtype=torch.bfloat16, device="cuda")
    t, _ = lin.swiglu_plan(M)
    assert t.rt == DENSE_RT and t.ksplit == 1
    lin.launch_swiglu(x, M, t, act, stream_ptr())
    plane = _launch8(lin, x, Tiling(DENSE_RT, 0, 0, 1, 0), True)
    want = torch.empty_like(act)
    check(lib().acorn_silu_mul(ptr(plane), 1, None, ptr(want), M, N // 2, 1, BF16, stream_ptr()),
          "silu_mul")
    assert torch.equal(act, want)


@pytest.mark.parametrize("N,K", [(6144, 4096), (4096, 4096), (24576, 4096), (4096, 12288),
                                 (1024, 3072), (4096, 1024), (1040, 512)])
def test_default_tilings_of_the_block_layouts_are_launchable(N, K):
    """The library's choice with nothing requested, asked for again in full, is
    accepted as it is, for every size from one row to a long prompt (no GPU)."""
    from acorninfer_amd._lib import WFMT_BF16B, WFMT_W4B, WFMT_W8B
    from acorninfer_amd.ops.quant_gemm import plan
    for fmt in (WFMT_W4B, WFMT_W8B, WFMT_BF16B):
        for M in (1, 2, 8, 9, 16, 17, 24, 25, 64, 65, 200, 255, 256, 511, 512, 1000, 8192):
            if N % 128 and 16 < M and not (fmt == WFMT_BF16B and M >= 256):
                continue                               # no tiled form: refused
            t, tiles = plan(M, N, K, fmt)
            assert tiles >= 1 and t.ksplit >= 1
            assert plan(M, N, K, fmt, t)[0] == t, (fmt, M, t)


@pytest.mark.parametrize("M,N,K", [(512, 4096, 4096), (1100, 1024, 4096), (300, 4096, 12288),
                                   (1000, 6144, 4096), (257, 1024, 3072), (700, 1040, 512)])
def test_partial_large_m_int8_requests_resolve_to_launchable_plans(M, N, K):
    """Requests for the large-M int8 kernel that leave entries to the planner: a
    division of the rows between the two kernels has one split (they share the
    output's rows, not its planes), a requested split or division is the one
    planned, and the resolved plan asked for again is itself (no GPU)."""
    from acorninfer_amd._lib import WFMT_W8B
    from acorninfer_amd.ops.quant_gemm import Tiling, plan
    mtiles = -(-M // 256)
    for upw in (0, 256):
        for nw in (0, 128):
            for ks in (0, 1, 2, 4):
                for first in (0, 1, 2, mtiles - 1, mtiles, mtiles + 3):
                    req = Tiling(DENSE_RT, upw, nw, ks, first)
                    try:
                        t, _ = plan(M, N, K, WFMT_W8B, req)
                    except NotImplementedError:
                        continue
                    assert t.tpw == (min(first, mtiles) if first else mtiles), (req, t)
                    assert t.tpw == mtiles or t.ksplit == 1, (req, t)
                    assert ks == 0 or t.ksplit == ks, (req, t)
                    assert plan(M, N, K, WFMT_W8B, t)[0] == t, (req, t)


@pytest.mark.gpu
def test_w8b_divided_rows_with_the_split_left_open():
    """A request that divides the rows and leaves the split to the planner, at a
    size where the undivided launch would split K: float64 (one bf16 rounding of
    fp32 sums), and the explicit one-split request bit for bit."""
    from acorninfer_amd.ops.quant_gemm import Tiling
    M, N, K = 300, 512, 1024
    lin, q, scale = _w8b(N, K, 5)
    x = torch.randn(M, K, generator=torch.Generator().manual_seed(6)).bfloat16().cuda()
    assert lin.plan(M, Tiling(DENSE_RT, 0, 0, 0, 0))[0].ksplit > 1
    want = x.double() @ (q.cuda().double() * scale.cuda().double()[:, None]).t()
    out = _launch8(lin, x, Tiling(DENSE_RT, 0, 0, 0, 1), False)
    assert ((out.double() - want).norm() / want.norm()) < 4e-3
    assert torch.equal(out, _launch8(lin, x, Tiling(DENSE_RT, 0, 0, 1, 1), False))


@pytest.mark.parametrize("N,K", [(6144, 4096), (4096, 4096), (24576, 4096), (4096, 12288),
                                 (1024, 3072), (1152, 4096), (2048, 384)])
def test_one_split_asked_for_is_one_split_on_the_blocks(N, K):
    """ksplit 1 with all else left open is a request, whose caller may hold no
    workspace: it is planned as one split at every row count (no GPU)."""
    from acorninfer_amd._lib import WFMT_BF16, WFMT_BF16B, WFMT_W4B, WFMT_W8B
    from acorninfer_amd.ops.quant_gemm import Tiling, plan
    for fmt in (WFMT_W8B, WFMT_W4B, WFMT_BF16B, WFMT_BF16):
        for M in (1, 8, 16, 17, 64, 255, 256, 300, 512, 1000, 2000, 8192):
            if (fmt == WFMT_W4B and K % 512) or (fmt == WFMT_BF16 and M <= 16):
                continue                   # no such blocks; K in pieces that fit the LDS
            t, _ = plan(M, N, K, fmt, Tiling(0, 0, 0, 1, 0))
            assert t.ksplit == 1, (fmt, M, t)


def test_int4_rows_without_an_int4_form_take_the_dequantise_route():
    """W4B weights of another row count than 128s have no int4 form above 64
    rows, the fused SwiGLU none above 16: a caller that holds a bf16 workspace gets
    the dequantise route from 512 rows on (no GPU)."""
    from acorninfer_amd._lib import WFMT_W4B
    from acorninfer_amd.models.qwen3 import DEQUANT_M_MIN, DEQUANT_RT, QLinear
    for N, K in ((1040, 512), (272, 1024), (576, 1024)):
        lin = QLinear(WFMT_W4B, None, N, K, None)
        for M in (512, 600, 703, 704, 5000):
            assert lin.plan(M, workspace=True)[0].rt == DEQUANT_RT
        with pytest.raises(NotImplementedError):
            lin.plan(600)
    for N in (1088, 1152):                            # the fused SwiGLU has no int4 form either
        for M in (512, 703, 704):
            lin = QLinear(WFMT_W4B, None, N, 512, None)
            assert lin.swiglu_plan(M, workspace=True)[0].rt == DEQUANT_RT
    assert lin.plan(DEQUANT_M_MIN - 1, workspace=True)[0].rt != DEQUANT_RT
    assert lin.plan(DEQUANT_M_MIN, workspace=True)[0].rt == DEQUANT_RT


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,swiglu", [(513, 272, 256, False), (300, 512, 1024, False),
                                          (600, 1056, 512, True)])
def test_w8b_large_m_operands_at_any_address(M, N, K, swiglu):
    """x one element and the weights one byte off their alignment, each and both
    (loads straight into LDS need 16 bytes): bit for bit the aligned launch, in
    bf16 and fp32, in one split and several."""
    from acorninfer_amd._lib import stream_ptr
    from acorninfer_amd.ops.quant_gemm import Tiling
    lin, _, _ = _w8b(N, K, 3 * N)
    lin.il16 = swiglu
    x = torch.randn(M, K, generator=torch.Generator().manual_seed(9)).bfloat16().cuda()
    xo = torch.empty(M * K + 1, dtype=x.dtype, device="cuda")[1:].view(M, K).copy_(x)
    w, wo = lin.w, torch.empty(N * K + 1, dtype=lin.w.dtype, device="cuda")[1:].view(lin.w.shape)
    wo.copy_(w)

    def outs(xs, ws):
        lin.w = ws
        if swiglu:
            act = torch.empty(M, N // 2, dtype=torch.bfloat16, device="cuda")
            lin.launch_swiglu(xs, M, lin.swiglu_plan(M)[0], act, stream_ptr())
            return [act]
        return [_launch8(lin, xs, Tiling(DENSE_RT, 0, 0, ks, 0), ks == 2) for ks in (1, 2)]
    want = outs(x, w)
    for xs, ws in ((xo, w), (x, wo), (xo, wo)):
        for a, b in zip(outs(xs, ws), want):
            assert torch.equal(a, b)


def test_default_tilings_where_one_split_or_eight_lose():
    """Sizes at which the general default loses, measured (no GPU): large int4
    weights past 8 rows keep several splits, small ones and fewer rows one; a bf16
    split of 128-row x tiles keeps 256 k."""
    from acorninfer_amd._lib import WFMT_BF16, WFMT_W4B
    from acorninfer_amd.ops.quant_gemm import plan
    for N, K in ((6144, 4096), (4096, 4096), (4096, 12288)):
        assert plan(8, N, K, WFMT_W4B)[0].ksplit == 1
        assert all(plan(M, N, K, WFMT_W4B)[0].ksplit > 1 for M in (9, 16))
    assert plan(16, 4096, 1024, WFMT_W4B)[0].ksplit == 1
    for N, K, M in ((2048, 1024, 255), (1024, 1024, 200), (4096, 2048, 160)):
        t = plan(M, N, K, WFMT_BF16)[0]
        assert t.upw == 128 and K // t.ksplit >= 256, t
    assert plan(17, 151936, 4096, WFMT_BF16)[0].nw == 64
    assert plan(64, 151936, 4096, WFMT_BF16)[0].nw == 128
