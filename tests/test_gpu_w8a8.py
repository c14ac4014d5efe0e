"""GPU parity of the W8A8 tier (per-token activation quantisation + fp8 x fp8 GEMM) against the CPU oracle.

Reference path: tybok/policies/pi05/models/triton_prefill_mlp.py:26-166 (`quantize_activation`, `_w8a8_gemm`,
`make_fp8_mlp_forward`).  Codes and scales of the quantiser are compared bit for bit; GEMM outputs within the
tolerance stated for bf16 op outputs (rtol 2e-2 / atol 2e-2).
"""

import pytest
import torch

from oracle import ops as oops
from oracle.inputs import ffn_case, gemm_case

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


def _close(got, want, what):
    got = got.float().cpu()
    want = want.float().cpu()
    assert torch.isfinite(got).all(), f"{what}: non-finite output"
    err = (got - want).abs()
    bad = err > 2e-2 + 2e-2 * want.abs()
    assert not bad.any(), f"{what}: {int(bad.sum())} / {bad.numel()} outside tolerance, max |err| {err.max():.4g}"


@pytest.fixture(scope="module")
def tk():
    from tybok_amd import ops

    return ops


@pytest.mark.parametrize("m,k", [(1, 64), (50, 720), (712, 2048), (257, 16384), (33, 8)])
@pytest.mark.parametrize("mode", [0, 1])
def test_activation_quantisation_is_bit_exact(tk, m, k, mode):
    g = torch.Generator().manual_seed(m * 131 + k)
    x = (torch.randn(m, k, generator=g) * torch.logspace(-2, 2, m)[:, None]).to(BF16)
    if m > 2:
        x[2] = 0.0
    a8, sa = tk.quant_act_rows(x.cuda(), mode)
    want8, want_s = oops.quantize_activation_rows(x, "bf16" if mode else "fp32")
    assert torch.equal(sa.cpu(), want_s), "per-token scales differ"
    assert torch.equal(a8.cpu().view(torch.uint8), want8.view(torch.uint8)), "e4m3fn codes differ"


def test_activation_quantisation_of_a_strided_view(tk):
    g = torch.Generator().manual_seed(7)
    big = torch.randn(40, 256, generator=g).to(BF16)
    x = big[:, 64:192]
    a8, sa = tk.quant_act_rows(big.cuda()[:, 64:192], 0)
    want8, want_s = oops.quantize_activation_rows(x)
    assert torch.equal(sa.cpu(), want_s) and torch.equal(a8.cpu().view(torch.uint8), want8.view(torch.uint8))


@pytest.mark.parametrize("m,k,n", [(257, 64, 36), (256, 2048, 2048), (385, 96, 260), (300, 720, 2048), (712, 2048, 16384), (712, 16384, 2048), (100, 64, 512), (5, 128, 64)])
def test_w8a8_gemm_matches_oracle(tk, m, k, n):
    x, w8, sw = gemm_case(m, k, n)
    a8, sa = oops.quantize_activation_rows(x)
    want = oops.lin_w8a8(a8, sa, w8, sw)
    pw = tk.pack_fp8_weight(w8.cuda(), sw.cuda())
    got = tk.w8a8_gemm(a8.cuda(), sa.cuda(), pw)
    _close(got, want, f"w8a8 gemm M={m} K={k} N={n}")


@pytest.mark.parametrize("resid_dtype", [None, torch.float32, BF16])
@pytest.mark.parametrize("m,k,n", [(385, 96, 260), (300, 256, 36)])
def test_w8a8_gemm_row_segment_stores_respect_n_and_the_pitch(tk, m, k, n, resid_dtype):
    # 16-byte row segment stores into a column slice of a wider buffer: the tail segment is cut to N, nothing
    # past N is written, and both residual types go through the coalesced path
    x, w8, sw = gemm_case(m, k, n)
    a8, sa = oops.quantize_activation_rows(x)
    want = oops.lin_w8a8(a8, sa, w8, sw)
    pitch = (n + 15) // 8 * 8
    buf = torch.full((m, pitch), 7.0, dtype=BF16, device="cuda")
    resid = None
    if resid_dtype is not None:
        r = torch.randn(m, pitch, generator=torch.Generator().manual_seed(3)).to(resid_dtype)
        want = (want.float() + r[:, :n].float()).to(BF16)
        resid = r.cuda()[:, :n]
    tk.w8a8_gemm(a8.cuda(), sa.cuda(), tk.pack_fp8_weight(w8.cuda(), sw.cuda()), resid=resid, out=buf[:, :n])
    _close(buf[:, :n], want, f"w8a8 gemm M={m} K={k} N={n} pitch={pitch}")
    assert bool((buf[:, n:] == 7.0).all()), "wrote past N"


def test_w8a8_gemm_exact_on_small_integers(tk):
    # integer-valued codes and power-of-two scales: every product and sum is exact in fp32, whatever the order --
    # a wrong pairing of k between the two operands of the matrix instruction cannot hide behind a tolerance
    g = torch.Generator().manual_seed(11)
    m, k, n = 130, 192, 96
    a = torch.randint(-3, 4, (m, k), generator=g).float()
    w = torch.randint(-2, 3, (n, k), generator=g).float()
    a8, w8 = a.to(torch.float8_e4m3fn), w.to(torch.float8_e4m3fn)
    sa = torch.exp2(torch.randint(-2, 3, (m,), generator=g).float())
    sw = torch.exp2(torch.randint(-2, 3, (n,), generator=g).float())
    want = ((a @ w.t()) * sa[:, None] * sw[None, :]).to(BF16)
    got = tk.w8a8_gemm(a8.cuda(), sa.cuda(), tk.pack_fp8_weight(w8.cuda(), sw.cuda()))
    assert torch.equal(got.cpu(), want)


@pytest.mark.parametrize("split", [1, 2, 5])
def test_w8a8_split_k_is_deterministic_and_matches(tk, split):
    x, w8, sw = gemm_case(300, 4096, 256)
    a8, sa = oops.quantize_activation_rows(x)
    pw = tk.pack_fp8_weight(w8.cuda(), sw.cuda())
    resid = torch.randn(300, 256, generator=torch.Generator().manual_seed(3)).to(BF16)
    a = tk.w8a8_gemm(a8.cuda(), sa.cuda(), pw, split_k=split, resid=resid.cuda())
    b = tk.w8a8_gemm(a8.cuda(), sa.cuda(), pw, split_k=split, resid=resid.cuda())
    assert torch.equal(a, b)
    want = (oops.lin_w8a8(a8, sa, w8, sw).float() + resid.float()).to(BF16)
    _close(a, want, f"w8a8 split_k={split}")


@pytest.mark.parametrize("mode", ["fp32", "bf16"])
@pytest.mark.parametrize("m,k,i,act", [(300, 256, 512, "silu"), (712, 2048, 16384, "gelu_tanh"), (64, 64, 32, "gelu_tanh")])
def test_w8a8_ffn_matches_oracle(tk, m, k, i, act, mode):
    x, wg8, sg, wu8, su, wd8, sd = ffn_case(m, k, i, seed=4)
    x = (x.float() * 1.5).to(BF16)
    want = oops.gated_ffn_w8a8(x, wg8, sg, wu8, su, wd8, sd, act, mode=mode)
    wgu = tk.pack_fp8_gate_up(wg8.cuda(), sg, wu8.cuda(), su)
    wd = tk.pack_fp8_weight(wd8.cuda(), sd)
    ws = tk.Workspace("cuda")
    got = tk.w8a8_gated_ffn(x.cuda(), wgu, wd, act, ws=ws, mode=mode)
    # Stage by stage on the library's own operands, so that no tolerance has to make room for a re-quantised row:
    # (1) the intermediate against the oracle's, plain tolerance; (2) its codes and scales are exactly the oracle's
    # quantisation of THAT intermediate; (3) the output against the oracle's down projection of THOSE codes, plain
    # tolerance, no outlier allowance.
    h_gpu, h8_gpu, sh_gpu = (t.cpu() for t in tk.w8a8_ffn_intermediates(ws, m, k, i))
    x8, sx = oops.quantize_activation_rows(x, mode)
    h_want = oops.act_fn(act, oops.lin_w8a8(x8, sx, wg8, sg)) * oops.lin_w8a8(x8, sx, wu8, su)
    _close(h_gpu, h_want, f"w8a8 ffn intermediate ({m},{k},{i}) {mode}")
    h8_want, sh_want = oops.quantize_activation_rows(h_gpu, mode)
    assert torch.equal(h8_gpu.view(torch.uint8), h8_want.view(torch.uint8)) and torch.equal(sh_gpu, sh_want)
    _close(got, oops.lin_w8a8(h8_gpu, sh_gpu, wd8, sd), f"w8a8 ffn down projection on the library's codes ({m},{k},{i}) {mode}")
    # End to end against the oracle's own chain: where the GPU's h differs from the oracle's by one bf16 step
    # (summation order of the gate / up products) in the element that sets a row's amax, that row's scale moves and
    # a few per cent of its codes re-round by one e4m3 step -- the stages above show that this is all there is to
    # it.  Here: at most 0.1 % of the outputs outside the plain tolerance, none farther than 2 % of the output range.
    got_c, want_c = got.float().cpu(), want.float()
    err = (got_c - want_c).abs()
    bad = err > 2e-2 + 2e-2 * want_c.abs()
    print(f"w8a8 ffn ({m},{k},{i}): {int(bad.sum())} / {bad.numel()} outside rtol/atol 2e-2, max |err| {err.max():.4g}, |y|max {want_c.abs().max():.4g}")
    assert bad.float().mean() <= 1e-3 and float(err.max()) <= 2e-2 * float(want_c.abs().max()) + 2e-2
    # with the residual
    got_r = tk.w8a8_gated_ffn(x.cuda(), wgu, wd, act, resid=x.cuda(), ws=ws, mode=mode)
    assert torch.equal(got_r.cpu(), (got.float().cpu() + x.float()).to(BF16))


@pytest.mark.parametrize("m,k,n", [(1, 16, 4), (257, 48, 36), (289, 144, 132), (319, 720, 388), (130, 2064, 260)])
@pytest.mark.parametrize("split", [0, 1, 2, 3])
def test_w8a8_gemm_edges_exact_on_small_integers(tk, m, k, n, split):
    # what the shapes pick by themselves (64 x 128 blocks; every shape of block: the next test):
    # k ranges that end inside a round of 128 (and, split, on any tile of 32), one past a row tile, N % 8 == 4; a8 is a column
    # slice of a wider buffer of NaN codes.  Integer codes and power-of-two scales: exact whatever the order of summation.
    if split > 1 and (k + 31) // 32 < split:
        pytest.skip("fewer k tiles than splits")
    g = torch.Generator().manual_seed(m + k + n)
    a = torch.randint(-3, 4, (m, k), generator=g).float()
    w = torch.randint(-2, 3, (n, k), generator=g).float()
    wide = torch.full((m, (k + 31) // 16 * 16), 0x7F, dtype=torch.uint8)
    wide[:, :k] = a.to(torch.float8_e4m3fn).view(torch.uint8)
    sa = torch.exp2(torch.randint(-2, 3, (m,), generator=g).float())
    sw = torch.exp2(torch.randint(-2, 3, (n,), generator=g).float())
    r = torch.randint(-16, 17, (m, n), generator=g).to(BF16)
    y = ((a @ w.t()) * sa[:, None] * sw[None, :]).to(BF16)
    want = (y.float() + r.float()).to(BF16)
    pw = tk.pack_fp8_weight(w.to(torch.float8_e4m3fn).cuda(), sw.cuda())
    got = tk.w8a8_gemm(wide.cuda()[:, :k], sa.cuda(), pw, split_k=split, resid=r.cuda())
    assert torch.equal(got.cpu(), want)
    assert torch.equal(tk.w8a8_gemm(wide.cuda()[:, :k], sa.cuda(), pw, split_k=split).cpu(), y)


W8A8_TILES = (408, 414, 204, 604, 28)  # 128 x 256, 128 x 128, 64 x 128, 192 x 128 blocks; 64 x 256 with weights in registers, no K split


def _integers(g, top, *shape):
    return torch.randint(-top, top + 1, shape, generator=g).float()


def _codes_before_nan(a):
    m, k = a.shape
    wide = torch.full((m, (k + 31) // 16 * 16), 0x7F, dtype=torch.uint8)
    wide[:, :k] = a.to(torch.float8_e4m3fn).view(torch.uint8)
    return wide.cuda()[:, :k]


@pytest.mark.parametrize("tile", W8A8_TILES)
@pytest.mark.parametrize("k", [16, 48, 144, 720, 2064, 4112])
def test_every_w8a8_block_shape_exact_on_small_integers(tk, tile, k):
    # rows and columns one (four) past a block and short of one, one row alone; K inside a round, more rounds than the ring
    # holds; even and uneven splits; NaN codes behind K, residuals, a pitch that allows only 8-byte stores (N + 4) and one with
    # room behind N.  Exact: |sum| <= 6 * 4112 times powers of two, rounded once to bf16 each time.
    rows, cols = {414: (128, 128), 28: (64, 256)}.get(tile, (tile // 100 * 32, tile % 100 * 32))
    for m, n in ((rows + 1, cols + 4), (1, 4), (2 * rows - 31, 36), (rows, 2 * cols - 60)):
        g = torch.Generator().manual_seed(m + k + n)
        a, w = _integers(g, 3, m, k), _integers(g, 2, n, k)
        sa, sw = torch.exp2(_integers(g, 2, m)), torch.exp2(_integers(g, 2, n))
        r = _integers(g, 16, m, n).to(BF16)
        y = ((a @ w.t()) * sa[:, None] * sw[None, :]).to(BF16)
        full = (y.float() + r.float()).to(BF16)
        pw = tk.pack_fp8_weight(w.to(torch.float8_e4m3fn).cuda(), sw.cuda())
        x, sac, rc = _codes_before_nan(a), sa.cuda(), r.cuda()
        for split in (1,) if tile == 28 else (s for s in (1, 2, 3, 5) if s <= (k + 31) // 32):
            assert torch.equal(tk.many_rows_gemm(x, pw, tile, sa=sac, split_k=split).cpu(), y), (m, n, split)
            for pitch in (n + 4, (n + 15) // 8 * 8):
                buf = torch.full((m, pitch), 7.0, dtype=BF16, device="cuda")
                tk.many_rows_gemm(x, pw, tile, sa=sac, split_k=split, resid=rc, out=buf[:, :n])
                assert torch.equal(buf[:, :n].cpu(), full) and bool((buf[:, n:] == 7.0).all()), (m, n, split, pitch)
            assert torch.equal(tk.many_rows_gemm(x, pw, tile, sa=sac, split_k=split, resid=rc.float()).cpu(), full), (m, n, split)


@pytest.mark.parametrize("m,k,n", [(1000, 48, 8196), (961, 1536, 8192), (960, 1536, 8192), (1000, 1552, 8192), (1025, 2048, 7940), (1024, 2048, 8192)])
def test_w8a8_gemm_where_the_rules_change_kernels(tk, m, k, n):
    # short K over a full generation of 64 x 256 blocks (512 on 256 CUs; 1536 columns, 2048 from 1025 rows on) and one step beside it
    g = torch.Generator().manual_seed(m + k)
    a, w = _integers(g, 2, m, k).cuda(), _integers(g, 1, n, k).cuda()
    sa, sw = torch.exp2(_integers(g, 1, m)).cuda(), torch.exp2(_integers(g, 1, n)).cuda()
    got = tk.w8a8_gemm(a.to(torch.float8_e4m3fn), sa, tk.pack_fp8_weight(w.to(torch.float8_e4m3fn), sw))
    assert torch.equal(got, ((a @ w.t()) * sa[:, None] * sw[None, :]).to(BF16))


@pytest.mark.parametrize("act", ["gelu_tanh", "silu"])
@pytest.mark.parametrize("m,k,i", [(1, 16, 32), (65, 80, 96), (129, 720, 160), (193, 2064, 32), (257, 144, 544)])
def test_every_w8a8_block_shape_gives_the_same_gated_bits(tk, m, k, i, act):
    # exact gate and up sums whatever the shape and the split, then one epilogue: the same bits from all of them
    g = torch.Generator().manual_seed(m + k + i)
    a, wg, wu = _integers(g, 3, m, k), _integers(g, 2, i, k), _integers(g, 2, i, k)
    sa, sg, su = torch.exp2(_integers(g, 1, m)), torch.exp2(_integers(g, 1, i) - 5), torch.exp2(_integers(g, 1, i) - 5)
    pre, up = ((a @ w.t()) * sa[:, None] * s for w, s in ((wg, sg), (wu, su)))
    want = (oops.act_fn(act, pre.to(BF16)).float() * up.to(BF16).float()).to(BF16)
    wgu = tk.pack_fp8_gate_up(wg.to(torch.float8_e4m3fn).cuda(), sg, wu.to(torch.float8_e4m3fn).cuda(), su)
    x, sac = _codes_before_nan(a), sa.cuda()
    first = None
    for tile in W8A8_TILES:
        for split in (1,) if tile == 28 or k < 64 else (1, 2):
            buf = torch.full((m, i + 4), 7.0, dtype=BF16, device="cuda")
            got = tk.many_rows_gemm(x, wgu, tile, sa=sac, split_k=split, act=act)
            tk.many_rows_gemm(x, wgu, tile, sa=sac, split_k=split, act=act, out=buf[:, :i])
            first = got if first is None else first
            assert torch.equal(got, first) and torch.equal(buf[:, :i], first) and bool((buf[:, i:] == 7.0).all()), (tile, split)
    _close(first, want, f"w8a8 gated M={m} K={k} I={i}")


def test_w8a8_rows_more_than_4_gib_of_lane_offset_apart(tk):
    m, k, n, ld = 9, 208, 96, 1 << 30  # (eight rows share a load's scalar base and 32-bit lane offsets otherwise)
    g = torch.Generator().manual_seed(3)
    a = torch.randint(-3, 4, (m, k), generator=g).float()
    w = torch.randint(-2, 3, (n, k), generator=g).float()
    far = torch.empty((m - 1) * ld + k, dtype=torch.uint8, device="cuda").as_strided((m, k), (ld, 1))
    far.copy_(a.to(torch.float8_e4m3fn).view(torch.uint8))
    pw = tk.pack_fp8_weight(w.to(torch.float8_e4m3fn).cuda(), torch.ones(n).cuda())
    assert torch.equal(tk.w8a8_gemm(far, torch.ones(m).cuda(), pw).cpu(), (a @ w.t()).to(BF16))


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("k", [8, 2048, 2056, 4104, 8200, 16384])
def test_activation_quantisation_at_the_edges_of_the_quotient(tk, k, mode):
    # every piece count of a row, a row of all finite bf16 magnitudes, signed zeros, scales at and beyond the range in which
    # the quotient comes from the reciprocal; whole rows of one scale each (scales that round to 0: the next test).
    # Infinities and NaN: as the division gives them.
    g = torch.Generator().manual_seed(k)
    rows = [torch.randn(k, generator=g) * 2.0**e for e in (-110, -100, -81, -72, -71, -70, -20, 0, 20, 70, 88, 89, 90, 100, 118)]
    codes = 0x7F7F - torch.arange(k, dtype=torch.int32) * 7 % 0x7F00
    rows.append(codes.to(torch.int16).view(BF16).float())
    rows.append(torch.where(torch.arange(k) % 3 == 0, -0.0, torch.randn(k, generator=g)))
    x = torch.stack(rows).to(BF16)
    a8, sa = tk.quant_act_rows(x.cuda(), mode)
    want8, want_s = oops.quantize_activation_rows(x, "bf16" if mode else "fp32")
    assert torch.equal(sa.cpu(), want_s) and torch.equal(a8.cpu().view(torch.uint8), want8.view(torch.uint8))
    odd = torch.randn(3, k, generator=g).to(BF16)
    odd[0, 1], odd[1, 2], odd[2, 3], odd[2, 4] = float("inf"), float("-inf"), float("nan"), float("inf")
    a8, sa = tk.quant_act_rows(odd.cuda(), mode)
    s = odd.float().abs().nan_to_num(0.0, float("inf")).amax(1) / 448  # (a maximum passes NaN by)
    q = odd.float() / s[:, None]
    got = a8.cpu().view(torch.float8_e4m3fn).float()
    assert torch.equal(sa.cpu(), s) and torch.equal(got.isnan(), q.isnan()) and bool((got[~q.isnan()] == 0).all())


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("k", [8, 2056, 16384])
def test_activation_quantisation_of_rows_whose_scale_rounds_to_zero(tk, k, mode):
    # amax / 448 as a bf16 value: 0 up to 448 * 2^-134 (a tie goes to the even 0), the smallest subnormal from the next
    # bf16 above; a scale of 0 gives zero codes (+0, whatever the signs) and a finite product.  In fp32 no bf16 row's does.
    g = torch.Generator().manual_seed(k)
    sign = torch.where(torch.rand(k, generator=g) < 0.5, -1.0, 1.0)
    top = 448 * 2.0**-134
    rows = [top * torch.rand(k, generator=g) * sign, sign * 2.0**-133, torch.where(torch.arange(k) == k - 1, top, 0.0), torch.where(torch.arange(k) == 1, top * (1 + 2**-7), -0.0)]
    x = torch.stack([*rows, torch.randn(k, generator=g) * 2.0**-126, torch.zeros(k), -torch.zeros(k)]).to(BF16)
    a8, sa = tk.quant_act_rows(x.cuda(), mode)
    want8, want_s = oops.quantize_activation_rows(x, "bf16" if mode else "fp32")
    assert torch.equal(sa.cpu(), want_s) and torch.equal(a8.cpu().view(torch.uint8), want8.view(torch.uint8))
    if mode:
        assert bool((sa[:3] == 0).all()) and bool((a8.view(torch.uint8)[:3] == 0).all()) and float(sa[3]) > 0
