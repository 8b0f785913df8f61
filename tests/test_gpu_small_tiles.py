"""GPU tests of the conv tiles that calls below a full chip take, at the edges
of their tiles and of the rules that choose them, against the fp64 definition
on the same rounded operands:

* conv_rows_kernel (16-bit activations): 1, 2 or 4 row blocks per wave, by the
  number of 16-row x 64-channel blocks (256, 512, 2,048);
* conv_f32_kernel: tiles of 32, 64 or 128 rows and channels;
* linear_skinny_rows_kernel: rows around a wave's 64, channels around its 128
  bytes;
* the halo-staged tiles at channel counts that keep few rows on them.

bf16 / f16 outputs are held to half an ulp of the output plus the f32 bound;
f32 outputs to 2e-5: the sum of 27 * Cin products in f32, whose error in any
order is below (27 * Cin) * 2^-24 of the sum of magnitudes and in practice near
its square root (about 2e-6 here)."""
import numpy as np
import pytest
import torch

from bevy_synth_amd import flex_gmm as F
from bevy_synth_amd import synth
from tests.test_gpu_plan import bf16_dev, cluster_coords, dev, ocfg, rbf
from tests.tolerance import assert_close

pytestmark = pytest.mark.gpu

TOL = {torch.float32: 2e-5, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11 + 2e-5}


def shell(n, seed=0):
    """n rows of a thick shell in (b, x, y, z) order."""
    r = 6.0
    while True:
        c = synth.sphere_shell_coords(int(2 * r) + 8, r, 1.5, (r + 4,) * 3)
        if len(c) >= n:
            return np.ascontiguousarray(c[:n])
        r *= 1.3


def conv_case(oracle, n, cin, cout, dtype, w="same", planned=False, ln=False, residual=False, groups=1, out=None,
              kernel=(3, 3, 3), coords=None, n_q=None, rows=None):
    rng = np.random.default_rng((n or 0) + 7 * cin + cout)
    cfg = F.SparseSubmConvConfig(cin, cout, *kernel, groups=groups)
    coords = shell(n) if coords is None else coords
    n = len(coords)
    K = F.kernel_rows(cfg)
    f16 = dtype == torch.float16
    rnd = (lambda a: a) if dtype == torch.float32 else (oracle.f16_round if f16 else rbf)
    to = dev if dtype == torch.float32 else ((lambda a: dev(a).half()) if f16 else bf16_dev)
    x = rnd(synth.normal_f32(rng, (n, cin)))
    cg = cin // groups
    if w == "i8":
        q, scale = synth.int8_weight(rng, cout, K, cg)
        scale = (scale / np.sqrt(K * cg / 3)).astype(np.float32)
        wv, wd, sd = q.astype(np.float64) * scale[:, None, None], dev(q), dev(scale)
    else:
        wv = rnd(synth.conv_weight(rng, cout, K, cg, 1 / np.sqrt(K * cg)))
        wd, sd = to(wv), None
    b = synth.normal_f32(rng, cout, 0.1)
    nbr = F.neighbor_rows_tensor_from_coords_tensor(cfg, dev(coords), query_rows=n_q)
    n_q = n if n_q is None else n_q
    od = dtype if out is None else out
    res = rbf(synth.normal_f32(rng, (n_q, cout))) if residual else None  # exact in bf16 and f32
    res = oracle.f16_round(res) if residual and f16 else res
    plan = F.build_conv_plan(cfg, dev(coords), nbr) if planned else None
    packed = F.pack_conv_weight(cfg, wd) if planned else None
    got = F.sparse_subm_conv_forward(cfg, to(x), nbr, wd, dev(b), sd, out_dtype=od,
                                     residual=None if res is None else dev(res).to(od), layer_norm=ln, silu=ln,
                                     plan=plan, packed_weight=packed).float().cpu().numpy()
    if planned:
        F.conv_plan_check(plan)
    m = nbr.cpu().numpy()
    sel = np.arange(n_q) if rows is None else rows(n_q)
    exp = oracle.conv_gemm_f64(ocfg(oracle, cfg), np.asarray(wv, np.float32), b, x, m[sel]) if w != "i8" else \
        oracle.conv_gemm_f64(ocfg(oracle, cfg), q, b, x, m[sel], w_scale=scale)
    if ln:
        exp = exp - exp.mean(1, keepdims=True)
        exp = exp / np.sqrt((exp * exp).mean(1, keepdims=True) + 1e-6)
        exp = exp / (1 + np.exp(-exp))
    if res is not None:
        exp = exp + res[sel]
    assert_close(got[sel], exp, TOL[od] if not ln else max(TOL[od], 4e-5), f"{n} rows {cin}->{cout}")


# rows at and past the ends of 16-, 32- and 64-row tiles, and on both sides of
# the rule's block counts (64 output channels: one block per 16 rows)
@pytest.mark.parametrize("n", [1, 15, 17, 63, 65, 4096, 4097, 8192, 8193, 32768, 32769])
@pytest.mark.parametrize("planned", [False, True])
def test_rows_tile_edges(oracle, n, planned):
    conv_case(oracle, n, 32, 64, torch.bfloat16, planned=planned, residual=n % 2 == 1,
              rows=lambda q: np.unique(np.r_[0:min(q, 300), max(0, q - 300):q]))


@pytest.mark.parametrize("dtype,w,cin,cout,groups,ln,out,n,planned", [
    (torch.float16, "same", 64, 96, 1, True, None, 1000, True),     # LayerNorm over two 64-channel columns
    (torch.bfloat16, "same", 64, 128, 1, True, None, 5000, False),
    (torch.bfloat16, "same", 32, 100, 1, True, torch.float32, 9001, True),
    (torch.bfloat16, "i8", 96, 24, 1, False, None, 700, False),     # int8 weights widened in registers
    (torch.bfloat16, "i8", 64, 72, 1, False, torch.float32, 700, True),
    (torch.float16, "same", 64, 7, 1, False, torch.float32, 333, False),  # scalar stores
    (torch.bfloat16, "same", 128, 192, 2, False, None, 777, True),  # groups
    (torch.bfloat16, "same", 128, 192, 2, False, None, 777, False),
    (torch.bfloat16, "same", 512, 256, 1, False, None, 3000, True),
])
def test_rows_tile_forms(oracle, dtype, w, cin, cout, groups, ln, out, n, planned):
    conv_case(oracle, n, cin, cout, dtype, w, planned, ln, not ln, groups, out)


@pytest.mark.parametrize("cin,cout,ln", [(32, 64, False), (96, 128, True), (64, 200, False)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_rows_tile_row_alone(cin, cout, ln, dtype):
    """A row's value, in every bit, is the one it has with no other row using
    any offset: which rows share its block does not enter its sum."""
    n = 90
    rng = np.random.default_rng(cin)
    nbr = np.where(rng.random((n, 27)) < 0.4, -1, rng.integers(0, n, (n, 27))).astype(np.int32)
    x, w = dev(synth.normal_f32(rng, (n, cin))).to(dtype), dev(synth.conv_weight(rng, cout, 27, cin, 0.05)).to(dtype)
    cfg = F.SparseSubmConvConfig(cin, cout)

    def conv(m):
        return F.sparse_subm_conv_forward(cfg, x, dev(m), w, layer_norm=ln, out_dtype=torch.float32)
    together = conv(nbr)
    for r in (0, 17, n - 1):
        alone = np.full_like(nbr, -1)
        alone[r] = nbr[r]
        assert torch.equal(conv(alone)[r], together[r]), r


@pytest.mark.parametrize("n,cin,cout,groups,ln,kernel,out", [
    (1, 16, 64, 1, False, (3, 3, 3), None),
    (31, 16, 24, 1, True, (3, 3, 3), None),
    (33, 48, 33, 1, False, (3, 3, 3), None),      # an odd slice count in the two-slice stages
    (6144, 32, 128, 1, True, (3, 3, 3), None),    # 192 tiles of 64 x 64: the last on 32 x 32
    (6145, 32, 128, 1, True, (3, 3, 3), None),    # and the first past it
    (12289, 16, 65, 1, False, (3, 1, 1), None),
    (28672, 16, 128, 1, True, (3, 3, 1), None),   # 224 tiles of 128 x 128
    (28545, 16, 100, 1, False, (3, 3, 1), None),
    (3000, 32, 128, 1, True, (3, 3, 3), torch.bfloat16),  # LayerNorm stays in the tile: no workspace
    (900, 64, 96, 2, False, (3, 3, 3), None),
    (500, 64, 129, 1, False, (1, 1, 1), None),
    (40, 16, 40, 1, False, (2, 4, 4), None),      # 32 offsets
])
def test_f32_tile_edges(oracle, n, cin, cout, groups, ln, kernel, out):
    conv_case(oracle, n, cin, cout, torch.float32, ln=ln, residual=True, groups=groups, kernel=kernel, out=out,
              rows=lambda q: np.unique(np.r_[0:min(q, 400), max(0, q - 400):q]))


# on both sides of the row counts up to which f32 stages a LayerNorm's rows
# through the output
@pytest.mark.parametrize("n,c", [(600, 64), (12288, 64), (12289, 64), (600, 128), (28544, 128), (28545, 128)])
@pytest.mark.parametrize("linear", [False, True])
def test_f32_layer_norm_residual_in_place(n, c, linear):
    """The output may be the residual's own buffer."""
    rng = np.random.default_rng(n + c)
    x, b, res = (dev(synth.normal_f32(rng, s)) for s in ((n, c), (c,), (n, c)))
    kw = dict(layer_norm=True, silu=True)
    if linear:
        w = dev(synth.normal_f32(rng, (c, c), 0.1))

        def call(r, out):
            return F.linear_forward(x, w, b, residual=r, out=out, **kw)
    else:
        cfg = F.SparseSubmConvConfig(c, c)
        nbr = F.neighbor_rows_tensor_from_coords_tensor(cfg, dev(shell(n)))
        w = dev(synth.conv_weight(rng, c, 27, c, 0.05))

        def call(r, out):
            return F.sparse_subm_conv_forward(cfg, x, nbr, w, b, residual=r, out=out, **kw)
    apart, buf = call(res, None), res.clone()
    call(buf, buf)
    # one sum order either way; the row kernel and the tile add LayerNorm's
    # statistics in different orders
    assert_close(buf.cpu().numpy(), apart.cpu().numpy(), 4e-5)


@pytest.mark.parametrize("n,c,dtype,w8,ln", [
    (300, 64, torch.float32, False, False), (6001, 128, torch.float32, False, False),
    (60000, 128, torch.float32, False, False), (600, 128, torch.float32, False, True),
    (300, 128, torch.bfloat16, False, True), (3000, 256, torch.float16, False, False),
    (45000, 256, torch.bfloat16, False, False),   # 176 tiles of 256 x 256
    (5000, 128, torch.bfloat16, True, False)])
def test_linear_over_its_input(n, c, dtype, w8, ln):
    """A linear whose row of output channels lies in one tile may write over
    its input, whatever the number of rows."""
    rng = np.random.default_rng(n)
    x = dev(synth.normal_f32(rng, (n, c))).to(dtype)
    w, b, scale = dev(synth.normal_f32(rng, (c, c), 0.1)).to(dtype), dev(synth.normal_f32(rng, c)), None
    if w8:
        q, scale = synth.int8_weight(rng, c, 1, c)
        w, scale = dev(q.reshape(c, c)), dev(scale)
    exp = x.double() @ (w.double() * (scale[:, None] if w8 else 1)).T + b.double()
    if ln:
        exp = torch.nn.functional.layer_norm(exp, (c,), eps=1e-6)
    buf = x.clone()
    assert F.linear_forward(buf, w, b, scale, layer_norm=ln, out=buf, out_dtype=dtype) is buf
    assert_close(buf.double().cpu().numpy(), exp.cpu().numpy(), max(TOL[dtype], 4e-5))


def test_f32_tile_isolated_rows(oracle):
    """Rows without any neighbour but one offset, and a map of -1 only."""
    cfg = F.SparseSubmConvConfig(16, 48)
    rng = np.random.default_rng(3)
    x, w, b = synth.normal_f32(rng, (70, 16)), synth.conv_weight(rng, 48, 27, 16, 0.1), synth.normal_f32(rng, 48)
    nbr = np.full((70, 27), -1, np.int32)
    got = F.sparse_subm_conv_forward(cfg, dev(x), dev(nbr), dev(w), dev(b)).cpu().numpy()
    assert np.array_equal(got, np.broadcast_to(b, got.shape))
    nbr[69, 26] = 3
    got = F.sparse_subm_conv_forward(cfg, dev(x), dev(nbr), dev(w), dev(b)).cpu().numpy()
    assert_close(got, oracle.conv_gemm_f64(ocfg(oracle, cfg), w, b, x, nbr), TOL[torch.float32])


@pytest.mark.parametrize("rows,cin,cout,dtype", [
    (1, 8, 8, torch.float16), (63, 64, 1, torch.bfloat16), (64, 72, 8, torch.bfloat16), (65, 4, 8, torch.float32),
    (129, 36, 5, torch.float32), (1000, 136, 7, torch.float16)])
def test_skinny_rows_edges(rows, cin, cout, dtype):
    rng = np.random.default_rng(rows + cin)
    x = dev(synth.normal_f32(rng, (rows, cin))).to(dtype)
    w, b = synth.normal_f32(rng, (cout, cin)), synth.normal_f32(rng, cout)
    got = F.linear_skinny(x, dev(w), dev(b)).cpu().numpy()
    assert_close(got, x.double().cpu().numpy() @ w.T.astype(np.float64) + b, TOL[torch.float32])


def test_skinny_more_rows_than_a_launch_has_threads():
    rows, cin = 2**32 + 3, 8  # 69 GB in, 17 GB out
    if torch.cuda.mem_get_info()[0] < 100 << 30:
        pytest.skip("needs 86 GB of free device memory")
    x = torch.empty((rows, cin), dtype=torch.float16, device="cuda")
    w = dev(np.arange(1, cin + 1, dtype=np.float32).reshape(1, cin))
    at = torch.tensor([0, 2**31, 2**32 - 1, 2**32, rows - 1], device="cuda")
    for i, r in enumerate(at.tolist()):
        x[r] = i + 1
    got = F.linear_skinny(x, w)[at].cpu().numpy().ravel()
    del x
    torch.cuda.empty_cache()
    assert np.array_equal(got, 36.0 * np.arange(1, 6))


# Cout a multiple of 8 (16-byte stores), of 4, of neither
@pytest.mark.parametrize("cout,form", [(1024, "plain"), (640, "residual"), (1028, "residual"), (1030, "residual")])
def test_halo_tiles_few_rows(oracle, cout, form):
    """Enough output channels that few rows stay on the halo-staged tiles:
    tiles over the LDS budget, mixed with others, and a partial last tile."""
    coords = cluster_coords(1300)
    extra = shell(4100).copy()
    extra[:, 1] += 200
    centres, rest = coords[:1300], coords[1300:]
    both = np.concatenate([centres, extra, rest])
    conv_case(oracle, None, 32, cout, torch.bfloat16, planned=True, residual=form == "residual", coords=both,
              n_q=1300 + len(extra), rows=lambda q: np.unique(np.r_[0:300, 1200:1500, q - 300:q]))
