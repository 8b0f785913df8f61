"""GPU tests of the persistent 256 x 256 tile of the dense linear
(dense_tile_kernel, from 160 tiles on) at its edges: a last row tile of one row,
a last column tile that is not full, the shortest ring (4 k-steps, 8 with child
lists), one, two and five tiles per workgroup, f32 output, the epilogue's forms;
child lists of very different lengths, one of them empty.

Against the float64 product of the same rounded operands: bf16 / f16 outputs to
half an ulp (2^-9, 2^-12 of the value; the bounds below leave a factor of two)
plus the f32 sum's error; f32 outputs to 2e-5 (a sum of Cin <= 544 products in
f32, whose error is near sqrt(Cin) 2^-24, about 2e-6)."""
import ctypes

import numpy as np
import pytest
import torch

from bevy_synth_amd import _capi
from bevy_synth_amd import decoder as D
from bevy_synth_amd import flex_gmm as F
from tests.test_gpu_plan import dev
from tests.test_gpu_small_tiles import TOL, shell
from tests.tolerance import assert_close

pytestmark = pytest.mark.gpu


def randn(shape, seed, scale=1.0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn(shape, generator=g, device="cuda") * scale


@pytest.mark.parametrize("rows,cin,cout,dtype,out,silu,residual", [
    (10241, 128, 1024, torch.bfloat16, torch.bfloat16, False, False),  # 164 tiles, 4 k-steps
    (10495, 128, 1024, torch.float16, torch.float32, True, True),      # 164, last row tile one row short
    (20481, 160, 488, torch.bfloat16, torch.float32, False, True),     # 162, last column tile 232 wide
    (40961, 192, 248, torch.float16, torch.float16, True, True),       # 161, 248 wide
    (10241, 544, 2560, torch.bfloat16, torch.bfloat16, True, False),   # 410, above 512 channels
    (70000, 128, 1024, torch.bfloat16, torch.bfloat16, False, True),   # 1,096: five rounds
])
def test_dense_tile_edges(rows, cin, cout, dtype, out, silu, residual):
    x, w = randn((rows, cin), 1).to(dtype), randn((cout, cin), 2, cin ** -0.5).to(dtype)
    b = randn((cout,), 3)
    res = randn((rows, cout), 4).to(out) if residual else None
    got = F.linear_forward(x, w, b, out_dtype=out, silu=silu, residual=res)
    exp = x.double() @ w.double().T + b.double()
    if silu:
        exp = exp * torch.sigmoid(exp)
    if residual:
        exp = exp + res.double()
    assert_close(got.double().cpu().numpy(), exp.cpu().numpy(), TOL[out], f"{rows} rows {cin}->{cout}")


@pytest.mark.parametrize("n,cin,cout,dtype", [
    (20001, 256, 256, torch.bfloat16), (12000, 288, 512, torch.float16),
    # the row-block tile's limit of 2,048 blocks over all children, and lists
    # that stay below it past that
    (1024, 256, 256, torch.bfloat16), (1025, 256, 256, torch.bfloat16), (3900, 64, 128, torch.float16)])
def test_dense_tile_child_lists(n, cin, cout, dtype):
    """Children of 0 (always), 3 (never), 7 (one parent), the rest at random;
    equal in every bit to the linear over all children."""
    parents = dev(shell(n))
    rng = np.random.default_rng(n)
    on = rng.random((n, 8)) < [1, 0.2, 0.5, 0, 0.9, 0.5, 0.4, 0]
    on[n - 1, 7] = True
    mask = dev(on.astype(np.uint8))
    x, w = randn((n, cin), 5).to(dtype), randn((8 * cout, cin), 6, cin ** -0.5).to(dtype)
    layer = D.ConvLayer(F.SparseSubmConvConfig(cin, 8 * cout, 1, 1, 1), w.reshape(8 * cout, 1, cin),
                        randn((8 * cout,), 7))
    _, got, idx = D.transposed_upsample(parents, x, layer, mask)
    _, every, _ = D.transposed_upsample(parents, x, layer, mask, active_only=False)
    full = (x.double() @ w.double().T + layer.bias.double()).reshape(n * 8, cout)
    assert_close(got.double().cpu().numpy(), full[torch.from_numpy(np.flatnonzero(on)).cuda()].cpu().numpy(), TOL[dtype])
    assert torch.equal(got, every)


@pytest.mark.parametrize("n,cout", [(1000, 128), (8000, 128), (30000, 256)])  # row blocks, dense_gemm, dense_tile
def test_child_list_of_another_size(n, cout):
    """Through the C ABI, a linear child plan built for fewer parents: nothing
    is written, and the plan's check reports it."""
    on = np.random.default_rng(n).random((n, 8)) < 0.5

    def lists(rows):
        _, _, child_rows = F.subdivision_build_indexed(dev(shell(n)[:rows]), mask=dev(on[:rows].astype(np.uint8)))
        return child_rows, F.build_linear_child_plan(child_rows, int(on[:rows].sum())).buf
    child_rows, own = lists(n)
    other = torch.zeros_like(own)
    short = lists(n - 300)[1]
    other[:len(short)] = short
    x, w = randn((n, 256), 5).bfloat16(), randn((8 * cout, 256), 6, 1 / 16).bfloat16()
    out = torch.full((int(on.sum()), cout), 7.0, dtype=torch.bfloat16, device="cuda")
    epi = _capi.ScConvEpilogue()
    epi.child_rows, epi.n_child_rows = ctypes.c_void_p(child_rows.data_ptr()), len(out)
    lib, stream = _capi.load(), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)

    def call(plan):
        p = [ctypes.c_void_p(t.data_ptr()) for t in (x, w, out, plan)]
        assert lib.sc_linear_forward_child_planned(1, p[0], n, 256, 8 * cout, 1, p[1], None, None, ctypes.byref(epi),
                                                   1, p[2], p[3], stream) == 0
        return lib.sc_conv_plan_check(p[3], stream)
    assert call(other) == 2 and (out == 7.0).all()
    assert call(own) == 0 and not (out == 7.0).all()
