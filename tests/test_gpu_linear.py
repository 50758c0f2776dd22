"""GPU parity of the fused Linear + bias + exact-GELU kernel (sah_linear).

Reference: the same op in float64 on the CPU from the same 16-bit operands,
``F.gelu(F.linear(x, w, b), approximate="none")``, i.e. the FFN input half of
the official block (oracle/forward.py, official order).  The kernel rounds an
fp32 result once to the operand dtype, so it must pass the 16-bit gate of
oracle.compare (|err| <= 2e-2 or |err| <= 1e-2 |ref|) elementwise; the tests
also bound the error by a few output ulps, which a dropped bias, a wrong
activation or a transposed operand would far exceed.
"""

from __future__ import annotations


import pytest
import torch
import torch.nn.functional as F

from oracle.compare import parity_gate

pytestmark = pytest.mark.gpu


def _operands(rows, k, n, dtype, seed, device, bias=True):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(rows, k, generator=g)
    w = (torch.rand(n, k, generator=g) * 2 - 1) * (6.0 / (k + n)) ** 0.5 * 2.0
    b = 0.5 * torch.randn(n, generator=g) if bias else None
    cast = lambda t: None if t is None else t.to(dtype)  # noqa: E731
    x, w, b = cast(x), cast(w), cast(b)
    return (x, w, b), tuple(None if t is None else t.to(device) for t in (x, w, b))


def _reference(x, w, b, gelu):
    y = F.linear(x.double(), w.double(), None if b is None else b.double())
    return F.gelu(y, approximate="none") if gelu else y


def _check(reference, got, dtype, what):
    got = got.float().cpu()
    result = parity_gate(reference.float(), got, dtype)
    err = (got.double() - reference).abs()
    # at most a couple of output ulps (bf16: 2^-8 relative, fp16: 2^-11) plus
    # the fp32 accumulation error
    ulp = 2.0**-8 if dtype == torch.bfloat16 else 2.0**-11
    bound = 2 * ulp * reference.abs() + 1e-3
    print(f"{what}: max_abs={result.max_abs_error:.3g} failed={result.failed_elements}", flush=True)
    assert result.passed, f"{what}: {result.failed_elements} of {result.total_elements} outside the gate"
    assert bool((err <= bound).all()), f"{what}: error {float((err - bound).max()):.3g} above a 2-ulp bound"


@pytest.mark.parametrize(
    "rows,k,n",
    [(1, 512, 2048), (255, 512, 2048), (300, 1024, 4096), (1025, 1024, 4096), (513, 2048, 8192), (700, 4096, 1024)],
)
def test_linear_exact_gelu_matches_float64(gpu_device, rows, k, n):
    from solution.kernels.ffn import prevalidated_hip_linear_exact_gelu

    (x, w, b), (xd, wd, bd) = _operands(rows, k, n, torch.bfloat16, seed=rows + k, device=gpu_device)
    with torch.inference_mode():
        hidden, marker = prevalidated_hip_linear_exact_gelu(xd, wd, bd)
    torch.cuda.synchronize()
    assert marker == "hip_linear_exact_gelu" and hidden.shape == (rows, n) and hidden.dtype == torch.bfloat16
    _check(_reference(x, w, b, True), hidden, torch.bfloat16, f"gelu rows={rows} k={k} n={n}")


@pytest.mark.parametrize("bias", [True, False])
def test_plain_linear_and_fp16(gpu_device, bias):
    from solution.kernels.ffn import prevalidated_hip_linear

    for dtype in (torch.bfloat16, torch.float16):
        (x, w, b), (xd, wd, bd) = _operands(777, 1024, 1024, dtype, seed=5, device=gpu_device, bias=bias)
        with torch.inference_mode():
            out, marker = prevalidated_hip_linear(xd, wd, bd)
        torch.cuda.synchronize()
        assert marker == "hip_linear"
        _check(_reference(x, w, b, False), out, dtype, f"linear bias={bias} {dtype}")


def test_strided_rows_and_untouched_tail_through_the_c_abi(gpu_device):
    """x with a padded row stride, y with a wider row stride and rows past the
    last one: the kernel reads only valid rows and writes only [rows, n]."""

    from solution.kernels.hip import _library

    rows, k, n, ldx, ldy = 333, 1024, 2048, 1024 + 64, 2048 + 256
    (x, w, b), (_, wd, bd) = _operands(rows, k, n, torch.bfloat16, seed=9, device=gpu_device)
    xs = torch.full((rows, ldx), float("nan"), dtype=torch.bfloat16)
    xs[:, :k] = x
    xs = xs.to(gpu_device)
    sentinel = -7.0
    y = torch.full((rows + 5, ldy), sentinel, dtype=torch.bfloat16, device=gpu_device)
    lib = _library.load_library()
    status = lib.sah_linear(
        xs.data_ptr(), wd.data_ptr(), bd.data_ptr(), y.data_ptr(), rows, k, n, ldx, ldy,
        _library.dtype_code(torch.bfloat16), _library.SAH_ACTIVATION_GELU_EXACT, 256, 256, 64, 8, 2,
        _library.stream_handle(gpu_device),
    )
    _library.check_status(status, "sah_linear")
    torch.cuda.synchronize()
    y = y.cpu()
    _check(_reference(x, w, b, True), y[:rows, :n], torch.bfloat16, "strided")
    assert bool((y[:rows, n:] == sentinel).all()) and bool((y[rows:] == sentinel).all())


def test_long_sequence_ffn_input_rows_sample(gpu_device):
    """The C5 chunk's FFN input projection (2e5 rows x 1024 -> 4096): rows from
    every part of the output, including the partial last tile, against
    float64, and the full output finite."""

    from solution.kernels.ffn import prevalidated_hip_linear_exact_gelu

    rows, k, n = 200_000, 1024, 4096
    g = torch.Generator(device=gpu_device).manual_seed(3)
    xd = torch.randn(rows, k, device=gpu_device, dtype=torch.bfloat16, generator=g)
    wd = ((torch.rand(n, k, device=gpu_device, generator=g) * 2 - 1) * 0.0765).to(torch.bfloat16)
    bd = (0.5 * torch.randn(n, device=gpu_device, generator=g)).to(torch.bfloat16)
    with torch.inference_mode():
        hidden, _ = prevalidated_hip_linear_exact_gelu(xd, wd, bd)
    torch.cuda.synchronize()
    assert bool(torch.isfinite(hidden).all())
    pick = torch.cat([torch.arange(0, 256), torch.randint(0, rows, (256,), generator=torch.Generator().manual_seed(1)),
                      torch.arange(rows - 64, rows)])
    x, w, b = xd[pick.to(gpu_device)].cpu(), wd.cpu(), bd.cpu()
    _check(_reference(x, w, b, True), hidden[pick.to(gpu_device)], torch.bfloat16, "C5 ffn_in sample")


def test_ineligible_inputs_raise(gpu_device):
    from solution.kernels.ffn import can_use_hip_linear_exact_gelu, prevalidated_hip_linear_exact_gelu

    x = torch.zeros(4, 1000, dtype=torch.bfloat16, device=gpu_device)
    w = torch.zeros(2048, 1000, dtype=torch.bfloat16, device=gpu_device)
    b = torch.zeros(2048, dtype=torch.bfloat16, device=gpu_device)
    assert not can_use_hip_linear_exact_gelu(x, w, b)
    with pytest.raises(RuntimeError, match="ineligible"):
        prevalidated_hip_linear_exact_gelu(x, w, b)
    with pytest.raises(ValueError, match="launch"):
        prevalidated_hip_linear_exact_gelu(x, w, b, block_m=128)


@pytest.mark.parametrize("k", [64, 128, 192, 320])
@pytest.mark.parametrize(
    "rows,n",
    # 64 x 64 (twice), 128 x 128, 128 x 256 and 256 x 256 tiles (256 CUs; the last
    # register-staged up to K 192); test_library_abi.py holds the rule to it
    [(1, 256), (129, 512), (777, 4096), (2047, 4096), (8191, 4096)],
)
def test_every_tile_kernel_at_its_edges(gpu_device, rows, n, k):
    """Each tile kernel with a partial last row tile and one to five K steps
    (odd and even: both stages, all prefetch tails; two tiles per workgroup
    for the largest), with and without GELU, bf16 and fp16, against
    float64.  The K order is the same in every kernel, so rows computed alone
    (the 64 x 64 tiles) equal the same rows of the whole call bit for bit."""

    from solution.kernels.ffn import prevalidated_hip_linear, prevalidated_hip_linear_exact_gelu

    for dtype in (torch.bfloat16, torch.float16):
        _, (xd, wd, bd) = _operands(rows, k, n, dtype, seed=rows + k, device=gpu_device)
        exact = F.linear(xd.double(), wd.double(), bd.double())
        for call, reference in ((prevalidated_hip_linear, exact), (prevalidated_hip_linear_exact_gelu, F.gelu(exact))):
            with torch.inference_mode():
                out, _ = call(xd, wd, bd)
                head, _ = call(xd[:100].contiguous(), wd, bd)
                tail, _ = call(xd[-77:].contiguous(), wd, bd)
            torch.cuda.synchronize()
            # one rounding of the result (unit roundoff 2^-8 at 8 significant
            # bits, 2^-11 at 11; half the smallest fp16 step near zero), and
            # fp32 accumulation of k products (k 2^-24 of sum |x| |w|, the
            # activation's slope is below 2)
            roundoff = 2.0**-8 if dtype == torch.bfloat16 else 2.0**-11
            slack = k * 2.0**-24 * F.linear(xd.double().abs(), wd.double().abs(), bd.double().abs())
            bound = roundoff * (reference.abs() + 2 * slack) + 2 * slack + 2.0**-25
            err = (out.double() - reference).abs()
            print(f"{call.__name__} {dtype} {rows}x{k}->{n}: max err {float(err.max()):.3g}", flush=True)
            assert bool((err <= bound).all())
            assert torch.equal(out[:100], head) and torch.equal(out[-77:], tail)


def test_rows_beyond_the_tile_kernels_offsets(gpu_device):
    """x rows more than 2^22 elements apart go to the register-staged kernel."""

    from solution.kernels.ffn import prevalidated_hip_linear
    from solution.kernels.hip import _library

    rows, k, n, ldx = 3, 128, 256, (1 << 22) + 8
    _, (xd, wd, bd) = _operands(rows, k, n, torch.bfloat16, seed=2, device=gpu_device)
    far = torch.empty(rows, ldx, dtype=torch.bfloat16, device=gpu_device)
    far[:, :k] = xd
    y = torch.empty(rows, n, dtype=torch.bfloat16, device=gpu_device)
    status = _library.load_library().sah_linear(
        far.data_ptr(), wd.data_ptr(), bd.data_ptr(), y.data_ptr(), rows, k, n, ldx, n,
        _library.dtype_code(torch.bfloat16), _library.SAH_ACTIVATION_NONE, 256, 256, 64, 8, 2,
        _library.stream_handle(gpu_device),
    )
    _library.check_status(status, "sah_linear")
    with torch.inference_mode():
        expected, _ = prevalidated_hip_linear(xd, wd, bd)
    torch.cuda.synchronize()
    assert torch.equal(y, expected)


@pytest.mark.parametrize("rows", [1, 31, 33, 256])
@pytest.mark.parametrize("k,n", [(128, 32), (256, 256), (384, 96), (512, 32), (1024, 64), (1152, 64), (512, 1024)])
def test_fp32_linear_at_its_edges(gpu_device, rows, k, n):
    """sah_linear_f32 about its 32 x 32 and 16 x 16 tiles and their load steps,
    with padded rows on both sides, against float64: k products and sums in
    fp32, (k + 4) 2^-24 of sum |x| |w| + |b|.  GELU: its slope (at most 1.13)
    times that, and 5 2^-24 |v| for 0.5 v (1 + erff(v / sqrt 2)) (erff to 2
    ulp, its argument and the sum to one rounding each, two products)."""

    from solution.kernels.hip import _library

    g = torch.Generator().manual_seed(rows + k + n)
    ldx, ldy = k + 4, n + 8
    xs = torch.full((rows, ldx), float("nan"))
    xs[:, :k] = torch.randn(rows, k, generator=g)
    w, b = torch.randn(n, k, generator=g).to(gpu_device), torch.randn(n, generator=g).to(gpu_device)
    xs = xs.to(gpu_device)
    for bias, act in ((b, 0), (None, 0), (b, 1)):
        y = torch.full((rows + 2, ldy), -7.0, device=gpu_device)
        status = _library.load_library().sah_linear_f32(
            xs.data_ptr(), w.data_ptr(), None if bias is None else bias.data_ptr(), y.data_ptr(), rows, k, n, ldx,
            ldy, act, _library.stream_handle(gpu_device),
        )
        _library.check_status(status, "sah_linear_f32")
        torch.cuda.synchronize()
        x = xs[:, :k].double()
        expected = F.linear(x, w.double(), None if bias is None else bias.double())
        size = F.linear(x.abs(), w.double().abs(), None if bias is None else bias.double().abs())
        bound = (k + 4) * 2.0**-24 * size
        if act:
            bound = 1.13 * bound + 5 * 2.0**-24 * expected.abs()
            expected = F.gelu(expected)
        error = (y[:rows, :n].double() - expected).abs()
        print(f"fp32 linear {rows}x{k}->{n} act {act}: max err {float(error.max()):.3g}", flush=True)
        assert bool((error <= bound).all())
        assert bool((y[:rows, n:] == -7.0).all()) and bool((y[rows:] == -7.0).all())


def test_model_projection_takes_what_it_serves(gpu_device):
    """project() against F.linear: the calls it serves agree to fp32 rounding, and
    every call that something observes or casts, or that the rule or the
    layout leaves out, is refused."""

    from solution.kernels.projection.hip_linear import project

    rows, k, n, dtype = 100, 256, 192, torch.float32
    linear = torch.nn.Linear(k, n, device=gpu_device, dtype=dtype)
    value = torch.randn(1, rows, k, device=gpu_device, dtype=dtype)
    with torch.no_grad():
        out = project(linear, value)
        exact = F.linear(value.double(), linear.weight.double(), linear.bias.double())
        size = F.linear(value.double().abs(), linear.weight.double().abs(), linear.bias.double().abs())
        bound = (k + 4) * 2.0**-24 * size
        assert out.shape == (1, rows, n) and bool(((out.double() - exact).abs() <= bound).all())
        hidden = project(linear, value, gelu=True)
        bound = 1.13 * bound + 5 * 2.0**-24 * exact.abs()
        assert bool(((hidden.double() - F.gelu(exact)).abs() <= bound).all())
        assert project(linear, torch.randn(1, rows, k + 8, device=gpu_device, dtype=dtype)[..., :k]) is None
        assert project(linear, value.cpu()) is None
        with torch.autocast("cuda", dtype=torch.float16):
            assert project(linear, value) is None
        handle = linear.register_forward_hook(lambda *_: None)
        assert project(linear, value) is None
        handle.remove()
        assert project(linear, value) is not None
    assert project(linear, value) is None  # grad enabled


def test_model_projection_leaves_no_guard_in_a_compiled_caller(gpu_device):
    """Under torch.compile the call is F.linear whatever the size: a caller of a
    dynamic row count compiles once, on both sides of the rule's line."""

    from torch._dynamo.testing import CompileCounter
    from solution.kernels.projection.hip_linear import project

    linear = torch.nn.Linear(256, 256, device=gpu_device)
    counter = CompileCounter()
    torch._dynamo.reset()

    @torch.compile(backend=counter, fullgraph=True)
    def call(value):
        output = project(linear, value)
        return linear(value) if output is None else output

    with torch.no_grad():
        for rows in (64, 250, 5000):
            value = torch.randn(rows, 256, device=gpu_device)
            torch._dynamo.mark_dynamic(value, 0)
            assert torch.equal(call(value), F.linear(value, linear.weight, linear.bias)), rows
    assert counter.frame_count == 1


@pytest.mark.parametrize("rows,k", [(1, 256), (300, 256), (300, 64), (20_000, 256)])
@pytest.mark.parametrize("act", [0, 1])
def test_256_columns_in_place_through_the_c_abi(gpu_device, rows, k, act):
    """y over x, 256 columns: the separate buffers' result bit for bit."""

    from solution.kernels.hip import _library

    n, dtype = 256, torch.bfloat16
    _, (xd, wd, bd) = _operands(rows, k, n, dtype, seed=rows + k, device=gpu_device)
    padded = torch.zeros(rows, n, dtype=dtype, device=gpu_device)
    padded[:, :k] = xd

    def call(x, y):
        status = _library.load_library().sah_linear(
            x.data_ptr(), wd.data_ptr(), bd.data_ptr(), y.data_ptr(), rows, k, n, n, n, _library.dtype_code(dtype), act,
            256, 256, 64, 8, 2, _library.stream_handle(gpu_device),
        )
        _library.check_status(status, "sah_linear")

    expected = torch.empty_like(padded)
    call(padded, expected)
    call(padded, padded)
    torch.cuda.synchronize()
    assert torch.equal(padded, expected)


@pytest.mark.parametrize("k", [64, 128, 192, 256])
@pytest.mark.parametrize("rows,n", [(10_000, 1024), (20_002, 512), (50_000, 256)])
def test_short_k_of_many_rows(gpu_device, rows, n, k):
    """About the line to the register-staged kernel (K up to 192, 256 in one round
    without GELU): rows computed alone (64 x 64 tiles) equal the same rows of the
    whole call bit for bit, the K order being the same in every kernel."""

    from solution.kernels.ffn import prevalidated_hip_linear, prevalidated_hip_linear_exact_gelu

    for dtype in (torch.bfloat16, torch.float16):
        _, (xd, wd, bd) = _operands(rows, k, n, dtype, seed=rows + k, device=gpu_device)
        for call in (prevalidated_hip_linear, prevalidated_hip_linear_exact_gelu):
            with torch.inference_mode():
                out, _ = call(xd, wd, bd)
                parts = [(first, call(xd[first : first + 100].contiguous(), wd, bd)[0])
                         for first in (0, 256 * 31 - 50, rows - 100)]
            torch.cuda.synchronize()
            for first, part in parts:
                assert torch.equal(out[first : first + 100], part), (dtype, call.__name__, first)


@pytest.mark.parametrize("rows,n,k", [
    # 128 x 256 tiles, two and three a workgroup: the next tile's loads issued inside
    # the epilogue, and the counted wait behind its stores (whole and partial last row tiles)
    (4133, 4096, 64), (4133, 4096, 128), (4133, 4096, 320), (4133, 4096, 1024),
    (5120, 4096, 64), (5120, 4096, 320),
    # 256 x 256 tiles, five and six a workgroup, one to four K steps
    (20_993, 4096, 64), (20_993, 4096, 128), (20_993, 4096, 192), (20_993, 4096, 256),
])
def test_persistent_tiles_of_several_rounds(gpu_device, rows, n, k):
    """The checks of every tile kernel where a workgroup walks several tiles."""

    test_every_tile_kernel_at_its_edges(gpu_device, rows, n, k)
