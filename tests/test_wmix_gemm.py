"""Mixed-input MFMA GEMM (csrc/kernels/wmix_gemm.hip): INT8 / INT4 / FP6 weight-only x bf16 activations against
an fp32 reference of the same op (dequantized weight, fp32 matmul). Reference parity: the CUTLASS mixed GEMM
(K37) and the FP6-LLM linear (K29), whose tests compare against a dequantized fp16 matmul."""
import pytest
import torch

from hcache_deepspeed_amd.ops import quantizer as Q

pytestmark = pytest.mark.gpu


def _ref(x, wq):
    return (x.float() @ wq.float().t())


@pytest.mark.parametrize("fmt", ["int8", "int4", "fp6_e3m2", "fp6_e2m3"])
@pytest.mark.parametrize("M,N,K,G", [(9, 384, 512, 128), (33, 1000, 1024, 32), (64, 4096, 4096, 128),
                                     (100, 520, 768, 64), (200, 256, 2048, 128)])
def test_wmix_matches_dequant_reference(fmt, M, N, K, G):
    torch.manual_seed(0)
    dev = "cuda"
    x = torch.randn(M, K, device=dev, dtype=torch.bfloat16)
    w = torch.randn(N, K, device=dev, dtype=torch.bfloat16) * 0.05
    bias = torch.randn(N, device=dev, dtype=torch.bfloat16)
    if fmt.startswith("int"):
        bits = int(fmt[3:])
        q, s, _ = Q.quantize(w.reshape(-1), G, bits, True)
        wd = Q.dequantize(q, s, None, G, bits, True, torch.float32).view(N, K)
        y = Q.wmix_gemm(x, q, s, N, K, G, fmt, bias=bias)
        y2 = Q.int_linear(x, q, s, N, K, G, bits=bits, bias=bias)  # dispatcher takes the same kernel
    else:
        mb = 2 if fmt.endswith("e3m2") else 3
        q, s = Q.quantize_minifloat(w.reshape(-1), G, 6, mb)
        wd = Q.dequantize_minifloat(q, s, G, 6, mb, torch.float32).view(N, K)
        y = Q.wmix_gemm(x, q, s, N, K, G, "fp6", 5 - mb, bias=bias)
        y2 = Q.fp6_linear(x, q, s, N, K, G, mb) + bias
    ref = _ref(x, wd) + bias.float()
    err = (y.float() - ref).abs().max().item()
    scale = ref.abs().max().item()
    # bf16 rounding of the dequantized weight (8 bits) + bf16 output: ~1e-2 relative of the largest output
    assert err <= 1e-2 * scale + 1e-2, (fmt, M, N, K, G, err, scale)
    assert (y2.float() - ref).abs().max().item() <= 1.5e-2 * scale + 2e-2


def test_wmix_split_k_deterministic():
    torch.manual_seed(1)
    x = torch.randn(48, 14336, device="cuda", dtype=torch.bfloat16)
    w = torch.randn(512, 14336, device="cuda", dtype=torch.bfloat16) * 0.02
    q, s, _ = Q.quantize(w.reshape(-1), 128, 8, True)
    from hcache_deepspeed_amd.ops import native
    assert native.kernels().hds_wmix_splits(48, 512, 14336) > 1
    a = Q.wmix_gemm(x, q, s, 512, 14336, 128, "int8")
    b = Q.wmix_gemm(x, q, s, 512, 14336, 128, "int8")
    assert torch.equal(a, b)
    ref = x.float() @ Q.dequantize(q, s, None, 128, 8, True, torch.float32).view(512, 14336).t()
    assert (a.float() - ref).abs().max().item() <= 1e-2 * ref.abs().max().item()


@pytest.mark.parametrize("fmt", ["int8", "int4", "fp6_e3m2", "fp6_e2m3"])
@pytest.mark.parametrize("M,N,K,G", [(1, 16, 128, 128), (8, 1000, 640, 128), (9, 16390, 512, 256), (16, 6160, 4224, 128),
                                     (17, 250, 1024, 1024), (32, 48, 14336, 128), (5, 40, 1024, 64),
                                     (3, 16380, 640, 128), (8, 16384, 4224, 128), (16, 16390, 4096, 512), (5, 33000, 2048, 128)])
def test_few_rows_keep_the_weights_exact(fmt, M, N, K, G):
    """The stream of packed weights: tails of the rows and of the 512-wide runs, one and two tiles of weight rows, four and
    eight waves, scales read by four and one by one, rows resident (from 16,384 weight rows of fp6 on) with one to three
    rounds of tiles; groups of 64 take the older kernels. The codes are exact and the
    scales 32-bit, so what is left are 32-bit sums (K terms) and the result's rounding."""
    torch.manual_seed(K + M)
    x = torch.randn(M, K, device="cuda", dtype=torch.bfloat16)
    w = torch.randn(N, K, device="cuda", dtype=torch.bfloat16) * 0.05
    if fmt.startswith("int"):
        bits = int(fmt[3:])
        q, s, _ = Q.quantize(w.reshape(-1), G, bits, True)
        wd = Q.dequantize(q, s, None, G, bits, True, torch.float32).view(N, K).double()
        bias = torch.randn(N, device="cuda", dtype=torch.bfloat16)
        y = Q.int_linear(x, q, s, N, K, G, bits=bits, bias=bias)
        ref = x.double() @ wd.t() + bias.double()
        stream = G % 128 == 0 and (bits == 8) < M <= 16
    else:
        mb = 2 if fmt.endswith("e3m2") else 3
        q, s = Q.quantize_minifloat(w.reshape(-1), G, 6, mb)
        wd = Q.dequantize_minifloat(q, s, G, 6, mb, torch.float32).view(N, K).double()
        y = Q.fp6_linear(x, q, s, N, K, G, mb)
        ref = x.double() @ wd.t()
        stream = G % 128 == 0
    bound = 2**-8 * ref.abs() + 1e-5 * (x.double().abs() @ wd.abs().t()) if stream else 0.02 * ref.abs().max()
    assert ((y.double() - ref).abs() <= bound).all()


@pytest.mark.parametrize("fmt,M,N,K", [
    ("fp6_e3m2", 1, 4090, 2176), ("fp6_e2m3", 8, 4200, 4224), ("fp6_e3m2", 9, 4000, 2176), ("fp6_e3m2", 16, 5000, 4352),
    ("int8", 3, 4096, 4224), ("int8", 8, 4112, 4608), ("int4", 1, 4096, 14336), ("int4", 7, 5000, 8320), ("int8", 1, 16400, 2176),
    ("int8", 16, 20500, 4096), ("int4", 16, 32790, 1920), ("fp6_e3m2", 5, 16390, 2176), ("int4", 2, 16384, 3200), ("int4", 5, 16390, 4224),
    ("int4", 16, 16380, 4224), ("int4", 9, 16400, 4224), ("fp6_e3m2", 12, 16400, 4224), ("fp6_e2m3", 9, 19300, 4224)])
def test_whole_lines_of_packed_weights(fmt, M, N, K):
    """The kernels that load whole lines, to the stream's bound: walks that end inside a run of 512 or leave waves without one,
    four, six and eight waves, partial tiles, one to three rounds of resident rows, many weight rows beside them; packed weights 8 bytes off a line."""
    torch.manual_seed(K + M)
    x = torch.randn(M, K, device="cuda", dtype=torch.bfloat16)
    w = torch.randn(N, K, device="cuda", dtype=torch.bfloat16) * 0.05
    off = lambda q: torch.cat([q.new_zeros(8), q.reshape(-1)])[8:]  # noqa: E731
    if fmt.startswith("int"):
        bits = int(fmt[3:])
        q, s, _ = Q.quantize(w.reshape(-1), 128, bits, True)
        wd = Q.dequantize(q, s, None, 128, bits, True, torch.float32).view(N, K).double()
        y = Q.int_linear(x, off(q), s, N, K, 128, bits=bits)
    else:
        mb = 2 if fmt.endswith("e3m2") else 3
        q, s = Q.quantize_minifloat(w.reshape(-1), 128, 6, mb)
        wd = Q.dequantize_minifloat(q, s, 128, 6, mb, torch.float32).view(N, K).double()
        y = Q.fp6_linear(x, off(q), s, N, K, 128, mb)
    ref = x.double() @ wd.t()
    assert ((y.double() - ref).abs() <= 2**-8 * ref.abs() + 1e-5 * (x.double().abs() @ wd.abs().t())).all()


@pytest.mark.parametrize("fmt,M,N,K,gemv", [
    ("int4", 1, 1024, 1024, True), ("int4", 1, 4096, 11648, True), ("int4", 1, 4096, 11776, False), ("int4", 1, 12200, 8192, True),
    ("int4", 1, 12224, 8192, False), ("int4", 2, 3900, 1024, True), ("int4", 2, 3920, 1024, False), ("int8", 2, 1000, 640, True),
    ("int8", 2, 6500, 640, True), ("int8", 2, 6560, 640, False), ("int8", 2, 4096, 640, False), ("fp6", 1, 3900, 1024, True),
    ("fp6", 1, 3920, 1024, False)])
def test_one_and_two_rows_keep_the_weights_exact_on_both_kernels(fmt, M, N, K, gemv):
    """Both sides of the sizes at which the packed GEMVs give way to the stream, to the stream's bound: 32-bit sums of K exact
    products and the result's rounding."""
    assert Q._gemv_wins(M, N, K, fmt) == gemv
    torch.manual_seed(K + M)
    x = torch.randn(M, K, device="cuda", dtype=torch.bfloat16)
    w = torch.randn(N, K, device="cuda", dtype=torch.bfloat16) * 0.05
    if fmt == "fp6":
        q, s = Q.quantize_minifloat(w.reshape(-1), 128, 6, 2)
        wd = Q.dequantize_minifloat(q, s, 128, 6, 2, torch.float32).view(N, K).double()
        y = Q.fp6_linear(x, q, s, N, K, 128, 2)
    else:
        bits = int(fmt[3:])
        q, s, _ = Q.quantize(w.reshape(-1), 128, bits, True)
        wd = Q.dequantize(q, s, None, 128, bits, True, torch.float32).view(N, K).double()
        y = Q.int_linear(x, q, s, N, K, 128, bits=bits)
    ref = x.double() @ wd.t()
    assert ((y.double() - ref).abs() <= 2**-8 * ref.abs() + 1e-5 * (x.double().abs() @ wd.abs().t())).all()


@pytest.mark.parametrize("fmt", ["int8", "int4", "fp6"])
@pytest.mark.parametrize("act", ["silu", "gelu_tanh", "relu"])
@pytest.mark.parametrize("M,N,K,G", [(2, 7, 128, 128), (8, 1000, 640, 128), (16, 4104, 4224, 128), (9, 8200, 4096, 128),
                                     (5, 8189, 1024, 256)])
def test_gated_projection_of_packed_weights(fmt, act, M, N, K, G):
    """act(x . gate^T) * (x . up^T) in one kernel: remainders of a tile's 8 rows, one and two tiles, rows resident."""
    torch.manual_seed(K + M)
    x = torch.randn(M, K, device="cuda", dtype=torch.bfloat16)
    w = torch.randn(2 * N, K, device="cuda", dtype=torch.bfloat16) * K**-0.5
    if fmt == "fp6":
        q, s = Q.quantize_minifloat(w.reshape(-1), G, 6, 2)
        wd = Q.dequantize_minifloat(q, s, G, 6, 2, torch.float32)
    else:
        q, s, _ = Q.quantize(w.reshape(-1), G, int(fmt[3:]), True)
        wd = Q.dequantize(q, s, None, G, int(fmt[3:]), True, torch.float32)
    wd = wd.view(2 * N, K).double()
    y = Q.packed_glu(x, q, s, N, K, G, fmt, act)
    gate, up = (x.double() @ wd.t()).split(N, 1)
    f = {"silu": torch.nn.functional.silu, "gelu_tanh": lambda t: torch.nn.functional.gelu(t, approximate="tanh"),
         "relu": torch.relu}[act]
    ref = f(gate) * up
    eg, eu = (1e-5 * (x.double().abs() @ wd.abs().t())).split(N, 1)
    # each factor within half a unit of the last place and its sum's error; |act'| <= 1.13
    bound = 2**-8 * (1.13 * gate.abs() * up.abs() + 2 * ref.abs()) + 1.13 * (eg * up.abs() + eu * gate.abs()) + 1e-6
    assert ((y.double() - ref).abs() <= bound).all()


@pytest.mark.parametrize("fmt", ["int8", "int4", "fp6"])
@pytest.mark.parametrize("M", [3, 9, 16, 32])
def test_groups_that_do_not_divide_a_row(fmt, M):
    """Groups that run on from one row to the next (384 columns in groups of 256) are no case for the packed-weight kernels:
    the linears dequantize then. Few rows of fp6 are refused, as the GEMV of up to 8 rows does."""
    torch.manual_seed(M)
    N, K, G = 128, 384, 256
    x = torch.randn(M, K, device="cuda", dtype=torch.bfloat16)
    w = torch.randn(N, K, device="cuda", dtype=torch.bfloat16) * K**-0.5
    if fmt == "fp6":
        q, s = Q.quantize_minifloat(w.reshape(-1), G, 6, 2)
        wd = Q.dequantize_minifloat(q, s, G, 6, 2, torch.float32).view(N, K).double()
        if M <= 8:
            with pytest.raises(RuntimeError):
                Q.fp6_linear(x, q, s, N, K, G)
            return
        y = Q.fp6_linear(x, q, s, N, K, G)
    else:
        bits = int(fmt[3:])
        q, s, _ = Q.quantize(w.reshape(-1), G, bits, True)
        wd = Q.dequantize(q, s, None, G, bits, True, torch.float32).view(N, K).double()
        y = Q.int_linear(x, q, s, N, K, G, bits=bits)
    assert Q.packed_glu(x, q, s, N // 2, K, G, fmt, "silu") is None
    # the dequantized weight and the result, each rounded to bf16
    bound = 2**-8 * ((x.double() @ wd.t()).abs() + x.double().abs() @ wd.abs().t())
    assert ((y.double() - x.double() @ wd.t()).abs() <= bound).all()


@pytest.mark.parametrize("M", [1, 8])
@pytest.mark.parametrize("mantissa", [1, 2, 3])
def test_fp6_formats_that_only_the_gemv_takes(M, mantissa):
    """e4m1 beside the formats of the packed-weight kernels: up to 8 rows the GEMV decodes them."""
    torch.manual_seed(M)
    N, K, G = 64, 256, 128
    x = torch.randn(M, K, device="cuda", dtype=torch.bfloat16)
    q, s = Q.quantize_minifloat((torch.randn(N, K, device="cuda") * K**-0.5).bfloat16().reshape(-1), G, 6, mantissa)
    wd = Q.dequantize_minifloat(q, s, G, 6, mantissa, torch.float32).view(N, K).double()
    y = Q.fp6_linear(x, q, s, N, K, G, mantissa)
    bound = 2**-8 * ((x.double() @ wd.t()).abs() + x.double().abs() @ wd.abs().t())
    assert ((y.double() - x.double() @ wd.t()).abs() <= bound).all()


@pytest.mark.parametrize("bits,M", [(8, 1), (8, 2), (4, 2), (8, 3)])
def test_int_linear_with_a_32_bit_bias(bits, M):
    """One and two rows with a 32-bit bias give 32 bits (the products are bf16), more rows bf16."""
    torch.manual_seed(M)
    N, K, G = 128, 256, 128
    x = torch.randn(M, K, device="cuda", dtype=torch.bfloat16)
    w = torch.randn(N, K, device="cuda", dtype=torch.bfloat16) * K**-0.5
    q, s, _ = Q.quantize(w.reshape(-1), G, bits, True)
    b = torch.randn(N, device="cuda")
    y = Q.int_linear(x, q, s, N, K, G, bits=bits, bias=b)
    assert y.dtype == (torch.float32 if M <= 2 else torch.bfloat16)
    narrow = b.bfloat16().requires_grad_()
    assert Q.int_linear(x, q, s, N, K, G, bits=bits, bias=narrow).requires_grad == (M <= 2)
    ref = x.double() @ Q.dequantize(q, s, None, G, bits, True, torch.float32).view(N, K).double().t()
    assert ((y.double() - (ref + b.double())).abs() <= 2**-8 * (ref.abs() + b.abs() + x.double().abs() @ w.double().abs().t())).all()


@pytest.mark.parametrize("M,N,K", [(1, 8200, 4096), (4, 8190, 2304), (16, 16400, 1920)])
def test_gated_projection_of_resident_rows(M, N, K):
    """One row of int8 in the gated kernel, waves without a run, two tiles at work at a time."""
    test_gated_projection_of_packed_weights("int8", "silu", M, N, K, 128)
