"""Products of more rows on packed weights (csrc/kernels/linear_packed.hip)."""
import pytest
import torch

from hcache_deepspeed_amd.ops import quantizer as Q

pytestmark = pytest.mark.gpu


def _packed(fmt, N, K, G):
    w = torch.randn(N, K, device="cuda", dtype=torch.bfloat16) * K**-0.5
    if fmt.startswith("int"):
        q, s, _ = Q.quantize(w.reshape(-1), G, int(fmt[3:]), True)
        return q, s, Q.dequantize(q, s, None, G, int(fmt[3:]), True, torch.float32).view(N, K).double()
    mb = 2 if fmt.endswith("e3m2") else 3
    q, s = Q.quantize_minifloat(w.reshape(-1), G, 6, mb)
    return q, s, Q.dequantize_minifloat(q, s, G, 6, mb, torch.float32).view(N, K).double()


@pytest.mark.parametrize("fmt", ["int8", "int4", "fp6_e3m2", "fp6_e2m3"])
@pytest.mark.parametrize("M,N,K,G", [(17, 68, 256, 128), (24, 4100, 2048, 128), (32, 12296, 1152, 384), (33, 1000, 640, 128),
                                     (64, 4104, 4224, 128), (65, 520, 5632, 256), (100, 16392, 1024, 1024), (128, 2052, 896, 128),
                                     (256, 3080, 1152, 128), (512, 260, 4096, 4096), (16, 8204, 8320, 128)])
def test_rows_on_packed_weights(fmt, M, N, K, G):
    """All tiles, with remainders of rows and of weight rows; one slice and several, whose groups begin inside a slice; a bias.
    The codes are exact in bf16: 32-bit sums of K exact products, each rounded once more with its scale, and the result's rounding."""
    torch.manual_seed(K + M)
    x = torch.randn(M, K, device="cuda", dtype=torch.bfloat16)
    q, s, wd = _packed(fmt, N, K, G)
    assert N * K < 1 << 23 and M <= 32 and fmt[0] == "f" or Q._packed_plan(M, N, K, G, fmt[:4] if fmt[0] == "i" else "fp6", 0)
    if fmt[0] == "i":
        bias = torch.randn(N, device="cuda").bfloat16()
        y = Q.int_linear(x, q, s, N, K, G, bits=int(fmt[3:]), bias=bias)
    else:
        bias = torch.zeros(N, device="cuda").bfloat16()
        y = Q.fp6_linear(x, q, s, N, K, G, 2 if fmt.endswith("e3m2") else 3)
    ref = x.double() @ wd.t() + bias.double()
    bound = 2**-8 * ref.abs() + 1e-5 * (x.double().abs() @ wd.abs().t() + bias.double().abs())
    assert ((y.double() - ref).abs() <= bound).all()


@pytest.mark.parametrize("fmt", ["int8", "int4", "fp6"])
@pytest.mark.parametrize("M,N,K,act", [(17, 36, 256, "silu"), (32, 4100, 4224, "gelu_tanh"), (64, 2052, 1024, "relu"),
                                       (100, 1028, 8320, "silu"), (256, 516, 640, "silu")])
def test_gated_rows_on_packed_weights(fmt, M, N, K, act):
    """The gated unit in the epilogue and in the sum of slices, tiles of 32 and 64 columns with remainders."""
    torch.manual_seed(K + M)
    x = torch.randn(M, K, device="cuda", dtype=torch.bfloat16)
    q, s, wd = _packed(fmt if fmt[0] == "i" else "fp6_e3m2", 2 * N, K, 128)
    y = Q.packed_glu(x, q, s, N, K, 128, fmt, act)
    if fmt == "fp6" and M <= 32 and 2 * N * K < 1 << 23:
        assert y is None
        return
    gate, up = (x.double() @ wd.t()).split(N, 1)
    f = {"silu": torch.nn.functional.silu, "gelu_tanh": lambda t: torch.nn.functional.gelu(t, approximate="tanh"),
         "relu": torch.relu}[act]
    ref = f(gate) * up
    eg, eu = (1e-5 * (x.double().abs() @ wd.abs().t())).split(N, 1)
    # each factor within half a unit of the last place and its sum's error; |act'| <= 1.13
    bound = 2**-8 * (1.13 * gate.abs() * up.abs() + 2 * ref.abs()) + 1.13 * (eg * up.abs() + eu * gate.abs()) + 1e-6
    assert ((y.double() - ref).abs() <= bound).all()


def test_packed_rows_leave_autocast():
    """Of 65 rows and more the weights are dequantized for a library product, whose type autocast decides."""
    q, s, _ = _packed("int8", 4096, 4096, 128)
    x = torch.ones(128, 4096, dtype=torch.bfloat16, device="cuda")
    with torch.no_grad(), torch.autocast("cuda", torch.float16):
        assert Q._packed_rows(x, q, s, 4096, 4096, 128, "int8", 3, None, 0) is None
        assert Q.int_linear(x, q, s, 4096, 4096, 128).dtype == torch.float16


TILES = [(16, 64), (32, 64), (64, 64), (128, 128)]  # kTiles: rows, weight rows


@pytest.mark.parametrize("fmt", ["int8", "int4", "fp6_e3m2", "fp6_e2m3"])
@pytest.mark.parametrize("glu", [False, True])
@pytest.mark.parametrize("S", [1, 3])
@pytest.mark.parametrize("tile", range(len(TILES)))
def test_each_tile_on_packed_weights(tile, S, glu, fmt):
    """Every kernel by name, whatever the choice: one tile of rows and two, remainders, reductions that the ring holds and longer ones,
    groups of a stage and of several; the bounds of the tests above."""
    from hcache_deepspeed_amd.ops import native
    R, W = TILES[tile]
    torch.manual_seed(tile)
    for M, K, G in ((R - 3, 512, 128), (R + 5, 2304, 1152), (4, 1536, 768)):
        N = (W // 2 if glu else W) + 12
        rows = 2 * N if glu else N
        q, s, wd = _packed(fmt, rows, K, G)
        x = torch.randn(M, K, device="cuda", dtype=torch.bfloat16)
        bias = None if glu else torch.randn(N, device="cuda").bfloat16()
        y = torch.full((M + 1, N), 7.0, device="cuda", dtype=torch.bfloat16)
        part = torch.empty(S, M, rows, device="cuda")
        native.check(native.kernels().hds_packed_rows(
            x.data_ptr(), q.data_ptr(), s.data_ptr(), native.ptr(bias), y.data_ptr(), part.data_ptr(), M, N, K, G,
            {"int8": 0, "int4": 1}.get(fmt, 2), 2 if fmt == "fp6_e2m3" else 3, 1 if glu else 0, tile + 16 * S, native.stream()), "packed_rows")
        ref, err = x.double() @ wd.t(), 1e-5 * (x.double().abs() @ wd.abs().t())
        if glu:
            (gate, up), (eg, eu) = ref.split(N, 1), err.split(N, 1)
            ref = torch.nn.functional.silu(gate) * up
            bound = 2**-8 * (1.13 * gate.abs() * up.abs() + 2 * ref.abs()) + 1.13 * (eg * up.abs() + eu * gate.abs()) + 1e-6
        else:
            ref = ref + bias.double()
            bound = 2**-8 * ref.abs() + err + 1e-5 * bias.double().abs()
        assert ((y[:M].double() - ref).abs() <= bound).all() and (y[M:] == 7).all(), (M, K)
