"""Products of 9 to 1,100 rows that split their reduction (csrc/kernels/linear.hip)."""
import pytest
import torch

from hcache_deepspeed_amd.ops import gemv

# smallest and largest rows of either rule, one and several row tiles, rows and columns behind the last tile, slices that
# differ by a stage, slices of fewer stages than the ring holds
SHAPES = [(9, 16384, 4096), (16, 32000, 2048), (13, 32008, 2112), (30, 33000, 1088), (64, 28672, 4096), (128, 12296, 2048), (17, 4096, 8192), (31, 4104, 8256), (33, 2056, 14336), (65, 2048, 8192), (80, 4096, 4096), (129, 4096, 4160), (193, 6144, 4096),
          (256, 8192, 8192), (256, 4120, 4096), (35, 72, 256), (40, 2048, 320), (32, 6144, 4096), (256, 8, 2048), (257, 4096, 8192), (521, 4096, 14336), (700, 3080, 8192), (1100, 4096, 8192)]


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_linear_rows_match_64_bits(M, N, K):
    g = torch.Generator(device="cuda").manual_seed(M + N)
    w = (torch.randn(N, K, device="cuda", generator=g) * K**-0.5).to(torch.bfloat16)
    x = torch.randn(M, K + 8, device="cuda", generator=g).to(torch.bfloat16)[:, :K]
    x[-1, -64:] = 100  # what the last row's last stage holds counts
    b = torch.randn(N, device="cuda", generator=g).to(torch.bfloat16) if M % 2 else None
    assert gemv._plan(M, N, K)
    with torch.no_grad():
        y, again = gemv.linear(x, w, b), gemv.linear(x, w, b)
    ref = x.double() @ w.double().t() + (0 if b is None else b.double())
    # 32-bit sums of K products, then one rounding
    bound = 2**-8 * ref.abs() + 2**-24 * K**0.5 * 8 * (x.double().abs() @ w.double().abs().t()) + 1e-6
    assert y.shape == ref.shape and ((y.double() - ref).abs() <= bound).all()
    assert torch.equal(y, again)


@pytest.mark.gpu
def test_linear_rows_all_tiles_exact():
    """The tiles and numbers of slices that the choice takes for one matrix over its range of rows: small integers, whose sums are
    exact in 32 bits and the result in bf16."""
    g = torch.Generator(device="cuda").manual_seed(1)
    K, N = 8192, 4096
    w = torch.randint(-1, 2, (N, K), device="cuda", generator=g).bfloat16()
    x = (torch.randint(-1, 2, (1100, K), device="cuda", generator=g) * (torch.rand(1100, K, device="cuda", generator=g) < 0.05)).bfloat16()
    ref = x.float() @ w.float().t()
    assert ref.abs().max() <= 256
    for M in list(range(17, 300, 16)) + list(range(300, 1100, 97)):
        with torch.no_grad():
            assert torch.equal(gemv.linear(x[:M], w).float(), ref[:M]), M


TILES = [(32, 64), (32, 128), (64, 64), (64, 128), (128, 128), (192, 128), (256, 128), (256, 256)]  # kTiles: rows, columns


@pytest.mark.gpu
@pytest.mark.parametrize("glu", [0, 3])  # 3: relu, exact on integers
@pytest.mark.parametrize("S", [1, 3])
@pytest.mark.parametrize("tile", range(len(TILES)))
def test_linear_rows_each_tile(tile, S, glu):
    """Every kernel by name, whatever the choice: one tile of rows and two, remainders of rows and columns, reductions that the ring holds
    and longer ones, walks apart; nothing is written beside the result."""
    from hcache_deepspeed_amd.ops import native
    R, W = TILES[tile]
    g = torch.Generator(device="cuda").manual_seed(tile)
    for M, K in ((R - 3, 448), (R + 5, 2048), (9, 1088)):
        N = (W // 2 if glu else W) + 24
        rows = 2 * N if glu else N
        w = torch.randint(-1, 2, (rows, K), device="cuda", generator=g).bfloat16()
        x = (torch.randint(-1, 2, (M, K), device="cuda", generator=g) * (torch.rand(M, K, device="cuda", generator=g) < 8 / K)).bfloat16()
        b = torch.randint(-2, 3, (rows, ), device="cuda", generator=g).bfloat16()
        y = torch.full((M + 1, N + 8), 7.0, device="cuda", dtype=torch.bfloat16)
        part = torch.empty(S, M, rows, device="cuda")
        native.check(native.kernels().hds_linear_bf16(x.data_ptr(), K, w.data_ptr(), b.data_ptr(), y.data_ptr(), N + 8, part.data_ptr(), M,
                                                      N, K, glu, tile + 16 * S, native.stream()), "linear_bf16")
        ref = x.float() @ w.float().t() + b.float()
        if glu:
            ref = ref[:, :N].relu() * ref[:, N:]
        assert 0 < ref.abs().max() <= 256
        assert torch.equal(y[:M, :N].float(), ref) and (y[M:] == 7).all() and (y[:, N:] == 7).all(), (M, K)


@pytest.mark.gpu
@pytest.mark.parametrize("act", ["silu", "gelu_tanh", "relu"])
@pytest.mark.parametrize("M,N,K", [(9, 14336, 4096), (16, 16392, 2112), (17, 8, 256), (33, 1000, 2048), (64, 5632, 2048), (129, 72, 8192), (200, 4096, 4160), (256, 14336, 4096)])
def test_linear_rows_gated(act, M, N, K):
    """One and several slices, features behind the last tile, against 64 bits with the projections rounded first."""
    g = torch.Generator(device="cuda").manual_seed(M + N)
    w = (torch.randn(2 * N, K, device="cuda", generator=g) * K**-0.5).to(torch.bfloat16)
    x = torch.randn(M, K + 8, device="cuda", generator=g).to(torch.bfloat16)[:, :K]
    b = torch.randn(2 * N, device="cuda", generator=g).to(torch.bfloat16) if M % 2 else None
    with torch.no_grad():
        y = gemv.glu_linear(x, w, b, act)
    ref = x.double() @ w.double().t() + (0 if b is None else b.double())
    sums = 2**-24 * K**0.5 * 8 * (x.double().abs() @ w.double().abs().t())
    gate, up = ref[:, :N], ref[:, N:]
    f = {"silu": torch.nn.functional.silu, "gelu_tanh": lambda t: torch.nn.functional.gelu(t, approximate="tanh"), "relu": torch.relu}[act]
    # each factor within half a unit of the last place and its sum's error; |act'| <= 1.13
    bound = 2**-8 * (1.13 * gate.abs() * up.abs() + 2 * (f(gate) * up).abs()) + 1.13 * (sums[:, :N] * up.abs() + sums[:, N:] * gate.abs())
    assert y.shape == (M, N) and ((y.double() - f(gate) * up).abs() <= bound + 1e-6).all()


@pytest.mark.gpu
def test_linear_rows_refuse():
    """What the kernel does not take goes where it went: rows, K, widths, types, alignment, gradients and transforms."""
    assert not any(gemv._plan(*s) for s in [(8, 32768, 4096), (32, 4096, 4096), (16, 4096, 8192), (1101, 4096, 8192), (128, 4096, 4000), (128, 4095, 8192), (129, 32768, 4096),
                                              (321, 4096, 4096), (257, 4096, 8192, 1)])
    x = torch.zeros(128, 8200, dtype=torch.bfloat16, device="cuda")
    w = torch.zeros(4096, 8192, dtype=torch.bfloat16, device="cuda")
    with torch.no_grad():
        assert gemv.rows_linear(x[:, :8192], w) is not None and gemv.rows_linear(x[:, :8192].view(2, 64, -1), w).shape == (2, 64, 4096)
        for a, b in ((x[:, 4:8196], w), (x[:, :8192].half(), w), (x, w), (x[:, :8192], w.t().contiguous().t())):
            assert gemv.rows_linear(a, b) is None
        with pytest.raises(RuntimeError):
            gemv.linear(x, w)
        rows = x[:, :8192].contiguous().view(2, 64, 8192)
        assert torch.func.vmap(gemv.linear, in_dims=(0, None))(rows, w).shape == (2, 64, 4096)
    w.requires_grad_()
    assert gemv.linear(x[:, :8192], w).grad_fn is not None


@pytest.mark.gpu
def test_linear_rows_leave_autocast_and_other_devices(monkeypatch):
    """Autocast to another type decides the result's type; a tensor of another device than the current one is the library's."""
    x = torch.ones(64, 4096, dtype=torch.bfloat16, device="cuda")
    w = torch.ones(4096, 4096, dtype=torch.bfloat16, device="cuda")
    with torch.no_grad():
        assert gemv.rows_linear(x, w) is not None
        with torch.autocast("cuda", torch.float16):
            assert gemv.linear(x, w).dtype == torch.float16
        monkeypatch.setattr(torch.cuda, "current_device", lambda: 1)
        assert gemv.rows_linear(x, w) is None


@pytest.mark.gpu
def test_linear_rows_heed_the_switches(monkeypatch):
    """HDS_SKINNY_GEMM=0 and HDS_SKINNY_MIN_M leave 9 to 16 rows to the library, as those of the skinny kernel; 17 are not theirs."""
    w = torch.ones(28672, 4096, dtype=torch.bfloat16, device="cuda")
    asked = []
    monkeypatch.setattr(gemv, "rows_linear", lambda x, *a: asked.append(x.shape[0]))
    with torch.no_grad():
        def call(M):
            x = torch.ones(M, 4096, dtype=torch.bfloat16, device="cuda")
            gemv.linear(x, w), gemv.glu_linear(x, w, None, "silu")
        call(12)
        monkeypatch.setattr(gemv, "SKINNY_MIN_M", 13)
        call(12), call(13)
        monkeypatch.setattr(gemv, "SKINNY", False)
        call(13), call(17)
    assert asked == [12, 12, 13, 13, 17, 17]


@pytest.mark.gpu
def test_linear_rows_leave_watched_calls():
    """Of 17 rows and more the product is the library's wherever something records or replaces operations: a dispatch mode (a
    trace by make_fx, a counter), a function mode other than a default device, torch.compile."""
    from torch.fx.experimental.proxy_tensor import make_fx
    from torch.overrides import TorchFunctionMode
    from torch.utils.flop_counter import FlopCounterMode
    M, N, K = 64, 4096, 4096
    g = torch.Generator(device="cuda").manual_seed(0)
    x, other = (torch.randn(M, K, device="cuda", generator=g).bfloat16() for _ in range(2))
    w = (torch.randn(N, K, device="cuda", generator=g) * K**-0.5).bfloat16()
    with torch.no_grad():
        traced = make_fx(lambda t: gemv.linear(t, w))(x)
        assert torch.equal(traced(other), torch.nn.functional.linear(other, w))
        with FlopCounterMode(display=False) as count:
            gemv.linear(x, w)
        assert count.get_total_flops() == 2 * M * N * K
        seen = []

        class Names(TorchFunctionMode):

            def __torch_function__(self, f, types, args=(), kwargs=None):
                seen.append(f)
                return f(*args, **(kwargs or {}))

        with Names():
            gemv.linear(x, w)
        assert torch.nn.functional.linear in seen
        graphs = []
        whole = torch.compile(gemv.linear, backend=lambda m, a: graphs.append(m) or m.forward, fullgraph=True)
        assert torch.equal(whole(x, w), torch.nn.functional.linear(x, w)) and len(graphs) == 1
        with torch.device("cuda"):
            assert gemv.rows_linear(x, w) is not None
