"""mi355_linear_few (prompts of few rows) against products in float64: tiles of every shape, edges of rows and columns, splits of K, K
tiles that its two groups of waves share unevenly, and the conditions under which ops.linear_few leaves a call to another kernel."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.fixture(scope="module")
def ops():
    from sglang_custom_amd import ops as o

    return o


def _bound(x, w, dtype):
    """Half an ulp of the result's type (2 for an error that crosses a rounding boundary) and 2^-24 per addition of K, which a random walk
    turns into its root; 8 x that."""
    k = x.shape[1]
    return (2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11), 8 * k ** 0.5 * 2.0 ** -24 * ((x ** 2) @ (w ** 2).T).sqrt()


# (rows, columns, K): tiles of 64 x 64, 128 x 64, 128 x 128; 1 to 8 splits; columns that end inside a tile; 2, 3, 9 and 33 K tiles
@pytest.mark.parametrize("m,n,k", [(65, 16, 128), (70, 2048, 2048), (128, 2064, 576), (129, 3072, 192), (207, 2048, 8192), (256, 16384, 256), (200, 8176, 2112),
                                   (100, 28672, 512), (1, 48, 1024)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_sixteen_bits(ops, m, n, k, dtype):
    g = torch.Generator().manual_seed(m + n + k)
    wide = torch.randn(m, k + 8, generator=g).to(dtype).to(DEV)
    x, w = wide[:, :k], torch.randn(n, k, generator=g).mul_(k ** -0.5).to(dtype).to(DEV)
    bias = torch.randn(n, generator=g).to(dtype).to(DEV)
    got = ops.linear_few(x, w, bias)
    assert got is not None
    ulp, sums = _bound(x.double(), w.double(), dtype)
    want = x.double() @ w.double().T + bias.double()
    assert ((got.double() - want).abs() <= ulp * want.abs() + sums + 1e-7).all()
    plain = ops.linear_few(x, w)
    # gate and up are rounded first: an error d of either moves the product by at most d |up| (1.1 is silu's steepest slope) or d |silu|, and the
    # result is rounded twice more; 2^-24 for the smallest fp16 numbers
    fused = ops.linear_few(x, w, None, silu_mul=True)
    gate, up = (x.double() @ w.double().T).chunk(2, 1)
    dg, du = ((ulp * z.abs() + sz + 2.0 ** -24) for z, sz in zip((gate, up), sums.chunk(2, 1)))
    silu = gate * torch.sigmoid(gate)
    assert ((fused.double() - silu * up).abs() <= 1.1 * dg * (up.abs() + du) + du * silu.abs() + 3 * ulp * (silu * up).abs() + 2.0 ** -23).all()
    if dtype == torch.bfloat16:
        assert torch.equal(ops.linear_few(x * 2, w), plain * 2)      # (powers of two change no rounding)
    if m > 64:
        order = torch.randperm(m, generator=g).to(DEV)
        assert torch.equal(ops.linear_few(x[order].contiguous(), w), plain[order])


@pytest.mark.parametrize("m,n,k", [(65, 48, 256), (88, 6144, 4096), (207, 4096, 14336), (512, 6144, 384), (300, 4096, 640)])
def test_eight_bits(ops, m, n, k):
    g = torch.Generator().manual_seed(m + n + k)
    x = torch.randn(m, k, generator=g).to(torch.float8_e4m3fn).to(DEV)
    w = torch.randn(n, k, generator=g).to(torch.float8_e4m3fn).to(DEV)
    xs, ws = torch.rand(m, 1, generator=g).add_(0.5).to(DEV), torch.rand(n, generator=g).add_(0.5).to(DEV) * k ** -0.5
    got = ops.linear_few(x, w, None, False, xs, ws, torch.bfloat16)
    # the matrix unit adds a K step's fp8 products with fewer bits than fp32: this kernel, the 256 x 256 one and torch._scaled_mm are all the same
    # 11 to 58 x 2^-24 sqrt(K) beyond half an ulp at these sizes
    ulp, sums = _bound(x.double() * xs.double(), w.double() * ws.double()[:, None], torch.bfloat16)
    want = (x.double() @ w.double().T) * xs.double() * ws.double()
    assert ((got.double() - want).abs() <= ulp * want.abs() + 16 * sums + 1e-7).all()
    off = lambda y: ((y.double() - want).norm() / want.norm()).item()
    assert off(got) <= 1.01 * off(ops.fp8_scaled_mm_tiled(x, w, xs, ws, torch.bfloat16))


def test_what_is_left_to_others(ops):
    x, w = torch.zeros(128, 1024, dtype=torch.bfloat16, device=DEV), torch.zeros(2048, 1024, dtype=torch.bfloat16, device=DEV)
    assert ops.linear_few(x, w) is not None
    assert ops.linear_few(torch.zeros(257, 1024, dtype=torch.bfloat16, device=DEV), w) is None                 # rows
    assert ops.linear_few(x, torch.zeros(65536, 1024, dtype=torch.bfloat16, device=DEV)) is None                # a second round of tiles
    assert ops.linear_few(x.t()[:128].contiguous().t(), w[:, :128].contiguous()) is None                        # rows that are columns
    assert ops.linear_few(torch.zeros(128 * 1024 + 1, dtype=torch.bfloat16, device=DEV)[1:].view(128, 1024), w) is None    # 2-byte aligned
    assert ops.linear_few(x, w, torch.zeros(2048, device=DEV)) is None                                          # a bias of another type
    assert ops.linear_few(x.float(), w.float()) is None


# one split and several (their sums' memory is the graph's own), both epilogues
@pytest.mark.parametrize("m,n,k,fp8,silu", [(96, 2048, 2048, False, False), (128, 2048, 8192, False, False), (96, 4096, 1024, False, True), (96, 4096, 4096, True, False)])
def test_captured(ops, m, n, k, fp8, silu):
    """Decode steps of more than 64 rows are captured too where they are asked for: replays over new rows give the eager call's bits."""
    g = torch.Generator().manual_seed(m + n)
    cast = lambda t: t.to(torch.float8_e4m3fn if fp8 else torch.bfloat16).to(DEV)
    x, w = cast(torch.randn(m, k, generator=g)), cast(torch.randn(n, k, generator=g))
    scales = (torch.rand(m, 1, generator=g).to(DEV), torch.rand(n, generator=g).to(DEV), torch.bfloat16) if fp8 else ()
    run = lambda: ops.linear_few(x, w, None, silu, *scales)
    run()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = run()
    for _ in range(4):
        x.copy_(cast(torch.randn(m, k, generator=g)))
        graph.replay()
        torch.cuda.synchronize()
        got = y.clone()
        assert torch.equal(got, run())
