"""mui_linear_ws: the prompt linear with a caller-provided workspace (parity gate: north_star's 1e-2
relative against the fp32-accumulating oracle; bit-equal results call after call)."""
import pytest
import torch

from muillm_amd import _lib
import oracle
from tests.util import assert_parity

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _gen(seed):
    g = torch.Generator(device="cpu")
    g.manual_seed(seed)
    return g


def _mk(shape, g, std=1.0, mean=0.0, dtype=torch.float16):
    return (mean + std * torch.randn(shape, generator=g)).to(dtype)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("tokens,n,k", [(64, 4096, 14336), (256, 4096, 14336), (33, 4096, 14336), (200, 1000, 6152)])
def test_linear_workspace_entry_shares_k_between_workgroups(tokens, n, k, dtype):
    """mui_linear_ws through the C ABI: few output tiles and a long K, so K is shared between
    workgroups that exchange partial tiles through the caller's workspace. Checked against the oracle
    and against the call without a workspace; three calls in a row on the same workspace (its
    counters must be back at zero after each) give the same bits, whichever workgroup arrived last."""
    lib = _lib.load()
    s = torch.cuda.current_stream().cuda_stream
    g = _gen(11)
    w, x = _mk((n, k), g, 0.02, dtype=dtype), _mk((tokens, k), g, dtype=dtype)
    r, b = _mk((tokens, n), g, dtype=dtype), _mk((n,), g, 0.5, dtype=dtype)
    ref = oracle.linear(x, w, None, 0.0, b, r)
    wd, xd, rd, bd = w.to(DEV), x.to(DEV), r.to(DEV), b.to(DEV)
    ws = torch.zeros(lib.mui_linear_workspace_bytes(), dtype=torch.uint8, device=DEV)
    code = 0 if dtype == torch.float16 else 1
    outs = []
    for _ in range(3):
        y = torch.zeros(tokens, n, dtype=dtype, device=DEV)
        st = lib.mui_linear_ws(s, code, wd.data_ptr(), k, xd.data_ptr(), None, 0.0, None, bd.data_ptr(), rd.data_ptr(),
                               y.data_ptr(), n, k, tokens, ws.data_ptr(), ws.numel())
        assert st == 0
        outs.append(y)
    torch.cuda.synchronize()
    assert_parity(outs[0], ref, 1e-2, f"prompt linear with workspace {tokens}x{n}x{k}")
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])
    assert int(ws[:4096].to(torch.int32).sum()) == 0  # every counter returned to zero
    plain = torch.zeros(tokens, n, dtype=dtype, device=DEV)
    assert lib.mui_linear(s, code, wd.data_ptr(), k, xd.data_ptr(), None, 0.0, None, bd.data_ptr(), rd.data_ptr(),
                          plain.data_ptr(), n, k, tokens) == 0
    assert_parity(outs[0], plain.double().cpu(), 1e-2, "workspace vs plain call",
                  elementwise=None)
    # a workspace that is too small or misaligned is not used (the call is then mui_linear); a size without a pointer is refused
    small = torch.zeros(tokens, n, dtype=dtype, device=DEV)
    assert lib.mui_linear_ws(s, code, wd.data_ptr(), k, xd.data_ptr(), None, 0.0, None, bd.data_ptr(), rd.data_ptr(),
                             small.data_ptr(), n, k, tokens, ws.data_ptr(), 1024) == 0
    assert torch.equal(small, plain)
    assert lib.mui_linear_ws(s, code, wd.data_ptr(), k, xd.data_ptr(), None, 0.0, None, bd.data_ptr(), rd.data_ptr(),
                             small.data_ptr(), n, k, tokens, None, 4096) == -1


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("tokens,n,k", [(17, 4096, 14344), (33, 1000, 10248), (41, 1000, 6152), (64, 4096, 14344), (96, 1000, 6152),
                                        (128, 4096, 14344), (128, 1000, 6152), (256, 4096, 14336)])
def test_tile_exchange_at_a_k_that_steps_do_not_divide(tokens, n, k, dtype):
    """K no multiple of 256 (or more than 128 tokens): 128 x 128 tiles whose workgroups exchange partial tiles and count themselves in.
    The scratch behind the counters has been written, the counters are back at zero, and call after call gives the same bits."""
    lib = _lib.load()
    g = _gen(tokens + k)
    w, x, r = _mk((n, k), g, 0.02, dtype=dtype), _mk((tokens, k), g, dtype=dtype), _mk((tokens, n), g, dtype=dtype)
    ref = oracle.linear(x, w, None, 0.0, None, r)
    wd, xd, rd = w.to(DEV), x.to(DEV), r.to(DEV)
    ws = torch.zeros(lib.mui_linear_workspace_bytes(), dtype=torch.uint8, device=DEV)
    outs = []
    for _ in range(4):
        y = torch.zeros(tokens, n, dtype=dtype, device=DEV)
        _lib.check(lib.mui_linear_ws(torch.cuda.current_stream().cuda_stream, 0 if dtype == torch.float16 else 1, wd.data_ptr(), k, xd.data_ptr(),
                                     None, 0.0, None, None, rd.data_ptr(), y.data_ptr(), n, k, tokens, ws.data_ptr(), ws.numel()), "mui_linear_ws")
        assert int(ws[:4096].count_nonzero()) == 0
        outs.append(y)
    assert int(ws[4096:].count_nonzero()) > 0, "K was not shared"
    assert_parity(outs[0], ref, 1e-2, f"tile exchange {tokens}x{n}x{k}")
    assert all(torch.equal(outs[0], y) for y in outs[1:])


@torch.no_grad()
def test_threads_on_one_stream():
    """Threads share the stream that they start on, and its scratch: what a linear's first launch leaves there is its own until its second has read it."""
    import threading

    from muillm_amd import muillm_ext

    def product(seed, kind, n, k, tokens):
        g = torch.Generator(device=DEV).manual_seed(seed)
        x, res = torch.randn(tokens, k, device=DEV, generator=g).half(), torch.randn(tokens, n, device=DEV, generator=g).half()
        if kind == "16":
            w = (torch.randn(n, k, device=DEV, generator=g) * k ** -0.5).half()
            return lambda: muillm_ext.muillm_linear_forward(None, x, w, residual=res)
        codes, scales = torch.randint(-128, 128, (n, k), device=DEV, generator=g, dtype=torch.int16).to(torch.int8), torch.full((n,), 1e-3, device=DEV).half()
        return lambda: muillm_ext.mui_int8_channel_linear_forward(x, codes, scales, residual=res)

    # two launches beyond 128 tokens and up to them, of codes, and one whose last workgroups add up
    calls = [product(1, "16", 2048, 8192, 333), product(2, "16", 4096, 14336, 48), product(3, "8", 2048, 8192, 100), product(4, "16", 1024, 8200, 200), product(5, "8", 4096, 8192, 333)]
    wants, wrong, start = [call() for call in calls], [], threading.Barrier(len(calls))
    torch.cuda.synchronize()

    def work(i):
        start.wait()
        for _ in range(40):
            outs = [calls[i]() for _ in range(5)]
            if not all(torch.equal(o, wants[i]) for o in outs):
                wrong.append(i)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(calls))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert not wrong
