"""Decode products at the edges of what their entry points take (csrc/kernels/decode_linear.hip, rows_gemm.hip)."""
import pytest
import torch
import torch.nn.functional as F

from penroz.ops import _ext

pytestmark = pytest.mark.gpu
DEV, BF = "cuda", torch.bfloat16


@pytest.mark.parametrize("M", [1, 3, 4])
@pytest.mark.parametrize("act", [0, 1, 2])
def test_products_over_no_columns(M, act):
    """A row of no columns has no last piece for a load to be held to: the sum is nothing, the result act(bias)."""
    N, k = 48, _ext.kernels()
    x, w, b = torch.empty(M, 8, device=DEV, dtype=BF)[:, :0], torch.empty(N, 0, device=DEV, dtype=BF), torch.randn(N, device=DEV).to(BF)
    none, rows = torch.empty(0, device=DEV), torch.empty(M, 0, device=DEV)
    for bias in (b, None):
        want = torch.zeros(N, device=DEV) if bias is None else b.float()
        if act:
            want = F.gelu(want, approximate="tanh" if act == 2 else "none")
        for call in (lambda o: k.decode_gemv(x, None, None, None, None, None, None, 0.0, w, bias, o, act),
                     lambda o: k.decode_gemv(None, rows, None, None, None, none, none, 1e-5, w, bias, o, act),
                     lambda o: k.decode_ln_gemm(rows, none, none, 1e-5, w, bias, o, act)):
            big = torch.full((M + 1, N + 8), 7.0, device=DEV, dtype=BF)
            call(big[:M, :N])
            # the erf of another implementation may fall on the other side of a tie of the one rounding
            assert torch.all((big[:M, :N].float() - want).abs() <= 2.0 ** -8 * want.abs())
            assert (big[M] == 7).all() and (big[:, N:] == 7).all()


@pytest.mark.parametrize("M", [1, 4, 5, 33])
def test_other_products_over_no_columns(M):
    N, D, k = 64, 16, _ext.kernels()
    x, w, b = torch.empty(M, 8, device=DEV, dtype=BF)[:, :0], torch.empty(N, 0, device=DEV, dtype=BF), torch.randn(N, device=DEV).to(BF)
    for bias in (b, None):
        old = torch.randn(M, N, device=DEV)
        got = old.clone()
        k.decode_gemm_acc(x, w, bias, got)
        assert torch.equal(got, old if bias is None else old + b.float())
    if M > 4:
        none = torch.empty(0, device=DEV)
        out = torch.empty(M, N, device=DEV, dtype=BF)
        k.decode_ln_gemm(torch.empty(M, 0, device=DEV), none, none, 1e-5, w, b, out, 0)
        assert torch.equal(out, b.expand(M, N))
        return
    cs = torch.ones(D // 2, device=DEV)
    for mode, n in ((1, N // 2), (2, N)):
        out = torch.full((M, n), 7.0, device=DEV, dtype=BF)
        k.decode_gemv_pair(x, w, out, mode, 2, D, 2, cs, cs)
        assert (out == 0).all()
    with pytest.raises(RuntimeError):  # its norms are over the columns
        k.decode_norm_pair(x, None, None, torch.empty(0, device=DEV, dtype=BF), 3, 0.0, 1e-6, None, w, out, 2, 0, D, 2, cs, cs)


def test_prompt_rows_of_no_width():
    qkv, cache = torch.empty(1, 2, 0, device=DEV, dtype=BF), torch.empty(1, 1, 4, 0, device=DEV, dtype=BF)
    assert _ext.kernels().prompt_kv(qkv, None, cache, cache, 0, 1, 1) is None


def test_tables_of_no_rows_are_refused():
    """Token and position are held to the table's rows, of which the last would be -1."""
    k, C, N = _ext.kernels(), 64, 128
    z = lambda *s, dt=BF: torch.zeros(*s, device=DEV, dtype=dt)
    tok, pos, out, w = z(1, dt=torch.int64), z(1, dt=torch.int64), z(1, N), z(N, C)
    f = torch.float32
    for wte, wpe in ((z(0, C), z(4, C)), (z(4, C), z(0, C))):
        with pytest.raises(RuntimeError):
            k.decode_gemv(None, None, None, None, z(1, C, dt=f), z(C, dt=f), z(C, dt=f), 1e-5, w, None, out, 0, emb_idx=tok, emb_wte=wte,
                          emb_wpe=wpe, emb_pos=pos)
    with pytest.raises(RuntimeError):
        k.decode_norm_pair(None, None, None, z(C), 3, 0.0, 1e-6, z(1, C), w, out[:, :N // 2], 1, 2, tok=tok, table=z(0, C))
