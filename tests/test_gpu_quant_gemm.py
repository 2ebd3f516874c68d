"""GPU parity of the raw-row products of many tokens on the fp16 matrix cores
(gpeed_matmul_rows_ws): tile and split edges against the oracle, precision
against float64, non-finite values against the float32 kernels.
"""
import numpy as np
import pytest

import gpeed_amd as G
import oracle
from gpeed_amd import synth
from conftest import rel_err

pytestmark = pytest.mark.gpu
TYPES = [1, 8, 10, 11, 14, 18, 21, 22, 23, 30]
# products of exactly decoded weights, float32 sums: as the other raw-row
# products (tests/test_gpu_quant_formats.py)
TIGHT = 2e-5


def dev(a, device):
    import torch

    return torch.from_numpy(np.ascontiguousarray(a)).to(device)


def uses_ws(dt, in_dim, out_dim, n_tok):
    return G.lib().gpeed_matmul_rows_ws_bytes(dt, in_dim, out_dim, n_tok) > 0


def rows_f32(dt, w, n_rows, row0, in_dim, out_dim, x):
    """The entry point without a workspace (float32 products)."""
    import torch

    y = torch.empty(x.shape[0], out_dim, device=x.device)
    assert G.lib().gpeed_matmul_rows(dt, G._ptr(w), n_rows, row0, in_dim, out_dim, G._ptr(x), x.shape[0], G._ptr(y),
                                     G._stream()) == 0
    return y


# (in_dim, rows, row0, tokens): one row past a row tile and an odd row count
# whose bytes end inside a dword; one token past 16, 32, 64 and 128; K splits of
# unequal length (9 blocks); one K split (4096 rows x 257 tokens)
SIZES = [(2304, 129, 3, 5), (2048, 127, 1, 17), (2304, 33, 0, 33), (2048, 200, 37, 65), (1024, 64, 0, 129),
         (1024, 4100, 1, 257)]


@pytest.mark.parametrize("dt", TYPES)
@pytest.mark.parametrize("in_dim,rows,row0,n_tok", SIZES)
def test_edges_vs_oracle(gpu, dt, in_dim, rows, row0, n_tok):
    assert uses_ws(dt, in_dim, rows, n_tok)
    w = synth.quant_matrix(61, dt, dt, rows + row0, in_dim)
    X = synth.normal(61, n_tok, n_tok * in_dim).reshape(n_tok, in_dim)
    Y = G.matmul_rows(dt, dev(w.reshape(-1), gpu), rows + row0, row0, in_dim, rows, dev(X, gpu)).cpu().numpy()
    keep = np.r_[0:3, n_tok - 2:n_tok]  # the oracle is slow: the first and last tokens
    assert np.isfinite(Y).all()
    assert rel_err(Y[keep], oracle.matmul_rows(dt, w, row0, in_dim, rows, X[keep])) < TIGHT


@pytest.mark.parametrize("dt", [1, 8, 30])
@pytest.mark.parametrize("in_dim", [1056, 2080, 8224])
def test_partial_last_chunk(gpu, dt, in_dim):
    """Formats whose rows need not be whole 128-column chunks (and rows past
    what the preparation keeps in registers)."""
    rows, n_tok = 70, 19
    w = synth.quant_matrix(62, dt, dt, rows, in_dim)
    X = synth.normal(62, in_dim, n_tok * in_dim).reshape(n_tok, in_dim)
    assert uses_ws(dt, in_dim, rows, n_tok)
    Y = G.matmul_rows(dt, dev(w.reshape(-1), gpu), rows, 0, in_dim, rows, dev(X, gpu)).cpu().numpy()
    assert rel_err(Y, oracle.matmul_rows(dt, w, 0, in_dim, rows, X)) < TIGHT


@pytest.mark.parametrize("dt", [1, 11])
@pytest.mark.parametrize("n_tok", [66, 96, 128, 200, 300])
def test_token_tiles_vs_float32(gpu, dt, n_tok):
    """A 6144 x 6144 product at the token counts where the launch takes 4, 6, 7
    and 8 token tiles of 16 a workgroup, partly filled ones among them."""
    n = 6144
    w = dev(synth.quant_matrix(68, dt, dt, n, n).reshape(-1), gpu)
    X = dev(synth.normal(68, n_tok, n_tok * n).reshape(n_tok, n), gpu)
    Y = G.matmul_rows(dt, w, n, 0, n, n, X).cpu().numpy()
    assert rel_err(Y, rows_f32(dt, w, n, 0, n, n, X).cpu().numpy()) < 2 * TIGHT  # (both sides' order)


@pytest.mark.parametrize("dt", TYPES)
@pytest.mark.parametrize("n_tok", [8, 40, 300])
def test_no_less_precise_than_float32(gpu, dt, n_tok):
    """Against float64, no further off than the float32 kernels (5% for the
    chance of one sample)."""
    in_dim, rows = 4096, 128
    w = synth.quant_matrix(63, dt, dt, rows, in_dim)
    X = synth.normal(63, n_tok, n_tok * in_dim).reshape(n_tok, in_dim)
    X[:, ::64] *= 8
    wd, xd = dev(w.reshape(-1), gpu), dev(X, gpu)
    ref = X.astype(np.float64) @ oracle.dequantize(w.reshape(-1), rows * in_dim, dtype=dt).reshape(
        rows, in_dim).astype(np.float64).T
    err = [np.linalg.norm(y.cpu().numpy() - ref) / np.linalg.norm(ref)
           for y in (G.matmul_rows(dt, wd, rows, 0, in_dim, rows, xd), rows_f32(dt, wd, rows, 0, in_dim, rows, xd))]
    assert err[0] <= 1.05 * err[1], err


@pytest.mark.parametrize("dt", [1, 8, 11, 30])
@pytest.mark.parametrize("rows,n_tok", [(200, 40), (4096, 300)])
def test_non_finite_values(gpu, dt, rows, n_tok):
    """Infinities and NaN in X and in the weights give what the float32
    kernels give, with and without K splits; a token of zeros and one near the
    largest float stay exact."""
    import torch

    in_dim = 1024
    w = synth.quant_matrix(64, dt, dt, rows, in_dim).reshape(rows, -1).copy()
    at = {1: 8, 8: 34, 11: 108, 30: 8}[dt]  # an F16 / BF16 weight, the second block's d, the first block's
    w[7, at:at + 2] = [0, 0x7C] if dt != 30 else [0x80, 0x7F]  # infinity
    w[rows - 1, at:at + 2] = [1, 0x7C] if dt != 30 else [0xC0, 0x7F]  # NaN
    X = synth.normal(64, rows, n_tok * in_dim).reshape(n_tok, in_dim)
    X[3, 5], X[17, 100], X[20, 7], X[21, 9], X[22] = np.inf, np.nan, -np.inf, 3e38, 0.0
    wd, xd = dev(w.reshape(-1), gpu), dev(X, gpu)
    assert uses_ws(dt, in_dim, rows, n_tok)
    y, ref = G.matmul_rows(dt, wd, rows, 0, in_dim, rows, xd), rows_f32(dt, wd, rows, 0, in_dim, rows, xd)
    for f in (torch.isnan, torch.isposinf, torch.isneginf):
        assert torch.equal(f(y), f(ref))
    ok = torch.isfinite(ref)
    assert float(((y - ref).abs()[ok] / torch.where(ok, ref, 0.0).pow(2).mean(1, keepdim=True).sqrt().clamp_min(
        1e-30).expand_as(ref)[ok]).max()) < TIGHT


@pytest.mark.parametrize("dt", [8, 11, 18, 21, 22])
@pytest.mark.parametrize("n_tok", [1, 3])
def test_last_row_ends_inside_a_dword(gpu, dt, n_tok):
    """Few-token slices over an odd number of rows of 2 bytes more than whole
    dwords: the last row's last bytes count."""
    in_dim, rows = (160, 127) if dt == 8 else (256, 127)
    w = synth.quant_matrix(65, dt, dt, rows, in_dim)
    X = synth.normal(65, n_tok, n_tok * in_dim).reshape(n_tok, in_dim)
    Y = G.matmul_rows(dt, dev(w.reshape(-1), gpu), rows, 0, in_dim, rows, dev(X, gpu)).cpu().numpy()
    assert rel_err(Y, oracle.matmul_rows(dt, w, 0, in_dim, rows, X)) < TIGHT


def test_captured_and_on_another_stream(gpu):
    """A captured call replays (no launch depends on host state), and a call on
    a stream of its own matches."""
    import torch

    in_dim, rows, n_tok = 2048, 256, 20
    w = dev(synth.quant_matrix(66, 14, 14, rows, in_dim).reshape(-1), gpu)
    X = torch.randn(n_tok, in_dim, device=gpu)
    ref = G.matmul_rows(14, w, rows, 0, in_dim, rows, X)
    out = torch.empty_like(ref)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        G.matmul_rows(14, w, rows, 0, in_dim, rows, X, out=out)
    for _ in range(3):
        X.copy_(torch.randn(n_tok, in_dim, device=gpu))
        ref = G.matmul_rows(14, w, rows, 0, in_dim, rows, X)
        out.zero_()
        g.replay()
        assert torch.equal(out, ref)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    y = torch.empty_like(ref)
    G.matmul_rows(14, w, rows, 0, in_dim, rows, X, out=y, stream=s)
    s.synchronize()
    assert torch.equal(y, ref)


def test_workspace_errors(gpu):
    import torch

    in_dim, rows, n_tok = 2048, 64, 20
    w = dev(synth.quant_matrix(67, 8, 8, rows, in_dim).reshape(-1), gpu)
    X, Y = torch.zeros(n_tok, in_dim, device=gpu), torch.zeros(n_tok, rows, device=gpu)
    need = G.lib().gpeed_matmul_rows_ws_bytes(8, in_dim, rows, n_tok)
    ws = torch.empty(need, dtype=torch.uint8, device=gpu)

    def call(p, n):
        return G.lib().gpeed_matmul_rows_ws(8, G._ptr(w), rows, 0, in_dim, rows, G._ptr(X), n_tok, G._ptr(Y), p, n,
                                            G._stream())

    assert call(None, need) == -1 and call(G._ptr(ws), need - 1) == -1
    assert call(G._ptr(ws), need) == 0
    assert G.lib().gpeed_matmul_rows_ws_bytes(0, in_dim, rows, n_tok) == 0  # F32 rows take none
    assert G.lib().gpeed_matmul_rows_ws_bytes(8, in_dim, rows, 1) == 0
