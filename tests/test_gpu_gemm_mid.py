"""The kernels that jh_op_gemm_splitk takes between the small-batch kernel's first round of tiles and the tiled
kernels: the slab-resident GEMM at K = 384 (csrc/gemm_slab.hip), and the weight-stationary one reading W row-major at
K = 768 and 1152 (csrc/gemm_ws.hip).  Sizes lie at the edges of the dispatch rule, of the 16-token units and of the
steps of two units, and where a range has one unit."""
import numpy as np
import pytest
import torch

from julia1_amd import abi, hip

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16
ALL = [abi.EPI_STORE_BF16, abi.EPI_ROPE_BF16, abi.EPI_GEGLU_BF16, abi.EPI_RESID_F32, abi.EPI_BIAS_BF16,
       abi.EPI_BIAS_RELU_BF16, abi.EPI_BIAS_F32]


def _operands(rows, n, k, epi, seed, ldx):
    """x (row stride ldx), w, keyword operands, and the result in 64 bits with the sum of its terms' magnitudes."""
    g = torch.Generator("cuda").manual_seed(seed)
    x = torch.randn(rows, ldx, generator=g, device="cuda").to(BF16)[:, :k]
    w = (torch.randn(n, k, generator=g, device="cuda") * 0.05).to(BF16)
    prod, size = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    kw = {}
    if epi == abi.EPI_ROPE_BF16:
        rc = 64 * (n // 64 - n // 192)
        cos, sin = (torch.from_numpy(t).cuda() for t in hip.rope_table(10000.0, 8192))
        pos = torch.randint(0, 8192, (rows,), device="cuda", generator=g, dtype=torch.int32)
        kw = dict(pos=pos, cos=cos, sin=sin, rope_cols=rc)
        c, s = (t[pos.long()].double()[:, None] for t in (cos, sin))
        a = prod[:, :rc].reshape(rows, -1, 2, 32)
        rot = torch.stack([a[:, :, 0] * c - a[:, :, 1] * s, a[:, :, 1] * c + a[:, :, 0] * s], 2).reshape(rows, rc)
        m = size[:, :rc].reshape(rows, -1, 2, 32).sum(2, keepdim=True).expand(-1, -1, 2, -1).reshape(rows, rc)
        prod, size = torch.cat([rot, prod[:, rc:]], 1), torch.cat([m, size[:, rc:]], 1)
    if epi == abi.EPI_GEGLU_BF16:
        a, m = prod.reshape(rows, -1, 2, 32), size.reshape(rows, -1, 2, 32)
        up = a[:, :, 1].abs()
        prod = (torch.nn.functional.gelu(a[:, :, 0]) * a[:, :, 1]).reshape(rows, -1)
        # an error of the gate is scaled by up, one of up by gelu(gate) <= |gate|; |gelu'| < 1.13
        size = (1.13 * m[:, :, 0] * (up + m[:, :, 1] * 2.0 ** -20) + a[:, :, 0].abs() * m[:, :, 1]).reshape(rows, -1)
    if epi in (abi.EPI_BIAS_BF16, abi.EPI_BIAS_RELU_BF16, abi.EPI_BIAS_F32, abi.EPI_RESID_F32):
        kw["bias"] = torch.randn(n, generator=g, device="cuda")
        prod = prod + kw["bias"].double()
        if epi == abi.EPI_BIAS_RELU_BF16:
            prod = prod.clamp_min(0.0)
    return x, w, kw, prod, size


def _out(rows, width, epi, col, pad, seed):
    g = torch.Generator("cuda").manual_seed(seed)
    f32 = epi in (abi.EPI_RESID_F32, abi.EPI_BIAS_F32)
    return torch.randn(rows + 1, col + width + pad, generator=g, device="cuda").to(torch.float32 if f32 else BF16)


# (rows, n): the first ones each one row past (or at) the small-batch kernel's last size and the rule's end; then a
# 128-row slab count that is no multiple of three, 2^22 * 3 outputs (from where few columns of bf16 run here again), and
# 384-row slabs from 16384 rows on
SLAB = [(2721, 384), (1345, 1152), (1792, 1152), (673, 2304), (4097, 256), (4323, 384), (16384, 768), (16384, 1152), (16385, 2304),
        (20003, 1536)]


@pytest.mark.parametrize("rows,n", SLAB)
@pytest.mark.parametrize("epi", ALL)
def test_slab_against_64_bits(rows, n, epi):
    """Each epilogue at K = 384, strided X and a column offset in a wider output.  FP32 sums of 384 products err by at
    most 384 * 2^-24 of their terms' magnitudes (and two roundings more for bias and residual); bf16 outputs add half
    a bf16 step, 2^-9, and the rational erf 1e-6."""
    k, col, pad = 384, 64, 16
    x, w, kw, want, size = _operands(rows, n, k, epi, 7 * rows + n + epi, k + 64)
    out = _out(rows, want.shape[1], epi, col, pad, rows + epi)
    before = out.clone()
    ws = torch.empty(6 << 20, device="cuda")
    hip.op_gemm_splitk(epi, x, w, out[:rows], ws, col=col, **kw)
    torch.cuda.synchronize()
    got = out[:rows, col:col + want.shape[1]].double()
    if epi == abi.EPI_RESID_F32:
        old = before[:rows, col:col + want.shape[1]].double()
        want, size = want + old, size + old.abs()
    tol = 384 * 2.0 ** -24 * size + 2.0 ** -22 * want.abs() + 1e-6
    if got.shape and out.dtype == BF16:
        tol = tol + 2.0 ** -8 * want.abs() + (2e-6 * size if epi == abi.EPI_GEGLU_BF16 else 0)
    assert bool(((got - want).abs() <= tol).all()), ((got - want).abs() - tol).max().item()
    out[:rows, col:col + want.shape[1]] = before[:rows, col:col + want.shape[1]]
    assert torch.equal(out, before)  # nothing outside the output's rows and columns


@pytest.mark.parametrize("rows,n,k,epi", [
    (673, 768, 768, abi.EPI_RESID_F32), (2687, 768, 768, abi.EPI_BIAS_F32), (2049, 256, 768, abi.EPI_STORE_BF16),
    (2053, 256, 768, abi.EPI_BIAS_F32), (449, 2304, 768, abi.EPI_ROPE_BF16), (896, 2304, 768, abi.EPI_GEGLU_BF16),
    (6001, 2304, 768, abi.EPI_ROPE_BF16), (6000, 2304, 768, abi.EPI_GEGLU_BF16), (382, 3072, 768, abi.EPI_BIAS_RELU_BF16),
    (700, 768, 768, abi.EPI_BIAS_BF16), (673, 384, 1152, abi.EPI_RESID_F32), (2049, 128, 1152, abi.EPI_RESID_F32),
    (321, 768, 1152, abi.EPI_RESID_F32), (4323, 384, 1152, abi.EPI_RESID_F32)])
def test_row_major_equals_packed(rows, n, k, epi):
    """jh_op_gemm_splitk on row-major W gives the bits of jh_op_gemm_ws on the packed copy."""
    x, w, kw, _, _ = _operands(rows, n, k, epi, rows + n + k, k + 8)
    width = n // 2 if epi == abi.EPI_GEGLU_BF16 else n
    out = _out(rows, width, epi, 0, 16, 3)
    again = out.clone()
    ws = torch.empty(6 << 20, device="cuda")
    hip.op_gemm_splitk(epi, x, w, out[:rows], ws, **kw)
    hip.op_gemm_ws(epi, x, hip.pack_ws(w), n, k, again[:rows], **kw)
    torch.cuda.synchronize()
    assert torch.equal(out, again)
    assert np.isfinite(out.float().cpu().numpy()).all()


def test_wide_output_stride():
    """Output rows 2^26 elements apart: 16 of them are 2^31 bytes, so the kernels that address them with 32-bit byte
    offsets leave the call to the others.  Tolerance: 768 sums of bf16 products and half a bf16 step, as above."""
    rows, n, k = 449, 2304, 768
    if torch.cuda.mem_get_info()[0] < (rows + 64) << 27:
        pytest.skip("needs 56 GiB of free device memory")
    x, w, _, want, size = _operands(rows, n, k, abi.EPI_STORE_BF16, 5, k)
    out = torch.empty(rows, 1 << 26, device="cuda", dtype=BF16)  # 56 GiB, of which the first 2304 columns are touched
    hip.op_gemm_splitk(abi.EPI_STORE_BF16, x, w, out, torch.empty(6 << 20, device="cuda"))
    torch.cuda.synchronize()
    got = out[:, :n].double()
    del out
    torch.cuda.empty_cache()
    tol = 768 * 2.0 ** -24 * size + 2.0 ** -8 * want.abs() + 1e-6
    assert bool(((got - want).abs() <= tol).all()), ((got - want).abs() - tol).max().item()
