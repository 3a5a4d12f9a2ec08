"""GPU parity of the per-token quantizer (pq_quant_rows) against the CPU oracle: bit-exact int8 codes and
fp32 scales (deploy/int8_exec.py:508-509 semantics), incl. the routed row gather, row-slice views, the
per-element kernel, all-zero rows, exact ties and the full c1 / c2a shapes."""
import numpy as np
import pytest
import torch

from conftest import bits, dcode

pytestmark = pytest.mark.gpu


def _check(oracle, x, row_idx=None, q=None, s=None):
    from pyraquant_amd import int8_exec as E

    if q is None:
        q, s = E.quant_rows(x, row_idx)
    torch.cuda.synchronize()
    xb = bits(x.cpu() if x.stride(1) == 1 else x.contiguous())
    ri = None if row_idx is None else row_idx.cpu().numpy()
    qo, so = oracle.quant_rows(xb, dcode(x.dtype), ri)
    qg, sg = q.cpu().numpy(), s.cpu().numpy()
    assert qg.shape == qo.shape and sg.shape == so.shape
    mism = int((qg != qo).sum())
    assert mism == 0, f"{mism} code mismatches of {qo.size}"
    assert np.array_equal(sg.view(np.uint32), so.view(np.uint32)), "scales differ"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,K", [(1, 3072), (7, 1280), (64, 640), (300, 3072), (33, 12288), (17, 15360),
                                 (5, 2048), (9, 2560), (3, 8), (2, 16384)])
def test_quant_rows_shapes(oracle, cuda, dtype, M, K):
    from pyraquant_amd.workloads import make_x

    x = make_x(M, K, dtype, seed=M * 7 + K).to(cuda)
    _check(oracle, x)


@pytest.mark.parametrize("K", [1, 5, 100, 1000, 3000])
def test_quant_rows_scalar_kernel(oracle, cuda, K):
    """K % 8 != 0 takes the per-element kernel."""
    from pyraquant_amd.workloads import make_x

    x = make_x(37, K, torch.bfloat16, seed=K).to(cuda)
    _check(oracle, x)


def test_quant_rows_unaligned_view(oracle, cuda):
    """A row-slice view (ldx > K, odd column offset) runs without a copy on the per-element kernel and a
    16-byte aligned view on the vector kernel."""
    from pyraquant_amd.workloads import make_x

    base = make_x(100, 3072 + 15360, torch.bfloat16, seed=5).to(cuda)
    _check(oracle, base[:, 3072:])          # aligned offset (3072 * 2 bytes), ldx = 18432
    _check(oracle, base[:, 1:3073])         # unaligned offset -> per-element kernel


def test_quant_rows_edge_values(oracle, cuda):
    """All-zero rows (scale 1e-8/127), tiny rows, exact ties (x = (k + 1/2) s), +-0, subnormals, a row
    whose absmax is negative, and huge magnitudes."""
    K = 512
    x = torch.zeros(8, K)
    x[1, :] = 1e-12                                   # below the 1e-8 clamp
    # row 2: exact half-integer multiples of the scale: a = 127 -> s = 1, x = k + 0.5
    x[2, 0] = 127.0
    x[2, 1:255] = torch.arange(-127, 127).float() + 0.5
    x[3, 0] = -127.0                                  # negative absmax
    x[3, 1:] = torch.linspace(-127, 127, K - 1)
    x[4, :] = torch.randn(K) * 1e-39                  # subnormal fp32 -> bf16 subnormals
    x[5, :] = torch.randn(K) * 1e30
    x[6, ::2] = -0.0
    x[6, 1] = 3.0
    x[7, :] = torch.randn(K)
    xb = x.to(torch.bfloat16).to(cuda)
    _check(oracle, xb)
    # ties at a non-unit scale: a = 254 -> s = 2, x = 2k + 1 are exact ties in x / s
    y = torch.zeros(2, K)
    y[0, 0] = 254.0
    y[0, 1:128] = torch.arange(-127, 0).float() * 2 + 1
    y[1, 0] = 63.5
    y[1, 1:200] = torch.arange(1, 200).float() * 0.25
    _check(oracle, y.to(torch.bfloat16).to(cuda))
    _check(oracle, y.to(torch.float16).to(cuda))


def test_quant_rows_gather(oracle, cuda):
    """Routed gather fused into the quantizer: output row m quantizes x[row_idx[m]]; duplicates allowed."""
    from pyraquant_amd.workloads import make_x

    x = make_x(1000, 3072, torch.bfloat16, seed=11).to(cuda)
    g = torch.Generator().manual_seed(3)
    idx = torch.randint(0, 1000, (513,), generator=g, dtype=torch.int32)
    idx[:4] = torch.tensor([999, 0, 0, 5], dtype=torch.int32)
    _check(oracle, x, idx.to(cuda))


def test_quant_rows_empty(cuda):
    from pyraquant_amd import int8_exec as E

    x = torch.empty(0, 3072, dtype=torch.bfloat16, device=cuda)
    q, s = E.quant_rows(x)
    assert q.shape == (0, 3072) and s.shape == (0,)


@pytest.mark.parametrize("cfg", ["c1", "c2a"])
def test_quant_rows_full_size(oracle, cuda, cfg):
    """Full c1 / c2a shapes, bit-exact against the oracle."""
    from pyraquant_amd.workloads import CONFIGS, make_x

    c = CONFIGS[cfg]
    x = make_x(c.M, c.K, c.dtype).to(cuda)
    _check(oracle, x)


def test_quant_rows_routed_c4(oracle, cuda):
    """Config 4: gather of the 33,316 routed rows of the 65,536-row canvas."""
    from pyraquant_amd.workloads import make_x, routed_rows

    x = make_x(65536, 3072, torch.bfloat16).to(cuda)
    idx = routed_rows(cuda)
    assert idx.numel() == 33316
    _check(oracle, x, idx)


@pytest.mark.parametrize("fixture", ["quant_bf16.npz", "quant_f16.npz"])
def test_quant_rows_golden_fixture(cuda, fixture):
    """The HIP quantizer reproduces the committed golden vectors (torch CPU, deploy/int8_exec.py:508-509)."""
    import os

    from pyraquant_amd import int8_exec as E

    f = np.load(os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", fixture), allow_pickle=False)
    dt = torch.bfloat16 if int(f["dtype"]) == 0 else torch.float16
    x = torch.from_numpy(f["x_bits"].view(np.int16)).view(dt).to(cuda)
    q, s = E.quant_rows(x)
    assert np.array_equal(q.cpu().numpy(), f["q"])
    assert np.array_equal(s.cpu().numpy().view(np.uint32), f["s"].view(np.uint32))


def test_linear_golden_fixture(cuda):
    """Golden layer (tests/golden/linear_lr.npz): codes, int32 accumulator and no-low-rank fp32 epilogue
    bit-exact, low-rank output within the tolerance of the float64 value."""
    import os

    from conftest import MAX_REL, MEAN_REL, rel_errors
    from pyraquant_amd import int8_exec as E

    f = np.load(os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "linear_lr.npz"), allow_pickle=False)
    x = torch.from_numpy(f["x_bits"].view(np.int16)).view(torch.bfloat16).to(cuda)
    wq = torch.from_numpy(f["w_q"]).to(cuda)
    ws = torch.from_numpy(f["w_s"]).to(cuda)
    b = torch.from_numpy(f["bias"]).to(cuda)
    l1 = torch.from_numpy(f["l1_bits"].view(np.int16)).view(torch.bfloat16)
    l2 = torch.from_numpy(f["l2_bits"].view(np.int16)).view(torch.bfloat16)
    q, s = E.quant_rows(x)
    assert np.array_equal(q.cpu().numpy(), f["q"])
    acc = E.int8_gemm_i32(q, wq)
    assert np.array_equal(acc.cpu().numpy(), f["acc"])
    y = E.int8_gemm_fused(q, s, wq, ws, b, torch.bfloat16)
    ref = torch.from_numpy(f["y_nolr"]).to(torch.bfloat16)
    assert torch.equal(y.cpu(), ref)
    t = E.lowrank_down(x, l1.t().contiguous().to(cuda))
    ylr = E.int8_gemm_lr(q, s, wq, ws, b, t, l2.to(cuda), torch.bfloat16)
    mx, mean = rel_errors(ylr.float().cpu().numpy(), f["y_lr_f64"])
    assert mx <= MAX_REL and mean <= MEAN_REL, (mx, mean)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_quant_rows_every_mantissa_pair(oracle, cuda, dtype):
    """Codes come from a branch-free Newton step, whose rounding depends on the row maximum's and the element's
    mantissas and their exponent difference alone: every maximum (all 128 mantissas in bf16, all 1024 in fp16) against
    every element mantissa at exponent differences 0 .. 9 (below that every code is 0), both signs; and the floor's scale
    (rows with no element above 1e-8, in bf16) against every element that has a code; against the oracle bit for bit,
    in the packed and the row-major kernel."""
    from pyraquant_amd import int8_exec as E

    bf = dtype == torch.bfloat16
    n, base = (128, 0x3F80) if bf else (1024, 0x4C00)
    maxima = torch.arange(n) + base
    elems = (torch.arange(-9 * n, n) + base).to(torch.int16)
    elems = torch.cat([elems, elems | torch.tensor(-32768, dtype=torch.int16)])
    rows = []
    for a in maxima.tolist():
        keep = torch.where((elems & 0x7FFF) <= a, elems, torch.zeros_like(elems))
        keep[0] = a
        rows.append(keep)
    if bf:
        floor = int(torch.tensor(1e-8).bfloat16().view(torch.int16)) - 1   # the largest below 1e-8, and nine binades
        low = torch.arange(floor - 9 * n, floor + 1).to(torch.int16)
        low = torch.cat([low, low | torch.tensor(-32768, dtype=torch.int16)])
        assert float(low[9 * n].view(dtype)) <= 1e-8
        rows.append(torch.nn.functional.pad(low, (0, elems.numel() - low.numel())))
    x = torch.stack(rows).view(dtype)
    x = torch.nn.functional.pad(x, (0, (-x.shape[1]) % 64))
    for r0 in range(0, x.shape[0], 64):
        part = x[r0:r0 + 64].contiguous()
        for c0 in range(0, part.shape[1], 8192):   # (the vectorised kernels take rows up to 16384)
            xc = part[:, c0:c0 + 8192].clone()
            xc[:, 0] = part[:, 0]
            q, s = E.quant_rows(xc.to(cuda))
            qo, so = oracle.quant_rows(bits(xc), dcode(dtype))
            assert (q.cpu().numpy() == qo).all() and (s.cpu().numpy() == so).all()
            qp, _ = E.quant_rows_packed(xc.to(cuda))
            assert torch.equal(qp, E.pack_k64(q))


def _codes_of(x):
    """Codes and scales of rows that need not be finite: a row with a NaN has the floor's scale, an infinite or NaN
    element code 0, every other clamp(rint(x / s)) (on the CPU, IEEE divisions)."""
    xf = x.float()
    a = torch.where(xf.isnan().any(1), torch.zeros(()), xf.abs().nan_to_num(nan=0.0, posinf=float("inf")).amax(1))
    s = a.clamp_min(1e-8) / 127
    q = torch.where(xf.isfinite(), (xf / s[:, None]).round().clamp(-127, 127), torch.zeros(()))
    return q.to(torch.int8), s


def _not_finite(M, K, dtype, seed):
    """Finite rows, and at `rows` ones with a NaN, an infinity or both beside elements of every magnitude."""
    from pyraquant_amd.workloads import make_x

    x = make_x(M, K, dtype, seed=seed)
    g = torch.Generator().manual_seed(seed)
    rows = sorted({0, 1, 2, 17 % M, M // 2, M - 3, M - 2, M - 1})
    for i, r in enumerate(rows):
        x[r] = torch.randint(-32768, 32768, (K,), generator=g).to(torch.int16).view(dtype).nan_to_num(0.0, 0.0, 0.0)
        x[r, 3:19] = torch.tensor([1e-8, -1e-8, 1.01e-8, 1e-7, -1e-6, 1e-5, -1e-4, 1e-3, 0.5, 1.0, -1.0, 2.0, 0.0, -0.0, 64.0, 3e4])
        if i % 3 < 2:
            x[r, (5 * r + 40) % K] = float("nan")
        if i % 3 > 0:
            x[r, K - 1], x[r, 1] = float("inf"), -float("inf")
    return x, rows


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,K", [(24, 64), (24, 520), (40, 1280), (24, 3072), (24, 12288), (24, 16384), (24, 1003)])
def test_rows_that_are_not_finite(cuda, dtype, M, K):
    """Codes of rows with NaN and infinite elements: in [-127, 127] and the same in the vectorised kernel (K % 8 == 0),
    its packed form, and the per-element kernel, which an unaligned view takes."""
    from pyraquant_amd import int8_exec as E

    x, _ = _not_finite(M, K, dtype, seed=K)
    qo, so = _codes_of(x)
    wide = torch.zeros(M, K + 8, dtype=dtype, device=cuda)
    wide[:, 1:K + 1] = x.to(cuda)
    for q, s in (E.quant_rows(x.to(cuda)), E.quant_rows(wide[:, 1:K + 1])):
        assert torch.equal(s.cpu(), so)
        assert torch.equal(q.cpu(), qo)
    if K % 64 == 0:
        qp, s = E.quant_rows_packed(x.to(cuda))
        assert torch.equal(s.cpu(), so) and torch.equal(qp, E.pack_k64(qo.to(cuda)))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,K", [(40, 1024), (40, 1280), (40, 2560), (40, 3072),             # one-pass kernel: 16, 4, 8 waves
                                 (40, 4096), (40, 12288), (4120, 12288), (2072, 15360)])      # wide kernel, and its tail
def test_rows_that_are_not_finite_lowrank(cuda, dtype, M, K):
    """The fused quantizer + down-projection: the same codes, NaN in every column of t for a row with a NaN, and no
    other row touched by it."""
    from pyraquant_amd import int8_exec as E

    x, rows = _not_finite(M, K, dtype, seed=K)
    l1t = (torch.randn(32, K, generator=torch.Generator().manual_seed(1)) * 0.05).to(dtype).to(cuda)
    clean = x.clone()
    clean[rows] = 0
    q0, s0, t0 = E.quant_rows_lowrank(clean.to(cuda), l1t)
    q, s, t = E.quant_rows_lowrank(x.to(cuda), l1t)
    qo, so = _codes_of(x)
    assert torch.equal(s.cpu(), so) and torch.equal(q, E.pack_k64(qo.to(cuda)))
    keep = torch.ones(M, dtype=torch.bool)
    keep[rows] = False
    assert torch.equal(t[keep.to(cuda)], t0[keep.to(cuda)])
    assert t[x.isnan().any(1).to(cuda)].isnan().all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("K", [64, 1280, 2048, 4096])
def test_rows_that_are_not_finite_small_layer(cuda, dtype, K):
    """The layer as one kernel against quantizer and GEMM on such rows, with weights large enough to show their codes."""
    from pyraquant_amd import int8_exec as E

    M, N = 24, 128
    x, rows = _not_finite(M, K, dtype, seed=K)
    lin = torch.nn.Linear(K, N, bias=False, device=cuda)
    with torch.no_grad():
        lin.weight.mul_(1e8 / K ** 0.5)
    m = E.Int8Linear(lin)
    xc = x.to(cuda)
    q, s = E.quant_rows_packed(xc)
    y2 = E.int8_gemm_packed(q, s, m.weight_packed, m.w_scale, None, M, N, K, dtype)
    y = m(xc)
    assert torch.equal(y.isnan(), y2.isnan()) and torch.equal(y.nan_to_num(0.0), y2.nan_to_num(0.0))
    nan_only = [r for r in rows if x[r].isnan().any()]
    assert (y[nan_only].abs() > 1e-3).any(1).all()
