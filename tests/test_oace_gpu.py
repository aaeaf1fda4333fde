"""GPU parity of the OACE loss head (include/afa.h oace_*) against the 40-digit golden fixtures
and the float64 oracle (oracle/oace_oracle.py): fused_oace_softmax_loss (src/model.py:180-240)
and fused_linear_oace (src/kernels/pallas_oace.py:59-293), forward and backward, on the MFMA path
(bf16/fp16) and the generic path (every dtype), in both weight layouts.

Tolerances (normwise max error, the reference's metric): fp64 1e-10 against 40-digit values;
fp32 and the bf16/fp16 loss (inputs exact, fp32 arithmetic) 2e-5; bf16/fp16 gradients 2e-2
(dz and the outputs are rounded to the element type; the reference gates bf16 at 2e-2)."""
import math
import os

import numpy as np
import pytest
import torch

import algebraic_intelligence_amd as A
from algebraic_intelligence_amd import _lib
from oracle import oace_oracle as O
from tests.helpers import normwise, to_f64

pytestmark = pytest.mark.gpu
DEV = "cuda"
GOLD = np.load(os.path.join(os.path.dirname(__file__), "golden", "oace_golden.npz"))
LOW = (torch.bfloat16, torch.float16)


def _t(x, dtype):
    return torch.from_numpy(np.asarray(x, dtype=np.float64)).to(dtype).to(DEV)


def _case(N, d, V, dtype, seed, scale=1.0):
    rng = np.random.default_rng(seed)
    h = _t(rng.standard_normal((N, d)) * scale, dtype)
    w = _t(rng.standard_normal((d, V)) * scale, dtype)
    t = torch.from_numpy(rng.integers(0, V, size=N)).to(DEV)
    return h, w, t


def _fwd(h, w, t, flags=0, eps=100.0, gamma=2.0):
    loss, cache = A.fused_linear_oace_forward(h, w, t, eps, gamma, flags=flags)
    return loss, cache


def _grads(cache, g=1.0):
    dh, dw, _ = A.fused_linear_oace_backward(cache, torch.tensor(g, dtype=torch.float64, device=DEV))
    return dh, dw


def _tied(w):
    """The same (d, V) weight as the transposed view of a contiguous (V, d) embedding."""
    return w.t().contiguous().t()


# ------------------------------------------------------------------------------ golden
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("name", ["lin_small", "lin_d32"])
@pytest.mark.parametrize("tied", [False, True])
def test_linear_matches_golden(name, dtype, tied):
    h, w = _t(GOLD[f"{name}_h"], dtype), _t(GOLD[f"{name}_w"], dtype)
    if tied:
        w = _tied(w)
    t = torch.from_numpy(GOLD[f"{name}_t"]).to(DEV)
    eps, gamma = (float(x) for x in GOLD[f"{name}_cfg"])
    loss, cache = _fwd(h, w, t, eps=eps, gamma=gamma)
    rows = cache[3]
    ref = float(GOLD[f"{name}_loss"])
    tol_f = 1e-10 if dtype == torch.float64 else 2e-5
    tol_g = 1e-10 if dtype == torch.float64 else (2e-5 if dtype == torch.float32 else 2e-2)
    assert abs(float(loss) - ref) <= tol_f * abs(ref)
    assert normwise(to_f64(rows[:, 6]), GOLD[f"{name}_row_loss"]) <= tol_f
    assert normwise(to_f64(rows[:, 0]), GOLD[f"{name}_tau"]) <= tol_f
    dh, dw = _grads(cache)
    e_h = normwise(to_f64(dh), GOLD[f"{name}_dh"])
    e_w = normwise(to_f64(dw), GOLD[f"{name}_dw"])
    print(f"{name} {dtype} tied={tied}: loss {abs(float(loss) - ref) / abs(ref):.2e} dh {e_h:.2e} dw {e_w:.2e}")
    assert e_h <= tol_g and e_w <= tol_g


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32, torch.bfloat16])
def test_softmax_loss_matches_golden(dtype):
    z = _t(GOLD["sm_z"], dtype).requires_grad_(True)
    t = torch.from_numpy(GOLD["sm_t"]).to(DEV)
    eps, gamma = (float(x) for x in GOLD["sm_cfg"])
    loss = A.fused_oace_softmax_loss(z, t, eps, gamma)
    loss.backward()
    ref = float(GOLD["sm_loss"])
    tol = 1e-10 if dtype == torch.float64 else 2e-5
    assert abs(float(loss) - ref) <= tol * abs(ref)
    assert normwise(to_f64(z.grad), GOLD["sm_dz"]) <= (tol if dtype != torch.bfloat16 else 1e-2)


# ------------------------------------------------------------------------------ oracle
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32, torch.bfloat16])
@pytest.mark.parametrize("shape", [(5, 203), (4, 50257), (33, 1000)])
def test_softmax_loss_vs_oracle(shape, dtype):
    N, V = shape
    rng = np.random.default_rng(N + V)
    z = _t(rng.standard_normal((N, V)) * 30.0, dtype).requires_grad_(True)
    t = torch.from_numpy(rng.integers(0, V, size=N)).to(DEV)
    loss = A.fused_oace_softmax_loss(z, t)
    g = 0.7
    (loss * g).backward()
    ref, cache = O.oace_softmax_loss(to_f64(z), t.cpu().numpy())
    rz = O.oace_softmax_loss_vjp(cache, g)
    tol = 1e-12 if dtype == torch.float64 else 2e-5
    assert abs(float(loss) - ref) <= tol * abs(ref)
    assert normwise(to_f64(z.grad), rz) <= (tol if dtype != torch.bfloat16 else 1e-2)


@pytest.mark.parametrize("dtype,epc", [(torch.float32, 4), (torch.bfloat16, 8), (torch.float16, 8)])
@pytest.mark.parametrize("chunks", [0, 1, 64, 128, 256, 512, 1024, 2048, 3328, 6656, 12800])
def test_softmax_loss_row_kernels(dtype, epc, chunks):
    """Rows at each limit of the register-resident row kernels (16-byte chunks per row), whose odd
    lengths start every row at another offset from a 16-byte boundary, from an aligned base and from
    one an element past it (its dz, allocated aligned, then takes the element-wise kernel); and the
    mean over more rows than one workgroup sums.  Tolerances as test_softmax_loss_vs_oracle; fp16
    dz (2^-11 rounding, entries of 1e-4 and up at 2^10 times the loss) 2e-3."""
    for V in sorted({max(1, chunks * epc - epc), max(1, chunks * epc - 1), chunks * epc + 1, chunks * epc + epc}):
        N = 4099 if V <= 9 else 3
        rng = np.random.default_rng(V)
        for off in (0, 1):
            buf = torch.empty(N * V + off, dtype=dtype, device=DEV)
            buf[off:] = _t(rng.standard_normal(N * V) * 10.0, dtype)
            z = buf[off:].view(N, V).requires_grad_(True)
            t = torch.from_numpy(rng.integers(0, V, size=N)).to(DEV)
            loss = A.fused_oace_softmax_loss(z, t)
            g = 1024.0
            (dz,) = torch.autograd.grad(loss * g, z)
            ref, cache = O.oace_softmax_loss(to_f64(z), t.cpu().numpy())
            # at V = 1 the loss is 0, the difference of terms of 2 * 64/7 = 18.3 whose S^(1/8) and
            # reciprocals are within about 8 roundings of 2^-24: 8.7e-6
            assert abs(float(loss) - ref) <= 2e-5 * abs(ref) + (8.7e-6 if V == 1 else 0.0), (V, off)
            tol = {torch.float32: 2e-5, torch.bfloat16: 1e-2, torch.float16: 2e-3}[dtype]
            if V > 1:
                assert normwise(to_f64(dz), O.oace_softmax_loss_vjp(cache, g)) <= tol, (V, off)


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("shape", [(16, 32, 256), (10, 20, 203), (7, 48, 1031)])
@pytest.mark.parametrize("tied", [False, True])
def test_linear_generic_vs_oracle(shape, dtype, tied):
    N, d, V = shape
    h, w, t = _case(N, d, V, dtype, seed=N * d + V, scale=1.5)
    if tied:
        w = _tied(w)
    loss, cache = _fwd(h, w, t)
    dh, dw = _grads(cache, 1.3)
    hf, wf, tn = to_f64(h), to_f64(w), t.cpu().numpy()
    ref, rows = O.fused_linear_oace_forward(hf, wf, tn)
    rh, rw = O.fused_linear_oace_backward(hf, wf, tn, rows, g=1.3)
    tol = 1e-11 if dtype == torch.float64 else 2e-5
    assert abs(float(loss) - ref) <= tol * abs(ref)
    assert normwise(to_f64(cache[3][:, 5]), rows["radial"][:, 0]) <= (tol if dtype == torch.float64 else 1e-4)
    assert normwise(to_f64(dh), rh) <= (tol if dtype == torch.float64 else 1e-4)
    assert normwise(to_f64(dw), rw) <= (tol if dtype == torch.float64 else 1e-4)


@pytest.mark.parametrize("shape", [(1, 1, 1), (31, 33, 63), (128, 64, 256), (129, 65, 257), (255, 127, 513),
                                   (257, 288, 130), (300, 40, 270000)])
@pytest.mark.parametrize("tied", [False, True])
@pytest.mark.parametrize("pad", [0, 3])
def test_linear_fp32_split_planes(shape, tied, pad):
    """fp32 through the three-plane bf16 products at the edges of tiles, steps and splits, with odd
    row strides (pad), and in row chunks (270000 entries: 224 rows at a time), against the fp64
    path.  Tolerance: sums of up to 270000 terms, 16 to a rounding of 2^-24, add up to about
    sqrt(270000 / 16) 2^-24 = 8e-6 of the largest result."""
    N, d, V = shape
    h, w, t = _case(N, d, V, torch.float32, seed=N + V)
    hs = torch.zeros((N, d + pad), device=DEV)
    hs[:, :d] = h
    rows_n, cols = (V, d) if tied else (d, V)
    ws = torch.zeros((rows_n, cols + pad), device=DEV)
    ws[:, :cols] = w.t() if tied else w
    wv = ws[:, :cols].t() if tied else ws[:, :cols]
    loss, cache = _fwd(hs[:, :d], wv, t)
    dh, dw = _grads(cache, 1.3)
    ref, rcache = _fwd(h.double(), w.double(), t)
    rh, rw = _grads(rcache, 1.3)
    # at V = 1 the loss is 0: as test_softmax_loss_row_kernels
    assert abs(float(loss) - float(ref)) <= 2e-5 * abs(float(ref)) + (8.7e-6 if V == 1 else 0.0)
    if V > 1:
        # in place of a new forward: weights changed since, or hidden rows changed since
        assert normwise(to_f64(dh), to_f64(rh)) <= 1e-5 and normwise(to_f64(dw), to_f64(rw)) <= 1e-5
        loss2, cache2 = _fwd(hs[:, :d], wv, t)
        hs.add_(0.0)  # a new version: the backward forms h's planes and the logits again
        dh2, dw2 = _grads(cache2, 1.3)
        assert torch.equal(dh, dh2) and torch.equal(dw, dw2) and torch.equal(loss, loss2)


def test_linear_fp32_keeps_infinities_and_nan():
    """An infinite or NaN hidden row, and values past the largest bf16, as in the fp32 sums: only
    the rows that hold them lose their finite results."""
    h, w, t = _case(5, 40, 300, torch.float32, seed=4)
    h[1, 3], h[2, 0], h[4] = float("inf"), float("nan"), 0.0
    h[4, 0], w[0] = 3.4e38, 1e-38
    loss, cache = _fwd(h, w, t)
    ref, rcache = _fwd(h.double(), w.double(), t)
    rows, rrows = cache[3][:, 6], rcache[3][:, 6]
    assert torch.equal(torch.isfinite(rows), torch.tensor([True, False, False, True, True], device=DEV))
    ok = torch.isfinite(rows)
    assert normwise(to_f64(rows[ok]), to_f64(rrows[ok])) <= 2e-5


@pytest.mark.parametrize("dtype", LOW)
@pytest.mark.parametrize("shape", [(8, 64, 300), (130, 96, 1000), (512, 768, 50257), (3, 32, 7)])
@pytest.mark.parametrize("tied", [False, True])
def test_linear_mfma_vs_oracle_and_generic(shape, dtype, tied):
    """The MFMA path (one GEMM sweep keeping the fp32 logits, the octic sums and dz from them,
    the MFMA GEMMs of oace_bwd_gemm.hip for dh and dW) against the float64 oracle on the same
    exact inputs and against the generic kernels (AFA_FLAG_GENERIC); (512, 768, 50257) is the
    reference benchmark's configuration (scripts/benchmark_kernels.py:118)."""
    N, d, V = shape
    h, w, t = _case(N, d, V, dtype, seed=N + d + V, scale=1.0 if dtype == torch.bfloat16 else 0.5)
    if tied:
        w = _tied(w)
    loss, cache = _fwd(h, w, t)
    dh, dw = _grads(cache, 1.0)
    gl, gcache = _fwd(h, w, t, flags=_lib.FLAG_GENERIC)
    gh, gw = _grads(gcache, 1.0)
    hf, wf, tn = to_f64(h), to_f64(w), t.cpu().numpy()
    ref, rows = O.fused_linear_oace_forward(hf, wf, tn)
    rh, rw = O.fused_linear_oace_backward(hf, wf, tn, rows, g=1.0)
    e_loss = abs(float(loss) - ref) / abs(ref)
    e_rows = normwise(to_f64(cache[3][:, 6]), rows["loss"][:, 0])
    e_h, e_w = normwise(to_f64(dh), rh), normwise(to_f64(dw), rw)
    e_gh, e_gw = normwise(to_f64(dh), to_f64(gh)), normwise(to_f64(dw), to_f64(gw))
    print(f"{shape} {dtype} tied={tied}: loss {e_loss:.2e} rows {e_rows:.2e} dh {e_h:.2e} dw {e_w:.2e} "
          f"vs generic loss {abs(float(loss) - float(gl)) / abs(float(gl)):.2e} dh {e_gh:.2e} dw {e_gw:.2e}")
    assert e_loss <= 2e-5 and e_rows <= 2e-5
    assert abs(float(loss) - float(gl)) <= 2e-5 * abs(float(gl))
    assert e_h <= 2e-2 and e_w <= 2e-2
    assert e_gh <= 2e-2 and e_gw <= 2e-2


@pytest.mark.parametrize("dtype", LOW)
@pytest.mark.parametrize("shape", [(130, 96, 1000), (512, 768, 50257), (3, 32, 7)])
@pytest.mark.parametrize("tied", [False, True])
def test_kept_logits_match_recomputed(shape, dtype, tied):
    """The forward that keeps the fp32 logits (octic sums from them) against the two-sweep forward
    (OACE_FLAG_RECOMPUTE_Z): the same sums in another order.  On one forward's row records, the
    backward's dz from the kept logits (OACE_FLAG_Z_READY) against the dz GEMM sweep: the same
    fp32 logits and arithmetic, so dh and dW are bitwise equal.  The gradients from the two
    forwards' records agree to one rounding of the element type."""
    N, d, V = shape
    h, w, t = _case(N, d, V, dtype, seed=N + 2 * d + V, scale=1.0 if dtype == torch.bfloat16 else 0.5)
    if tied:
        w = _tied(w)
    loss, cache = _fwd(h, w, t)
    rloss, rcache = _fwd(h, w, t, flags=A.oace.FLAG_RECOMPUTE_Z)
    assert abs(float(loss) - float(rloss)) <= 1e-6 * abs(float(rloss))
    assert normwise(to_f64(cache[3][:, :7]), to_f64(rcache[3][:, :7])) <= 1e-6
    dh, dw = _grads(cache, 1.0)
    stale_h = cache[:-1] + (-1,)  # as if h had changed: the backward recomputes z by the GEMM sweep
    gh, gw = _grads(stale_h, 1.0)
    assert torch.equal(dh, gh) and torch.equal(dw, gw)
    rh, rw = _grads(rcache, 1.0)
    # the two records differ in the order of their fp32 sums, so an output that sits at a rounding
    # boundary of the element type can round the other way: at most one unit in the last place of
    # the largest element (the element type's eps), and in few elements
    ulp = torch.finfo(dtype).eps
    for x, y in ((dh, rh), (dw, rw)):
        assert normwise(to_f64(x), to_f64(y)) <= ulp
        assert (x != y).double().mean().item() <= 1e-2


def test_backward_after_inputs_change_in_place():
    """The forward's kept logits are reused only while h and w_vocab are unchanged; after an
    in-place update of h the backward recomputes them with the current h."""
    h, w, t = _case(16, 64, 700, torch.bfloat16, seed=23)
    loss, cache = _fwd(h, w, t)
    h.mul_(0.5)
    dh, dw = _grads(cache, 1.0)
    hf, wf, tn = to_f64(h), to_f64(w), t.cpu().numpy()
    rows = {k: to_f64(cache[3][:, i:i + 1]) for i, k in enumerate(O.ROW_FIELDS)}
    rh, rw = O.fused_linear_oace_backward(hf, wf, tn, rows, g=1.0)
    assert normwise(to_f64(dh), rh) <= 2e-2 and normwise(to_f64(dw), rw) <= 2e-2


def test_linear_autograd_and_chunk_size():
    """fused_linear_oace through torch autograd; chunk_size does not change the result."""
    h, w, t = _case(6, 32, 500, torch.float32, seed=5)
    h.requires_grad_(True)
    w.requires_grad_(True)
    loss = A.fused_linear_oace(h, w, t, chunk_size=64)
    loss.backward()
    ref, rows = O.fused_linear_oace_forward(to_f64(h), to_f64(w), t.cpu().numpy())
    rh, rw = O.fused_linear_oace_backward(to_f64(h), to_f64(w), t.cpu().numpy(), rows)
    assert abs(float(loss) - ref) <= 2e-5 * abs(ref)
    assert normwise(to_f64(h.grad), rh) <= 1e-4 and normwise(to_f64(w.grad), rw) <= 1e-4
    assert float(A.fused_linear_oace(h.detach(), w.detach(), t, chunk_size=7)) == float(loss)
    with pytest.raises(ValueError):
        A.fused_linear_oace(h, w, t, chunk_size=0)


@pytest.mark.parametrize("dtype,flags", [(torch.float32, 0), (torch.bfloat16, 0), (torch.bfloat16, 2)])
def test_target_outside_vocabulary_gives_infinite_loss(dtype, flags):
    """As in the reference, a target that no vocabulary chunk contains leaves rho_t = 0."""
    h, w, t = _case(4, 32, 100, dtype, seed=9)
    t[1] = 100
    loss, cache = _fwd(h, w, t, flags=flags)
    assert torch.isinf(cache[3][1, 6]) and torch.isfinite(cache[3][[0, 2, 3], 6]).all()
    assert torch.isinf(loss)


def test_backward_after_weights_change_in_place():
    """The backward reuses the transposed weights the forward left in its workspace only while
    w_vocab is unchanged; an in-place update in between must not leave a stale copy in use."""
    h, w, t = _case(16, 64, 700, torch.bfloat16, seed=21)
    loss, cache = _fwd(h, w, t)
    w.mul_(0.5)
    dh, dw = _grads(cache, 1.0)
    # the forward's row records belong to the old weights; the backward recomputes the logits with
    # the current ones, exactly as the oracle backward does with those records
    hf, wf, tn = to_f64(h), to_f64(w), t.cpu().numpy()
    rows = {k: to_f64(cache[3][:, i:i + 1]) for i, k in enumerate(O.ROW_FIELDS)}
    rh, rw = O.fused_linear_oace_backward(hf, wf, tn, rows, g=1.0)
    assert normwise(to_f64(dh), rh) <= 2e-2 and normwise(to_f64(dw), rw) <= 2e-2


# ------------------------------------------------------------------------------ dW row strides
@pytest.mark.parametrize("tied,V,pad,off", [(False, 1000, 3, 0), (False, 517, 0, 0), (False, 517, 1, 1),
                                            (False, 50257, 0, 1), (False, 2049, 8, 1), (True, 700, 1, 1),
                                            (True, 700, 0, 0)])
def test_dw_rows_of_any_stride_and_start(tied, V, pad, off):
    """dW stored into rows of any stride (the weight's, odd ones included) starting at any 2-byte
    boundary: equal to the result in a buffer of the Python layer's own, and no element outside
    each row's dW columns changes.  Rows that are not dword aligned take the overlapping-tile stores whose seam dwords
    are written whole; this is where an element of a neighbouring tile, of the next row or of
    the padding would be overwritten if they were wrong."""
    N, d = 70, 64
    h, w, t = _case(N, d, V, torch.bfloat16, seed=V + 7 * pad + off)
    # the weight with the padded row stride; dW gets that stride too (include/afa.h).  The
    # reference is the Python layer's backward on the same weight (the same kernels: an odd
    # stride of a tied embedding is not matrix-core eligible), into a buffer of its own.
    rows_n, cols = (V, d) if tied else (d, V)
    wide = torch.zeros((rows_n, cols + pad), dtype=torch.bfloat16, device=DEV)
    wide[:, :cols] = w.t() if tied else w
    wv = wide[:, :cols].t() if tied else wide[:, :cols]
    _, cache = _fwd(h, wv, t)
    dh_ref, dw_ref = _grads(cache)
    hf, wop, tt, rows, gamma, _c, _s, flags, ws, _wv, _hv = cache
    ldw = cols + pad
    sentinel = 0x7F7B  # a bf16 NaN pattern no gradient takes
    store = torch.full((rows_n * ldw + off + 64,), sentinel, dtype=torch.int16, device=DEV)
    g = torch.ones((), dtype=rows.dtype, device=DEV)
    dh = torch.empty((N, d), dtype=torch.bfloat16, device=DEV)
    lay = A.oace.OACE_W_VD if tied else A.oace.OACE_W_DV
    rc = _lib.lib().oace_linear_bwd(_lib.dtype_code(torch.bfloat16), N, d, V, hf.data_ptr(), hf.stride(0),
                                    wop.data_ptr(), lay, ldw, tt.data_ptr(), float(gamma), rows.data_ptr(),
                                    g.data_ptr(), dh.data_ptr(), store.data_ptr() + 2 * off, flags, ws.data_ptr(),
                                    ws.numel(), _lib.stream_ptr(torch.device(DEV)))
    _lib.check(rc, "oace_linear_bwd")
    torch.cuda.synchronize()
    mat = store[off:off + rows_n * ldw].view(rows_n, ldw)
    got = mat[:, :cols].view(torch.bfloat16)
    ref = dw_ref.t() if tied else dw_ref
    assert normwise(to_f64(got), to_f64(ref)) <= 1e-6
    assert normwise(to_f64(dh), to_f64(dh_ref)) <= 1e-6
    assert bool((mat[:, cols:] == sentinel).all()), "padding columns changed"
    assert bool((store[:off] == sentinel).all()) and bool((store[off + rows_n * ldw:] == sentinel).all())


@pytest.mark.parametrize("dtype", LOW)
@pytest.mark.parametrize("shape", [(2049, 32, 9), (1500, 96, 1003), (1024, 64, 257), (4100, 288, 520)])
@pytest.mark.parametrize("tied", [False, True])
def test_dw_split_over_the_rows(shape, dtype, tied):
    """dW from parts of its contraction over the rows (few tiles, many rows), with ragged last parts
    and tiles in both dimensions, against the fp64 path: the element type's rounding of dz and of
    dW, 2e-2 normwise as the other gradients; and repeated calls bitwise equal."""
    N, d, V = shape
    h, w, t = _case(N, d, V, dtype, seed=N + V, scale=1.0 if dtype == torch.bfloat16 else 0.5)
    wv = _tied(w) if tied else w
    g = 1.0 if dtype == torch.bfloat16 else 4096.0  # fp16: dz of a mean over this many rows is small
    _, cache = _fwd(h, wv, t)
    dh, dw = _grads(cache, g)
    dh2, dw2 = _grads(cache, g)
    assert torch.equal(dh, dh2) and torch.equal(dw, dw2)
    _, rcache = _fwd(h.double(), wv.double(), t)
    rh, rw = _grads(rcache, g)
    assert normwise(to_f64(dh), to_f64(rh)) <= 2e-2 and normwise(to_f64(dw), to_f64(rw)) <= 2e-2


@pytest.mark.parametrize("V", [4095, 4096, 4097])
@pytest.mark.parametrize("N", [3, 130])
def test_forward_rows_at_the_kernel_change(N, V):
    """Kept logits on both sides of the row length at which the forward changes its row kernel
    (4096), against the fp64 path: fp32 sums of exact inputs, 2e-5 as test_linear_matches_golden."""
    h, w, t = _case(N, 64, V, torch.bfloat16, seed=N + V, scale=0.5)
    loss, cache = _fwd(h, w, t)
    ref, rcache = _fwd(h.double(), w.double(), t)
    assert abs(float(loss) - float(ref)) <= 2e-5 * abs(float(ref))
    for f in range(7):
        assert normwise(to_f64(cache[3][:, f]), to_f64(rcache[3][:, f])) <= (1e-4 if f == 5 else 2e-5), f


@pytest.mark.parametrize("dtype", LOW)
@pytest.mark.parametrize("shape", [(3, 32, 8), (130, 64, 248), (33, 96, 264), (520, 32, 1088), (257, 160, 2056)])
def test_head_read_in_place_equals_its_aligned_copy(shape, dtype):
    """A (d, V) head whose rows are whole 16-byte chunks is read where it lies; the same weights at an
    odd offset or row stride go through the aligned copy.  Same products in the same order: equal."""
    N, d, V = shape
    h, w, t = _case(N, d, V, dtype, seed=N + V, scale=0.5)
    loss, cache = _fwd(h, w, t)
    dh, dw = _grads(cache, 1.0)
    for off, ld in [(0, V + 8), (8, V + 16), (1, V + 8), (3, V + 7), (0, V + 1)]:
        store = torch.full((d * ld + off + 16,), float("nan"), dtype=dtype, device=w.device)
        view = store[off:off + d * ld].view(d, ld)[:, :V]
        view.copy_(w)
        loss2, cache2 = _fwd(h, view, t)
        dh2, dw2 = _grads(cache2, 1.0)
        assert float(loss2) == float(loss), (off, ld)
        assert torch.equal(cache2[3], cache[3]) and torch.equal(dh2, dh) and torch.equal(dw2, dw), (off, ld)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("V", [1, 2, 3, 5, 9, 15, 17, 65, 129, 1031])
def test_softmax_loss_small_row_sums(dtype, V):
    """Row records of negative logits, whose octic sum (V terms near 9e-4) is far below the 1 that an
    entry outside the row would add to it, from every start of a row against the fp64 kernel.  Bounds as
    test_algebraic_softmax_small_row_sums: 3.3e-6 for a weight and for the sums; the target's is one of
    them, so p_target^(-1/8), S^(1/8) and sum p^(7/8) are within 3.3e-6 (1 + 7/8) of theirs, and the loss
    within that of its terms."""
    N = 16
    rng = np.random.default_rng(V)
    z = _t(-60.0 - rng.random((N, V)), dtype)
    t = torch.from_numpy(rng.integers(0, V, size=N)).to(DEV)
    stream = _lib.stream_ptr(z.device)

    def records(x):
        acc = _lib.accum_dtype(x.dtype)
        loss, rec = torch.empty((), dtype=acc, device=DEV), torch.empty((N, A.oace.ROW_FIELDS), dtype=acc, device=DEV)
        _lib.check(_lib.lib().oace_softmax_loss_fwd(_lib.dtype_code(x.dtype), N, V, x.data_ptr(), t.data_ptr(), 100.0, 2.0,
                                                    loss.data_ptr(), rec.data_ptr(), stream), "oace_softmax_loss_fwd")
        return rec.double()

    ref = records(z.double())
    for start in range(0, 16 // z.element_size(), 3):
        got = records(torch.empty(N * V + start, dtype=dtype, device=DEV)[start:].view(N, V).copy_(z))
        for f in range(5):  # tau, 1/S, S^(1/8), sum p^(7/8), p_target^(-1/8)
            assert ((got[:, f] - ref[:, f]).abs() <= 6.2e-6 * ref[:, f].abs()).all(), (start, f)
        terms = 2.0 * (8.0 * ref[:, 4] + 8.0 / 7.0 * ref[:, 3])
        assert ((got[:, 6] - ref[:, 6]).abs() <= 6.2e-6 * terms).all(), start


@pytest.mark.parametrize("N,V,dtype", [(700, 12289, torch.bfloat16), (700, 12289, torch.float16),
                                       (1400, 3075, torch.float32)])
def test_softmax_loss_many_chunks_per_lane(N, V, dtype):
    """dz of enough rows that a lane takes four chunks of a row: several spans per row, ragged rows of
    every start, and targets in each of the four chunk positions, on both sides of a span's edge and at
    both ends of the row; against the fp64 kernel, tolerances as test_softmax_loss_row_kernels."""
    rng = np.random.default_rng(V)
    z = _t(rng.standard_normal((N, V)) * 10.0, dtype).requires_grad_(True)
    t = rng.integers(0, V, size=N)
    epc = 16 // z.element_size()
    edges = [c * 64 * epc + o for c in range(V // (64 * epc) + 1) for o in (-epc, -1, 0, 1, epc)] + [0, 1, V - 2, V - 1]
    edges = [e for e in edges if 0 <= e < V]
    t[:len(edges)] = edges
    t = torch.from_numpy(t).to(DEV)
    g = 1024.0
    (dz,) = torch.autograd.grad(A.fused_oace_softmax_loss(z, t) * g, z)
    zd = z.detach().double().requires_grad_(True)
    (ref,) = torch.autograd.grad(A.fused_oace_softmax_loss(zd, t) * g, zd)
    tol = {torch.float32: 2e-5, torch.bfloat16: 1e-2, torch.float16: 2e-3}[dtype]
    err = (dz.double() - ref).abs()
    assert (err.amax(-1) <= tol * ref.abs().amax(-1)).all()  # every row by itself


@pytest.mark.parametrize("shape", [(130, 96, 1000), (1100, 288, 50257), (70, 32, 800000), (300, 40, 270000)])
@pytest.mark.parametrize("tied", [False, True])
def test_fp32_kept_logits_match_recomputed(shape, tied):
    """The fp32 head with and without kept logits (OACE_FLAG_RECOMPUTE_Z: other row chunks, down to 32 rows
    at 800000 entries): the same fp32 logits, so the same row records, and dh and dW but for the order
    of their sums (1e-5 as test_linear_fp32_split_planes); bitwise equal where no logits were kept but the
    chunks are the same."""
    N, d, V = shape
    h, w, t = _case(N, d, V, torch.float32, seed=N + V)
    wv = _tied(w) if tied else w
    loss, cache = _fwd(h, wv, t)
    rloss, rcache = _fwd(h, wv, t, flags=A.oace.FLAG_RECOMPUTE_Z)
    assert float(loss) == float(rloss) and torch.equal(cache[3], rcache[3])
    dh, dw = _grads(cache, 1.3)
    rh, rw = _grads(rcache, 1.3)
    assert normwise(to_f64(rh), to_f64(dh)) <= 1e-5 and normwise(to_f64(rw), to_f64(dw)) <= 1e-5
    if N * V * 10 <= 1 << 28:
        assert torch.equal(rh, dh) and torch.equal(rw, dw)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("N,V", [(3, 1031), (4099, 9), (700, 6145)])
def test_softmax_loss_infinite_cotangent(dtype, N, V):
    """An infinite loss cotangent gives infinite dlogits, of the sign and with the NaN (an entry whose
    bracket is 0) that a finite one predicts."""
    rng = np.random.default_rng(V)
    z = _t(rng.standard_normal((N, V)) * 10.0, dtype).requires_grad_(True)
    t = torch.from_numpy(rng.integers(0, V, size=N)).to(DEV)
    zd = z.detach().double().requires_grad_(True)
    (ref,) = torch.autograd.grad(A.fused_oace_softmax_loss(zd, t), zd)
    (dz,) = torch.autograd.grad(A.fused_oace_softmax_loss(z, t) * math.inf, z)
    # entries not within rounding of 0 (2e-5 of a row's largest, as test_softmax_loss_vs_oracle)
    clear = ref.abs() > 2e-5 * ref.abs().amax(-1, keepdim=True)
    assert torch.equal(dz[clear].double(), ref[clear].sign() * math.inf) and not torch.isfinite(dz).any()


@pytest.mark.parametrize("d", [1792, 2048, 2080, 2304])
@pytest.mark.parametrize("V", [1100, 1531])
def test_tied_dw_tile_orders(d, V):
    """dW of a (V, d) embedding on both sides of the 8 m tiles (256 features each) at which their order over the
    workgroups changes, with more n tiles (128 entries) than m tiles and ragged ones: every tile once.
    Against the fp32 path on the same operands: the element type's rounding of dz and of dW, 2e-2."""
    h, w, t = _case(160, d, V, torch.bfloat16, seed=d + V, scale=0.2)
    _, cache = _fwd(h, _tied(w), t)
    dh, dw = _grads(cache)
    _, rcache = _fwd(h.float(), _tied(w).float(), t)
    rh, rw = _grads(rcache)
    assert normwise(to_f64(dh), to_f64(rh)) <= 2e-2 and normwise(to_f64(dw), to_f64(rw)) <= 2e-2
    blocks = (dw.double() - rw.double()).abs()[: d // 32 * 32].reshape(d // 32, 32, V).amax(1)
    assert (blocks <= 2e-2 * rw.double().abs().max()).all()


@pytest.mark.parametrize("shape", [(1, 40, 300), (1, 130, 1031), (1, 33, 50257)])
@pytest.mark.parametrize("tied", [False, True])
def test_linear_fp32_infinite_cotangent(shape, tied):
    """dh and dW of the fp32 head where the loss cotangent is infinite: infinite, of the sign that a finite
    one predicts, and NaN where infinite terms of both signs or a zero factor meet, as the generic fp32
    kernels have them.  Feature 0 is 0 in h, so its weights are free to take the signs of dz."""
    N, d, V = shape
    h, w, t = _case(N, d, V, torch.float32, seed=V)
    h[:, 0] = 0.0
    wv = _tied(w) if tied else w
    dz = (_grads(_fwd(h, wv, t)[1])[1][1] / h[0, 1]).double()
    # an entry within rounding of 0 (2e-5 of the largest, as test_softmax_loss_vs_oracle) has no sign to predict
    clear = dz.abs() > 2e-5 * dz.abs().max()
    wv[0] = (dz.sign() * (0.5 + torch.rand(V, device=DEV, dtype=torch.float64))).float()
    dh, dw = _grads(_fwd(h, wv, t)[1], math.inf)
    gh, gw = _grads(_fwd(h, wv, t, flags=_lib.FLAG_GENERIC)[1], math.inf)
    assert torch.isinf(dw[1:, clear]).all() and torch.isnan(dw[0]).all()
    for got, want in ((dw[:, clear], gw[:, clear]), (dh[:, 1:], gh[:, 1:])):
        assert torch.equal(got.nan_to_num(9e9), want.nan_to_num(9e9))
    if clear.all():
        assert float(dh[0, 0]) == float(gh[0, 0]) == math.inf
