"""The matrix-core tile kernels (16-byte aligned operands and outputs, output rows of whole
16-byte units, full K chunks) against the kernels the same C entry points take otherwise (here:
operands offset by one element for the inner product, an output offset by one element for the
fp4 metrics and the bit-packed rows): identical inputs, bit-identical outputs, edge tiles and
long K.
The inner-product paths form each dot product from the same MFMA sequence (the tile kernel
with the operands swapped); the boolean counts are exact integers on every path; all of them
finish with the same epilogue functions."""
import ctypes as C

import pytest
import torch

from tests._util import rand, randn
from torchpairwise_amd import _capi as capi

pytestmark = pytest.mark.gpu
DEV = "cuda"



class Launches:
    """The launches of one kernel family inside a ``with`` block: which path a call took."""

    def __init__(self, family):
        self.timer = capi.LaunchTimer(family, 16)

    def __enter__(self):
        self.timer.arm()
        return self

    def __exit__(self, *exc):
        self.count = len(self.timer.read()[0])


EPIS = [capi.EPI_DOT, capi.EPI_EUCLIDEAN, capi.EPI_SQEUCLIDEAN, capi.EPI_COSINE_SIM,
        capi.EPI_COSINE_DIST, capi.EPI_CORRELATION]


def _inner(x1, x2, epi, misaligned):
    """tpw_pairwise_inner on 16-byte aligned inputs (the tile kernel), or on copies of them
    offset by one element (not 16-byte aligned: the register-staged kernel with element loads);
    the output is aligned either way."""
    B, n, d = x1.shape
    m = x2.shape[1]
    if misaligned:
        s1 = torch.empty(B * n * d + 16, dtype=x1.dtype, device=DEV)
        s2 = torch.empty(B * m * d + 16, dtype=x2.dtype, device=DEV)
        a, b = s1[1:1 + B * n * d].view(B, n, d), s2[1:1 + B * m * d].view(B, m, d)
        a.copy_(x1)
        b.copy_(x2)
    else:
        a, b = x1, x2
    squared = epi in (capi.EPI_EUCLIDEAN, capi.EPI_SQEUCLIDEAN)
    n1 = capi.row_norms(x1, squared) if epi != capi.EPI_DOT else None
    n2 = capi.row_norms(x2, squared) if epi != capi.EPI_DOT else None
    out = torch.empty((B, n, m), dtype=x1.dtype, device=DEV)
    capi.call("tpw_pairwise_inner", C.c_void_p(a.data_ptr()), C.c_void_p(b.data_ptr()), capi._dtype_code(x1),
              B, n, m, d, capi._ptr(n1), capi._ptr(n2), epi, C.c_void_p(out.data_ptr()), capi._stream())
    return out


def _same_bits(a, b):
    ia = a.view(torch.int32) if a.dtype == torch.float32 else a.view(torch.int16)
    ib = b.view(torch.int32) if b.dtype == torch.float32 else b.view(torch.int16)
    return torch.equal(ia, ib)


# batches of more than 256 tiles of 128 x 128, which the small-output kernel does not take
@pytest.mark.parametrize("dtype,B,n,m,d", [
    (torch.float32, 29, 300, 260, 32),
    (torch.float32, 65, 129, 136, 96),
    (torch.float32, 129, 128, 256, 256),
    (torch.float32, 43, 130, 260, 512),     # 16 chunks: the double-buffered long-K variant
    (torch.float32, 29, 300, 259, 64),      # ragged rows: 16-byte units at any dword
    (torch.float32, 65, 129, 142, 512),
    (torch.bfloat16, 29, 300, 264, 64),
    (torch.bfloat16, 18, 257, 520, 192),
    (torch.bfloat16, 257, 128, 128, 256),
    (torch.bfloat16, 65, 200, 136, 1024),   # long K
    # bf16 ragged rows (m % 8 = 1 .. 7): 16-byte units at any value
    (torch.bfloat16, 29, 300, 259, 64),
    (torch.bfloat16, 65, 129, 133, 192),
    (torch.bfloat16, 43, 130, 262, 1024),
    (torch.bfloat16, 257, 70, 7, 128),
    (torch.bfloat16, 43, 257, 140, 256),
])
@pytest.mark.parametrize("epi", EPIS)
def test_inner_tile_kernel_equals_staged_kernel(dtype, B, n, m, d, epi):
    x1 = randn(B, n, d, seed=1).to(DEV, dtype)
    x2 = randn(B, m, d, seed=2).to(DEV, dtype)
    x2[:, 3] = 0  # a zero row: the guarded cosine divide
    if m > 7:
        x2[:, 7] = x1[:, 0]  # an identical pair: the clamped euclidean floor
    with Launches("inner_tile_kernel") as on_tile:
        tile = _inner(x1, x2, epi, False)
    with Launches("pairwise_inner_kernel") as on_staged:
        staged = _inner(x1, x2, epi, True)
    with Launches("inner_small_kernel") as on_small:
        _inner(x1, x2, epi, False), _inner(x1, x2, epi, True)
    assert (on_tile.count, on_staged.count, on_small.count) == (1, 1, 0)
    if dtype == torch.bfloat16 and epi >= capi.EPI_COSINE_SIM:
        # tiles without a zero row divide by reciprocal norms (2 ulp of float, 2^-22 near 1, before the
        # bf16 rounding): one bf16 ulp, 2^-7 relative, or 2^-21 where 1 - q cancels
        assert torch.allclose(tile.float(), staged.float(), rtol=2.0 ** -7, atol=2.0 ** -21)
    else:
        assert _same_bits(tile, staged)


# Small outputs (64 x 64 tiles, norms formed in the kernel or given) against the 128 x 128 kernels,
# which the same rows take inside a batch of 260: the same products and norms in the same order, so
# the same bits.  Tile edges, ragged m, rows of whole and partial 16-byte pieces, chunks (32 fp32,
# 64 bf16) and 256-byte stages, vector norms of 1 .. 64 lanes, unaligned operands.  bf16 cosine
# rounds its quotient by reciprocal norms where the whole tile allows it (2 ulp of float before the
# bf16 rounding), and a tile with a zero row divides: one bf16 ulp between the two.
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n,m,d", [(64, 64, 64), (65, 63, 50), (1, 129, 1), (33, 100, 128), (130, 7, 257),
                                   # the tile kernel with ragged rows (16-byte units at any alignment)
                                   (65, 63, 64), (130, 131, 128), (40, 1, 64), (129, 142, 1024),
                                   (40, 66, 100), (31, 32, 516)])
@pytest.mark.parametrize("epi", EPIS)
def test_small_output_kernel_equals_tile_kernels(dtype, n, m, d, epi):
    B = 260
    x1, x2 = randn(B, n, d, seed=21).to(DEV, dtype), randn(B, m, d, seed=22).to(DEV, dtype)
    x2[:, min(3, m - 1)] = 0
    def small(a, c, b):
        return capi.lib().tpw_pairwise_inner_forms_norms(capi._ptr(a), capi._ptr(c), capi._dtype_code(a), b, n, m, d)

    assert not small(x1, x2, B)
    want = _inner(x1, x2, epi, False)
    for b in (0, B - 1):
        given = _inner(x1[b:b + 1].contiguous(), x2[b:b + 1].contiguous(), epi, b > 0)
        own = torch.empty((1, n, m), dtype=dtype, device=DEV)
        a, c = x1[b].clone(), x2[b].clone()
        assert small(a, c, 1)
        capi.call("tpw_pairwise_inner_own_norms", capi._ptr(a), capi._ptr(c), capi._dtype_code(a), 1, n, m, d, epi,
                  capi._ptr(own), capi._stream())
        assert _same_bits(own, given)
        if dtype == torch.bfloat16 and epi >= capi.EPI_COSINE_SIM:
            assert torch.allclose(own[0].float(), want[b].float(), rtol=2.0 ** -7, atol=2.0 ** -8)
        else:
            assert _same_bits(own[0], want[b])


def _fp4_metric(x1, x2, metric, misaligned):
    (fa, ca), (fb, cb) = capi.pack_bool_fp4(x1), capi.pack_bool_fp4(x2)
    B, n, d = x1.shape
    m = x2.shape[1]
    store = torch.empty(B * n * m + 16, dtype=torch.float32, device=DEV)
    out = store[1:1 + B * n * m] if misaligned else store[:B * n * m]
    capi.call("tpw_bool_fp4_count_metric", capi._ptr(fa), capi._ptr(fb), capi._ptr(ca), capi._ptr(cb), B, n, m, d,
              metric, C.c_void_p(out.data_ptr()), capi._stream())
    return out.view(B, n, m)


@pytest.mark.parametrize("B,n,m,d", [(1, 300, 260, 100), (2, 129, 136, 1000), (1, 128, 256, 256), (1, 70, 132, 3000),
                                     (1, 130, 131, 1000), (2, 70, 134, 300)])
@pytest.mark.parametrize("metric", range(10))
def test_fp4_tile_kernel_equals_staged_kernel(B, n, m, d, metric):
    x1 = (rand(B, n, d, seed=3) < 0.3).to(DEV)
    x2 = (rand(B, m, d, seed=4) < 0.3).to(DEV)
    x2[:, 0] = False  # an all-zero row: the guarded 0 / 0 cases
    tile = _fp4_metric(x1, x2, metric, False)
    staged = _fp4_metric(x1, x2, metric, True)
    assert torch.equal(torch.nan_to_num(tile, nan=-7.0).view(torch.int32),
                       torch.nan_to_num(staged, nan=-7.0).view(torch.int32))


# --------------------------------------------------------------------------------------
# Bit-packed rows on the fp4 matrix cores (bool_bits_tile_kernel: the count metrics at any d,
# the reductions over more than 256 features) against the popcount kernel the same entry points
# take for an output offset by one element: every count metric, jaccard, and every op x
# reduction of the counted entry; partial last chunks (d = 1 .. 256: one chunk of one or two
# pieces; 257: 3 of 8 pieces; 1500: 2 chunks, the second half full; 2081: 3 chunks, the last
# one piece), edge tiles, ragged output rows (m % 4 != 0).  Bit-identical.
# --------------------------------------------------------------------------------------
def _bits_call(x1, x2, kind, code, misaligned):
    wa, pa = capi.pack_bool(x1)
    wb, pb = capi.pack_bool(x2)
    B, n, d = x1.shape
    m = x2.shape[1]
    store = torch.empty(B * n * m + 16, dtype=torch.float32, device=DEV)
    out = store[1:1 + B * n * m] if misaligned else store[:B * n * m]
    o = C.c_void_p(out.data_ptr())
    if kind == "metric":
        capi.call("tpw_bool_count_metric", capi._ptr(wa), capi._ptr(wb), capi._ptr(pa), capi._ptr(pb), B, n, m, d,
                  code, o, capi._stream())
    elif kind == "jaccard":
        capi.call("tpw_jaccard_bool", capi._ptr(wa), capi._ptr(wb), capi._ptr(pa), capi._ptr(pb), B, n, m, d, o,
                  capi._stream())
    else:
        op, red = code
        capi.call("tpw_bool_pairwise_reduce_counted", capi._ptr(wa), capi._ptr(wb), capi._ptr(pa), capi._ptr(pb),
                  B, n, m, d, op, red, o, capi._stream())
    return out.view(B, n, m)


BITS_CASES = ([("metric", k) for k in range(10)] + [("jaccard", 0)] +
              [("reduce", (op, red)) for op in range(5) for red in range(2)])


@pytest.mark.parametrize("B,n,m,d", [(1, 130, 132, 1), (1, 70, 136, 33), (2, 129, 136, 128), (1, 130, 132, 256),
                                     (1, 300, 260, 257), (2, 129, 136, 1024), (1, 130, 132, 1500),
                                     (1, 70, 132, 2081),
                                     # ragged rows (m % 4 != 0): dword rows (counts) or unaligned units
                                     (1, 130, 131, 1024), (2, 70, 133, 300), (1, 129, 130, 100),
                                     (1, 257, 259, 33), (1, 40, 1, 512)])
@pytest.mark.parametrize("kind,code", BITS_CASES)
def test_bits_tile_kernel_equals_popcount_kernel(B, n, m, d, kind, code):
    x1 = (rand(B, n, d, seed=5) < 0.3).to(DEV)
    x2 = (rand(B, m, d, seed=6) < 0.3).to(DEV)
    x2[:, 0] = False  # an all-zero row: the guarded 0 / 0 cases
    x1[:, 1] = True   # an all-one row
    tile = _bits_call(x1, x2, kind, code, False)
    ref = _bits_call(x1, x2, kind, code, True)
    assert torch.equal(torch.nan_to_num(tile, nan=-7.0).view(torch.int32),
                       torch.nan_to_num(ref, nan=-7.0).view(torch.int32))


# Ragged output rows of at most 256 features: few rows leave by dwords (the aligned stores' blocks would
# be nearly empty), more by aligned whole lines; the bits of the same columns among m + 1 (m % 4 == 0).
@pytest.mark.parametrize("B,n,m,d,lines", [(1, 1, 70003, 166, False), (1, 43, 70003, 166, False), (1, 44, 70003, 166, True),
                                           (1, 25, 70003, 60, False), (1, 26, 70003, 60, True), (9, 5, 3003, 166, False),
                                           (1, 5, 3003, 166, True), (1, 300, 20003, 250, True), (3, 257, 3003, 33, True)])
def test_popcount_ragged_rows(B, n, m, d, lines):
    x1, x2 = (rand(B, n, d, seed=7) < 0.3).to(DEV), (rand(B, m + 1, d, seed=8) < 0.3).to(DEV)
    x2m = x2[:, :m].contiguous()
    want = torch.ops.torchpairwise.hamming_distances(x1, x2)[..., :m]
    for family, count in (("bool_reduce_kernel", 1), ("bool_reduce_ragged_kernel", int(lines))):
        with Launches(family) as launches:
            got = torch.ops.torchpairwise.hamming_distances(x1, x2m)
        assert launches.count == count
        assert torch.equal(got, want)


# --------------------------------------------------------------------------------------
# fp32 backward of small problems with aligned inputs and with inputs offset by one element: the
# weight pass and the split-K GEMM (polynomial), op_backward_kernel with whole and element loads
# (the others; the kernels of larger problems are in test_backward_paths_of_large_problems).
# Bar: float64 autograd of the reference's composite on the CPU, rtol 1e-4 (+ 1e-4 * max);
# the two calls agree to 1e-5 * max (different summation orders).
# --------------------------------------------------------------------------------------
BWD_OPS = [("euclidean_distances", {}), ("sqeuclidean_distances", {}), ("cosine_distances", {}),
           ("cosine_similarity", {}), ("correlation_distances", {}),
           ("polynomial_kernel", dict(degree=3, gamma=0.05)), ("sigmoid_kernel", dict(gamma=0.02)),
           ("linear_kernel", {})]


def _leaf(x, misaligned):
    if not misaligned:
        return x.to(DEV).requires_grad_()
    buf = torch.empty(x.numel() + 16, dtype=x.dtype, device=DEV)
    v = buf[1:1 + x.numel()].view(x.shape)
    v.copy_(x)
    return v.requires_grad_()


@pytest.mark.parametrize("B,n,m,d", [(1, 96, 160, 36), (2, 256, 128, 64), (1, 544, 512, 132), (1, 128, 96, 300)])
@pytest.mark.parametrize("name,kw", BWD_OPS)
def test_backward_products_tile_fp32(name, kw, B, n, m, d):
    import torchpairwise_amd as tp
    from tests._util import assert_close

    print(f"{name} {kw} B={B} n={n} m={m} d={d}", flush=True)
    fn = getattr(tp, name)
    x1, x2, g = randn(B, n, d, seed=0), randn(B, m, d, seed=1), randn(B, n, m, seed=2)
    grads = {}
    for misaligned in (False, True):
        a, b = _leaf(x1, misaligned), _leaf(x2, misaligned)
        assert (a.data_ptr() % 16 != 0) == misaligned
        fn(a, b, **kw).backward(g.to(DEV))
        grads[misaligned] = (a.grad.cpu(), b.grad.cpu())
    ra, rb = x1.double().requires_grad_(), x2.double().requires_grad_()
    fn(ra, rb, **kw).backward(g.double())
    for k, want in enumerate((ra.grad, rb.grad)):
        tile, split = grads[False][k], grads[True][k]
        scale = float(want.abs().max())
        assert_close(tile, want, rtol=1e-4, atol=1e-4 * scale, what=f"{name} grad_x{k + 1} (aligned)")
        assert_close(split, want, rtol=1e-4, atol=1e-4 * scale, what=f"{name} grad_x{k + 1} (offset)")
        assert_close(tile, split.double(), rtol=0, atol=1e-5 * scale, what=f"{name} grad_x{k + 1} aligned vs offset")


# Both gradients in one launch (op_backward_kernel): edges of its 64-row tiles, 64- and 128-feature
# tiles, 32-row K chunks and splits (also of one direction alone), sums long enough to be blocked (512), vector and element
# loads; a zero row (norm 0) and rows out of the fast cosine terms' norm range.  fp32 against the
# derived per-element bounds (euclidean, cosine) or, like the kernel functions above, rtol 1e-4;
# bf16 at the bf16 tolerance of the other paths.
@pytest.mark.parametrize("B,n,m,d", [(1, 1, 1, 1), (1, 63, 65, 64), (2, 65, 33, 65), (1, 31, 1100, 30),
                                     (1, 1601, 64, 128), (3, 130, 97, 131), (4, 9000, 40, 130)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("name,kw", [o for o in BWD_OPS if o[0] != "polynomial_kernel"])
def test_backward_one_launch(name, kw, dtype, B, n, m, d):
    import torchpairwise_amd as tp
    from tests import _gradbound as GB
    from tests._util import assert_close

    print(f"one launch {name} {dtype} B={B} n={n} m={m} d={d}", flush=True)
    fn = getattr(tp, name)
    x1, x2, g = (randn(B, r, c, seed=k, dtype=dtype) for k, (r, c) in enumerate(((n, d), (m, d), (n, m))))
    if n > 40 and name.startswith("cosine"):
        x1[:, 7] = 0
        x1[:, 33] *= 2.0 ** 58  # norm about 2^61
    a, b = x1.to(DEV).requires_grad_(), x2.to(DEV).requires_grad_()
    fn(a, b, **kw).backward(g.to(DEV))
    ra, rb = x1.double().requires_grad_(), x2.double().requires_grad_()
    fn(ra, rb, **kw).backward(g.double())
    plain = slice(34, None) if n > 40 and name.startswith("cosine") else slice(None)
    for k, (got, want) in enumerate(((a.grad, ra.grad), (b.grad, rb.grad))):
        if dtype == torch.float32 and name in ("euclidean_distances", "cosine_similarity") and d > 1:
            for bb in range(B):
                own, other, gs = (x1, x2, g[bb]) if k == 0 else (x2, x1, g[bb].T)
                if name == "euclidean_distances":
                    bound = GB.euclidean_grad_bound(own[bb], other[bb], gs)
                elif k == 0:  # rows of ordinary norms
                    GB.check(got[bb].cpu()[plain], want[bb][plain],
                             GB.cosine_grad_bound(own[bb], other[bb], gs, True)[plain], f"{name} grad_x1")
                    continue
                else:
                    ok = torch.ones(n, dtype=torch.bool)
                    if n > 40:
                        ok[7] = False  # the zero row's pairs: no quotient
                    bound = GB.cosine_grad_bound(own[bb], other[bb][ok], gs[:, ok], True)
                GB.check(got[bb].cpu(), want[bb], bound, f"{name} grad_x{k + 1}")
        tol = 1e-4 if dtype == torch.float32 else 1e-2
        # one feature: the cosine's two terms, each at most |g| / |own| a pair, cancel to zero, and
        # what is left is their rounding (4 u a term, u = 2^-24 or 2^-9)
        own = (x1, x2)[k].double()
        left = 0.0
        if d == 1:
            u = 2.0 ** -24 if dtype == torch.float32 else 2.0 ** -9
            left = 4 * u * float(g.double().abs().sum()) / max(float(own.abs().min()), 1e-3)
        # (the row scaled by 2^58 has gradients 2^-58 of the others': the floor covers them)
        assert_close(got.float(), want, rtol=tol, atol=tol * float(want.abs().max()) + left,
                     what=f"{name} grad_x{k + 1}")


# past op_backward_kernel's limit (3 2^23 pairs): the weight pass and the products, fp32 split-K
# and tile kernel and bf16 with W^T and transposed copies, ragged and aligned, against float64 on
# the GPU's plain torch operations
@pytest.mark.parametrize("n,m,d", [(5201, 5003, 70), (5120, 5120, 64)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("name", ["euclidean_distances", "cosine_similarity", "linear_kernel"])
def test_backward_passes_above_one_launch(name, dtype, n, m, d):
    import torchpairwise_amd as tp
    from tests._util import assert_close

    x1, x2, g = randn(n, d, seed=0, dtype=dtype), randn(m, d, seed=1, dtype=dtype), randn(n, m, seed=2, dtype=dtype)
    a, b, gd = x1.to(DEV).requires_grad_(), x2.to(DEV).requires_grad_(), g.to(DEV)
    getattr(tp, name)(a, b).backward(gd)
    ra, rb = (x.to(DEV).double().requires_grad_() for x in (x1, x2))
    s = ra @ rb.T
    if name == "euclidean_distances":
        s = (ra.square().sum(1)[:, None] + rb.square().sum(1)[None] - 2 * s).clamp_min(0).sqrt()
    elif name == "cosine_similarity":
        s = s / (ra.norm(dim=1)[:, None] * rb.norm(dim=1)[None])
    s.backward(gd.double())
    tol = 1e-4 if dtype == torch.float32 else 1e-2
    for got, want in ((a.grad, ra.grad), (b.grad, rb.grad)):
        assert_close(got.float(), want, rtol=tol, atol=tol * float(want.abs().max()), what=name)


# The backward's kernels for problems past op_backward_kernel's limit, each with aligned inputs and
# with inputs offset by one element, which take the weight pass and the split-K GEMM (fp32) or W^T,
# transposed copies and the register-staged kernel (bf16):
#   fused:  the weights formed inside the grad_x1 product (128 x 256 tiles that fill the GPU), grad_x2
#           on the 128 x 128 tile kernel, W and x1 read k-major in place;
#   tiles:  half as many 128 x 256 tiles, so the weight pass, then both products on the tile kernel;
#   wide:   bf16's fused path with grad_x2 on 128 x 256 tiles;
#   passes: ragged sizes in two batches, where both inputs take the offset inputs' path.
# The tile kernels' launches in the backward tell the paths apart.  Bar: float64 autograd of plain
# torch on the GPU, rtol 1e-4 or 1e-2 (+ that times the largest).
PATHS = {"fused": (2, 4096, 2048, 2048), "tiles": (1, 4096, 4096, 2048), "wide": (1, 8192, 8192, 2048),
         "passes": (2, 3101, 3003, 300)}


def _op64(name, kw, a, b):
    """The named metric of one batch in plain torch (float64 inputs)."""
    if name == "correlation_distances":
        a, b = a - a.mean(1, keepdim=True), b - b.mean(1, keepdim=True)
    s = a @ b.T
    if "euclidean" in name:
        sq = (a.square().sum(1)[:, None] + b.square().sum(1)[None] - 2 * s).clamp_min(0)
        return sq if name.startswith("sq") else sq.sqrt()
    if name.startswith(("cosine", "correlation")):
        s = s / (a.norm(dim=1)[:, None] * b.norm(dim=1)[None])
        return s if name == "cosine_similarity" else 1 - s
    if name == "linear_kernel":
        return s
    return (s * kw["gamma"] + 1).pow(kw["degree"]) if name == "polynomial_kernel" else (s * kw["gamma"] + 1).tanh()


@pytest.mark.parametrize("path,dtype", [(p, t) for p in PATHS for t in (torch.float32, torch.bfloat16)
                                        if p != "wide" or t == torch.bfloat16])
@pytest.mark.parametrize("name,kw", BWD_OPS)
def test_backward_paths_of_large_problems(name, kw, path, dtype):
    import torchpairwise_amd as tp
    from tests._util import assert_close

    B, n, m, d = PATHS[path]
    print(f"{path} {name} {dtype} B={B} n={n} m={m} d={d}", flush=True)
    gen = torch.Generator(DEV).manual_seed(5)
    x1, x2, g = (torch.randn(B, r, c, generator=gen, device=DEV).to(dtype) for r, c in ((n, d), (m, d), (n, m)))
    want = ([], [])
    for i in range(B):
        ra, rb = x1[i].double().requires_grad_(), x2[i].double().requires_grad_()
        for lst, t in zip(want, torch.autograd.grad(_op64(name, kw, ra, rb), (ra, rb), g[i].double())):
            lst.append(t)
    tol = 1e-4 if dtype == torch.float32 else 1e-2
    for offset in (False, True):
        a, b = _leaf(x1, offset), _leaf(x2, offset)
        out = getattr(tp, name)(a, b, **kw)
        count = {}
        for family in ("op_backward_kernel", "inner_tile_kernel", "grad_wide_bf16_kernel"):
            with Launches(family) as launches:
                got = torch.autograd.grad(out, (a, b), g, retain_graph=True)
            count[family] = launches.count
        print(offset, count, flush=True)
        assert count["op_backward_kernel"] == 0
        # (sqeuclidean takes the power-sum kernels, polynomial and linear other mixes of these products)
        if name.startswith(("euclidean", "cosine", "correlation", "sigmoid")) and not offset:
            tiles, wide = {"fused": (1, 0), "tiles": (2, 0), "wide": (0, 1), "passes": (0, 0)}[path]
            assert (count["inner_tile_kernel"], count["grad_wide_bf16_kernel"]) == (tiles, wide)
        for k in (0, 1):
            w = torch.stack(want[k])
            assert_close(got[k].float(), w, rtol=tol, atol=tol * float(w.abs().max()),
                         what=f"{name} {path} offset={offset} grad_x{k + 1}")


# Batches whose weight pass and products end sooner than the one-launch kernel (regression: cosine up to 1.7
# times and bf16 of aligned sizes 1.6 times as slow on it), and their neighbours that stay; long blocks of
# either direction first.  Bar as above.
@pytest.mark.parametrize("name,dtype,B,n,m,d,one", [
    ("cosine_distances", torch.float32, 50, 128, 1664, 200, 0), ("cosine_distances", torch.float32, 50, 64, 300, 200, 1),
    ("cosine_distances", torch.bfloat16, 200, 128, 128, 427, 0), ("cosine_distances", torch.bfloat16, 50, 66, 3468, 200, 1),
    ("linear_kernel", torch.bfloat16, 200, 128, 128, 640, 0), ("linear_kernel", torch.bfloat16, 200, 128, 127, 640, 1),
    ("euclidean_distances", torch.bfloat16, 200, 192, 128, 384, 0), ("euclidean_distances", torch.float32, 16, 2880, 93, 427, 1),
])
def test_backward_batches_one_launch_or_passes(name, dtype, B, n, m, d, one):
    import torchpairwise_amd as tp
    from tests._util import assert_close

    print(f"{name} {dtype} B={B} n={n} m={m} d={d}", flush=True)
    gen = torch.Generator(DEV).manual_seed(6)
    x1, x2, g = (torch.randn(B, r, c, generator=gen, device=DEV).to(dtype) for r, c in ((n, d), (m, d), (n, m)))
    a, b = x1.clone().requires_grad_(), x2.clone().requires_grad_()
    out = getattr(tp, name)(a, b)
    with Launches("op_backward_kernel") as launches:
        got = torch.autograd.grad(out, (a, b), g)
    assert launches.count == one
    tol = 1e-4 if dtype == torch.float32 else 1e-2
    for i in (0, B - 1):
        ra, rb = x1[i].double().requires_grad_(), x2[i].double().requires_grad_()
        for t, w in zip(got, torch.autograd.grad(_op64(name, {}, ra, rb), (ra, rb), g[i].double())):
            assert_close(t[i].float(), w, rtol=tol, atol=tol * float(w.abs().max()), what=f"{name} batch {i}")


# bf16 backward of small problems with aligned inputs and with inputs offset by one element
# (polynomial: the weight pass and the products; the others: op_backward_kernel with whole and element
# loads): bar: the bf16 tolerance against float64 autograd, 1e-2 (+ 1e-2 * max), and the two calls
# within one bf16 ulp of each other (2^-7 relative, the ulp of values in [1, 2), + 1e-3 * max).
@pytest.mark.parametrize("B,n,m,d", [(2, 128, 192, 64), (1, 1088, 1024, 72), (1, 256, 128, 264), (1, 128, 65536, 256)])
@pytest.mark.parametrize("name", ["euclidean_distances", "cosine_distances", "polynomial_kernel", "sigmoid_kernel"])
def test_backward_products_kmajor_bf16(name, B, n, m, d):
    import torchpairwise_amd as tp
    from tests._util import assert_close

    print(f"{name} bf16 B={B} n={n} m={m} d={d}", flush=True)
    fn = getattr(tp, name)
    kw = {"polynomial_kernel": dict(degree=2, gamma=0.05), "sigmoid_kernel": dict(gamma=0.02)}.get(name, {})
    x1 = randn(B, n, d, seed=0, dtype=torch.bfloat16)
    x2 = randn(B, m, d, seed=1, dtype=torch.bfloat16)
    g = randn(B, n, m, seed=2, dtype=torch.bfloat16)
    grads = {}
    for misaligned in (False, True):
        a, b = _leaf(x1, misaligned), _leaf(x2, misaligned)
        fn(a, b, **kw).backward(g.to(DEV))
        grads[misaligned] = (a.grad.float().cpu(), b.grad.float().cpu())
    ra, rb = x1.double().requires_grad_(), x2.double().requires_grad_()
    fn(ra, rb, **kw).backward(g.double())
    for k, want in enumerate((ra.grad, rb.grad)):
        kmaj, other = grads[False][k], grads[True][k]
        scale = float(want.abs().max())
        assert_close(kmaj, want, rtol=1e-2, atol=1e-2 * scale, what=f"{name} grad_x{k + 1} (aligned)")
        assert_close(kmaj, other.double(), rtol=2.0 ** -7, atol=1e-3 * scale,
                     what=f"{name} grad_x{k + 1} aligned vs offset")


# --------------------------------------------------------------------------------------
# Rows that are not whole 128-byte chunks: for outputs of 2^20 entries or more that the
# small-output kernel does not take, the public inner-product ops copy the operands zero-padded to
# whole chunks and take the tile kernel, against the staged kernel of the C entry, which zero-fills
# its last chunk.  Bit-identical either way.
# --------------------------------------------------------------------------------------
@pytest.mark.parametrize("dtype,n,m,d", [
    (torch.float32, 2100, 2000, 127), (torch.float32, 2049, 2080, 130), (torch.float32, 2060, 2048, 1),
    (torch.float32, 2050, 2047, 700), (torch.bfloat16, 2060, 2048, 255), (torch.bfloat16, 2049, 2056, 200),
])
@pytest.mark.parametrize("op,epi", [("euclidean_distances", capi.EPI_EUCLIDEAN),
                                    ("cosine_similarity", capi.EPI_COSINE_SIM),
                                    ("linear_kernel", capi.EPI_DOT)])
def test_padded_rows_equal_staged_kernel(dtype, n, m, d, op, epi):
    print(f"padded {op} {dtype} {n}x{m}x{d}", flush=True)
    x1 = randn(1, n, d, seed=11).to(DEV, dtype)
    x2 = randn(1, m, d, seed=12).to(DEV, dtype)
    x2[:, 5] = x1[:, 0]
    with Launches("inner_tile_kernel") as on_tile:
        got = getattr(torch.ops.torchpairwise, op)(x1[0], x2[0])
    with Launches("inner_small_kernel") as on_small:
        getattr(torch.ops.torchpairwise, op)(x1[0], x2[0])
    with Launches("pairwise_inner_kernel") as on_staged:
        want = _inner(x1, x2, epi, True)[0]
    assert (on_tile.count, on_small.count, on_staged.count) == (1, 0, 1)
    assert _same_bits(got, want)

