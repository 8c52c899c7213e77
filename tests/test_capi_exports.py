"""The C-ABI library loads without a GPU and exports every symbol include/*.h declares."""
import ctypes
from pathlib import Path

from torchpairwise_amd import _capi


def test_header_declares_entry_points():
    syms = _capi.header_symbols()
    for name in ("tpw_pack_bool_rows", "tpw_bool_pairwise_reduce", "tpw_jaccard_bool",
                 "tpw_pairwise_inner", "tpw_lp_distances", "tpw_directed_hausdorff"):
        assert name in syms


def test_library_exports_every_declared_symbol():
    lib = ctypes.CDLL(str(_capi.LIB_PATH))
    headers = sorted(Path(_capi.HEADER).parent.glob("*.h"))
    missing = []
    for h in headers:
        for name in _capi.header_symbols(h):
            if not hasattr(lib, name):
                missing.append(f"{h.name}:{name}")
    assert not missing, f"declared but not exported: {missing}"


def test_binding_covers_header():
    assert set(_capi.header_symbols()) <= set(_capi._SIGNATURES), \
        set(_capi.header_symbols()) - set(_capi._SIGNATURES)


def test_pure_host_entry_points():
    l = _capi.lib()
    assert l.tpw_packed_words(1) == 4
    assert l.tpw_packed_words(128) == 4
    assert l.tpw_packed_words(129) == 8
    assert l.tpw_packed_words(1024) == 32
    assert l.tpw_runtime_version() > 0
    assert l.tpw_inner_backward_workspace_size(1, 10, 20, 8) >= 4 * 10 * 20
    assert l.tpw_hausdorff_workspace_size(1, 2, 10, 3, 20, 3) > 0


def test_hausdorff_workspace_fits_the_static_buffer():
    # regression: sized for the dense kernels' keys where those never run (pairs x p1 > 2^28), which
    # the allocation-free entry then refused: 101, 155 and 119 MiB
    l = _capi.lib()
    for sizes in ((1, 255, 13000, 255, 1000, 3), (1, 255, 20000, 255, 200, 2), (1, 200, 25000, 200, 500, 1)):
        assert l.tpw_hausdorff_workspace_size(*sizes) <= 96 << 20, sizes


def test_lp_backward_splits_fill_three_blocks():
    """The Lp backward's workspace holds the narrow kernel's partials for three blocks per CU (256 CUs):
    8 splits of 12000 x 12000 x 64 (94 row blocks), 6 of 16384^2 x 16, 12 of 8192^2 x 64 (regression: it
    was split for two, up to 11 % slower)."""
    l = _capi.lib()
    for n, d, splits in ((12000, 64, 8), (16384, 16, 6), (8192, 64, 12)):
        size = l.tpw_lp_backward_workspace_size(1, n, n, d) - 4 * n * n  # beside the weights
        assert splits * 4 * n * d <= size < (splits + 1) * 4 * n * d


def test_small_output_rule():
    """Where the 64 x 64 inner-product kernel runs (256 CUs): not where the 128 x 128 tile kernel,
    padded copies or not, takes less (regression: wide rows went there, up to 2.2 times as slow)."""
    l = _capi.lib()

    def small(dtype, b, n, m, d, offset=0):
        return bool(l.tpw_pairwise_inner_forms_norms(4096 + offset, 8192, dtype, b, n, m, d))

    f32, bf16 = 0, 1
    for d in (256, 512, 1000, 1024, 2048):  # ragged m and partial chunks at 256 tiles
        assert not small(f32, 1, 2048, 2047, d) and not small(f32, 1, 2000, 2047, d)
        if d >= 1000:
            assert not small(bf16, 1, 2048, 2048, d) and not small(bf16, 1, 2000, 2047, d)
    assert not small(f32, 1, 2048, 2048, 500) and not small(f32, 1, 1664, 2048, 500)
    assert not small(f32, 1, 1700, 1999, 512) and not small(f32, 1, 1280, 2048, 768)
    for d in (1024, 2048, 4096, 65536):  # bf16 rows of whole chunks
        assert not small(bf16, 1, 1024, 2048, d) and not small(bf16, 1, 300, 5000, d)
        assert not small(bf16, 1, 64, 64, d)
    for n, m, d in ((64, 64, 128), (37, 1003, 50), (1000, 1000, 4096), (1024, 2048, 1000), (1280, 2041, 128)):
        assert small(f32, 1, n, m, d) and small(bf16, 1, n, m, min(d, 500))
        assert small(f32, 1, n, m, d, 4) and small(bf16, 1, n, m, min(d, 500), 2)
    assert small(f32, 250, 128, 128, 1000) and small(bf16, 250, 128, 128, 3000) and small(bf16, 1, 16000, 60, 768)
    assert not small(f32, 260, 64, 64, 50) and not small(bf16, 260, 64, 64, 50)

    def dot(dtype, b, n, m, d, offset=0):
        return bool(l.tpw_pairwise_inner_is_small(4096 + offset, 8192, dtype, b, n, m, d, _capi.EPI_DOT))

    # without norms (regression: the lines above, up to 1.9 times as slow here)
    assert dot(f32, 1, 1920, 1920, 340) and dot(f32, 1, 906, 3692, 1001) and dot(f32, 14, 500, 470, 2100)
    assert not dot(f32, 1, 1920, 1920, 1001) and not dot(f32, 1, 906, 3692, 2100) and not dot(f32, 1, 2048, 2047, 512)
    assert dot(bf16, 1, 1024, 1024, 2048) and dot(bf16, 1, 1300, 1900, 3000) and dot(bf16, 14, 500, 470, 3000)
    assert dot(bf16, 1, 1024, 1024, 4100) and dot(bf16, 1, 1000, 1050, 2048) and dot(bf16, 1, 1920, 1920, 2500, 2)
    assert dot(bf16, 1, 1300, 1900, 4100) and dot(bf16, 14, 500, 470, 4001) and dot(bf16, 1, 2000, 1700, 3000)
    assert not dot(bf16, 1, 1000, 2048, 1024) and not dot(bf16, 1, 1300, 1900, 8000) and not dot(bf16, 1, 1920, 1920, 4001)
    assert not dot(f32, 260, 64, 64, 50) and not dot(bf16, 260, 64, 64, 50)


def test_argument_errors_are_reported_without_gpu():
    l = _capi.lib()
    # invalid sizes are rejected on the host before any launch
    rc = l.tpw_lp_distances(None, None, 1, 4, 4, 3, -1.0, None, None)
    assert rc == 1
    assert b"p must be non-negative" in l.tpw_last_error()
    rc = l.tpw_bool_pairwise_reduce(None, None, 1, 4, 4, 0, 0, 0, None, None)
    assert rc == 1


def test_workspace_queries_accept_empty_sizes():
    # regression: split counts divided by the number of output tiles, 0 for an empty side;
    # run in a child so that a host fault fails this test instead of ending the session
    import subprocess
    import sys

    code = (
        "from torchpairwise_amd import _capi\n"
        "l = _capi.lib()\n"
        "for n, m, d in ((0, 37, 5), (41, 0, 5), (0, 0, 5), (5, 7, 0)):\n"
        "    for b in (0, 1):\n"
        "        [l.tpw_family_backward_workspace_size(k, b, n, m, d) for k in range(6)]\n"
        "        l.tpw_lp_backward_workspace_size(b, n, m, d)\n"
        "        l.tpw_inner_backward_workspace_size(b, n, m, d)\n"
        "        l.tpw_haversine_workspace_size(b, n, m)\n"
        "        l.tpw_hausdorff_workspace_size(b, 2, n, 3, m, d)\n"
        "print('ok')\n")
    root = Path(__file__).resolve().parents[1]
    r = subprocess.run([sys.executable, "-c", code], cwd=root, capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.strip() == "ok", (r.returncode, r.stderr[-2000:])
