"""GPU parity of the quantized prefill matmul (Q4_0 / Q8_0 and Q4_K / Q5_K / Q6_K weights, fp16 activations,
fp16 MFMA with fp32 accumulation) against the CPU oracle, through the C ABI.

Oracle definition: Y[m][n] = sum_k h(deq(W)[n][k]) * X[m][k] with h = round-to-nearest-even to fp16 and
fp32 accumulation.  The kernels form the fp16 weight bit-exactly (h(d*q); for the K-quants the reference's
fp32 dequantization operation by operation, then h), so only the accumulation order differs.
Gate (north_star): max|y - ref| / max|ref| <= 1e-3; asserted: PARITY_TOL.
"""
import os
import subprocess
import sys

import numpy as np
import pytest

import ggufref as G
from openagents_amd import _ffi, backend
from openagents_amd.records import launched_kernels

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
GATE = 1e-3
PARITY_TOL = 2e-5
TILES = [(64, 64), (64, 128), (128, 128), (128, 256), (256, 128), (256, 256)]


def say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


_cache = {}


def weights(orc, qname, seed, n, k):
    key = (qname, seed, n, k)
    if key not in _cache:
        _cache[key] = orc.quantize(getattr(orc, qname), G.seeded_weights(seed, n, k))
    return _cache[key]


@pytest.mark.parametrize("qname", ["Q4_0", "Q8_0"])
@pytest.mark.parametrize("tile", TILES)
def test_every_tile_ragged_shapes(hip, orc, qname, tile):
    """m and n are ragged against every tile; k = 768 and 1280 exercise the partial last round of the
    256-wide register chunks for the 64- and 128-column tiles."""
    t = getattr(orc, qname)
    for m, n, k in ((1, 70, 768), (37, 300, 1280), (200, 130, 512), (333, 516, 1024)):
        say(f"prefill {qname} tile={tile} m={m} n={n} k={k}")
        W = weights(orc, qname, 800, n, k)
        X = G.seeded_acts(801 + m, m, k).astype(np.float16)
        ref = orc.prefill(t, W, X, n, k)
        ws = tile in ((64, 64), (64, 128), (128, 128), (128, 256))   # tiles with the producer/consumer (16) kernel
        for waves in (4,) + ((16,) if ws else ()):
            for ksplit in (1, 2, 4):
                if ksplit > 1 and (m * n) % 4:
                    continue
                y = hip.matmul_host(t, W, X, n, k, tile + (ksplit, waves))
                err = G.max_rel_err(y, ref)
                assert np.all(np.isfinite(y)) and err < PARITY_TOL, (tile, ksplit, waves, m, n, k, err)


@pytest.mark.parametrize("qname", ["Q4_K", "Q5_K", "Q6_K"])
@pytest.mark.parametrize("tile", TILES)
def test_k_quant_prefill_every_tile_ragged_shapes(hip, orc, qname, tile):
    """The K-quants run the four-wave family: weights dequantized in fp32 exactly as the reference does
    (one rounding per operation) and rounded to fp16 for the MFMA.  Ragged m and n against every tile; k of
    three and five super-blocks exercises the partial last round of the register chunks; Q6_K's 210-byte
    super-blocks put every second one on an odd dword boundary."""
    t = getattr(orc, qname)
    for m, n, k in ((1, 70, 768), (37, 300, 1280), (200, 130, 512), (333, 516, 1024)):
        say(f"prefill {qname} tile={tile} m={m} n={n} k={k}")
        W = weights(orc, qname, 830, n, k)
        X = G.seeded_acts(831 + m, m, k).astype(np.float16)
        ref = orc.prefill(t, W, X, n, k)
        families = (4, 16) if tile == (128, 256) and qname != "Q6_K" else (4,)   # Q4_K / Q5_K: also the producer / consumer kernel
        for waves in families:
            for ksplit in (1, 2, 4):
                if ksplit > 1 and (m * n) % 4:
                    continue
                y = hip.matmul_host(t, W, X, n, k, tile + (ksplit, waves))
                err = G.max_rel_err(y, ref)
                assert np.all(np.isfinite(y)) and err < PARITY_TOL, (tile, ksplit, waves, m, n, k, err)


@pytest.mark.parametrize("qname", ["Q4_K", "Q5_K", "Q6_K"])
def test_k_quant_prefill_default_plan_and_refusals(hip, orc, qname):
    """psn_qmatmul_prefill picks a four-wave tile by itself for the K-quants (a slice of the 4096 -> 14336
    projection at M = 64 and M = 512); the other kernel families exist for Q4_0 / Q8_0 only."""
    t = getattr(orc, qname)
    n, k = 1024, 4096
    W = weights(orc, qname, 840, n, k)
    for m in (64, 512):
        say(f"prefill {qname} default plan m={m} n={n} k={k}")
        X = G.seeded_acts(841 + m, m, k).astype(np.float16)
        err = G.max_rel_err(hip.matmul_host(t, W, X, n, k), orc.prefill(t, W, X, n, k))
        say(f"  max_rel_err={err:.3e}")
        assert err < PARITY_TOL
    X = G.seeded_acts(842, 64, k).astype(np.float16)
    for tile in ((128, 128, 1, 16), (256, 256, 1, 32)):
        with pytest.raises(backend.PsnError) as e:
            hip.matmul_host(t, W, X, n, k, tile)
        assert e.value.code == _ffi.E_UNSUPPORTED


@pytest.mark.parametrize("qname", ["Q4_0", "Q8_0", "Q4_K", "Q5_K", "Q6_K"])
def test_skinny_kernel_ragged_shapes(hip, orc, qname):
    """The M <= 64 kernel (waves code 64): every combination of ragged m and n, K ranges of one to many
    256-wide chunks (one chunk: the load rings are deeper than the whole range), with and without K split.
    Q6_K rows must be whole 16-byte words (K a multiple of 2048); its eight chunks per 2048 start at all eight
    possible offsets inside their aligned windows."""
    t = getattr(orc, qname)
    shapes = ((1, 70, 256), (37, 300, 768), (64, 130, 1280), (50, 516, 4096), (64, 64, 14336))
    if qname == "Q6_K":
        shapes = ((1, 70, 2048), (37, 300, 4096), (64, 130, 6144), (50, 516, 4096), (64, 64, 14336))
        with pytest.raises(backend.PsnError) as e:
            hip.matmul_host(t, weights(orc, qname, 859, 70, 768), G.seeded_acts(1, 4, 768).astype(np.float16), 70, 768, (64, 64, 1, 64))
        assert e.value.code == _ffi.E_UNSUPPORTED
    for m, n, k in shapes:
        say(f"skinny {qname} m={m} n={n} k={k}")
        W = weights(orc, qname, 860, n, k)
        X = G.seeded_acts(861 + m, m, k).astype(np.float16)
        ref = orc.prefill(t, W, X, n, k)
        for ksplit in (1, 2, 4, 8):
            if ksplit > 1 and (m * n) % 4:
                continue
            y = hip.matmul_host(t, W, X, n, k, (64, 64, ksplit, 64))
            err = G.max_rel_err(y, ref)
            assert np.all(np.isfinite(y)) and err < PARITY_TOL, (ksplit, m, n, k, err)
    # the result without K split does not depend on the run (fixed summation order)
    W = weights(orc, qname, 860, 516, 4096)
    X = G.seeded_acts(861 + 50, 50, 4096).astype(np.float16)
    ys = [hip.matmul_host(t, W, X, 516, 4096, (64, 64, 1, 64)) for _ in range(3)]
    assert np.array_equal(ys[0], ys[1]) and np.array_equal(ys[0], ys[2])
    with pytest.raises(backend.PsnError) as e:
        hip.matmul_host(t, W, G.seeded_acts(1, 65, 4096).astype(np.float16), 516, 4096, (64, 64, 1, 64))
    assert e.value.code == _ffi.E_UNSUPPORTED


@pytest.mark.parametrize("qname", ["Q4_0", "Q8_0"])
def test_prefill_m1_matches_matvec_f32_scheme(hip, orc, qname):
    """One row of the prefill is the F32-scheme matvec on the same fp16 activations, up to the fp16
    rounding of the weights (about 1.5e-4 of the output scale)."""
    t = getattr(orc, qname)
    n, k = 512, 4096
    W = weights(orc, qname, 810, n, k)
    X = G.seeded_acts(811, 1, k).astype(np.float16)
    y = hip.matmul_host(t, W, X, n, k)
    mv = hip.matvec_host(t, W, X[0].astype(np.float32), n, k, _ffi.ACT_F32)
    assert G.max_rel_err(y[0], mv) < GATE


@pytest.mark.parametrize("n,k", [(14336, 4096), (4096, 14336)])
@pytest.mark.parametrize("qname", ["Q4_0", "Q8_0", "Q4_K", "Q5_K", "Q6_K"])
def test_prefill_baseline_shapes_m64(hip, orc, qname, n, k):
    say(f"prefill {qname} m=64 n={n} k={k} (full oracle)")
    t = getattr(orc, qname)
    W = weights(orc, qname, 820, n, k)
    X = G.seeded_acts(821, 64, k).astype(np.float16)
    y = hip.matmul_host(t, W, X, n, k)
    err = G.max_rel_err(y, orc.prefill(t, W, X, n, k))
    say(f"  max_rel_err={err:.3e}")
    assert err < PARITY_TOL


@pytest.mark.parametrize("m", [512, 2048])
@pytest.mark.parametrize("n,k", [(14336, 4096), (4096, 14336)])
@pytest.mark.parametrize("qname", ["Q4_0", "Q8_0"])
def test_prefill_baseline_shapes_large_m_sampled(hip, orc, qname, m, n, k):
    """The GPU computes the full [m, n] product; the oracle re-computes a sample of 96 activation rows x
    160 weight rows (tile corners, edges and random interior rows) that the full result must match."""
    t = getattr(orc, qname)
    say(f"prefill {qname} m={m} n={n} k={k} (sampled oracle)")
    W = weights(orc, qname, 820, n, k)
    X = G.seeded_acts(830 + m, m, k).astype(np.float16)
    y = hip.matmul_host(t, W, X, n, k)
    rng = np.random.default_rng(m + n)
    mi = np.unique(np.concatenate([[0, 31, 32, 63, 64, 127, 128, 255, 256, m - 1], rng.integers(0, m, 86)]))
    ni = np.unique(np.concatenate([[0, 31, 32, 63, 64, 127, 128, 255, 256, n - 1], rng.integers(0, n, 150)]))
    ref = orc.prefill(t, W[ni], X[mi], len(ni), k)
    err = G.max_rel_err(y[np.ix_(mi, ni)], ref)
    say(f"  max_rel_err={err:.3e}")
    assert err < PARITY_TOL
    assert np.all(np.isfinite(y))


def test_prefill_linearity_and_zero(hip, orc):
    """Size-independent properties at a full shape: Y(X1 + X2) = Y(X1) + Y(X2) when X1, X2 have disjoint
    supports (exact in fp16), and zero activations give exactly zero."""
    t, n, k, m = orc.Q8_0, 4096, 4096, 128
    W = weights(orc, "Q8_0", 840, n, k)
    X = G.seeded_acts(841, m, k).astype(np.float16)
    X1, X2 = X.copy(), X.copy()
    X1[:, k // 2:] = 0
    X2[:, :k // 2] = 0
    y, y1, y2 = (hip.matmul_host(t, W, A, n, k) for A in (X, X1, X2))
    assert G.max_rel_err(y, y1 + y2) < PARITY_TOL
    assert not hip.matmul_host(t, W, np.zeros((m, k), np.float16), n, k).any()


@pytest.mark.parametrize("qname", ["Q4_0", "Q8_0"])
def test_wide_kernel_ragged_shapes(hip, orc, qname):
    """The large-M kernel (waves code 32, 256 x 256 tiles, weights decoded from raw bytes by the multiplying
    wave): ragged m and n against the tile, K ranges from one 256-chunk (the load rings are as deep as the
    whole range) to many, with and without K split; the result without K split is the same on every run."""
    t = getattr(orc, qname)
    for m, n, k in ((256, 256, 256), (1, 70, 512), (300, 296, 1280), (512, 768, 2048), (257, 513, 4096), (640, 260, 3584)):
        say(f"wide {qname} m={m} n={n} k={k}")
        W = weights(orc, qname, 870, n, k)
        X = G.seeded_acts(871 + m, m, k).astype(np.float16)
        ref = orc.prefill(t, W, X, n, k)
        for ksplit in (1, 2, 4):
            if ksplit > 1 and ((m * n) % 4 or k // 256 < ksplit):
                continue
            y = hip.matmul_host(t, W, X, n, k, (256, 256, ksplit, 32))
            err = G.max_rel_err(y, ref)
            assert np.all(np.isfinite(y)) and err < PARITY_TOL, (ksplit, m, n, k, err)
    W = weights(orc, qname, 870, 513, 4096)
    X = G.seeded_acts(871 + 257, 257, 4096).astype(np.float16)
    ys = [hip.matmul_host(t, W, X, 513, 4096, (256, 256, 1, 32)) for _ in range(3)]
    assert np.array_equal(ys[0], ys[1]) and np.array_equal(ys[0], ys[2])
    with pytest.raises(backend.PsnError) as e:
        hip.matmul_host(t, W, X, 513, 4096, (128, 256, 1, 32))          # the wide kernel has one tile
    assert e.value.code == _ffi.E_UNSUPPORTED


def test_prefill_errors(hip, orc):
    n, k = 64, 512
    W = weights(orc, "Q4_0", 850, n, k)
    w = hip.upload_weight(orc.Q4_0, W, n, k)
    x = hip.upload(np.zeros((4, k), np.float16))
    y = hip.alloc(4 * n * 4)
    with pytest.raises(backend.PsnError) as e:
        hip.quantized_matmul(w, x, y, 4, tile=(96, 96))
    assert e.value.code == _ffi.E_UNSUPPORTED
    with pytest.raises(backend.PsnError) as e:
        hip.quantized_matmul(w, x, y, 8)                      # X and Y too small for 8 rows
    assert e.value.code == _ffi.E_INVALID_ARG
    wk = hip.upload_weight(orc.Q6_K, weights(orc, "Q6_K", 851, n, k), n, k)
    with pytest.raises(backend.PsnError) as e:
        hip.quantized_matmul(wk, x, y, 4, tile=(64, 64, 1, 64))   # Q6_K rows of K = 512 are not whole 16-byte words
    assert e.value.code == _ffi.E_UNSUPPORTED
    hip.quantized_matmul(w, x, y, 4)
    hip.sync()


def test_prefill_default_plans_over_seeded_random_shapes(hip, orc):
    """The planner's own choice of family, tile and K split for shapes nobody tuned for, all five formats."""
    rng = np.random.default_rng(6150)
    for case in range(30):
        qname = ["Q4_0", "Q8_0", "Q4_K", "Q5_K", "Q6_K"][case % 5]
        qt = getattr(orc, qname)
        k = int(rng.choice([256, 512, 1024, 1536, 2048, 4096]))
        n = int(rng.integers(1, 900))
        m = int(rng.choice([1, 3, 17, 64, 65, 100, 128, 257, 300, 520]))
        say(f"random prefill #{case}: {qname} m={m} n={n} k={k} plan={backend.prefill_plan(m, n, k, hip.compute_units, qt)}")
        b = orc.quantize(qt, G.seeded_weights(6200 + case, n, k))
        x = G.seeded_acts(6300 + case, m, k).astype(np.float16)
        ref = orc.prefill(qt, b, x, n, k)
        got = hip.matmul_host(qt, b, x, n, k)
        assert G.max_rel_err(got, ref) < 2e-5, (qname, m, n, k)


@pytest.mark.parametrize("qname", ["Q4_0", "Q8_0", "Q4_K", "Q5_K", "Q6_K"])
def test_dense_family_ragged_shapes(hip, orc, qname):
    """Family 128: the matrix is rewritten as fp16 fragments once (psn_prefill_<fmt>_unpack), then multiplied
    on 256 x 256 or 128 x 256 tiles.  Ragged m and n against the tiles and against the 32-row fragment blocks,
    one to sixteen chunks of K, every K split the shape allows; the fp16 values are those of the other
    families, so the same tolerance holds."""
    t = getattr(orc, qname)
    for m, n, k in ((1, 40, 256), (37, 300, 1280), (260, 700, 2048), (333, 516, 1024), (257, 256, 512), (520, 33, 4096)):
        W = weights(orc, qname, 820, n, k)
        X = G.seeded_acts(821 + m, m, k).astype(np.float16)
        ref = orc.prefill(t, W, X, n, k)
        for ksplit in (1, 2, 4):
            if ksplit > 1 and ((m * n) % 4 or k // 256 < ksplit):
                continue
            for bm in (256, 128):
                say(f"dense prefill {qname} m={m} n={n} k={k} rows per tile={bm} ksplit={ksplit}")
                y = hip.matmul_host(t, W, X, n, k, (bm, 256, ksplit, 128))
                err = G.max_rel_err(y, ref)
                assert np.all(np.isfinite(y)) and err < PARITY_TOL, (qname, bm, ksplit, m, n, k, err)
    with pytest.raises(backend.PsnError) as e:
        hip.matmul_host(t, W, X, n, k, (128, 128, 1, 128))                      # the dense kernels' tiles are 256 columns wide
    assert e.value.name == "PSN_E_UNSUPPORTED"


def test_dense_family_in_graphs_needs_its_workspace_first(hip, orc):
    """Large M takes the dense family by default.  Its fp16 copy of the matrix lives in the stream's
    workspace, which cannot be allocated during a capture: on a stream that has none the default plan falls
    back to the other families (same result), a forced dense launch is refused, and after psn_prefill_reserve
    the capture contains the dense launches and replays to the eager result."""
    t, n, k, m = orc.Q4_K, 3000, 768, 3000
    assert backend.prefill_plan(m, n, k, hip.compute_units, t)[3] == 128
    assert backend.prefill_plan(64, n, k, hip.compute_units, t)[3] != 128
    W = weights(orc, "Q4_K", 830, n, k)
    X = G.seeded_acts(831, m, k).astype(np.float16)
    ref = orc.prefill(t, W, X, n, k)
    w, x = hip.upload_weight(t, W, n, k), hip.upload(X)
    y = hip.alloc(m * n * 4)
    s2 = hip.new_stream()
    try:
        with hip.on_stream(s2):
            hip.begin_capture()
            try:
                hip.quantized_matmul(w, x, y, m)                                  # no workspace on this stream: not dense
                with pytest.raises(backend.PsnError) as e:
                    hip.quantized_matmul(w, x, y, m, (256, 256, 1, 128))
                assert e.value.name == "PSN_E_INVALID_ARG"
            finally:
                g = hip.end_capture()
            hip.launch_graph(g)
            hip.sync()
            assert G.max_rel_err(y.download(np.float32, (m, n)), ref) < PARITY_TOL
            hip.destroy_graph(g)
            hip.reserve_prefill(n, k)
            y.fill_zero()
            hip.begin_capture()
            try:
                hip.quantized_matmul(w, x, y, m)                                  # dense now
                hip.quantized_matmul(w, x, y, m, (256, 256, 2, 128))
            finally:
                g = hip.end_capture()
            for _ in range(3):
                hip.launch_graph(g)
                hip.sync()
                assert G.max_rel_err(y.download(np.float32, (m, n)), ref) < PARITY_TOL
            hip.destroy_graph(g)
    finally:
        hip.destroy_stream(s2)


OUT_OF_MEMORY = """
import ctypes, sys
fake = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)          # its hipMalloc comes before the runtime's for what is loaded from here on
import numpy as np
from openagents_amd import _ffi, backend, quantize
from openagents_amd.records import launched_kernels
hip = backend.HipBackend(0)
m, n, k, rng = 4096, 4096, 4096, np.random.default_rng(5)
assert backend.prefill_choice(m, n, k, _ffi.Q4_0)[3] == 128
w = hip.upload_weight(_ffi.Q4_0, quantize.quantize(_ffi.Q4_0, rng.standard_normal((n, k), dtype=np.float32), 8), n, k)
x, y = hip.upload(rng.standard_normal((m, k), dtype=np.float32).astype(np.float16)), hip.alloc(m * n * 4)
def out():
    y.upload(np.full((m, n), np.nan, np.float32))
    names = launched_kernels(hip, lambda: hip.quantized_matmul(w, x, y, m))
    return names, y.download(np.float32, (m, n))
hip.reserve(4096, 8)                                              # a small workspace, which stays
copy = ctypes.c_size_t.in_dll(fake, "refuse_from")
asked = ctypes.c_int.in_dll(fake, "refused")
copy.value = n * k * 2
names, got = out()
assert asked.value == 1 and "dense" not in names, (asked.value, names)
again, same = out()
assert asked.value == 1 and again == names and np.array_equal(got, same)       # not asked for again
assert hip.lib.hipGetLastError() == 0
xv = hip.upload(rng.standard_normal((8, k), dtype=np.float32))
yv = hip.alloc(8 * n * 4)
hip.begin_capture()                                               # the small workspace is there: nothing has to grow while capturing
hip.quantized_matvec(w, xv, yv, 8, _ffi.ACT_Q8)
hip.destroy_graph(hip.end_capture())
try:
    hip.quantized_matmul(w, x, y, m, (256, 256, 1, 128))          # asked for by name: refused as before
    raise SystemExit("no error")
except backend.PsnError as e:
    assert e.name == "PSN_E_OOM", e
copy.value = 1 << 62
hip.reserve_prefill(n, k)
names, dense = out()
assert "dense" in names and float(np.max(np.abs(dense - got)) / np.max(np.abs(got))) < 2e-6, names
print("fell back")
"""


def test_a_copy_that_does_not_fit_the_device_leaves_the_kernels_that_need_none(hip, tmp_path):
    """A process of its own in which hipMalloc answers out-of-memory from a size on: psn_qmatmul_prefill runs without the dequantized copy instead of failing, keeps the workspace it had,
    leaves no error behind, does not ask for the copy at every call, and takes the dense family again once psn_prefill_reserve has got it."""
    src, so = tmp_path / "fake.c", tmp_path / "fake.so"
    src.write_text("""
#include <dlfcn.h>
#include <stddef.h>
size_t refuse_from = (size_t)1 << 62;
int refused = 0;
int hipMalloc(void **p, size_t n) {
    static int (*real)(void **, size_t);
    if (!real) real = (int (*)(void **, size_t))dlsym(dlopen("libamdhip64.so", RTLD_NOW | RTLD_LOCAL), "hipMalloc");
    if (n >= refuse_from) { ++refused; *p = 0; return 2; }
    return real(p, n);
}
""")
    subprocess.check_call(["gcc", "-shared", "-fPIC", "-o", str(so), str(src), "-ldl", "-L/opt/rocm/lib", "-Wl,-rpath,/opt/rocm/lib"])
    say("prefill without room for the copy")
    got = subprocess.run([sys.executable, "-c", OUT_OF_MEMORY, str(so)], cwd=ROOT, capture_output=True, text=True, timeout=100)
    assert got.returncode == 0 and got.stdout.strip().endswith("fell back"), got.stdout + got.stderr


@pytest.mark.parametrize("qname", ["Q4_0", "Q8_0", "Q4_K", "Q5_K", "Q6_K"])
def test_packed_weights_multiply_like_the_dense_family(hip, orc, qname):
    """psn_prefill_pack once, psn_qmatmul_prefill_packed for several X of different heights: the oracle's
    result each time, and the dense family's (same fragments, same multiply) up to the order of the K ranges' sums."""
    t = getattr(orc, qname)
    n, k = 700, 2048
    W = weights(orc, qname, 840, n, k)
    w = hip.upload_weight(t, W, n, k)
    packed = hip.pack_for_prefill(w)
    assert packed.nbytes >= 768 * k * 2
    for m in (1, 260, 37, 384, 1100):                                                    # (64 x 64 tiles at this width, with and without a K cut)
        X = G.seeded_acts(841 + m, m, k).astype(np.float16)
        y = hip.alloc(m * n * 4)
        hip.quantized_matmul_packed(packed, hip.upload(X), y, m, n, k)
        got = y.download(np.float32, (m, n))
        assert G.max_rel_err(got, orc.prefill(t, W, X, n, k)) < PARITY_TOL, (qname, m)
        same = hip.matmul_host(t, W, X, n, k, (256, 256, 1, 128))
        assert G.max_rel_err(got, same) < 2e-6                                          # the library may cut K (atomic adds): not bit for bit
    with pytest.raises(backend.PsnError) as e:
        hip.quantized_matmul_packed(hip.alloc(1024), hip.upload(X), y, m, n, k)          # not a packed buffer of this shape
    assert e.value.name == "PSN_E_INVALID_ARG"
    with pytest.raises(backend.PsnError) as e:
        hip.quantized_matmul_packed(packed, hip.upload(X), y, m, n, 2000)
    assert e.value.name == "PSN_E_SHAPE"


@pytest.mark.parametrize("qname", ["Q4_0", "Q8_0", "Q4_K", "Q5_K", "Q6_K"])
def test_packed_fragments_hold_the_reference_fp16_values_bit_for_bit(hip, orc, qname):
    """psn_prefill_pack writes h(deq(W)): every weight as the fp16 rounding of the value the reference's
    dequantizer returns, in fragment order [row / 32][k / 16][half][row % 32][8].  Read back and compared
    bit for bit (up to the sign of a zero) with numpy.float16 of the oracle's dequantization -- rows scaled over twelve binades so that
    block scales, mins and fp16 roundings of every size occur, and a ragged last row panel."""
    t = getattr(orc, qname)
    n, k = 200, 2048
    rng = np.random.default_rng(8100)
    w = rng.standard_normal((n, k), dtype=np.float32) * np.exp2(rng.integers(-8, 4, (n, k // 32))).astype(np.float32).repeat(32, axis=1)
    blocks = orc.quantize(t, w)
    wt = hip.upload_weight(t, blocks, n, k)
    packed = hip.pack_for_prefill(wt)
    npanel = -(-n // 32)
    raw = packed.download(np.uint16, (packed.nbytes // 2,))[:npanel * (k // 16) * 64 * 8].reshape(npanel, k // 16, 2, 32, 8)
    # [panel][kslice][half][row % 32][j] -> [row][k]
    got = raw.transpose(0, 3, 1, 2, 4).reshape(npanel * 32, k)[:n]
    want = orc.dequantize(t, blocks, k).reshape(n, k).astype(np.float16).view(np.uint16)
    # a zero keeps no sign: the reference's d * sc * (q - 32) is -0 where d * sc is negative and q = 32, the
    # kernels' fused form d sc q - 32 d sc returns +0 (Q6_K; the other formats agree in the sign of zero too)
    zero = (want & 0x7fff) == 0
    got, want = np.where(zero, got & 0x7fff, got), np.where(zero, want & 0x7fff, want)
    differ = np.argwhere(got != want)
    assert differ.size == 0, [(int(r), int(c), hex(int(got[r, c])), hex(int(want[r, c]))) for r, c in differ[:6]]


def test_prefill_refuses_operands_beyond_32_bit_offsets(hip, orc):
    """Several families address X and W with 32-bit byte offsets: shapes that would overflow them are
    refused by the host before any buffer is looked at."""
    w = hip.upload_weight(orc.Q4_0, weights(orc, "Q4_0", 850, 64, 4096), 64, 4096)
    x, y = hip.alloc(1 << 20), hip.alloc(1 << 20)
    with pytest.raises(backend.PsnError) as e:
        hip.quantized_matmul(w, x, y, 1 << 20)                       # X would be 8 GiB
    assert e.value.name == "PSN_E_SHAPE" and "4 GiB" in str(e.value)
    with pytest.raises(backend.PsnError) as e:
        hip.quantized_matmul_packed(x, x, y, 1 << 20, 64, 4096)
    assert e.value.name == "PSN_E_SHAPE"


@pytest.mark.parametrize("qname", ["Q4_0", "Q8_0", "Q4_K", "Q5_K", "Q6_K"])
def test_in_loop_kernels_at_tile_and_range_edges(hip, orc, qname):
    """The eight-wave kernels (family 4, tiles of 64 and 128 columns) one row and column either side of their tiles, with K
    ranges of one, two, an odd and an even number of 256-wide chunks (their loop takes chunks in pairs and asks for raw
    bytes two chunks ahead), and a K split that leaves a range empty.  fp16 products are exact in fp32, so only the order
    of at most 2048 sums differs from the oracle: PARITY_TOL is far above 2048 * 2^-24."""
    t = getattr(orc, qname)
    for tile in ((64, 64), (64, 128), (128, 128), (256, 128)):
        for m, n, k in ((tile[0] - 1, tile[1] + 1, 256), (tile[0] + 1, tile[1] - 1, 512), (tile[0], tile[1], 768), (65, 3 * tile[1], 2048)):
            say(f"in-loop {qname} tile={tile} m={m} n={n} k={k}")
            W = weights(orc, qname, 880, n, k)
            X = G.seeded_acts(881 + m, m, k).astype(np.float16)
            ref = orc.prefill(t, W, X, n, k)
            for ksplit in (1, 4) if (m * n) % 4 == 0 else (1,):
                y = hip.matmul_host(t, W, X, n, k, tile + (ksplit, 4))
                err = G.max_rel_err(y, ref)
                assert np.all(np.isfinite(y)) and err < PARITY_TOL, (tile, ksplit, m, n, k, err)


@pytest.mark.parametrize("qname", ["Q4_0", "Q8_0", "Q4_K", "Q5_K", "Q6_K"])
def test_thin_kernels_at_tile_and_range_edges(hip, orc, qname):
    """Family 8 (16 to 64 rows of X, 16 to 64 of W), every kernel of the format by name: X at either end of its sixteens and below, fewer weight
    rows than a tile, ragged last tiles, K ranges in which no, some and all of the eight waves have a chunk, one and several, with and without
    a cut of K (one that leaves ranges empty, too).  fp16 products are exact in fp32, so only the order of at most 4096 sums differs from the
    oracle: PARITY_TOL is far above 2^-24 sqrt(4096)."""
    t = getattr(orc, qname)
    kernels = [(tm, rt) for tm in (1, 2, 3, 4) for rt in (1, 2, 4) if rt < 4 or tm in {"Q8_0": (1,), "Q6_K": (1, 2, 3)}.get(qname, (2, 3))]
    for n, k in ((5, 256), (17, 768), (300, 2304), (132, 4096)):
        W = weights(orc, qname, 890, n, k)
        X = G.seeded_acts(891, 64, k).astype(np.float16)
        ref = orc.prefill(t, W, X, n, k)
        for tm, rt in kernels:
            for m in sorted({1, 16 * tm - 15, 16 * tm - 4, 16 * tm}):
                for ksplit in (1, 2, 5) if (m * n) % 4 == 0 else (1,):
                    say(f"thin {qname} {tm} {rt} m={m} n={n} k={k} ksplit={ksplit}")
                    hip.lib.psn_launch_log_clear()
                    y = hip.matmul_host(t, W, X[:m], n, k, (16 * tm, 16 * rt, ksplit, 8))
                    assert f"psn_prefill_{qname[0].lower() + qname[1:]}_thin_{tm}_{rt}" in hip.lib.psn_launch_log().decode().split(";")
                    err = G.max_rel_err(y, ref[:m])
                    assert np.all(np.isfinite(y)) and err < PARITY_TOL, (tm, rt, ksplit, m, n, k, err)
    for tile in {(16 * tm, 16 * rt) for tm in (1, 2, 3, 4) for rt in (1, 2, 4)} - {(16 * tm, 16 * rt) for tm, rt in kernels} | {(0, 16), (80, 16), (24, 16), (16, 128), (-16, 16)}:
        with pytest.raises(backend.PsnError) as e:
            hip.matmul_host(t, W, X[:1], n, k, tile + (1, 8))
        assert e.value.name == "PSN_E_UNSUPPORTED"
    for tile, m in (((16, 16, 1, 8), 17), ((64, 32, 0, 8), 64), ((64, 32, 65, 8), 64)):                     # more rows than the tile, cuts outside 1..64
        with pytest.raises(backend.PsnError) as e:
            hip.matmul_host(t, W, X[:m], n, k, tile)
        assert e.value.name == "PSN_E_UNSUPPORTED"


@pytest.mark.parametrize("qname", ["Q4_0", "Q8_0", "Q4_K", "Q5_K", "Q6_K"])
def test_the_choice_is_what_runs(hip, orc, qname):
    """psn_qmatmul_prefill_choice names the launch of psn_qmatmul_prefill: the same kernels with and without it as an explicit tile."""
    t = getattr(orc, qname)
    for n, k, ms in ((300, 2304, (1, 17, 33, 49, 64, 65)), (4104, 1280, (1, 33, 64)), (8209, 1024, (16, 18, 48)), (2048, 2048, (64, 200, 2048))):
        w = hip.upload_weight(t, weights(orc, qname, 895, n, k), n, k)
        for m in ms:
            x, y = hip.upload(G.seeded_acts(896, m, k).astype(np.float16)), hip.alloc(m * n * 4)
            say(f"choice {qname} m={m} n={n} k={k}")
            ran = []
            for tile in (None, backend.prefill_choice(m, n, k, t, hip.compute_units)):
                hip.lib.psn_launch_log_clear()
                hip.quantized_matmul(w, x, y, m, tile)
                ran.append(hip.lib.psn_launch_log().decode())
            hip.sync()
            assert ran[0] == ran[1], (m, n, k, ran, tile)


@pytest.mark.parametrize("qname", ["Q4_0", "Q8_0", "Q4_K", "Q5_K", "Q6_K"])
def test_values_that_are_not_finite_stay_in_their_row_and_column(hip, orc, qname):
    """A block scale that is infinite or NaN spoils its weight row's column of Y, an infinity or NaN in X its row, and nothing else changes by a
    bit: thin and in-loop kernels, ragged against every tile (rows past the end repeat the last one, tiles past it are moved back)."""
    t = getattr(orc, qname)
    n, k = 300, 768
    clean_w = weights(orc, qname, 897, n, k)
    bad_w = clean_w.copy().reshape(n, -1)
    d_at = 208 if qname == "Q6_K" else 0
    cols, size = [0, 17, 250, n - 1], len(bad_w[0])
    for i, c in enumerate(cols):
        block = size - 210 if qname == "Q6_K" and i == 3 else 0
        bad_w[c, block + d_at:block + d_at + 2] = np.array([0x7c00, 0x7e00, 0xfc00, 0x7c01], np.uint16)[i:i + 1].view(np.uint8)
    for tile, m in (((16, 16), 13), ((48, 16), 37), ((64, 32), 62), ((64, 64), 70), ((64, 128), 70), ((128, 128), 150), ((256, 128), 270)):
        say(f"not finite {qname} tile={tile}")
        x = G.seeded_acts(898, m, k).astype(np.float16)
        bad_x = x.copy()
        rows = [2, m - 1]
        bad_x[2, 5], bad_x[m - 1, k - 1] = np.inf, np.nan
        tile = tile + (1, 4 if m > 64 else 8)
        clean, y = hip.matmul_host(t, clean_w, x, n, k, tile), hip.matmul_host(t, bad_w, bad_x, n, k, tile)
        assert not np.isfinite(y[rows]).any() and not np.isfinite(y[:, cols]).any(), tile
        keep = np.ix_(np.setdiff1d(np.arange(m), rows), np.setdiff1d(np.arange(n), cols))
        assert np.isfinite(clean).all() and np.array_equal(clean[keep], y[keep]), tile


@pytest.mark.parametrize("m,n,k", [(1, 1, 256), (63, 65, 512), (64, 64, 2048), (65, 130, 768), (129, 127, 1280), (128, 1000, 2560), (257, 255, 256), (300, 2050, 512), (1025, 1021, 256),
                                   (2049, 4100, 256)])
def test_packed_multiply_at_tile_edges(hip, orc, m, n, k):
    """Shapes a row and a column either side of the tiles' edges, odd row lengths of Y (stored word by word), and K in several ranges; mostly 64 x 64 tiles, the last ones 64 x 128
    and 256 x 256.  Products are exact in fp32, so only the order of at most 2560 sums differs from the oracle: PARITY_TOL is far above 2560 * 2^-24."""
    W = weights(orc, "Q4_K", 870, n, k)
    X = G.seeded_acts(871 + m, m, k).astype(np.float16)
    packed = hip.pack_for_prefill(hip.upload_weight(orc.Q4_K, W, n, k))
    y = hip.upload(np.full((m, n), np.nan, np.float32))
    say(f"packed multiply m={m} n={n} k={k}")
    hip.quantized_matmul_packed(packed, hip.upload(X), y, m, n, k)
    err = G.max_rel_err(y.download(np.float32, (m, n)), orc.prefill(orc.Q4_K, W, X, n, k))
    assert err < PARITY_TOL, (m, n, k, err)


@pytest.mark.parametrize("m,n,k,plan", [(130, 129, 1280, (64, 64, 1)), (2, 2, 5120, (64, 64, 8)), (193, 4097, 1280, (64, 128, 1)), (193, 4100, 1280, (64, 128, 1)),
                                        (1, 4100, 3840, (64, 128, 4)), (2052, 65, 5120, (64, 128, 4)), (1281, 1537, 1280, (128, 128, 1)), (2049, 1000, 1280, (128, 128, 1)),
                                        (65, 4100, 5120, (128, 128, 4)), (1281, 3073, 1280, (128, 256, 1)), (4100, 1000, 1280, (128, 256, 1)), (4001, 2049, 1280, (256, 256, 1)),
                                        (4001, 2052, 1280, (256, 256, 1))])
def test_every_tile_of_the_packed_multiply(hip, orc, m, n, k, plan):
    """Ragged rows and columns, K long enough that every slot of the rings is used again, rows of Y that are whole 16-byte words and not, K cut and not, on the tile that the plan
    names and the launch runs.  fp16 products are exact in fp32: PARITY_TOL is far above the rounding of 5120 sums."""
    assert backend.packed_plan(m, n, k, hip.compute_units) == plan
    W = weights(orc, "Q8_0", 875, n, k)
    X = G.seeded_acts(876, m, k).astype(np.float16)
    packed = hip.pack_for_prefill(hip.upload_weight(orc.Q8_0, W, n, k))
    x, y = hip.upload(X), hip.upload(np.full((m, n), np.nan, np.float32))
    say(f"packed multiply m={m} n={n} k={k} plan={plan}")
    name = "psn_prefill_dense_f16" + {(256, 256): "", (128, 256): "_m128"}.get(plan[:2], f"_m{plan[0]}_n{plan[1]}")
    assert launched_kernels(hip, lambda: hip.quantized_matmul_packed(packed, x, y, m, n, k)) == ("psn_fill_zero + " if plan[2] > 1 else "") + name
    ref = X.astype(np.float64) @ orc.dequantize(orc.Q8_0, W, k).reshape(n, k).astype(np.float16).astype(np.float64).T
    err = G.max_rel_err(y.download(np.float32, (m, n)), ref)
    assert err < PARITY_TOL, (m, n, k, err)


@pytest.mark.parametrize("qname", ["Q4_0", "Q8_0", "Q4_K", "Q5_K", "Q6_K"])
def test_few_rows_over_more_weight_rows_than_one_round_of_64(hip, orc, qname):
    """64 rows of W per compute unit and one more: from there on psn_qmatmul_prefill may take family 4's tiles for M <= 64, and in every format it does (Q4_0 and Q8_0 at K = 768).
    fp16 products are exact in fp32, so only the order of at most 768 sums differs from the oracle: PARITY_TOL is far above 768 * 2^-24."""
    t = getattr(orc, qname)
    edge = 64 * hip.compute_units
    beyond = set()
    for n, k in ((edge, 512), (edge + 1, 256), (edge + 4, 512), (edge + 4, 768)):
        W = weights(orc, qname, 885, n, k)
        w, X = hip.upload_weight(t, W, n, k), G.seeded_acts(886, 64, k).astype(np.float16)
        ref = orc.prefill(t, W, X, n, k)
        for m in (1, 33, 64):
            choice = backend.prefill_choice(m, n, k, t, hip.compute_units)
            say(f"few rows {qname} m={m} n={n} k={k} {choice}")
            if n > edge:
                beyond.add((choice[3], m > 16))
            y = hip.upload(np.full((m, n), np.nan, np.float32))
            hip.quantized_matmul(w, hip.upload(X[:m]), y, m)
            err = G.max_rel_err(y.download(np.float32, (m, n)), ref[:m])
            assert err < PARITY_TOL, (m, n, k, err)
    assert (4, True) in beyond and (8, False) in beyond, beyond


@pytest.mark.parametrize("qname", ["Q4_0", "Q8_0", "Q4_K", "Q5_K", "Q6_K"])
def test_256_row_tiles_on_either_side_of_the_line_between_their_two_kernels(hip, orc, qname):
    """11 of 16 compute units with a workgroup: up to there 256 x 128 tiles multiply 32 x 32 x 16, beyond 16 x 16 x 32.  Ragged rows and columns, rows of Y that are whole 16-byte words
    and not, K cut and not.  fp16 products are exact in fp32, so what differs from float64 over the oracle's fp16 weights
    is the rounding of at most 1280 sums: PARITY_TOL is far above sqrt(1280) * 2^-24."""
    t = getattr(orc, qname)
    line = hip.compute_units * 11 // 16
    for m, k, ksplit in ((2041, 256, 1), (1793, 512, 1), (260, 1280, 4), (516, 1024, 2)):
        rows = -(-m // 256) * ksplit
        for n, name in ((line // rows * 128, "_pp32"), (line // rows * 128 - 127, "_pp32"), (line // rows * 128 + 1, "_pp"), (line // rows * 128 + 126, "_pp")):
            if ksplit > 1 and (m * n) % 4:
                continue
            W = weights(orc, qname, 890, n, k)
            w, X = hip.upload_weight(t, W, n, k), G.seeded_acts(891, m, k).astype(np.float16)
            y = hip.upload(np.full((m, n), np.nan, np.float32))
            x = hip.upload(X)
            say(f"256-row tiles {qname} m={m} n={n} k={k} ksplit={ksplit}")
            assert launched_kernels(hip, lambda: hip.quantized_matmul(w, x, y, m, (256, 128, ksplit, 4))).endswith(name), (m, n, k, ksplit)
            ref = X.astype(np.float64) @ orc.dequantize(t, W, k).reshape(n, k).astype(np.float16).astype(np.float64).T
            err = G.max_rel_err(y.download(np.float32, (m, n)), ref)
            assert err < PARITY_TOL, (m, n, k, ksplit, err)


@pytest.mark.parametrize("m,n", [(4, 1), (64, 512), (64, 516), (1024, 1024), (1028, 1025)])
def test_zero_fill_in_front_of_a_k_cut_at_the_lines_between_its_stores(hip, orc, m, n):
    """One 16-byte word, 128 KB of Y (the last with plain stores) and a little more, 4 MB (the last with a thread for every store) and a little more: nothing of what Y held is left.
    fp16 products are exact in fp32: PARITY_TOL is far above the rounding of 512 sums."""
    k = 512
    W = weights(orc, "Q4_0", 895, n, k)
    X = G.seeded_acts(896, m, k).astype(np.float16)
    w, x, y = hip.upload_weight(orc.Q4_0, W, n, k), hip.upload(X), hip.upload(np.full((m, n), np.nan, np.float32))
    hip.quantized_matmul(w, x, y, m, (64, 64, 2, 4))
    ref = X.astype(np.float64) @ orc.dequantize(orc.Q4_0, W, k).reshape(n, k).astype(np.float16).astype(np.float64).T
    assert G.max_rel_err(y.download(np.float32, (m, n)), ref) < PARITY_TOL
