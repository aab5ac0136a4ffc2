"""fp32 convolutions on bf16 matrix cores at the edges of their tiles: row
counts below, at and past 32, 64 and 96, on narrow, flat and square boards,
channel counts that give uneven and empty K groups (two to 24 16-channel
chunks) and column tiles of 32 and 64, through whole nets against the
oracle; and the same bits for a row on every tile."""
import numpy as np
import pytest

from katago_amd import modelgen, nn
from test_gpu_conv_stream import TRANSFORMER, _nbt, _regular
from test_gpu_parity import _run_parity

pytestmark = pytest.mark.gpu

NARROW = modelgen.Arch("narrowtflrs", 17, 48, 48, 16, ["attention", "ffn"], 16, 16, 32, 48, "ACTIVATION_SILU", heads=2, kv_heads=2,
                       q_head_dim=32, v_head_dim=32, ffn_c=96, learnable_rope=True, trunk_rmsnorm=True)
NETS = [NARROW, _regular(80), _regular(96), _nbt(384, 192), TRANSFORMER]


def _file(model_dir, arch):
    return modelgen.write_model(arch, 91, f"{model_dir}/{arch.name}-fp32.bin.gz")


@pytest.mark.parametrize("nn_x,nn_y", [(2, 2), (15, 2), (2, 16), (11, 3), (9, 7), (8, 8), (13, 5), (19, 5), (6, 16), (7, 14), (19, 19)], ids=str)
@pytest.mark.parametrize("arch", NETS, ids=lambda a: a.name)
def test_edges_match_oracle(model_dir, arch, nn_x, nn_y):
    """Tolerances are _compare's fp32 bounds (1e-3 absolute on the raw
    outputs): edges and layouts; test_sums_match_float64 holds the products."""
    _run_parity(_file(model_dir, arch), False, 1, board_sizes=((nn_x, nn_y),), label=f"fp32 {nn_x}x{nn_y}", nn_x=nn_x, nn_y=nn_y)


@pytest.mark.parametrize("arch", [_regular(64), _nbt(384, 192), TRANSFORMER, NARROW], ids=lambda a: a.name)
def test_rows_do_not_depend_on_batch(model_dir, arch):
    """Batches whose convolutions run on 32-, 64- and 96-row tiles and with K
    or columns over the waves."""
    h = nn.ComputeHandle(nn.ComputeContext(nn.LoadedModel(_file(model_dir, arch)), use_fp16=False), max_batch=60)
    sp, gl = modelgen.synthetic_inputs(5, 60, board_sizes=(19, 9))
    want = h.get_output(sp, gl)
    for n in (1, 7, 13, 30, 46):
        got = h.get_output(sp[:n], gl[:n])
        for k in want:
            assert np.array_equal(got[k], want[k][:n]), (n, k)


def _conv_text(w):
    return "c %d %d %d %d 1 1\n%s\n" % (*w.shape, " ".join(repr(float(v)) for v in w.reshape(-1)))


def _conv(x, w):
    """The device's conv of x [n, y, x, cin] with w [ky, kx, cin, cout]."""
    n, h, wd, _ = x.shape
    out = nn.test_evaluate(nn.TEST_CONV, _conv_text(w), n, wd, h, False, True, x, None, w.shape[3])
    return out.reshape(n, h, wd, w.shape[3])


def _conv64(x, w, dtype=np.float64):
    """The same as a sum of products in float64 (or float32, in some order)."""
    k = w.shape[0]
    xp = np.pad(x.astype(dtype), ((0, 0), (k // 2, k // 2), (k // 2, k // 2), (0, 0)))
    h, wd = x.shape[1:3]
    with np.errstate(all="ignore"):
        return sum(xp[:, dy:dy + h, dx:dx + wd] @ w[dy, dx].astype(dtype) for dy in range(k) for dx in range(k))


SHAPES = [(3, 32, 32, 1, 9), (3, 64, 64, 2, 19), (3, 192, 64, 16, 19), (3, 96, 64, 40, 19), (1, 384, 192, 1, 19), (1, 192, 384, 30, 19)]


def _pieces(a):
    """A float32 array as three bf16 arrays, each the rounded rest (nearest even)."""
    out, rest = [], a.astype(np.float32)
    for _ in range(3):
        bits = rest.view(np.uint32).astype(np.uint64)
        p = ((bits + 0x7FFF + ((bits >> 16) & 1)) & 0xFFFF0000).astype(np.uint32).view(np.float32)
        out.append(p)
        rest = rest - p
    return out


@pytest.mark.parametrize("k,cin,cout,n,side", SHAPES + [(3, 384, 64, 1, 19), (3, 80, 96, 3, 13), (1, 1024, 384, 4, 19), (1, 48, 96, 2, 7)], ids=str)
def test_sums_match_float64(k, cin, cout, n, side):
    """One conv on every tile against float64, in the 2-norm. A sum rounds once
    per 16 channels and tap (up to 216 times), each time by 2^-24 / sqrt(12) of
    a partial sum: 1.8e-7 if they were all of the final size; measured 0.5e-7 to
    1.7e-7 (numpy's float32 sums 1.2e-7 to 3.6e-7). Any of the three products of
    2^-18 left out of the six would give 1e-6 and more."""
    rng = np.random.default_rng(k + cin)
    x = rng.standard_normal((n, side, side, cin)).astype(np.float32)
    w = (rng.standard_normal((k, k, cin, cout)) * np.sqrt(2.0 / (k * k * cin))).astype(np.float32)
    want = _conv64(x, w)
    size = np.linalg.norm(want)
    assert np.linalg.norm(_conv(x, w) - want) <= 5e-7 * size
    if n == 1:  # what a product left out is, on the CPU
        a, b = _pieces(x), _pieces(w)
        for i, j in ((0, 2), (1, 1), (2, 0)):
            assert np.linalg.norm(_conv64(a[i], b[j])) > 1e-6 * size


@pytest.mark.parametrize("k,cin,cout,n,side", SHAPES, ids=str)
def test_infinite_and_largest_inputs(k, cin, cout, n, side):
    """Infinities, NaN and numbers past the largest bf16 (and past the last that
    rounds to it) among ordinary ones: sums are infinite and NaN where a float32
    conv's are, the others are right to 1e-5 of the sum of their terms' sizes."""
    rng = np.random.default_rng(k + cin)
    x = rng.standard_normal((n, side, side, cin)).astype(np.float32)
    w = (rng.standard_normal((k, k, cin, cout)) / cin).astype(np.float32)
    for i, v in enumerate((np.inf, -np.inf, np.nan, 3.4028235e38, -3.4e38, 3.396e38, 3.39e38)):
        x[0, (i * 2) % side, (i * 3) % side, (i * 5) % cin] = v
    got, want = _conv(x, w), _conv64(x, w)
    assert np.isinf(want).any() and np.isnan(want).any()
    assert np.array_equal(np.isnan(got), np.isnan(want))
    inf = np.isinf(want)
    assert np.array_equal(got[inf], want[inf].astype(np.float32))
    fin = np.isfinite(want)
    size = _conv64(np.abs(np.where(np.isfinite(x), x, 0)), np.abs(w))
    assert np.isfinite(got[fin]).all() and (np.abs(got[fin] - want[fin]) <= 1e-5 * size[fin]).all()


@pytest.mark.parametrize("x,y,n", [(155, 2, 1), (156, 2, 60), (187, 3, 1), (188, 3, 1), (300, 2, 2), (182, 181, 1)], ids=str)
def test_boards_wider_than_a_window(x, y, n):
    """A conv by itself on boards at and past the widest that the tiles' windows
    hold (155 for 96 rows, 187 for 32), and of more positions than their
    divisions take: the direct kernel has those."""
    rng = np.random.default_rng(x)
    inp = rng.standard_normal((n, y, x, 32)).astype(np.float32)
    w = (rng.standard_normal((3, 3, 32, 64)) / 17).astype(np.float32)
    got, want = _conv(inp, w), _conv64(inp, w)
    assert np.abs(got - want).max() <= 1e-5
