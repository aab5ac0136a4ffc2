"""fp32 attention on the matrix cores at the edges of its tiles: key counts
below, at and one past a 32-key tile, a 64-key chunk and a 128-query
workgroup, masked boards, grouped and shared kv heads, every head shape the
kernel is built for, through whole nets against the oracle."""
import numpy as np
import pytest

from katago_amd import modelgen, nn
from test_gpu_parity import _run_parity, _tiny_transformer

pytestmark = pytest.mark.gpu

HEADS = [(2, 2, 32, 32, 64), (4, 2, 32, 16, 64), (2, 1, 64, 64, 128)]


def _model(model_dir, heads, kv, dq, dv, c):
    arch = _tiny_transformer(heads, kv, dq, dv, c, True, True)
    return modelgen.write_model(arch, 31 + heads + dq, f"{model_dir}/{arch.name}-edges.bin.gz")


@pytest.mark.parametrize("nn_x,nn_y,boards", [(5, 5, (5, 4)), (8, 4, ((8, 4), 3)), (8, 8, (8, 5)), (13, 5, ((13, 5), 5)), (16, 8, ((16, 8), 7)),
                                              (19, 7, ((19, 7), 6)), (19, 19, (19, 9))], ids=lambda v: str(v))
@pytest.mark.parametrize("heads", HEADS, ids=["mha-q32v32", "gqa-q32v16", "mqa-q64v64"])
def test_key_counts_match_oracle(model_dir, heads, nn_x, nn_y, boards):
    """Tolerances are _compare's fp32 bounds (1e-3 absolute on the raw
    outputs; the sums of fp32 products agree to about 1e-6)."""
    _run_parity(_model(model_dir, *heads), False, 3, board_sizes=boards, label=f"attention {nn_x}x{nn_y}", nn_x=nn_x, nn_y=nn_y)


def test_rows_do_not_depend_on_batch(model_dir):
    lm = nn.LoadedModel(_model(model_dir, *HEADS[2]))
    h = nn.ComputeHandle(nn.ComputeContext(lm, 13, 13, use_fp16=False), max_batch=21)
    sp, gl = modelgen.synthetic_inputs(77, 21, 13, 13, board_sizes=(13, 9))
    full = h.get_output(sp, gl)
    one = h.get_output(sp[20:], gl[20:])
    for k in full:
        assert np.array_equal(full[k][20], one[k][0]), k
