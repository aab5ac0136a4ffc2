"""fp16 attention with an item's queries over one, two and three workgroups:
batches on both sides of each rule, at query counts that fill the parts
unevenly, leave some without a query wave, or end in a partial wave. Rows are
the same bits at every batch."""
import numpy as np
import pytest

from katago_amd import modelgen, nn
from test_gpu_attention_fp32 import HEADS, _model

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nn_x,nn_y", [(19, 19), (19, 14), (16, 10), (13, 10), (16, 8), (8, 4)], ids=str)
@pytest.mark.parametrize("heads", HEADS, ids=["mha-q32v32", "gqa-q32v16", "mqa-q64v64"])
def test_rows_do_not_depend_on_batch(model_dir, heads, nn_x, nn_y):
    most = 257 // heads[0] + 1  # more items than CUs: one workgroup per item, some of which take two
    lm = nn.LoadedModel(_model(model_dir, *heads))
    h = nn.ComputeHandle(nn.ComputeContext(lm, nn_x, nn_y, use_fp16=True), max_batch=most)
    sp, gl = modelgen.synthetic_inputs(78, most, nn_x, nn_y, board_sizes=((nn_x, nn_y), (nn_x - 1, nn_y)))
    full = h.get_output(sp, gl)
    for n in (1, 85 // heads[0], 85 // heads[0] + 1, 128 // heads[0], 128 // heads[0] + 1):
        got = h.get_output(sp[:n], gl[:n])
        for k in full:
            assert np.array_equal(got[k], full[k][:n]), (n, k)
