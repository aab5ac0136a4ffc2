"""Low-latency mode (hipLowLatency / kgh_handle_set_low_latency): 3x3
convolutions whose sums are cut into up to eight splits, for handles of at
most 16 rows. Checked against the CPU oracle at the fp16 whole-net tolerances
(the summation order differs from the default kernels, so these rows are not
bitwise equal to a default handle's), against recorded bits, and for
batch-size independence within the mode."""
import ctypes
import os

import numpy as np
import pytest

from katago_amd import modelgen, nn
from oracle import oracle
from conftest import GOLDEN
from golden import make_low_latency_golden as recorded
from test_gpu_parity import _compare

pytestmark = pytest.mark.gpu


def _handle(lm, n, low_latency=True):
    ctx = nn.ComputeContext(lm, 19, 19, use_fp16=True, low_latency=low_latency)
    return ctx, nn.ComputeHandle(ctx, max_batch=n)


@pytest.mark.parametrize("n,board_sizes,cfg_idx", [
    (1, (19,), 2),
    (4, (19,), 2),
    (8, (9, 13, 19), 3),
    (16, (19, 9), 3),
], ids=["c2-b1", "c2-b4", "c3-b8-mixed", "c3-b16-mixed"])
def test_low_latency_matches_oracle(model_dir, n, board_sizes, cfg_idx):
    cfg = modelgen.configs()[cfg_idx]
    path = modelgen.ensure_model(model_dir, cfg)
    om = oracle.OracleModel(path, 19, 19)
    lm = nn.LoadedModel(path)
    ctx, h = _handle(lm, n)
    sp, gl = modelgen.synthetic_inputs(cfg.input_seed + n, n, board_sizes=board_sizes)
    sym = np.arange(n) % 8
    opt = (np.arange(n) % 3) / 2.0
    gpu = h.get_output(sp, gl, sym, opt)
    ora = om.forward(sp, gl, sym, opt)
    _compare(gpu, ora, True, lm.info.output_scale_multiplier, board_sizes, n, f"low-latency C{cfg_idx} n={n}")
    for k in gpu:
        assert np.isfinite(gpu[k]).all(), k


def test_low_latency_rows_do_not_depend_on_batch(model_dir):
    """Within the mode every call adds the same splits in the same order, so a
    row's outputs are bitwise the same at batch 1 and inside a batch of 12; the mode
    is deterministic (a repeat gives the same bits)."""
    cfg = modelgen.configs()[3]
    lm = nn.LoadedModel(modelgen.ensure_model(model_dir, cfg))
    ctx, h = _handle(lm, 12)
    sp, gl = modelgen.synthetic_inputs(cfg.input_seed, 12, board_sizes=(9, 13, 19))
    full = h.get_output(sp, gl)
    again = h.get_output(sp, gl)
    for k in full:
        assert np.array_equal(full[k], again[k]), k
    for r in (0, 5, 11):
        one = h.get_output(sp[r:r + 1], gl[r:r + 1])
        for k in full:
            assert np.array_equal(full[k][r], one[k][0]), (r, k)


def test_low_latency_close_to_default_kernels(model_dir):
    """The splits' sums differ from the default kernels only by fp32 rounding
    order: the outputs agree far inside the fp16 tolerances, but are not the
    same bits."""
    cfg = modelgen.configs()[2]
    lm = nn.LoadedModel(modelgen.ensure_model(model_dir, cfg))
    sp, gl = modelgen.synthetic_inputs(cfg.input_seed, 4)
    _, fast = _handle(lm, 4, True)
    _, dflt = _handle(lm, 4, False)
    a = fast.get_output(sp, gl)
    b = dflt.get_output(sp, gl)
    for k in a:
        d = np.abs(a[k] - b[k]).max()
        assert d <= 5e-3, (k, d)
    assert not np.array_equal(a["policy"], b["policy"])


@pytest.mark.parametrize("arch", recorded.NETS, ids=lambda a: a.name)
def test_low_latency_gives_the_recorded_bits(model_dir, arch):
    """A row is rounded as it always was in this mode, whichever kernels add
    the splits: in registers up to 704 channels, split-K workgroups above; at
    a batch of two and, on the 64-row tiles, of 16."""
    lm = nn.LoadedModel(recorded.model_file(model_dir, arch))
    want = np.load(os.path.join(GOLDEN, "low_latency.npz"))
    ctx = nn.ComputeContext(lm, 19, 19, use_fp16=True, low_latency=True)
    rows = recorded.inputs()
    for n in (2, 16):
        got = nn.ComputeHandle(ctx, max_batch=n).get_output(*(np.concatenate([r] * (n // 2)) for r in rows))
        for k in got:
            assert np.array_equal(got[k][:2], want[f"{arch.name}/{k}"]) and np.array_equal(got[k][-2:], got[k][:2]), (n, k)

    dm = nn.DeviceModel(lm, use_fp16=True)
    h = nn.DeviceHandle(dm, 2)
    h.set_low_latency(True)
    h.set_profiling(True)
    dev = [nn.DeviceBuffer.from_array(r) for r in rows]
    out = nn.DeviceBuffer(2 * h.row_floats * 4)
    h.forward_device(2, *(b.ptr for b in dev), out.ptr)
    h.synchronize()
    kernels = " ".join(r[4] for r in h.profile_kernels() if r[0] == 0)
    assert ("split-K" if arch.mid_c > 704 else "partial sums") in kernels, kernels
    dm.close()


def test_low_latency_device_handle_limits(model_dir):
    """kgh_handle_set_low_latency on a device handle: accepted up to 16 rows,
    refused above with a message, and it can be switched off again."""
    cfg = modelgen.configs()[2]
    lm = nn.LoadedModel(modelgen.ensure_model(model_dir, cfg))
    dm = nn.DeviceModel(lm, use_fp16=True)
    big = nn.DeviceHandle(dm, max_batch=17)
    with pytest.raises(nn.StringError, match="low-latency"):
        big.set_low_latency(True)
    big.close()
    h = nn.DeviceHandle(dm, max_batch=2)
    h.set_low_latency(True)
    h.set_low_latency(False)
    h.close()
    dm.close()


@pytest.mark.parametrize("arch,allocates", [(recorded.NETS[2], False), (recorded.NETS[6], True)], ids=["c384-192", "c768"])
def test_partial_sum_buffer_only_for_nets_that_use_it(model_dir, arch, allocates):
    """Enabling the mode allocates the split-K partial sums (8 * 16 * 361 *
    channels floats: 142 MB at 768 channels) only where a conv is too wide to
    add them in registers."""
    hip = nn.hip_library()  # its handle finds the runtime it is linked with

    def free():
        now, total = ctypes.c_size_t(), ctypes.c_size_t()
        assert hip.hipMemGetInfo(ctypes.byref(now), ctypes.byref(total)) == 0
        return now.value

    dm = nn.DeviceModel(nn.LoadedModel(recorded.model_file(model_dir, arch)), use_fp16=True)
    h = nn.DeviceHandle(dm, 16)
    h.synchronize()
    before = free()
    h.set_low_latency(True)
    assert (before - free() > 30e6) == allocates
    dm.close()
