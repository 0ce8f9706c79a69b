"""Backward of the SOFT window edge on each of its paths (initial-value rows up to four edge
keys, edge factors, one exp per element) against the float64 oracle, with sequence lengths
around the workgroups' 128 queries and 32-key tiles; tolerances as in test_gpu_bwd."""
import pytest
import torch

import dsalt._hip as hip
from test_gpu_bwd import run_case

pytestmark = pytest.mark.gpu


# (tau, edge): rows; rows without an edge key; fewer edge keys than the rows hold; the widest
# that takes rows; factors in both kernels; in dq only; in neither
@pytest.mark.parametrize("tau,edge", [(1.0, 4.0), (1.0, 0.0), (2.0, 0.5), (0.05, 4.0), (1.0, 4.5), (0.45, 6.0),
                                      (0.2, 6.0)])
@pytest.mark.parametrize("D", [64, 128])
def test_edge_paths(tau, edge, D):
    print(f"bwd edges tau={tau} edge={edge} D={D}", flush=True)
    run_case(hip.MODE_SOFT, [127, 1, 129, 31, 257, 33], 2, D, 9, seed=71, n_min=1, n_max=70, tau=tau, edge=edge)


# windows of one or two keys put P near 1 and gradients near 11, where bf16's rounding of P
# and dS alone (2^-9 of the sum) passes the absolute bar of 0.02: fp16 (2^-12) there
@pytest.mark.parametrize("n_min,n_max,dtype", [(1, 2, torch.float16), (3, 5, torch.float16), (500, 900, torch.float16),
                                               (500, 900, torch.bfloat16)])
@pytest.mark.parametrize("mode", [hip.MODE_HARD, hip.MODE_SOFT])
def test_window_extremes(mode, dtype, n_min, n_max):
    """Windows of a key or two (every band key is an edge key) and longer than the sequence."""
    print(f"bwd windows {mode} {dtype} {n_min}..{n_max}", flush=True)
    run_case(mode, [128, 96, 385], 2, 64, 5, seed=72, n_min=n_min, n_max=n_max, dtype=dtype)


# dq's workgroups: more than 64 sequences of a block each (the dispatch order of their blocks),
# and at head_dim 128 with edges wider than the rows hold the four waves that long sequences
# take (2 x 2048 tokens x 8 heads give every CU a workgroup), with both edge forms, against
# the two waves of the same batch with fewer heads
@pytest.mark.parametrize("mode,lens,H,D,tau,edge", [
    (hip.MODE_HARD, [64] * 66 + [1, 0, 63], 2, 64, 1.0, 4.0), (hip.MODE_SOFT, [33, 64, 31] * 23, 3, 128, 1.0, 4.0),
    (hip.MODE_SOFT, [64] * 65, 2, 128, 1.0, 8.0), (hip.MODE_SOFT, [2047, 2049], 8, 128, 1.0, 6.0),
    (hip.MODE_SOFT, [2047, 2049], 8, 128, 0.2, 6.0), (hip.MODE_SOFT, [2047, 2049], 1, 128, 1.0, 6.0)],
    ids=["hard-64s", "soft-short-d128", "soft-wide-64s", "four-waves", "four-waves-exact", "two-waves"])
def test_workgroup_shapes(mode, lens, H, D, tau, edge):
    print(f"bwd workgroups mode={mode} {len(lens)} x {lens[0]} H={H} D={D} tau={tau} edge={edge}", flush=True)
    run_case(mode, lens, H, D, 9, seed=73, n_min=1, n_max=60, tau=tau, edge=edge)
