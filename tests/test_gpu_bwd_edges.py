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
