"""First-order calls by the sweeps that take them: the linear-domain sweeps take
temperatures from 0.2 on (and lengths of up to 2048 in all), the log-domain sweeps the
others.  The same problem in other units (scores, gaps and temperature times one factor)
has the same marginals, so a test states its case once and runs it through either."""
import ctypes

import torch

from _capi import check, lib

LOG_T = 0.19
SWEEPS = ("as stated", "log domain")


def in_units(sweeps, s, gaps, T):
    """(scores, gaps, temperature) of the case for these sweeps."""
    if sweeps == "as stated":
        return s, tuple(gaps), T
    k = LOG_T / T
    return s * k, tuple(g * k for g in gaps), LOG_T


def kernels_launched(fn):
    """The labels of the launches that fn makes."""
    lib().d2p_profile_reset()
    check(lib().d2p_profile_enable(1))
    try:
        fn()
        torch.cuda.synchronize()
    finally:
        check(lib().d2p_profile_enable(0))
    buf = ctypes.create_string_buffer(1 << 16)
    check(lib().d2p_profile_report(buf, len(buf)))
    return {line.split()[0] for line in buf.value.decode().splitlines()}


def assert_log_domain(fn):
    """fn's first-order calls run the log-domain sweeps: no launch that ends linear-domain
    ones."""
    names = kernels_launched(fn)
    assert names and not any(n.endswith("_redo") for n in names), names
