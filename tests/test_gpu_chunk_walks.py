"""The wavefront walks over a chunk against the oracle, at the sizes where they turn over: BDA maps of
baselines of 1, 63..65 and 129 rows and of 1..130 channels (64 rows and 64 channels are one turn of the
walk), and the flag selections of 1..130 channels and up to more antennas than a block can sum in LDS.
Maps, flags and fractions are whole numbers and their quotients: equal word for word."""
import numpy as np
import pytest
import torch

from ddfacet_amd import bda, chunk
from oracle import bda as obda
from oracle import chunk as ochunk

pytestmark = pytest.mark.gpu


def _rows_of(counts, na, seed):
    """Baseline (p, q) number k of the upper triangle has counts[k % len(counts)] rows, shuffled."""
    rng = np.random.default_rng(seed)
    pairs = [(p, q) for p in range(na) for q in range(p + 1, na)]
    a0, a1, uvw = [], [], []
    for k, (p, q) in enumerate(pairs):
        n = counts[k % len(counts)]
        t = np.arange(n)
        b = rng.uniform(30, 4000)
        ha = 2 * np.pi / 86400 * 8.0 * t + rng.uniform(0, 6)
        uvw.append(np.stack([b * np.cos(ha), b * np.sin(ha), 0.1 * b * np.cos(ha + 1)], 1))
        a0 += [p] * n
        a1 += [q] * n
    a0, a1, uvw = np.array(a0, np.int32), np.array(a1, np.int32), np.concatenate(uvw)
    at = np.argsort(rng.random(a0.size), kind="stable")
    return np.ascontiguousarray(uvw[at]), a0[at], a1[at]


@pytest.mark.parametrize("mode", [1, 2])
@pytest.mark.parametrize("nchan", [1, 2, 63, 64, 65, 130])
@pytest.mark.parametrize("decorr", [0.0005, 0.02, 0.5])
def test_map_turns(mode, nchan, decorr):
    uvw, a0, a1 = _rows_of((1, 2, 63, 64, 65, 129, 200), 7, nchan)
    freqs = np.linspace(1.2e9, 1.3e9, nchan) if nchan > 1 else np.array([1.25e9])
    dfreq = freqs[1] - freqs[0] if nchan > 1 else 1e6
    chan_map = (np.arange(nchan) * 3 // nchan).astype(np.int32)
    cell = 1.5 * np.pi / 180 / 3600
    host = (obda.bda_map_mode1 if mode == 1 else obda.bda_map_mode2)(uvw, a0, a1, freqs, dfreq, decorr, cell, 455,
                                                                    chan_map)
    dev = bda.bda_map_device(uvw, a0, a1, freqs, dfreq, decorr, cell, 455, chan_map, mode=mode).cpu().numpy()
    np.testing.assert_array_equal(dev, host)


@pytest.mark.parametrize("na,nrow,nchan,ncorr", [(2, 1, 1, 1), (5, 255, 1, 4), (5, 257, 2, 2), (7, 1000, 3, 1),
                                                 (7, 1000, 63, 2), (64, 4097, 64, 4), (9, 333, 65, 4), (9, 100, 130, 1),
                                                 (4096, 3000, 5, 4), (4097, 3000, 5, 4)])
def test_selection_turns(na, nrow, nchan, ncorr):
    rng = np.random.default_rng(na + nchan)
    a0, a1 = (rng.integers(0, na, nrow).astype(np.int32) for _ in range(2))
    uvw = rng.normal(0, 2000, (nrow, 3))
    # the same on every correlation, as the flag preparation leaves them
    flags = np.repeat(rng.random((nrow, nchan, 1)) < 0.1, ncorr, axis=2)
    flags[(a0 == 1) | (a1 == 1)] = True
    data = np.ones((nrow, nchan, ncorr), np.complex64)
    f_ref, d_ref = flags.copy(), data.copy()
    frac_ref = ochunk.update_flags(f_ref, uvw, d_ref, a0, a1, na, uv_range_km=(0.5, 3.0), named_antennas=(0,))
    d = lambda x: torch.from_numpy(np.ascontiguousarray(x)).cuda()  # noqa: E731
    tf, td = d(flags.view(np.uint8)), d(data)
    frac, _ = chunk.update_flags(tf, d(uvw), td, d(a0), d(a1), uv_range_km=(0.5, 3.0), named_antennas=(0,), na=na)
    np.testing.assert_array_equal(frac.cpu().numpy(), frac_ref)
    np.testing.assert_array_equal(tf.cpu().numpy().view(bool), f_ref)
    np.testing.assert_array_equal(td.cpu().numpy(), d_ref)
