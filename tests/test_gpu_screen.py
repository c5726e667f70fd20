"""First-pass screen of the peeler without energies from the assembler: which bins it stamps, at the edges of
its row counts (64, 128, 256 rows per column) and of its column groups."""
import ctypes

import numpy as np
import pytest
import torch

from qsft_amd import _lib as L
from qsft_amd import device as dv
from qsft_amd import kernels as K

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("P", [2, 63, 64, 65, 127, 128, 129, 193, 256])
@pytest.mark.parametrize("q,b,C", [(4, 3, 1), (3, 3, 2), (2, 1, 3), (3, 4, 1)])
def test_screen_stamps_the_bins_above_the_cutoff(P, q, b, C):
    print(f"screen P={P} q={q} b={b} C={C}", flush=True)
    rng = np.random.default_rng(P + q)
    n, Q, cutoff = P - 1, q ** b, 0.25
    dev, n_pad = dv.current_device(), dv.n_pad_of(P - 1)
    # energy per row well below or above the cutoff: in one row of the column (any row, the last
    # included), in all of them, or too little of it
    U = np.zeros((C * Q, P), complex)
    kind = rng.integers(0, 4, size=C * Q)
    for t in range(C * Q):
        if kind[t] == 1:
            U[t, rng.choice([0, P - 1, rng.integers(P)])] = 2 * np.sqrt(cutoff * P)
        elif kind[t] == 2:
            U[t] = 2 * np.sqrt(cutoff) * np.exp(2j * np.pi * rng.uniform(size=P))
        elif kind[t] == 3:
            U[t] = np.sqrt(cutoff) / 2 * np.exp(2j * np.pi * rng.uniform(size=P))
    D = np.zeros((C, P, n_pad), np.int8)
    D[:, :, :n] = np.eye(P, n, -1, dtype=np.int8)
    Mt = torch.from_numpy(rng.integers(0, q, size=(C, b, n_pad)).astype(np.int8)).to(dev)
    batch = K.PeelBatch([dict(q=q, n=n, b=b, C=C, P=P, p1=P, method=L.QSFT_DETECT_NSO1, cutoff=cutoff, Mt=Mt,
                              D=torch.from_numpy(D).to(dev),
                              U=torch.from_numpy(U.reshape(C, Q, P)).to(dev))])
    vp = ctypes.c_void_p
    L.check(L.lib.qsft_peel_init(vp(batch.dptr), vp(batch.pre_b), vp(batch.pre_s), 1, batch.tot_b, batch.tot_s,
                                 K.stream_handle()), "qsft_peel_init")
    at = batch.descs[0].mark - batch.ws[0].data_ptr()
    mark = batch.ws[0][at:at + 4 * C * Q].view(torch.int32).cpu().numpy()
    np.testing.assert_array_equal(mark, np.where((kind == 1) | (kind == 2), 0, -1))
