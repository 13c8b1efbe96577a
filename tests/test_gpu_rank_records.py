"""Which SVDs the learned rank form records (needs a GPU): all whose matrix has
more than 96 columns or takes more than 159 KiB with 64 bytes a column, by the
log of the SVDs themselves. Whatever else one workgroup may hold, a bond's
history begins there."""

import gc

import numpy as np
import pytest

import oqupy_amd as oqupy

from tests import models

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("predictor", [None, "previous", "adaptive"])
def test_records_begin_at_96_columns(predictor, tmp_path, monkeypatch):
    print(f"[gpu-case] rank records {predictor}", flush=True)
    log = tmp_path / "svd.csv"
    monkeypatch.setenv("PTE_SVD_TRACE", str(log))
    _, bath, params = models.spin_boson(0.7, 4.0, 0.1, 0.05, 20, 1e-7)
    config = {"rank_trace": 200000, "chi_cap": 4096}
    if predictor:
        config["rank_predictor"] = predictor
    ptt = oqupy.PtTempo(bath, 0.0, 26 * 0.05 + 1e-9, params, backend_config=config)
    ptt.compute()
    records = ptt.backend.rank_trace()
    del ptt
    gc.collect()            # the log is complete when the engine is gone
    m, n = np.loadtxt(log, delimiter=",", usecols=(0, 1)).T
    beyond = (n > 96) | (16 * m * n + 64 * n > 159 * 1024)
    one_workgroup = beyond & (n <= 126) & (m <= 152)
    assert one_workgroup.any()
    assert len(records) == beyond.sum()
