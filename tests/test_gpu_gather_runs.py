"""Gather at the edges of its runs: every head size, lengths at, under and over
a run's end, zeros past a length and on an invalid page, outputs that end
inside a run, pages that split runs, and outputs 2 bytes off a word."""
import numpy as np
import pytest

import emelk
import oracle
from kvsetup import Scenario

pytestmark = pytest.mark.gpu

CASES = [  # D, n_kv, page, kv, lengths, out_tokens, invalid page of sequence 0, byte offset
    (64, 3, 16, emelk.KV_Q8_0, [64, 1, 130], 131, -1, 0),
    (64, 2, 12, emelk.KV_F16, [33, 31, 64], 70, -1, 0),
    (128, 8, 32, emelk.KV_Q8_0, [33, 95, 32], 97, 0, 2),
    (128, 1, 16, emelk.KV_F16, [100], 65, 2, 0),
    (256, 1, 16, emelk.KV_Q8_0, [17, 15], 16, -1, 2),
    (256, 2, 32, emelk.KV_F16, [40, 5], 40, -1, 0),
    (512, 2, 8, emelk.KV_Q8_0, [9, 30], 31, 1, 0),
    (512, 1, 16, emelk.KV_F16, [7, 50], 51, -1, 0),
]


@pytest.mark.parametrize("case", CASES, ids=[f"gather{i}" for i in range(len(CASES))])
def test_gather_runs(device, case):
    import torch
    D, n_kv, bt, kv, lens, n_out, bad, off = case
    print(f"\n[gpu-case] gather runs {case}", flush=True)
    sc = Scenario(n_layer=2, n_head=n_kv, n_kv=n_kv, head_dim=D, block_tokens=bt, lens=lens,
                  kv_type=kv, seed=61)
    t = sc.tables_host.copy()
    if bad >= 0:
        t[0, bad] = 0xFFFF
    tables = torch.from_numpy(np.ascontiguousarray(t).view(np.int16)).to(device)
    row = D * 2 if kv == emelk.KV_F16 else D // 32 * 34
    size = len(lens) * n_kv * n_out * row
    buf = [torch.full((size + 64,), 0xAB, dtype=torch.uint8, device=device) for _ in range(2)]
    emelk.gather(sc.g, sc.k_pool, sc.v_pool, 1, torch.tensor(lens, dtype=torch.int32, device=device),
                 tables, buf[0][off:off + size], buf[1][off:off + size], n_out)
    torch.cuda.synchronize()
    for which, rows in ((0, sc.k_rows[1]), (1, sc.v_rows[1])):
        host = buf[which].cpu().numpy()
        assert (host[:off] == 0xAB).all() and (host[off + size:] == 0xAB).all()
        got = host[off:off + size].reshape(len(lens), n_kv, n_out, row)
        for s, n in enumerate(lens):
            stored = (oracle.fp32_to_fp16(rows[s]).view(np.uint8) if kv == emelk.KV_F16 else
                      oracle.quantize_q8_0(rows[s]).view(np.uint8)).reshape(n, n_kv, row)
            want = np.zeros((n_kv, n_out, row), np.uint8)
            m = min(n, n_out)
            want[:, :m] = stored[:m].transpose(1, 0, 2)
            for p in range(m):
                if t[s, p // bt] == 0xFFFF:
                    want[:, p] = 0
            np.testing.assert_array_equal(got[s], want, err_msg=f"pool {which} seq {s}")
