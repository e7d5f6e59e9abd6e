"""Chunked prefill with the keys split over workgroups (calls with fewer query
tiles than compute units), against the fp64 ideal on the rounded inputs and
against the unsplit entry point: every head size, contexts around the smallest
one that splits, ragged sequences of which some split and some do not, empty
and negative starts, chunks that end inside a row block, pages that do and do
not hold a whole 32-key sub-tile, an invalid page, and workspaces that hold
fewer splits than the call would take."""
import ctypes

import numpy as np
import pytest

import emelk
import oracle
from kvsetup import Scenario

pytestmark = pytest.mark.gpu

F16, Q8 = emelk.KV_F16, emelk.KV_Q8_0
CASES = [
    # D, n_kv, group, page, kv, starts, n_q, invalid page of sequence 0
    (128, 8, 4, 32, F16, [1900, 411, 0], 6, -1),
    (128, 2, 1, 16, F16, [441, 442, 505, 506], 7, -1),      # 7, 8 and 9 key tiles
    (128, 1, 8, 12, F16, [700], 33, -1),
    (128, 2, 2, 64, Q8, [900, 60], 40, -1),
    (64, 2, 4, 32, F16, [1200, -5, 300], 5, -1),
    (64, 1, 1, 16, Q8, [2000], 3, -1),
    (64, 4, 2, 32, F16, [1500, 700], 70, 9),
    (256, 1, 8, 32, F16, [1000], 50, -1),
    (256, 2, 2, 16, Q8, [300, 513], 17, -1),
    (512, 1, 8, 32, F16, [640, 100], 19, -1),
    (512, 1, 2, 8, F16, [500], 33, 20),
]


def _size(g, n_seq, n_q, stride):
    out = ctypes.c_uint64(0)
    assert emelk.lib.emelk_attn_prefill_workspace_size(ctypes.byref(g), n_seq, n_q, stride,
                                                       ctypes.byref(out)) == emelk.ERR_NONE
    return out.value


@pytest.mark.parametrize("case", CASES, ids=[f"split{i}" for i in range(len(CASES))])
def test_split_prefill(device, case):
    import torch
    D, n_kv, group, bt, kv, starts, n_q, bad = case
    n_head = n_kv * group
    print(f"\n[gpu-case] split prefill {case}", flush=True)
    sc = Scenario(n_layer=1, n_head=n_head, n_kv=n_kv, head_dim=D, block_tokens=bt,
                  lens=[max(s, 0) + n_q for s in starts], seed=D + n_q, kv_type=kv,
                  outlier_frac=0.01 if kv == Q8 else 0.0)
    t = sc.tables_host.copy()
    if bad >= 0:
        t[0, bad] = 0xFFFF
    tables = torch.from_numpy(np.ascontiguousarray(t).view(np.int16)).to(device)
    q = np.random.default_rng(1).standard_normal((sc.n_seq, n_q, n_head, D)).astype(np.float32)
    qd = torch.from_numpy(q).to(device)
    qs = torch.tensor(starts, dtype=torch.int32, device=device)
    scale = 1.0 / np.sqrt(D)
    stride = int(tables.shape[1])
    need = _size(sc.g, sc.n_seq, n_q, stride)
    rows = sc.n_seq * n_q * n_head * (D + 2) * 4
    assert need >= 2 * rows and need % rows == 0

    def call(ws_bytes):
        ws = torch.full((max(ws_bytes // 4, 1),), float("nan"), device=device)
        out = torch.full_like(qd, float("nan"))
        p = lambda x: ctypes.c_void_p(x.data_ptr())  # noqa: E731
        e = emelk.lib.emelk_attn_prefill_chunk_ws(
            ctypes.byref(sc.g), p(sc.k_pool), p(sc.v_pool), 0, p(qd), p(out), sc.n_seq, n_q,
            p(qs), p(tables), stride, scale, p(ws) if ws_bytes else None, ws_bytes,
            ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
        assert e == emelk.ERR_NONE
        torch.cuda.synchronize()
        return out.cpu().numpy()

    whole, split, two = call(0), call(need), call(2 * rows + rows // 2)
    assert np.array_equal(whole, call(rows)), "a workspace of one split runs unsplit"
    assert np.array_equal(split, call(need)), "deterministic"
    out = torch.full_like(qd, float("nan"))
    emelk.prefill_chunk(sc.g, sc.k_pool, sc.v_pool, 0, qd, out, qs, tables, scale)
    assert np.array_equal(split, out.cpu().numpy()), "the binding runs the split plan"

    stored = ((lambda r: oracle.dequantize_q8_0(oracle.quantize_q8_0(r))) if kv == Q8 else
              (lambda r: oracle.fp16_to_fp32(oracle.fp32_to_fp16(r))))
    # f16 pools round each probability to fp16 (2^-11 of sum p |v| at most; q8_0
    # pools carry it to 2^-22); 2^-13 covers the 32-bit scores and sums of both
    bound = (2.0 ** -11 if kv == F16 else 0.0) + 2.0 ** -13
    for s, start in enumerate(starts):
        if start < 0:
            assert not whole[s].any() and not split[s].any() and not two[s].any()
            continue
        kf, vf = stored(sc.k_rows[0][s]), stored(sc.v_rows[0][s])
        for r in sorted({0, n_q // 2, n_q - 1}):
            limit = start + r + 1
            keep = np.array([t[s, p // bt] != 0xFFFF for p in range(limit)])
            qr = oracle.fp16_to_fp32(oracle.fp32_to_fp16(q[s, r].ravel()))
            kk, vv, n = kf[:limit][keep], vf[:limit][keep], int(keep.sum())
            ideal = np.asarray(oracle.attention_f64(qr, kk, vv, n_head, n_kv, D, n, scale))
            mag = np.asarray(oracle.attention_f64(qr, kk, np.abs(vv), n_head, n_kv, D, n, scale))
            for name, got in (("unsplit", whole), ("split", split), ("two splits", two)):
                err = np.abs(got[s, r].ravel() - ideal)
                assert (err <= bound * mag + 1e-6).all(), \
                    f"{name}: seq {s} row {r}: {(err / (bound * mag + 1e-6)).max():.2f} of the bound"


def test_which_calls_split(device):
    g = emelk.geometry(1, 32, 8, 128, 32, 4096)
    assert _size(g, 1, 4, 8) == 0           # 256 keys: a few tiles, one workgroup per head group
    assert _size(g, 1, 4, 64) > 0
    assert _size(g, 1, 512, 16) == 0        # the prompt's first 512 rows: partials cost more
    assert _size(g, 1, 512, 80) > 0
    assert _size(g, 8, 512, 144) == 0       # two full rounds of workgroups
    assert _size(g, 3, 337, 4096) <= 64 << 20
