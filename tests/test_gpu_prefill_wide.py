"""Chunked prefill through block tables much wider than the sequences.  The
table's width bounds the split plan, the device knows the lengths: a sequence
too short for the planned splits to pay is computed as without splits, bit for
bit, also beside a long one that does split.  With max_kv_len the binding plans
for that length."""
import ctypes

import numpy as np
import pytest

import emelk
import oracle
from kvsetup import Scenario, assert_close

pytestmark = pytest.mark.gpu

F16, Q8 = emelk.KV_F16, emelk.KV_Q8_0
WIDE = 1000  # pages of a table row
CASES = [
    # D, n_kv, group, kv, starts, rows, which sequences split
    (128, 8, 4, F16, [176] * 8, 64, []),
    (128, 8, 4, Q8, [176] * 8, 64, []),
    (128, 8, 4, F16, [176] * 6 + [3000, 0], 64, [6]),
    (64, 8, 4, F16, [176, 60, 180, 190, 2500, -4, 176, 176], 64, [4]),
    (256, 1, 8, F16, [60] * 7 + [1500], 64, [7]),
    (512, 1, 8, F16, [60] * 6 + [700, 20], 64, [6]),
]


def _setup(device, D, n_kv, group, kv, starts, n_q):
    import torch
    sc = Scenario(n_layer=1, n_head=n_kv * group, n_kv=n_kv, head_dim=D, block_tokens=32,
                  lens=[max(s, 0) + n_q for s in starts], kv_type=kv, seed=81)
    wide = np.full((sc.n_seq, WIDE), 0xFFFF, np.uint16)
    wide[:, :sc.tables_host.shape[1]] = sc.tables_host
    wide = torch.from_numpy(wide.view(np.int16)).to(device)
    q = np.random.default_rng(82).standard_normal((sc.n_seq, n_q, sc.n_head, D)).astype(np.float32)
    qd = torch.from_numpy(q).to(device)
    start = torch.tensor(starts, dtype=torch.int32, device=device)

    def call(entry, **kw):
        out = torch.full_like(qd, float("nan"))
        entry(out, **kw)
        torch.cuda.synchronize()
        return out.cpu().numpy()

    def unsplit(out):
        assert emelk.lib.emelk_attn_prefill_chunk(
            ctypes.byref(sc.g), sc.k_pool.data_ptr(), sc.v_pool.data_ptr(), 0, qd.data_ptr(),
            out.data_ptr(), sc.n_seq, n_q, start.data_ptr(), wide.data_ptr(), WIDE,
            1.0 / np.sqrt(D), torch.cuda.current_stream().cuda_stream) == emelk.ERR_NONE

    def chunk(out, **kw):
        emelk.prefill_chunk(sc.g, sc.k_pool, sc.v_pool, 0, qd, out, start, wide, 1.0 / np.sqrt(D),
                            **kw)

    return sc, q, call, unsplit, chunk


@pytest.mark.parametrize("case", CASES, ids=[f"wide{i}" for i in range(len(CASES))])
def test_short_sequences_stay_whole(device, case):
    D, n_kv, group, kv, starts, n_q, split = case
    print(f"\n[gpu-case] prefill through a wide table {case}", flush=True)
    sc, q, call, unsplit, chunk = _setup(device, D, n_kv, group, kv, starts, n_q)
    need = ctypes.c_uint64(0)
    assert emelk.lib.emelk_attn_prefill_workspace_size(
        ctypes.byref(sc.g), sc.n_seq, n_q, WIDE, ctypes.byref(need)) == emelk.ERR_NONE
    assert need.value > 0
    whole, got = call(unsplit), call(chunk)
    r16 = lambda x: oracle.fp16_to_fp32(oracle.fp32_to_fp16(x))  # noqa: E731
    for s, start in enumerate(starts):
        if s not in split:
            np.testing.assert_array_equal(got[s], whole[s], err_msg=f"seq {s}")
            continue
        assert not np.array_equal(got[s], whole[s]), f"seq {s} of {start} tokens did not split"
        k, v = r16(sc.k_rows[0][s]), r16(sc.v_rows[0][s])
        for r in (0, n_q - 1):
            want = oracle.attention_f64(r16(q[s, r].ravel()), k, v, sc.n_head, n_kv, D,
                                        start + r + 1, 1.0 / np.sqrt(D))
            assert_close(got[s, r].ravel(), want, what=f"seq {s} row {r}")


def test_max_kv_len_plans_for_the_length(device):
    """512 rows of an empty sequence run unsplit when the caller says how long
    it is; a longer claim, or one past the table, changes the plan alone."""
    print("\n[gpu-case] prefill with max_kv_len", flush=True)
    sc, q, call, unsplit, chunk = _setup(device, 128, 8, 4, F16, [0], 512)
    stride = []
    size = emelk._prefill_workspace
    try:
        emelk._prefill_workspace = lambda g, n, r, w, s: stride.append(w) or size(g, n, r, w, s)
        whole = call(unsplit)
        for kv_len, pages in ((512, 16), (513, 17), (0, 1), (10 ** 6, WIDE), (None, WIDE)):
            assert_close(call(chunk, max_kv_len=kv_len), whole, what=f"max_kv_len {kv_len}")
            assert stride.pop() == pages
        np.testing.assert_array_equal(call(chunk, max_kv_len=512), whole)
    finally:
        emelk._prefill_workspace = size
