"""Values past the f16 range are stored as infinities, and attention over them
is an infinity of their sign in that dim, as it is without splits: every merge
of split partials leaves the places that hold no split out, rather than adding
0 * inf.  Decode (one sequence, a ragged batch) and chunked prefill with split
keys, at every head size, against the fp64 ideal on the stored values."""
import ctypes

import numpy as np
import pytest

import emelk
import oracle
from kvsetup import Scenario, assert_close

pytestmark = pytest.mark.gpu

F16 = emelk.KV_F16


def _same(got, want, what):
    inf = np.isinf(want)
    assert inf.any() and not np.isnan(want).any()
    assert not np.isnan(got).any(), f"{what}: {np.isnan(got).sum()} NaN"
    np.testing.assert_array_equal(got[inf], want[inf], err_msg=what)
    assert_close(got[~inf], want[~inf], what=what)


def _scenario(D, n_kv, group, bt, lens):
    sc = Scenario(n_layer=1, n_head=n_kv * group, n_kv=n_kv, head_dim=D, block_tokens=bt,
                  lens=lens, kv_type=F16, seed=71, fill=False)
    for s, n in enumerate(lens):
        sc.v_rows[0][s][n // 9, 3] = 70000.0            # in the first splits
        sc.v_rows[0][s][n // 2, D - 1] = -70000.0       # another dim, another split
    sc.append_all()
    return sc


DECODE = [  # D, n_kv, group, page, lengths
    (64, 8, 4, 16, [1500]),
    (128, 8, 4, 32, [1000]),
    (128, 8, 2, 32, [900, 300, 40]),
    (128, 2, 4, 12, [2000]),
    (256, 1, 8, 32, [1200, 60]),
    (512, 1, 8, 16, [700]),
]


@pytest.mark.parametrize("case", DECODE, ids=[f"decode{i}" for i in range(len(DECODE))])
def test_decode_merge_of_infinities(device, case):
    D, n_kv, group, bt, lens = case
    print(f"\n[gpu-case] decode, infinite values {case}", flush=True)
    sc = _scenario(D, n_kv, group, bt, lens)
    assert emelk.decode_plan(sc.g, len(lens), max(lens))[1] > 1
    q = np.random.default_rng(72).standard_normal((len(lens), sc.n_head * D)).astype(np.float32)
    _same(sc.gpu_decode(0, q), sc.ideal_decode(0, q), f"decode {case}")


PREFILL = [  # D, n_kv, group, page, starts, rows
    (64, 4, 2, 32, [1500, 700], 5),
    (128, 8, 4, 32, [1900, 411], 6),
    (128, 1, 8, 12, [700], 33),
    (256, 1, 8, 32, [1000], 50),
    (512, 1, 8, 32, [640], 19),
]


@pytest.mark.parametrize("case", PREFILL, ids=[f"prefill{i}" for i in range(len(PREFILL))])
def test_prefill_merge_of_infinities(device, case):
    import torch
    D, n_kv, group, bt, starts, n_q = case
    print(f"\n[gpu-case] split prefill, infinite values {case}", flush=True)
    sc = _scenario(D, n_kv, group, bt, [s + n_q for s in starts])
    H = sc.n_head
    need = ctypes.c_uint64(0)
    assert emelk.lib.emelk_attn_prefill_workspace_size(
        ctypes.byref(sc.g), sc.n_seq, n_q, int(sc.tables.shape[1]),
        ctypes.byref(need)) == emelk.ERR_NONE and need.value > 0
    q = np.random.default_rng(73).standard_normal((sc.n_seq, n_q, H, D)).astype(np.float32)
    qd = torch.from_numpy(q).to(device)
    out = torch.full_like(qd, float("nan"))
    scale = 1.0 / np.sqrt(D)
    emelk.prefill_chunk(sc.g, sc.k_pool, sc.v_pool, 0, qd, out,
                        torch.tensor(starts, dtype=torch.int32, device=device), sc.tables, scale)
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    f16r = lambda x: oracle.fp16_to_fp32(oracle.fp32_to_fp16(x))  # noqa: E731
    for s, start in enumerate(starts):
        k, v = f16r(sc.k_rows[0][s]), f16r(sc.v_rows[0][s])
        for r in (0, n_q - 1):
            want = oracle.attention_f64(f16r(q[s, r].ravel()), k, v, H, n_kv, D, start + r + 1,
                                        scale)
            _same(got[s, r].ravel(), want, f"prefill {case} seq {s} row {r}")
