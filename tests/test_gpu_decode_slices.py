"""Decode where several waves of a workgroup walk one KV head in turn (token
slices) and the split count follows the lengths: lengths around one tile and
around one tile per wave, one long sequence among short ones, batches of more
than 64 sequences, few KV heads, every head size, with the step's token stored
in the same call, against the fp64 ideal on the stored values and the stored
bytes."""
import numpy as np
import pytest

import emelk
import oracle
from kvsetup import Scenario

pytestmark = pytest.mark.gpu

F16, Q8 = emelk.KV_F16, emelk.KV_Q8_0
CASES = [
    # D, n_kv, group, page, kv, lengths
    (128, 8, 2, 16, F16, [1]),
    (128, 8, 4, 32, F16, [16, 17, 127, 128, 129]),
    (128, 1, 8, 16, Q8, [2050]),
    (128, 2, 4, 12, F16, [333, 1]),                        # pages that split a wave tile
    (64, 8, 4, 16, F16, [4097] + [3] * 15),                # one long among 16, then 17 and 33
    (64, 8, 1, 16, Q8, [3000, 1] + [40] * 15),
    (64, 8, 2, 16, F16, [5000] + list(range(1, 33))),
    (64, 6, 2, 16, F16, [700, 90]),                        # 6 KV heads: two per workgroup at most
    (256, 1, 8, 32, F16, [4000]),
    (256, 2, 4, 16, Q8, [8, 9, 65, 64, 1100]),
    (512, 1, 8, 16, F16, [1300, 5]),
    (512, 1, 2, 32, Q8, [900, 33, 1]),
    # two sequences per lane in the plan, and the batches on either side
    (64, 8, 1, 16, F16, [70] * 64),
    (64, 8, 2, 16, F16, [3000] + [2 + i for i in range(64)]),
    (64, 8, 1, 16, Q8, [9] * 80 + [1500] + [130] * 19),
    (128, 1, 8, 32, F16, [40 + 7 * i for i in range(126)] + [2500]),
    (256, 2, 4, 16, Q8, [1] * 90 + [700, 3]),
    (64, 16, 2, 16, F16, [300] * 70),                     # more splits than run at once
    (64, 8, 1, 16, F16, [60] * 127 + [2000]),             # 128: the host plan
]


@pytest.mark.parametrize("case", CASES, ids=[f"slices{i}" for i in range(len(CASES))])
def test_decode_slices(device, case):
    import torch
    D, n_kv, group, bt, kv, lens = case
    H = n_kv * group
    print(f"\n[gpu-case] decode slices {case}", flush=True)
    sc = Scenario(n_layer=1, n_head=H, n_kv=n_kv, head_dim=D, block_tokens=bt, lens=lens,
                  kv_type=kv, seed=41, outlier_frac=0.01 if kv == Q8 else 0.0)
    n = len(lens)
    q = np.random.default_rng(42).standard_normal((n, H * D)).astype(np.float32)
    # the last token of every sequence is stored again by the call under test
    want_k, want_v = sc.k_pool.clone(), sc.v_pool.clone()
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(device)  # noqa: E731
    k = dev(np.stack([sc.k_rows[0][s][m - 1] for s, m in enumerate(lens)]))
    v = dev(np.stack([sc.v_rows[0][s][m - 1] for s, m in enumerate(lens)]))
    pos = torch.tensor([m - 1 for m in lens], dtype=torch.int32, device=device)
    zero = torch.zeros((n, 1, n_kv * D), device=device)
    emelk.append(sc.g, sc.k_pool, sc.v_pool, 0, zero, zero, pos, sc.tables)
    assert not torch.equal(sc.k_pool, want_k)
    out = torch.full((n, H, D), float("nan"), device=device)
    ws = torch.full((emelk.decode_workspace_bytes(sc.g, n, max(lens)) // 4,), float("nan"),
                    device=device)
    emelk.decode_append(sc.g, sc.k_pool, sc.v_pool, 0, k, v, dev(q).view(n, H, D), out,
                        torch.tensor(lens, dtype=torch.int32, device=device), max(lens), sc.tables,
                        1.0 / np.sqrt(D), ws)
    torch.cuda.synchronize()
    assert torch.equal(sc.k_pool, want_k) and torch.equal(sc.v_pool, want_v)
    got = out.view(n, -1).cpu().numpy()
    ideal = sc.ideal_decode(0, q)
    # Per output, relative to sum p |v|: f16 pools round each probability to
    # fp16 (2^-11), and 2^-13 covers the 32-bit scores and sums.  q8_0 pools
    # keep the weights to 2^-22, but add bytes biased by 1152 in 32 bits.  Scores:
    # a 16-dim chunk's sum starts at 1152 sum|q| (about 15000), rounds at 2^-24
    # of that four times, and the outlier blocks' scale (0.5) and the softmax
    # scale (1/8) carry 4 * 6e-5 of it into the exponent, doubled by chunks of
    # like sign: 2^-11.  Values: sum p d (v + 1152) rounds at 2^-24 of 1152 sum
    # p d, taken 64 times (a wave adds at most 3000 / (8 waves * 4 tokens) times
    # two weights, roundings of either sign).
    bound = 2.0 ** -11 + 2.0 ** -13
    bias = 64 * 1152 * 2.0 ** -24 if kv == Q8 else 0.0
    stored = ((lambda r: oracle.dequantize_q8_0(oracle.quantize_q8_0(r))) if kv == Q8 else
              (lambda r: oracle.fp16_to_fp32(oracle.fp32_to_fp16(r))))

    def scales(rows):  # each value's block scale
        d = oracle.fp16_to_fp32(oracle.quantize_q8_0(rows)["d"])
        return np.repeat(d.reshape(rows.shape[0], -1), 32, axis=1)

    qr = oracle.fp16_to_fp32(oracle.fp32_to_fp16(q))
    for s, m in enumerate(lens):
        k64, v64 = stored(sc.k_rows[0][s]), stored(sc.v_rows[0][s])
        limit = bound * np.asarray(oracle.attention_f64(qr[s], k64, np.abs(v64), H, n_kv, D, m,
                                                        1.0 / np.sqrt(D))) + 1e-6
        if kv == Q8:
            limit += bias * np.asarray(oracle.attention_f64(
                qr[s], k64, np.ascontiguousarray(scales(sc.v_rows[0][s])), H, n_kv, D, m,
                1.0 / np.sqrt(D)))
        err = np.abs(got[s] - ideal[s]) / limit
        assert err.max() <= 1.0, f"seq {s} of {m}: {err.max():.2f} of the bound"
