"""Norm + RoPE + append at the edges of the kernel's launch shapes, bit-exact
against the oracle: every row-slot count that a launch of each head size takes
(by its token count), row counts that leave a wave partly filled, adjacent,
halved and partial pairings, a norm on q or on k alone, v norm with several v
heads per wave, and rows and weights that lie 4 bytes off any wider boundary."""
import numpy as np
import pytest

import emelk
import oracle
from kvsetup import Scenario

pytestmark = pytest.mark.gpu

ADJ, HALF = emelk.NORMAL_PAIRING, emelk.NEOX_PAIRING
F16, Q8 = emelk.KV_F16, emelk.KV_Q8_0
CASES = [
    # kv, n_head, n_kv, D, page, pairing, n_rot, norms, v_rms, sequences, tokens
    (F16, 16, 8, 128, 16, HALF, 128, "qk", False, 3, 1),
    (F16, 16, 8, 128, 16, HALF, 128, "qk", False, 5, 129),    # more row slots
    (F16, 16, 8, 128, 16, ADJ, 128, "k", False, 1, 1023),
    (F16, 16, 8, 128, 16, HALF, 128, "qk", True, 1, 2049),
    (Q8, 8, 1, 64, 16, HALF, 64, "q", False, 7, 600),
    (Q8, 32, 8, 64, 16, ADJ, 31, "", True, 2, 700),
    (F16, 8, 1, 256, 12, HALF, 256, "qk", True, 1, 700),
    (Q8, 8, 2, 256, 16, HALF, 100, "qk", False, 1, 530),      # partial: through LDS
    (F16, 4, 2, 512, 8, HALF, 512, "qk", False, 1, 1100),
    (Q8, 8, 1, 512, 16, ADJ, 400, "", False, 3, 2),
    (F16, 8, 1, 64, 16, HALF, 64, "qk", False, 3, 2),
    # 256 and 512 dims at two and four row slots, which a prompt chunk takes
    (F16, 8, 1, 256, 16, ADJ, 256, "qk", False, 1, 900),
    (Q8, 8, 1, 256, 16, HALF, 256, "qk", True, 3, 500),
    (F16, 8, 1, 256, 12, HALF, 100, "q", False, 1, 1500),
    (F16, 8, 1, 512, 16, HALF, 512, "qk", True, 1, 1500),
    (Q8, 8, 1, 512, 8, ADJ, 400, "k", False, 5, 300),
    (F16, 8, 1, 512, 16, HALF, 300, "qk", False, 1, 1500),
    # no norm at all (kernels of their own), from one slot to the most
    (F16, 32, 8, 64, 16, HALF, 64, "", False, 2, 700),
    (F16, 8, 1, 64, 16, ADJ, 64, "", False, 7, 600),
    (Q8, 16, 8, 128, 16, HALF, 128, "", False, 1, 2049),
    (F16, 16, 8, 128, 16, HALF, 128, "", False, 3, 1),
    (F16, 8, 1, 256, 16, HALF, 256, "", False, 1, 900),
    (Q8, 8, 1, 256, 12, HALF, 100, "", False, 3, 500),
    (F16, 8, 1, 512, 16, HALF, 512, "", False, 1, 900),
    (Q8, 4, 2, 512, 8, ADJ, 512, "", False, 1, 1100),
    (F16, 8, 1, 512, 16, ADJ, 512, "", False, 3, 2),
]


@pytest.mark.parametrize("case", CASES, ids=[f"rows{i}" for i in range(len(CASES))])
def test_rope_rows_bit_exact(device, case):
    import torch
    kv, H, HK, D, bt, pairing, n_rot, norms, v_rms, n_seq, n_tok = case
    print(f"\n[gpu-case] rope rows {case}", flush=True)
    starts = [3 * s for s in range(n_seq)]
    sc = Scenario(n_layer=1, n_head=H, n_kv=HK, head_dim=D, block_tokens=bt,
                  lens=[s + n_tok for s in starts], kv_type=kv, seed=5, fill=False,
                  outlier_frac=0.01 if kv == Q8 else 0.0)
    rng = np.random.default_rng(6)
    q = rng.standard_normal((n_seq, n_tok, H * D)).astype(np.float32)
    k = np.stack([sc.k_rows[0][s][starts[s]:] for s in range(n_seq)])
    v = np.stack([sc.v_rows[0][s][starts[s]:] for s in range(n_seq)])
    w = {c: rng.standard_normal(D).astype(np.float32) if c in norms else None for c in "qk"}

    def off(a):  # on the device, one float past an aligned address
        if a is None:
            return None
        flat = torch.empty(a.size + 1, dtype=torch.float32, device=device)
        flat[1:] = torch.from_numpy(a.ravel()).to(device)
        return flat[1:].view(a.shape)

    rope = emelk.RopeTable(n_rot, D, max(sc.lens), 1e4, pairing)
    out = off(np.full_like(q, 7.0))
    emelk.qkv_rope_append(sc.g, sc.k_pool, sc.v_pool, 0, off(q), out, off(k), off(v),
                          torch.tensor(starts, dtype=torch.int32, device=device), sc.tables, rope,
                          off(w["q"]), off(w["k"]), v_rms, 1e-6)
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    for s in range(n_seq):
        sc.k_rows[0][s][:starts[s]] = 0.0
        sc.v_rows[0][s][:starts[s]] = 0.0
        for t in range(n_tok):
            qo, ko, vo = oracle.qkv_rope_rows(q[s, t], k[s, t], v[s, t], H, HK, D, pairing, n_rot,
                                              1e4, starts[s] + t, q_norm=w["q"], k_norm=w["k"],
                                              v_rms=v_rms, eps=1e-6)
            np.testing.assert_array_equal(got[s, t].view(np.uint32), qo.view(np.uint32),
                                          err_msg=f"q of seq {s} token {t}")
            sc.k_rows[0][s][starts[s] + t] = ko
            sc.v_rows[0][s][starts[s] + t] = vo
    for which, pool in (("k", sc.k_pool), ("v", sc.v_pool)):
        np.testing.assert_array_equal(pool.cpu().numpy(), sc.expected_pool(which), err_msg=which)
    rope.close()
