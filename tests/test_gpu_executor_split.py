"""The step executor's multi-token steps where the prefill splits its keys: a
long sequence that splits beside a short one that does not, on the workspace
that the decode steps around them use too, with both split plans, and the layer
calls captured once and replayed after the sequences have grown."""
import ctypes

import numpy as np
import pytest

import emelk
import oracle
from kvsetup import assert_close

pytestmark = pytest.mark.gpu

H, HKV, D, BT, L = 8, 2, 128, 16, 2
MAX_KV = 2048
BASE = 1e4
SCALE = 1.0 / np.sqrt(D)


class Rig:
    """An executor over `n` sequences and the oracle's stored rows of each."""

    def __init__(self, device, kv_type, n, seed, stream=None):
        import torch
        self.torch, self.device = torch, device
        self.rng = np.random.default_rng(seed)
        blocks = n * (MAX_KV // BT)
        self.g = emelk.geometry(L, H, HKV, D, BT, blocks, kv_type)
        self.actor = emelk.KvActor()
        assert self.actor.reserve(n, blocks, BT)[0]
        self.actor.set_free_order(self.rng.permutation(blocks).astype(np.uint16))
        for s in range(n):
            assert self.actor.allocate_sequence(s)[0]
        self.cache = emelk.KvCache(self.g, stream=stream)
        self.rope = emelk.RopeTable(D, D, MAX_KV, BASE, emelk.NEOX_PAIRING, stream=stream)
        self.dec = emelk.BatchDecoder(self.g, self.actor, self.cache, self.rope, max_batch=n,
                                      max_kv_len=MAX_KV, stream=stream)
        self.rows = [[([], []) for _ in range(L)] for _ in range(n)]
        self.stored = ((lambda x: oracle.fp16_to_fp32(oracle.fp32_to_fp16(x)))
                       if kv_type == emelk.KV_F16 else
                       (lambda x: oracle.dequantize_q8_0(oracle.quantize_q8_0(x))))

    def draw(self, n, tokens):
        d = lambda w: self.rng.standard_normal((n, tokens, w)).astype(np.float32)  # noqa: E731
        return [(d(H * D), d(HKV * D), d(HKV * D)) for _ in range(L)]

    def want(self, ids, pos, rows, only=None):
        """The oracle's outputs [layer][seq][token] (token t in `only`, all of
        them by default), the rows stored as it goes."""
        out = {}
        for layer in range(L):
            for i, s in enumerate(ids):
                q, k, v = (x[i] for x in rows[layer])
                ks, vs = self.rows[s][layer]
                for t in range(q.shape[0]):
                    assert len(ks) == pos[i] + t
                    qo, ko, vo = oracle.qkv_rope_rows(q[t], k[t], v[t], H, HKV, D,
                                                      emelk.NEOX_PAIRING, D, BASE, pos[i] + t)
                    ks.append(self.stored(ko))
                    vs.append(self.stored(vo))
                    if only is None or t in only:
                        q16 = oracle.fp16_to_fp32(oracle.fp32_to_fp16(qo))
                        out[layer, i, t] = oracle.attention_f64(q16, np.stack(ks), np.stack(vs), H,
                                                                HKV, D, pos[i] + t + 1, SCALE)
        return out

    def check(self, got, want, what):
        for (layer, i, t), w in want.items():
            assert_close(got[layer][i, t], w, what=f"{what}: layer {layer} seq {i} token {t}")

    def step(self, ids, tokens, what, only=None):
        torch = self.torch
        rows = self.draw(len(ids), tokens)
        pos = self.dec.begin_step(ids, tokens)
        outs, roped = [], []
        for layer in range(L):
            q, k, v = (torch.from_numpy(x).to(self.device) for x in rows[layer])
            out = torch.full_like(q, float("nan"))
            self.dec.layer(layer, q, q, k, v, out, SCALE)
            outs.append(out)
            roped.append(q)
        torch.cuda.synchronize()
        self.check([o.cpu().numpy() for o in outs], self.want(ids, pos, rows, only), what)
        return pos, outs, roped

    def unsplit(self, layer, ids, pos, roped):
        """The same attention through the entry point without a workspace."""
        torch = self.torch
        stride = MAX_KV // BT
        t = self.actor.export_block_tables(ids, stride)
        t = torch.from_numpy(np.ascontiguousarray(t).view(np.int16)).to(self.device)
        start = torch.tensor(pos, dtype=torch.int32, device=self.device)
        out = torch.full_like(roped, float("nan"))
        assert emelk.lib.emelk_attn_prefill_chunk(
            ctypes.byref(self.g), emelk.lib.emelk_kv_cache_k_pool(self.cache.handle),
            emelk.lib.emelk_kv_cache_v_pool(self.cache.handle), layer, roped.data_ptr(),
            out.data_ptr(), len(ids), int(roped.shape[1]), start.data_ptr(), t.data_ptr(), stride,
            SCALE, torch.cuda.current_stream().cuda_stream) == emelk.ERR_NONE
        torch.cuda.synchronize()
        return out


@pytest.mark.parametrize("fixed", [False, True], ids=["step", "fixed"])
@pytest.mark.parametrize("kv_type", [emelk.KV_F16, emelk.KV_Q8_0], ids=["f16", "q8_0"])
def test_steps_that_split(device, kv_type, fixed):
    import torch
    print(f"\n[gpu-case] executor with split prefill steps, kv {kv_type}, fixed plan {fixed}",
          flush=True)
    rig = Rig(device, kv_type, 2, 91)
    rig.dec.set_fixed_plan(fixed)
    rig.step([0], 1500, "long prompt", only=(0, 777, 1499))
    rig.step([1], 40, "short prompt", only=(0, 39))
    for ids, what in (([0, 1], "both"), ([1, 0], "the other way round")):
        pos, outs, roped = rig.step(ids, 6, what)
        for layer in range(L):
            whole = rig.unsplit(layer, ids, pos, roped[layer])
            for i, s in enumerate(ids):  # the long one's sums come in another order
                assert torch.equal(whole[i], outs[layer][i]) == (s == 1)
        rig.step(ids, 1, f"{what}, a decode step after")
    rig.dec.close()


def test_captured_layers_that_split(device):
    import torch
    print("\n[gpu-case] executor, multi-token layers captured once and replayed", flush=True)
    side = torch.cuda.Stream()
    ids, tokens = [0, 1], 6
    with torch.cuda.stream(side):
        rig = Rig(device, emelk.KV_F16, 2, 92, stream=side.cuda_stream)
        rig.dec.set_fixed_plan(True)
        buf = [[torch.zeros((2, tokens, w), device=device) for w in (H * D, HKV * D, HKV * D)]
               for _ in range(L)]
        roped = [torch.zeros_like(b[0]) for b in buf]
        outs = [torch.zeros_like(b[0]) for b in buf]

        def layers():
            for layer in range(L):
                q, k, v = buf[layer]
                rig.dec.layer(layer, q, roped[layer], k, v, outs[layer], SCALE)

        rig.step([0], 700, "prompt of one", only=(699,))
        graph = None
        for grow in (0, 30, 600):  # 0: the second sequence starts with this step
            if grow:
                rig.step([1], grow, "prompt of the other", only=(grow - 1,))
                rig.step([0], 3 * grow // 4, "the first one grows", only=(0,))
            rows = rig.draw(2, tokens)
            for layer in range(L):
                for dst, src in zip(buf[layer], rows[layer]):
                    dst.copy_(torch.from_numpy(src))
            pos = rig.dec.begin_step(ids, tokens)
            if graph is None:
                graph = torch.cuda.CUDAGraph()
                with torch.cuda.graph(graph, stream=side):
                    layers()
            graph.replay()
            side.synchronize()
            got = [o.cpu().numpy() for o in outs]
            rig.check(got, rig.want(ids, pos, rows), f"replay at {pos}")
            for layer in range(L):
                whole = rig.unsplit(layer, ids, pos, roped[layer])
                for i in range(2):
                    assert torch.equal(whole[i], outs[layer][i]) == (pos[i] < 100)
        rig.dec.close()
