"""Prefill query blocks split over several workgroups, each over a share of the
block's key tiles, and the merge of their partials: against the CPU oracle at
the bars every attention result is held to (max-abs 1e-5, mean-abs 1e-6). Few
queries over many keys (many shares of few tiles, shares no early row of the
block sees), causal prompts whose blocks take different share counts, ragged
ends, windows, two kv heads, V past the fp16 range; and the no-alloc entry
point, whose partials end past its 64 MiB of scratch, bit-identical."""
import numpy as np
import pytest

import g4a
import g4a.synth as synth
import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,S,Dh,W,Hkv,vscale", [
    (16, 4099, 512, 0, 1, 1.0), (17, 2500, 256, 0, 1, 1.0), (23, 1033, 512, 0, 2, 1.0), (16, 16, 512, 0, 1, 1.0),
    (200, 200, 512, 0, 1, 1.0), (130, 130, 256, 0, 2, 1.0), (70, 900, 256, 512, 1, 1.0), (97, 640, 512, 100, 1, 1.0),
    (33, 1500, 512, 0, 1, 1e5), (33, 1500, 256, 0, 1, 1e5),
])
def test_split_blocks_match_the_oracle(ctx, T, S, Dh, W, Hkv, vscale):
    ins = synth.gemma_inputs(T=T, S=S, Dh=Dh, seed=T + S, Hq=8 * Hkv, Hkv=Hkv)
    v = (ins.v * np.float32(vscale)).astype(np.float32)
    print(f"[gpu] T={T} S={S} Dh={Dh} window={W} Hkv={Hkv} v x {vscale:g}", flush=True)
    want = oracle.attention(ins.q, ins.k, v, ins.q_pos, ins.k_pos, window=W)
    got = g4a.attention_host(ctx, ins.q, ins.k, v, q_pos=ins.q_pos, k_pos=ins.k_pos, window=W)
    # errors scale with |v|: in units of the factor
    d = np.abs(got.astype(np.float64) - np.asarray(want, np.float64)) / vscale
    print(f"  max-abs {d.max():.3e} mean-abs {d.mean():.3e}", flush=True)
    assert d.max() <= 1e-5 and d.mean() <= 1e-6


@pytest.mark.parametrize("T,S", [(2400, 2400), (64, 15600), (1500, 6000)])
def test_noalloc_split_is_bit_identical(ctx, T, S):
    ins = synth.gemma_inputs(T=T, S=S, Dh=512, seed=7)
    bufs = [ctx.upload(x) for x in (ins.q, ins.k, ins.v)]
    outs = [ctx.empty((T, 8 * 512)) for _ in range(2)]
    kw = dict(T=T, S=S, Hq=8, Hkv=1, Dh=512, Dv=512, q_pos0=S - T)
    try:
        print(f"[gpu] T={T} S={S}", flush=True)
        ctx.attention(*(b.ptr for b in bufs), outs[0].ptr, **kw)
        ctx.attention_noalloc(*(b.ptr for b in bufs), outs[1].ptr, **kw)
        assert np.array_equal(outs[0].to_host(), outs[1].to_host())
    finally:
        for b in bufs + outs:
            b.free()


@pytest.mark.parametrize("Dh", [256, 512])
def test_capture_with_room_for_the_keys_only(Dh):
    # the workspace, grown by a projection's split of 4 Dh rows (2056 floats each), holds the key
    # splits (8 Dh bytes a key) but no partial slot: the capture records unsplit blocks
    T, S, M, N, K = 64, 4096, 4 * Dh, 64, 2048
    ins = synth.gemma_inputs(T=T, S=S, Dh=Dh, seed=11)
    want = oracle.attention(ins.q, ins.k, ins.v, ins.q_pos, ins.k_pos)
    with g4a.Context(0) as own:
        bufs, out = [own.upload(x) for x in (ins.q, ins.k, ins.v)], own.empty((T, 8 * Dh))
        x, y = own.upload(np.zeros((M, K), np.float32)), own.empty((M, N))
        qb, sc = own.upload(np.zeros((N, K // 2), np.uint8)), own.upload(np.ones(N, np.float32))
        w = g4a.DeviceQWeight(g4a.QWeightArgs(qb.ptr, sc.ptr, N, K, 4, 0, K), None, None)
        print(f"[gpu] Dh={Dh}", flush=True)
        own.linear_q(w, x.ptr, y.ptr, M)
        own.sync()
        own.capture_begin()
        own.attention(*(b.ptr for b in bufs), out.ptr, T=T, S=S, Hq=8, Hkv=1, Dh=Dh, Dv=Dh, q_pos0=S - T)
        graph = own.capture_end()
        for _ in range(2):
            graph.launch()
            d = np.abs(out.to_host().astype(np.float64) - want)
            assert d.max() <= 1e-5 and d.mean() <= 1e-6
        graph.free()
        for b in bufs + [out, x, y, qb, sc]:
            b.free()
