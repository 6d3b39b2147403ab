"""The choice of a prefill's key shares, on the host side of the library over a
stand-in for the HIP runtime: what it chooses for some calls, that the pre-pass is
enqueued ahead of it, and that it takes little enough host time to hide there."""
import time

import pytest

import hip_standin as hip
from hip_standin import PTR


@pytest.fixture(scope="module")
def ctx():
    with hip.binding().Context(0) as c:
        yield c


def _args(T, past, Dh, window):
    return dict(q=PTR, k=PTR, v=PTR, out=PTR, T=T, S=past + T, Hq=8, Hkv=1, Dh=Dh, Dv=Dh, q_pos0=past, window=window)


CALLS = [  # T, earlier keys, head_dim, window; workgroups, workgroups of the merge
    (2048, 0, 256, 512, 256, 0),      # every CU has one block: whole
    (2048, 0, 512, 0, 510, 170 * 8),  # causal: the later blocks in two or three
    (173, 6001, 512, 0, 242, 22 * 8),
    (16, 16000, 512, 0, 256, 2 * 8),
    (512, 0, 256, 512, 238, 54 * 4),
    (300, 0, 256, 512, 140, 32 * 4),
]


@pytest.mark.parametrize("T,past,Dh,window,workgroups,merge", CALLS)
def test_shares(ctx, T, past, Dh, window, workgroups, merge):
    ctx.attention_batch(ctx.prepare_batch([_args(T, past, Dh, window)]))
    hip.launches()
    ctx.attention_batch(ctx.prepare_batch([_args(T, past, Dh, window)]))  # (its workspace is there by now)
    got = hip.launches()
    assert [x.name for x in got] == ["g4a_split_kv"] + ["g4a_prefill2_d256" if Dh == 256 and not merge else
                                                        f"g4a_prefill2_{'split_' if Dh == 256 else ''}d{Dh}"] + (
        [f"g4a_prefill_merge_d{Dh}"] if merge else [])
    assert got[1].gx == workgroups and (not merge or got[2].gx == merge)


def test_no_second_round_for_a_few_workgroups(ctx):
    # 513 .. 700 tokens in shares of 257 .. 263 workgroups on 256 CUs took up to a half more than
    # in fewer shares; a head_dim, a window and earlier keys of each kind
    for Dh, window in ((256, 0), (256, 512), (512, 0)):
        for past in (0, 100, 1000, 3000, 6001):
            for T in range(17, 800, 29):
                ctx.attention_batch(ctx.prepare_batch([_args(T, past, Dh, window)]))
                grid = next(x.gx for x in hip.launches() if "prefill2" in x.name)
                assert not 256 < grid < 280, (T, past, Dh, window, grid)


def test_a_workspace_that_grows_for_the_partials_has_the_splits_too():
    with hip.binding().Context(0) as c:
        c.linear_q(hip.weight(64, 2048, 4), PTR, PTR, 3700)  # 30 MB of workspace: the K/V splits' place, 16.8 MB
        hip.launches()
        call = c.prepare_batch([_args(2048, 2048, 512, 0)])  # and 68 MB of partials
        c.attention_batch(call)
        names = [x.name for x in hip.launches()]
        assert names == ["g4a_split_kv", "g4a_split_kv", "g4a_prefill2_d512", "g4a_prefill_merge_d512"]
        c.attention_batch(call)
        assert [x.name for x in hip.launches()] == names[1:]


def test_host_time(ctx):
    # 64 calls at a time, the least of several runs: a call is its launches (recorded here in
    # well under 1 us each) and the choice; with every count played through these calls took
    # 14, 18, 8, 1, 16 and 3 us, now 1, 9, 3, 1, 3 and 2
    for T, past, Dh, window, *_ in CALLS:
        calls = ctx.prepare_batch([_args(T, past, Dh, window)] * 64)
        least = 1e9
        for _ in range(30):
            t = time.perf_counter()
            ctx.attention_batch(calls)
            least = min(least, (time.perf_counter() - t) / 64 * 1e6)
            hip.launches()
        print(f"T={T} past={past} Dh={Dh}: {least:.1f} us")
        # (on a machine several times slower too)
        assert least < {(2048, 256): 8, (512, 256): 12, (2048, 512): 40}.get((T, Dh), 30)
