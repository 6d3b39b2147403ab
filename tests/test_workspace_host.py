"""How a context's workspace grows, on the host side of the library over a stand-in
for the HIP runtime: a projection of many rows takes a larger one if there is memory
for it and else runs the kernel that needs none, with the workspace it found left
as it was; growth by doubling does not ask for more than a tight device has; and
errors that are not a lack of memory come back to the caller. A prefill without
memory for the partials of split query blocks runs them whole, and a batch of sequences without
room for its finer splits' partials takes fewer."""
import pytest

import hip_standin as hip
from hip_standin import PTR

MB = 1 << 20


@pytest.fixture
def ctx():
    c = hip.binding().Context(0)
    hip.launches()
    yield c
    hip.budget()
    hip.sync_error(0)
    c.close()


def _split_bytes(M, K):
    return (M + 31) // 32 * 32 * (K + (K + 255) // 256) * 4


def _project(ctx, M, K=1536):
    ctx.linear_q(hip.weight(256, K, 4), PTR, PTR, M)
    return [x.name for x in hip.launches()]


def _attend(ctx, S):
    ctx.attention(PTR, PTR, PTR, PTR, T=64, S=S, Hq=8, Hkv=1, Dh=512, Dv=512, q_pos0=S - 64)
    return [x.name for x in hip.launches()]


def test_a_projection_without_memory_for_its_split_leaves_the_workspace(ctx):
    _attend(ctx, 8192)
    before = hip.used()
    hip.budget(before + MB)
    for _ in range(2):
        names = _project(ctx, 20000)  # 120 MB
        assert len(names) == 1 and names[0].startswith("g4a_linear_q_mfma_b4")
        assert hip.used() == before
        assert hip.last_error() == 0  # nothing for the next launch check of this thread
        # the attention call still has the workspace it made
        assert "g4a_prefill2_d512" in _attend(ctx, 8192)


def test_a_tight_device_gives_the_bytes_asked_for(ctx):
    _attend(ctx, 8192)  # about 42 MB
    need = _split_bytes(10000, 1536)  # 59 MB, less than twice that
    hip.budget(hip.used() + need + MB)
    assert _project(ctx, 10000)[0] == "g4a_split_x_b4"
    hip.budget(hip.used())
    assert _project(ctx, 10000)[0] == "g4a_split_x_b4"


def test_growth_makes_room_with_the_old_workspace_when_a_call_must_have_it(ctx):
    _attend(ctx, 8192)
    # no room for both: the call that cannot do without takes the old one's place
    hip.budget(hip.used() + 8 * MB)
    assert "g4a_prefill2_d512" in _attend(ctx, 9000)


def test_a_call_that_cannot_have_its_workspace_leaves_room_for_smaller_ones(ctx):
    _attend(ctx, 8192)
    hip.budget(hip.used() + 8 * MB)
    with pytest.raises(hip.binding().G4aError) as e:
        _attend(ctx, 65536)
    assert e.value.code == -6
    assert "g4a_prefill2_d512" in _attend(ctx, 8192)


def test_errors_other_than_a_lack_of_memory_reach_the_caller(ctx):
    _attend(ctx, 1024)
    hip.sync_error(719)  # a launch failure found when the growth waits for the stream
    with pytest.raises(hip.binding().G4aError) as e:
        _project(ctx, 20000)
    assert e.value.code == -1
    hip.sync_error(0)
    assert _project(ctx, 20000)[0] == "g4a_split_x_b4"


@pytest.mark.parametrize("Dh", [256, 512])
def test_a_prefill_with_memory_for_its_key_splits_only_runs_whole_blocks(ctx, Dh):
    S, T = 8192, 64
    splits = 256 + 2 * S * Dh * 4 + S // 16 * 4
    hip.budget(hip.used() + splits + 256)

    def attend():
        ctx.attention(PTR, PTR, PTR, PTR, T=T, S=S, Hq=8, Hkv=1, Dh=Dh, Dv=Dh, q_pos0=S - T)
        return {x.name: x.gx for x in hip.launches()}

    whole = {256: "g4a_prefill2_d256", 512: "g4a_prefill2_d512"}[Dh]
    got = attend()
    assert got[whole] == T // 8 and len(got) == 2
    hip.budget()
    got = attend()
    assert f"g4a_prefill_merge_d{Dh}" in got


def _batch(ctx, n, S):
    calls = ctx.prepare_batch([dict(q=PTR, k=PTR, v=PTR, out=PTR, T=1, S=S, Hq=8, Hkv=1, Dh=512, Dv=512, q_pos0=S - 1)
                               for _ in range(n)])
    assert ctx.attention_decode_batch(calls) == n
    return [(x.name, x.gx) for x in hip.launches()]


def test_a_captured_batch_takes_the_splits_its_workspace_has_room_for(ctx):
    # 128 sequences of 160 keys: 4 splits each (48 keys) have partials of 8.03 MiB, 3 of 64 keys 6.02
    ctx.attention(PTR, PTR, PTR, PTR, T=1, S=1000, Hq=8, Hkv=1, Dh=512, Dv=512, q_pos0=999)  # 8 MiB of workspace
    hip.launches()
    ctx.capture_begin()
    got = _batch(ctx, 128, 160)
    ctx.capture_end().free()
    assert got == 2 * [("g4a_decode_wave_batch_d512", 3), ("g4a_combine_rows_batch_d512", 8)]
    # the same without memory to grow it, and eagerly
    hip.budget(hip.used())
    assert _batch(ctx, 128, 160) == got
    hip.budget()
    assert _batch(ctx, 128, 160) == 2 * [("g4a_decode_wave_batch_d512", 4), ("g4a_combine_rows_batch_d512", 8)]


def test_a_capture_after_the_eager_call_records_its_kernels(ctx):
    def calls():
        got = _attend(ctx, 8192) + _project(ctx, 3000)
        return got + _batch(ctx, 128, 160)

    calls()
    eager = calls()  # (the workspace is there by now)
    ctx.capture_begin()
    captured = calls()
    ctx.capture_end().free()
    assert captured == eager and "g4a_prefill_merge_d512" in eager and "g4a_split_x_b4" in eager
