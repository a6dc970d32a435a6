"""Packets of several streams that share their launches: each stream's PCM is
the bits it gets alone, whatever the other streams' packet sizes, and every
packet size agrees with the float64 whole-utterance model."""
import ctypes as C

import numpy as np
import pytest

import codec_model as M

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def codec():
    import qwen3_tts_codec_hip

    qwen3_tts_codec_hip.load()
    return qwen3_tts_codec_hip


@pytest.fixture(scope="module")
def weights():
    return M.make_weights(3)


@pytest.fixture(scope="module")
def model(codec, weights):
    return codec.SharedModel(weights)


# packet sizes per round: groups of one to six equal packets, mixed sizes, a
# leader that changes between rounds
@pytest.mark.parametrize("rounds", [
    [(4, 4, 4, 4, 4, 4), (1, 1, 1, 1, 1, 1), (4, 4, 4, 4, 4, 4)],
    [(1, 4, 1), (4, 4, 1), (2, 3, 2)],
    [(2, 3, 2, 3, 4), (3, 3, 3, 3, 3), (1, 2, 2, 2, 2)]])
def test_shared_launches_give_each_stream_its_own_bits(codec, model, rounds):
    n = len(rounds[0])
    streams = [M.random_codes(sum(r[i] for r in rounds), 50 + i) for i in range(n)]
    batch = [model.session() for _ in range(n)]
    alone = [model.session() for _ in range(n)]
    at = [0] * n
    for sizes in rounds:
        parts = [streams[i][at[i]:at[i] + sizes[i]] for i in range(n)]
        got = codec.process_batch(batch, parts)
        for i in range(n):
            want, _ = alone[i].packet(parts[i])
            pcm, result = got[i]
            assert result.frame_count == sizes[i] and result.first_frame_position == at[i]
            assert np.array_equal(pcm, want), (sizes, i)
            at[i] += sizes[i]
    # the same sessions go on alone, in the other order
    for i in reversed(range(n)):
        a, _ = batch[i].packet(streams[i][:2])
        b, _ = alone[i].packet(streams[i][:2])
        assert np.array_equal(a, b)


@pytest.mark.parametrize("frames", [1, 2, 3, 4])
def test_packet_size_matches_float64(model, weights, frames):
    """Final convolution before and after the clamp, within the published bar
    of the reference's own checkpoint (5e-6 on the final pre-clamp)."""
    codes = M.random_codes(2 * frames, 9)
    whole = M.F64Decoder(weights).run(codes)
    s = model.session()
    got = np.concatenate([s.debug_checkpoint(codes[at:at + frames], 12, 1920 * frames, 1) for at in (0, frames)])
    assert np.abs(got - whole[12]).max() <= 5e-6 * max(1.0, np.abs(whole[12]).max())


def test_batches_allocate_no_device_memory(codec, model):
    """A batch works in its members' own memory: sessions that lead their
    first batch (of several packet sizes, and of one) leave the device's free
    memory as it was, and report the same bytes as before."""
    hip = C.CDLL("libamdhip64.so")
    sessions = [model.session() for _ in range(6)]
    streams = [M.random_codes(12, 70 + i) for i in range(6)]
    # the launches' own first-use allocations, on other sessions' buffers
    codec.process_batch([model.session() for _ in range(2)], [s[:4] for s in streams[:2]])
    before = [s.memory().device_bytes for s in sessions]
    free, after, total = C.c_size_t(), C.c_size_t(), C.c_size_t()
    assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    for order in (range(6), reversed(range(6))):
        order = list(order)
        codec.process_batch([sessions[i] for i in order], [streams[i][:4] for i in order])
    codec.process_batch(sessions, [streams[i][8:8 + 1 + i // 2] for i in range(6)])
    assert hip.hipMemGetInfo(C.byref(after), C.byref(total)) == 0
    assert after.value == free.value
    assert [s.memory().device_bytes for s in sessions] == before


def test_failed_launches_cancel_their_members_alone(codec, model, monkeypatch):
    """Shared launches that fail to queue (forced on the leader, behind its
    launches) fail all their items, whose sessions then refuse packets until a
    reset; what was queued before completes, what comes after is not begun and
    goes on where it was."""
    def leader():
        with monkeypatch.context() as m:
            m.setenv("QWEN3_TTS_CODEC_TEST_FAIL_GROUP", "1")
            return model.session()

    sessions = [model.session(), leader(), model.session(), model.session()]
    sizes = [1, 3, 2, 3]  # launched as (0), (1, 3), (2)
    streams = [M.random_codes(8, 80 + i) for i in range(4)]
    for s, c in zip(sessions, streams):
        s.packet(c[:4])
    results = [codec.PacketResult() for _ in sessions]
    pcms = [np.zeros(7680, np.int16) for _ in sessions]
    items = (codec.BatchItem * 4)()
    parts = [np.ascontiguousarray(c[4:4 + n]) for c, n in zip(streams, sizes)]
    for i, s in enumerate(sessions):
        items[i] = codec.BatchItem(s.handle, parts[i].ctypes.data, sizes[i], 0, pcms[i].ctypes.data, 7680,
                                   C.pointer(results[i]))
    with pytest.raises(codec.CodecError) as e:
        codec.call("qwen3_tts_codec_session_process_batch_v1", items, 4)
    assert e.value.status == -2 and "launch decoder packet" in e.value.message
    assert [r.frame_count for r in results] == [1, 0, 0, 0]
    assert [s.state().frame_position for s in sessions] == [5, 4, 4, 4]
    for i in (1, 3):
        with pytest.raises(codec.CodecError) as e:
            sessions[i].packet(parts[i])
        assert e.value.status == -3
        sessions[i].reset()
    for i, (s, c) in enumerate(zip(sessions, streams)):
        alone = model.session()
        want = [alone.packet(c[:4])[0], alone.packet(parts[i])[0]]
        if i in (1, 3):
            assert np.array_equal(s.packet(c[:4])[0], want[0])
        got = pcms[i][:1920] if i == 0 else s.packet(parts[i])[0]
        assert np.array_equal(got, want[1]), i
