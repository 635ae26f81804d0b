"""The delta rule's prompt scan with two chunks to a barrier (delta_scan_pairs_kernel): every number of chunks modulo its unrolled loop, whole and ragged
last chunks, wave tiles past the last channel, and launches that end inside a segment, against the recurrence in 64 bits."""
import pytest

from tests.test_bokulorn_gpu import Delta, close, lib  # noqa: F401  (lib: the fixture)


pytestmark = pytest.mark.gpu


# one and two channel tiles a wave, all of them used, one and a half of the four waves idle, three of four idle
@pytest.mark.parametrize("shape", [(2, 2, 128, 128, 4), (3, 1, 80, 48, 3), (2, 1, 64, 32, 2), (4, 4, 16, 200, 2)])
@pytest.mark.parametrize("lengths,chunks", [([15, 16, 17, 32, 48], 64), ([64, 65, 80, 95, 112], 64), ([128, 129, 144, 193], 64), ([180, 33, 70], 5), ([200, 200], 9)])
def test_chunks_in_pairs(lib, shape, lengths, chunks):  # noqa: F811
    x = Delta(lib, *shape, lengths, seed=sum(shape) + sum(lengths))
    close(*x.step([(i, n) for i, n in enumerate(lengths)], chunks=chunks), 1)
    for i in range(len(lengths)):
        x.check_state(i)


# value columns: whole quads short of a tile, one past 64 and 128, no whole quad; keys of two rounds of lanes, of one past 128; bf16 and fp32 outputs
@pytest.mark.parametrize("shape", [(2, 1, 32, 20, 4), (5, 5, 16, 68, 3), (2, 2, 48, 132, 1), (3, 1, 24, 30, 4), (2, 1, 144, 64, 4), (1, 1, 256, 128, 5)])
def test_edges_of_columns(lib, shape):  # noqa: F811
    for f32 in (0, 1):
        x = Delta(lib, *shape, [40, 17, 2], seed=sum(shape))
        close(*x.step([(0, 40), (1, 17), (2, 2)], f32), f32)
        for i in range(3):
            x.check_state(i)


# one long segment in two parts at the same time: second parts of 0 .. 3 chunks by themselves and a ragged last one, one and two channel tiles a
# wave with waves idle and not; the next segment starts from the joined state
@pytest.mark.parametrize("shape", [(2, 2, 128, 128, 4), (16, 16, 128, 128, 4), (3, 1, 80, 80, 3), (4, 2, 64, 64, 2), (2, 1, 20, 20, 4), (1, 1, 7, 16, 1)])
@pytest.mark.parametrize("first,second", [(1008, 1024), (1024, 1056), (1025, 1071), (1055, 1036), (1500, 2)])
def test_long_segments_in_two_parts(lib, shape, first, second):  # noqa: F811
    x = Delta(lib, *shape, [first + second], seed=sum(shape) + first, strong=shape[0] == 4)
    close(*x.step([(0, first)], chunks=256), 1)
    close(*x.step([(0, second)], 0, chunks=256), 0)
    x.check_state(0)


# pieces of a segment that the workspace holds: two of them in two parts, the rest not; beside it a sequence too short, and with another one neither goes in parts
@pytest.mark.parametrize("lengths,chunks", [([2300], 70), ([1100, 40], 256), ([1100], 63)])
def test_parts_and_pieces(lib, lengths, chunks):  # noqa: F811
    x = Delta(lib, 4, 4, 128, 128, 4, lengths, seed=len(lengths) + chunks)
    close(*x.step([(i, n) for i, n in enumerate(lengths)], chunks=chunks), 1)
    for i in range(len(lengths)):
        x.check_state(i)


# heads of 128 on more CUs than three parts leave
@pytest.mark.parametrize("heads", [12, 16])
@pytest.mark.parametrize("first,second", [(1136, 1152), (1152, 1168), (1151, 1153)])
def test_two_parts_that_share_cus(lib, heads, first, second):  # noqa: F811
    test_long_segments_in_two_parts(lib, (heads, heads, 128, 128, 4), first, second)


# a chunk below the line (one scan), on it, and a ragged one above; a workspace that holds just so many, and one less
@pytest.mark.parametrize("shape", [(16, 16, 128, 128, 4), (3, 1, 128, 128, 2), (4, 4, 64, 64, 4), (20, 20, 96, 96, 3), (1, 1, 7, 16, 1)])
@pytest.mark.parametrize("first,second,chunks", [(752, 768, 256), (753, 770, 256), (768, 1000, 48), (800, 769, 47)])
def test_line_of_two_parts(lib, shape, first, second, chunks):  # noqa: F811
    x = Delta(lib, *shape, [first + second], seed=sum(shape) + first)
    close(*x.step([(0, first)], chunks=chunks), 1)
    close(*x.step([(0, second)], 0, chunks=chunks), 0)
    x.check_state(0)


# the replies' rooms of a second part: 16 dkp numbers a head and chunk, for heads that have CUs for one (16 of 128 on 256 CUs), and not for one head more
def test_rooms_for_replies(lib):  # noqa: F811
    import torch
    from tests.bokulorn_cases import config, delta
    from vllm_neuron_amd._native import NativeModel
    from vllm_neuron_amd.models import config_from_dict, fill_sizes
    heads, length = torch.cuda.get_device_properties(0).multi_processor_count // 16, 4096

    def workspace(n):
        c = config_from_dict(config(256, 256, [delta(n, n, 128, 128, 4)]))
        fill_sizes(c, lambda name: (128, 256))
        m = NativeModel(stack=dict(c.stack, compute_dtype=1), ctx_buckets=[length], num_blocks=129, block_size=32, max_num_seqs=1, max_model_len=length, device_id=0, use_graphs=0)
        m.init_synthetic_weights(1, 0.02)
        m.finalize()
        got = m.kv_stats()["workspace_bytes"]
        m.close()
        return got
    at = {n: workspace(n) for n in (heads - 1, heads, heads + 1, heads + 2)}
    chunks = length // 16 + 1
    # what a head takes besides is the same either way (a row's columns come in sixteens: none of the pairs crosses one)
    assert (at[heads] - at[heads - 1]) - (at[heads + 2] - at[heads + 1]) == chunks * 16 * 128 * 4
