"""Index tables of a ragged batch against the lists they stand for."""
import random

import pytest
import torch

from deepspeedsyclsupport_amd.inference.model_implementations.transformer import RaggedMeta
from deepspeedsyclsupport_amd.ops.native import cpu_ops, gemv_ops


@pytest.mark.parametrize("seed", range(6))
def test_tables_hold_the_batch(seed):
    r = random.Random(seed)
    n_decode, slots = r.randint(0, 3), r.random() < 0.5
    n = [1] * n_decode + sorted(r.choice((0, 1, 16, 17, 64)) for _ in range(r.randint(0, 3))) + [65, 128, 129, 300][:r.randint(1, 4)]
    S, block = len(n), 16
    starts = [r.randint(1, 40) if i < n_decode else r.choice((0, 5, 64)) for i in range(S)]
    blocks = [[r.randint(0, 99) for _ in range(-(-(st + k) // block))] for st, k in zip(starts, n)]
    toks = [torch.randint(0, 1000, (k, )) for k in n]
    rows = [0, sum(n) - 1] if seed % 2 else None
    m = RaggedMeta.build(starts, n, blocks, n_decode, block, None, list(range(7, 7 + S)) if slots else None, rows, toks)
    cu = [sum(n[:i]) for i in range(S + 1)]
    assert m.cu_host == cu and m.cu_q.tolist() == cu and m.start_pos.tolist() == starts == m.start_host
    assert m.pos_ids.tolist() == [st + j for st, k in zip(starts, n) for j in range(k)]
    assert m.seq_ids.tolist() == [i for i, k in enumerate(n) for _ in range(k)]
    assert m.seq_lens.tolist() == [st + k for st, k in zip(starts, n)]
    assert m.work.tolist() == [[i, b] for i in range(n_decode, S) for b in range(-(-n[i] // 128))]
    last = rows or [c - 1 for c in cu[1:]]
    assert m.last_idx.tolist() == last == m.last_rows.tolist() and m.last_idx.dtype == torch.int64 and not m.all_rows
    assert torch.equal(m.ids, torch.cat(toks))
    width = max(len(b) for b in blocks)
    assert m.block_tables.tolist() == [b + [0] * (width - len(b)) for b in blocks] and m.max_len == width * block
    assert m.slots.tolist() == (list(range(7, 7 + S)) if slots else [])
    long = [i for i in range(S) if n[i] > RaggedMeta.STEP_TOKENS] if slots else []
    assert m.seq_list.tolist() == ([i for i in range(S) if i not in long] if slots else [])
    work = [[i, c] for i in long for c in range(-(-n[i] // RaggedMeta.STATE_CHUNK))]
    assert m.chunk_work.tolist() == work and m.chunk_seqs.tolist() == [[i, work.index([i, 0])] for i in long]
    assert m.n_short == next((i for i in range(n_decode, S) if n[i] > RaggedMeta.SHORT_TOKENS), S)
    ctx = [starts[i] + n[i] for i in range(m.n_short, S)]
    assert m.kv_offs.tolist() == [sum(ctx[:i]) for i in range(len(ctx) + 1)] and m.kv_total == sum(ctx)


@pytest.mark.parametrize("what", ["starts", "tokens", "sum", "block", "slot", "row"])
def test_what_32_bits_do_not_hold_is_refused(what):
    big = 1 << 31
    a = dict(starts=[4, 0], n_new=[1, 2], block_lists=[[1], [2]], n_decode=1, block_size=16, device=None, slots=[0, 1], logit_rows=[0, 2])
    RaggedMeta.build(**a)
    a.update({"starts": dict(starts=[big, 0]), "tokens": dict(n_new=[1, big]), "sum": dict(starts=[4, big - 2]), "block": dict(block_lists=[[1], [big]]),
              "slot": dict(slots=[0, -big - 1]), "row": dict(logit_rows=[0, big + 2])}[what])
    with pytest.raises(OverflowError):
        RaggedMeta.build(**a)


def test_range_of_host_tokens():
    f = cpu_ops().int_range
    assert f([]) == (0, -1) and f([torch.empty(0, dtype=torch.int64)]) == (0, -1)
    assert f([torch.tensor([3, -1]), torch.tensor([7], dtype=torch.int32)]) == (-1, 7)


@pytest.mark.gpu
@pytest.mark.parametrize("S,new", [(1, 1), (12, 1), (50, 1), (60, 1), (90, 1), (3, 40), (2, 700)])
def test_tables_on_the_device(S, new):
    """Short tables go as a kernel's arguments, long ones as a copy: the same tables either way, twice in a row."""
    args = [5 + i for i in range(S)], [new] * S, [[i, 2 * i + 1, 7] for i in range(S)], S if new == 1 else 0, 256
    toks = [torch.arange(new) + i for i in range(S)]
    for slots in (list(range(S)), list(range(S, 2 * S))):
        want = RaggedMeta.build(*args, None, slots, None, toks)
        for device in ("cuda", "cuda:0", torch.device("cuda")):
            got = RaggedMeta.build(*args, device, slots, None, toks)
            for name, a in vars(want).items():
                b = getattr(got, name)
                if torch.is_tensor(a):
                    assert b.device == torch.device("cuda:0") and b.dtype == a.dtype and torch.equal(b.cpu(), a), name
                else:
                    assert b == a, name


@pytest.mark.gpu
def test_words_as_arguments():
    most = gemv_ops().upload_most()
    assert gemv_ops().upload(torch.zeros(most + 1, dtype=torch.int32), 0) is None
    for n in (0, 1, 239, 240, 241, 256, 257, most - 1, most):
        host, outs, want = torch.empty(n, dtype=torch.int32), [], []
        for k in range(4):
            host.copy_(torch.randint(-2**31, 2**31 - 1, (n, )))   # (free again as soon as the call returns)
            want.append(host.clone())
            outs.append(gemv_ops().upload(host, 0))
        assert all(torch.equal(a.cpu(), b) for a, b in zip(outs, want))
