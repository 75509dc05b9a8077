"""Decode attention of many sequences of unequal length: the order in which workgroups take them, and blocks of keys around the ends of the
wavefronts' shares."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _step(lens, heads, kv_heads, dim, seed):
    gen = torch.Generator().manual_seed(seed)
    pages = [-(-n // 16) for n in lens]
    k = torch.randn((sum(pages) + 1, kv_heads, 16, dim), generator=gen).to(torch.bfloat16)
    v = torch.randn((sum(pages) + 1, kv_heads, dim, 16), generator=gen).to(torch.bfloat16)
    order = torch.randperm(sum(pages), generator=gen) + 1
    tables, at = torch.zeros((len(lens), max(pages)), dtype=torch.int32), 0
    for i, n in enumerate(pages):
        tables[i, :n] = order[at:at + n].int()
        at += n
    for i, n in enumerate(lens):                  # what lies behind a context in its last page is nobody's
        if n % 16:
            k[tables[i, n // 16], :, n % 16:] = float("nan")
            v[tables[i, n // 16], :, :, n % 16:] = float("nan")
    q = torch.randn((len(lens), heads * dim), generator=gen).to(torch.bfloat16)
    return q, k, v, tables


def _reference(q, k, v, tables, lens, heads, kv_heads, dim):
    out = torch.empty(q.shape, dtype=torch.float64)
    for i, n in enumerate(lens):
        pages = tables[i, :-(-n // 16)].long()
        keys = k[pages].double().permute(1, 0, 2, 3).reshape(kv_heads, -1, dim)[:, :n]
        values = v[pages].double().permute(1, 0, 3, 2).reshape(kv_heads, -1, dim)[:, :n]
        rows = q[i].double().view(kv_heads, heads // kv_heads, dim)
        p = torch.softmax(torch.matmul(rows, keys.transpose(1, 2).contiguous()) * dim ** -0.5, dim=-1)
        out[i] = torch.matmul(p, values).reshape(-1)
    return out


# more workgroups than compute units: two rounds and a part, equal lengths among them, padding sequences of one token, one kv head more than
# divides the compute units, several rounds of 16 sequences
@pytest.mark.parametrize("sequences,kv_heads,dim", [(33, 8, 64), (40, 8, 64), (64, 8, 64), (37, 7, 64), (61, 16, 32), (64, 8, 128)])
@pytest.mark.parametrize("waves", [4, 8])
def test_any_order_of_sequences_gives_the_same_bits(sequences, kv_heads, dim, waves):
    from paged_llm_amd.csrc import ops
    gen = torch.Generator().manual_seed(sequences * kv_heads + dim)
    lens = torch.randint(1, 700, (sequences,), generator=gen).tolist()
    lens[0], lens[-1], lens[5], lens[9] = 700, 1, 321, 321
    heads = 2 * kv_heads
    q, k, v, tables = _step(lens, heads, kv_heads, dim, sequences)
    args = (q.cuda(), k.cuda(), v.cuda(), tables.cuda(), torch.arange(sequences + 1, dtype=torch.int32).cuda(), torch.tensor(lens, dtype=torch.int32).cuda(),
            heads, kv_heads, dim, dim ** -0.5, 0, 1, 0, 1, waves, 0)
    plain = ops.paged_attention_mfma(*args)
    assert torch.equal(ops.paged_attention_mfma(*args, max_k_len=700), plain)
    # probabilities rounded to bfloat16 (2^-9 each) weigh values of size 1 (up to 4.5 here), the result is rounded once more
    want = _reference(q, k, v, tables, lens, heads, kv_heads, dim)
    assert (plain.double().cpu() - want).abs().max() <= 2.0 ** -8 * want.abs().max()


# a wavefront with no block, one, two, three (the loop ends with a block alone or with a pair), a last block of one key and of all, and partitions
@pytest.mark.parametrize("dim", [32, 64, 256])
@pytest.mark.parametrize("waves,partition", [(4, 0), (8, 0), (4, 256), (8, 512)])
def test_ends_of_the_wavefronts_shares(dim, waves, partition):
    from paged_llm_amd.csrc import ops
    if dim == 256 and waves == 8:
        pytest.skip("eight wavefronts of heads of 256 do not fit LDS") if ops._merge_lds_bytes(1, 8, 256) > ops._max_lds_bytes(torch.device("cuda")) else None
    step = 64 * waves
    lens = [1, 15, 64, 65, step - 63, step, step + 1, 2 * step, 2 * step + 64, 3 * step - 1, 3 * step + 1, 4 * step + 17]
    q, k, v, tables = _step(lens, 4, 2, dim, dim + waves)
    parts = -(-max(lens) // partition) if partition else 1
    got = ops.paged_attention_mfma(q.cuda(), k.cuda(), v.cuda(), tables.cuda(), torch.arange(len(lens) + 1, dtype=torch.int32).cuda(),
                                   torch.tensor(lens, dtype=torch.int32).cuda(), 4, 2, dim, dim ** -0.5, 0, 1, partition, parts, waves, 0)
    want = _reference(q, k, v, tables, lens, 4, 2, dim)
    assert (got.double().cpu() - want).abs().max() <= 2.0 ** -8 * want.abs().max()          # (as above)
