"""qh_attention_fp8_noalloc against qh_attention_fp8, through the C ABI (MI355X only).

The no-alloc entry point has no workspace to scan q-tiles into: its waves
count them. Calls of many and of few sequences, on either side of where the
workspace entry point scans, must each be bit-identical to it on the same
inputs, values and scales. A call past the sequence limit is refused on the
host.
"""

import math

import pytest
import torch

from quail_amd import _hip, kernels, layout

pytestmark = pytest.mark.gpu

DEV = "cuda"
PAGE = 16
N_Q, N_KV, D = 32, 8, 128


def _case(seed, n_seqs, prefix, max_suffix):
    """n_seqs sequences over a shared prefix node plus own suffix pages,
    physical pages permuted; every table entry is a valid page."""
    g = torch.Generator().manual_seed(seed)
    lens = torch.randint(1, max_suffix + 1, (n_seqs,), generator=g).tolist()
    node_pages = -(-prefix // PAGE)
    own = [-(-(prefix + n) // PAGE) - prefix // PAGE for n in lens]
    n_pages = node_pages + sum(own) + 4
    perm = torch.randperm(n_pages, generator=g).tolist()
    shared, cursor = perm[:node_pages], node_pages
    tables, used = [], []
    for n, extra in zip(lens, own):
        pages = shared[:prefix // PAGE] + perm[cursor:cursor + extra]
        cursor += extra
        assert len(pages) * PAGE >= prefix + n
        tables.append(pages)
        used.append(prefix + n)
    width = max(map(len, tables))
    table = torch.zeros(n_seqs, width, dtype=torch.int32)
    for i, p in enumerate(tables):
        table[i, :len(p)] = torch.tensor(p, dtype=torch.int32)
    cu_q = torch.zeros(n_seqs + 1, dtype=torch.int32)
    cu_q[1:] = torch.cumsum(torch.tensor(lens), 0)
    T = int(cu_q[-1])
    q = (torch.randn(T, N_Q, D, generator=g) / math.sqrt(D)).to(torch.bfloat16)
    k_rows = (torch.randn(n_pages * PAGE, N_KV, D, generator=g) / math.sqrt(D)).to(torch.bfloat16)
    v_rows = (torch.randn(n_pages * PAGE, N_KV, D, generator=g) / math.sqrt(D)).to(torch.bfloat16)
    return dict(q=q.to(DEV), kp=layout.k_pool_from_rows(k_rows).to(DEV),
                vp=layout.v_pool_from_rows(v_rows).to(DEV), table=table.to(DEV),
                used=torch.tensor(used, dtype=torch.int32, device=DEV), cu_q=cu_q.to(DEV),
                max_q=max(lens), n_seqs=n_seqs, T=T, n_pages=n_pages)


def _call(c, no_alloc):
    T = c["T"]
    out_q = torch.full((T, N_Q * D), 0x7F, dtype=torch.uint8, device=DEV)
    scales = kernels.col_major_scales(T, N_Q * D, DEV)
    scales.fill_(float("nan"))
    args = [c["q"].data_ptr(), c["q"].stride(0), T, None, c["kp"].data_ptr(),
            c["vp"].data_ptr(), c["n_pages"], c["table"].data_ptr(), c["table"].shape[1], PAGE,
            c["cu_q"].data_ptr(), c["used"].data_ptr(), c["n_seqs"], T, c["max_q"], N_Q, N_KV,
            D, 1.0 / math.sqrt(D), 1, out_q.data_ptr(), out_q.stride(0), scales.data_ptr(), 0]
    stream = torch.cuda.current_stream().cuda_stream
    if no_alloc:
        _hip.call("qh_attention_fp8_noalloc", *args, stream)
    else:
        ws = torch.empty(_hip.workspace_bytes(c["n_seqs"]), dtype=torch.uint8, device=DEV)
        _hip.call("qh_attention_fp8", *args, ws.data_ptr(), ws.numel(), stream)
    torch.cuda.synchronize()
    return out_q.cpu(), scales.cpu()


def test_noalloc_attention_matches_the_workspace_entry_point_twice():
    big = _case(71, n_seqs=48, prefix=256, max_suffix=200)
    small = _case(72, n_seqs=5, prefix=40, max_suffix=90)
    scanned = _case(73, n_seqs=300, prefix=40, max_suffix=60)
    for case in (big, small, scanned):
        want_q, want_s = _call(case, no_alloc=False)
        got_q, got_s = _call(case, no_alloc=True)
        assert torch.equal(got_q, want_q)
        assert torch.equal(got_s, want_s)
        assert not torch.isnan(got_s).any()


def test_noalloc_attention_refuses_more_sequences_than_its_scratch_holds():
    with pytest.raises(ValueError, match="a call takes at most 131072"):
        _hip.call("qh_attention_fp8_noalloc", None, 4096, 0, None, None, None, 1, None, 1,
                  PAGE, None, None, 131073, 1, 1, N_Q, N_KV, D, 0.1, 1, None, 4096, None, 0,
                  None)
