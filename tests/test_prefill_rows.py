"""Which rows a workgroup of the prefill attention has (ops/paged_prefill.py ``prefill_rows``)."""
import types

import pytest
import torch

from hcache_deepspeed_amd.ops import paged_prefill as P


@pytest.mark.parametrize("seqs,heads,rows", [
    ([(2048, 0)], 32, 128), ([(512, 789)], 32, 128), ([(16000, 0)], 16, 256), ([(256, 60)] * 4, 32, 128),
    ([(200, 60)] * 8, 32, 256), ([(200, 60)] * 16, 32, 256), ([(200, 60)] * 12, 32, 128),      # one, two and one and a half rounds
    ([(200, 150 * i) for i in range(8)], 32, 128), ([(128, 60)] * 16, 32, 128), ([(9, 1500)] * 24, 8, 128),
    ([(256, 60)] * 17, 32, 256)])
def test_rows_of_a_workgroup(seqs, heads, rows):
    assert P.prefill_rows(seqs, heads) == rows


def test_estimates_are_of_the_kernel_that_runs():
    """Lists of up to 512 workgroups: the faster of both; the longest workgroup, the load, whole rounds."""
    for seqs, heads in (([(2048, 0)], 32), ([(200, 60)] * 8, 32), ([(40, 3000)] * 16, 32)):
        assert P._many_us(seqs, heads) == P._launch_us(seqs, heads, P.prefill_rows(seqs, heads))
    assert P._many_us([(256, 0)] * 17, 32) == P._prefill_us([(256, 0)] * 17, 32)
    (a, b), (c, d) = P._WALK_US[128], P._WALK_US[256]
    assert P._launch_us([(256, 0)] * 8, 32, 256) == pytest.approx(c + d * 256)
    assert P._launch_us([(256, 0)] * 9, 32, 256) == pytest.approx(2 * (c + d * 256))
    assert P._launch_us([(1024, 0)], 1, 128) == pytest.approx(a + b * 1024)


def test_a_step_carries_its_rows(monkeypatch):
    """The batch hands the choice of its portions on to the kernel where there is one: not of single tokens, nor of lists whose
    length says it."""
    from hcache_deepspeed_amd.inference.v2 import build_engine_from_model
    from hcache_deepspeed_amd.models.llama import LlamaForCausalLM, tiny
    eng = build_engine_from_model(LlamaForCausalLM(tiny()).eval(), {"dtype": "fp32"}, device=torch.device("cpu"), num_kv_blocks=8)
    asked = []
    monkeypatch.setattr(P, "prefill_rows", lambda seqs, heads: asked.append(([tuple(s) for s in seqs], heads)) or 256)
    for heads, rows in ((128, 0), (130, 256), (256, 256)):
        eng._batch.set_attention_geometry(heads, 2, 128)
        eng.put([1, 2], [torch.arange(20) % 7, torch.arange(3)], capture_latents=False)
        assert eng._batch.prefill_rows == rows
        eng.flush(1), eng.flush(2)
    assert asked == [([(20, 0)], 130), ([(20, 0)], 256)]
    eng.put([1], [torch.arange(1)], capture_latents=False)
    assert eng._batch.prefill_rows == 0


def test_rows_reach_the_kernel(monkeypatch):
    calls = []
    lib = types.SimpleNamespace(hds_paged_prefill=lambda *a: calls.append(a) or 0)
    monkeypatch.setattr(P.native, "kernels", lambda: lib)
    monkeypatch.setattr(P.native, "stream", lambda: 0)
    t = torch.zeros(1, dtype=torch.int32)
    batch = types.SimpleNamespace(block_tables=t.view(1, 1), seq_meta=t)
    P.paged_attention_portions(torch.zeros(2, 1, 128), torch.zeros(1, 64, 2, 1, 128), None, t.view(-1, 1), batch, 1, 1, 1.0, rows=256)
    P.paged_attention_portions(torch.zeros(2, 1, 128), torch.zeros(1, 64, 2, 1, 128), None, t.view(-1, 1), batch, 1, 1, 1.0)
    assert [c[-2] for c in calls] == [256, 0]
