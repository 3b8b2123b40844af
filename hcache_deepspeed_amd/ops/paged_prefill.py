"""Serving steps with more than single tokens: portions of prompts on the FlashAttention kernels over block tables
(csrc/kernels/flash_attn_pair.hip, flash_attn_w64.hip) or in row blocks, single tokens on the split-key kernel (both
csrc/kernels/paged_attn.hip)."""
import torch

from . import native
from .paged import DECODE_MAX, ROWS_PER_ATOM

# new tokens of an entry of the prefill kernels' list: one workgroup a head, or two of half the rows (``prefill_rows``)
PREFILL_ROWS = 256


def make_portions(seq_meta_host, portions=None):
    """How a step with more than single tokens is divided: (rows of the tokens that run one by one, flat list of (sequence,
    first new token) of the prefill kernel's workgroups, those that see the most keys first). ``portions``: the sequences
    that run on it (default: those of more than ``DECODE_MAX`` new tokens)."""
    toks, blocks = [], []
    for s, (q0, n, seen) in enumerate(seq_meta_host):
        if n <= DECODE_MAX if portions is None else s not in portions:
            toks += range(q0, q0 + n)
        else:
            blocks += [(seen + min(r + PREFILL_ROWS, n), s, r) for r in range(0, n, PREFILL_ROWS)]
    blocks.sort(reverse=True)
    return toks, [v for b in blocks for v in b[1:]]


# Microseconds of the kernels, fitted to 1 to 64 sequences of 2 to 256 new tokens behind 60 to 4,000 earlier ones, 8 / 1 to 64 / 8
# and 32 / 32 heads (within a fifth, at least about the lines between them). Prefill kernel and row blocks: the longest
# workgroup, or all of them over the CUs (256 at a time, by 256 rows; of the row blocks about 270). One by one: the contexts
# are read from memory once, from the caches once a token.
def _prefill_us(seqs, heads):
    longest = max(7 + 0.031 * (seen + n) for n, seen in seqs)
    return max(longest, heads / 256 * sum(-(-n // PREFILL_ROWS) * (7 + 0.031 * (seen + n / 2)) for n, seen in seqs))


# The prefill kernels on lists of up to so many workgroups of 256 rows, by the rows of a workgroup: us of one, and a key (of 1,736
# lists of 9 to 2,048 new tokens, 4 / 4 to 32 / 32 heads, 130 to 512 workgroups: 13 % rms)
SHORT_LIST = 512
_WALK_US = {128: (7.5, 0.0145), 256: (8.5, 0.033)}


def _launch_us(seqs, heads, rows):
    """The longest workgroup, all of them over the CUs, or the rounds of 256 that workgroups of much the same length take."""
    us, per_key = _WALK_US[rows]
    last = []  # the workgroups' last keys
    for n, seen in seqs:
        last.append(seen + n)
        last += range(seen + (n - 1) // rows * rows, seen, -rows)
    last.sort(reverse=True)
    rounds = max((k + 1) * (us + per_key * last[256 * k // heads]) for k in range((heads * len(last) - 1) // 256 + 1))
    return max(rounds, heads / 256 * (us * len(last) + per_key * sum(last)))


def prefill_rows(seqs, heads):
    """Rows of a workgroup of the prefill kernel for these (new, earlier) tokens, 128 (csrc/kernels/flash_attn_pair.hip) or 256
    (flash_attn_w64.hip). Half of the rows take half of the time in twice the workgroups: where those of 256 fill the chip
    in whole rounds, twice as many rounds of 128 take as long and longer (8 sequences of 200 tokens behind 60, 32 / 8 heads
    23.0 us by 128 rows, 20.8 by 256; 16 43.2 and 38.8), unless lengths differ (8 behind up to 1,500 44 and 61) or the second
    halves are empty (16 of 64 behind 500 30 and 44). Over 1,736 lists of 130 to 512 workgroups 0.77 of the time of 256 rows, at
    most 1.07; with 128 rows for all of them 0.78 and 1.27 (profiles/main_paths/prefill_rows.txt)."""
    blocks = heads * sum(-(-n // PREFILL_ROWS) for n, _ in seqs)
    if blocks > SHORT_LIST:
        return 256
    if 2 * blocks <= 256 or max(n for n, _ in seqs) <= 128:  # (no question: 128 rows are the faster ones)
        return 128
    return 128 if _launch_us(seqs, heads, 128) <= _launch_us(seqs, heads, 256) else 256


def _rows_us(seqs, heads, kv_heads):
    G, R = heads // kv_heads, ROWS_PER_ATOM
    longest = max(4 + 0.05 * (seen + n) for n, seen in seqs)
    return max(longest, kv_heads / 270 * sum(-(-n * G // R) * (2.5 + 4.5 * min(1, n * G / R) + 0.05 * (seen + n / 2))
                                             for n, seen in seqs))


def _tokens_us(seqs, kv_heads):
    return 6 + kv_heads * sum((seen + n) * (6e-5 + 3.8e-5 * n) + 6e-3 * n for n, seen in seqs)


def _many_us(seqs, heads):
    """``_prefill_us``, of short lists by the rows that they run with: of 257 to 512 workgroups the division by it is 0.4 % slower
    than the better of both (at most 1.16 of its time), by the estimate of 256 rows 5.6 % (2.25)."""
    rows = prefill_rows(seqs, heads)
    short = heads * sum(-(-n // PREFILL_ROWS) for n, _ in seqs) <= SHORT_LIST
    return _launch_us(seqs, heads, rows) if short else _prefill_us(seqs, heads)


def divide_step(seq_meta_host, heads, kv_heads):
    """``make_portions`` for these head counts, and flat list of (sequence, kv head, first row) of the sequences that run in
    row blocks: (tokens, blocks, atoms). Two cases leave ``make_portions``'s division:

    * many portions of few tokens: the prefill kernel has a workgroup a query head for each of them, 256 at a time, row
      blocks have one a key head (32 sequences of 16 tokens, up to 4,000 keys, 32 / 8 heads: 331 us against 226; 16
      sequences 76 / 206, up to 60 keys 16 / 10);
    * many sequences of 2 to ``DECODE_MAX`` tokens, whose contexts are read once a token: 32 of 8 tokens there 237 us
      against 221 in row blocks, up to 1,000 keys 69 / 58, up to 300 34 / 20; of 4 tokens 155 / 224, 41 / 57, 20 / 20.

    Beside row blocks single tokens join them where that takes less than a launch of their own (32 of them and 32 sequences
    of 8 tokens, up to 2,000 keys: 161 us apart, 129 together)."""
    short = blocks = 0
    for _, n, _ in seq_meta_host:
        if n > DECODE_MAX:
            blocks += -(-n // PREFILL_ROWS)
        elif n > 1:
            short += n
    if kv_heads * short <= 512 and heads * blocks <= 256:  # neither case (8 us of host time a step otherwise, 4 so)
        return (*make_portions(seq_meta_host), [])
    new = {s: (n, seen) for s, (_, n, seen) in enumerate(seq_meta_host) if n}
    ones = [s for s, (n, _) in new.items() if n == 1]
    few = [s for s, (n, _) in new.items() if 1 < n <= DECODE_MAX]
    many = [s for s, (n, _) in new.items() if n > DECODE_MAX]
    of = lambda which: [new[s] for s in which]  # noqa: E731
    best = lambda which: min(_prefill_us(of(which), heads), _rows_us(of(which), heads, kv_heads)) if which else 0  # noqa: E731
    if kv_heads * sum(new[s][0] for s in few) > 512 and _tokens_us(of(few), kv_heads) > best(few + many) - best(many):
        few, many = [], few + many
    if heads * sum(-(-new[s][0] // PREFILL_ROWS) for s in many) <= 256 or \
            _many_us(of(many), heads) <= _rows_us(of(many), heads, kv_heads):
        return (*make_portions(seq_meta_host, set(many)), [])
    if ones and _tokens_us(of(ones), kv_heads) > _rows_us(of(ones + many), heads, kv_heads) - _rows_us(of(many), heads, kv_heads):
        many = many + ones
    G, gone = heads // kv_heads, set(many)
    toks = [t for s, (q0, n, _) in enumerate(seq_meta_host) if s not in gone for t in range(q0, q0 + n)]
    atoms = []
    for s in sorted(many, key=lambda s: -sum(new[s])):  # those that see the most keys first
        for r in range(0, new[s][0] * G, ROWS_PER_ATOM)[::-1]:
            for h in range(kv_heads):
                atoms += (s, h, r)
    return toks, [], atoms


def portions_ok(q, cache, n_q, n_kv, scale=1.0):
    """Does the prefill kernel take these heads, this cache and this scale (it keeps the maximum of the raw scores, so a positive
    one; row blocks take any)?"""
    return (2**-64 <= scale <= 2**64 and native.use_native(q) and q.dtype == torch.bfloat16 and cache.dtype == q.dtype and cache.dim() == 5
            and q.shape[2] == 128 and cache.is_contiguous() and cache.shape[1] % 64 == 0 and n_q % n_kv == 0
            and cache.shape[0] * cache.shape[1] < 2**31 and cache.stride(0) // cache.shape[1] <= 2**23
            and q.stride(0) % 8 == 0 and q.stride(1) == 128 and q.data_ptr() % 16 == 0)


def paged_attention_portions(q, cache, toks, blocks, batch, n_q, n_kv, scale, window=0, atoms=None, rows=0):
    """``paged_attention`` of a step that mixes single tokens and portions of prompts: ``toks`` (int32 rows of q) on the
    split-key kernel, which spreads a token's context over the chip, ``blocks`` ([n, 2] int32) on the prefill kernel by ``rows``
    (``prefill_rows``; 0: by the length of the list), ``atoms`` ([n, 3] int32) in row blocks. There a single token walks its
    whole context in one workgroup (9 such tokens, up to 3,000 keys, 8 key heads, beside 512 new ones: 171 us; apart 29 + 38
    us)."""
    T, _, D = q.shape
    o = torch.empty(T, n_q, D, device=q.device, dtype=q.dtype)
    lib, st, tab = native.kernels(), native.stream(), batch.block_tables
    mb, bs = tab.shape[1], cache.shape[1]
    n = 0 if toks is None else toks.numel()
    if n:
        keys = mb * bs
        splits = lib.hds_paged_decode_splits(n, n_kv, min(keys, window) if window else keys)
        part_o = part_ml = None
        if splits > 1:
            part_o = torch.empty(n * n_q * splits * D, device=q.device, dtype=torch.float32)
            part_ml = torch.empty(n * n_q * splits * 2, device=q.device, dtype=torch.float32)
        native.check(
            lib.hds_paged_decode(native.dt(q), 0, q.data_ptr(), q.stride(0), cache.data_ptr(), o.data_ptr(), n_q * D,
                                 native.ptr(part_o), native.ptr(part_ml), None, toks.data_ptr(),
                                 batch.tok_seq.data_ptr(), batch.tok_pos.data_ptr(), tab.data_ptr(), mb, bs, n, n_q,
                                 n_kv, D, D, splits, float(scale), int(window), 0, 0, 0.0, None, None, 0, 1, None, st),
            "paged_decode")
    if blocks is not None and blocks.shape[0]:
        native.check(
            lib.hds_paged_prefill(q.data_ptr(), q.stride(0), cache.data_ptr(), o.data_ptr(), n_q * D,
                                  blocks.data_ptr(), blocks.shape[0], batch.seq_meta.data_ptr(), tab.data_ptr(), mb, bs,
                                  n_q, n_kv, float(scale), int(window), int(rows), st), "paged_prefill")
    if atoms is not None and atoms.shape[0]:
        native.check(
            lib.hds_paged_attn(q.data_ptr(), q.stride(0), cache.data_ptr(), o.data_ptr(), n_q * D, atoms.data_ptr(),
                               atoms.shape[0], batch.seq_meta.data_ptr(), tab.data_ptr(), mb, bs, n_q, n_kv, D, D,
                               float(scale), int(window), 0, 0, 0.0, None, None, 0, 1, st), "paged_attn")
    return o
