// Host-side ragged batch metadata for the inference-v2 (FastGen + HCache) engine, built in one pass into ONE
// int32 buffer (pinned by the caller) so a forward ships its whole batch description with a single H2D copy.
//
// Capability parity: reference inference/v2/ragged/csrc/ragged_ops.cpp (`RaggedBatchWrapper` finalize: the
// inflight sequence descriptors, token -> sequence map, KV block table) and
// inference/v2/kernels/ragged_ops/atom_builder/atom_builder.cpp:10-52 (`build_atoms`: one attention work item per
// (sequence, kv head, query-row chunk)). The reference runs them per forward in C++ for exactly the reason the
// Python versions were slow here: a decode step of B sequences is O(B * n_kv) small items per layer-forward.
//
// Layout of `out` (int32), S = n_seqs, T = sum(n_new), A = atoms:
//   [0, 3S)                 seq_meta  (q_start, n_new, seen) per sequence
//   [3S, 3S+T)              tok_seq   sequence index of every token
//   [3S+T, 3S+2T)           tok_pos   absolute position of every token (seen + i)
//   [3S+2T, 4S+2T)          last      index of each sequence's last token (logits rows)
//   [4S+2T, 4S+2T+S*MB)     tables    KV block ids per sequence, MB = max_blocks columns, zero padded
//   [..., + 3A)             atoms     (seq, kv_head, row_start) with rows = n_new * (n_q / n_kv) per (seq, kv head)
#include <cstdint>
#include <cstring>

#define HDS_EXPORT extern "C" __attribute__((visibility("default")))

namespace {

struct Seq {
  int32_t n_new, seen;
  const int32_t* blocks;
  int64_t n_blocks;
};

Seq seq_of(const int64_t* seqs, int s) {
  const int64_t* q = seqs + 5 * (int64_t)s;
  return Seq{(int32_t)q[1], (int32_t)q[2], reinterpret_cast<const int32_t*>(q[3]), q[4]};
}

struct Counts {
  int64_t tokens, atoms;
};

Counts count(const int64_t* seqs, int n_seqs, int n_q, int n_kv, int rows_per_atom) {
  Counts c{0, 0};
  for (int s = 0; s < n_seqs; ++s) {
    const int64_t n = seq_of(seqs, s).n_new;
    c.tokens += n;
    c.atoms += (int64_t)n_kv * ((n * (n_q / n_kv) + rows_per_atom - 1) / rows_per_atom);
  }
  return c;
}

void build(const int64_t* seqs, int n_seqs, int64_t T, int max_blocks, int n_q, int n_kv, int rows_per_atom, int32_t* out) {
  const int G = n_q / n_kv;
  int32_t* meta = out;
  int32_t* tok_seq = meta + 3LL * n_seqs;
  int32_t* tok_pos = tok_seq + T;
  int32_t* last = tok_pos + T;
  int32_t* tables = last + n_seqs;
  int32_t* atoms = tables + (int64_t)n_seqs * max_blocks;
  int64_t q0 = 0, a = 0;
  for (int s = 0; s < n_seqs; ++s) {
    const Seq q = seq_of(seqs, s);
    const int32_t n = q.n_new, sn = q.seen;
    meta[3 * s] = (int32_t)q0;
    meta[3 * s + 1] = n;
    meta[3 * s + 2] = sn;
    for (int32_t i = 0; i < n; ++i) {
      tok_seq[q0 + i] = s;
      tok_pos[q0 + i] = sn + i;
    }
    last[s] = (int32_t)(q0 + (n > 0 ? n - 1 : 0));
    int32_t* row = tables + (int64_t)s * max_blocks;
    const int64_t ncopy = q.n_blocks < max_blocks ? q.n_blocks : max_blocks;
    if (ncopy > 0) std::memcpy(row, q.blocks, sizeof(int32_t) * ncopy);
    if (ncopy < max_blocks) std::memset(row + ncopy, 0, sizeof(int32_t) * (max_blocks - ncopy));
    const int64_t rows = (int64_t)n * G;
    for (int hk = 0; hk < n_kv; ++hk)
      for (int64_t r0 = 0; r0 < rows; r0 += rows_per_atom) {
        atoms[3 * a] = s;
        atoms[3 * a + 1] = hk;
        atoms[3 * a + 2] = (int32_t)r0;
        ++a;
      }
    q0 += n;
  }
}

}  // namespace

// A whole step in one call, from the sequences' own buffers: the 64-bit token ids, the layout above and `n_extra` further values
// go to `out` (8-byte aligned) one behind the other. seqs [n_seqs][5]: address of the tokens (int64), their number, tokens
// seen, address of the KV blocks (int32), their number. id_limit: ids must lie in [0, id_limit) (0: any). info: ints needed,
// smallest and largest id. Returns the number of atoms; -1 when `cap` is too small (nothing is written), -3 with an id outside.
HDS_EXPORT int64_t hds_ragged_step_build(const int64_t* seqs, int n_seqs, int max_blocks, int n_q, int n_kv,
                                         int rows_per_atom, int64_t id_limit, const int32_t* extra, int64_t n_extra,
                                         int32_t* out, int64_t cap, int64_t* info) {
  if (n_seqs < 0 || n_kv <= 0 || n_q % n_kv != 0 || rows_per_atom <= 0 || max_blocks < 0 || n_extra < 0) return -2;
  const Counts c = count(seqs, n_seqs, n_q, n_kv, rows_per_atom);
  const int64_t size = 4LL * n_seqs + 2 * c.tokens + (int64_t)n_seqs * max_blocks + 3 * c.atoms;
  info[0] = 2 * c.tokens + size + n_extra;
  if (info[0] > cap) return -1;
  int64_t* ids = reinterpret_cast<int64_t*>(out);
  int64_t lo = INT64_MAX, hi = INT64_MIN;
  for (int s = 0; s < n_seqs; ++s) {
    const int64_t* t = reinterpret_cast<const int64_t*>(seqs[5 * (int64_t)s]);
    const int64_t n = seqs[5 * (int64_t)s + 1];
    for (int64_t i = 0; i < n; ++i) {
      lo = t[i] < lo ? t[i] : lo;
      hi = t[i] > hi ? t[i] : hi;
      *ids++ = t[i];
    }
  }
  info[1] = lo;
  info[2] = hi;
  if (c.tokens > 0 && id_limit > 0 && (lo < 0 || hi >= id_limit)) return -3;
  int32_t* meta = out + 2 * c.tokens;
  build(seqs, n_seqs, c.tokens, max_blocks, n_q, n_kv, rows_per_atom, meta);
  if (n_extra > 0) std::memcpy(meta + size, extra, sizeof(int32_t) * (size_t)n_extra);
  return c.atoms;
}
