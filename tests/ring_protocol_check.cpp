// Host-side replay of the ring kernels' tile pipeline (no GPU): built and run by tests/test_ring_protocol.py.
//
// For a protocol (sample_efficient_gpt_amd/csrc/ring_protocol.hpp: the numbers the kernels themselves compile in) and
// a tile count, the order of operations ONE wave executes is generated in the kernels' control flow:
//   requests of tiles / row blocks (direct global->LDS loads, `loads` vector-memory operations each),
//   s_waitcnt vmcnt(N), workgroup barriers, fragment reads of a stage.
// All waves of a workgroup run the same order and each loads its quarter of every tile, so the replay keeps one
// symbolic wave plus the count of barriers passed ("epoch"):
//   - vector memory retires in order: a wait with immediate N retires everything but the youngest N operations;
//   - a read of a stage in epoch e is safe iff the stage holds the expected content and ALL of that content's loads
//     were retired by a wait in an epoch < e (every wave waited for its own quarter before a barrier that the reader
//     has passed);
//   - a request that refills a stage in epoch e is safe iff the last read of the stage's previous content happened
//     in an epoch < e (a barrier separates the slowest reader from the first new byte) and that content had landed; content
//     that nobody read must have been retired in an epoch < e (every wave's part of it).
// Exit code 0 and "ok" per line when everything holds; the deliberately broken protocols at the end must each be
// reported as a violation, or the program fails: a checker that cannot see the known bug proves nothing.
#include <cstdio>
#include <cstring>
#include <string>
#include <vector>

#include "ring_protocol.hpp"

using segpt::ring::Protocol;

namespace {

enum Kind { REQUEST, WAIT, BARRIER, READ };
struct Op {
  Kind kind;
  int stage;    // REQUEST / READ
  int content;  // REQUEST / READ: tile index >= 0, kRows, kPreRows, kEpilogueRows, kSlots or kScratch
  int n;        // REQUEST: loads issued by the wave (0: plain LDS stores, e.g. the epilogue's scratch); WAIT: the vmcnt immediate
};
constexpr int kRows = -1, kPreRows = -3, kEpilogueRows = -5, kScratch = -4, kSlots = -6;

// The order of operations of one wave, following fwd_mfma.hip / bwd_mfma.hip:
//   [first start-up phase: row blocks in stages 0 .., wait for everything, barrier, rows -> registers, barrier;]
//   start-up: early tiles, row blocks, wait for everything, barrier, rows -> registers, barrier, late tiles,
//             [wait + barrier], fragment request of tile 0;
//   iteration jt: [request at top], blocks of tile jt (its stage; the second block also requests the row-major
//             fragments of tile jt+1 from the NEXT stage), [request at bottom], wait, barrier;
//   [behind the loop: `epilogue_rows` row blocks (at most p.epilogue_row_stages) requested into stages 0 .., beside them the
//    accumulators that two waves hand over (plain stores), wait for everything, barrier, rows and hand-over -> registers,
//    barrier if there were rows, scratch stores over the ring; dQ reads the hand-over only behind that second barrier].
std::vector<Op> wave_program(const Protocol& p, int n_tiles, int row_loads_per_stage, int epilogue_rows = 0) {
  std::vector<Op> ops;
  auto request_tile = [&](int t) { ops.push_back({REQUEST, t % p.stages, t, p.loads_per_tile}); };
  if (p.pre_row_stages > 0) {
    for (int i = 0; i < p.pre_row_stages; ++i) ops.push_back({REQUEST, i, kPreRows, row_loads_per_stage});
    ops.push_back({WAIT, 0, 0, 0});
    ops.push_back({BARRIER, 0, 0, 0});
    for (int i = 0; i < p.pre_row_stages; ++i) ops.push_back({READ, i, kPreRows, 0});
    ops.push_back({BARRIER, 0, 0, 0});
  }
  for (int t = 0; t < p.early_tiles; ++t)
    if (t < n_tiles) request_tile(t);
  for (int i = 0; i < p.row_stages; ++i) ops.push_back({REQUEST, p.row_stage_first + i, kRows, row_loads_per_stage});
  ops.push_back({WAIT, 0, 0, 0});
  ops.push_back({BARRIER, 0, 0, 0});
  for (int i = 0; i < p.row_stages; ++i) ops.push_back({READ, p.row_stage_first + i, kRows, 0});
  ops.push_back({BARRIER, 0, 0, 0});
  for (int t = p.early_tiles; t < p.startup_tiles; ++t)
    if (t < n_tiles) request_tile(t);
  if (p.wait_before_loop) {
    const int keep = n_tiles >= p.startup_tiles ? segpt::ring::loads_kept_before_loop(p, p.startup_tiles) : 0;
    ops.push_back({WAIT, 0, 0, keep});
    ops.push_back({BARRIER, 0, 0, 0});
  }
  if (n_tiles > 0) ops.push_back({READ, 0, 0, 0});  // row-major fragments of the first block
  for (int jt = 0; jt < n_tiles; ++jt) {
    const bool requested = p.always_requests || jt + p.issue_ahead < n_tiles;  // past the end: a tile nobody reads
    if (p.issue_at_top && requested) request_tile(jt + p.issue_ahead);
    ops.push_back({READ, jt % p.stages, jt, 0});                                      // both blocks, both orientations
    if (jt + 1 < n_tiles) ops.push_back({READ, (jt + 1) % p.stages, jt + 1, 0});      // next tile's first fragments
    if (!p.issue_at_top && requested) request_tile(jt + p.issue_ahead);
    ops.push_back({WAIT, 0, 0, segpt::ring::loads_kept_after_iteration(p, requested)});
    ops.push_back({BARRIER, 0, 0, 0});
  }
  if (p.always_requests) {
    ops.push_back({WAIT, 0, 0, 0});
    ops.push_back({BARRIER, 0, 0, 0});
  }
  const int slots_end = p.merge_stage_first + p.merge_stages;
  for (int i = p.merge_stage_first; i < slots_end; ++i) ops.push_back({REQUEST, i, kSlots, 0});
  for (int i = 0; i < epilogue_rows; ++i) ops.push_back({REQUEST, i, kEpilogueRows, row_loads_per_stage});
  if (epilogue_rows > 0 || p.merge_stages > 0) {
    ops.push_back({WAIT, 0, 0, 0});
    ops.push_back({BARRIER, 0, 0, 0});
  }
  for (int i = 0; i < epilogue_rows; ++i) ops.push_back({READ, i, kEpilogueRows, 0});
  if (epilogue_rows > 0 && p.epilogue_reuses_ring) ops.push_back({BARRIER, 0, 0, 0});
  for (int i = p.merge_stage_first; i < slots_end; ++i) ops.push_back({READ, i, kSlots, 0});
  if (p.epilogue_reuses_ring)
    for (int i = 0; i < (p.scratch_stages ? p.scratch_stages : p.stages); ++i) ops.push_back({REQUEST, i, kScratch, 0});
  return ops;
}

// returns "" or the first violation
std::string replay(const Protocol& p, const std::vector<Op>& ops) {
  struct Load { int stage, content; };
  struct StageState { int content = -2; int loads_pending = 0; int retired_epoch = -1; int last_read_epoch = -1; bool ever = false; };
  std::vector<StageState> st(p.stages);
  std::vector<Load> queue;  // this wave's vector-memory operations still in flight, oldest first
  int epoch = 0;
  char buf[256];
  for (size_t i = 0; i < ops.size(); ++i) {
    const Op& o = ops[i];
    switch (o.kind) {
      case REQUEST: {
        if (o.stage < 0 || o.stage >= p.stages) return "request outside the ring";
        StageState& s = st[o.stage];
        if (s.ever) {
          if (s.loads_pending > 0) {
            snprintf(buf, sizeof buf, "op %zu: stage %d refilled with content %d while content %d is still in flight", i, o.stage, o.content, s.content);
            return buf;
          }
          if (s.last_read_epoch < 0 && s.retired_epoch >= epoch) {  // never read: nothing else says that the other waves' parts have landed
            snprintf(buf, sizeof buf, "op %zu: stage %d refilled with content %d in the epoch of this wave's wait for content %d (no barrier in between)", i, o.stage, o.content, s.content);
            return buf;
          }
          if (s.last_read_epoch >= epoch) {
            snprintf(buf, sizeof buf, "op %zu: stage %d refilled with content %d in the epoch of the last read of content %d (no barrier in between)", i, o.stage, o.content, s.content);
            return buf;
          }
        }
        s.content = o.content; s.loads_pending = o.n; s.retired_epoch = o.n == 0 ? epoch : -1; s.last_read_epoch = -1; s.ever = true;
        for (int k = 0; k < o.n; ++k) queue.push_back({o.stage, o.content});
        break;
      }
      case WAIT: {
        while ((int)queue.size() > o.n) {
          const Load l = queue.front();
          queue.erase(queue.begin());
          StageState& s = st[l.stage];
          if (s.content == l.content && s.loads_pending > 0 && --s.loads_pending == 0) s.retired_epoch = epoch;
        }
        break;
      }
      case BARRIER: ++epoch; break;
      case READ: {
        StageState& s = st[o.stage];
        if (!s.ever || s.content != o.content) {
          snprintf(buf, sizeof buf, "op %zu: read of content %d from stage %d, which holds content %d", i, o.content, o.stage, s.content);
          return buf;
        }
        if (s.loads_pending > 0 || s.retired_epoch < 0 || s.retired_epoch >= epoch) {
          snprintf(buf, sizeof buf, "op %zu: read of content %d (stage %d) before it has landed and been published (pending loads %d, waited in epoch %d, read in epoch %d)",
                   i, o.content, o.stage, s.loads_pending, s.retired_epoch, epoch);
          return buf;
        }
        s.last_read_epoch = epoch;
        break;
      }
    }
  }
  return "";
}

// every streamed-tile count from min_tiles on, with every count of epilogue row blocks the protocol allows
std::string check(const Protocol& p, int max_tiles, int min_tiles = 1) {
  if (!segpt::ring::well_formed(p)) return "not well formed";
  for (int rows = 0; rows <= p.epilogue_row_stages; ++rows)
    for (int n = min_tiles; n <= max_tiles; ++n) {
      const std::string v = replay(p, wave_program(p, n, 2 * p.loads_per_tile, rows));
      if (!v.empty()) return "n_tiles " + std::to_string(n) + " + " + std::to_string(rows) + " epilogue row blocks: " + v;
    }
  return "";
}

// ---- the split-key decode kernel (decode_mfma.hip).  Buffers: the K, V and V_first rows of a block are a wave's own, the table
// rows (two buffers) the workgroup's.  A private buffer is readable once its loads were retired by a wait and may be requested
// over once the reads of it have returned (LDS_DONE); a shared one follows the rules of a stage above.
enum DecodeBuffer { TAB0, TAB1, KBUF, VBUF, FBUF, kDecodeBuffers };
constexpr Kind LDS_DONE = (Kind)(READ + 1);

// `reads`: false for a wave of the last workgroup without a (batch, kv head) pair, which only brings its pieces of the tables;
// reading them stands for what the other waves do with those pieces
std::vector<Op> decode_program(const segpt::ring::DecodeLoads& d, int n_blocks, bool reads) {
  std::vector<Op> ops;
  auto request = [&](int buffer, int block, int loads) { if (loads) ops.push_back({REQUEST, buffer, block, loads}); };
  if (n_blocks > 0) {
    request(TAB0, 0, d.tables);
    if (reads) { request(KBUF, 0, d.rows); request(VBUF, 0, d.rows); request(FBUF, 0, d.first); }
  }
  ops.push_back({WAIT, 0, 0, 0});
  for (int n = 0; n < n_blocks; ++n) {
    const bool more = n + 1 < n_blocks;
    ops.push_back({WAIT, 0, 0, reads ? segpt::ring::decode_kept_at_top(d) : 0});
    if (d.tables) {
      ops.push_back({BARRIER, 0, 0, 0});
      if (more) request(TAB0 + (n + 1) % 2, n + 1, d.tables);
      ops.push_back({READ, TAB0 + n % 2, n, 0});
    }
    if (reads) {
      ops.push_back({READ, KBUF, n, 0});
      ops.push_back({LDS_DONE, 0, 0, 0});
      if (more) request(KBUF, n + 1, d.rows);
      ops.push_back({WAIT, 0, 0, segpt::ring::decode_kept_before_v(d, more)});
      ops.push_back({READ, VBUF, n, 0});
      if (d.first) ops.push_back({READ, FBUF, n, 0});
      ops.push_back({LDS_DONE, 0, 0, 0});
      if (more) { request(VBUF, n + 1, d.rows); request(FBUF, n + 1, d.first); }
    }
  }
  return ops;
}

std::string replay_decode(const std::vector<Op>& ops) {
  struct State { int content = -2, pending = 0, retired_epoch = -1, read_epoch = -1; bool read_open = false; } st[kDecodeBuffers];
  std::vector<std::pair<int, int>> queue;  // (buffer, content), oldest first
  int epoch = 0;
  for (size_t i = 0; i < ops.size(); ++i) {
    const Op& o = ops[i];
    const std::string at = "op " + std::to_string(i) + ": buffer " + std::to_string(o.stage) + ", block " + std::to_string(o.content) + ": ";
    const bool shared = o.stage <= TAB1;
    State& s = st[o.stage];
    if (o.kind == REQUEST) {
      if (s.pending > 0) return at + "requested over a block in flight";
      if (shared ? s.read_epoch >= epoch : s.read_open) return at + "requested over a block that may still be read";
      s = State{};
      s.content = o.content; s.pending = o.n;
      for (int k = 0; k < o.n; ++k) queue.push_back({o.stage, o.content});
    } else if (o.kind == WAIT) {
      while ((int)queue.size() > o.n) {
        State& r = st[queue.front().first];
        queue.erase(queue.begin());
        if (--r.pending == 0) r.retired_epoch = epoch;
      }
    } else if (o.kind == BARRIER) {
      ++epoch;
    } else if (o.kind == LDS_DONE) {
      for (State& b : st) b.read_open = false;
    } else {
      if (s.content != o.content) return at + "read while the buffer holds block " + std::to_string(s.content);
      if (s.pending > 0 || (shared && s.retired_epoch >= epoch)) return at + "read before it has landed and been published";
      s.read_epoch = epoch;
      s.read_open = true;
    }
  }
  return "";
}

}  // namespace

int main() {
  using namespace segpt::ring;
  struct Named { const char* name; Protocol p; };
  int failures = 0;
  // wave-wide 16-byte loads per wave and [64, D] tile: 2 at head_dim 64, 4 at head_dim 128
  for (const int passes : {2, 4}) {
    const Named shipped[] = {
        {"forward, 32 rows per wave (3 stages; head_dim 64 up to 2048 keys, head_dim 128)", forward(3, 1, passes)},
        {"forward, 64 rows per wave (4 stages; head_dim 64 beyond 2048 keys)", forward(4, 2, passes)},
        {"dQ", dq(passes, false)},
        {"dQ with a rotary embedding (two start-up phases, table rows once more behind the loop)", dq_rope(passes, false)},
        {"dK/dV (k, v, v_first rows behind the loop; a key tile may see no query at all)", dkdv(passes, false)},
        {"dQ requesting a tile in every iteration", dq(passes, true)},
        {"dQ with a rotary embedding requesting a tile in every iteration", dq_rope(passes, true)},
        {"dK/dV requesting a tile in every iteration", dkdv(passes, true)},
    };
    for (const Named& k : shipped) {
      const bool can_be_empty = k.p.loads_per_tile == 2 * passes + 1;  // dK/dV: key tiles beyond every query
      const std::string v = check(k.p, 70, can_be_empty ? 0 : 1);
      printf("passes %d  %-82s %s\n", passes, k.name, v.empty() ? "ok" : ("VIOLATION: " + v).c_str());
      failures += !v.empty();
    }
  }
  // 64-row workgroups: a 64-key tile at either head size, two waves per row block
  for (const int passes : {2, 4}) {
    const Named shipped[] = {
        {"forward, two waves per row block", forward_parts(3, 1, passes)},
        {"dQ, two waves per row block", dq_parts(passes)},
        {"dQ with a rotary embedding, two waves per row block", dq_rope_parts(passes)},
        {"dK/dV, two waves per key block", dkdv_parts(passes)},
    };
    for (const Named& k : shipped) {
      const std::string v = check(k.p, 70, k.p.loads_per_tile == 2 * passes + 1 ? 0 : 1);
      printf("passes %d  %-82s %s\n", passes, k.name, v.empty() ? "ok" : ("VIOLATION: " + v).c_str());
      failures += !v.empty();
    }
  }
  // decode: a wave loads the 32 rows of a block in 4 (head_dim 64) or 8 accesses, its quarter of a pair of table tiles in 2 or 4
  for (const int rows : {4, 8})
    for (const int tables : {0, rows / 2})
      for (const int first : {0, rows}) {
        const DecodeLoads d{tables, rows, first};
        std::string v;
        for (int n = 0; n <= 40 && v.empty(); ++n)
          for (const bool reads : {true, false})
            if (v.empty()) v = replay_decode(decode_program(d, n, reads));
        printf("decode: %d loads per tensor, %d of tables, %d of the value residual %34s\n", rows, tables, first, v.empty() ? "ok" : ("VIOLATION: " + v).c_str());
        failures += !v.empty();
      }
  const int passes = 2;
  // Other ring depths and borrowed-stage layouts the formulas claim to cover (not shipped): must hold as well.
  for (int stages = 3; stages <= 6; ++stages)
    for (int q_stages = 1; q_stages <= stages - 2; ++q_stages) {
      const std::string v = check(forward(stages, q_stages, passes), 40);
      if (!v.empty()) { printf("forward(%d stages, %d row stages): VIOLATION: %s\n", stages, q_stages, v.c_str()); ++failures; }
    }

  // ---- protocols that are wrong on purpose: each must be caught
  struct Broken { const char* name; Protocol p; };
  Protocol dq_no_wait[2], dq_keep2[2], dkdv_ahead4[2];
  for (const bool always : {false, true}) {
    dq_no_wait[always] = dq_keep2[always] = dq(passes, always);
    dkdv_ahead4[always] = dkdv(passes, always);
    dq_no_wait[always].wait_before_loop = false;  // the start-up that shipped once: tile 1, a late request, not awaited before iteration 0
    dq_keep2[always].keep_tiles = 2;              // the iteration's wait leaves the tile in flight that the next iteration prefetches from
    dkdv_ahead4[always].issue_ahead = 4;          // refills the stage the iteration has just read, before the barrier
  }
  Protocol fwd_early_into_rows = forward(4, 2, passes);
  fwd_early_into_rows.early_tiles = 3;  // an early tile lands in a stage the query rows borrow
  const Broken broken[] = {
      {"dQ without the wait before the loop", dq_no_wait[0]},
      {"dQ leaving two tiles in flight per iteration", dq_keep2[0]},
      {"dK/dV requesting four tiles ahead in a ring of four", dkdv_ahead4[0]},
      {"dQ, always requesting, without the wait before the loop", dq_no_wait[1]},
      {"dQ, always requesting, leaving two tiles in flight per iteration", dq_keep2[1]},
      {"dK/dV, always requesting, four tiles ahead in a ring of four", dkdv_ahead4[1]},
      {"forward with an early tile in a borrowed stage", fwd_early_into_rows},
  };
  for (const Broken& k : broken) {
    const std::string v = replay(k.p, wave_program(k.p, 12, 2 * k.p.loads_per_tile));
    printf("%-93s %s\n", k.name, v.empty() ? "NOT CAUGHT" : ("caught: " + v).c_str());
    failures += v.empty();
  }
  for (const bool always : {false, true}) {  // a vmcnt unit larger than what a wave really issues per tile (say the statistics
     // load was dropped from the kernel but not from the count): the iteration's wait then leaves part of the next tile in flight
    const Protocol p = dkdv(passes, always);
    std::vector<Op> ops = wave_program(p, 12, 2 * p.loads_per_tile);
    for (Op& o : ops)
      if (o.kind == REQUEST && o.content >= 0) o.n = p.loads_per_tile - 1;
    const std::string v = replay(p, ops);
    printf("%-82s %s\n", "dK/dV counting five loads per tile while issuing four", v.empty() ? "NOT CAUGHT" : ("caught: " + v).c_str());
    failures += v.empty();
  }
  // ---- the row blocks around the loop, broken by leaving out one barrier or wait of the generated order
  auto drop = [](std::vector<Op> ops, Kind kind, int which_from_end) {  // removes the which-th last op of a kind
    for (int i = (int)ops.size() - 1; i >= 0; --i)
      if (ops[i].kind == kind && which_from_end-- == 0) { ops.erase(ops.begin() + i); break; }
    return ops;
  };
  auto drop_nth = [](std::vector<Op> ops, Kind kind, int which) {        // removes the which-th op of a kind
    for (size_t i = 0; i < ops.size(); ++i)
      if (ops[i].kind == kind && which-- == 0) { ops.erase(ops.begin() + i); break; }
    return ops;
  };
  struct BrokenOps { const char* name; Protocol p; std::vector<Op> ops; };
  const Protocol dr = dq_rope(passes, false), dk = dkdv(passes, false), da = dq(passes, true), ka = dkdv(passes, true);
  const int iterations = 12;
  // an iteration that requested nothing waits as if it had: the tail of the loop reads tiles that are still in flight
  std::vector<Op> keeping = wave_program(dk, iterations, 2 * dk.loads_per_tile);
  for (size_t i = keeping.size(), left = (size_t)dk.issue_ahead; i-- > 0 && left > 0;)
    if (keeping[i].kind == WAIT) { keeping[i].n = dk.keep_tiles * dk.loads_per_tile; --left; }
  const BrokenOps broken_ops[] = {
      {"dK/dV reading its epilogue row blocks without the wait behind their requests", dk,
       drop(wave_program(dk, 12, 2 * dk.loads_per_tile, 3), WAIT, 0)},
      {"dK/dV reading its epilogue row blocks without the barrier behind the wait", dk,
       drop(wave_program(dk, 12, 2 * dk.loads_per_tile, 3), BARRIER, 0)},
      {"dQ (rotary) requesting the second start-up phase without the barrier behind the first phase's reads", dr,
       drop_nth(wave_program(dr, 12, 2 * dr.loads_per_tile, 2), BARRIER, 1)},
      {"dQ (rotary) writing the epilogue's scratch over the ring without a barrier behind the table-row reads", dr,
       drop(wave_program(dr, 12, 2 * dr.loads_per_tile, 2), BARRIER, 0)},
      {"dK/dV ending iterations that requested nothing with the wait of those that did", dk, keeping},
      {"dQ, always requesting, writing scratch data over a tile in flight: no wait behind the loop", da,
       drop(wave_program(da, iterations, 2 * da.loads_per_tile), WAIT, 0)},
      {"dQ, always requesting, writing scratch data over another wave's part of a tile: no barrier behind the wait", da,
       drop(wave_program(da, iterations, 2 * da.loads_per_tile), BARRIER, 0)},
      {"dK/dV, always requesting, row blocks over a tile in flight: no wait behind the loop", ka,
       drop(wave_program(ka, iterations, 2 * ka.loads_per_tile, 3), WAIT, 1)},
      {"dK/dV, always requesting, row blocks over another wave's part of a tile: no barrier behind the wait", ka,
       drop(wave_program(ka, iterations, 2 * ka.loads_per_tile, 3), BARRIER, 1)},
  };
  for (const BrokenOps& k : broken_ops) {
    const std::string v = replay(k.p, k.ops);
    printf("%-104s %s\n", k.name, v.empty() ? "NOT CAUGHT" : ("caught: " + v).c_str());
    failures += v.empty();
  }
  // ---- the hand-over behind the loop
  const Protocol fp = forward_parts(3, 1, passes), dp = dq_parts(passes);
  Protocol dp_scratch = dp;
  dp_scratch.scratch_stages = 0;  // the scale-gradient staging over all of the ring
  const std::vector<Op> fwd_ops = wave_program(fp, 11, 2 * fp.loads_per_tile);  // the last tile lies in stage 1, a hand-over stage
  const int fwd_barriers = 2 + 11 + 1;  // start-up, iterations, hand-over
  const BrokenOps broken_merge[] = {
      {"forward reading the other wave's accumulators without the barrier behind their stores", fp, drop(fwd_ops, BARRIER, 0)},
      {"forward storing its accumulators without the barrier that ends the last iteration", fp, drop_nth(fwd_ops, BARRIER, fwd_barriers - 2)},
      {"dQ staging the scale gradient over the accumulators it is reading", dp_scratch, wave_program(dp_scratch, 12, 2 * dp.loads_per_tile)},
  };
  for (const BrokenOps& k : broken_merge) {
    const std::string v = replay(k.p, k.ops);
    printf("%-104s %s\n", k.name, v.empty() ? "NOT CAUGHT" : ("caught: " + v).c_str());
    failures += v.empty();
  }
  // ---- decode: a count that is off, a missing wait or barrier
  const DecodeLoads dl{2, 4, 4};
  const std::vector<Op> dec = decode_program(dl, 12, true);
  auto add_to_waits = [](std::vector<Op> ops, int immediate, int more) {
    for (Op& o : ops)
      if (o.kind == WAIT && o.n == immediate) o.n += more;
    return ops;
  };
  struct BrokenDecode { const char* name; std::vector<Op> ops; };
  const BrokenDecode broken_decode[] = {
      {"decode leaving one load too many in flight at the top of a block", add_to_waits(dec, decode_kept_at_top(dl), 1)},
      {"decode counting V_first among the loads younger than V", add_to_waits(dec, decode_kept_before_v(dl, true), dl.first)},
      {"decode awaiting V as if a next block were in flight behind the last one",
       [&] { std::vector<Op> o = dec; for (size_t i = o.size(); i-- > 0;) if (o[i].kind == WAIT) { o[i].n = dl.tables + dl.rows; break; } return o; }()},
      {"decode requesting K over the tile it is reading", drop_nth(dec, LDS_DONE, 0)},
      {"decode reading the tables without the workgroup's barrier", drop_nth(dec, BARRIER, 3)},
  };
  for (const BrokenDecode& k : broken_decode) {
    const std::string v = replay_decode(k.ops);
    printf("%-104s %s\n", k.name, v.empty() ? "NOT CAUGHT" : ("caught: " + v).c_str());
    failures += v.empty();
  }
  return failures ? 1 : 0;
}
