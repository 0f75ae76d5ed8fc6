// Internal representation of a compiled program.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <memory>
#include <vector>

#include "plaquette_amd.h"
#include "pq_common.h"
#include "pq_frame.h"

constexpr uint64_t kCus = 256;               // compute units of an MI355X
constexpr uint32_t kProgramThreadsMax = 768;  // largest block of the persistent kernel builds
// Gate segments with more qubits than a row tile of kWindowCutRows rows can
// hold (in the default LDS budget) are cut into qubit windows, each small
// enough for a tile of kWindowRows rows.
constexpr uint32_t kWindowCutRows = 32;
constexpr uint32_t kWindowRows = 48;

struct pq_program_s {
  uint64_t n = 0, W = 0, R = 0;
  std::vector<pq_op> ops;
  uint64_t ngates = 0, nmeas = 0, nnoise = 0;
  std::vector<pq::DSegment> segs;
  std::vector<pq::DInstr> instrs;
  std::vector<pq::NoiseDesc> noise;
  std::vector<uint32_t> segq;  // qubit lists of row-tiled gate segments
  bool tiled = false;          // some gate segment runs row-tiled
  bool masked = false;         // noise or flagged ops
  bool uniform = false;        // no flagged H/S/CX/CZ: X/Z change in every shot alike
  pq::DSegment *d_segs = nullptr;
  uint32_t *d_segq = nullptr;
  pq::DInstr *d_instrs = nullptr;
  pq::NoiseDesc *d_noise = nullptr;
  uint64_t *d_planes = nullptr;  // noise planes [nnoise][2][W]
  uint64_t *d_side = nullptr;    // frame form, two-part runs: [W][2n + nref] words
  uint32_t threads = 0, blocks = 0;
  // the graph form's captured launches, by which kernels they hold (0,
  // kSharedKnown, kSharedVerify); each replay takes the one of its state
  struct Graph {
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    uint64_t state_id = 0, arena_gen = 0;  // the state whose buffers it holds
    void drop() {
      if (exec) (void)hipGraphExecDestroy(exec);
      if (graph) (void)hipGraphDestroy(graph);
      exec = nullptr;
      graph = nullptr;
    }
  } graphs[3];
  hipStream_t alloc_stream = nullptr;  // stream-ordered allocation (server use)
  unsigned long long *d_census = nullptr;  // 8 counters when census is on
  bool census_on = false;
  bool timing_on = false;
  std::vector<hipEvent_t> ev;  // start/end pairs of timed kernel launches
  size_t ev_used = 0;
  std::shared_ptr<FramePlan> frame;  // frame form plan, built on first use (may be shared)
  // prepare_records' check of the record ids, for a state holding
  // prep_start records (prep_end after the run), and the measured slots
  bool prep_valid = false;
  uint64_t prep_start = 0, prep_end = 0;
  std::vector<uint32_t> m_slots;
  // end of the last run's device work (on last_stream): a run on another
  // stream waits for it, since the noise planes and side buffer are shared
  hipEvent_t done_ev = nullptr;
  hipStream_t last_stream = nullptr;
  // workgroups per word group in persistent runs: requested (0: chosen from
  // the state size and the device), last used, and the slices' barrier
  // counters ([W] words) and give-up flag (one word after them)
  uint32_t slices_req = 0, slices_used = 1;
  bool slices_set = false;     // pq_program_set_slices was called: per-shot kernel
  uint64_t *d_packed = nullptr;  // the shared X/Z columns, where a kernel of its own expands them
  uint32_t *d_done = nullptr;  // shared-X/Z runs that verify: groups that ran, [W]
  uint32_t slice_wait = 0;  // polls before a barrier gives up (0: default)
  unsigned int *d_sync = nullptr;
  uint64_t sync_words = 0;
  void drop_graph();
  ~pq_program_s();
};

int compile_program(pq_program_s *p);
// What the frame form alone needs: the noise descriptors (noise ops and
// random flags, numbered in program order as compile_program numbers them)
// and the op counts, without the persistent form's segments.
int compile_frame_only(pq_program_s *p);
int validate_ops(uint64_t n, const pq_op *ops, uint64_t nops);

constexpr uint64_t kProgramLdsBytes = 158 * 1024;  // dynamic-LDS cap (kProgramLdsBudget there)

// Shared with the batch runner.  check_records validates the record ids
// and sets p->prep_end without allocating; prepare_records also sizes the
// state's record arena and marks the measured records' host copies stale.
int check_records(pq_state s, pq_program p);
int prepare_records(pq_state s, pq_program p);
pq::ProgramArgs program_args(pq_state s, pq_program p, uint64_t lds_budget);
// Whether a persistent run of p on s from |0...0> may take the shared-X/Z
// kernel, and the buffers such a run needs (made once per program).
bool shared_allowed(const pq_state_s *s, const pq_program_s *p);
int ensure_shared(pq_state s, pq_program p, uint32_t shared, bool split);
// pq_program_create for a server-owned state: stream-ordered allocation and
// copies on the state's stream.
int create_program_on(pq_state s, const pq_op *ops, uint64_t nops, pq_program *out);
