// Host-side planning of one step of the gfx950 paged-KV path: validation of
// a batch description, the decode and block-prefill work lists, and the
// staged host->device upload of the plan. Plain C++ with no HIP types: the
// device side is reached through MemOps, so the planner also builds and runs
// on a CPU-only host (the sanitizer tests link it with a fake MemOps).
#pragma once

#include <cstddef>
#include <functional>
#include <vector>

#include "../csrc/tge_records.h"

namespace tge::plan {

// Device memory, pinned host memory, copies and ordering, as status-returning
// calls (TGE_OK or a tge_status). A stream or event is an opaque handle.
struct MemOps {
  virtual ~MemOps() = default;
  virtual int host_alloc(char** p, std::size_t bytes) = 0;
  virtual void host_free(char* p) = 0;
  virtual int dev_alloc(char** p, std::size_t bytes) = 0;
  virtual void dev_free(char* p) = 0;
  virtual int copy_to_device(char* dev, const char* host, std::size_t bytes, void* stream) = 0;
  // Record a marker after the work queued on `stream` (creating it when
  // *event is null); wait for a marker; wait for a stream.
  virtual int record(void** event, void* stream) = 0;
  virtual int wait_event(void* event) = 0;
  virtual int wait_stream(void* stream) = 0;
  virtual void event_free(void* event) = 0;
};

// A device buffer filled from pinned host staging. Both grow on demand and
// are reused across uploads. The recorded capacities always describe
// buffers that exist: a failed allocation leaves the buffer empty (capacity
// 0), so a later, smaller upload allocates again instead of writing through
// a freed pointer.
struct Staged {
  char* host = nullptr;
  std::size_t host_bytes = 0;
  char* dev = nullptr;
  std::size_t dev_bytes = 0;
  void* staged = nullptr;  // marker after the last copy out of `host`

  // Copy `bytes` (at least 256) written by `fill` into the host buffer to
  // the device buffer on `stream`. Waits for the previous copy out of the
  // host buffer first.
  int upload(MemOps& m, std::size_t bytes, void* stream, const std::function<void(char*)>& fill);
  void release(MemOps& m);
};

// A device array that grows on demand (split-K partials). Same capacity
// rule as Staged.
struct Scratch {
  char* dev = nullptr;
  std::size_t bytes = 0;
  // Make room for `need` bytes; waits for `stream` before freeing a smaller
  // buffer that queued work may still use.
  int reserve(MemOps& m, std::size_t need, void* stream);
  void release(MemOps& m);
};

// The sessions of one step (host copies of the plan records).
struct Step {
  std::vector<SessionRec> sessions;
  std::vector<int> tables;
  std::vector<RowRec> rows;
  int kv_heads = 0;
  int head_dim = 0;
  int block_dims = 0;  // width of the page blocks: 64, 128 or 256 (block_dims_for)
  int q_heads = 0;
  int group = 1;
  int pages = 0;     // pages of the pool
  int max_rows = 0;  // largest n_new * group
};

// Builds `step` from a batch description (the fields of tge_batch_desc),
// validating every rule first; on failure returns TGE_ERR_INVALID with a
// message and leaves `step` untouched.
int build_step(Step& step, int n_sessions, const int* ctx, const int* n_new,
               const int* table_offsets, const int* page_ids, int q_heads, int kv_heads,
               int head_dim, int pool_pages, const char** message);

// The step's new rows page by page (TileRec) when its append should store
// whole pages, empty when it should go row by row. By page a launch has a
// longer fixed time (four tokens per lane, staged: f16 4.9 us, int8 6.0,
// against 3.8-4.2) and the better rate. The lines are drawn through measured
// crossings, which lie at fewer values the wider a row is and at more for
// int8, whose 1-byte stores write half as much. Values here are rows x 2 x KV
// heads x block width, a row's width its K dims: f16 from 2^20 values on, 2^21
// where a row is narrower than 1024 dims; int8 from 3 * 2^20, 9 * 2^19 below
// 1024 dims, never below 256. Row kernel / page kernel, us:
//   f16   8 x 256, 257 rows 6.3 / 4.8; 8 x 128, 513 5.4 / 4.8; 4 x 128, 2048
//         7.4 / 5.7; 2 x 128, 4097 6.6 / 5.5; 1 x 128, 8200 6.1 / 5.7; 1 x
//         256, 4100 6.7 / 5.8; below the line 4 x 128, 1100 (a part of a
//         page last) 5.1 / 5.6, 1500 5.8 / 5.9; 1 x 128, 6000 4.9 / 5.3
//   int8  8 x 256, 768 8.9 / 8.0; 8 x 128, 2048 9.9 / 8.5; 4 x 128, 5000
//         10.2 / 10.3, 8192 17.6 / 15.3; 2 x 128, 12000 10.8 / 10.8; below
//         the line 8 x 256, 512 6.7 / 6.7; 2 x 256, 2048 5.7 / 6.9; 1 x 128,
//         16384 7.8 / 8.5, 32768 14.3 / 15.4
// 64-dim blocks stay with the row kernel (2 heads, 20,000 rows: int8 9.3 /
// 10.5, f16 11.5 / 10.8 with a page kernel for them and an earlier f16
// encoder), and so do steps whose rows fill their pages to less than three
// quarters on average. No line lies below kAppendPageWork lanes (8 values
// each) times block width.
constexpr long kAppendPageWork = 1L << 24;
void build_append_tiles(const Step& s, std::vector<TileRec>& tiles, bool i8 = false);

// Work lists of one attention kind for the current step.
struct AttnLists {
  std::vector<WorkRec> work;
  std::vector<ReduceRec> reduce;
  std::vector<int> wg_first;  // [groups + 1] first item of each workgroup, or empty
  int groups = 0;             // workgroups of the launch
  int row_groups = 1;         // 16-row groups per unit
  int tile_rows = 0;          // prefill: rows of a tile (prefill_tile_rows, or 64)
  int parts = 0;              // split-K partial slots
  int max_splits = 0;
  // Decode launches that store the step's new rows (build_decode_appends):
  // the rows each wave stores, those of the pages it reads itself, as
  // records {page id, position, k/v row * kv_heads + KV head, work item};
  // wave w of workgroup g stores records [app_first[g*app_waves + w],
  // app_first[g*app_waves + w + 1]). kAppPad zero records follow the last.
  // app_waves 0: no lists (the launch cannot store the rows).
  std::vector<int> app_first;
  std::vector<int> app_recs;
  int app_waves = 0;
};


// Resident workgroups of the decode launch and the device's compute units;
// workgroup g is the (g / cus)-th to land on its compute unit.
struct Residency {
  int groups;
  int cus;
};

// Sessions a decode unit holds (n_new * group <= kMaxRows); `only`: 0 every
// session, 1 those, 2 the others.
bool decode_session(const Step& s, const SessionRec& r);
bool take_session(const Step& s, const SessionRec& r, int only);

// Decode schedule: every (session, KV head) is a segment of pages; the
// segments are laid end to end and cut into one share per resident
// workgroup (balanced by pages, per-piece cost and dispatch rank); a
// segment cut into several items is merged by the split reduction.
void build_decode(const Step& s, Residency res, AttnLists& out, int only);

// The new-row records of a decode plan whose launch of `waves` waves per
// workgroup stores the rows: page j (from page_begin) of work item `item`
// is read by wave (j + item) mod waves, which stores the new rows that page
// holds. No lists
// (app_waves 0) when `waves` is 0 or a wave would hold more than max_rows.
void build_decode_appends(const Step& s, AttnLists& pl, int waves, int max_rows);

// Block-prefill work: (session, KV head, query tile) x page pieces, longest
// items first. `halves`: groups of four waves per workgroup (2: an item's
// pages are shared by two halves). A launch of its own (`only` 0) takes the
// shortest of a few ways to cut the tiles, by a model of the launch's length
// on `cus` compute units (`i8`: int8 pages); at 128 dims with two halves the
// tiles may be 64 rows (tile_rows). Otherwise the pieces are of about equal
// length and cover the compute units about twice.
void build_prefill(const Step& s, int cus, AttnLists& out, int only, int halves = 1,
                   bool i8 = false);

// A small decode step in one launch (paged_step_kernel): one workgroup per
// piece of a (session, KV head) segment; pieces of a split segment own
// consecutive partial slots and the segment's arrival counter.
struct StepLists {
  std::vector<StepRec> recs;
  std::vector<int> first_ids;  // [recs][kStepFirstIds]
  int row_groups = 1;
  int piece_pages = 0;  // pages of every piece but a segment's first
  int parts = 0;        // partial slots
  int segments = 0;     // arrival counters
  int max_pieces = 0;
};

// Builds the one-launch lists when every session's rows fit a decode unit
// (at most 48 rows at head_dim above 64) and the step holds at most
// kStepMaxBlocks page blocks; returns false (and leaves `out` empty)
// otherwise. Pieces are whole batches of the kernel's page loads
// (kStepWaves x step_batch_pages), at most kStepMaxParts per segment; the
// segment's last piece holds every page with a new position and stores the
// new rows.
constexpr int kStepMaxBlocks = 4096;
bool build_step_lists(const Step& s, bool i8, bool scale_f32, StepLists& out);

// The plan image of `lists` (work | reduce | wg_first, each 256-aligned):
// total bytes and the offsets of the reduce and wg_first parts.
// [ work | reduce | wg_first | app_first | app_recs ], each part 256-byte aligned.
std::size_t image_layout(const AttnLists& lists, std::size_t* off_reduce, std::size_t* off_first,
                         std::size_t* off_app = nullptr);
void write_image(const AttnLists& lists, std::size_t off_reduce, std::size_t off_first, char* dst,
                 std::size_t off_app = 0);

}  // namespace tge::plan
