// Plan-level fusion of kernel groups (see fusion.cc).
#pragma once
#include <string>
#include <vector>

#include "polygrad_abi.h"
#include "templates.h"

namespace polyhip {

// A set of schedule items replaced by one launch.
struct FusedGroup {
  std::vector<int> items;           // schedule items the fused kernel stands for
  int launch_item = -1;             // the fused kernel runs at this item's place in exec_order
  std::vector<int> internal_slots;  // buffers that are never materialised
  std::vector<int> arg_slots;       // slot of each kernel argument, in order
  RenderedKernel rk;
  // a row chain: the item it was grown from and the buffer its last kernel stores (-1: none)
  int row_chain_from = -1, row_chain_stores = -1;
  // ... what a product that computes those rows itself needs of it (rows.code empty: its rows are not
  // dealt to at most a wave each, or it stores more than them): `n_rows` rows of `row_len`
  // elements, stored row after row; the arguments behind the first are its parameters
  MatmulRows rows;
  int64_t n_rows = 0, row_len = 0;
  // a product that computes those rows itself: buffers of the caller's that it writes, each with
  // one that its workgroups read whole rows of; where the two share memory the launches are two
  std::vector<std::pair<int, int>> apart;
  // Two groups that only work together (a chain that stores bf16 values into an fp32 buffer
  // and the product that reads them as such) name each other's launch item here: dropping
  // one drops the other.
  int needs_group_at = -1;
  int matched_from = -1;            // the item the matcher started from
  // An attention group whose keys lie in the output of a product, in blocks of 64 keys x 64
  // features that are blocks of 64 rows x 64 columns there (row-major, `pitch` columns,
  // `rows` rows): what that product would have to leave for the kernel to bound the
  // products of masked key blocks without computing them (MatmulEpilogue::block_maxima).
  struct KeyBounds {
    bool possible = false, used = false;
    int slot = -1;
    int64_t pitch = 0, rows = 0, lo = 0, hi = 0;
    std::string index;
    size_t bytes = 0, offset = 0;   // of the table, and where it lies in the kernel's scratch memory
  } key_bounds;
};

// Finds the fusable groups of a schedule.  graphs[k] is the analysed kernel of item k.
// Setting POLY_HIP_NO_FUSION in the environment disables the search.
void find_fused_groups(const PolySchedule *s, const std::vector<KernelGraph> &graphs, std::vector<FusedGroup> *out);
// What is done with the groups once they are known: pairs that work together are rendered again,
// and groups that would launch out of order are dropped.  !buffers_apart: only what does as the
// kernels do also where buffers of the caller's share memory (FusedGroup::apart).
void refine_fused_groups(const PolySchedule *s, const std::vector<KernelGraph> &graphs, bool buffers_apart, std::vector<FusedGroup> *out);
// The groups (indices into `groups`) whose place of launch breaks the order of two kernels
// of the schedule that share a buffer, one of them writing it; refine_fused_groups drops such
// groups itself, so that its result always passes.
std::vector<int> fused_groups_out_of_order(const PolySchedule *s, const std::vector<KernelGraph> &graphs, const std::vector<FusedGroup> &groups);

// What matmul_hint_param_kinds takes for the lowering of item `item`: 1 for every fp32
// buffer parameter that is an intermediate of the plan with one writer, whose one store
// puts a bf16 value cast to fp32 there (2 where `narrow_slots` names the buffer: its writer
// has been made to store the bf16 values themselves).
std::vector<int> matmul_param_kinds_of(const PolySchedule *s, const std::vector<KernelGraph> &graphs, int item, const std::vector<int> &narrow_slots);

// A schedule as it is planned: its kernels analysed, grouped, and without the copies that
// need no launch (copies.cc).  `sched` is the schedule itself where there are none.
struct PlannedSchedule {
  PolySchedule sched;
  std::vector<KernelGraph> graphs;          // of the items of `sched`
  std::vector<FusedGroup> groups;
  std::vector<char> unused;                 // per slot: an intermediate that no kernel touches any more
  std::vector<int> written_early;           // the caller's buffers that are written before their copy's place
  std::vector<int> held_by;                 // per slot: the one that has its value, -1: itself (empty: all themselves)
  PlannedSchedule() = default;
  PlannedSchedule(const PlannedSchedule &) = delete;
  PlannedSchedule &operator=(PlannedSchedule &&) = default;
  std::vector<PolyExecItem> items;          // what `sched` points to, where it is not the caller's
  std::vector<std::vector<int>> args;
  std::vector<int> order;
};
// Analyses and groups schedule `s` (POLY_HIP_NO_COPY_DROP in the environment, or
// !buffers_apart: every copy keeps its launch).  False with a message on a malformed kernel.
bool plan_schedule(const PolySchedule *s, bool buffers_apart, PlannedSchedule *out, std::string *err);

}  // namespace polyhip
