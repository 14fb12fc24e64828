// Copies of a schedule that no launch is spent on.
//
// A scheduler realizes more tensors than its kernels need: the output of a LayerNorm once as
// it is made and once more as the layer behind it reads it, a parameter's new value in a
// temporary and then in the parameter.  Such a kernel is dst[i] = src[i] over a whole buffer,
// the same type on both sides, and no group of fusion.cc has it as a member.  Each is a launch
// between two others that wait for it, 2-5 us whatever it moves: 37 of the 131 launches of
// GPT-2 small in fp32, six of the 17 or 22 of a classifier's training step.  Without them:
// GPT-2 small of 128 fp32 tokens 969 -> 888 us, a classifier's step at batch 33 48.1 -> 37.6, at
// batch 4096 179 -> 166.
//
//   dst an intermediate:  its readers read src instead;
//   dst the caller's:     the kernel that wrote src writes dst instead, and whoever read src
//                         reads dst.  The caller's buffer is then written earlier than the
//                         schedule says, which nobody sees unless buffers of the caller share
//                         memory: PlannedSchedule::written_early, for which the plan keeps the
//                         schedule as it stands (poly_hip_plan_run).
//
// Reference: src/exec_plan.c:1000-1057 launches every scheduled kernel.
#include <algorithm>
#include <cstdlib>

#include "fusion.h"
#include "templates.h"

namespace polyhip {

bool slot_fully_written(const PolySchedule *s, int slot, const std::vector<KernelGraph> &graphs);

namespace {

// Item `g` as dst[i] = src[i] (the positions of the two parameters), every i of a walk that
// slot_fully_written can vouch for.
bool is_identity(const KernelGraph &g, int *dst, int *src) {
  if (!g.reduces.empty() || g.stores.size() != 1 || g.stores[0].gate >= 0 || !g.vars.empty() || g.params.size() != 2) return false;
  const StoreInfo &st = g.stores[0];
  const KNode &v = g.n(st.value);
  if (v.op != POLY_OP_LOAD || v.guard >= 0 || v.dt != g.n(st.param).dt || v.src.size() != 1) return false;
  const KNode &ix = g.n(v.src[0]), &sx = g.n(st.index);
  if (ix.src.size() != 2 || sx.src.size() != 2) return false;
  const int ll = g.n(ix.src[1]).lin, ls = g.n(sx.src[1]).lin;
  if (ll < 0 || ls < 0) return false;
  const Lin &a = g.lins[(size_t)ll], &b = g.lins[(size_t)ls];
  if (a.c0 != b.c0 || a.terms.size() != b.terms.size()) return false;
  for (size_t i = 0; i < a.terms.size(); i++)
    if (a.terms[i].atom != b.terms[i].atom || a.terms[i].coef != b.terms[i].coef) return false;
  *dst = g.param_slot(st.param);
  *src = g.param_slot(ix.src[0]);
  return *dst >= 0 && *src >= 0 && *dst != *src && !g.params[(size_t)*dst].read;
}

// Whether kernel `g` reads parameter `p` nowhere but at the element it stores, once that
// element's sum (if it has one) is complete.
bool reads_only_its_element(const KernelGraph &g, int p) {
  if (g.stores.size() != 1 || g.stores[0].gate >= 0) return false;
  const KNode &sx = g.n(g.stores[0].index);
  const int ls = sx.src.size() == 2 ? g.n(sx.src[1]).lin : -1;
  if (ls < 0) return false;
  uint64_t mine = 0;
  for (int r : g.stores[0].ranges) {
    if (r >= 64) return false;
    mine |= 1ull << r;
  }
  const Lin &b = g.lins[(size_t)ls];
  for (const KNode &n : g.nodes) {
    if (n.op != POLY_OP_LOAD || n.src.empty()) continue;
    const KNode &ix = g.n(n.src[0]);
    if (ix.src.empty() || g.param_slot(ix.src[0]) != p) continue;
    const int ll = ix.src.size() == 2 ? g.n(ix.src[1]).lin : -1;
    if (ll < 0 || (n.deps & ~mine)) return false;
    const Lin &a = g.lins[(size_t)ll];
    if (a.c0 != b.c0 || a.terms.size() != b.terms.size()) return false;
    for (size_t i = 0; i < a.terms.size(); i++)
      if (a.terms[i].atom != b.terms[i].atom || a.terms[i].coef != b.terms[i].coef) return false;
  }
  return true;
}

struct Rewrite {
  const PolySchedule *s;
  const std::vector<KernelGraph> &graphs;
  std::vector<std::vector<int>> args;       // per item: its slots, as rewritten
  std::vector<char> dropped;                // items without a launch
  std::vector<int> step;
  std::vector<int> early;                   // the caller's buffers that are written before their copy's place
  std::vector<int> held_by;                 // per slot: the one that has its value, -1: itself

  bool uses(int item, int slot, bool written) const {
    const KernelGraph &g = graphs[(size_t)item];
    for (size_t p = 0; p < args[(size_t)item].size(); p++)
      if (args[(size_t)item][p] == slot && (written ? g.params[p].written : g.params[p].read)) return true;
    return false;
  }
  // the one item that writes `slot`, -1 if there is not exactly one
  int writer(int slot) const {
    int w = -1;
    for (int k = 0; k < s->n_items; k++)
      if (!dropped[(size_t)k] && uses(k, slot, true)) {
        if (w >= 0) return -1;
        w = k;
      }
    return w;
  }
  void rename(int from, int to) {
    for (auto &a : args) std::replace(a.begin(), a.end(), from, to);
    std::replace(held_by.begin(), held_by.end(), from, to);
    held_by[(size_t)from] = to;
  }

  bool drop(int c) {
    const KernelGraph &g = graphs[(size_t)c];
    int pd, ps;
    if (!is_identity(g, &pd, &ps)) return false;
    const int dst = args[(size_t)c][(size_t)pd], src = args[(size_t)c][(size_t)ps];
    const PolyScheduleBufSlot &d = s->buf_slots[dst], &t = s->buf_slots[src];
    if (dst == src || !t.is_intermediate || t.numel != d.numel || t.nbytes != d.nbytes) return false;
    const int w = writer(src);
    if (w < 0 || writer(dst) != c || step[(size_t)w] >= step[(size_t)c]) return false;
    if (!slot_fully_written(s, s->items[c].buf_slot_indices[pd], graphs)) return false;
    if (d.is_intermediate) {
      for (int k = 0; k < s->n_items; k++) {
        if (dropped[(size_t)k] || k == c || !uses(k, dst, false)) continue;
        if (step[(size_t)k] < step[(size_t)c] || uses(k, src, false)) return false;
      }
      dropped[(size_t)c] = 1;
      rename(dst, src);
      return true;
    }
    // (src as a whole comes from its one writer: what a writer leaves out reads as zero in an
    // intermediate, and as whatever it was in a buffer of the caller's)
    const KernelGraph &gw = graphs[(size_t)w];
    if (gw.stores.size() != 1 || !gw.vars.empty() || !slot_fully_written(s, written_slot(w), graphs)) return false;
    for (int k = 0; k < s->n_items; k++) {
      if (dropped[(size_t)k] || k == c) continue;
      const bool reads_old = uses(k, dst, false);
      if (k == w) {
        for (size_t p = 0; p < args[(size_t)k].size(); p++)
          if (args[(size_t)k][p] == dst && !reads_only_its_element(gw, (int)p)) return false;
      } else if (reads_old && (step[(size_t)k] > step[(size_t)w] && (step[(size_t)k] < step[(size_t)c] || uses(k, src, false)))) {
        return false;
      }
    }
    dropped[(size_t)c] = 1;
    rename(src, dst);
    early.push_back(dst);
    return true;
  }
  // the slot that the schedule itself names for what item `w` stores
  int written_slot(int w) const {
    const KernelGraph &g = graphs[(size_t)w];
    const int p = g.param_slot(g.stores[0].param);
    return s->items[w].buf_slot_indices[p];
  }
};

int n_launches(const PolySchedule *s, const std::vector<FusedGroup> &groups) {
  int n = s->n_items;
  for (const FusedGroup &fg : groups) n -= (int)fg.items.size() - 1;
  return n;
}

}  // namespace

bool plan_schedule(const PolySchedule *s, bool buffers_apart, PlannedSchedule *out, std::string *err) {
  MatmulsOfPlan of_plan;
  out->graphs.clear();
  out->graphs.resize((size_t)s->n_items);
  for (int k = 0; k < s->n_items; k++) {
    if (s->items[k].kind != POLY_EXEC_COMPUTE) { *err = strf("non-COMPUTE item %d not supported", k); return false; }
    if (!out->graphs[(size_t)k].build(s->items[k].root)) { *err = strf("kernel %d: %s", k, out->graphs[(size_t)k].error.c_str()); return false; }
  }
  out->sched = *s;
  out->unused.assign((size_t)s->n_buf_slots, 0);
  out->written_early.clear();
  out->held_by.clear();
  find_fused_groups(s, out->graphs, &out->groups);
  auto as_it_is = [&]() {
    refine_fused_groups(s, out->graphs, buffers_apart, &out->groups);
    return true;
  };
  // (a dropped copy is two buffers of the schedule in one place, which POLY_HIP_NO_ALIAS is about)
  if (!buffers_apart || getenv("POLY_HIP_NO_FUSION") || getenv("POLY_HIP_NO_COPY_DROP") || getenv("POLY_HIP_NO_ALIAS")) return as_it_is();

  // (what a group has taken in costs no launch, and the matchers know those copies)
  std::vector<char> grouped((size_t)s->n_items, 0);
  for (const FusedGroup &fg : out->groups) {
    bool copies = true;
    int pd, ps;
    for (int it : fg.items) copies = copies && is_identity(out->graphs[(size_t)it], &pd, &ps);
    if (!copies) for (int it : fg.items) grouped[(size_t)it] = 1;
  }
  Rewrite rw{s, out->graphs, {}, {}, {}, {}, {}};
  rw.held_by.assign((size_t)s->n_buf_slots, -1);
  rw.dropped.assign((size_t)s->n_items, 0);
  rw.step.assign((size_t)s->n_items, 0);
  for (int st = 0; st < s->n_items; st++) rw.step[(size_t)s->exec_order[st]] = st;
  for (int k = 0; k < s->n_items; k++) {
    const PolyExecItem &it = s->items[k];
    if ((int)out->graphs[(size_t)k].params.size() != it.n_buf_slots) return as_it_is();
    for (int i = 0; i < it.n_buf_slots; i++)
      if (it.buf_slot_indices[i] < 0 || it.buf_slot_indices[i] >= s->n_buf_slots) return as_it_is();
    rw.args.push_back(std::vector<int>(it.buf_slot_indices, it.buf_slot_indices + it.n_buf_slots));
  }
  int n_dropped = 0;
  for (int st = 0; st < s->n_items; st++) {
    const int k = s->exec_order[st];
    if (!grouped[(size_t)k] && out->graphs[(size_t)k].reduces.empty() && rw.drop(k)) n_dropped++;
  }
  if (n_dropped == 0) return as_it_is();

  PlannedSchedule p;
  p.sched = *s;
  std::vector<int> number((size_t)s->n_items, -1);
  auto keep_copies = [&]() {
    for (int k = 0; k < s->n_items; k++)
      if (number[(size_t)k] >= 0) out->graphs[(size_t)k] = std::move(p.graphs[(size_t)number[(size_t)k]]);
    return as_it_is();
  };
  for (int k = 0; k < s->n_items; k++) {
    if (rw.dropped[(size_t)k]) continue;
    number[(size_t)k] = (int)p.items.size();
    p.items.push_back(s->items[k]);
    p.args.push_back(rw.args[(size_t)k]);
    p.graphs.push_back(std::move(out->graphs[(size_t)k]));
  }
  for (size_t i = 0; i < p.items.size(); i++) p.items[i].buf_slot_indices = p.args[i].data();
  for (int st = 0; st < s->n_items; st++)
    if (number[(size_t)s->exec_order[st]] >= 0) p.order.push_back(number[(size_t)s->exec_order[st]]);
  p.sched.items = p.items.data();
  p.sched.n_items = (int)p.items.size();
  p.sched.exec_order = p.order.data();
  p.written_early = rw.early;
  p.held_by = rw.held_by;
  p.unused.assign((size_t)s->n_buf_slots, 1);
  for (const auto &a : p.args) for (int sl : a) p.unused[(size_t)sl] = 0;
  std::vector<char> used_before((size_t)s->n_buf_slots, 0);
  for (int k = 0; k < s->n_items; k++)
    for (int i = 0; i < s->items[k].n_buf_slots; i++) used_before[(size_t)s->items[k].buf_slot_indices[i]] = 1;
  for (int sl = 0; sl < s->n_buf_slots; sl++)
    if (!used_before[(size_t)sl] || !s->buf_slots[sl].is_intermediate) p.unused[(size_t)sl] = 0;
  find_fused_groups(&p.sched, p.graphs, &p.groups);
  if (n_launches(&p.sched, p.groups) >= n_launches(s, out->groups)) return keep_copies();
  // (a kernel that reads the old contents of such a buffer is not in one launch with the one
  // that writes it: what one workgroup has stored, another might still have to read)
  for (const FusedGroup &fg : p.groups)
    for (int sl : p.written_early)
      for (int a : fg.items)
        for (int b : fg.items) {
          bool writes = false, reads = false;
          for (size_t i = 0; i < p.args[(size_t)a].size(); i++) writes = writes || (p.args[(size_t)a][i] == sl && p.graphs[(size_t)a].params[i].written);
          for (size_t i = 0; i < p.args[(size_t)b].size(); i++) reads = reads || (p.args[(size_t)b][i] == sl && p.graphs[(size_t)b].params[i].read);
          if (writes && reads && std::find(p.order.begin(), p.order.end(), b) < std::find(p.order.begin(), p.order.end(), a)) return keep_copies();
        }
  if (getenv("POLY_HIP_DEBUG")) fprintf(stderr, "polygrad: compile_schedule: %d copies need no launch, %zu buffers of the caller are written by the kernel in front\n", n_dropped, p.written_early.size());
  refine_fused_groups(&p.sched, p.graphs, buffers_apart, &p.groups);
  *out = std::move(p);
  return true;
}

}  // namespace polyhip
