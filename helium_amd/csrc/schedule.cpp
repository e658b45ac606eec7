// The launch list of a plan (exec.h: Schedule): what an execution does, worked out once per graph, so that a call only
// fills in addresses. A small graph's execution is bound by the host, which spent a third of it in maps from nodes to
// tensors and in one allocation per intermediate value (a training step of 157 launches: 214 of 630 us).
#include <algorithm>
#include <functional>
#include <future>
#include <map>
#include <set>

#include "exec.h"

namespace he::exec {

// Small elementwise launches whose work may share a launch with others': a launch costs the host 2.5 us and the device
// about as much, whatever it does. (Larger ones gain nothing from company, and moving them keeps their operands alive.)
bool can_share_launch(const plan::Instr& instr) {
    constexpr size_t kMostBytes = 32u << 20;
    if (instr.kind() != plan::InstrKind::Pointwise) return false;
    const auto kernel = std::dynamic_pointer_cast<TileKernel>(instr.kernel());
    if (!kernel || !kernel->can_join()) return false;
    size_t bytes = 0;
    for (const tp::Arg& a : kernel->args()) bytes += storage_bytes(a.dtype, (size_t)a.numel);
    return bytes <= kMostBytes;
}

namespace {

// An instruction that only renames a shape: its result is its operand's storage.
bool is_view(const plan::Instr& instr, const ir::OpGraph& g) {
    if (instr.kind() != plan::InstrKind::Pointwise || instr.carried() || instr.absorbed() || instr.subgraph().nodes().size() != 1) return false;
    const ir::Node& n = g.get(instr.subgraph().nodes()[0]);
    return n.op.kind == ir::OpKind::Reshape && g.get(n.op.inputs[0]).desc.dtype == n.desc.dtype;
}

// Launches on their way to the list: plan instructions, one or several to a launch.
struct Item {
    std::vector<const plan::Instr*> instrs;
    std::vector<NodeId> reads, writes;
    uint8_t side = 0;  // Prepared::Side::side
    bool mergeable = false;
    std::shared_ptr<KernelBase> kernel;  // of several instructions
};

Item item_of(const plan::Instr& instr, uint8_t side) {
    Item it;
    it.instrs = {&instr};
    it.reads = instr.all_inputs();
    it.writes = instr.all_outputs();
    it.side = side;
    return it;
}

// Makes the kernels of the groups that have none yet, in parallel. A group without one - it does not compile, or there are no
// tiles that all members can take - goes out as its members, whose own kernels are there.
void compile_joins(std::vector<Item>* items, const std::function<std::shared_ptr<KernelBase>(const std::vector<std::shared_ptr<KernelBase>>&)>& join) {
    std::vector<std::future<std::shared_ptr<KernelBase>>> jobs(items->size());
    for (size_t i = 0; i < items->size(); i++) {
        const Item& it = (*items)[i];
        if (it.instrs.size() < 2 || it.kernel) continue;
        std::vector<std::shared_ptr<KernelBase>> members;
        for (auto* instr : it.instrs) members.push_back(instr->kernel());
        jobs[i] = std::async(std::launch::async, [&join, members]() -> std::shared_ptr<KernelBase> {
            try {
                return join(members);
            } catch (const Error&) {
                return nullptr;
            }
        });
    }
    std::vector<Item> list;
    for (size_t i = 0; i < items->size(); i++) {
        Item& it = (*items)[i];
        if (jobs[i].valid() && !(it.kernel = jobs[i].get())) {
            for (auto* instr : it.instrs) list.push_back(item_of(*instr, it.side));
            continue;
        }
        list.push_back(std::move(it));
    }
    *items = std::move(list);
}

// Joins launches of a one-stream list. Each mergeable launch may run anywhere between the last launch that makes what it
// reads and the first that reads what it makes; a group goes out when the first of its members has to, and takes every
// launch along that can run by then: the fewest launches there can be (the casts of all filters at the head of a
// training step, the parameters' updates at its end).
void join_launches(std::vector<Item>* items) {
    constexpr size_t kMostMembers = 24, kMostArgs = 160;
    const size_t n = items->size();
    std::map<NodeId, size_t> made_by;
    std::vector<std::vector<size_t>> deps(n), users(n);
    for (size_t i = 0; i < n; i++) {
        std::set<size_t> from;
        for (NodeId r : (*items)[i].reads) {
            auto it = made_by.find(r);
            if (it != made_by.end()) from.insert(it->second);
        }
        for (size_t d : from) {
            deps[i].push_back(d);
            users[d].push_back(i);
        }
        for (NodeId w : (*items)[i].writes) made_by[w] = i;
    }
    // the position by which a launch has to be out: its first user's own, or that user's place if it stays where it is
    std::vector<size_t> due(n, n);
    for (size_t i = n; i-- > 0;)
        for (size_t u : users[i]) due[i] = std::min(due[i], (*items)[u].mergeable ? due[u] : u);
    std::vector<uint8_t> out(n, 0);
    std::vector<Item> list;
    std::vector<size_t> waiting;  // mergeable launches passed by and not out yet, in order
    auto ready = [&](size_t i) {
        for (size_t d : deps[i])
            if (!out[d]) return false;
        return true;
    };
    // sends out what is due by `pos`, with company
    auto flush = [&](size_t pos) {
        for (;;) {
            bool any_due = false;
            for (size_t i : waiting) any_due = any_due || due[i] <= pos;
            if (!any_due) return;
            Item group;
            size_t args = 0;
            std::vector<size_t> members, rest;
            // (those that are due first: the company must not fill the launch ahead of them)
            for (int pass = 0; pass < 2; pass++)
                for (size_t i : waiting) {
                    if ((due[i] <= pos) != (pass == 0)) continue;
                    const size_t more = (*items)[i].reads.size() + (*items)[i].writes.size();
                    // (one of more arguments than that goes out alone)
                    if (ready(i) && members.size() < kMostMembers && (members.empty() || args + more <= kMostArgs)) {
                        members.push_back(i);
                        args += more;
                    } else {
                        rest.push_back(i);
                    }
                }
            std::sort(members.begin(), members.end());
            std::sort(rest.begin(), rest.end());
            for (size_t i : members) {
                Item& m = (*items)[i];
                group.instrs.insert(group.instrs.end(), m.instrs.begin(), m.instrs.end());
                group.reads.insert(group.reads.end(), m.reads.begin(), m.reads.end());
                group.writes.insert(group.writes.end(), m.writes.begin(), m.writes.end());
                out[i] = 1;
            }
            HE_REQUIRE(!members.empty(), HE_ERR_INTERNAL, "no launch of the group that is due can run");
            list.push_back(std::move(group));
            waiting.swap(rest);
        }
    };
    // (what reads nothing but the graph's inputs can come along from the start)
    std::vector<uint8_t> queued(n, 0);
    for (size_t i = 0; i < n; i++)
        if ((*items)[i].mergeable && deps[i].empty()) {
            waiting.push_back(i);
            queued[i] = 1;
        }
    for (size_t i = 0; i < n; i++) {
        if ((*items)[i].mergeable) {
            if (!queued[i]) waiting.push_back(i);
            continue;
        }
        flush(i);
        list.push_back(std::move((*items)[i]));
        out[i] = 1;
    }
    flush(n);
    *items = std::move(list);
    compile_joins(items, [](const std::vector<std::shared_ptr<KernelBase>>& kernels) {
        std::vector<std::shared_ptr<TileKernel>> members;
        for (auto& k : kernels) members.push_back(std::dynamic_pointer_cast<TileKernel>(k));
        return std::make_shared<JoinedKernel>(members);
    });
}

// Joins products that follow each other in the list and do not depend on each other: a layer's data gradient and filter
// gradient, a block's two convolutions of one activation.
void join_products(std::vector<Item>* items) {
    constexpr size_t kMostMembers = 4;
    std::vector<Item> list;
    for (Item& it : *items) {
        const auto joinable = [](const Item& i) {
            for (auto* instr : i.instrs)
                if (instr->kind() != plan::InstrKind::Gemm || instr->carried() || !JoinedProducts::can_join(*instr->kernel())) return false;
            return true;
        };
        bool join = !list.empty() && list.back().instrs.size() < kMostMembers && joinable(it) && joinable(list.back());
        if (join)
            for (NodeId r : it.reads) join = join && std::find(list.back().writes.begin(), list.back().writes.end(), r) == list.back().writes.end();
        if (!join) {
            list.push_back(std::move(it));
            continue;
        }
        Item& group = list.back();
        group.instrs.push_back(it.instrs[0]);
        group.reads.insert(group.reads.end(), it.reads.begin(), it.reads.end());
        group.writes.insert(group.writes.end(), it.writes.begin(), it.writes.end());
    }
    *items = std::move(list);
    compile_joins(items, [](const std::vector<std::shared_ptr<KernelBase>>& kernels) { return std::make_shared<JoinedProducts>(kernels); });
}

}  // namespace

void build_schedule(Prepared* pr) {
    const ir::OpGraph& g = *pr->graph;
    const plan::Plan& plan = *pr->plan;
    for (uint8_t f : pr->fan_out)
        if (f) return;  // runs step by step over several streams
    Schedule S;
    // ---- slots: one per value that exists in memory
    std::map<NodeId, uint32_t> slot_of;
    auto new_slot = [&](NodeId node, Schedule::Slot::Where where) {
        const ir::Descriptor& d = g.get(node).desc;
        Schedule::Slot s;
        s.where = where;
        s.dtype = d.dtype;
        s.len = (size_t)ir::num_elements(d.shape);
        s.bytes = storage_bytes(d.dtype, s.len);
        slot_of[node] = (uint32_t)S.slots.size();
        S.slots.push_back(s);
        return (uint32_t)S.slots.size() - 1;
    };
    for (NodeId in : g.inputs()) S.inputs.push_back({pr->caller_input(in), new_slot(in, Schedule::Slot::Input)});
    std::sort(S.inputs.begin(), S.inputs.end(), [](const Schedule::Named& a, const Schedule::Named& b) { return a.node < b.node; });
    // ---- launches in the order they go out
    std::vector<Item> items;
    std::map<NodeId, NodeId> view_of;
    auto base = [&](NodeId n) {
        for (auto it = view_of.find(n); it != view_of.end(); it = view_of.find(n)) n = it->second;
        return n;
    };
    for (auto& step : plan.steps) {
        S.steps += !step.instrs.empty();
        for (auto& instr : step.instrs) {
            if (instr->absorbed()) continue;
            S.instrs++;
            if (is_view(*instr, g)) view_of[instr->outputs()[0]] = instr->inputs()[0];
        }
    }
    // A result is memory of its own, which its owner may write: one that would be another result's or an input's under another
    // shape is copied after all.
    for (bool again = true; again;) {
        again = false;
        std::map<NodeId, NodeId> held_by;  // storage -> the result that has it
        for (NodeId in : g.inputs()) held_by[in] = in;
        for (NodeId out : g.outputs()) {
            const NodeId n = g.inbound(out)[0], other = held_by.emplace(base(n), n).first->second;
            if (other == n) continue;
            view_of.erase(view_of.count(n) ? n : other);
            again = true;
            break;
        }
    }
    auto renames = [&](const plan::Instr& instr) { return is_view(instr, g) && view_of.count(instr.outputs()[0]); };
    const Prepared::Side& side = pr->side;
    if (side.side.empty()) {
        for (auto& step : plan.steps)
            for (auto& instr : step.instrs) {
                if (instr->absorbed() || renames(*instr)) continue;
                Item it = item_of(*instr, 0);
                it.mergeable = can_share_launch(*instr);
                items.push_back(std::move(it));
            }
        for (Item& it : items)
            for (NodeId& r : it.reads) r = base(r);
        join_launches(&items);
        join_products(&items);
        for (Item& it : items)
            for (NodeId& r : it.reads) r = base(r);
    } else {
        // The early instructions first, on the side stream, in one launch where they can share it; then the main chain in
        // plan order. A side instruction goes out where the plan has it, and the side instructions that read its results
        // alone follow at once (a filter gradient's update), which saves them a wait of their own.
        std::vector<uint8_t> issued(side.order.size(), 0);
        std::vector<Item> early;
        for (size_t i = 0; i < side.order.size(); i++) {
            if (side.side[i] != 2) continue;
            issued[i] = 1;
            if (renames(*side.order[i])) continue;
            Item it = item_of(*side.order[i], 2);
            it.mergeable = can_share_launch(*side.order[i]);
            early.push_back(std::move(it));
        }
        for (Item& it : early)
            for (NodeId& r : it.reads) r = base(r);
        join_launches(&early);
        for (Item& it : early) it.side = 2;
        items = std::move(early);
        auto issue = [&](auto&& self, size_t i) -> void {
            issued[i] = 1;
            if (!renames(*side.order[i])) items.push_back(item_of(*side.order[i], side.side[i]));
            if (side.side[i] != 1) return;
            for (uint32_t d : side.dependents[i]) {
                if (issued[d] || side.side[d] != 1) continue;
                bool ready = true;
                for (uint32_t dep : side.deps[d]) ready = ready && issued[dep];
                if (ready) self(self, d);
            }
        };
        for (size_t i = 0; i < side.order.size(); i++)
            if (!issued[i]) issue(issue, i);
        for (Item& it : items)
            for (NodeId& r : it.reads) r = base(r);
    }
    // ---- which values the caller gets
    std::set<NodeId> results;
    for (NodeId out : g.outputs()) results.insert(base(g.inbound(out)[0]));
    for (Item& it : items)
        for (NodeId w : it.writes) new_slot(w, results.count(w) ? Schedule::Slot::Result : Schedule::Slot::Arena);
    auto slot = [&](NodeId n) {
        auto it = slot_of.find(base(n));
        HE_REQUIRE(it != slot_of.end(), HE_ERR_INTERNAL, "missing storage for node %u", n);
        return it->second;
    };
    for (NodeId out : g.outputs()) S.outputs.push_back({pr->caller_output.empty() ? out : pr->caller_output.at(out), slot(g.inbound(out)[0])});
    std::sort(S.outputs.begin(), S.outputs.end(), [](const Schedule::Named& a, const Schedule::Named& b) { return a.node < b.node; });
    // ---- kernels, arguments, waits
    std::set<std::pair<uint8_t, uint32_t>> seen_inputs;
    bool main_dirty = false, early_pending = false;
    size_t last_main = SIZE_MAX;
    std::set<uint32_t> early_made;
    for (Item& it : items) {
        Schedule::Launch L;
        L.stream = it.side ? 1 : 0;
        if (it.kernel) {
            L.kernel = it.kernel;
        } else if (it.instrs[0]->kind() == plan::InstrKind::Permute) {
            L.permute = it.instrs[0]->permute();
            L.args = {slot(it.instrs[0]->inputs()[0]), slot(it.instrs[0]->outputs()[0])};
        } else {
            L.kernel = it.instrs[0]->kernel();
        }
        if (L.kernel)
            for (const tp::Arg& a : L.kernel->args()) L.args.push_back(slot((NodeId)a.node));
        for (NodeId r : it.reads) {
            const uint32_t s = slot(r);
            if (S.slots[s].where == Schedule::Slot::Input && seen_inputs.insert({L.stream, s}).second) L.new_inputs.push_back(s);
            if (L.stream == 0 && early_pending && early_made.count(s)) {
                L.waits_for_early = true;
                early_pending = false;
            }
        }
        if (it.side == 2) {
            for (NodeId w : it.writes) early_made.insert(slot(w));
            early_pending = true;
            S.early_launches = S.launches.size() + 1;
        } else if (it.side == 1) {
            if (main_dirty) {
                L.waits_for_main = true;
                S.launches[last_main].marks_end = true;
            }
            main_dirty = false;
        } else {
            main_dirty = true;
            last_main = S.launches.size();
        }
        S.uses_side = S.uses_side || L.stream == 1;
        S.launches.push_back(std::move(L));
    }
    // the last launch carries the execution's event when it runs on the main stream
    if (!S.launches.empty() && S.launches.back().stream == 0) S.launches.back().closes = true;
    // ---- where the values that nobody else sees lie: the largest first, each at the lowest address of the first block that has
    // it free for as long as it is needed. What the side stream touches stays until the streams join. A block holds what a page
    // of the pool does (DevicePool::kMinPage), or one value that is larger: one block for everything took a page of the next
    // power of two, 64 GB for 33 GB of values.
    const size_t n = S.launches.size();
    std::vector<size_t> from(S.slots.size(), SIZE_MAX), to(S.slots.size(), 0);
    for (size_t i = 0; i < n; i++)
        for (uint32_t s : S.launches[i].args) {
            from[s] = std::min(from[s], i);
            to[s] = std::max(to[s], S.launches[i].stream == 1 ? n : i);
        }
    std::vector<uint32_t> order;
    for (uint32_t s = 0; s < S.slots.size(); s++)
        if (S.slots[s].where == Schedule::Slot::Arena) order.push_back(s);
    std::stable_sort(order.begin(), order.end(), [&](uint32_t a, uint32_t b) { return S.slots[a].bytes > S.slots[b].bytes; });
    const char* env = tuning::get("HELIUM_HIP_ARENA_BLOCK");
    const uint64_t most = env ? (uint64_t)atoll(env) : DevicePool::kMinPage;
    struct Placed {
        uint64_t start, end;
        size_t from, to;
    };
    struct Block {
        std::vector<Placed> placed;  // by address
        uint64_t capacity;
        size_t from, to;
    };
    std::vector<Block> blocks;
    for (uint32_t s : order) {
        if (from[s] == SIZE_MAX) from[s] = 0, to[s] = n;  // (written by a launch that names it otherwise: keep it whole)
        const uint64_t size = std::max<uint64_t>((S.slots[s].bytes + DevicePool::kAlign - 1) / DevicePool::kAlign * DevicePool::kAlign, DevicePool::kAlign);
        uint64_t at = 0;
        size_t b = 0;
        for (;; b++) {
            if (b == blocks.size()) {
                blocks.push_back({{}, std::max(most, size), SIZE_MAX, 0});
                S.blocks.push_back(0);
            }
            at = 0;
            for (const Placed& p : blocks[b].placed) {
                if (p.to < from[s] || p.from > to[s]) continue;
                if (at + size <= p.start) break;
                at = std::max(at, p.end);
            }
            if (at + size <= blocks[b].capacity) break;
        }
        Block& block = blocks[b];
        S.slots[s].block = (uint32_t)b;
        S.slots[s].offset = at;
        S.blocks[b] = std::max(S.blocks[b], at + size);
        block.from = std::min(block.from, from[s]);
        block.to = std::max(block.to, to[s]);
        Placed mine{at, at + size, from[s], to[s]};
        block.placed.insert(std::upper_bound(block.placed.begin(), block.placed.end(), mine, [](const Placed& a, const Placed& b) { return a.start < b.start; }), mine);
    }
    // One block (most graphs): everything is allocated ahead of the first launch. Several: blocks and results as they are first
    // needed, and blocks given back behind their last launch, so that what comes later can have their memory.
    const bool at_once = S.blocks.size() < 2;
    for (uint32_t b = 0; b < S.blocks.size(); b++) {
        S.launches[at_once ? 0 : blocks[b].from].opens_blocks.push_back(b);
        if (!at_once && blocks[b].to < n) S.launches[blocks[b].to].closes_blocks.push_back(b);
    }
    for (uint32_t s = 0; s < S.slots.size(); s++)
        if (S.slots[s].where == Schedule::Slot::Result) S.launches[at_once || from[s] == SIZE_MAX ? 0 : from[s]].opens_results.push_back(s);
    pr->schedule = std::make_shared<const Schedule>(std::move(S));
}

}  // namespace he::exec
