// Launch plans.  A forward or backward pass of one (stage, micro-batch) is the same thirty to several hundred launches on
// the same static buffers in every batch; what its Python callers spend on it -- descriptors, checks, foreign-function
// calls, about 10 us a launch -- is more than a small kernel runs.  The pass is recorded while it is issued for the first
// time (bb_launch copies each launch's kernel, grid and argument bytes here) and afterwards issued by one call that walks
// the records: about 2 us a launch, and unlike a captured graph it needs no special stream, and dropout keys can change.
// What a pass is given -- its input, the gradient it receives, key lengths -- is not part of the records: the places that
// hold those addresses are found once (bb_plan_operands) and filled in at every launch.
#include "common.h"

#include <new>
#include <vector>

thread_local BbPlan* bb_recording = nullptr;

struct BbPlan {
    struct Launch {
        const void* fn;
        dim3 grid, block;
        uint32_t lds, first_arg;
    };
    struct Drop {
        size_t at;     // byte offset of a DropKey among the argument bytes
        int32_t key;   // which of `keys`
    };
    struct Key {
        int64_t base_seed, micro_batch, layer, site;
    };
    struct Slot {
        size_t at;         // byte offset of a pointer among the argument bytes
        int32_t operand;   // whose address it takes ...
        uint64_t offset;   // ... and how far behind it
    };
    std::vector<Launch> launches;
    std::vector<size_t> arg_at;           // byte offset of every argument
    std::vector<unsigned char> bytes;     // argument bytes, 16-byte aligned each
    std::vector<void*> args;              // arg_at as pointers, once `bytes` has stopped growing
    std::vector<Drop> drops;
    std::vector<Key> keys;
    std::vector<size_t> pointers;         // byte offsets of all pointers
    std::vector<Slot> slots;
    int operands = 0;
    bool incomplete = false;              // a record found no memory
};

void bb_record_launch(const void* fn, dim3 grid, dim3 block, size_t lds, int nargs, void* const* args, const BbArgType* types) {
    BbPlan& p = *bb_recording;
    try {
        p.launches.push_back({fn, grid, block, (uint32_t)lds, (uint32_t)p.arg_at.size()});
        for (int i = 0; i < nargs; ++i) {
            const BbArgType& t = types[i];
            const size_t at = p.bytes.size();
            p.bytes.resize(at + (t.size + 15) / 16 * 16);
            memcpy(p.bytes.data() + at, args[i], t.size);
            p.arg_at.push_back(at);
            for (uint32_t k = 0; k < t.pointers; ++k) p.pointers.push_back(at + t.pointer_at[k]);
            if (t.drop_at >= 0) {
                DropKey k;
                memcpy(&k, p.bytes.data() + at + t.drop_at, sizeof(k));
                if (k.thresh) p.drops.push_back({at + (size_t)t.drop_at, -1});
            }
        }
    } catch (const std::bad_alloc&) {   // the launch itself has gone out; bb_plan_end refuses the plan
        p.incomplete = true;
    }
}

// the key of one dropout mask: a splitmix64 chain over what identifies it (the host mirror of it is
// bamboo_amd.hip.dropout_key)
static void dropout_key(const int64_t (&id)[5], uint32_t& k0, uint32_t& k1) {
    uint64_t z = 0x9E3779B97F4A7C15ull;
    for (int64_t v : id) {
        z += (uint64_t)v * 0xBF58476D1CE4E5B9ull + 0x9E3779B97F4A7C15ull;
        z ^= z >> 30; z *= 0xBF58476D1CE4E5B9ull;
        z ^= z >> 27; z *= 0x94D049BB133111EBull;
        z ^= z >> 31;
    }
    k0 = (uint32_t)z;
    k1 = (uint32_t)(z >> 32);
}

#define BB_NO_MEMORY(what)                    \
    catch (const std::bad_alloc&) {           \
        bb_set_error(what ": out of memory"); \
        return BB_EINVAL;                     \
    }

extern "C" int bb_plan_begin(void) {
    BB_REQUIRE(!bb_recording, "bb_plan_begin: this thread is already recording a plan");
    bb_recording = new (std::nothrow) BbPlan;
    BB_REQUIRE(bb_recording, "bb_plan_begin: out of memory");
    return BB_OK;
}

extern "C" int bb_plan_abort(void) {
    delete bb_recording;
    bb_recording = nullptr;
    return BB_OK;
}

extern "C" int bb_plan_end(void** plan_out) {
    BB_REQUIRE(bb_recording && plan_out, "bb_plan_end: this thread is not recording a plan");
    BbPlan* p = bb_recording;
    bb_recording = nullptr;
    try {
        p->args.reserve(p->arg_at.size() + 1);
    } catch (const std::bad_alloc&) {
        p->incomplete = true;
    }
    if (p->incomplete) {
        delete p;
        bb_set_error("bb_plan_end: out of memory");
        return BB_EINVAL;
    }
    for (size_t at : p->arg_at) p->args.push_back(p->bytes.data() + at);
    p->args.push_back(nullptr);
    *plan_out = p;
    return BB_OK;
}

extern "C" int bb_plan_dropout(void* plan, int count, const uint32_t* k0, const uint32_t* k1, const int64_t* base_seed,
                               const int64_t* micro_batch, const int64_t* layer, const int64_t* site) {
    BB_REQUIRE(plan && count >= 0 && (count == 0 || (k0 && k1 && base_seed && micro_batch && layer && site)), "bb_plan_dropout: null argument");
    BbPlan& p = *(BbPlan*)plan;
    try {
        p.keys.clear();
        for (int i = 0; i < count; ++i) p.keys.push_back({base_seed[i], micro_batch[i], layer[i], site[i]});
    }
    BB_NO_MEMORY("bb_plan_dropout")
    for (BbPlan::Drop& d : p.drops) {
        DropKey k;
        memcpy(&k, p.bytes.data() + d.at, sizeof(k));
        d.key = -1;
        for (int i = 0; i < count && d.key < 0; ++i)
            if (k.k0 == k0[i] && k.k1 == k1[i]) d.key = i;
        BB_REQUIRE(d.key >= 0, "bb_plan_dropout: the plan holds a dropout key that is not listed");
    }
    return BB_OK;
}

extern "C" int bb_plan_operands(void* plan, int count, const uint64_t* address, const int64_t* bytes) {
    BB_REQUIRE(plan && count >= 0 && (count == 0 || (address && bytes)), "bb_plan_operands: null argument");
    BbPlan& p = *(BbPlan*)plan;
    BB_REQUIRE(p.operands == 0, "bb_plan_operands: this plan's operands have been named");
    for (int i = 0; i < count; ++i)
        for (int j = 0; j < i; ++j)
            BB_REQUIRE(bytes[i] <= 0 || bytes[j] <= 0 || address[i] + (uint64_t)bytes[i] <= address[j] || address[j] + (uint64_t)bytes[j] <= address[i],
                       "bb_plan_operands: operands %d and %d overlap: whose a pointer is cannot be told", j, i);
    try {
        for (size_t at : p.pointers) {
            uint64_t v;
            memcpy(&v, p.bytes.data() + at, sizeof(v));
            for (int i = 0; i < count; ++i)
                if (bytes[i] > 0 && v - address[i] < (uint64_t)bytes[i]) p.slots.push_back({at, i, v - address[i]});
        }
    } catch (const std::bad_alloc&) {
        p.slots.clear();
        bb_set_error("bb_plan_operands: out of memory");
        return BB_EINVAL;
    }
    p.operands = count;
    return BB_OK;
}

extern "C" int bb_plan_launches(void* plan) { return plan ? (int)((BbPlan*)plan)->launches.size() : 0; }

extern "C" int bb_plan_launch(void* plan, int64_t step, void* stream) { return bb_plan_launch_on(plan, 0, nullptr, step, stream); }

extern "C" int bb_plan_launch_on(void* plan, int count, const uint64_t* address, int64_t step, void* stream) {
    BB_REQUIRE(plan, "bb_plan_launch: null plan");
    BbPlan& p = *(BbPlan*)plan;
    BB_REQUIRE(count == p.operands && (count == 0 || address), "bb_plan_launch: the plan has %d operands, %d are given", p.operands, count);
    for (const BbPlan::Drop& d : p.drops) {
        BB_REQUIRE(d.key >= 0, "bb_plan_launch: the plan's dropout keys have not been named (bb_plan_dropout)");
        const BbPlan::Key& k = p.keys[d.key];
        DropKey* dst = (DropKey*)(p.bytes.data() + d.at);
        dropout_key({k.base_seed, step, k.micro_batch, k.layer, k.site}, dst->k0, dst->k1);
    }
    for (const BbPlan::Slot& s : p.slots) {
        const uint64_t v = address[s.operand] + s.offset;
        memcpy(p.bytes.data() + s.at, &v, sizeof(v));
    }
    for (const BbPlan::Launch& l : p.launches)
        BB_HIP_CHECK(hipLaunchKernel(l.fn, l.grid, l.block, p.args.data() + l.first_arg, l.lds, (hipStream_t)stream));
    return BB_OK;
}

extern "C" int bb_plan_destroy(void* plan) {
    delete (BbPlan*)plan;
    return BB_OK;
}
