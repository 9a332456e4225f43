// Host side of the packed databases (gv_graph_set_owner, gv_resident_mine)
// without a device: one case a run, named by the first argument.
#include "fake_hip.h"
#include "geneva_hip.h"
#include "geneva_host.h"

#include <algorithm>
#include <new>

// host allocations until one throws (-1: none does)
static int fail_new = -1;
static bool new_failed = false;
void* operator new(size_t n) {
    if (fail_new >= 0 && fail_new-- == 0) {
        new_failed = true;
        throw std::bad_alloc();
    }
    if (void* p = std::malloc(n ? n : 1)) return p;
    throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }

namespace {

int fails = 0;
#define CHECK(x)                                                    \
    do {                                                            \
        if (!(x)) {                                                 \
            std::printf("line %d: not so: %s\n", __LINE__, #x);     \
            ++fails;                                                \
        }                                                           \
    } while (0)

// two graphs of one edge each: vertices 1-2 and 3-4, labels 1 and 2
const uint32_t kLabels[] = {4, 1, 2, 1, 2};
const uint32_t kBlock[] = {18, 4, 1, 0, 9, /*sources*/ 1, 0, 4, 0, /*lists*/ 0, 1, 2, 3, 4, /*neighbours*/ 2, 1, 4, 3};
const uint32_t kOwner[] = {0, 0, 0, 1, 1};

struct Db {
    gv_ctx_t c = nullptr;
    gv_graph_t g = nullptr;
    explicit Db(int device = 0) {
        const uint32_t* blocks[] = {kBlock};
        const uint32_t edge_label = 1;
        CHECK(gv_ctx_create(device, &c) == GV_OK);
        CHECK(gv_graph_create(c, kLabels, 1, blocks, &edge_label, &g) == GV_OK);
    }
    ~Db() {
        gv_graph_destroy(g);
        gv_ctx_destroy(c);
    }
    int mine() {
        gv_query_t q{};
        q.k = 2;
        q.step[1].label = 1;
        q.step[1].col = 1;
        q.step[1].nback = 1;
        q.step[1].restrict_col = GV_NONE;
        const gv_query_t* qs[] = {&q};
        uint64_t count = 0, bytes = 0;
        uint32_t word = 0, *bits[] = {&word};
        return gv_resident_mine(c, g, 1, qs, nullptr, &count, &bytes, bits, 1, nullptr);
    }
};

// accumulators that a call adds to start at zero, and results have a place
hipError_t accumulators(const std::string& name, void** args) {
    if (name.find("k_resident_out") == std::string::npos) return hipSuccess;
    const char* acc = *(char**)args[0];
    const uint32_t nacc = *(uint32_t*)args[1];
    CHECK(*(void**)args[2] != nullptr);
    bool zero = acc != nullptr;
    for (uint32_t i = 0; zero && i < 8 * nacc; ++i) zero = acc[i] == 0;
    CHECK(zero);
    return hipSuccess;
}

// After a call that found no memory the next one works.
void failed_allocation() {
    fake::on_launch = accumulators;
    for (int i = 0;; ++i) {
        Db db;
        CHECK(gv_graph_set_owner(db.g, kOwner, 2) == GV_OK);
        fake::failed = false;
        fake::fail_alloc = i;
        const int first = db.mine();
        fake::fail_alloc = -1;
        std::printf("allocation %d: %d\n", i, first);
        std::fflush(stdout);
        CHECK(fake::failed == (first != GV_OK));
        CHECK(db.mine() == GV_OK);
        if (!fake::failed) break;
        CHECK(i < 100);
    }
}

// A call that finds no memory says what a database that does not fit says
// (the caller's table engines mine it), and leaves no error behind.
void no_memory_is_capacity() {
    fake::sticky = true;
    for (int i = 0;; ++i) {
        Db db;
        CHECK(gv_graph_set_owner(db.g, kOwner, 2) == GV_OK);
        fake::failed = false;
        fake::fail_alloc = i;
        const int first = db.mine();
        fake::fail_alloc = -1;
        CHECK(first == (fake::failed ? GV_ERR_CAPACITY : GV_OK));
        CHECK(fake::last == hipSuccess);
        CHECK(db.mine() == GV_OK);
        if (!fake::failed) break;
        CHECK(i < 100);
    }
}

// What packing needs of its kernels: labels, and one segment with one
// neighbour for each vertex.
hipError_t pack_kernels(const std::string& name, void** args) {
    if (name.find("k_pack_labels") != std::string::npos) {
        const uint32_t* lverts = *(uint32_t**)args[0];
        const uint64_t n = *(uint64_t*)args[1], *lvoff = *(uint64_t**)args[2];
        const uint32_t nl = *(uint32_t*)args[3];
        uint32_t* lab = *(uint32_t**)args[4];
        for (uint32_t l = 0; l < nl; ++l)
            for (uint64_t i = lvoff[l]; i < lvoff[l + 1] && i < n; ++i) lab[lverts[i]] = l;
    } else if (name.find("k_pack_count") != std::string::npos) {
        const uint64_t nv1 = *(uint64_t*)args[2];
        for (int a : {3, 4})
            for (uint64_t v = 1; v < nv1; ++v) (*(uint32_t**)args[a])[v] = 1;
    }
    return hipSuccess;
}
uint64_t device_bytes(gv_graph_t g) {
    uint64_t b = 0;
    CHECK(gv_graph_info(g, nullptr, nullptr, nullptr, nullptr, &b) == GV_OK);
    return b;
}
uint64_t packed_bytes(gv_graph_t g) {
    uint32_t blocks = 0;
    uint64_t b = 0;
    CHECK(gv_resident_info(g, &blocks, &b) == GV_OK);
    CHECK((blocks == 0) == (b == 0));
    return b;
}

// The packed form counts once in a graph's bytes, however often its owners are set.
void owners_twice() {
    fake::on_launch = pack_kernels;
    Db db;
    const uint64_t bare = device_bytes(db.g);
    for (int i = 0; i < 3; ++i) {
        CHECK(gv_graph_set_owner(db.g, kOwner, 2) == GV_OK);
        CHECK(packed_bytes(db.g) > 0);
        CHECK(device_bytes(db.g) == bare + packed_bytes(db.g));
    }
    const uint32_t one[5] = {};   // one graph is not packed
    CHECK(gv_graph_set_owner(db.g, one, 1) == GV_OK);
    CHECK(packed_bytes(db.g) == 0);
    CHECK(device_bytes(db.g) == bare);
}

// Packing runs on the graph's device, whichever the calling thread used last.
hipError_t on_device_1(const std::string& name, void** args) {
    CHECK(fake::device == 1);
    return pack_kernels(name, args);
}
void owners_on_their_device() {
    Db db(1);
    fake::on_launch = on_device_1;
    fake::device = 0;
    CHECK(gv_graph_set_owner(db.g, kOwner, 2) == GV_OK);
    CHECK(packed_bytes(db.g) > 0);
}

// Owners are set also where the database cannot be packed: a launch of the
// packing fails, or a device allocation of its own.
int fail_launch = -1;
hipError_t some_launch_fails(const std::string& name, void** args) {
    if (fail_launch >= 0 && fail_launch-- == 0) {
        fake::failed = true;
        return hipErrorLaunchFailure;
    }
    return pack_kernels(name, args);
}
void packing_fails() {
    fake::on_launch = some_launch_fails;
    fake::sticky = true;
    for (int what = 0; what < 2; ++what)
        for (int i = 0;; ++i) {
            Db db;
            fake::failed = false;
            // allocation 0 is the owners' own
            (what ? fail_launch : fake::fail_alloc) = i + (what ? 0 : 1);
            CHECK(gv_graph_set_owner(db.g, kOwner, 2) == GV_OK);
            fail_launch = fake::fail_alloc = -1;
            CHECK(fake::last == hipSuccess);
            uint32_t n = 0;
            CHECK(gv_graph_owners(db.g, &n) == GV_OK && n == 2);
            CHECK((packed_bytes(db.g) == 0) == fake::failed);
            CHECK(db.mine() == (fake::failed ? GV_ERR_CAPACITY : GV_OK));
            if (!fake::failed) break;
            CHECK(i < 100);
        }
}

// No exception leaves the library: without host memory to pack in a database
// stays unpacked, without host memory for a call the table engines mine it.
void no_host_memory() {
    fake::on_launch = pack_kernels;
    for (int what = 0; what < 2; ++what)
        for (int i = 0;; ++i) {
            Db db;
            if (what) CHECK(gv_graph_set_owner(db.g, kOwner, 2) == GV_OK);
            new_failed = false;
            fail_new = i;
            const int rc = what ? db.mine() : gv_graph_set_owner(db.g, kOwner, 2);
            fail_new = -1;
            CHECK(rc == (what && new_failed ? GV_ERR_CAPACITY : GV_OK));
            uint32_t n = 0;
            CHECK(gv_graph_owners(db.g, &n) == GV_OK && n == 2);
            CHECK(db.mine() == (packed_bytes(db.g) ? GV_OK : GV_ERR_CAPACITY));
            if (!new_failed) break;
            CHECK(i < 1000);
        }
}

// Reading the slot engine's counters, or turning its profile off, makes no
// slot engine (device memory of slots x two tables) on a database that is
// mined without it.
void counters_without_slot_engine() {
    fake::on_launch = pack_kernels;
    const uint32_t labels[] = {0, 1, 2, 1, 2}, edges[] = {1, 2, 1, 3, 4, 1};
    gh_dataset_t ds = gh_ds_from_arrays(4, labels, 2, edges, kOwner, 2);
    CHECK(ds != nullptr);
    int rc = 0;
    gh_engine_t e = gh_engine_create(ds, 0, 1 << 20, &rc);
    CHECK(e != nullptr && rc == GV_OK);
    CHECK(gh_engine_resident_blocks(e) > 0);
    CHECK(gh_engine_batch_config(e, 4, 1 << 20, 1 << 16, 0, 0) == GV_OK);
    const char* q = "v 0 1\nv 1 2\ne 0 1 1\n";
    uint64_t count = 0, bytes = 0;
    uint32_t word = 0;
    CHECK(gh_engine_batch_mine(e, &q, 1, 0, &count, &bytes, &word, 1, nullptr) == GV_OK);
    const int held = fake::allocations;
    CHECK(gh_engine_batch_profile(e, 0) == GV_OK);
    uint64_t a = 1, b = 1, rows = 1, cand = 1;
    CHECK(gh_engine_batch_profile_bytes(e, &a, &b) == GV_OK && a == 0 && b == 0);
    uint32_t n = 1;
    CHECK(gh_engine_batch_history(e, &rows, &cand, 1, &n) == GV_OK && n == 0);
    CHECK(fake::allocations == held);
    gh_engine_free(e);
    gh_ds_free(ds);
}

// A packed database of two graphs: 60 vertices of label 1, all joined, and a
// pair; path(k) is a path of k vertices of label 1.
struct Served {
    gh_dataset_t ds = nullptr;
    gh_engine_t e = nullptr;
    double stats[6] = {};
    Served() {
        std::vector<uint32_t> labels(63, 1), edges, owner(63, 0);
        for (uint32_t a = 1; a <= 60; ++a)
            for (uint32_t b = a + 1; b <= 60; ++b) edges.insert(edges.end(), {a, b, 1});
        edges.insert(edges.end(), {61, 62, 1});
        owner[61] = owner[62] = 1;
        ds = gh_ds_from_arrays(62, labels.data(), edges.size() / 3, edges.data(), owner.data(), 2);
        int rc = 0;
        e = gh_engine_create(ds, 0, 1 << 20, &rc);
        CHECK(e != nullptr && rc == GV_OK);
        CHECK(gh_engine_resident_blocks(e) > 0);
        CHECK(gh_engine_batch_config(e, 4, 1 << 20, 1 << 16, 0, 0) == GV_OK);
    }
    ~Served() {
        gh_engine_free(e);
        gh_ds_free(ds);
    }
    static std::string path(int k) {
        std::string q;
        for (int i = 0; i < k; ++i) q += "v " + std::to_string(i) + " 1\n";
        for (int i = 0; i + 1 < k; ++i) q += "e " + std::to_string(i) + " " + std::to_string(i + 1) + " 1\n";
        return q;
    }
    std::vector<double> latency;
    int serve(std::vector<int> ks, uint64_t budget, double apart = 0.0) {   // requests this far apart
        std::vector<std::string> text;
        std::vector<const char*> q;
        for (int k : ks) text.push_back(path(k));
        for (auto& t : text) q.push_back(t.c_str());
        std::vector<double> at;
        for (size_t i = 0; i < ks.size(); ++i) at.push_back(apart * (double)i);
        latency.assign(ks.size(), 0.0);
        return gh_engine_serve(e, q.data(), at.data(), (uint32_t)ks.size(), 0, budget, latency.data(), nullptr, nullptr, 0, stats);
    }
};

// The memory bound of a turn holds after a request whose estimate is out of
// range as well.
void bound_after_huge_estimate() {
    fake::on_launch = pack_kernels;
    Served s;
    CHECK(s.serve({5, 5}, 1ull << 30) == GV_OK && s.stats[1] == 1);    // both in one turn
    CHECK(s.serve({14, 5}, 1ull << 30) == GV_OK && s.stats[1] == 2);   // 2^64 - 1 and some MB
    CHECK(s.serve({5, 14}, 1ull << 30) == GV_OK && s.stats[1] == 2);
}

// Requests that a turn could not take are reported as overflowed, not as sent
// straight to the plain path.
void refused_turn_is_overflow() {
    fake::on_launch = pack_kernels;
    Served s;
    fake::failed = false;
    fake::fail_alloc = 3;   // after the side worker's context: the turn's first buffer
    CHECK(s.serve({5, 5}, 1ull << 30) == GV_OK);
    fake::fail_alloc = -1;
    CHECK(fake::failed && s.stats[3] == 2 && s.stats[4] == 0);
    CHECK(s.serve({5, 5}, 1ull << 30) == GV_OK && s.stats[3] == 0 && s.stats[4] == 0);
}

// A query of 16 vertices whose levels take 27 KiB a wave, on a database with a
// graph of nearly 64 KiB: with three waves it fits LDS.
void wide_levels_beside_a_large_graph() {
    fake::on_launch = pack_kernels;
    // a path of n vertices and a pair, one label, as a partition block
    const uint32_t n = 4600, nv = n + 2;
    std::vector<uint32_t> labels(nv + 1, 1), owner(nv + 1, 0), at(1, 0), list;
    labels[0] = nv;
    owner[n + 1] = owner[n + 2] = 1;
    for (uint32_t v = 1; v <= nv; ++v) {
        if (v != 1 && v != n + 1) list.push_back(v - 1);
        if (v != n && v != nv) list.push_back(v + 1);
        at.push_back((uint32_t)list.size());
    }
    std::vector<uint32_t> block{0, nv, 1, 0, 4 + nv + 1, /*sources*/ 1, 0, nv, 0};
    block.insert(block.end(), at.begin(), at.end());
    // a list of up to 130 neighbours has no skip index before it
    block.insert(block.end(), list.begin(), list.end());
    block[0] = (uint32_t)block.size();
    const uint32_t* blocks[] = {block.data()};
    const uint32_t edge_label = 1;
    gv_ctx_t c = nullptr;
    gv_graph_t g = nullptr;
    CHECK(gv_ctx_create(0, &c) == GV_OK);
    CHECK(gv_graph_create(c, labels.data(), 1, blocks, &edge_label, &g) == GV_OK);
    CHECK(gv_graph_set_owner(g, owner.data(), 2) == GV_OK);
    CHECK(packed_bytes(g) > 64000);
    gv_query_t q{};
    q.k = 16;
    for (uint32_t w = 1; w < q.k; ++w) {
        gv_step_t& s = q.step[w];
        s.col = w;
        s.nback = 1;   // column 0
        s.restrict_col = GV_NONE;
    }
    // columns 0 to 9 are read by the last two steps, so every table keeps them
    q.step[15].nback = 3;
    q.step[15].back_col[1] = 1;
    q.step[15].back_col[2] = 2;
    q.step[15].ncoll = q.step[14].ncoll = 4;
    for (uint32_t i = 0; i < 4; ++i) {
        q.step[15].coll_col[i] = 3 + i;
        q.step[14].coll_col[i] = 6 + i;
    }
    const gv_query_t* qs[] = {&q};
    uint64_t count = 0, bytes = 0;
    CHECK(gv_resident_mine(c, g, 1, qs, nullptr, &count, &bytes, nullptr, 0, nullptr) == GV_OK);
    gv_graph_destroy(g);
    gv_ctx_destroy(c);
}

// A request that comes long after the one before it is mined at once, also
// with others to come.
void lone_request_does_not_wait() {
    fake::on_launch = pack_kernels;
    Served s;
    CHECK(s.serve(std::vector<int>(100, 5), 1ull << 30, 0.5e-3) == GV_OK);
    double least = 1e9;
    for (size_t i = 0; i + 1 < s.latency.size(); ++i) least = std::min(least, s.latency[i]);
    std::printf("least latency %.1f us\n", least * 1e3);
    CHECK(least < 20e-3);
}

// A call that sets aside more than there is room for gets more room in the
// next one, and does without where there is no memory for it.
uint32_t set_aside = 0;   // what the next launch sets aside
hipError_t sets_aside(const std::string& name, void** args) {
    if (name.find("k_resident_out") != std::string::npos) {
        **(uint32_t**)args[9] = set_aside;
        set_aside = 0;
    }
    return hipSuccess;
}
void room_for_tables_set_aside() {
    fake::on_launch = sets_aside;
    fake::sticky = true;
    Db db;
    CHECK(gv_graph_set_owner(db.g, kOwner, 2) == GV_OK);
    CHECK(db.mine() == GV_OK);
    int held = fake::allocations;
    set_aside = 5;
    CHECK(db.mine() == GV_OK && db.mine() == GV_OK && fake::allocations == held);
    set_aside = 1u << 20;
    CHECK(db.mine() == GV_OK && fake::allocations == held);
    fake::fail_alloc = 0;
    CHECK(db.mine() == GV_OK && fake::allocations == held && fake::last == hipSuccess);
    set_aside = 1u << 20;
    CHECK(db.mine() == GV_OK && db.mine() == GV_OK && fake::allocations == held + 1);
    set_aside = 1u << 20;
    CHECK(db.mine() == GV_OK && db.mine() == GV_OK && fake::allocations == held + 1);
}

}  // namespace

int main(int, char** argv) {
    const std::string what = argv[1];
    if (what == "failed_allocation") failed_allocation();
    else if (what == "no_memory_is_capacity") no_memory_is_capacity();
    else if (what == "owners_twice") owners_twice();
    else if (what == "owners_on_their_device") owners_on_their_device();
    else if (what == "packing_fails") packing_fails();
    else if (what == "no_host_memory") no_host_memory();
    else if (what == "counters_without_slot_engine") counters_without_slot_engine();
    else if (what == "bound_after_huge_estimate") bound_after_huge_estimate();
    else if (what == "refused_turn_is_overflow") refused_turn_is_overflow();
    else if (what == "wide_levels_beside_a_large_graph") wide_levels_beside_a_large_graph();
    else if (what == "lone_request_does_not_wait") lone_request_does_not_wait();
    else if (what == "room_for_tables_set_aside") room_for_tables_set_aside();
    else return 2;
    std::printf("%s: %d wrong\n", what.c_str(), fails);
    return fails ? 1 : 0;
}
