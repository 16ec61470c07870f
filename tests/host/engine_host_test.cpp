// engine_host_test.cpp -- the engine's host code over the stand-in device
// (stub_device.cpp): stream contexts, their output pools, and copies to the host.
// Run with the name of a case; exits 0 when it holds.
#include "../../eagleimp_amd/csrc/eimp_engine.cpp"

#include <chrono>
#include <ctime>

#include "stub_device.h"

namespace {

#define REQUIRE(x)                                                                          \
    do {                                                                                    \
        if (!(x)) {                                                                         \
            std::fprintf(stderr, "%s:%d: %s (%s)\n", __FILE__, __LINE__, #x, g_err.c_str()); \
            std::exit(1);                                                                   \
        }                                                                                   \
    } while (0)

constexpr size_t kN = 512, kM = 80000;

eimp_engine *engine() {
    static std::vector<uint64_t> site(kM * kN / 64, 0x5555555555555555ull);
    static std::vector<float> cM(kM, 0.5f);
    eimp_engine *e = nullptr;
    REQUIRE(eimp_engine_create(0, &e) == EIMP_OK);
    REQUIRE(eimp_engine_initialize(e, 2, unit_words(2), kM, kN, kN, kN / 8, site.data()) == EIMP_OK);
    REQUIRE(eimp_engine_set_panel_extras(e, cM.data(), nullptr, 0, nullptr) == EIMP_OK);
    return e;
}

struct Batch {
    std::vector<eimp_target> t;
    explicit Batch(const std::vector<std::pair<uint64_t, uint64_t>> &wk) {
        static const std::vector<uint64_t> gt(2 * unit_words(kM), 0);
        for (auto &x : wk) t.push_back(eimp_target{gt.data(), 0, x.first, x.second, -1});
    }
};

void submit(eimp_stream *s, const Batch &b) {
    REQUIRE(eimp_stream_submit(s, b.t.size(), b.t.data(), 0.125f) == EIMP_OK);
}
std::vector<eimp_target_result> wait(eimp_stream *s, const Batch &b) {
    std::vector<eimp_target_result> r(b.t.size());
    size_t nd = 0;
    REQUIRE(eimp_stream_wait(s, r.data(), &nd, nullptr) == EIMP_OK);
    REQUIRE(nd == 0);
    return r;
}
// rows of target j copied out, their digest the stand-in kernels'
void check_copy(eimp_stream *s, const Batch &b, size_t j) {
    const uint64_t W = b.t[j].W, K = b.t[j].K, Mp = 2 * (W / 4) + 1;
    const uint32_t RS = row_stride((uint32_t)K, LAYOUT_GPU);
    std::vector<uint32_t> rows(2 * Mp * RS);
    std::vector<int32_t> c0(Mp);
    REQUIRE(eimp_stream_copy_target(s, j, nullptr, nullptr, nullptr, nullptr, nullptr, c0.data(), rows.data(),
                                    nullptr) == EIMP_OK);
    uint64_t d = 0;
    for (size_t i = 0; i < rows.size(); i++) d += dig_word(i, rows[i]);
    REQUIRE(d == stub_digest((uint32_t)W, (uint32_t)K, LAYOUT_GPU));
    for (uint32_t r = 0; r < Mp; r++) REQUIRE(c0[r] == (int32_t)(r ^ W));
}

std::vector<eimp_stream *> shared_contexts(eimp_engine *e, int n, uint32_t flags) {
    std::vector<eimp_stream *> s(n, nullptr);
    REQUIRE(eimp_stream_create(e, 4, kM, kN, 64u << 20, flags, &s[0]) == EIMP_OK);
    for (int i = 1; i < n; i++) REQUIRE(eimp_stream_create_shared(s[0], 4, kM, kN, flags, &s[i]) == EIMP_OK);
    return s;
}

// Timed passes over two contexts on one pool, the digests of the last outputs,
// one target copied out, the context that made the pool closed first, then the
// same with contexts that are not timed.
void shared_pool_sequence(int rounds) {
    eimp_engine *e = engine();
    const std::vector<Batch> all = {Batch({{30000, 512}, {4000, 300}, {900, 64}}), Batch({{8000, 512}, {25000, 500}}),
                                    Batch({{40000, 65}}), Batch({{64, 1}, {20000, 511}, {1, 33}, {31000, 300}})};
    stub.build_us = 300;
    stub.prep_us = 100;
    for (int r = 0; r < rounds; r++)
        for (uint32_t flags : {(uint32_t)EIMP_STREAM_TIMED, 0u}) {
            auto s = shared_contexts(e, 2, flags);
            size_t next = r;
            std::vector<const Batch *> in(2, nullptr);
            for (int c = 0; c < 2; c++) submit(s[c], *(in[c] = &all[next++ % 4]));
            for (int k = 0; k < 8; k++) {
                const int c = k & 1;
                auto res = wait(s[c], *in[c]);
                for (size_t j = 0; j < res.size(); j++) REQUIRE(res[j].Mp == 2 * (in[c]->t[j].W / 4) + 1);
                if (k < 6) submit(s[c], *(in[c] = &all[next++ % 4]));
            }
            uint64_t dig[8];
            REQUIRE(eimp_stream_digest_outputs(s[0], dig) == EIMP_ERR_STATE);
            eimp_stream_destroy(s[0]);
            REQUIRE(eimp_stream_digest_outputs(s[1], dig) == EIMP_OK);
            for (size_t j = 0; j < in[1]->t.size(); j++) {
                REQUIRE(dig[2 * j] == stub_digest((uint32_t)in[1]->t[j].W, (uint32_t)in[1]->t[j].K, LAYOUT_GPU));
                check_copy(s[1], *in[1], j);
            }
            eimp_stream_destroy(s[1]);
        }
    eimp_engine_destroy(e);
}

// Two contexts on one pool, each driven by its own thread.
void shared_pool_threads(int rounds) {
    eimp_engine *e = engine();
    auto s = shared_contexts(e, 2, 0);
    std::atomic<int> copied{0}, refused{0};
    auto drive = [&](int c) {
        Batch b({{(uint64_t)(12000 + 9000 * c), 512}, {700, 90}});
        std::vector<uint32_t> rows(2 * (2 * (b.t[0].W / 4) + 1) * row_stride(512, LAYOUT_GPU));
        for (int r = 0; r < rounds; r++) {
            submit(s[c], b);
            wait(s[c], b);
            const int rc = eimp_stream_copy_target(s[c], 0, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr,
                                                   rows.data(), nullptr);
            if (rc == EIMP_ERR_STATE) {
                refused++;
                continue;
            }
            REQUIRE(rc == EIMP_OK);
            uint64_t d = 0;
            for (size_t i = 0; i < rows.size(); i++) d += dig_word(i, rows[i]);
            REQUIRE(d == stub_digest((uint32_t)b.t[0].W, 512, LAYOUT_GPU));
            copied++;
        }
    };
    std::thread a(drive, 0), b(drive, 1);
    a.join();
    b.join();
    std::printf("copied %d refused %d\n", copied.load(), refused.load());
    for (auto *x : s) eimp_stream_destroy(x);
    eimp_engine_destroy(e);
}

// A context with a pool of its own replays its two graphs; contexts on a pool
// that more than one context uses launch their kernels one by one, the one that
// made the pool included, also after the others are closed.
void shared_pool_without_graphs(int) {
    eimp_engine *e = engine();
    const Batch b({{30000, 512}, {4000, 300}});
    auto s = shared_contexts(e, 1, 0);
    auto pass = [&](eimp_stream *x) {
        stub.graphs = 0;
        submit(x, b);
        wait(x, b);
        check_copy(x, b, 0);
        check_copy(x, b, 1);
        return stub.graphs.load();
    };
    REQUIRE(pass(s[0]) == 2);
    eimp_stream *other = nullptr;
    REQUIRE(eimp_stream_create_shared(s[0], 4, kM, kN, 0, &other) == EIMP_OK);
    REQUIRE(pass(s[0]) == 0);
    REQUIRE(pass(other) == 0);
    eimp_stream_destroy(other);
    REQUIRE(pass(s[0]) == 0);
    eimp_stream_destroy(s[0]);
    eimp_engine_destroy(e);
}

// A copy that fails returns only when nothing writes to the caller's memory any
// more: the rows go straight to pinned memory, then the chunks' buffer cannot be
// had, or the gather of the other array does not start.
void failed_copy_leaves_nothing_in_flight(int) {
    eimp_engine *e = engine();
    const Batch b({{20000, 512}});
    auto s = shared_contexts(e, 1, 0);
    submit(s[0], b);
    wait(s[0], b);
    const size_t Mp = 2 * (20000 / 4) + 1, words = 2 * Mp * row_stride(512, LAYOUT_GPU);
    void *rows = nullptr;
    REQUIRE(hipHostMalloc(&rows, words * 4, 0) == hipSuccess);
    std::vector<int32_t> c0(Mp);
    stub.copy_us = 30000;
    for (int way = 0; way < 2; way++) {
        stub.copies = stub.copies_done = stub.gathers = 0;
        stub.fail_host_malloc = way == 0;
        stub.fail_gather = way == 1 ? 0 : -1;
        REQUIRE(eimp_stream_copy_target(s[0], 0, nullptr, nullptr, nullptr, nullptr, nullptr, c0.data(),
                                        static_cast<uint32_t *>(rows), nullptr) != EIMP_OK);
        REQUIRE(stub.copies == 1 && stub.copies_done == 1);
    }
    stub.fail_host_malloc = false;
    stub.fail_gather = -1;
    stub.copy_us = 0;
    check_copy(s[0], b, 0);
    (void)hipHostFree(rows);
    eimp_stream_destroy(s[0]);
    eimp_engine_destroy(e);
}

// The threads that move chunks on do not run while the device has not filled
// them: five chunks, 60 ms each, are copied with far less processor time than
// they take.
void waiting_for_the_device_is_idle(int) {
    eimp_engine *e = engine();
    const Batch b({{80000, 512}});  // 10.2 MB of rows
    auto s = shared_contexts(e, 1, 0);
    submit(s[0], b);
    wait(s[0], b);
    const size_t Mp = 2 * (80000 / 4) + 1;
    std::vector<uint32_t> rows(2 * Mp * row_stride(512, LAYOUT_GPU));
    auto copy = [&] {
        REQUIRE(eimp_stream_copy_target(s[0], 0, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, rows.data(),
                                        nullptr) == EIMP_OK);
    };
    copy();  // makes the buffers and the threads, touches the rows
    auto cpu_ms = [] { return 1e3 * (double)std::clock() / CLOCKS_PER_SEC; };
    stub.gathers = 0;
    stub.gather_us = 60000;
    const auto t0 = std::chrono::steady_clock::now();
    const double c0 = cpu_ms();
    copy();
    const double cpu = cpu_ms() - c0;
    const double wall = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
    std::fprintf(stderr, "%d chunks: %.1f ms, %.1f ms of processor time\n", stub.gathers.load(), wall, cpu);
    REQUIRE(stub.gathers >= 4 && wall > 200);
    REQUIRE(cpu < wall / 4);
    stub.gather_us = 0;
    check_copy(s[0], b, 0);
    eimp_stream_destroy(s[0]);
    eimp_engine_destroy(e);
}

// The chains of targets with these row counts at this K are all cut, from one
// workgroup on a compute unit to eight.
void cut(int argc, char **argv) {
    std::vector<uint32_t> nblk, Kpad;
    for (int i = 3; i < argc; i++) {
        nblk.push_back(((uint32_t)std::atoi(argv[i]) + 15) / 16);
        Kpad.push_back((uint32_t)round_up(std::atoi(argv[2]), 64));
    }
    REQUIRE(!nblk.empty());
    for (uint32_t occ = 1; occ <= 8; occ++) {
        bool latency = false;
        const uint32_t L = choose_segments(nblk, Kpad, 256 * (10 + 2 * (occ - 1)), kSegBytes / 2, ~0u, 256, &latency);
        for (uint32_t nb : nblk) {
            uint32_t len = 0;
            REQUIRE(seg_split(nb, L, len) >= 3);
        }
    }
}

// Several arrays in one copy, as the drop-in call has: ends on, before and behind
// the edges of chunks, of the four buffers and of the pieces that a chunk holds.
void arrays_at_chunk_edges(int) {
    HostCopier c;
    hipStream_t s = nullptr;
    REQUIRE(hipStreamCreateWithFlags(&s, 0) == hipSuccess);
    constexpr size_t C = HostCopier::kChunk;
    const std::vector<std::vector<size_t>> sets = {
        {C}, {C - 4}, {C + 4}, {C, C}, {C - 16, 16, C}, {C - 16, 4, 4}, {C - 4, 4, 4}, {4 * C, 4}, {4 * C - 8, C + 8, 12},
        {8 * C + 4, 0, C - 4}, std::vector<size_t>(kGatherPieces, 20), std::vector<size_t>(kGatherPieces + 1, 20),
        std::vector<size_t>(3 * kGatherPieces + 2, C / kGatherPieces / 4 * 4)};
    for (const auto &set : sets) {
        std::vector<std::vector<uint32_t>> src, dst;
        std::vector<HostCopier::Job> jobs;
        for (size_t b : set) {
            src.emplace_back(b / 4 + 1);
            for (size_t i = 0; i < src.back().size(); i++) src.back()[i] = (uint32_t)((i + b) * 2654435761u + src.size());
            dst.emplace_back(b / 4 + 1, 7u);
        }
        for (size_t i = 0; i < set.size(); i++) jobs.push_back({dst[i].data(), src[i].data(), set[i]});
        REQUIRE(c.run(jobs, s) == EIMP_OK);
        for (size_t i = 0; i < set.size(); i++) {
            REQUIRE(std::equal(dst[i].begin(), dst[i].end() - 1, src[i].begin()));
            REQUIRE(dst[i].back() == 7u);
        }
    }
    c.release();
    (void)hipStreamDestroy(s);
}

}  // namespace

int main(int argc, char **argv) {
    const std::string name = argc > 1 ? argv[1] : "";
    const int rounds = argc > 2 ? std::atoi(argv[2]) : 3;
    if (name == "shared_pool_sequence") shared_pool_sequence(rounds);
    else if (name == "shared_pool_threads") shared_pool_threads(rounds);
    else if (name == "shared_pool_without_graphs") shared_pool_without_graphs(rounds);
    else if (name == "failed_copy_leaves_nothing_in_flight") failed_copy_leaves_nothing_in_flight(rounds);
    else if (name == "waiting_for_the_device_is_idle") waiting_for_the_device_is_idle(rounds);
    else if (name == "cut") cut(argc, argv);
    else if (name == "arrays_at_chunk_edges") arrays_at_chunk_edges(rounds);
    else return 2;
    std::printf("ok %s\n", name.c_str());
    return 0;
}
