// Host-side tests of the engine on a device in host memory (fake_device.hpp): what a prefill reports and how it is cut
// into chunks, the buffers of sessions, and allocations that fail.
#include "fake_device.hpp"

#include <memory>
#include <string>
#include <vector>

using namespace jfh;

namespace {

int failures = 0;

void expect(bool ok, const std::string& what) {
    if (ok) return;
    ++failures;
    std::printf("FAIL: %s\n", what.c_str());
}

constexpr uint32_t kVocab = 512, kCtx = 8192, kLayers = 3, kEmbd = 512, kFf = 768, kHeads = 8, kKvHeads = 2, kDim = 64;

std::unique_ptr<Engine> engine(uint32_t layer_start = 0, uint32_t layer_end = kLayers, uint32_t kv_heads = kKvHeads) {
    SynthSpec spec;
    spec.params = {kLayers, kEmbd, kFf, kHeads, kv_heads, kCtx, kVocab, kDim, 1.0e6F, 1.0e-6F};
    const auto model = HostModel::synthesize(spec);
    if (layer_start == 0 && layer_end == kLayers) return std::make_unique<Engine>(*model, EngineOptions{});
    return std::make_unique<Engine>(*model->slice(layer_start, layer_end), EngineOptions{});
}

std::vector<int32_t> prompt(uint32_t n) {
    std::vector<int32_t> ids(n);
    for (uint32_t i = 0; i < n; ++i) ids[i] = static_cast<int32_t>(i * 7 % kVocab);
    return ids;
}

// The workspace a prefill reports: what its longest chunk's rows take, with logits rows and attention partials for
// the rows of a step only.
void test_prefill_scratch() {
    const auto e = engine();
    auto act8 = [](uint64_t K) { return K + K / 32 * 4 + K / 16 * 2; };
    constexpr uint64_t F = 4;
    const uint64_t row = (kEmbd + 2 * kHeads * kDim + kFf) * F + act8(kHeads * kDim) + act8(kFf) + act8(kEmbd);
    for (uint32_t n : {1u, 100u, 256u, 300u, 1500u, 2048u, 2200u, 5000u}) {
        const auto s = e->create_session(n);
        e->prefill(*s, prompt(n).data(), n, nullptr);
        const uint32_t chunks = s->prefill_metrics().steps;
        const BufferMetrics m = e->buffer_metrics(n, n, s->prefill_metrics());
        const uint64_t wide = m.decode_scratch_bytes - row;  // a row's logits and attention partials
        // the longest of about equally long chunks
        const uint64_t longest = chunks == 1 ? n : ((n + chunks - 1) / chunks + 127) / 128 * 128;
        expect(wide >= kVocab * F && wide <= kVocab * F + 32 * kHeads * (kDim + 2) * F, "decode scratch of a row");
        expect(m.prefill_scratch_bytes == longest * row + std::min<uint64_t>(longest, 256) * wide,
               "prefill scratch of " + std::to_string(n) + " tokens: " + std::to_string(m.prefill_scratch_bytes));
        expect(m.prefill_scratch_bytes <= fake::live_bytes, "prefill scratch exceeds what is allocated");
    }
}

// A prefill's allocation time holds the clearing of its session's cache (48 MB), in a new buffer and in one kept from a
// closed session; its compute time does not.
void test_allocation_time() {
    const auto e = engine(0, kLayers, kHeads);
    for (int i = 0; i < 3; ++i) {
        const auto s = e->create_session(kCtx);
        const double clearing = 100.0 * static_cast<double>(s->kv_bytes()) / (1 << 20);
        e->prefill(*s, prompt(2500).data(), 2500, nullptr);
        const PrefillMetrics& m = s->prefill_metrics();
        expect(m.allocation_ms >= 0.999 * clearing, "allocation time " + std::to_string(m.allocation_ms) + " ms, clearing " + std::to_string(clearing));
        expect(m.compute_ms > 0.0 && m.compute_ms < 0.5 * clearing, "compute time " + std::to_string(m.compute_ms));
    }
}

template <typename F>
bool refused(F&& f) {
    try {
        f();
    } catch (const Error&) {
        return true;
    }
    return false;
}

// A session that the device has no memory for leaves the engine and its open sessions usable.
void test_failed_capacity() {
    for (size_t limit : {size_t{0}, size_t{100} << 10, size_t{3} << 20}) {  // refusing the rope table, the partials, the cache
        const auto e = engine();
        const auto s = e->create_session(300);
        e->prefill(*s, prompt(200).data(), 200, nullptr);
        SeqStep st;
        const int32_t id = 3;
        st.session = s.get();
        st.tokens = &id;
        st.n = 1;
        e->forward({st}, nullptr, nullptr, nullptr);
        fake::fail_from = (size_t{100} << 10) + limit;
        fake::memory = fake::live_bytes + limit;
        expect(refused([&] { (void) e->create_session(kCtx); }), "a session larger than the device's memory");
        fake::memory = fake::fail_from = ~size_t{0};
        try {
            e->forward({st}, nullptr, nullptr, nullptr);
        } catch (const std::exception& err) {
            expect(false, std::string("step after a refused session: ") + err.what());
            continue;
        }
        expect(s->position() == 202, "step after a refused session");
        const auto t = e->create_session(kCtx);
        e->forward({st}, nullptr, nullptr, nullptr);
    }
}

// Buffers kept for later sessions are given back before any allocation of any engine is refused.
void test_kept_buffers_given_back() {
    const auto e = engine();
    { const auto warm = e->create_session(kCtx); }  // the rope table and partials of the longest session
    const auto other = engine();
    auto full = [&](auto&& call, const std::string& what) {
        { const auto s = e->create_session(kCtx); }  // 8 MB, kept
        fake::memory = fake::live_bytes;
        try {
            call();
        } catch (const Error& err) {
            expect(false, what + ": " + err.what());
        }
        fake::memory = ~size_t{0};
    };
    std::vector<float> x(kEmbd), y(kVocab * kEmbd);
    full([&] { e->matmul("blk.0.attn_output.weight", x.data(), 1, y.data()); }, "matmul");
    full([&] { e->dequantize("blk.0.attn_output.weight", 0, 1, y.data()); }, "dequantize");
    full([&] { (void) other->create_session(1000); }, "another engine's session");
    full([&] { (void) other->create_session(1050); }, "another engine's rope table and partials");
}

// What depends on another thread or on the time between two calls may fail on a busy machine, though not every time.
template <typename F>
bool sooner_or_later(F&& f) {
    for (int i = 0; i < 8; ++i) {
        if (f()) return true;
    }
    return false;
}

template <typename F>
void elsewhere(F&& f) {
    std::thread(f).join();
}

// A prompt alone runs in few long chunks; while another session steps, in chunks that hold the engine for 384 rows at
// most and let every waiting step pass.
void test_prefill_shares_the_engine() {
    const auto e = engine();
    constexpr uint32_t n = 4200;
    const std::vector<int32_t> ids = prompt(n);
    auto chunks = [&](bool steps_between = true) {
        const auto s = e->create_session(n);
        e->prefill(*s, ids.data(), n, nullptr, steps_between);
        return s->prefill_metrics().steps;
    };
    auto step = [&](Session& s) {
        const int32_t id = 5;
        SeqStep st;
        st.session = &s;
        st.tokens = &id;
        st.n = 1;
        e->forward({st}, nullptr, nullptr, nullptr);
    };
    expect(chunks() == 3, "chunks of a prompt alone");
    {
        const auto other = e->create_session(4000);
        e->prefill(*other, ids.data(), 300, nullptr);
        expect(chunks() == 3, "chunks beside a session that does not step");
        step(*other);
        expect(chunks() == 3, "chunks after a step of the same thread");
        elsewhere([&] { step(*other); });
        expect(chunks(false) == 3, "chunks of a caller that lets no session step meanwhile");
        expect(sooner_or_later([&] {
                   elsewhere([&] { step(*other); });
                   return chunks() > 3;
               }), "chunks beside a session that has just stepped");
        std::this_thread::sleep_for(std::chrono::milliseconds(40));
        expect(chunks() == 3, "chunks beside a session that stepped long ago");
        elsewhere([&] { step(*other); });
    }
    expect(chunks() == 3, "chunks after the other session was closed");

    const auto other = e->create_session(4000);
    e->prefill(*other, ids.data(), 10, nullptr);
    std::atomic<bool> done{false};
    std::atomic<int> steps{0};
    fake::us_per_256_rows = 1000;
    std::thread decoder([&] {
        while (!done) {
            step(*other);
            ++steps;
        }
    });
    while (steps < 5) std::this_thread::yield();
    std::string seen;
    const bool shared = sooner_or_later([&] {
        fake::longest_step = 0;
        const int before = steps;
        const uint32_t count = chunks();
        const int during = steps - before;
        seen = std::to_string(during) + " steps passed " + std::to_string(count) + " chunks of up to " + std::to_string(fake::longest_step) + " rows";
        return fake::longest_step <= 384 && count >= 11 && during >= 8;
    });
    expect(shared, "beside a decoding session " + seen);
    done = true;
    decoder.join();
    fake::us_per_256_rows = 0;
}

// A stage's rows come out where they belong whatever the chunks.
void test_stage_rows() {
    const auto e = engine(1, 2);
    for (uint32_t n : {1u, 300u, 1500u, 2049u, 2600u}) {
        std::vector<float> rows(static_cast<size_t>(n) * kEmbd), out(rows.size());
        for (size_t i = 0; i < rows.size(); ++i) rows[i] = static_cast<float>(i % 9973);
        for (bool busy : {false, true}) {
            const auto other = e->create_session(kCtx);
            e->stage_prefill(*other, nullptr, rows.data(), 1, out.data());
            uint32_t chunks = 0;
            const uint32_t want = busy ? (n + 383) / 384 : (n + 2047) / 2048;
            const bool cut = sooner_or_later([&] {
                if (busy) elsewhere([&] { e->stage_decode(*other, nullptr, rows.data(), out.data()); });
                const auto s = e->create_session(n);
                std::fill(out.begin(), out.end(), -1.0F);
                e->stage_prefill(*s, nullptr, rows.data(), n, out.data());
                expect(rows == out && s->position() == n, "rows of a stage, " + std::to_string(n));
                chunks = s->prefill_metrics().steps;
                return chunks == want;
            });
            expect(cut, "chunks of a stage, " + std::to_string(n) + ": " + std::to_string(chunks));
        }
    }
}

}  // namespace

int main() {
    test_prefill_shares_the_engine();
    test_stage_rows();
    test_failed_capacity();
    test_kept_buffers_given_back();
    test_allocation_time();
    test_prefill_scratch();
    failures += fake::faults;
    if (failures == 0) std::printf("engine tests passed\n");
    return failures == 0 ? 0 : 1;
}
