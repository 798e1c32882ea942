// Driver for test_layered_steps.py: a layered decoder whose device calls are stubs, so that what a step asks of the device can be looked at without one.
// One command a line on standard input, one JSON line out:
//     steps <config.json> <mode> <max sequences> <max rows>  then per step  s <entries>  and per entry  <sequence> <tokens> <copies of the last place wanted>;  f  recordings fail from here on;  n  no
//     place for logits is given from here on
#include <iostream>
#include <sstream>

#include "../m40-llm_amd/host/layered_decoder.hpp"

using namespace m40host;

namespace {

// The context of the program, the one that records if there is one, and what went where.
struct World {
    const void* own = nullptr;
    const void* capturing = nullptr;
    int launched = 0, recorded = 0, replays = 0, recordings = 0, destroyed = 0, blocking_copies = 0, recorders = 0;
    bool captured_shared = false, fail_recording = false;
    std::vector<std::string> head;         // what the head's norms and the last sums of the streams were given, launches only
    std::string order;                     // L a launch, R a recorded one, G a replay, B / E a recording's begin and end, X given up
    bool call(const void* ctx) {           // whether it is a launch
        const bool records = ctx == capturing;
        ++(records ? recorded : launched);
        if (order.empty() || order.back() != (records ? 'R' : 'L')) order += records ? 'R' : 'L';
        return !records;
    }
};
World world;

}  // namespace

#define STUB(name, result) extern "C" long long stub_##name(const void* ctx) asm(#name); long long stub_##name(const void* ctx) { (void)ctx; return result; }
#define LAUNCH(name) STUB(name, (!world.call(ctx) && world.fail_recording ? -1 : 0))
LAUNCH(m40llm_ext_advance_rows_async) LAUNCH(m40llm_ext_channel_delta_async) LAUNCH(m40llm_ext_clear_u32_async) LAUNCH(m40llm_ext_conv_state_async)
LAUNCH(m40llm_ext_copy_words_async) LAUNCH(m40llm_ext_delta_split_async) LAUNCH(m40llm_ext_embed_tokens_async) LAUNCH(m40llm_ext_gate_group_norm_rows_async)
LAUNCH(m40llm_ext_gather_rows_async) LAUNCH(m40llm_ext_head_attention_async) LAUNCH(m40llm_ext_latent_attention_async) LAUNCH(m40llm_ext_latent_split_append_async)
LAUNCH(m40llm_ext_layer_norm_rows_async) LAUNCH(m40llm_ext_lightning_async) LAUNCH(m40llm_ext_matrix_memory_async) LAUNCH(m40llm_ext_norm_add_rows_async)
LAUNCH(m40llm_ext_norm_gate_rows_async) LAUNCH(m40llm_ext_pack_tiles_async) LAUNCH(m40llm_ext_packed_gemm_async) LAUNCH(m40llm_ext_pair_attention_async)
LAUNCH(m40llm_ext_pair_split_append_async) LAUNCH(m40llm_ext_poly_norm_rows_async) LAUNCH(m40llm_ext_qkv_split_append_async) LAUNCH(m40llm_ext_rotation_angles_async)
LAUNCH(m40llm_ext_route_rows_async) LAUNCH(m40llm_ext_space_split_async) LAUNCH(m40llm_ext_time_mixing_async) LAUNCH(m40llm_ext_token_mix_async)
LAUNCH(m40llm_ext_top2_parts_async) LAUNCH(m40llm_ext_fill_random_bf16_async) LAUNCH(m40llm_memcpy_d2d_async)
STUB(m40llm_ext_channel_delta_state_floats, 4) STUB(m40llm_ext_expert_max_jobs, 64) STUB(m40llm_ext_expert_slots, 64) STUB(m40llm_ext_head_attention_serves, 1)
STUB(m40llm_ext_latent_attention_max_m_tiles, 4) STUB(m40llm_ext_latent_attention_partial_floats, 4) STUB(m40llm_ext_lightning_scratch_bytes, 4)
STUB(m40llm_ext_lightning_serves, 1) STUB(m40llm_ext_matrix_memory_state_floats, 4) STUB(m40llm_ext_memory_scratch_bytes, 4) STUB(m40llm_ext_memory_serves, 1)
STUB(m40llm_ext_pair_attention_partial_floats, 4) STUB(m40llm_ext_pair_attention_tile_queries, 64) STUB(m40llm_ext_pair_page_elements, 4)
STUB(m40llm_stream_synchronize, 0)

extern "C" {
int m40llm_device_malloc(M40llmCudaContext*, size_t bytes, void** out) { return (*out = std::calloc(bytes, 1)) ? 0 : -1; }
int m40llm_device_free(M40llmCudaContext*, void* p) { std::free(p); return 0; }
int m40llm_ext_pinned_malloc(M40llmCudaContext* ctx, size_t bytes, void** out) { return m40llm_device_malloc(ctx, bytes, out); }
int m40llm_ext_pinned_free(M40llmCudaContext* ctx, void* p) { return m40llm_device_free(ctx, p); }
int m40llm_memcpy_h2d(M40llmCudaContext*, void* dst, const void* src, size_t n) { std::memcpy(dst, src, n); return 0; }
int m40llm_memcpy_d2h(M40llmCudaContext*, void* dst, const void* src, size_t n) {
    if (!dst) return -1;
    std::memcpy(dst, src, n);
    ++world.blocking_copies;
    return 0;
}
int m40llm_ext_norm_rows_async(M40llmCudaContext* ctx, uint32_t, void*, const void*, uint32_t n_planes, uint64_t plane_stride, const void*, const uint32_t* index, uint32_t rows,
                               uint32_t, float, void*, uint32_t, uint32_t, uint32_t) {
    if (world.call(ctx) && index) world.head.push_back("norm " + std::to_string(n_planes) + " planes " + std::to_string(plane_stride) + " apart, rows " + std::to_string(rows));
    return 0;
}
int m40llm_ext_stream_update_async(M40llmCudaContext* ctx, const M40llmStreamUpdate* u, uint32_t) {
    if (world.call(ctx) && u->discard)
        world.head.push_back("sum " + std::to_string(u->n_planes) + " planes " + std::to_string(u->plane_stride) + " apart, mix " + std::to_string(u->mix != nullptr) +
                             ", experts " + std::to_string(u->expert_out != nullptr) + ", fresh " + std::to_string(u->x0 != nullptr) + ", rows " + std::to_string(u->rows));
    return 0;
}
static char recorder;
M40llmCudaContext* m40llm_ext_create_recorder(M40llmCudaContext* ctx) {
    ++world.recorders;
    return ctx == world.own ? reinterpret_cast<M40llmCudaContext*>(&recorder) : nullptr;
}
void m40llm_destroy_context(M40llmCudaContext*) {}
int m40llm_cuda_graph_begin_capture(M40llmCudaContext* ctx, uint32_t) {
    if (ctx == world.own) world.captured_shared = true;
    world.capturing = ctx;
    world.order += 'B';
    ++world.recordings;
    return 0;
}
int m40llm_cuda_graph_end_capture(M40llmCudaContext* ctx, uint32_t, M40llmCudaGraphExec** out) {
    if (ctx != world.capturing) return -1;
    world.capturing = nullptr;
    world.order += 'E';
    *out = reinterpret_cast<M40llmCudaGraphExec*>(new char);
    return 0;
}
int m40llm_cuda_graph_cancel_capture(M40llmCudaContext*, uint32_t) { world.capturing = nullptr; world.order += 'X'; return 0; }
int m40llm_cuda_graph_launch(M40llmCudaContext* ctx, M40llmCudaGraphExec*, uint32_t) {
    if (ctx != world.own || world.capturing) return -1;
    world.order += 'G';
    ++world.replays;
    return 0;
}
void m40llm_cuda_graph_destroy(M40llmCudaGraphExec* g) { delete reinterpret_cast<char*>(g); ++world.destroyed; }
}

static std::string quoted(const std::string& s) { return "\"" + s + "\""; }

static void steps(std::istream& in) {
    std::string path, op;
    uint32_t mode;
    LayeredOptions opt;
    opt.max_tokens = 65536;
    in >> path >> mode >> opt.max_sequences >> opt.max_rows;
    world = World{};
    char own;
    world.own = &own;
    RandomTensors tensors(1, 0.1f);
    std::ostringstream log;
    {
        LayeredDecoder d(reinterpret_cast<M40llmCudaContext*>(&own), read_decoder_spec(read_text_file(path)), tensors, opt);
        d.set_mode(mode);
        bool first = true, place = true;
        while (in >> op) {
            if (op == "n") {
                place = false;
                continue;
            }
            if (op == "f") {
                world.fail_recording = true;
                continue;
            }
            uint32_t n;
            in >> n;
            std::vector<std::vector<uint32_t>> tokens(n), want(n);
            std::vector<StepEntry> entries;
            size_t rows = 0;
            for (uint32_t i = 0; i < n; ++i) {
                uint32_t seq, len, copies;
                in >> seq >> len >> copies;
                tokens[i].assign(len, 1);
                want[i].assign(copies, len - 1);
                rows += copies;
                entries.push_back({seq, tokens[i].data(), len, want[i].data(), copies});
            }
            std::vector<float> logits(rows * d.vocab() + 1);
            const World before = world;
            world.head.clear();
            world.order.clear();
            d.step(entries, place ? logits.data() : nullptr);
            log << (first ? "" : ", ") << "{\"replays\": " << world.replays - before.replays << ", \"recordings\": " << world.recordings - before.recordings
                << ", \"destroyed\": " << world.destroyed - before.destroyed << ", \"recorders\": " << world.recorders - before.recorders << ", \"blocking_copies\": " << world.blocking_copies - before.blocking_copies << ", \"order\": " << quoted(world.order) << ", \"head\": [";
            for (size_t i = 0; i < world.head.size(); ++i) log << (i ? ", " : "") << quoted(world.head[i]);
            log << "]}";
            first = false;
        }
    }
    std::cout << "{\"steps\": [" << log.str() << "], \"captured_shared\": " << (world.captured_shared ? "true" : "false") << "}\n";
}

int main() {
    std::string line;
    while (std::getline(std::cin, line)) {
        std::istringstream in(line);
        std::string what;
        in >> what;
        try {
            if (what == "steps") steps(in);
        } catch (const std::exception& e) {
            std::cout << "{\"error\": " << quoted(e.what()) << "}\n";
        }
        std::cout.flush();
    }
    return 0;
}
