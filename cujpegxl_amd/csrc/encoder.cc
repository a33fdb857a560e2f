// Frame encoder orchestration (frame_encoder.cu:88-352 in the reference):
// one stream, buffers allocated once per configuration, every stage on the
// device, and exactly two host synchronizations per frame -- one to learn the
// file size, one after copying the file out.
#include "encoder.h"

#include <algorithm>
#include <atomic>
#include <cstring>
#include <memory>
#include <mutex>
#include <new>
#include <utility>

#include "kernels.h"
#include "prefix.h"

namespace cjx {
namespace {

// Host bit writer over a growable word vector.
struct HostBits {
    std::vector<std::uint32_t> words = std::vector<std::uint32_t>(16, 0u);
    std::uint32_t pos{0};
    void write(std::uint32_t n, std::uint32_t v) {
        while ((pos + n + 64) / 32 >= words.size()) {
            words.resize(words.size() * 2, 0u);
        }
        BitSink s{words.data(), pos, static_cast<std::uint32_t>(words.size() * 32)};
        s.write(n, v);
        pos = s.pos;
    }
    void pad() { pos = (pos + 7u) & ~7u; }
    void append(const HostBits& o) { copy_bits(*this, o.words.data(), o.pos); }
};

constexpr Distr kDimEnc[4]{{false, 1, 9}, {false, 1, 13}, {false, 1, 18}, {false, 1, 30}};
constexpr Distr kGlobalScaleEnc[4]{{false, 1, 11}, {false, 2049, 11}, {false, 4097, 12}, {false, 8193, 16}};
constexpr Distr kQuantDcEnc[4]{{true, 16, 0}, {false, 1, 5}, {false, 1, 8}, {false, 1, 16}};
constexpr Distr kOrderEnc[4]{{true, 0x5F, 0}, {true, 0x13, 0}, {true, 0, 0}, {false, 0, 13}};

// write_prefix_histograms (histogram_writer.cc:59-83) for constant alphabets.
void prefix_histograms(HostBits& w, const std::uint32_t* hist, int length, int num_contexts, std::uint32_t se,
                       std::uint32_t msb, std::uint32_t lsb, std::uint8_t* depth, std::uint16_t* bits) {
    auto scratch{std::make_unique<HuffScratch>()};
    w.write(1, 0);
    if (num_contexts > 1) {
        w.write(1, 1);
        w.write(2, 0);
    }
    w.write(1, 1);
    write_uint_config(w, se, msb, lsb);
    write_var_len_u16(w, static_cast<std::uint32_t>(length - 1));
    std::fill(depth, depth + length, 0);
    std::fill(bits, bits + length, 0);
    if (length > 1) {
        build_and_store_huffman(hist, length, depth, bits, w, *scratch);
    }
}

// context_map.cc:43-168: the smallest of complex, complex+MTF and simple.
void complex_cmap(HostBits& w, const std::uint8_t* map, int n, bool mtf) {
    std::vector<std::uint8_t> sym(map, map + n);
    if (mtf) {
        std::uint8_t s[256];
        for (int i{0}; i < 256; ++i) {
            s[i] = static_cast<std::uint8_t>(i);
        }
        for (int i{0}; i < n; ++i) {
            int r{0};
            while (s[r] != map[i]) {
                ++r;
            }
            sym[i] = static_cast<std::uint8_t>(r);
            const std::uint8_t v{s[r]};
            for (; r > 0; --r) {
                s[r] = s[r - 1];
            }
            s[0] = v;
        }
    }
    std::uint32_t hist[16]{};
    for (std::uint8_t v : sym) {
        std::uint32_t t, nb, b;
        hybrid_uint(2, 0, 1, v, t, nb, b);
        ++hist[t];
    }
    int alpha{1};
    for (int i{0}; i < 16; ++i) {
        if (hist[i]) {
            alpha = i + 1;
        }
    }
    w.write(1, 0);
    w.write(1, mtf ? 1 : 0);
    std::uint8_t depth[16];
    std::uint16_t bits[16];
    prefix_histograms(w, hist, alpha, 1, 2, 0, 1, depth, bits);
    for (std::uint8_t v : sym) {
        std::uint32_t t, nb, b;
        hybrid_uint(2, 0, 1, v, t, nb, b);
        w.write(depth[t], bits[t]);
        w.write(nb, b);
    }
}

HostBits best_context_map(const std::uint8_t* map, int n, int nclusters) {
    HostBits cx, cm, sp;
    complex_cmap(cx, map, n, false);
    complex_cmap(cm, map, n, true);
    const HostBits* sel{&cx};
    if (cm.pos < sel->pos) {
        sel = &cm;
    }
    if (nclusters <= 8) {
        const std::uint32_t bpe{ceil_log2(static_cast<std::uint32_t>(nclusters))};
        sp.write(1, 1);
        sp.write(2, bpe);
        for (int i{0}; i < n; ++i) {
            sp.write(bpe, map[i]);
        }
        if (sp.pos <= sel->pos) {
            sel = &sp;
        }
    }
    return *sel;
}

// ac_context.h:108-131 on the host (the fixed 32-cluster context map).
int cluster_of(std::uint32_t ctx) {
    constexpr std::uint32_t count_contexts{15u * 37u};
    if (ctx < count_contexts) {
        const std::uint32_t bucket{ctx / 15u};
        const int group{static_cast<int>(ctx % 15u) < 7 ? 0 : 1};
        return group * 4 + (bucket < 4 ? 0 : (bucket < 12 ? 1 : (bucket < 24 ? 2 : 3)));
    }
    const std::uint32_t rel{ctx - count_contexts};
    const int group{static_cast<int>(rel / 458u) < 7 ? 0 : 1};
    const std::uint32_t z{rel % 458u};
    static const std::uint32_t edges[11]{32, 64, 96, 128, 160, 200, 240, 280, 328, 376, 424};
    int band{11};
    for (int i{0}; i < 11; ++i) {
        if (z < edges[i]) {
            band = i;
            break;
        }
    }
    return 8 + group * 12 + band;
}

const HostBits& ac_context_map_bits() {
    static const HostBits bits{[] {
        std::vector<std::uint8_t> map(kNumAcContexts);
        for (int i{0}; i < kNumAcContexts; ++i) {
            map[i] = static_cast<std::uint8_t>(cluster_of(static_cast<std::uint32_t>(i)));
        }
        return best_context_map(map.data(), kNumAcContexts, kNumClusters);
    }()};
    return bits;
}

// frame_assembly.cc:70-101 up to (not including) the data alphabet size:
// GroupHeader, single-leaf tree with `predictor`, the data histogram's fixed
// leading fields.
void modular_prefix(HostBits& w, int predictor) {
    w.write(1, 0);
    w.write(1, 1);
    w.write(2, 0);
    const std::uint32_t tokens[5]{0, static_cast<std::uint32_t>(predictor), 0, 0, 0};
    std::uint32_t th[16]{};
    int tl{1};
    for (std::uint32_t t : tokens) {
        ++th[t];
        tl = std::max(tl, static_cast<int>(t) + 1);
    }
    std::uint8_t td[16];
    std::uint16_t tb[16];
    prefix_histograms(w, th, tl, 6, 4, 2, 0, td, tb);
    for (std::uint32_t t : tokens) {
        w.write(td[t], tb[t]);
    }
    w.write(1, 0);  // data container: no LZ77
    w.write(1, 1);  // prefix codes
    write_uint_config(w, 4, 2, 0);
}

std::once_flag g_tables_once[64];
bool g_tables_ok[64];

// Test hook: the runtime object (stream, event, page-locked or device memory)
// whose creation brings the countdown from 1 to 0 is refused as if there were
// none left (0: no failure pending).
std::atomic<int> g_fail_alloc_countdown{0};

bool injected_alloc_failure() {
    int n{g_fail_alloc_countdown.load()};
    while (n > 0) {
        if (g_fail_alloc_countdown.compare_exchange_weak(n, n - 1)) {
            return n == 1;
        }
    }
    return false;
}

// Everything an encoder creates comes from the four calls below, so that the
// hook can refuse each of them.
bool create_stream(hipStream_t* s) {
    return !injected_alloc_failure() && hipStreamCreateWithFlags(s, hipStreamNonBlocking) == hipSuccess;
}

bool create_event(hipEvent_t* e, unsigned int flags = hipEventDefault) {
    return !injected_alloc_failure() && hipEventCreateWithFlags(e, flags) == hipSuccess;
}

bool alloc_host(void** p, std::size_t bytes, unsigned int flags) {
    return !injected_alloc_failure() && hipHostMalloc(p, bytes, flags) == hipSuccess;
}

bool alloc_device(void** p, std::size_t bytes) {
    return !injected_alloc_failure() && hipMalloc(p, bytes) == hipSuccess;
}

// The stream of a destroyed encoder, one per device, for the next one:
// creating a stream takes the runtime up to 0.8 ms, most of the creation of a
// small encoder (640x360 one-shot encodes 950 -> 325 us).  Only one, because a
// stream keeps its hardware queue (of four): two kept streams may share one,
// and two frames in flight then run one after the other (2560x1440 352 -> 375
// us with four kept), while new streams take the least used queues.
class StreamPool {
public:
    hipStream_t take(int device) {
        hipStream_t s{nullptr};
        if (device < kDevices) {
            const std::lock_guard<std::mutex> lock{mutex_};
            std::swap(s, idle_[device]);
        }
        return s != nullptr || create_stream(&s) ? s : nullptr;
    }

    // `s` has nothing queued.
    void give(int device, hipStream_t s) {
        if (device >= 0 && device < kDevices) {
            const std::lock_guard<std::mutex> lock{mutex_};
            if (idle_[device] == nullptr) {
                std::swap(s, idle_[device]);
                return;
            }
        }
        (void)hipStreamDestroy(s);
    }

private:
    static constexpr int kDevices{64};
    std::mutex mutex_;
    hipStream_t idle_[kDevices]{};
};

// Never destroyed: encoders may be destroyed after this file's statics.
StreamPool& stream_pool() {
    static StreamPool* const pool{new StreamPool};
    return *pool;
}

}  // namespace

bool ensure_device_tables(int device) {
    std::call_once(g_tables_once[device & 63], [device] { g_tables_ok[device & 63] = init_device_tables(); });
    return g_tables_ok[device & 63];
}

void fail_allocation_after(int n) {
    g_fail_alloc_countdown.store(n < 0 ? 0 : n);
}

bool device_exists(int ordinal) {
    int count{0};
    if (hipGetDeviceCount(&count) != hipSuccess) {
        return false;
    }
    return ordinal >= 0 && ordinal < count;
}

bool device_has_matrix_cores(int ordinal) {
    hipDeviceProp_t p{};
    if (hipGetDeviceProperties(&p, ordinal) != hipSuccess) {
        return false;
    }
    const std::string arch{p.gcnArchName};
    return arch.rfind("gfx90a", 0) == 0 || arch.rfind("gfx94", 0) == 0 || arch.rfind("gfx95", 0) == 0;
}

std::size_t Encoder::max_output_size(std::uint32_t width, std::uint32_t height) {
    const std::size_t bw{width / 8u}, bh{height / 8u};
    const std::size_t nac{((bw + 31) / 32) * ((bh + 31) / 32)};
    const std::size_t ndc{((bw + 255) / 256) * ((bh + 255) / 256)};
    return 3 * bw * bh * 384 + 48 * bw * bh + (nac + ndc) * 2048 + 16384;
}

Encoder::~Encoder() {
    release();
}

void Encoder::release() {
    if (device_ >= 0) {
        (void)hipSetDevice(device_);
    }
    // A frame queued by encode_async and never finished may still run.
    const bool idle{stream_ != nullptr && hipStreamSynchronize(stream_) == hipSuccess};
    pending_ = false;
    for (void* p : allocations_) {
        (void)hipFree(p);
    }
    allocations_.clear();
    input_ = nullptr;
    copy_team_.reset();
    team_shared_ = false;
    if (total_host_ != nullptr) {
        (void)hipHostFree(total_host_);
        total_host_ = nullptr;
    }
    if (stage_host_ != nullptr) {
        (void)hipHostFree(stage_host_);
        stage_host_ = nullptr;
        stage_dev_ = nullptr;
    }
    for (hipEvent_t& e : stage_ready_) {
        if (e != nullptr) {
            (void)hipEventDestroy(e);
            e = nullptr;
        }
    }
    for (hipEvent_t& e : events_) {
        if (e != nullptr) {
            (void)hipEventDestroy(e);
            e = nullptr;
        }
    }
    for (hipEvent_t* e : {&ev_size_, &ev_end_, &ev_done_, &ev_caller_, &ev_input_free_}) {
        if (*e != nullptr) {
            (void)hipEventDestroy(*e);
            *e = nullptr;
        }
    }
    if (stream_ != nullptr) {
        if (idle) {
            stream_pool().give(device_, stream_);
        } else {
            (void)hipStreamDestroy(stream_);
        }
        stream_ = nullptr;
    }
    null_buffers();
    total_dev_ = nullptr;
    configured_ = false;
    workspace_ = false;
}

// Every device buffer member back to null (their memory was freed with
// allocations_), so nothing can reach freed memory after a failed configure.
void Encoder::null_buffers() {
    coeffs_ = nullptr;
    acs_ = nullptr;
    qf_ = nullptr;
    cfl_part_ = nullptr;
    ytox_ = ytob_ = nullptr;
    ac_ = nullptr;
    dc_ = nullptr;
    nz_grid_ = nullptr;
    nz_count_ = nullptr;
    hists_ = fb_count_ = nullptr;
    codes_ = constants_ = layout_ = nullptr;
    tokens_ = nullptr;
    item_tokens_ = nullptr;
    item_list_ = item_count_ = hist_partial_ = ac_staging_ = dc_staging_ = nullptr;
    ac_run_bits_ = nullptr;
    ac_group_bits_ = dc_group_bits_ = ac_base_ = dc_base_ = nullptr;
    ac_group_bytes_ = dc_group_bytes_ = chunk_bits_ = nullptr;
    out_ = nullptr;
    out_cap_ = 0;
    features_ = nullptr;
    export_ = false;
    const_gs_ = const_qdc_ = 0;
}

bool Encoder::configure(std::uint32_t width, std::uint32_t height, float distance, int device) {
    if (width == 0 || height == 0 || width % 8 || height % 8) {
        return false;
    }
    const Geometry geo{Geometry::of(width, height)};
    if (geo.num_dc > 32) {
        return false;  // per-group tables are sized for up to 32 DC groups
    }
    const bool same_shape{configured_ && device == device_ && width == geo_.width && height == geo_.height};
    if (pending_) {
        return false;  // a frame queued by encode_async is still owed to finish()
    }
    distance_ = distance;
    prm_ = make_frame_params(distance);
    prm_.mode = mode_;
    if (same_shape) {
        return true;
    }
    release();
    device_ = device;
    geo_ = geo;
    if (!setup(device)) {
        // Leave nothing half-built: no buffers, no shape a later configure
        // could mistake for its own, and every encode refused until a
        // configure succeeds.
        release();
        device_ = -1;
        geo_ = Geometry{};
        return false;
    }
    configured_ = true;
    return true;
}

bool Encoder::setup(int device) {
    if (hipSetDevice(device) != hipSuccess) {
        return false;
    }
    std::call_once(g_tables_once[device & 63], [device] { g_tables_ok[device & 63] = init_device_tables(); });
    if (!g_tables_ok[device & 63]) {
        return false;
    }
    stream_ = stream_pool().take(device);
    if (stream_ == nullptr) {
        return false;
    }
    for (hipEvent_t* e : {&ev_done_, &ev_caller_, &ev_input_free_}) {
        if (!create_event(e, hipEventDisableTiming)) {
            return false;
        }
    }
    // Bound to kernels' completion at launch (timing-capable events).
    for (hipEvent_t* e : {&ev_size_, &ev_end_}) {
        if (!create_event(e)) {
            return false;
        }
    }
    for (hipEvent_t& e : events_) {
        if (!create_event(&e)) {
            return false;
        }
    }
    if (!alloc_host(reinterpret_cast<void**>(&total_host_), sizeof(std::uint64_t), hipHostMallocDefault) ||
        hipHostGetDevicePointer(reinterpret_cast<void**>(&total_dev_), total_host_, 0) != hipSuccess ||
        !alloc_host(reinterpret_cast<void**>(&stage_host_), 2 * kStageChunk, hipHostMallocMapped) ||
        hipHostGetDevicePointer(reinterpret_cast<void**>(&stage_dev_), stage_host_, 0) != hipSuccess) {
        return false;
    }
    // Also bound to the upload's copies (timing-capable events).
    for (hipEvent_t& e : stage_ready_) {
        if (!create_event(&e)) {
            return false;
        }
    }
    return alloc();
}

template <class Get>
void Encoder::carve(Get& get) {
    const std::size_t nblk{geo_.nblocks};
    const std::size_t tiles{static_cast<std::size_t>(geo_.cmw) * geo_.cmh};
    const std::size_t regions{static_cast<std::size_t>(geo_.rw) * geo_.rh};
    const std::size_t nh{static_cast<std::size_t>(kNumClusters) + 2 * geo_.num_dc};
    const std::size_t dc_chunks{static_cast<std::size_t>(geo_.num_dc) * dc_chunks_per_group(geo_)};
    get(coeffs_, 3 * nblk * 64 * sizeof(std::uint16_t));
    get(acs_, nblk);
    get(qf_, nblk * sizeof(std::int32_t));
    get(cfl_part_, regions * 3 * sizeof(float));
    get(ytox_, tiles);
    get(ytob_, tiles);
    get(ac_, 3 * nblk * 64 * sizeof(std::int16_t));
    get(dc_, 3 * nblk * sizeof(std::int32_t));
    get(nz_grid_, 3 * nblk);
    get(nz_count_, 3 * nblk * sizeof(std::uint16_t));
    get(hists_, nh * kHistStride * sizeof(std::uint32_t));
    get(fb_count_, 64 * sizeof(std::uint32_t));
    get(codes_, sizeof_codeset());
    get(constants_, sizeof_constants());
    get(tokens_, 3 * nblk * 64 * sizeof(std::uint32_t));
    get(item_tokens_, 3 * nblk * sizeof(std::uint16_t));
    get(item_list_, 3 * nblk * sizeof(std::uint32_t));
    get(item_count_, 2 * sizeof(std::uint32_t));
    get(hist_partial_, ac_partial_words() * sizeof(std::uint32_t));
    get(ac_staging_, static_cast<std::size_t>(geo_.num_ac) * ac_group_slot_words() * sizeof(std::uint32_t));
    get(dc_staging_, dc_chunks * dc_chunk_slot_words() * sizeof(std::uint32_t));
    get(ac_run_bits_, geo_.num_ac * ac_group_runs() * sizeof(std::uint16_t));
    get(ac_group_bytes_, geo_.num_ac * sizeof(std::uint32_t));
    get(ac_group_bits_, geo_.num_ac * sizeof(std::uint64_t));
    get(chunk_bits_, dc_chunks * sizeof(std::uint32_t));
    get(dc_group_bytes_, geo_.num_dc * sizeof(std::uint32_t));
    get(dc_group_bits_, geo_.num_dc * sizeof(std::uint64_t));
    get(layout_, sizeof_layout());
    get(ac_base_, geo_.num_ac * sizeof(std::uint64_t));
    get(dc_base_, geo_.num_dc * sizeof(std::uint64_t));
}

// Consecutive 256-byte aligned ranges from offset 0 of a workspace (`base`
// null: sizing only).
namespace {
struct Bump {
    std::uint8_t* base;
    std::size_t used{0};
    template <class T>
    void operator()(T*& p, std::size_t bytes) {
        p = base != nullptr ? reinterpret_cast<T*>(base + used) : nullptr;
        used += (std::max<std::size_t>(bytes, 1) + 255) & ~static_cast<std::size_t>(255);
    }
};
}  // namespace

// One allocation holds every buffer: a program that creates an encoder for a
// single frame pays for each allocation, mapped on creation and unmapped on
// destruction (one-shot encode of a host frame with 31 allocations and with
// one: 1920x1080 3,790 and 1,270 us, 3840x2160 5,170 and 2,540).
bool Encoder::alloc() {
    out_cap_ = (max_output_size(geo_.width, geo_.height) + 64 + 3) & ~static_cast<std::size_t>(3);
    const_gs_ = const_qdc_ = 0;
    Bump size{nullptr};
    carve(size);
    size(out_, out_cap_);
    void* arena{nullptr};
    if (!alloc_device(&arena, size.used)) {
        return false;
    }
    allocations_.push_back(arena);
    Bump place{static_cast<std::uint8_t*>(arena)};
    carve(place);
    place(out_, out_cap_);
    return true;
}

std::size_t Encoder::workspace_bytes(std::uint32_t width, std::uint32_t height) {
    Encoder probe;
    probe.geo_ = Geometry::of(width, height);
    Bump b{nullptr};
    probe.carve(b);
    probe.null_buffers();
    return b.used;
}

bool Encoder::bind_workspace(std::uint32_t width, std::uint32_t height, float distance, int device, void* base,
                             std::size_t bytes) {
    if (!allocations_.empty() || stream_ != nullptr || base == nullptr || width == 0 || height == 0 ||
        width % 8 || height % 8) {
        return false;  // an encoder that owns allocations is never rebound
    }
    const Geometry geo{Geometry::of(width, height)};
    if (geo.num_dc > 32 || workspace_bytes(width, height) > bytes) {
        return false;
    }
    if (hipSetDevice(device) != hipSuccess) {
        return false;
    }
    std::call_once(g_tables_once[device & 63], [device] { g_tables_ok[device & 63] = init_device_tables(); });
    if (!g_tables_ok[device & 63]) {
        return false;
    }
    const bool same{workspace_ && configured_ && device == device_ && geo.width == geo_.width &&
                    geo.height == geo_.height &&
                    static_cast<void*>(coeffs_) == base};
    device_ = device;
    distance_ = distance;
    prm_ = make_frame_params(distance);
    prm_.mode = mode_;
    if (!same) {
        geo_ = geo;
        Bump b{static_cast<std::uint8_t*>(base)};
        carve(b);
        out_ = nullptr;
        out_cap_ = 0;
        const_gs_ = const_qdc_ = 0;  // the constants depend on the shape
    }
    workspace_ = true;
    configured_ = true;
    return true;
}

bool Encoder::fill_job(FrameJob& j, hipStream_t s, std::uint8_t* out_dev, std::size_t cap, std::uint64_t* size_dev) {
    if (!workspace_ || !configured_ || hipSetDevice(device_) != hipSuccess ||
        !build_constants(prm_.global_scale, prm_.quant_dc, s)) {
        return false;
    }
    j.geo = geo_;
    j.prm = prm_;
    j.coeffs = coeffs_;
    j.acs = acs_;
    j.qf = qf_;
    j.cfl_part = cfl_part_;
    j.ytox = ytox_;
    j.ytob = ytob_;
    j.ac = ac_;
    j.dc = dc_;
    j.nz_grid = nz_grid_;
    j.nz_count = nz_count_;
    j.hists = hists_;
    j.fb_count = fb_count_;
    j.codes = static_cast<CodeSet*>(codes_);
    j.k = static_cast<const Constants*>(constants_);
    j.tokens = tokens_;
    j.item_tokens = item_tokens_;
    j.item_list = item_list_;
    j.item_count = item_count_;
    j.hist_partial = hist_partial_;
    j.ac_staging = ac_staging_;
    j.dc_staging = dc_staging_;
    j.ac_run_bits = ac_run_bits_;
    j.ac_group_bytes = ac_group_bytes_;
    j.ac_group_bits = ac_group_bits_;
    j.chunk_bits = chunk_bits_;
    j.dc_group_bytes = dc_group_bytes_;
    j.dc_group_bits = dc_group_bits_;
    j.lay = static_cast<Layout*>(layout_);
    j.ac_base = ac_base_;
    j.dc_base = dc_base_;
    j.out = reinterpret_cast<std::uint32_t*>(out_dev);
    j.cap = cap;
    j.size_out = size_dev;
    j.clr = entropy_clears();
    j.dc_chunks = dc_chunks_per_group(geo_);
    return true;
}

#ifdef CJX_REGION_CUT
bool Encoder::region_only(const std::uint8_t* luma, std::size_t luma_pitch, const std::uint8_t* chroma,
                          std::size_t chroma_pitch) {
    if (!configured_ || workspace_ || pending_ || hipSetDevice(device_) != hipSuccess) {
        return false;
    }
    launch_region(stream_, geo_, prm_, luma, luma_pitch, chroma, chroma_pitch, coeffs_, acs_, qf_, cfl_part_,
                  item_count_, entropy_clears());
    return hipStreamSynchronize(stream_) == hipSuccess;
}
#endif

// One frame queued on `s`; nothing waits on the host unless the constant bit
// strings change (a new shape or distance), which copies them in order on
// `s` and waits for that copy.
bool Encoder::encode_on(hipStream_t s, const std::uint8_t* luma, std::size_t luma_pitch, const std::uint8_t* chroma,
                        std::size_t chroma_pitch, std::uint8_t* out_dev, std::size_t cap, std::uint64_t* size_dev) {
    if (!workspace_ || !configured_ || hipSetDevice(device_) != hipSuccess ||
        !build_constants(prm_.global_scale, prm_.quant_dc, s)) {
        return false;
    }
    auto* codes{static_cast<CodeSet*>(codes_)};
    auto* k{static_cast<const Constants*>(constants_)};
    auto* lay{static_cast<Layout*>(layout_)};
    launch_region(s, geo_, prm_, luma, luma_pitch, chroma, chroma_pitch, coeffs_, acs_, qf_, cfl_part_, item_count_,
                  entropy_clears());
    launch_tile_quantize(s, geo_, prm_, coeffs_, acs_, qf_, cfl_part_, ac_, nz_grid_, nz_count_,
                         ItemList{item_list_, item_count_}, dc_, ytox_, ytob_);
    launch_ac_tokens(s, geo_, ac_, acs_, nz_grid_, nz_count_, tokens_, item_tokens_, hist_partial_, hists_,
                     ItemList{item_list_, item_count_}, dc_, qf_, ytox_, ytob_, fb_count_);
    launch_huffman(s, kNumClusters + static_cast<int>(2 * geo_.num_dc), hists_, codes);
    launch_emit(s, geo_, acs_, item_tokens_, tokens_, codes, k, fb_count_, dc_, qf_, ytox_, ytob_, ac_staging_,
                ac_run_bits_, dc_staging_, chunk_bits_);
    launch_layout(s, geo_, k, codes, ac_run_bits_, chunk_bits_, dc_group_bytes_, dc_group_bits_, ac_group_bytes_,
                  ac_group_bits_, lay, ac_base_, dc_base_, size_dev);
    launch_assemble(s, geo_, k, lay, dc_staging_, ac_staging_, dc_group_bits_, ac_run_bits_, chunk_bits_,
                    dc_base_, ac_base_, out_dev, cap);
    return hipGetLastError() == hipSuccess;
}

// Constant bit strings of a configuration (codestream.cc, frame_assembly.cc).
bool Encoder::build_constants(std::uint32_t global_scale, std::uint32_t quant_dc, hipStream_t s) {
    if (global_scale == const_gs_ && quant_dc == const_qdc_) {
        return true;
    }
    HostBits head;
    head.write(8, 0xff);
    head.write(8, 0x0a);
    const bool small{geo_.width % 8 == 0 && geo_.height % 8 == 0 && geo_.width <= 256 && geo_.height <= 256};
    head.write(1, small);
    if (small) {
        head.write(5, geo_.height / 8 - 1);
    } else {
        write_u32(head, kDimEnc, geo_.height);
    }
    head.write(3, 0);
    if (small) {
        head.write(5, geo_.width / 8 - 1);
    } else {
        write_u32(head, kDimEnc, geo_.width);
    }
    head.write(1, 1);  // ImageMetadata all_default
    head.write(1, 1);  // CustomTransformData all_default
    head.pad();
    // FrameHeader (codestream.cc:67-85).
    const Distr ft[4]{{true, 0, 0}, {true, 1, 0}, {true, 2, 0}, {true, 3, 0}};
    const Distr ups[4]{{true, 1, 0}, {true, 2, 0}, {true, 4, 0}, {true, 8, 0}};
    const Distr passes[4]{{true, 1, 0}, {true, 2, 0}, {true, 3, 0}, {false, 4, 3}};
    const Distr blend[4]{{true, 0, 0}, {true, 1, 0}, {true, 2, 0}, {false, 3, 2}};
    const Distr name[4]{{true, 0, 0}, {false, 0, 4}, {false, 16, 5}, {false, 48, 10}};
    head.write(1, 0);
    write_u32(head, ft, 0);
    head.write(1, 0);
    head.write(2, 0);  // flags = 0 (U64)
    write_u32(head, ups, 1);
    head.write(3, 2);
    head.write(3, 2);
    write_u32(head, passes, 1);
    head.write(1, 0);
    write_u32(head, blend, 0);
    head.write(1, 1);
    write_u32(head, name, 0);
    head.write(1, 1);
    head.write(2, 0);  // extensions = 0 (U64)

    HostBits dcg;  // vardct_frame.cc:533-540
    dcg.write(1, 1);
    write_u32(dcg, kGlobalScaleEnc, global_scale);
    write_u32(dcg, kQuantDcEnc, quant_dc);
    dcg.write(1, 1);
    dcg.write(1, 1);
    dcg.write(1, 0);

    HostBits acp;  // frame_assembly.cc:131-146 + histogram_writer.cc:85-104
    acp.write(1, 1);
    acp.write(ceil_log2(geo_.num_ac), 0);
    write_u32(acp, kOrderEnc, 0);
    acp.write(1, 0);
    acp.append(ac_context_map_bits());
    acp.write(1, 1);
    for (int c{0}; c < kNumClusters; ++c) {
        write_uint_config(acp, 4, 2, 0);
    }

    HostBits pre;  // DecodeVarDCTDC extra_precision + modular prefix
    pre.write(2, 0);
    modular_prefix(pre, 5);
    HostBits mid;
    modular_prefix(mid, 0);

    if (!constants_fit(head.pos, acp.pos, pre.pos, mid.pos)) {
        return false;
    }
    std::vector<std::uint8_t> host(sizeof_constants());
    fill_constants(host.data(), head.words.data(), head.pos, dcg.words.data(), dcg.pos, acp.words.data(),
                   acp.pos, pre.words.data(), pre.pos, mid.words.data(), mid.pos);
    const hipStream_t on{s != nullptr ? s : stream_};
    if (hipMemcpyAsync(constants_, host.data(), host.size(), hipMemcpyHostToDevice, on) != hipSuccess ||
        hipStreamSynchronize(on) != hipSuccess) {
        return false;
    }
    const_gs_ = global_scale;
    const_qdc_ = quant_dc;
    return true;
}

void Encoder::mark(Stage s) {
    if (profiling_ == 1 || (profiling_ == 2 && (s == Stage::kRegion || s == Stage::kQuantize))) {
        (void)hipEventRecord(events_[static_cast<int>(s)], stream_);
    }
}

namespace {

// True for host memory the runtime can DMA into directly (allocated or
// registered through HIP); such an output skips the pinned staging copy.
bool host_pinned(const void* p) {
    hipPointerAttribute_t a{};
    if (p == nullptr || hipPointerGetAttributes(&a, p) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    return a.type == hipMemoryTypeHost;
}

}  // namespace

// The caller's output as a device address when it is page-locked host memory
// mapped for the device: the assembly kernel then writes the file there
// itself (over the host link, as a DMA would) and no copy follows it.
std::uint8_t* Encoder::mapped_output(std::uint8_t* dst) const {
    hipPointerAttribute_t a{};
    if (dst == nullptr || hipPointerGetAttributes(&a, dst) != hipSuccess) {
        (void)hipGetLastError();
        return nullptr;
    }
    if (a.type != hipMemoryTypeHost || a.devicePointer == nullptr || a.hostPointer == nullptr) {
        return nullptr;
    }
    // Base-relative: correct whether the runtime reports the allocation's
    // base or the queried address in both fields.  The kernel stores words,
    // so an unaligned output takes the copy path instead.
    std::uint8_t* const dev{static_cast<std::uint8_t*>(a.devicePointer) +
                            (dst - static_cast<std::uint8_t*>(a.hostPointer))};
    return reinterpret_cast<std::uintptr_t>(dev) % 4 == 0 ? dev : nullptr;
}

// The readback's first half.  The layout kernel writes the size into the
// pinned word.  A mapped page-locked output `direct` holds the file once the
// assembly has finished; for any other output (or none yet, for encode_async)
// the assembly also writes the file's first two chunks into the pinned
// staging buffer.
void Encoder::queue_readback(std::uint8_t* direct) {
    mark(Stage::kReadback);
    direct_dst_ = direct;
    pending_ = true;
}

// Queues the next n bytes of the device's file into a pinned slot.
bool Encoder::stage_chunk(int slot, std::size_t n) {
    const bool ok{hipMemcpyAsync(stage_host_ + slot * kStageChunk, reinterpret_cast<const std::uint8_t*>(out_) + staged_,
                                 n, hipMemcpyDeviceToHost, stream_) == hipSuccess &&
                  hipEventRecord(stage_ready_[slot], stream_) == hipSuccess};
    staged_ += n;
    return ok;
}

// Polls `e` until it has completed (false on an error).
bool Encoder::spin_on(hipEvent_t e) {
    for (;;) {
        const hipError_t r{hipEventQuery(e)};
        if (r == hipSuccess) {
            return true;
        }
        if (r != hipErrorNotReady) {
            return false;
        }
        __builtin_ia32_pause();
    }
}

// The end of a frame: the assembly kernel's own completion when it writes
// the output and ends the frame, else an event after the last copy.  The
// host polls it, and so would the runtime's own wait: hipEventSynchronize takes
// the thread's whole time on events of either kind (60 ms of 60, also with
// hipEventBlockingSync).
bool Encoder::wait_done() {
    if (end_bound_) {
        end_bound_ = false;
        return spin_on(ev_end_);
    }
    return hipEventRecord(ev_done_, stream_) == hipSuccess && spin_on(ev_done_);
}

// The readback's second half: waits for the frame, then moves the bytes into
// `dst` -- one DMA when `dst` is pinned, else from the staging chunks, which
// hold the file's start; the host copies a chunk out while the next one is in
// flight, then reuses its slot for the chunk after that.
bool Encoder::finish(std::uint8_t* dst, std::size_t cap, std::size_t* size) {
    if (!pending_) {
        return false;
    }
    pending_ = false;
    // Poll for the size, or for the frame's end when no size event was bound
    // (the assembly writes the file into `dst`): an event in mid-chain, to wait
    // for in two parts, costs about 5 us of idle device time after the kernel
    // that carries it.
    const bool ended{!size_bound_};
    if (!(ended ? wait_done() : spin_on(ev_size_))) {
        return false;
    }
    const std::uint64_t total{*total_host_};
    *size = static_cast<std::size_t>(total);
    bool ok{total <= out_cap_};
    bool queued{false};  // work on the stream behind the frame
    if (ok && total <= cap && dst != nullptr) {
        if (direct_dst_ != nullptr && dst == direct_dst_) {
            // The assembly kernel writes the file into `dst`; the frame's end
            // (waited for above without a size event, else below) completes it.
        } else if (host_pinned(dst)) {
            ok = hipMemcpyAsync(dst, out_, total, hipMemcpyDeviceToHost, stream_) == hipSuccess;
            queued = true;
        } else {
            if (!ended && !wait_done()) {
                return false;
            }
            staged_ = std::min<std::size_t>(2 * kStageChunk, total);
            std::size_t done{0};
            for (int slot{0}; ok && done < total; slot ^= 1) {
                const std::size_t n{std::min(kStageChunk, static_cast<std::size_t>(total) - done)};
                if (done >= 2 * kStageChunk && !spin_on(stage_ready_[slot])) {
                    return false;
                }
                std::memcpy(dst + done, stage_host_ + slot * kStageChunk, n);
                done += n;
                if (staged_ < total) {
                    ok = stage_chunk(slot, std::min<std::size_t>(kStageChunk, total - staged_));
                }
            }
        }
    }
    direct_dst_ = nullptr;
    if (!ended || queued) {
        mark(Stage::kCount);
        if (!wait_done()) {
            return false;
        }
    }
    if (profiling_ != 0) {
        for (int i{0}; i < static_cast<int>(Stage::kCount); ++i) {
            float ms{0.0f};
            if (profiling_ == 1 || i == static_cast<int>(Stage::kRegion)) {
                (void)hipEventElapsedTime(&ms, events_[i], events_[i + 1]);
            }
            stage_ms_[i] = ms;
        }
    }
    return ok;
}

bool Encoder::submit_nv12(const std::uint8_t* luma, std::size_t luma_pitch, const std::uint8_t* chroma,
                          std::size_t chroma_pitch, hipStream_t caller, bool release_caller, std::uint8_t* dst,
                          std::size_t cap) {
    if (!configured_ || workspace_ || pending_ || hipSetDevice(device_) != hipSuccess ||
        !build_constants(prm_.global_scale, prm_.quant_dc)) {
        return false;
    }
    // The frame starts after the work already queued on `caller` (the null
    // stream for the synchronous entry points: a caller that filled the
    // planes there, as callers of the reference did, is ordered before the
    // region kernel reads them).  A null stream with nothing left to run
    // needs no event: that saves a marker and a barrier packet ahead of the
    // region kernel on every frame of a synchronous loop.
    const bool settled{caller == nullptr && hipStreamQuery(nullptr) == hipSuccess};
    if (!settled &&
        (hipEventRecord(ev_caller_, caller) != hipSuccess || hipStreamWaitEvent(stream_, ev_caller_, 0) != hipSuccess)) {
        return false;
    }
    // With profiling on, the region kernel's own start and end times open the
    // region and quantize stages.
    const bool timed{profiling_ != 0};
    launch_region(stream_, geo_, prm_, luma, luma_pitch, chroma, chroma_pitch, coeffs_, acs_, qf_, cfl_part_,
                  item_count_, entropy_clears(),
                  timed ? events_[static_cast<int>(Stage::kRegion)] : nullptr,
                  timed ? events_[static_cast<int>(Stage::kQuantize)] : nullptr, export_ ? features_ : nullptr);
    // The planes are read by the region kernel only: later work on the
    // caller's stream may overwrite them once it has finished.
    if (release_caller && (hipEventRecord(ev_input_free_, stream_) != hipSuccess ||
                           hipStreamWaitEvent(caller, ev_input_free_, 0) != hipSuccess)) {
        return false;
    }
    // The quantizer lists the non-empty items for the tokenizer and leaves
    // the DC values and colour maps.
    launch_tile_quantize(stream_, geo_, prm_, coeffs_, acs_, qf_, cfl_part_, ac_, nz_grid_, nz_count_,
                         ItemList{item_list_, item_count_}, dc_, ytox_, ytob_);
    // A mapped page-locked output receives the file from the assembly kernel.
    std::uint8_t* const direct{mapped_output(dst)};
    if (!run_entropy(direct != nullptr ? direct : reinterpret_cast<std::uint8_t*>(out_),
                     direct != nullptr ? cap : out_cap_, true, profiling_ != 0)) {
        return false;
    }
    queue_readback(direct != nullptr ? dst : nullptr);
    return true;
}

bool Encoder::encode_nv12(const std::uint8_t* luma, std::size_t luma_pitch, const std::uint8_t* chroma,
                          std::size_t chroma_pitch, std::uint8_t* out, std::size_t cap, std::size_t* size) {
    if (!submit_nv12(luma, luma_pitch, chroma, chroma_pitch, nullptr, false, out, cap)) {
        pending_ = false;
        (void)hipStreamSynchronize(stream_);
        return false;
    }
    return finish(out, cap, size);
}

bool Encoder::encode_dct8_uniform(const std::uint8_t* luma, std::size_t luma_pitch, const std::uint8_t* chroma,
                                  std::size_t chroma_pitch, std::uint8_t* out, std::size_t cap, std::size_t* size) {
    if (!configured_ || pending_ || hipSetDevice(device_) != hipSuccess || !build_constants(prm_.global_scale, prm_.quant_dc)) {
        return false;
    }
    if (hipEventRecord(ev_caller_, nullptr) != hipSuccess || hipStreamWaitEvent(stream_, ev_caller_, 0) != hipSuccess) {
        return false;
    }
    mark(Stage::kRegion);
    launch_dct8_uniform(stream_, geo_, prm_, luma, luma_pitch, chroma, chroma_pitch, ac_, dc_, acs_, qf_, ytox_,
                        ytob_);
    mark(Stage::kQuantize);
    launch_nz(stream_, geo_, ac_, acs_, nz_grid_, nz_count_, entropy_clears());
    if (!run_entropy(reinterpret_cast<std::uint8_t*>(out_), out_cap_, false, profiling_ != 0)) {
        (void)hipStreamSynchronize(stream_);
        return false;
    }
    queue_readback(nullptr);
    return finish(out, cap, size);
}

bool Encoder::encode_async(const std::uint8_t* luma, std::size_t luma_pitch, const std::uint8_t* chroma,
                           std::size_t chroma_pitch, hipStream_t caller) {
    const bool ok{submit_nv12(luma, luma_pitch, chroma, chroma_pitch, caller, true, nullptr, 0)};
    if (!ok && pending_) {
        pending_ = false;
        (void)hipStreamSynchronize(stream_);
    }
    return ok;
}

// Host planes -> the encoder's device NV12 frame (width pitch), queued on the
// stream.  Pinned planes are copied by one 2D DMA each (the caller's frame has
// ended before encode_host returns), others go as row blocks through the two
// pinned staging chunks: the host copy of one chunk overlaps the transfer
// of the other, and from kTeamBytes up the copy is shared with a few helper threads
// (1920x1080: 216 us of copying by one thread, 36 by four; with the readback
// below a frame from and to ordinary memory 390 -> 249 us).
bool Encoder::upload_nv12(const std::uint8_t* luma, std::size_t luma_pitch, const std::uint8_t* chroma,
                          std::size_t chroma_pitch) {
    if (!configured_ || pending_ || hipSetDevice(device_) != hipSuccess) {
        return false;
    }
    const std::size_t w{geo_.width}, h{geo_.height};
    if (input_ == nullptr) {
        void* p{nullptr};
        if (!alloc_device(&p, w * h * 3 / 2)) {
            return false;
        }
        allocations_.push_back(p);
        input_ = static_cast<std::uint8_t*>(p);
    }
    struct Plane {
        const std::uint8_t* src;
        std::size_t pitch, rows;
        std::uint8_t* dst;
    };
    const Plane planes[2]{{luma, luma_pitch, h, input_}, {chroma, chroma_pitch, h / 2, input_ + w * h}};
    if (host_pinned(luma) && host_pinned(chroma)) {
        for (const Plane& pl : planes) {
            if (hipMemcpy2DAsync(pl.dst, w, pl.src, pl.pitch, w, pl.rows, hipMemcpyHostToDevice, stream_) !=
                hipSuccess) {
                (void)hipStreamSynchronize(stream_);
                return false;
            }
        }
        return true;
    }
    const std::size_t chunk_rows{kStageChunk / w};
    if (chunk_rows == 0) {
        return false;
    }
    const std::size_t luma_chunks{(h + chunk_rows - 1) / chunk_rows};
    const std::size_t chunks{luma_chunks + (h / 2 + chunk_rows - 1) / chunk_rows};
    if (chunks > CopyTeam::kGroups) {
        return false;
    }
    const bool shared{w * h * 3 / 2 >= kTeamBytes};
    if (copy_team_ == nullptr || (shared && !team_shared_)) {
        copy_team_.reset(new (std::nothrow) CopyTeam{shared ? kTeamHelpers : 0u});
        team_shared_ = shared;
        if (copy_team_ == nullptr) {
            return false;
        }
    }
    CopyTeam& team{*copy_team_};
    // Chunk c: rows [row, row + rows) of its plane, to slot c % 2, in
    // kChunkPieces runs of rows.
    constexpr std::size_t kChunkPieces{8};
    struct Chunk {
        const Plane* plane;
        std::size_t row, rows;
    };
    const auto chunk_at = [&](std::size_t c) {
        const Plane& pl{planes[c < luma_chunks ? 0 : 1]};
        const std::size_t row{(c < luma_chunks ? c : c - luma_chunks) * chunk_rows};
        return Chunk{&pl, row, std::min(chunk_rows, pl.rows - row)};
    };
    const auto copy_piece = [&](std::uint32_t i) {
        const Chunk k{chunk_at(i / kChunkPieces)};
        const std::size_t piece{i % kChunkPieces};
        const std::size_t r0{k.rows * piece / kChunkPieces}, r1{k.rows * (piece + 1) / kChunkPieces};
        std::uint8_t* const st{stage_host_ + (i / kChunkPieces % 2) * kStageChunk};
        const std::uint8_t* const src{k.plane->src + k.row * k.plane->pitch};
        if (k.plane->pitch == w) {
            std::memcpy(st + r0 * w, src + r0 * w, (r1 - r0) * w);
        } else {
            for (std::size_t r{r0}; r < r1; ++r) {
                std::memcpy(st + r * w, src + r * k.plane->pitch, w);
            }
        }
    };
    team.open(static_cast<std::uint32_t>(chunks * kChunkPieces), kChunkPieces,
              [&copy_piece](std::uint32_t i) { copy_piece(i); }, shared);
    bool ok{true};
    for (std::size_t c{0}; ok && c < chunks; ++c) {
        const std::size_t slot{c % 2};
        if (c == 0) {
            team.release(static_cast<std::uint32_t>(std::min<std::size_t>(2, chunks) * kChunkPieces));
        } else if (c >= 2) {
            if (!spin_on(stage_ready_[slot])) {
                ok = false;
                break;
            }
            team.release(static_cast<std::uint32_t>((c + 1) * kChunkPieces));
        }
        team.finish_group(static_cast<std::uint32_t>(c));
        const Chunk k{chunk_at(c)};
        launch_copy_in(stream_, k.plane->dst + k.row * w, stage_dev_ + slot * kStageChunk, k.rows * w,
                       stage_ready_[slot]);
    }
    team.close();
    return ok && hipGetLastError() == hipSuccess;
}

bool Encoder::encode_host(const std::uint8_t* luma, std::size_t luma_pitch, const std::uint8_t* chroma,
                          std::size_t chroma_pitch, std::uint8_t* out, std::size_t cap, std::size_t* size) {
    return upload_nv12(luma, luma_pitch, chroma, chroma_pitch) &&
           encode_nv12(input_, geo_.width, input_ + static_cast<std::size_t>(geo_.width) * geo_.height, geo_.width,
                       out, cap, size);
}

bool Encoder::encode_coefficients(const std::int16_t* ac, const std::int32_t* dc, const std::int8_t* acs,
                                  const std::int32_t* qf, const std::int8_t* ytox, const std::int8_t* ytob,
                                  std::uint32_t global_scale, std::uint32_t quant_dc, std::uint8_t* out,
                                  std::size_t cap, std::size_t* size) {
    if (!configured_ || pending_ || hipSetDevice(device_) != hipSuccess || !build_constants(global_scale, quant_dc)) {
        return false;
    }
    const std::size_t nblk{geo_.nblocks};
    const std::size_t tiles{static_cast<std::size_t>(geo_.cmw) * geo_.cmh};
    std::vector<std::int8_t> zeros(tiles, 0);
    const bool ok{
        hipMemcpyAsync(ac_, ac, 3 * nblk * 64 * sizeof(std::int16_t), hipMemcpyHostToDevice, stream_) == hipSuccess &&
        hipMemcpyAsync(dc_, dc, 3 * nblk * sizeof(std::int32_t), hipMemcpyHostToDevice, stream_) == hipSuccess &&
        hipMemcpyAsync(acs_, acs, nblk, hipMemcpyHostToDevice, stream_) == hipSuccess &&
        hipMemcpyAsync(qf_, qf, nblk * sizeof(std::int32_t), hipMemcpyHostToDevice, stream_) == hipSuccess &&
        hipMemcpyAsync(ytox_, ytox != nullptr ? ytox : zeros.data(), tiles, hipMemcpyHostToDevice, stream_) ==
            hipSuccess &&
        hipMemcpyAsync(ytob_, ytob != nullptr ? ytob : zeros.data(), tiles, hipMemcpyHostToDevice, stream_) ==
            hipSuccess &&
        hipStreamSynchronize(stream_) == hipSuccess};
    if (!ok) {
        return false;
    }
    mark(Stage::kRegion);
    mark(Stage::kQuantize);
    launch_nz(stream_, geo_, ac_, acs_, nz_grid_, nz_count_, entropy_clears());
    if (!run_entropy(reinterpret_cast<std::uint8_t*>(out_), out_cap_, false, profiling_ != 0)) {
        (void)hipStreamSynchronize(stream_);
        return false;
    }
    queue_readback(nullptr);
    return finish(out, cap, size);
}

// The histograms (AC clusters, then DC and AcMetadata per DC group) and the
// first-block counts start every frame at zero.
Clears Encoder::entropy_clears() const {
    Clears c{};
    c.ptr[0] = hists_;
    c.words[0] = static_cast<std::uint32_t>((kNumClusters + 2 * geo_.num_dc) * kHistStride);
    c.ptr[1] = fb_count_;
    c.words[1] = 64;
    return c;
}

// The entropy stage on the encoder's one stream: six launches, the DC
// groups' work beside the AC groups' in each (histograms beside the partial
// histograms' sum, codes beside codes, chunks beside parts).  A DC chain of
// its own on a second stream was six launches and two cross-stream
// dependencies (about 5 us each), and ran after the AC chain's start of its
// stage, not beside it, wherever the two streams shared a hardware queue
// (four per process: two encoders fill them).  Whole frames, before -> after,
// with three encoders alive and the DC values in the quantizer included:
// 320x240 159 -> 123 us, 7680x4320 1,145 -> 1,125 us, 3840x2160 unchanged at
// 364 us, a batch of 16 mixed frames 1,527 -> 1,486 us.  `size_event` binds
// ev_size_ to the layout kernel (the host then reads the size before the
// frame's end).
bool Encoder::run_entropy(std::uint8_t* out, std::size_t cap, bool listed, bool size_event) {
    auto* codes{static_cast<CodeSet*>(codes_)};
    auto* k{static_cast<const Constants*>(constants_)};
    auto* lay{static_cast<Layout*>(layout_)};
    mark(Stage::kHistograms);
    launch_ac_tokens(stream_, geo_, ac_, acs_, nz_grid_, nz_count_, tokens_, item_tokens_, hist_partial_, hists_,
                     listed ? ItemList{item_list_, item_count_} : ItemList{nullptr, nullptr}, dc_, qf_, ytox_, ytob_,
                     fb_count_);
    mark(Stage::kCodes);
    launch_huffman(stream_, kNumClusters + static_cast<int>(2 * geo_.num_dc), hists_, codes);
    mark(Stage::kSizes);
    launch_emit(stream_, geo_, acs_, item_tokens_, tokens_, codes, k, fb_count_, dc_, qf_, ytox_, ytob_, ac_staging_,
                ac_run_bits_, dc_staging_, chunk_bits_);
    size_bound_ = size_event;
    // Without a size event the output is written by the assembly kernel and
    // nothing follows it: its own completion ends the frame.
    end_bound_ = !size_event;
    launch_layout(stream_, geo_, k, codes, ac_run_bits_, chunk_bits_, dc_group_bytes_, dc_group_bits_,
                  ac_group_bytes_, ac_group_bits_, lay, ac_base_, dc_base_, total_dev_,
                  size_event ? ev_size_ : nullptr);
    mark(Stage::kEmit);
    // A file that stays on the device is read by the host from the staging
    // chunks first.
    const FileHead head{out == reinterpret_cast<std::uint8_t*>(out_)
                            ? FileHead{reinterpret_cast<std::uint32_t*>(stage_dev_), 2 * kStageChunk / 4}
                            : FileHead{nullptr, 0}};
    launch_assemble(stream_, geo_, k, lay, dc_staging_, ac_staging_, dc_group_bits_, ac_run_bits_, chunk_bits_,
                    dc_base_, ac_base_, out, cap, head, end_bound_ ? ev_end_ : nullptr);
    return hipGetLastError() == hipSuccess;
}

bool Encoder::export_features(bool on) {
    if (!configured_ || workspace_ || hipSetDevice(device_) != hipSuccess) {
        return false;
    }
    if (on && features_ == nullptr) {
        void* p{nullptr};
        if (!alloc_device(&p, static_cast<std::size_t>(geo_.rw) * geo_.rh * 108 * sizeof(float))) {
            return false;
        }
        allocations_.push_back(p);
        features_ = static_cast<float*>(p);
    }
    export_ = on;
    return true;
}

std::size_t Encoder::buffer_bytes(Buffer which) const {
    const std::size_t nblk{geo_.nblocks};
    const std::size_t tiles{static_cast<std::size_t>(geo_.cmw) * geo_.cmh};
    switch (which) {
        case Buffer::kCoeffs: return 3 * nblk * 64 * 2;
        case Buffer::kAcs: return nblk;
        case Buffer::kQuantField: return nblk * 4;
        case Buffer::kCflPartials: return static_cast<std::size_t>(geo_.rw) * geo_.rh * 12;
        case Buffer::kYtoX:
        case Buffer::kYtoB: return tiles;
        case Buffer::kAc: return 3 * nblk * 64 * 2;
        case Buffer::kDc: return 3 * nblk * 4;
        case Buffer::kNzGrid: return 3 * nblk;
        case Buffer::kNzCount: return 3 * nblk * 2;
        case Buffer::kHistograms: return (kNumClusters + 2 * geo_.num_dc) * kHistStride * 4;
        case Buffer::kAcGroupBytes: return geo_.num_ac * 4;
        case Buffer::kDcGroupBytes: return geo_.num_dc * 4;
        case Buffer::kCodeDepth: return (kNumClusters + 2 * geo_.num_dc) * kHistStride;
        case Buffer::kCodeBits: return (kNumClusters + 2 * geo_.num_dc) * kHistStride * 2;
        case Buffer::kFeatures: return features_ != nullptr ? static_cast<std::size_t>(geo_.rw) * geo_.rh * 108 * 4 : 0;
        default: return 0;
    }
}

bool Encoder::fetch(Buffer which, void* host, std::size_t bytes) {
    if (!configured_ || bytes > buffer_bytes(which) || hipSetDevice(device_) != hipSuccess) {
        return false;
    }
    const void* src{nullptr};
    switch (which) {
        case Buffer::kCoeffs: src = coeffs_; break;
        case Buffer::kAcs: src = acs_; break;
        case Buffer::kQuantField: src = qf_; break;
        case Buffer::kCflPartials: src = cfl_part_; break;
        case Buffer::kYtoX: src = ytox_; break;
        case Buffer::kYtoB: src = ytob_; break;
        case Buffer::kAc: src = ac_; break;
        case Buffer::kDc: src = dc_; break;
        case Buffer::kNzGrid: src = nz_grid_; break;
        case Buffer::kNzCount: src = nz_count_; break;
        case Buffer::kHistograms: src = hists_; break;
        case Buffer::kAcGroupBytes: src = ac_group_bytes_; break;
        case Buffer::kDcGroupBytes: src = dc_group_bytes_; break;
        case Buffer::kFeatures: src = features_; break;
        case Buffer::kCodeDepth:
        case Buffer::kCodeBits: {
            // Rows of the code set, one per histogram.
            const std::size_t nh{static_cast<std::size_t>(kNumClusters) + 2 * geo_.num_dc};
            const auto* cs{static_cast<const std::uint8_t*>(codes_)};
            const std::size_t row{static_cast<std::size_t>(which == Buffer::kCodeDepth ? kHistStride : kHistStride * 2)};
            const std::size_t base{static_cast<std::size_t>(which == Buffer::kCodeDepth ? 0 : 96 * kHistStride)};
            return hipMemcpy(host, cs + base, std::min(bytes, nh * row), hipMemcpyDeviceToHost) == hipSuccess;
        }
        default: return false;
    }
    return hipMemcpy(host, src, bytes, hipMemcpyDeviceToHost) == hipSuccess;
}

}  // namespace cjx
