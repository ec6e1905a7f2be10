// tx_capi.hip -- C ABI of the MI355X BC1-BC5 encoder (include/texpresso_hip.h).
//
// Host-buffer entry points (tx_compress, tx_decompress, ...) stage through a
// per-device scratch pool and run synchronously on the device's stream;
// device-buffer entry points only enqueue.  There is no CPU code path.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <mutex>
#include <string.h>
#include <vector>

#include "bcn_kernels.hpp"
#include "texpresso_hip.h"
#include "tx_context.hpp"
#include "tx_tables.hpp"

namespace {

constexpr txt::SingleLut kHostLut = txt::make_single_lut();

bool valid_format(int f) { return f >= TX_BC1 && f <= TX_BC5; }
bool valid_params(const tx_params* p) { return p && p->algorithm >= 0 && p->algorithm <= 2; }

// 4 * width * height without overflow; false when it does not fit
bool image_bytes(size_t w, size_t h, size_t* out)
{
    if (w != 0 && h > SIZE_MAX / 4 / w) return false;
    *out = 4 * w * h;
    return true;
}

}  // namespace

// Device scratch of tx_compress_device_noalloc: the binned pipeline's
// records, keys, sorted lists and counters for TX_NOALLOC_MAX_PIPELINE_BLOCKS
// blocks.  Every GPU the library's code object is loaded on holds its own
// copy.  In host code `scratch` names a host-side stand-in, not a device
// address: the per-device address comes from hipGetSymbolAddress
// (NoallocDevice::ptr), and only that address is passed to kernels.
static_assert(txp::PipeBufs::bytes_for(TX_NOALLOC_MAX_PIPELINE_BLOCKS) == TX_NOALLOC_SCRATCH_BYTES,
              "TX_NOALLOC_SCRATCH_BYTES holds the pipeline buffers of TX_NOALLOC_MAX_PIPELINE_BLOCKS blocks");
static __device__ __align__(256) uint8_t scratch[TX_NOALLOC_SCRATCH_BYTES];

namespace {

struct NoallocDevice {
    bool ready = false;
    uint8_t* ptr = nullptr;  // this device's copy of `scratch`
    uint32_t cus = 0;
};

constexpr int kNoallocDevices = 64;
std::mutex g_noalloc_mu;
NoallocDevice g_noalloc[kNoallocDevices];

// Set-up of the calling thread's current device, once per device: its
// address of `scratch` and its compute-unit count.  Allocates nothing.
int noalloc_device(const NoallocDevice** out)
{
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kNoallocDevices) return TX_ERR_NO_DEVICE;
    std::lock_guard<std::mutex> lock(g_noalloc_mu);
    NoallocDevice& d = g_noalloc[dev];
    if (!d.ready) {
        hipDeviceProp_t prop;
        if (hipGetDeviceProperties(&prop, dev) != hipSuccess || strncmp(prop.gcnArchName, "gfx950", 6) != 0)
            return TX_ERR_NO_DEVICE;
        void* p = nullptr;
        if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || p == nullptr) return TX_ERR_HIP;
        d.ptr = static_cast<uint8_t*>(p);
        d.cus = (uint32_t)prop.multiProcessorCount;
        d.ready = true;
    }
    *out = &d;
    return TX_OK;
}

}  // namespace

extern "C" {

tx_params tx_params_default(void)
{
    tx_params p;
    p.algorithm = TX_CLUSTER_FIT;
    p.weights[0] = 0.2126f;
    p.weights[1] = 0.7152f;
    p.weights[2] = 0.0722f;
    p.weigh_colour_by_alpha = 0;
    return p;
}

size_t tx_num_blocks(size_t size) { return (size + 3) / 4; }

size_t tx_block_size(int format)
{
    if (!valid_format(format)) return 0;
    return (format == TX_BC1 || format == TX_BC4) ? 8 : 16;
}

size_t tx_compressed_size(int format, size_t width, size_t height)
{
    return tx_num_blocks(width) * tx_num_blocks(height) * tx_block_size(format);
}

const char* tx_error_string(int code)
{
    switch (code) {
    case TX_OK: return "ok";
    case TX_ERR_FORMAT: return "invalid format or algorithm";
    case TX_ERR_ZERO_WIDTH: return "width is zero";
    case TX_ERR_INPUT_SHORT: return "input buffer shorter than the image";
    case TX_ERR_OUTPUT_SHORT: return "output buffer smaller than the compressed size";
    case TX_ERR_OUTPUT_PARTIAL: return "output buffer ends inside a block";
    case TX_ERR_ALIGN: return "device pointer misaligned";
    case TX_ERR_HIP: return "HIP runtime error";
    case TX_ERR_NO_DEVICE: return "no usable gfx950 device";
    case TX_ERR_BUSY: return "queue full";
    case TX_ERR_INVALID: return "invalid argument or handle";
    case TX_ERR_NOMEM: return "device memory budget exceeded";
    case TX_ERR_TOO_LARGE: return "texture exceeds the allocation-free scratch (TX_NOALLOC_MAX_PIPELINE_BLOCKS)";
    default: return "unknown error";
    }
}

void tx_single_lut(uint8_t out[6144]) { memcpy(out, &kHostLut, sizeof kHostLut); }

uint64_t tx_set_pipeline_threshold(uint64_t min_blocks)
{
    const uint64_t old = txc::pipeline_min_blocks();
    txc::set_pipeline_min_blocks(min_blocks);
    return old;
}

const char* tx_device_arch(void)
{
    txc::DeviceContext* ctx = txc::current_context(nullptr);
    return ctx ? ctx->arch : nullptr;
}

// Validation shared by the image entry points (lib.rs:295-305 semantics).
static int check_compress(int format, size_t width, size_t height, const tx_params* params, size_t out_len,
                          size_t* in_bytes)
{
    if (!valid_format(format) || !valid_params(params)) return TX_ERR_FORMAT;
    if (width == 0) return TX_ERR_ZERO_WIDTH;
    if (width > 0x7FFFFFFFu || height > 0x7FFFFFFFu) return TX_ERR_INVALID;
    if (!image_bytes(width, height, in_bytes)) return TX_ERR_INVALID;
    const size_t bs = tx_block_size(format);
    if (out_len < tx_compressed_size(format, width, height)) return TX_ERR_OUTPUT_SHORT;
    if (out_len % bs != 0) return TX_ERR_OUTPUT_PARTIAL;
    return TX_OK;
}

static txk::EncodeArgs encode_args(int format, const tx_params* p, const uint8_t* d_in, size_t w, size_t h,
                                   uint8_t* d_out, size_t out_len)
{
    txk::EncodeArgs a;
    a.format = format;
    a.algorithm = p->algorithm;
    a.rgba = d_in;
    a.width = (uint32_t)w;
    a.height = (uint32_t)h;
    a.blocks_wide = (uint32_t)tx_num_blocks(w);
    a.nblocks = out_len / tx_block_size(format);
    a.out = d_out;
    a.wr = p->weights[0];
    a.wg = p->weights[1];
    a.wb = p->weights[2];
    a.weigh_alpha = p->weigh_colour_by_alpha ? 1u : 0u;
    a.may_overlap = false;
    a.over_bus = false;
    return a;
}

// Blocks from which a texture goes through the binned pipeline, as a share of
// the set threshold (default 32,768), in sixteenths: the measured crossings
// against the direct kernels (square seeded textures, pipeline / direct us).
// BC2/BC3 IterativeClusterFit 205 / 196 at 30,976 blocks, 220 / 239 at 36,864.
// BC1 IterativeClusterFit runs two searches after classify, which textures with
// flat areas or few colours do not repay: of noise 250 / 247 at 57,600 blocks,
// 284 / 282 at 73,984, 344 / 348 at 92,416 (of 1024 x 1024 259 / 315), of the
// same with three quarters of its tiles flat 157 / 127, 172 / 140 and 189 / 154
// (161 / 141), with 8 levels a channel 149 / 52, 153 / 63 and 133 / 74 (152 / 67).
// ClusterFit on the library's own stream, where calls run one after another: BC1
// 52 / 61 at 16,384 blocks (the direct kernel's last full round of waves), 51 /
// 58 at 18,769, 60 / 63 at 25,600, 68 / 82 at 33,856, with flat tiles 38 / 38,
// 39 / 49 and 40 / 56; BC3 55 / 52, 59 / 70, 76 / 83 and 91 / 102, with flat
// tiles 40 / 43, 46 / 51 and 47 / 56.  (With 8 levels a channel the direct
// kernels stay ahead by 4-11 us up to 40,000 blocks, BC3 28 / 18 at 18,769.)
// With point weights from alpha classify takes longer: BC1 59 / 59 at 18,769, 71 /
// 64 at 25,600, 72 / 78 at 29,584; BC3 71 / 71 at 20,736, 86 / 86 at 25,600, 97 /
// 95 at 29,584 and 125 / 123 at 40,804.  A chain's small levels fill the direct
// launch badly, so there the pipeline starts as early as without weights and for
// BC1 IterativeClusterFit too (chains of noise of 61,801 blocks 274 / 316, 83,460
// 318 / 354, with flat tiles 229 / 189 and 234 / 212).
// Calls on a caller's stream may overlap those on other streams, which only the
// direct kernels allow (three streams, BC1 ClusterFit, per call: 100 / 73 at
// 40,000 blocks), so there the pipeline starts later.
static uint64_t pipeline_threshold(const txk::EncodeArgs& a, bool is_chain, bool own_stream)
{
    const uint64_t t = txc::pipeline_min_blocks();
    const bool bc1 = a.format == TX_BC1, iterative = a.algorithm == TX_ITERATIVE_CLUSTER_FIT;
    uint64_t sixteenths = bc1 ? (iterative ? 48 : 24) : (iterative ? 16 : 20);
    if (own_stream && !iterative) sixteenths = is_chain || !a.weigh_alpha ? 9 : bc1 ? 14 : 20;
    if (own_stream && iterative && bc1 && is_chain) sixteenths = 28;
    return t > UINT64_MAX / sixteenths ? UINT64_MAX : t * sixteenths / 16;
}

// Whether a texture goes through the binned pipeline: ClusterFit or
// IterativeClusterFit in BC1-BC3 with at least pipeline_threshold() blocks.
static bool takes_pipeline(const txk::EncodeArgs& a, bool is_chain, bool own_stream)
{
    const bool cluster = a.format <= TX_BC3 && a.algorithm != TX_RANGE_FIT;
    return cluster && a.nblocks >= pipeline_threshold(a, is_chain, own_stream) && a.nblocks <= 0xFFFFFFFFull;
}

// Whether `s` is being captured into a graph.
static bool capturing(hipStream_t s)
{
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    return hipStreamIsCapturing(s, &status) == hipSuccess && status != hipStreamCaptureStatusNone;
}

// Launch shape of the binned pipeline for one texture, or for the levels of
// `chain` (a.nblocks blocks in all), on a device with `cus` compute units.
static txp::PipeLaunch pipe_launch_for(const txk::EncodeArgs& a, const txk::ChainTable* chain, uint32_t cus)
{
    txp::PipeLaunch p{};
    p.d_tex = nullptr;
    p.tex0.rgba = a.rgba;
    p.tex0.out = a.out;
    p.tex0.width = a.width;
    p.tex0.height = a.height;
    p.tex0.blocks_wide = a.blocks_wide;
    p.tex0.nblocks = (uint32_t)a.nblocks;
    p.tex0.variant = 3u * (uint32_t)a.format + (uint32_t)a.algorithm;
    p.tex0.pad = 0;
    p.tex0.wr = a.wr;
    p.tex0.wg = a.wg;
    p.tex0.wb = a.wb;
    p.tex0.weigh_alpha = a.weigh_alpha;
    // persistent single-wave workgroups, 16 per CU for both passes.  Classify
    // runs one block per lane: chunks of 64 blocks fill a wave; a texture
    // with fewer than 64 blocks per SIMD is cut into chunks of at least 16
    // so that it still reaches every SIMD (one wave per SIMD with all lanes
    // busy beats several part-filled ones)
    const uint64_t cwaves = (uint64_t)cus * txp::kClassifyWavesPerCu;
    const uint64_t swaves = (uint64_t)cus * txp::kSearchWavesPerCu;
    const uint64_t simds = (uint64_t)cus * 4;
    uint64_t cb = (a.nblocks + simds - 1) / simds;
    cb = std::min<uint64_t>(64, std::max<uint64_t>(16, (cb + 15) & ~(uint64_t)15));
    p.chunk_blocks = (uint32_t)cb;
    if (chain) p.chain = *chain;
    p.nchunks = (uint32_t)(chain ? p.chain.number(p.chunk_blocks) : (a.nblocks + cb - 1) / cb);
    p.nslots = a.nblocks;
    p.d_chunks = nullptr;
    p.classify_grid = (uint32_t)std::min<uint64_t>(cwaves, p.nchunks);
    p.search_grid = (uint32_t)std::min<uint64_t>(swaves, (a.nblocks + 3) / 4);
    p.lists = txp::lists_for((uint32_t)a.format, (uint32_t)a.algorithm);
    return p;
}

// Encodes one texture on `s`: textures that take_pipeline() go through the
// binned pipeline (classify, bin, independent per-block searches),
// everything else through the direct kernel.  Both produce the same bytes.
// With `marks` (5 events) the pipeline records them between its kernels;
// `used_pipeline` says which path ran.  With `chain`, the levels of a chain
// instead of one texture (a.nblocks counts the blocks of them all).
static hipError_t encode_on(txc::DeviceContext* ctx, txk::EncodeArgs a, hipStream_t s,
                            const txk::ChainTable* chain = nullptr, hipEvent_t* marks = nullptr,
                            bool* used_pipeline = nullptr)
{
    if (used_pipeline) *used_pipeline = false;
    // the pipeline's shared buffers are ordered between streams by events, which
    // a captured stream cannot wait for
    const bool own = s == ctx->stream;
    a.may_overlap = !own && !chain;
    const auto direct = [&] { return chain ? txk::launch_encode_chain(a, *chain, s) : txk::launch_encode(a, s); };
    if (!takes_pipeline(a, chain != nullptr, own) || (!own && capturing(s))) return direct();
    std::lock_guard<std::mutex> lock(ctx->pipe_mu);
    txp::PipeBufs bufs;
    if (!ctx->pipe_scratch(a.nblocks, &bufs)) {
        // no memory for the records; the direct kernels need none.  The failed
        // allocation must not be taken for a failed launch.
        (void)hipGetLastError();
        return direct();
    }
    if (used_pipeline) *used_pipeline = true;
    if (!ctx->pipe_before(s)) return hipErrorUnknown;
    const hipError_t e = txp::launch_pipeline(pipe_launch_for(a, chain, (uint32_t)ctx->cus), bufs, s, marks);
    if (!ctx->pipe_after(s)) return hipErrorUnknown;
    return e;
}

// Kernels read pinned input themselves up to this size.  The decoder and the
// one-block-per-lane encoders read it once in long runs: no copy is faster at
// every staged size (RangeFit 512^2 71 us against 83 with one, 64^2 24 / 27;
// decoding 512^2 68 / 80, 64^2 16 / 21), and RangeFit takes its groups for few
// blocks of such input only (txk::range_group_blocks).  The 16-lane groups of the cluster
// fits fetch 16 bytes at a time over the bus, which a copy beats from about 64
// KiB on (BC1 ClusterFit 64^2 31 us against 32 with a copy, 128^2 41 / 40,
// 256^2 64 / 59).
constexpr size_t kDirectGroupBytes = 32u << 10;

static size_t direct_in_bytes(int format, int algorithm)
{
    return format <= TX_BC3 && algorithm != TX_RANGE_FIT ? kDirectGroupBytes : txc::kStageBytes;
}

namespace {

// Moves a host-staged call's input and output (txc::kStageBytes).  Used under
// the context's lock, by one call at a time, which ends with finish().
class HostCall {
public:
    HostCall(txc::DeviceContext* c, size_t in_total, size_t direct_in_max, size_t out_total) : ctx(c)
    {
        if (in_total <= txc::kStageBytes || out_total <= txc::kStageBytes) pin = ctx->staging();
        stage_in = pin && in_total <= txc::kStageBytes;
        direct_in = stage_in && in_total <= direct_in_max;
        stage_out = pin && out_total <= txc::kStageBytes;
    }
    // n bytes of `src` where kernels on the context's stream can read them:
    // d_buf, or the pinned memory itself at `at` of its input half (the parts
    // of a call's input follow one another).  Null on an error.
    const uint8_t* upload(uint8_t* d_buf, const void* src, size_t n, size_t at = 0)
    {
        if (n == 0) return d_buf;
        if (stage_in) {
            memcpy(pin + at, src, n);
            if (direct_in) return pin + at;
            src = pin + at;
        }
        return hipMemcpyAsync(d_buf, src, n, hipMemcpyHostToDevice, ctx->stream) == hipSuccess ? d_buf : nullptr;
    }
    // Whether upload() hands out the pinned memory itself.
    bool reads_pinned() const { return direct_in; }
    // Where kernels write the output: d_buf, or the pinned memory.
    uint8_t* output(uint8_t* d_buf) { return stage_out ? pin + txc::kStageBytes : d_buf; }
    // Waits for the call's work and leaves its n bytes of output in dst.
    int finish(void* dst, const uint8_t* d_buf, size_t n)
    {
        if (!stage_out && hipMemcpyAsync(dst, d_buf, n, hipMemcpyDeviceToHost, ctx->stream) != hipSuccess)
            return TX_ERR_HIP;
        if (hipStreamSynchronize(ctx->stream) != hipSuccess) return TX_ERR_HIP;
        if (stage_out) memcpy(dst, pin + txc::kStageBytes, n);
        return TX_OK;
    }

private:
    txc::DeviceContext* ctx;
    uint8_t* pin = nullptr;
    bool stage_in = false, direct_in = false, stage_out = false;
};

}  // namespace

int tx_compress(int format, const uint8_t* rgba, size_t rgba_len, size_t width, size_t height,
                const tx_params* params, uint8_t* output, size_t out_len)
{
    size_t in_bytes = 0;
    int rc = check_compress(format, width, height, params, out_len, &in_bytes);
    if (rc != TX_OK) return rc;
    if (rgba_len < in_bytes) return TX_ERR_INPUT_SHORT;
    if (out_len == 0) return TX_OK;
    if ((in_bytes && !rgba) || !output) return TX_ERR_INVALID;
    txc::DeviceContext* ctx = txc::current_context(&rc);
    if (!ctx) return rc;
    std::lock_guard<std::mutex> lock(ctx->mu);
    const size_t in_cap = (in_bytes + 255) & ~(size_t)255;
    uint8_t* d = ctx->scratch(in_cap + out_len);
    if (!d) return TX_ERR_NOMEM;
    HostCall call(ctx, in_bytes, direct_in_bytes(format, params->algorithm), out_len);
    const uint8_t* d_in = call.upload(d, rgba, in_bytes);
    uint8_t* d_out = call.output(d + in_cap);
    if (!d_in) return TX_ERR_HIP;
    txk::EncodeArgs a = encode_args(format, params, d_in, width, height, d_out, out_len);
    a.over_bus = call.reads_pinned();
    if (encode_on(ctx, a, ctx->stream) != hipSuccess) return TX_ERR_HIP;
    return call.finish(output, d_out, out_len);
}

int tx_compress_device(int format, const uint8_t* d_rgba, size_t width, size_t height, const tx_params* params,
                       uint8_t* d_output, size_t out_len, void* stream)
{
    size_t in_bytes = 0;
    int rc = check_compress(format, width, height, params, out_len, &in_bytes);
    if (rc != TX_OK) return rc;
    if (out_len == 0) return TX_OK;
    if ((in_bytes && !d_rgba) || !d_output) return TX_ERR_INVALID;
    if (((uintptr_t)d_rgba & 3u) || ((uintptr_t)d_output & (tx_block_size(format) - 1))) return TX_ERR_ALIGN;
    txc::DeviceContext* ctx = txc::current_context(&rc);
    if (!ctx) return rc;
    hipStream_t s = stream ? (hipStream_t)stream : ctx->stream;
    if (encode_on(ctx, encode_args(format, params, d_rgba, width, height, d_output, out_len), s) != hipSuccess)
        return TX_ERR_HIP;
    return TX_OK;
}

// ------------------------------------------------------------ allocation-free entry point

int tx_compress_device_noalloc(int format, const uint8_t* d_rgba, size_t width, size_t height,
                               const tx_params* params, uint8_t* d_output, size_t out_len, void* stream)
{
    size_t in_bytes = 0;
    int rc = check_compress(format, width, height, params, out_len, &in_bytes);
    if (rc != TX_OK) return rc;
    if (out_len == 0) return TX_OK;
    if ((in_bytes && !d_rgba) || !d_output) return TX_ERR_INVALID;
    if (((uintptr_t)d_rgba & 3u) || ((uintptr_t)d_output & (tx_block_size(format) - 1))) return TX_ERR_ALIGN;
    const NoallocDevice* dev = nullptr;
    rc = noalloc_device(&dev);
    if (rc != TX_OK) return rc;
    const hipStream_t s = (hipStream_t)stream;
    txk::EncodeArgs a = encode_args(format, params, d_rgba, width, height, d_output, out_len);
    a.may_overlap = true;
    if (!takes_pipeline(a, false, false)) return txk::launch_encode(a, s) == hipSuccess ? TX_OK : TX_ERR_HIP;
    if (a.nblocks > TX_NOALLOC_MAX_PIPELINE_BLOCKS) return TX_ERR_TOO_LARGE;
    txp::PipeBufs bufs;
    bufs.carve(dev->ptr, TX_NOALLOC_MAX_PIPELINE_BLOCKS);
    return txp::launch_pipeline(pipe_launch_for(a, nullptr, dev->cus), bufs, s) == hipSuccess ? TX_OK : TX_ERR_HIP;
}

// ------------------------------------------------------------ mip chains

static size_t mip_side(size_t v, uint32_t level) { return level >= 64 ? 1 : std::max<size_t>(1, v >> level); }

uint32_t tx_mip_levels(size_t width, size_t height)
{
    if (width == 0 || height == 0) return 0;
    uint32_t n = 1;
    for (size_t m = std::max(width, height); m > 1; m >>= 1) ++n;
    return n;
}

void tx_mip_dims(size_t width, size_t height, uint32_t level, size_t* w_out, size_t* h_out)
{
    if (w_out) *w_out = mip_side(width, level);
    if (h_out) *h_out = mip_side(height, level);
}

size_t tx_mip_chain_rgba_bytes(size_t width, size_t height, uint32_t levels)
{
    size_t total = 0;
    for (uint32_t k = 1; k < levels; ++k) {
        size_t b = 0;
        if (!image_bytes(mip_side(width, k), mip_side(height, k), &b) || total > SIZE_MAX - b) return SIZE_MAX;
        total += b;
    }
    return total;
}

size_t tx_mip_chain_compressed_size(int format, size_t width, size_t height, uint32_t levels)
{
    size_t total = 0;
    for (uint32_t k = 0; k < levels; ++k) total += tx_compressed_size(format, mip_side(width, k), mip_side(height, k));
    return total;
}

// Shared checks of the mip-chain entry points.
static int check_mips(size_t width, size_t height, uint32_t levels, size_t chain_len)
{
    if (width == 0) return TX_ERR_ZERO_WIDTH;
    if (height == 0 || width > 0x7FFFFFFFu || height > 0x7FFFFFFFu) return TX_ERR_INVALID;
    // the whole chain holds less than 4/3 of level 0: keep level 0 below half
    // the address space so every size computed from it fits
    size_t level0 = 0;
    if (!image_bytes(width, height, &level0) || level0 > SIZE_MAX / 2) return TX_ERR_INVALID;
    if (levels == 0 || levels > tx_mip_levels(width, height)) return TX_ERR_INVALID;
    if (chain_len < tx_mip_chain_rgba_bytes(width, height, levels)) return TX_ERR_OUTPUT_SHORT;
    return TX_OK;
}

// Levels 1..levels-1 into d_chain, kMipLevelsPerLaunch at a time.
static hipError_t mips_on(const uint8_t* d_rgba, size_t width, size_t height, uint32_t levels, uint8_t* d_chain,
                          hipStream_t s)
{
    const uint8_t* src = d_rgba;
    uint8_t* dst = d_chain;
    for (uint32_t k = 0; k + 1 < levels;) {
        const uint32_t n = std::min(levels - 1 - k, txk::kMipLevelsPerLaunch);
        const hipError_t e =
            txk::launch_mip_levels(src, (uint32_t)mip_side(width, k), (uint32_t)mip_side(height, k), n, dst, s);
        if (e != hipSuccess) return e;
        for (uint32_t m = 0; m < n; ++m) {  // dst ends up past the last of these levels, src on it
            ++k;
            src = dst;
            dst += 4 * mip_side(width, k) * mip_side(height, k);
        }
    }
    return hipSuccess;
}

// Levels of more blocks than this are encoded by launches of their own and the
// rest of the chain by one: a level takes one block's latency however small it
// is (13-70 us, eleven levels in series for a 1024^2 chain), while a large
// level fills the GPU by itself and would only enlarge the record buffers.
constexpr uint64_t kChainLevelMaxBlocks = 1u << 20;

// Every level of the chain (level 0 = d_rgba, then d_chain) compressed back
// to back into d_output, level 0 first.
static hipError_t compress_chain_on(txc::DeviceContext* ctx, int format, const tx_params* params,
                                    const uint8_t* d_rgba, size_t width, size_t height, uint32_t levels,
                                    const uint8_t* d_chain, uint8_t* d_output, hipStream_t s)
{
    txk::ChainTable chain{};  // the levels that go together
    uint64_t chain_blocks = 0;
    uint8_t* chain_out = d_output;
    const uint8_t* src = d_rgba;
    size_t in_off = 0, out_off = 0;
    for (uint32_t k = 0; k < levels; ++k) {
        const size_t w = mip_side(width, k), h = mip_side(height, k);
        const size_t n = tx_compressed_size(format, w, h);
        if (k > 0) {
            src = d_chain + in_off;
            in_off += 4 * w * h;
        }
        const txk::EncodeArgs a = encode_args(format, params, src, w, h, d_output + out_off, n);
        if (a.nblocks > kChainLevelMaxBlocks || levels == 1) {
            const hipError_t e = encode_on(ctx, a, s);
            if (e != hipSuccess) return e;
        } else {
            if (chain.count == 0) chain_out = a.out;
            if (chain.count == txk::kMaxChainLevels) return hipErrorInvalidValue;
            chain.level[chain.count++] = txk::ChainTable::Level{
                src, (uint32_t)w, (uint32_t)h, a.blocks_wide, (uint32_t)a.nblocks, (uint32_t)chain_blocks};
            chain_blocks += a.nblocks;
        }
        out_off += n;
    }
    if (chain.count == 0) return hipSuccess;
    txk::EncodeArgs a = encode_args(format, params, chain.level[0].rgba, chain.level[0].width, chain.level[0].height,
                                    chain_out, chain_blocks * tx_block_size(format));
    return encode_on(ctx, a, s, chain.count > 1 ? &chain : nullptr);
}

int tx_generate_mips_device(const uint8_t* d_rgba, size_t width, size_t height, uint32_t levels, uint8_t* d_chain,
                            size_t chain_len, void* stream)
{
    int rc = check_mips(width, height, levels, chain_len);
    if (rc != TX_OK) return rc;
    if (levels == 1) return TX_OK;
    if (!d_rgba || !d_chain) return TX_ERR_INVALID;
    if (((uintptr_t)d_rgba & 3u) || ((uintptr_t)d_chain & 3u)) return TX_ERR_ALIGN;
    txc::DeviceContext* ctx = txc::current_context(&rc);
    if (!ctx) return rc;
    return mips_on(d_rgba, width, height, levels, d_chain, stream ? (hipStream_t)stream : ctx->stream) == hipSuccess
               ? TX_OK
               : TX_ERR_HIP;
}

int tx_compress_mips_device(int format, const uint8_t* d_rgba, size_t width, size_t height, const tx_params* params,
                            uint32_t levels, uint8_t* d_chain, size_t chain_len, uint8_t* d_output, size_t out_len,
                            void* stream)
{
    if (!valid_format(format) || !valid_params(params)) return TX_ERR_FORMAT;
    int rc = check_mips(width, height, levels, chain_len);
    if (rc != TX_OK) return rc;
    if (out_len < tx_mip_chain_compressed_size(format, width, height, levels)) return TX_ERR_OUTPUT_SHORT;
    if (!d_rgba || !d_output || (levels > 1 && !d_chain)) return TX_ERR_INVALID;
    if (((uintptr_t)d_rgba & 3u) || ((uintptr_t)d_chain & 3u) || ((uintptr_t)d_output & (tx_block_size(format) - 1)))
        return TX_ERR_ALIGN;
    txc::DeviceContext* ctx = txc::current_context(&rc);
    if (!ctx) return rc;
    hipStream_t s = stream ? (hipStream_t)stream : ctx->stream;
    if (mips_on(d_rgba, width, height, levels, d_chain, s) != hipSuccess) return TX_ERR_HIP;
    if (compress_chain_on(ctx, format, params, d_rgba, width, height, levels, d_chain, d_output, s) != hipSuccess)
        return TX_ERR_HIP;
    return TX_OK;
}

int tx_compress_mips(int format, const uint8_t* rgba, size_t rgba_len, size_t width, size_t height,
                     const tx_params* params, uint32_t levels, uint8_t* output, size_t out_len)
{
    if (!valid_format(format) || !valid_params(params)) return TX_ERR_FORMAT;
    const size_t chain_len = tx_mip_chain_rgba_bytes(width, height, levels);
    int rc = check_mips(width, height, levels, chain_len);
    if (rc != TX_OK) return rc;
    size_t in_bytes = 0;
    if (!image_bytes(width, height, &in_bytes)) return TX_ERR_INVALID;
    if (rgba_len < in_bytes) return TX_ERR_INPUT_SHORT;
    const size_t need = tx_mip_chain_compressed_size(format, width, height, levels);
    if (out_len < need) return TX_ERR_OUTPUT_SHORT;
    if (!rgba || !output) return TX_ERR_INVALID;
    txc::DeviceContext* ctx = txc::current_context(&rc);
    if (!ctx) return rc;
    std::lock_guard<std::mutex> lock(ctx->mu);
    auto up = [](size_t x) { return (x + 255) & ~(size_t)255; };
    uint8_t* d = ctx->scratch(up(in_bytes) + up(chain_len) + need);
    if (!d) return TX_ERR_NOMEM;
    uint8_t* d_chain = d + up(in_bytes);
    HostCall call(ctx, in_bytes, direct_in_bytes(format, params->algorithm), need);
    const uint8_t* d_in = call.upload(d, rgba, in_bytes);
    uint8_t* d_out = call.output(d_chain + up(chain_len));
    if (!d_in) return TX_ERR_HIP;
    if (mips_on(d_in, width, height, levels, d_chain, ctx->stream) != hipSuccess) return TX_ERR_HIP;
    if (compress_chain_on(ctx, format, params, d_in, width, height, levels, d_chain, d_out, ctx->stream) !=
        hipSuccess)
        return TX_ERR_HIP;
    return call.finish(output, d_out, need);
}

int tx_compress_block_masked(int format, const uint8_t rgba[64], uint32_t mask, const tx_params* params,
                             uint8_t* output, size_t out_len)
{
    if (!valid_format(format) || !valid_params(params)) return TX_ERR_FORMAT;
    if (!rgba || !output) return TX_ERR_INVALID;
    if (out_len < tx_block_size(format)) return TX_ERR_OUTPUT_SHORT;
    return tx_compress_blocks(format, rgba, &mask, 1, params, output);
}

int tx_compress_blocks(int format, const uint8_t* blocks, const uint32_t* masks, size_t nblocks,
                       const tx_params* params, uint8_t* output)
{
    if (!valid_format(format) || !valid_params(params)) return TX_ERR_FORMAT;
    if (nblocks == 0) return TX_OK;
    if (!blocks || !masks || !output) return TX_ERR_INVALID;
    if (nblocks > SIZE_MAX / 64) return TX_ERR_INVALID;
    int rc = TX_OK;
    txc::DeviceContext* ctx = txc::current_context(&rc);
    if (!ctx) return rc;
    std::lock_guard<std::mutex> lock(ctx->mu);
    const size_t bs = tx_block_size(format);
    const size_t pix = 64 * nblocks, msk = (4 * nblocks + 255) & ~(size_t)255;
    uint8_t* d = ctx->scratch(pix + msk + nblocks * bs);
    if (!d) return TX_ERR_NOMEM;
    HostCall call(ctx, pix + 4 * nblocks, kDirectGroupBytes, nblocks * bs);
    const uint8_t* d_pix = call.upload(d, blocks, pix);
    const uint8_t* d_mask = call.upload(d + pix, masks, 4 * nblocks, pix);
    uint8_t* d_out = call.output(d + pix + msk);
    if (!d_pix || !d_mask) return TX_ERR_HIP;
    txk::BlockListArgs a;
    a.format = format;
    a.algorithm = params->algorithm;
    a.blocks = d_pix;
    a.masks = reinterpret_cast<const uint32_t*>(d_mask);
    a.nblocks = nblocks;
    a.out = d_out;
    a.wr = params->weights[0];
    a.wg = params->weights[1];
    a.wb = params->weights[2];
    a.weigh_alpha = params->weigh_colour_by_alpha ? 1u : 0u;
    if (txk::launch_encode_blocks(a, ctx->stream) != hipSuccess) return TX_ERR_HIP;
    return call.finish(output, d_out, nblocks * bs);
}

int tx_decompress(int format, const uint8_t* data, size_t data_len, size_t width, size_t height, uint8_t* output,
                  size_t out_len)
{
    if (!valid_format(format)) return TX_ERR_FORMAT;
    if (width == 0) return TX_ERR_ZERO_WIDTH;
    if (width > 0x7FFFFFFFu || height > 0x7FFFFFFFu) return TX_ERR_INVALID;
    size_t px_bytes = 0;
    if (!image_bytes(width, height, &px_bytes)) return TX_ERR_INVALID;
    const size_t need = tx_compressed_size(format, width, height);
    if (data_len < need) return TX_ERR_INPUT_SHORT;
    if (out_len < px_bytes) return TX_ERR_OUTPUT_SHORT;
    if (px_bytes == 0) return TX_OK;
    if (!data || !output) return TX_ERR_INVALID;
    int rc = TX_OK;
    txc::DeviceContext* ctx = txc::current_context(&rc);
    if (!ctx) return rc;
    std::lock_guard<std::mutex> lock(ctx->mu);
    const size_t in_cap = (need + 255) & ~(size_t)255;
    uint8_t* d = ctx->scratch(in_cap + px_bytes);
    if (!d) return TX_ERR_NOMEM;
    HostCall call(ctx, need, txc::kStageBytes, px_bytes);
    const uint8_t* d_in = call.upload(d, data, need);
    uint8_t* d_out = call.output(d + in_cap);
    if (!d_in) return TX_ERR_HIP;
    if (txk::launch_decode(format, d_in, (uint32_t)width, (uint32_t)height, d_out, ctx->stream) != hipSuccess)
        return TX_ERR_HIP;
    return call.finish(output, d_out, px_bytes);
}

int tx_decompress_device(int format, const uint8_t* d_data, size_t width, size_t height, uint8_t* d_output,
                         void* stream)
{
    if (!valid_format(format)) return TX_ERR_FORMAT;
    if (width == 0) return TX_ERR_ZERO_WIDTH;
    if (width > 0x7FFFFFFFu || height > 0x7FFFFFFFu) return TX_ERR_INVALID;
    if (height == 0) return TX_OK;
    if (!d_data || !d_output) return TX_ERR_INVALID;
    if ((uintptr_t)d_output & 3u) return TX_ERR_ALIGN;
    int rc = TX_OK;
    txc::DeviceContext* ctx = txc::current_context(&rc);
    if (!ctx) return rc;
    hipStream_t s = stream ? (hipStream_t)stream : ctx->stream;
    if (txk::launch_decode(format, d_data, (uint32_t)width, (uint32_t)height, d_output, s) != hipSuccess)
        return TX_ERR_HIP;
    return TX_OK;
}

int tx_util_malloc(void** d_ptr, size_t bytes)
{
    if (!d_ptr) return TX_ERR_INVALID;
    int rc = TX_OK;
    if (!txc::current_context(&rc)) return rc;
    if (hipMalloc(d_ptr, bytes ? bytes : 1) != hipSuccess) return TX_ERR_NOMEM;
    return TX_OK;
}

int tx_util_free(void* d_ptr)
{
    if (!d_ptr) return TX_OK;
    return hipFree(d_ptr) == hipSuccess ? TX_OK : TX_ERR_HIP;
}

int tx_util_upload(void* d_dst, const void* src, size_t bytes)
{
    if (bytes == 0) return TX_OK;
    if (!d_dst || !src) return TX_ERR_INVALID;
    return hipMemcpy(d_dst, src, bytes, hipMemcpyHostToDevice) == hipSuccess ? TX_OK : TX_ERR_HIP;
}

int tx_util_download(void* dst, const void* d_src, size_t bytes)
{
    if (bytes == 0) return TX_OK;
    if (!dst || !d_src) return TX_ERR_INVALID;
    int rc = TX_OK;
    txc::DeviceContext* ctx = txc::current_context(&rc);
    if (!ctx) return rc;
    if (hipStreamSynchronize(ctx->stream) != hipSuccess) return TX_ERR_HIP;
    return hipMemcpy(dst, d_src, bytes, hipMemcpyDeviceToHost) == hipSuccess ? TX_OK : TX_ERR_HIP;
}

int tx_util_copy(void* d_dst, const void* d_src, size_t bytes)
{
    if (bytes == 0) return TX_OK;
    if (!d_dst || !d_src) return TX_ERR_INVALID;
    int rc = TX_OK;
    txc::DeviceContext* ctx = txc::current_context(&rc);
    if (!ctx) return rc;
    if (hipMemcpyAsync(d_dst, d_src, bytes, hipMemcpyDeviceToDevice, ctx->stream) != hipSuccess) return TX_ERR_HIP;
    return hipStreamSynchronize(ctx->stream) == hipSuccess ? TX_OK : TX_ERR_HIP;
}

int tx_util_elementary(const float* in, size_t n, float u8f[256], float sqrt_counts[17], float sqrt_alpha[4096],
                       float* snap31, float* snap63, int32_t* round255)
{
    if (!u8f || !sqrt_counts || !sqrt_alpha || n > ((size_t)1 << 26) || (n && (!in || !snap31 || !snap63 || !round255)))
        return TX_ERR_INVALID;
    int rc = TX_OK;
    txc::DeviceContext* ctx = txc::current_context(&rc);
    if (!ctx) return rc;
    constexpr size_t kTables = 256 + 17 + 4096;
    const size_t m = n ? n : 1;
    uint8_t* d = nullptr;
    const size_t bytes = 4 * (kTables + 4 * m);
    if (hipMalloc(&d, bytes) != hipSuccess) return TX_ERR_NOMEM;
    float* d_tables = reinterpret_cast<float*>(d);
    float* d_in = d_tables + kTables;
    float* d_s31 = d_in + m;
    float* d_s63 = d_s31 + m;
    int32_t* d_r = reinterpret_cast<int32_t*>(d_s63 + m);
    rc = TX_OK;
    if (n && hipMemcpyAsync(d_in, in, 4 * n, hipMemcpyHostToDevice, ctx->stream) != hipSuccess) rc = TX_ERR_HIP;
    if (rc == TX_OK && txk::launch_elementary(d_in, (uint32_t)n, d_tables, d_s31, d_s63, d_r, ctx->stream) != hipSuccess)
        rc = TX_ERR_HIP;
    if (rc == TX_OK && hipStreamSynchronize(ctx->stream) != hipSuccess) rc = TX_ERR_HIP;
    float tables[kTables];
    if (rc == TX_OK && hipMemcpy(tables, d_tables, sizeof tables, hipMemcpyDeviceToHost) != hipSuccess) rc = TX_ERR_HIP;
    if (rc == TX_OK && n &&
        (hipMemcpy(snap31, d_s31, 4 * n, hipMemcpyDeviceToHost) != hipSuccess ||
         hipMemcpy(snap63, d_s63, 4 * n, hipMemcpyDeviceToHost) != hipSuccess ||
         hipMemcpy(round255, d_r, 4 * n, hipMemcpyDeviceToHost) != hipSuccess))
        rc = TX_ERR_HIP;
    if (rc == TX_OK) {
        memcpy(u8f, tables, 4 * 256);
        memcpy(sqrt_counts, tables + 256, 4 * 17);
        memcpy(sqrt_alpha, tables + 256 + 17, 4 * 4096);
    }
    (void)hipFree(d);
    return rc;
}

int tx_util_reciprocal(const float* in, size_t n, float* out)
{
    if (n > ((size_t)1 << 26) || (n && (!in || !out))) return TX_ERR_INVALID;
    int rc = TX_OK;
    txc::DeviceContext* ctx = txc::current_context(&rc);
    if (!ctx) return rc;
    if (n == 0) return TX_OK;
    float* d = nullptr;
    if (hipMalloc(&d, 8 * n) != hipSuccess) return TX_ERR_NOMEM;
    if (hipMemcpyAsync(d, in, 4 * n, hipMemcpyHostToDevice, ctx->stream) != hipSuccess ||
        txk::launch_reciprocal(d, (uint32_t)n, d + n, ctx->stream) != hipSuccess ||
        hipMemcpyAsync(out, d + n, 4 * n, hipMemcpyDeviceToHost, ctx->stream) != hipSuccess)
        rc = TX_ERR_HIP;
    if (hipStreamSynchronize(ctx->stream) != hipSuccess) rc = TX_ERR_HIP;
    (void)hipFree(d);
    return rc;
}

int tx_util_time_compress(int format, const uint8_t* d_rgba, size_t width, size_t height, const tx_params* params,
                          uint8_t* d_output, size_t out_len, int iters, float* ms_total)
{
    if (!ms_total || iters < 1) return TX_ERR_INVALID;
    int rc = TX_OK;
    txc::DeviceContext* ctx = txc::current_context(&rc);
    if (!ctx) return rc;
    hipEvent_t e0, e1;
    if (hipEventCreate(&e0) != hipSuccess) return TX_ERR_HIP;
    if (hipEventCreate(&e1) != hipSuccess) {
        (void)hipEventDestroy(e0);
        return TX_ERR_HIP;
    }
    rc = hipEventRecord(e0, ctx->stream) == hipSuccess ? TX_OK : TX_ERR_HIP;
    for (int i = 0; i < iters && rc == TX_OK; ++i)
        rc = tx_compress_device(format, d_rgba, width, height, params, d_output, out_len, ctx->stream);
    if (rc == TX_OK && hipEventRecord(e1, ctx->stream) != hipSuccess) rc = TX_ERR_HIP;
    if (rc == TX_OK && hipEventSynchronize(e1) != hipSuccess) rc = TX_ERR_HIP;
    if (rc == TX_OK && hipEventElapsedTime(ms_total, e0, e1) != hipSuccess) rc = TX_ERR_HIP;
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    return rc;
}

int tx_util_time_phases(int format, const uint8_t* d_rgba, size_t width, size_t height, const tx_params* params,
                        uint8_t* d_output, size_t out_len, int iters, float ms_phase[4], int* used_pipeline)
{
    if (!ms_phase || !used_pipeline || iters < 1) return TX_ERR_INVALID;
    size_t in_bytes = 0;
    int rc = check_compress(format, width, height, params, out_len, &in_bytes);
    if (rc != TX_OK) return rc;
    if (!d_rgba || !d_output) return TX_ERR_INVALID;
    txc::DeviceContext* ctx = txc::current_context(&rc);
    if (!ctx) return rc;
    hipEvent_t ev[5] = {};
    for (int i = 0; i < 5 && rc == TX_OK; ++i)
        if (hipEventCreate(&ev[i]) != hipSuccess) rc = TX_ERR_HIP;
    for (int k = 0; k < 4; ++k) ms_phase[k] = 0.0f;
    const txk::EncodeArgs a = encode_args(format, params, d_rgba, width, height, d_output, out_len);
    for (int it = 0; it < iters && rc == TX_OK; ++it) {
        bool pipe = false;
        if (encode_on(ctx, a, ctx->stream, nullptr, ev, &pipe) != hipSuccess) rc = TX_ERR_HIP;
        *used_pipeline = pipe ? 1 : 0;
        if (rc != TX_OK || !pipe) break;
        if (hipEventSynchronize(ev[4]) != hipSuccess) rc = TX_ERR_HIP;
        for (int k = 0; k < 4 && rc == TX_OK; ++k) {
            float ms = 0.0f;
            if (hipEventElapsedTime(&ms, ev[k], ev[k + 1]) != hipSuccess) rc = TX_ERR_HIP;
            ms_phase[k] += ms;
        }
    }
    if (rc == TX_OK && hipStreamSynchronize(ctx->stream) != hipSuccess) rc = TX_ERR_HIP;
    for (int i = 0; i < 5; ++i)
        if (ev[i]) (void)hipEventDestroy(ev[i]);
    return rc;
}

int tx_decompress_block(int format, const uint8_t* block, size_t block_len, uint8_t rgba_out[64])
{
    if (!valid_format(format)) return TX_ERR_FORMAT;
    if (block_len < tx_block_size(format)) return TX_ERR_INPUT_SHORT;
    return tx_decompress(format, block, tx_block_size(format), 4, 4, rgba_out, 64);
}

}  // extern "C"
