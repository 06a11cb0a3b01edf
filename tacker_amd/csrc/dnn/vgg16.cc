#include "vgg16.h"

#include <cmath>
#include <mutex>
#include <stdexcept>
#include <unordered_map>

#include "../Creator.h"
#include "../Logger.h"
#include "direct.h"
#include "../rng.h"

extern Logger logger;
extern std::unordered_map<std::string, void *> fmap;

namespace {

int pad128(int x) { return ((x + 127) / 128) * 128; }

void launch1d(const char *key, long work, void **args, cudaStream_t stream)
{
    long blocks = (work + 255) / 256;
    const long cap = (long)cuCount() * 8;
    if (blocks > cap) blocks = cap;
    if (blocks < 1) blocks = 1;
    TK_SAFE_CALL(tkLaunchKernel(fmap.at(key), dim3((unsigned)blocks).raw(), dim3(256).raw(), args, 0, stream));
}

// A task's device buffers, given back together.  The small ones -- four in five -- lie in slabs: tkFree waits for the device and
// unmaps, 50 to 350 us a call, which made a task of one allocation a buffer 8 ms to give back.
class Buffers {
public:
    ~Buffers()
    {
        for (void *p : slabs_) tkErrCheck(tkFree(p));
    }
    void *get(size_t bytes)
    {
        bytes = (bytes + 255) / 256 * 256;
        void *p = nullptr;
        if (bytes > left_) {
            const bool own = bytes > SLAB / 2;
            TK_SAFE_CALL(tkMalloc(&p, own ? bytes : SLAB));
            slabs_.push_back(p);
            if (own) return p;
            next_ = (char *)p;
            left_ = SLAB;
        }
        p = next_;
        next_ += bytes;
        left_ -= bytes;
        return p;
    }

private:
    static constexpr size_t SLAB = (size_t)64 << 20;
    std::vector<void *> slabs_;
    char *next_ = nullptr;
    size_t left_ = 0;
};

void *zeroed(Buffers &buffers, size_t bytes)
{
    void *p = buffers.get(bytes);
    TK_SAFE_CALL(tkMemset(p, 0, bytes));
    return p;
}
float *devAlloc(Buffers &buffers, size_t floats) { return (float *)zeroed(buffers, floats * sizeof(float)); }

// f16 [rows_pad][cols_pad] with uniform[-1,1]*scale in the top-left rows x cols, zero elsewhere
void *randomHalfMatrix(Buffers &buffers, tk::Rng &rng, int rows, int cols, int rows_pad,
                       int cols_pad, float scale)
{
    std::vector<uint16_t> host((size_t)rows_pad * cols_pad, 0);
    for (int r = 0; r < rows; ++r)
        for (int c = 0; c < cols; ++c)
            host[(size_t)r * cols_pad + c] = tk::float_to_half_bits(rng.uniform(-1.0f, 1.0f) * scale);
    void *p = buffers.get(host.size() * 2);
    TK_SAFE_CALL(tkMemcpy(p, host.data(), host.size() * 2, TK_MEMCPY_H2D));
    return p;
}

float *randomBias(Buffers &buffers, tk::Rng &rng, int n, int n_pad)
{
    std::vector<float> host(n_pad, 0.0f);
    for (int i = 0; i < n; ++i) host[i] = rng.uniform(-0.1f, 0.1f);
    float *p = devAlloc(buffers, n_pad);
    TK_SAFE_CALL(tkMemcpy(p, host.data(), (size_t)n_pad * sizeof(float), TK_MEMCPY_H2D));
    return p;
}

// The direct kernels (kernels/dnn_direct.hip) run a layer that has its launch to itself; a device layer without them
// runs every layer through its operand builder and tzgemm, as a layer fused with a best-effort kernel always does.
bool haveDirectKernels() { return fmap.count("conv3x3_image") != 0; }

// The weights [rows][K] once more, in the order the direct kernels read them.
void *weightFragments(Buffers &buffers, void *weights, int rows, int K)
{
    if (!haveDirectKernels()) return nullptr;
    void *p = buffers.get((size_t)rows * K * 2);
    void *args[] = {&weights, &p, &rows, &K};
    launch1d("pack_weight_fragments", (long)rows * K / 8, args, nullptr);
    return p;
}

// How tzgemm cuts the reduction of a (padded) GEMM: the segments' number -- 4 per part (tz_use_ksplit), or 1 -- and the
// 64-k chunk each begins with.  Chunks from `real` on are padding: zeros, which nobody needs to add.
int reductionCut(int M, int N, int K, int real, int begin[DNN_MAX_SEGMENTS + 1])
{
    const int chunks = K / TZ_BLOCK_K;
    if (!tz_use_ksplit(M, N, K)) {
        begin[0] = 0;
        begin[1] = std::min(real, chunks);
        return 1;
    }
    const int parts = tz_ksplit_parts(M, N, K), segments = 4 * parts;
    static_assert(4 * TZ_KSPLIT_MAX_PARTS <= DNN_MAX_SEGMENTS, "the table holds every cut");
    for (int i = 0; i <= segments; ++i) {   // as tzgemm_role_ksplit
        const int part = i / 4, first = part * chunks / parts, count = (part + 1) * chunks / parts - first;
        begin[i] = std::min(real, first + (i % 4) * count / 4);
    }
    begin[segments] = std::min(real, chunks);
    return segments;
}

// d -> what dnn_div takes for a division by d
unsigned reciprocal(int d) { return d == 1 ? 0u : (unsigned)((1ull << 32) / (unsigned)d + 1); }

// Whether the activation that a layer's direct kernel leaves for the next layer is what the layer's raw output and bias
// give.  A layer that ran fused, or not through its direct kernel, has written only the raw output; and a caller who has
// the raw output's or the bias's address may write there between two layers that are launched one by one.
struct Fresh {
    bool valid = false, exposed = false;
    const bool *wholeQuery = nullptr;   // the layers follow each other, nobody writes in between
    bool holds() const { return valid && (!exposed || *wholeQuery); }
};

// A layer's activation as the next layer's direct kernel reads it.
struct Activation {
    DnnOutput out{};
    int channels = 0;
    Fresh fresh;
    // bring it up to date, if it is not
    void need(cudaStream_t stream)
    {
        if (fresh.holds()) return;
        const int pixels = out.pool ? out.H * out.W / 4 : out.H * out.W;
        void *args[] = {&out, &channels};
        launch1d("dnn_activation", (long)pixels * (channels / 4), args, stream);
        fresh.valid = true;
    }
};

// Shared GEMM machinery of conv and FC layers: persistent objects built once.
class GemmLayer : public LcGemmKernel {
public:
    // tile_end > 0: only the reference tiles [0, tile_end) are computed (the others would be padding)
    GemmLayer(VGG16 &task, int id, const std::string &name, int M, int N, int K, const void *A, const void *B, float *C,
              int tile_end = 0)
        : task_(task), M_(M), N_(N), K_(K)
    {
        this->Id = id;
        this->kernelName = name;
        ori_.reset(new OriTZGEMMKernel(id, M, N, K, A, B, C));
        tiles_ = tile_end > 0 ? tile_end : getTZGEMMGridDim(M, N, K)[3];
        gptb_.reset(new GPTBKernel(id, "tzgemm", "gptb_tzgemm", ori_.get(), dim3(cuCount(), 1, 1),
                                   dim3(TZ_THREADS, 1, 1), 0, tiles_));
    }
    std::vector<int> gemmDims() const override { return {M_, N_, K_}; }
    // somebody may write the weights from now on, of which a direct kernel reads a copy: tzgemm reads them as they are
    virtual void weightsHandedOut() {}

protected:
    virtual void before(cudaStream_t stream) = 0;   // operand staging (im2col / pack)
    virtual void fused() {}                         // tzgemm runs the layer: its raw output is all this launch writes
    virtual void run(cudaStream_t stream)
    {
        before(stream);
        gptb_->execute(stream);
    }
    void executeImpl(cudaStream_t stream) final
    {
        task_.layerByItself(stream);
        run(stream);
    }

public:
    void executeMixed(GPTBKernel *be, int be_start, int be_end, cudaStream_t stream,
                      const std::string &variant = "") override
    {
        if (be_end <= be_start) {
            executeImpl(stream);
            return;
        }
        task_.layerByItself(stream);
        before(stream);
        fused();
        std::unique_ptr<MixKernel> mix(createTzgemmMix(be, gptb_.get(), be_start, be_end, 0, tiles_, variant, 0, 0));
        mix->execute(stream);
    }

protected:
    VGG16 &task_;
    int M_, N_, K_, tiles_;
    std::unique_ptr<OriTZGEMMKernel> ori_;
    std::unique_ptr<GPTBKernel> gptb_;
};

class ConvKernel : public GemmLayer {
public:
    // act_bias != nullptr: act is the raw output of the previous convolution; its bias and
    // ReLU are applied while the operand is gathered.  pooled: act is that output at twice the
    // height and width, and the 2x2 max pooling between the two layers happens on the way in too.
    ConvKernel(VGG16 &task, int id, const std::string &name, const float *act, const float *act_bias, bool pooled, int H,
               int W, int C, int c_stride, int Cout, void *A, const void *Wt, float *out)
        : GemmLayer(task, id, name, pad128(H * W), pad128(Cout), pad128(9 * C), A, Wt, out), act_(act),
          act_bias_(act_bias), pool_(pooled ? 1 : 0), H_(H), W_(W), C_(C), cs_(c_stride), Cout_(Cout), A_(A)
    {
        this->mixable = 2;
        if (pooled && !(C % 8 == 0 && c_stride % 4 == 0))
            logger.ERROR("vgg16: a pooled input needs a channel count that is a multiple of 8");
    }
    // {n,c,h,w, k,c,kh,kw, pad,pad, stride,stride, dil,dil}
    std::vector<int> getArgs() override { return {1, C_, H_, W_, Cout_, C_, 3, 3, 1, 1, 1, 1, 1, 1}; }

    // Run through the direct kernel from now on: `in` (null: the layer reads the image) to `out`, weights as
    // fragments.  A workgroup's output channels are as many as still leave a workgroup for three CUs in four -- every
    // workgroup reads its tile's input and its channels' weights once, so larger ones read less -- and, where tzgemm cuts
    // the reduction, as many as 16 wavefronts serve with a segment each; a wavefront takes two 16-channel slices
    // where 8 are left.  Segments that are too many for that are taken a part (four of them) a wavefront.
    void useDirect(Activation *in, Activation *out, const void *fragments)
    {
        in_ = in;
        next_ = out;
        direct_.reset(new DnnConv{});
        DnnConv &d = *direct_;
        d.act = in ? in->out.act : nullptr;
        d.weights = fragments;
        d.out = out->out;
        d.C = C_;
        d.chunks = K_ / TZ_BLOCK_K;
        d.tiles_x = (W_ + DNN_TILE - 1) / DNN_TILE;
        d.tiles = d.tiles_x * ((H_ + DNN_TILE - 1) / DNN_TILE);
        d.per_group = reciprocal(d.tiles);
        d.per_row = reciprocal(d.tiles_x);
        int ct = 8, &slices = slices_;
        bool &part = part_, &low = low_;
        if (in) {
            const int segments = reductionCut(M_, N_, K_, 9 * C_ / TZ_BLOCK_K, d.segment_begin);
            while (ct > 1 && (Cout_ % (16 * ct) != 0 || (segments > 1 && ct * segments > 16) ||
                              (long)d.tiles * (Cout_ / (16 * ct)) * 4 < (long)cuCount() * 3))
                ct /= 2;
            part = segments > 16;
            // More workgroups than CUs, but not twice as many, leave a few CUs with two in turn: as half as many with twice the channels
            // every CU has one.  us of the layers before and after: conv4_2 at 320 x 416 (280 workgroups -> 140) 27.5 / 20.5, at
            // 160 x 416 (336) 13.8 / 9.8, conv3_2 at 192 x 192 (288) 10.3 / 8.0, at 224 x 192 (336) 11.1 / 8.3, at 160 x 128 (320) 8.8 / 8.4, at
            // 224 x 416 (364) 13.2 / 12.9, conv1_2 with the first layer in it at 96 x 96 10.0 / 8.0.
            // Where 16 wavefronts cannot take a segment each any more, each takes a part, if a workgroup had 16 channels only: conv4_2
            // at 160 x 160 (288) 11.4 / 9.1, at 128 x 288 (320) 11.1 / 10.9, at 224 x 160 (384) 10.6 / 10.7 and conv4_3 there 11.1 / 10.9, at
            // 96 x 416 (448) 11.1 / 10.9, conv5_1 at 288 x 416 (384) 11.9 / 9.2.  Of two slices of eight segments and of four of four it makes
            // eight longer wavefronts out of 16 and loses: conv4_2 at 224 x 288 (320) 13.0 / 14.0, at 160 x 352 (288) 12.5 / 13.9, at
            // 352 x 352 (288) 19.3 / 22.7.
            const long workgroups = (long)d.tiles * (Cout_ / (16 * ct));
            if (!part && workgroups > cuCount() && workgroups < 2L * cuCount() && ct < 8 && Cout_ % (32 * ct) == 0) {
                if (segments == 1 || 2 * ct * segments <= 16) {
                    ct *= 2;
                } else if (ct == 1 && C_ > 64) {   // (C = 64: the form that takes the first layer)
                    ct *= 2;
                    part = true;
                }
            }
            slices = !part && ct % 2 == 0 && ct / 2 * segments >= 8 ? 2 : 1;
            d.runs = part ? segments / 4 : segments;
            // Tiles of four rows where an image has no more, and where those of eight make workgroups for half of the CUs or
            // fewer: us with tiles of eight and four rows, conv5_1 at 224 x 224 (128 workgroups of 8 x 8) 8.0 / 6.7, conv4_2 at
            // 64 x 96 (64) 9.0 / 7.3, conv3_2 there (96) 6.2 / 5.2.
            low = slices == 1 && (H_ <= DNN_TILE / 2 || (ct == 1 && 2L * d.tiles * (Cout_ / 16) <= cuCount()));
            if (low) {
                d.tiles = d.tiles_x * ((H_ + DNN_TILE / 2 - 1) / (DNN_TILE / 2));
                d.per_group = reciprocal(d.tiles);
            }
            key_ = std::string("conv3x3_direct_") + (slices == 2 ? "2" : "1") + (part ? "_1" : "_0") + (low ? "_low" : "");
            lds_ = std::max((size_t)(C_ / 64) * DNN_PLANE_BYTES, (size_t)ct * d.runs * DNN_PARTIAL_BYTES);
        } else {
            ct = Cout_ / 16;
            d.runs = 1;
            key_ = "conv3x3_image";
        }
        d.ct_count = ct;
        d.workgroups = d.tiles * (Cout_ / (16 * ct));
        threads_ = in ? 64u * (unsigned)(ct / slices * d.runs) : 256u;
        grid_ = (unsigned)(d.workgroups + TK_XCD_NUM - 1) / TK_XCD_NUM * TK_XCD_NUM;
    }

    void weightsHandedOut() override { direct_.reset(); }
    bool direct() const { return direct_ != nullptr; }
    // As part of a whole query.  raw: the output is written beside the activation.  image, keep: of the first layer, read
    // from `image` and stored where the layer has it as a rule.
    void executeInQuery(const float *image, float *keep, bool raw, cudaStream_t stream) { launchDirect(image, keep, raw, stream); }
    // Whether the second layer can compute the first one's activation for itself: where a wavefront of it serves one slice of
    // channels over segments of their own, the form its kernel for that has.  That is so at all sizes on 256 CUs: a reduction that
    // is cut is one of at most 128 pixel tiles, too few for a workgroup to take the four slices that make two a wavefront.  On
    // fewer CUs it may not be, and the first layer then has its launch.
    bool takesFirstLayer() const { return direct_ && slices_ == 1 && !part_ && threads_ <= 512; }
    // ... and both of them, the second as part of a whole query without its raw output
    void executeWithFirst(const ConvKernel &first, const float *image, float *keep, cudaStream_t stream)
    {
        DnnImage i{image, keep, first.direct_->weights, first.direct_->out.bias, first.direct_->chunks, (int)lds_};
        DnnConv c = *direct_;
        c.out.raw = nullptr;
        void *args[] = {&i, &c};
        const char *key = low_ ? "conv3x3_direct_image_low" : "conv3x3_direct_image";
        TK_SAFE_CALL(tkLaunchKernel(fmap.at(key), dim3(grid_).raw(), dim3(threads_).raw(), args, lds_ + DNN_IMAGE_BYTES, stream));
        first.next_->fresh.valid = false;
        next_->fresh.valid = true;
    }

protected:
    void fused() override
    {
        if (next_) next_->fresh.valid = false;
    }
    void run(cudaStream_t stream) override
    {
        if (!direct_) {
            fused();
            return GemmLayer::run(stream);
        }
        if (in_) in_->need(stream);
        launchDirect(act_, nullptr, true, stream);
    }
    void launchDirect(const float *image, float *keep, bool raw, cudaStream_t stream)
    {
        DnnConv c = *direct_;
        if (!raw) c.out.raw = nullptr;
        void *image_args[] = {&image, &keep, &c}, *act_args[] = {&c};
        void **args = in_ ? act_args : image_args;
        TK_SAFE_CALL(tkLaunchKernel(fmap.at(key_), dim3(grid_).raw(), dim3(threads_).raw(), args, lds_, stream));
        next_->fresh.valid = true;
    }
    void before(cudaStream_t stream) override
    {
        int KH = 3, KW = 3, pad = 1, stride = 1, Ho = H_, Wo = W_, Kp = K_;
        int relu = 1;
        if (C_ % 8 == 0 && cs_ % 4 == 0) {   // every layer but the first: each activation read once
            void *args[] = {&act_, &H_, &W_, &C_, &cs_, &A_, &Kp, &act_bias_, &relu, &pool_};
            launch1d("im2col3x3_scatter_nhwc_f16", (long)H_ * W_ * (C_ / 8), args, stream);
            return;
        }
        // the first layer (3 channels): an operand buffer of its own, zeroed once, of which only the
        // columns that hold data are rewritten
        int Kw = (9 * C_ + 7) / 8 * 8;
        void *args[] = {&act_, &H_, &W_, &C_, &cs_, &KH, &KW, &pad, &stride, &Ho, &Wo, &A_, &Kp, &act_bias_, &relu, &Kw};
        launch1d("im2col_nhwc_f16", (long)Ho * Wo * Kw, args, stream);
    }

private:
    const float *act_;
    const float *act_bias_;
    int pool_;
    int H_, W_, C_, cs_, Cout_;
    void *A_;
    std::unique_ptr<DnnConv> direct_;
    Activation *in_ = nullptr, *next_ = nullptr;
    std::string key_;
    int slices_ = 1;                     // of 16 channels a wavefront takes
    bool part_ = false, low_ = false;    // ... over a whole part of the reduction; tiles of four rows
    unsigned grid_ = 0, threads_ = 0;
    size_t lds_ = 0;
};

class FcKernel : public GemmLayer {
public:
    // C[128][out_pad] = X[128][K] * W[out_pad][K]^T with the batch-1 activation in row 0 of X, taken
    // from src with stride src_stride.  The activation is the M side so that the reference tiles that
    // hold the result, row 0 .. 63 of C, are the first out_pad / 64 of the tile order: only those are
    // launched, every one of them streams weights nobody else reads, and rows 64 .. 127 of C (all
    // padding) stay as allocated.
    // pool_W > 0: src is the raw output of the last convolution, [.][pool_W][pool_ld] with pool_C
    // channels, and the 2x2 max pooling in front of the classifier happens while the row is packed
    FcKernel(VGG16 &task, int id, const std::string &name, const float *src, long src_stride, const float *src_bias,
             int src_relu, int in_features, int out_features, const void *Wt, void *X, float *out,
             int pool_W = 0, int pool_ld = 0, int pool_C = 0)
        : GemmLayer(task, id, name, 128, pad128(out_features), pad128(in_features), X, Wt, out,
                    pad128(out_features) / TZ_REF_TILE),
          src_(src), stride_(src_stride), bias_(src_bias), relu_(src_relu), in_(in_features), out_(out_features),
          X_(X), poolW_(pool_W), poolLd_(pool_ld), poolC_(pool_C)
    {
        this->mixable = 1;
    }
    std::vector<int> getArgs() override { return {M_, N_, K_}; }

    // Run through the direct kernel from now on.  in, out: whether X's first row, and the next layer's (next_x), hold
    // this layer's input and activation (out null: the last layer).
    void useDirect(Fresh *in, Fresh *out, const void *fragments, float *raw, const float *bias, void *next_x)
    {
        inFresh_ = in;
        outFresh_ = out;
        direct_.reset(new DnnFc{});
        direct_->x = X_;
        direct_->weights = fragments;
        direct_->raw = raw;
        direct_->bias = bias;
        direct_->act = next_x;
        direct_->chunks = K_ / TZ_BLOCK_K;
        direct_->segments = reductionCut(M_, N_, K_, direct_->chunks, direct_->segment_begin);
        perWave_ = direct_->segments > 16 ? 2 : 1;
    }
    void weightsHandedOut() override { direct_.reset(); }

protected:
    void fused() override
    {
        if (inFresh_) inFresh_->valid = true;   // before() packed it
        if (outFresh_) outFresh_->valid = false;
    }
    void run(cudaStream_t stream) override
    {
        if (!direct_) {
            fused();
            return GemmLayer::run(stream);
        }
        if (!inFresh_->holds()) before(stream);
        inFresh_->valid = true;
        void *args[] = {direct_.get()};
        const int waves = (direct_->segments + perWave_ - 1) / perWave_;
        TK_SAFE_CALL(tkLaunchKernel(fmap.at(perWave_ == 2 ? "fc_direct_2" : "fc_direct_1"), dim3((unsigned)(N_ / 16)).raw(),
                                    dim3((unsigned)(64 * waves)).raw(), args, 0, stream));
        if (outFresh_) outFresh_->valid = true;
    }
    void before(cudaStream_t stream) override
    {
        if (poolW_ > 0) {
            void *args[] = {&src_, &poolW_, &poolLd_, &poolC_, &bias_, &relu_, &in_, &X_};
            launch1d("pack_fc_input_pooled", in_, args, stream);
            return;
        }
        void *args[] = {&src_, &stride_, &bias_, &relu_, &in_, &X_};
        launch1d("pack_fc_input", in_, args, stream);
    }

private:
    const float *src_;
    long stride_;
    const float *bias_;
    int relu_, in_, out_;
    void *X_;
    int poolW_, poolLd_, poolC_;
    std::unique_ptr<DnnFc> direct_;
    Fresh *inFresh_ = nullptr, *outFresh_ = nullptr;
    int perWave_ = 1;
};

// The stream images are staged on, one for all tasks, given back with the last of them.  (A stream for each task would
// soon share its hardware queue with the streams the queries run on.)
struct StagingStream {
    cudaStream_t stream = nullptr;
    StagingStream() { TK_SAFE_CALL(tkStreamCreateNonBlocking(&stream)); }
    ~StagingStream() { tkErrCheck(tkStreamDestroy(stream)); }
};
std::shared_ptr<StagingStream> stagingStream()
{
    static std::mutex lock;
    static std::weak_ptr<StagingStream> shared;
    std::lock_guard<std::mutex> held(lock);
    auto s = shared.lock();
    if (!s) shared = s = std::make_shared<StagingStream>();
    return s;
}

}  // namespace

namespace { constexpr size_t CONVOLUTIONS = 13; }

struct VGG16::Impl {
    Buffers buffers;
    bool direct = false;            // layers run through the direct kernels
    float *hostInput = nullptr;     // page-locked
    size_t pixels = 0;              // floats of it
    // executeQuery: two device images taken in turn, and an event behind the last query of each turn
    std::shared_ptr<StagingStream> staging;
    float *image[2] = {};
    tkEvent_t over[2] = {};
    int turn = 0;
    cudaStream_t lastStream = nullptr;   // the last query's
    tkEvent_t before = nullptr;          // recorded on the null stream for a query to wait for
    bool stepped = false;                // since the last whole query the task has been used otherwise
    bool watched = false;                // no query leaves anything out: somebody has an address of a raw output, a bias or weights, or has
                                         // recorded a launch that has, or something was left out that somebody needed
    bool lean = false;                   // the last query has left out the raw outputs ...
    int leanTurn = 0;                    // ... and read this image
    ~Impl()
    {
        for (tkEvent_t e : {over[0], over[1], before})
            if (e) tkErrCheck(tkEventDestroy(e));
        if (hostInput) tkErrCheck(tkHostFree(hostInput));
    }
    float *input = nullptr;
    std::vector<VGG16::Act> convOut;   // the 13 convolutions, then the 3 fully connected layers
    float *logits = nullptr;
    long logitsStride = 0;
    Activation act[13];             // of the convolutions; the last one's is fc1's input
    Fresh fcInput[3];               // fc2's and fc3's input vectors hold the layer before's activation ([0] unused: act[12])
};

VGG16::VGG16(int taskId, const VGG16Options &o) : Task(taskId, "vgg16"), opt(o), impl(new Impl)
{
    taskType = LC;
    if (opt.height % 32 || opt.width % 32) logger.ERROR("vgg16: input resolution must be a multiple of 32");
    tk::Rng rng(opt.seed);
    auto &fl = impl->buffers;

    int H = opt.height, W = opt.width, C = 3, ld = 3;
    impl->pixels = (size_t)H * W * 3;
    TK_SAFE_CALL(tkHostMalloc((void **)&impl->hostInput, impl->pixels * sizeof(float)));
    for (size_t i = 0; i < impl->pixels; ++i) impl->hostInput[i] = rng.uniform();
    impl->input = devAlloc(fl, impl->pixels);
    InputHost[0] = impl->hostInput;
    Input[0] = impl->input;
    InputSize[0] = (int)(impl->pixels * sizeof(float));
    // A larger image's tile numbers times its tiles pass 2^32, where dnn_div's reciprocals stop being exact; it runs
    // through the operand builders and tzgemm.
    const bool direct = impl->direct = haveDirectKernels() && (long)H * W <= 2048L * 2048;
    if (direct) {
        impl->staging = stagingStream();
        for (float *&image : impl->image) image = devAlloc(fl, impl->pixels);
    }
    TK_SAFE_CALL(tkEventCreate(&impl->before));
    for (tkEvent_t &e : impl->over) {
        TK_SAFE_CALL(tkEventCreate(&e));
        TK_SAFE_CALL(tkEventRecord(e, nullptr));   // nothing to wait for yet
    }

    // the largest im2col operand of the network, shared by every conv layer
    size_t maxA = 0;
    {
        int h = H, w = W, c = 3;
        const int plan[] = {64, 64, -1, 128, 128, -1, 256, 256, 256, -1, 512, 512, 512, -1, 512, 512, 512, -1};
        for (int p : plan) {
            if (p < 0) { h /= 2; w /= 2; continue; }
            maxA = std::max(maxA, (size_t)pad128(h * w) * pad128(9 * c));
            c = p;
        }
    }
    void *Abuf = zeroed(fl, maxA * 2);

    void *X1 = nullptr, *X2 = nullptr, *X3 = nullptr;   // the fully connected layers' operands
    auto halfBuf = [&](void **p, size_t n) { *p = zeroed(fl, n * 2); };

    // A convolution leaves 1.1 * A * B^T in its output buffer; bias and ReLU are applied by
    // whatever reads that buffer next (the next layer's operand gather, or the pooling).
    const float *act = impl->input;
    const float *act_bias = nullptr;   // bias the reader of act still has to apply
    int id = 100;
    const int plan[] = {64, 64, -1, 128, 128, -1, 256, 256, 256, -1, 512, 512, 512, -1, 512, 512, 512, -1};
    // A pooling layer is not a kernel either: the next convolution's operand, or the classifier's
    // input row, is built from the 2x2 maxima.
    bool pooled = false;
    int unpooled_W = 0;   // width of the raw convolution output a pending pooling reads
    int block = 1, layer = 1;
    const int n_plan = (int)(sizeof(plan) / sizeof(plan[0]));
    for (int step = 0; step < n_plan; ++step) {
        const int p = plan[step];
        if (p < 0) {
            pooled = true;
            unpooled_W = W;
            H /= 2;
            W /= 2;
            block++;
            layer = 1;
            continue;
        }
        const int Cout = p, Np = pad128(Cout), Kp = pad128(9 * C);
        const std::string name = "conv" + std::to_string(block) + "_" + std::to_string(layer++);
        void *Wt = randomHalfMatrix(fl, rng, Cout, 9 * C, Np, Kp, std::sqrt(2.0f / (9 * C)));
        float *bias = randomBias(fl, rng, Cout, Np);
        float *out = devAlloc(fl, (size_t)pad128(H * W) * Np);
        void *operand = Abuf;
        if (C % 8 != 0)   // gathered, and only its data columns rewritten: needs zeros nobody else disturbs
            operand = zeroed(fl, (size_t)pad128(H * W) * Kp * 2);
        auto *conv = new ConvKernel(*this, id++, "Convolution_" + name, act, act_bias, pooled, H, W, C, ld, Cout, operand, Wt, out);
        addKernel(conv);
        if (direct) {
            // what the next layer reads: this layer's activation, pooled if a pooling follows, in a frame of
            // zeros -- or, behind the last convolution, the classifier's input row
            const int i = (int)impl->convOut.size();
            Activation &a = impl->act[i];
            a.channels = Cout;
            a.out = DnnOutput{out, bias, nullptr, H, W, Np, 0, Cout, 0, plan[step + 1] < 0 ? 1 : 0};
            const int ho = a.out.pool ? H / 2 : H, wo = a.out.pool ? W / 2 : W;
            if (i < 12) {
                a.out.border = 1;
                a.out.act_pitch = wo + 2;
                halfBuf(&a.out.act, (size_t)(ho + 2) * (wo + 2) * Cout);
            } else {
                a.out.act_pitch = wo;
                halfBuf(&X1, (size_t)128 * pad128(ho * wo * Cout));
                a.out.act = X1;
            }
            conv->useDirect(i == 0 ? nullptr : &impl->act[i - 1], &a, weightFragments(fl, Wt, Np, Kp));
        }
        pooled = false;
        impl->convOut.push_back(Act{out, H, W, Cout, Np, Wt, bias, Np, Kp});
        act = out;
        act_bias = bias;
        C = Cout;
        ld = Np;
    }
    // classifier: 512*(H/32)*(W/32) -> 4096 -> 4096 -> classes; activations travel as
    // row 0 of the previous FC output, bias+ReLU applied while packing the next input
    const int feat = H * W * C;   // NHWC flatten (ld == C == 512 here)
    if (!X1) halfBuf(&X1, (size_t)128 * pad128(feat));
    halfBuf(&X2, (size_t)128 * 4096);
    halfBuf(&X3, (size_t)128 * 4096);
    void *W1 = randomHalfMatrix(fl, rng, 4096, feat, 4096, pad128(feat), std::sqrt(2.0f / feat));
    void *W2 = randomHalfMatrix(fl, rng, 4096, 4096, 4096, 4096, std::sqrt(2.0f / 4096));
    void *W3 = randomHalfMatrix(fl, rng, opt.classes, 4096, pad128(opt.classes), 4096, std::sqrt(2.0f / 4096));
    float *b1 = randomBias(fl, rng, 4096, 4096), *b2 = randomBias(fl, rng, 4096, 4096);
    float *o1 = devAlloc(fl, (size_t)128 * 4096), *o2 = devAlloc(fl, (size_t)128 * 4096);
    float *o3 = devAlloc(fl, (size_t)128 * pad128(opt.classes));
    // act is conv5_3's raw output; its pooling, bias and ReLU happen while fc1's input is packed
    auto *fc1 = new FcKernel(*this, id++, "Dot_fc1", act, 1, act_bias, 1, feat, 4096, W1, X1, o1, pooled ? unpooled_W : 0, ld, C);
    auto *fc2 = new FcKernel(*this, id++, "Dot_fc2", o1, 1, b1, 1, 4096, 4096, W2, X2, o2);
    auto *fc3 = new FcKernel(*this, id++, "Dot_fc3", o2, 1, b2, 1, 4096, opt.classes, W3, X3, o3);
    for (auto *fc : {fc1, fc2, fc3}) addKernel(fc);
    if (direct) {
        for (auto &a : impl->act) a.fresh.wholeQuery = &wholeQuery;
        Fresh *fresh = impl->fcInput;
        fresh[1].wholeQuery = fresh[2].wholeQuery = &wholeQuery;
        fc1->useDirect(&impl->act[12].fresh, &fresh[1], weightFragments(fl, W1, 4096, pad128(feat)), o1, b1, X2);
        fc2->useDirect(&fresh[1], &fresh[2], weightFragments(fl, W2, 4096, 4096), o2, b2, X3);
        fc3->useDirect(&fresh[2], nullptr, weightFragments(fl, W3, pad128(opt.classes), 4096), o3, nullptr, nullptr);
        TK_SAFE_CALL(tkDeviceSynchronize());   // the fragments are laid out before a kernel on any stream reads them
    }
    impl->convOut.push_back(Act{o1, 1, 1, 4096, 4096, W1, b1, 4096, pad128(feat)});
    impl->convOut.push_back(Act{o2, 1, 1, 4096, 4096, W2, b2, 4096, 4096});
    impl->convOut.push_back(Act{o3, 1, 1, opt.classes, pad128(opt.classes), W3, nullptr, pad128(opt.classes), 4096});
    impl->logits = o3;
    impl->logitsStride = 1;
}

void VGG16::captured()
{
    for (auto &a : impl->act) a.fresh.valid = false;
    for (Fresh &f : impl->fcInput) f.valid = false;
}

// The image goes over PCIe while the query before is still running: on a stream of its own, into the device image which
// the query before that one has read.  The copy has ended when the first kernel is launched, so nothing on the device
// waits for it, and the host's image may change as soon as this returns.  A copy on the query's stream waits for
// the query before and leaves the GPU idle until the host has seen its end and launched again: 45 us of a 206 us query
// at 224 x 224, 37 of 133 at 64 x 96.
//
// All of a task's launches share its buffers, so a query comes after the last one, whichever stream that ran on, and after
// what the null stream and the streams ordered with it have in front of them (a reader of the logits on a second stream, a
// recorded graph, a bias written on the null stream) -- what a query whose image is copied on the null stream waits for.
//  * On the null stream its launches wait for all that by themselves.
//  * On a stream that is not ordered with it, the device waits for an event recorded there, which is over by the time the
//    image is in place where the null stream is idle: 0 to 1 us a query.
//  * On a stream that is, the host waits, after the image has been staged: 158 us a query at 224 x 224 where the null stream
//    takes 144.  An event there, behind the stream's own last query, took 315 where the null stream took 163.
// Graphs and single layers on a caller's stream that is not ordered with the null stream are the caller's to order
// with a query on another stream.
void VGG16::executeQuery(cudaStream_t stream)
{
    Impl &m = *impl;
    // The null stream by its other name, hipStreamLegacy: kernels and events take it, but a question about it
    // (its flags, whether it is recorded) is answered for the handles of streams that were created only.
    if (stream == reinterpret_cast<cudaStream_t>(1)) stream = nullptr;
    if (stream) {
        // The copy on the null stream refuses to run while the stream is recorded.  The staged one would pass in a relaxed
        // recording, and every launch of the graph would see the image of this moment.
        int capturing = 0;
        TK_SAFE_CALL(tkStreamIsCapturing(stream, &capturing));
        if (capturing) throw std::runtime_error("vgg16: a query copies its image and cannot be recorded; captureQuery records its kernels");
    }
    const int turn = m.turn;
    const tkEvent_t last = m.over[turn ^ 1];
    // what comes after this query waits for what there is of it
    const auto launched = [&]() {
        m.turn ^= 1;
        m.lastStream = stream;
        return tkEventRecord(m.over[turn], stream);
    };
    auto *first = m.direct ? dynamic_cast<ConvKernel *>(kernels.front()) : nullptr;
    if (!first || !first->direct()) {
        // the copy on the null stream waits for the streams ordered with it; for the others the host does
        TK_SAFE_CALL(tkEventSynchronize(last));
        if (stream) TK_SAFE_CALL(tkStreamSynchronize(stream));
        Task::executeQuery(stream);
    } else {
        unsigned ordered = 0;   // with the null stream
        if (stream) TK_SAFE_CALL(tkStreamIsBlocking(stream, &ordered));
        if (stream && !ordered) TK_SAFE_CALL(tkEventRecord(m.before, nullptr));
        TK_SAFE_CALL(tkEventSynchronize(m.over[turn]));   // which read this image
        // by the copy engine, 602 KB in 19 us; a kernel that reads the host's memory takes 23 and slows the one it runs beside
        TK_SAFE_CALL(tkMemcpyAsync(m.image[turn], m.hostInput, (size_t)InputSize[0], TK_MEMCPY_H2D, m.staging->stream));
        TK_SAFE_CALL(tkStreamSynchronize(m.staging->stream));
        if (ordered) TK_SAFE_CALL(tkStreamSynchronize(nullptr));
        else if (stream) TK_SAFE_CALL(tkStreamWaitEvent(stream, m.before));
        if (stream || m.lastStream) TK_SAFE_CALL(tkStreamWaitEvent(stream, last));
        const WholeQuery whole(*this);
        m.lean = !m.stepped && !m.watched;
        m.leanTurn = turn;
        try {
            size_t next = 1;
            auto *second = static_cast<ConvKernel *>(kernels[1]);
            if (m.lean && !opt.firstLayerApart && second->takesFirstLayer()) {
                second->executeWithFirst(*first, m.image[turn], m.input, stream);
                next = 2;
            } else {
                first->executeInQuery(m.image[turn], m.input, !m.lean, stream);
            }
            for (; m.lean && next < CONVOLUTIONS; ++next)
                static_cast<ConvKernel *>(kernels[next])->executeInQuery(nullptr, nullptr, false, stream);
            for (; next < kernels.size(); ++next) kernels[next]->execute(stream);
        } catch (...) {
            (void)launched();
            throw;
        }
    }
    TK_SAFE_CALL(launched());
    m.stepped = false;
}

// The queries' kernels read each other's activations, every layer's in a buffer of its own, so what a query left out can be
// had afterwards from what it kept: its image and the activations, which stay as they are until the next query.  On the
// staging stream, behind the query, and waited for: the caller's stream may be recording.
void VGG16::complete() const
{
    Impl &m = *impl;
    if (!m.lean) return;
    const cudaStream_t stream = m.staging->stream;
    TK_SAFE_CALL(tkStreamWaitEvent(stream, m.over[m.leanTurn]));
    for (size_t i = 0; i < CONVOLUTIONS; ++i)
        static_cast<ConvKernel *>(kernels[i])->executeInQuery(m.image[m.leanTurn], nullptr, true, stream);
    TK_SAFE_CALL(tkStreamSynchronizeBesideCapture(stream));
    m.lean = false;   // (and no sooner: where one of these fails, the next call tries again)
    m.watched = true;   // (a caller who does something else between queries does it again: this, 0.2 ms, once in a task's life)
}

void VGG16::layerByItself(cudaStream_t stream)
{
    if (wholeQuery) return;
    complete();
    impl->stepped = true;
    // A launch that is recorded reads the outputs of the layers before it whenever the caller replays it.  (The null stream cannot be
    // recorded, also not by its other name; a stream that gives no answer is taken to be.)
    int capturing = 1;
    if (!impl->watched && stream && stream != reinterpret_cast<cudaStream_t>(1) &&
        (tkStreamIsCapturing(stream, &capturing) || capturing))
        impl->watched = true;
}

// A recorded query writes every output whenever it is launched, behind no call of the task's.
void VGG16::recording()
{
    complete();
    impl->watched = true;
}

VGG16::~VGG16()
{
    for (auto *k : kernels) delete k;
}

void VGG16::initExecution()
{
    layerByItself(nullptr);
    // (the last query's first kernel, which may still wait on a stream that the copy is not ordered with, stores its own image there)
    TK_SAFE_CALL(tkEventSynchronize(impl->over[impl->turn ^ 1]));
    TK_SAFE_CALL(tkMemcpy(Input[0], InputHost[0], (size_t)InputSize[0], TK_MEMCPY_H2D));
}

const float *VGG16::logits(long *stride) const
{
    if (stride) *stride = impl->logitsStride;
    return impl->logits;
}

void VGG16::weightsHandedOut(int layer)
{
    this->layer(layer);
    static_cast<GemmLayer *>(kernels.at(layer))->weightsHandedOut();
}

void VGG16::resultHandedOut(int layer)
{
    this->layer(layer);
    if (layer < 13) impl->act[layer].fresh.exposed = true;
    else if (layer < 15) impl->fcInput[layer - 12].exposed = true;
}

bool VGG16::leavesOutputsOut() const { return impl->direct && !impl->watched && !impl->stepped; }

const VGG16::Act &VGG16::layer(int idx) const
{
    complete();
    impl->watched = true;
    return impl->convOut.at(idx);
}

VGG16::Act VGG16::activation(int conv_index)
{
    resultHandedOut(conv_index);
    weightsHandedOut(conv_index);
    return layer(conv_index);
}

Task *createTask(const std::string &model)
{
    if (model == "vgg16") return new VGG16(1);
    logger.ERROR("createTask: model not found: " + model);
}
