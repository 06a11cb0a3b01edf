// Checks of the C++ interface, the VGG16 task's and launch sizes of lbm: what no C entry point reaches.  Usage: task_checks <check>; exit code 0 if it holds.
#include <cstdio>
#include <cstring>
#include <exception>
#include <string>
#include <unordered_map>
#include <vector>

#include "Creator.h"
#include "dnn/vgg16.h"
#include "ori_kernel/lbm_kernel.h"
#include "../include/tacker_amd.h"

extern std::unordered_map<std::string, void *> fmap;

namespace {

std::vector<float> read(const float *p, size_t n)
{
    std::vector<float> host(n);
    TK_SAFE_CALL(tkDeviceSynchronize());
    TK_SAFE_CALL(tkMemcpy(host.data(), p, n * sizeof(float), TK_MEMCPY_D2H));
    return host;
}

void write(float *p, const std::vector<float> &host)
{
    TK_SAFE_CALL(tkMemcpy(p, host.data(), host.size() * sizeof(float), TK_MEMCPY_H2D));
    TK_SAFE_CALL(tkDeviceSynchronize());
}

bool same(const std::vector<float> &a, const std::vector<float> &b)
{
    return a.size() == b.size() && memcmp(a.data(), b.data(), a.size() * sizeof(float)) == 0;
}

size_t size_of(const VGG16::Act &a) { return (size_t)a.H * a.W * a.ld; }

// the same network (weights and image come from the seed) with every layer through its operand and tzgemm
void use_tzgemm(VGG16 &task)
{
    for (int i = 0; i < 16; ++i) task.weightsHandedOut(i);
}

// Layer `i` run by itself, its raw output or its bias written, layer i + 1 run by itself, twice: each run sees what was written last.
bool written_between_layers(bool accessor, bool bias)
{
    VGG16Options opt;
    opt.height = 64, opt.width = 96;
    for (int i : {0, 1, 5, 9, 12, 13, 14}) {
        VGG16 task(1, opt), plain(2, opt);
        use_tzgemm(plain);
        task.executeQuery(nullptr);
        plain.executeQuery(nullptr);
        std::vector<float> before = read(task.layer(i + 1).ptr, size_of(task.layer(i + 1)));
        float *raw = nullptr;
        int dims[4];
        if (accessor) raw = task.activation(i).ptr;
        else if (tacker_task_activation(static_cast<Task *>(&task), i, &raw, dims)) return false;
        if (raw != task.layer(i).ptr) return false;
        for (float factor : {0.5f, 3.0f}) {
            for (VGG16 *t : {&task, &plain}) {
                const VGG16::Act &a = t->layer(i);
                std::vector<float> v = bias ? read(a.bias, a.C) : read(a.ptr, size_of(a));
                for (float &x : v) x *= factor;
                write(bias ? a.bias : a.ptr, v);
                t->kernels[i + 1]->execute((cudaStream_t) nullptr);
            }
            const std::vector<float> got = read(task.layer(i + 1).ptr, size_of(task.layer(i + 1)));
            if (!same(got, read(plain.layer(i + 1).ptr, size_of(plain.layer(i + 1)))) || same(got, before)) {
                printf("layer %d, factor %g: not what was written\n", i, factor);
                return false;
            }
            before = got;
        }
    }
    return true;
}

// more classes than tzgemm cuts the last layer's reduction for
bool many_classes(int classes)
{
    VGG16Options opt;
    opt.height = opt.width = 32;
    opt.classes = classes;
    VGG16 task(1, opt), plain(2, opt);
    use_tzgemm(plain);
    task.executeQuery(nullptr);
    plain.executeQuery(nullptr);
    return same(read(task.logits(nullptr), classes), read(plain.logits(nullptr), classes));
}

void image(VGG16 &t, float factor)
{
    float *host = static_cast<float *>(t.InputHost[0]);
    for (size_t i = 0; i < t.InputSize[0] / sizeof(float); ++i) host[i] = factor * (float)((i * 2654435761u) % 1000) / 1000.0f;
}

// What a whole query after a whole query leaves out is there as soon as anybody can see it: every raw output, behind two queries
// of different images, as the layers through their operands and tzgemm leave it.  After the queries: nothing, another image staged, a
// layer run by itself, its addresses handed out before or between the queries.
bool raw_outputs_after_queries(int height, int width, bool apart = false)
{
    VGG16Options opt;
    opt.height = height, opt.width = width;
    opt.firstLayerApart = apart;
    enum { Nothing, Staged, Layer, Before, Between };
    for (int use : {Nothing, Staged, Layer, Before, Between}) {
        VGG16 task(1, opt), plain(2, opt);
        use_tzgemm(plain);
        if (use == Before) task.resultHandedOut(3);
        for (float factor : {1.0f, 0.5f, 0.75f}) {
            for (VGG16 *t : {&task, &plain}) {
                image(*t, factor);
                t->executeQuery(nullptr);
            }
            if (use == Between && factor == 0.5f) task.resultHandedOut(9);
        }
        if (use == Staged)
            for (VGG16 *t : {&task, &plain}) {
                image(*t, 0.25f);
                t->initExecution();
                t->kernels[0]->execute((cudaStream_t) nullptr);
            }
        if (use == Layer)
            for (int i : {7, 1, 0, 14, 12})
                for (VGG16 *t : {&task, &plain}) t->kernels[i]->execute((cudaStream_t) nullptr);
        for (int again = 0; again < 2; ++again) {
            for (int i = 0; i < 16; ++i) {
                const VGG16::Act &a = task.layer(i), &b = plain.layer(i);
                const size_t n = i < 13 ? size_of(a) : (size_t)a.C;
                if (!same(read(a.ptr, n), read(b.ptr, n))) {
                    printf("%d x %d, use %d, round %d: layer %d differs\n", height, width, use, again, i);
                    return false;
                }
            }
            for (VGG16 *t : {&task, &plain}) {   // from now on every query leaves them
                image(*t, 0.6f);
                t->executeQuery(nullptr);
            }
        }
    }
    return true;
}

bool same_outputs(const char *what, VGG16 &task, VGG16 &plain)
{
    for (int i = 0; i < 16; ++i) {
        const VGG16::Act &a = task.layer(i), &b = plain.layer(i);
        const size_t n = i < 13 ? size_of(a) : (size_t)a.C;
        if (!same(read(a.ptr, n), read(b.ptr, n))) {
            printf("%s: layer %d differs\n", what, i);
            return false;
        }
    }
    return true;
}

struct Stream {
    cudaStream_t s = nullptr;
    explicit Stream(bool blocking) { TK_SAFE_CALL(blocking ? tkStreamCreate(&s) : tkStreamCreateNonBlocking(&s)); }
    ~Stream() { tkErrCheck(tkStreamDestroy(s)); }
};

// A part of a query that a caller records -- layers 1 .. 15, or layer `fused` beside a best-effort kernel and those behind it
// -- on a new task, behind one query or behind two (which runs what they left out, while the stream is being recorded), and
// replays: straight away, or behind other queries.  It reads what the last query left.
bool recorded_part(int fused, bool others)
{
    VGG16Options opt;
    opt.height = 64, opt.width = 96;
    GPTBKernel *be = fused ? createKernel("stencil") : nullptr;
    const auto part = [&](VGG16 &t, cudaStream_t stream) {
        for (int i = fused ? fused : 1; i < 16; ++i) {
            auto *layer = static_cast<LcGemmKernel *>(t.kernels[i]);
            if (i == fused) layer->executeMixed(be, 0, 256, stream);
            else layer->execute(stream);
        }
    };
    for (int queries : {1, 2}) {
        VGG16 task(1, opt), plain(2, opt);
        for (int i = 0; i < 16; ++i) plain.resultHandedOut(i);   // its queries leave nothing out
        Stream stream(true);
        for (int q = 0; q < queries; ++q) task.executeQuery(nullptr);
        plain.executeQuery(nullptr);
        TK_SAFE_CALL(tkDeviceSynchronize());
        tkGraphExec_t graph = nullptr;
        TK_SAFE_CALL(tkStreamBeginCapture(stream.s));
        part(task, stream.s);
        TK_SAFE_CALL(tkStreamEndCapture(stream.s, &graph));
        bool ok = true;
        for (int replay = 0; replay < 4; ++replay) {
            if (others)
                for (VGG16 *t : {&task, &plain}) {
                    image(*t, 0.25f * (float)(4 - replay));
                    t->executeQuery(nullptr);
                }
            TK_SAFE_CALL(tkGraphLaunch(graph, stream.s));
            part(plain, nullptr);
            const size_t n = (size_t)opt.classes;
            if (!same(read(task.logits(nullptr), n), read(plain.logits(nullptr), n))) {
                printf("fused %d, recorded behind %d queries, replay %d: not its logits\n", fused, queries, replay);
                ok = false;
            }
        }
        ok = ok && same_outputs("recorded part", task, plain);
        TK_SAFE_CALL(tkGraphExecDestroy(graph));
        if (!ok) return false;
    }
    return true;
}

// A whole query recorded, before or behind queries; it is launched on an image that was written on the device, and what it leaves stays.
bool recorded_query(bool first)
{
    VGG16Options opt;
    opt.height = 64, opt.width = 96;
    VGG16 task(1, opt), plain(2, opt);
    use_tzgemm(plain);
    Stream stream(true);
    tkGraphExec_t graph = nullptr;
    if (first) graph = task.captureQuery(stream.s);
    for (float factor : {1.0f, 0.5f}) {
        image(task, factor);
        task.executeQuery(nullptr);
    }
    if (!first) graph = task.captureQuery(stream.s);
    image(plain, 0.75f);
    plain.executeQuery(nullptr);
    const float *host = static_cast<float *>(plain.InputHost[0]);
    write(static_cast<float *>(task.Input[0]), std::vector<float>(host, host + plain.InputSize[0] / sizeof(float)));
    TK_SAFE_CALL(tkGraphLaunch(graph, stream.s));
    TK_SAFE_CALL(tkDeviceSynchronize());
    const bool ok = same_outputs("recorded query", task, plain);
    TK_SAFE_CALL(tkGraphExecDestroy(graph));
    return ok;
}

// A task that somebody uses otherwise between its queries pays for what they left out once.
bool paid_once()
{
    VGG16Options opt;
    opt.height = opt.width = 32;
    enum { Look, Stage, Layer, Record };
    for (int use : {Look, Stage, Layer, Record}) {
        VGG16 task(1, opt);
        bool left = task.leavesOutputsOut();   // a new task's
        for (int round = 0; round < 2; ++round) {
            for (int q = 0; q < 3; ++q) task.executeQuery(nullptr);
            left = left && task.leavesOutputsOut() == (round == 0);
            if (use == Look) task.layer(2);
            if (use == Stage) task.initExecution();
            if (use == Layer) task.kernels[14]->execute((cudaStream_t) nullptr);
            if (use == Record) {
                Stream stream(false);
                TK_SAFE_CALL(tkGraphExecDestroy(task.captureQuery(stream.s)));
            }
        }
        if (!left || task.leavesOutputsOut()) {
            printf("use %d\n", use);
            return false;
        }
    }
    return true;
}

// every output of a query as the layers through their operands and tzgemm leave it
bool outputs(int height, int width)
{
    VGG16Options opt;
    opt.height = height, opt.width = width;
    VGG16 task(1, opt), plain(2, opt);
    use_tzgemm(plain);
    for (VGG16 *t : {&task, &plain}) t->executeQuery(nullptr);
    return same_outputs("a query", task, plain);
}

// Queries on a stream that is not ordered with the null stream, and straight behind the last one, while it is running: its outputs
// looked at, another image staged, a layer run by itself.
bool straight_behind_queries(int height, int width, int most)
{
    VGG16Options opt;
    opt.height = height, opt.width = width;
    VGG16 plain(2, opt);
    use_tzgemm(plain);
    enum { Look, Stage, Layer };
    for (bool watched : {false, true})
        for (int use : {Look, Stage, Layer})
            for (int queries = 1; queries <= most; ++queries) {
                VGG16 task(1, opt);
                if (watched) task.resultHandedOut(3);
                Stream stream(false);
                for (int q = 0; q < queries; ++q) {
                    image(task, 1.0f / (float)(1 + q));
                    task.executeQuery(stream.s);
                }
                image(task, 0.3f);
                std::vector<float> first;
                if (use == Look) first = read(task.layer(0).ptr, size_of(task.layer(0)));
                if (use == Stage) task.initExecution();
                if (use == Layer) task.kernels[3]->execute(stream.s);
                TK_SAFE_CALL(tkStreamSynchronize(stream.s));
                image(plain, 1.0f / (float)queries);
                plain.executeQuery(nullptr);
                char what[100];
                snprintf(what, sizeof(what), "%d x %d, use %d behind %d queries, watched %d", height, width, use, queries, watched);
                if (!same_outputs(what, task, plain)) return false;
                if (use == Look && !same(first, read(plain.layer(0).ptr, size_of(plain.layer(0))))) return false;
                const float *staged = static_cast<float *>(task.Input[0]), *host = static_cast<float *>(task.InputHost[0]);
                const size_t n = task.InputSize[0] / sizeof(float);
                if (use == Stage && !same(read(staged, n), std::vector<float>(host, host + n))) {
                    printf("%s: not the image staged\n", what);
                    return false;
                }
            }
    return true;
}

// A launch that fails, in a query or while what queries left out is computed, is an error of that call: the next one has the
// outputs of the image the query read, or goes on from there.
bool after_a_failed_launch(bool query)
{
    VGG16Options opt;
    opt.height = 64, opt.width = 96;
    const auto fails = [](const char *prefix, auto call) {   // with the kernels of that prefix out of reach
        const auto kept = fmap;
        for (auto &k : kept)
            if (k.first.compare(0, strlen(prefix), prefix) == 0) fmap.erase(k.first);
        bool failed = false;
        try {
            call();
        } catch (const std::exception &) {
            failed = true;
        }
        fmap = kept;
        return failed;
    };
    for (int queries : {1, 2}) {
        VGG16 task(1, opt), plain(2, opt);
        use_tzgemm(plain);
        for (int q = 0; q < queries; ++q)
            for (VGG16 *t : {&task, &plain}) {
                image(*t, 1.0f / (float)(1 + q));
                t->executeQuery(nullptr);
            }
        if (query) {
            image(task, 0.75f);
            if (!fails("fc_direct", [&] { task.executeQuery(nullptr); })) return false;
            for (VGG16 *t : {&task, &plain}) {
                image(*t, 0.6f);
                t->executeQuery(nullptr);
            }
        } else {
            for (int again = 0; again < 2; ++again)
                if (!fails("conv3x3_direct", [&] { task.layer(3); })) return false;
        }
        if (!same_outputs("after a failed launch", task, plain)) return false;
    }
    return true;
}

// Ranges of lbm in workgroups of less than a wavefront, of a wavefront and a half, and of eight, are those of ordinary ones.
bool lbm_workgroups()
{
    OriLBMKernel ori(1);
    const int rows = ori.sizeY() * ori.sizeZ();
    const size_t floats = (size_t)ori.sizeX() * rows * 19;
    const std::vector<float> nothing(floats, -5.0f);
    for (const auto &range : {std::pair<int, int>(0, rows), {0, 1}, {rows / 2, rows / 2 + 77}, {rows - 3, rows + 2}}) {
        std::vector<float> want;
        for (int block : {256, 32, 48, 96, 512}) {
            write(ori.params()->dst, nothing);
            GPTBKernel k(2, "lbm", "gptb_lbm", &ori, dim3(block < 64 ? 1000 : 75, 1, 1), dim3(block, 1, 1), range.first, range.second);
            k.execute(nullptr);
            const std::vector<float> got = read(ori.params()->dst, floats);
            if (want.empty()) want = got;
            if (!same(got, want)) {
                printf("rows %d to %d, workgroups of %d\n", range.first, range.second, block);
                return false;
            }
        }
        if (same(want, nothing)) return false;
    }
    return true;
}

}  // namespace

int main(int argc, char **argv)
{
    const char *check = argc > 1 ? argv[1] : "";
    if (tacker_init(0, nullptr)) return 2;
    bool ok = false;
    try {
        if (!strcmp(check, "raw")) ok = written_between_layers(false, false) && written_between_layers(true, false);
        else if (!strcmp(check, "bias")) ok = written_between_layers(false, true) && written_between_layers(true, true);
        else if (!strcmp(check, "classes")) ok = many_classes(1000) && many_classes(8192) && many_classes(9000);
        else if (!strcmp(check, "lean"))
            ok = raw_outputs_after_queries(32, 32) && raw_outputs_after_queries(64, 96) && raw_outputs_after_queries(128, 160) &&
                 raw_outputs_after_queries(64, 96, true);
        else if (!strcmp(check, "recorded_layers")) ok = recorded_part(0, true);
        else if (!strcmp(check, "recorded_fused")) ok = recorded_part(5, true);
        else if (!strcmp(check, "recorded_behind_queries")) ok = recorded_part(0, false) && recorded_part(5, false);
        else if (!strcmp(check, "recorded_query")) ok = recorded_query(true) && recorded_query(false);
        else if (!strcmp(check, "sizes")) ok = outputs(160, 160) && outputs(160, 352) && outputs(352, 352) && outputs(96, 416);
        else if (!strcmp(check, "paid_once")) ok = paid_once();
        else if (!strcmp(check, "straight_behind")) ok = straight_behind_queries(64, 96, 4) && straight_behind_queries(224, 224, 2);
        else if (!strcmp(check, "failed_launch")) ok = after_a_failed_launch(true) && after_a_failed_launch(false);
        else if (!strcmp(check, "lbm_workgroups")) ok = lbm_workgroups();
        else return 2;
    } catch (const std::exception &e) {
        printf("%s\n", e.what());
    }
    printf("%s %s\n", check, ok ? "ok" : "FAILED");
    return ok ? 0 : 1;
}
