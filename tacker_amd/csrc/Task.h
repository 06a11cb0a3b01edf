// Task.h -- an ordered list of kernels run as one job (src/Task.h of the reference).
#pragma once
#include <string>
#include <vector>

#include "Kernel.h"

enum ExecutionMode { Aker = 0, Tacker };
enum TaskType { LC = 0, BE };

class Task {
public:
    Task(int taskId, std::string taskName);
    explicit Task(int taskId);
    virtual ~Task();
    void addKernel(Kernel *kernel);
    // every kernel in order, each timed with device events; times go to the
    // global Recorder in Aker mode
    void executeTask(ExecutionMode mode, cudaStream_t stream);
    void executeTask(ExecutionMode mode, int idx, cudaStream_t stream);
    // stage the job's input (host -> device copy for a DNN query)
    virtual void initExecution() = 0;
    // the whole job: its input staged (the host's copy may change once this returns), every kernel launched on `stream`
    virtual void executeQuery(cudaStream_t stream);
    // the job's launches recorded from `stream` (not the null stream) into one executable graph:
    // every kernel's execute() once, none of them run.  The job must have run before, so that no
    // kernel still has buffers to allocate, and the caller stages the input before each launch of
    // the graph.  The caller destroys the graph (tkGraphExecDestroy).
    tkGraphExec_t captureQuery(cudaStream_t stream);
    // set while a query's kernels are launched one behind the other, with nobody in between
    bool wholeQuery = false;
    struct WholeQuery {
        Task &task;
        explicit WholeQuery(Task &t) : task(t) { task.wholeQuery = true; }
        ~WholeQuery() { task.wholeQuery = false; }
    };
    // the kernels' execute() is about to be recorded
    virtual void recording() {}
    // the kernels' execute() has been recorded, not run: what a task remembers of its last run no longer holds
    virtual void captured() {}

    int taskId;
    std::string taskName;
    std::vector<Kernel *> kernels;
    TaskType taskType = LC;

    void *Input[3] = {nullptr, nullptr, nullptr};
    void **Result = nullptr;
    void *InputHost[3] = {nullptr, nullptr, nullptr};
    int InputSize[3] = {0, 0, 0};
};
