/*
 * xpu_jit.h - per-plan specialization of the kernels (host side).
 *
 * The kernel bodies of xpu_device.h are templates over the program runner.
 * Ahead of time they run the plan through the op interpreter; here the
 * plan is emitted into a HIP source as constant bytes, each program segment
 * as straight-line calls of the op semantics (xop_exec) with constant
 * operands, and compiled with hiprtc for gfx950.  The compiler folds the op
 * dispatch, the register numbers and every metadata load of the plan, so
 * the specialized kernel keeps the register file in plain VGPRs and has no
 * per-row scalar-load chains.  Results are those of the interpreter by
 * construction: both run the same device functions.
 */
#ifndef XPU_JIT_H
#define XPU_JIT_H
#include <atomic>
#include <memory>
#include <string>
#include <vector>

#include "xpu_program.h"

/* Kernels compiled together are those that one task launches: with all that a
 * plan could launch in one module, the first chunk waited twice as long
 * (hiprtc on one core: C1's group-by 7.8 s with its batched passes, 4.5 s
 * without; C0's scan 4.0 s with the passes for joins, 1.8 s without; C2's join
 * 6.8 s with its one-kernel form, 2.7 s without). */
enum xpu_jit_kind
{
    XJ_SCAN_AGG = 1,        /* scan + group-by task: scan, spill and dump passes (param: rows a lane) */
    XJ_PIPELINE = 2,        /* param 1: group-by over joins in one kernel; 0: the count and
                               write passes of a projection */
    XJ_SCAN_BATCH = 3,      /* the batched passes of a scan + group-by (param: rows a lane) */
    XJ_JOIN_PASSES = 4,     /* group-by over joins: the screen pass and one pass per depth */
};

/* HIP source of the specialized kernels */
std::string xpu_jit_source(const xplan *P, int kind, int param);

/* hiprtc compile for gfx950 into a code object; false with *log filled */
bool xpu_jit_compile(const std::string &src, std::vector<char> *code, std::string *log);

/* code object of the specialized kernel, compiled once per distinct source
 * in the process (thread-safe); nullptr with *log filled on failure */
const std::vector<char> *xpu_jit_code(const xplan *P, int kind, int param, std::string *log);

/* The same off the calling thread: a thread of the library compiles one
 * kernel after another and says so in *state.  It makes no call to the HIP
 * runtime.  Nothing happens if the state is not XJ_STATE_NONE, if the queue is
 * full, or once XJ_BG_MAX kernels have been asked for in the process (each
 * stays in the code cache); the caller may ask again. */
enum xpu_jit_state
{
    XJ_STATE_NONE = 0,
    XJ_STATE_QUEUED = 1,
    XJ_STATE_READY = 2,     /* xpu_jit_code finds it */
    XJ_STATE_FAILED = 3,
};
#define XJ_BG_QUEUE     16
#define XJ_BG_MAX       512
typedef std::shared_ptr<std::atomic<int>> xpu_jit_progress;
void xpu_jit_request(const xplan *P, int kind, int param, const xpu_jit_progress &state);

/* drops what is queued and waits for the kernel being compiled */
void xpu_jit_stop(void);

#endif
