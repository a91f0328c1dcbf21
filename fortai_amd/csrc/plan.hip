// The kernel variant each launcher chose, for plan recording: every launcher
// in the *.hip files calls note_launch() after it launches, and the decoders
// read last_launch() to record (operation, kernel, batch) steps -- the
// reference's PlanIR step (src/fortai_plan_ir.f90:7-21).  Outside a recording
// nobody reads the note and it is not formatted: in a program of single
// operations about half of the launches would pay for one (0.8B, four layers,
// host bound, 24 processes a side: 201.2 us a token with them, 196.8 without).
#include "fortai_hip_kernels.h"

#include <cstdarg>
#include <cstdio>

namespace fortai_hip {

namespace {
thread_local char g_last[256] = "";
thread_local bool g_noting = false;
}

void note_launches(bool on) { g_noting = on; }

void note_launch(const char *fmt, ...) {
    if (!g_noting) return;
    va_list ap;
    va_start(ap, fmt);
    std::vsnprintf(g_last, sizeof(g_last), fmt, ap);
    va_end(ap);
}

const char *last_launch() { return g_last; }

const char *prologue_name(Prologue p) {
    switch (p) {
    case Prologue::Q8: return "q8";
    case Prologue::F32: return "f32";
    case Prologue::RMSNORM: return "rmsnorm";
    case Prologue::Q8L: return "q8l";
    case Prologue::GATED: return "gated";
    }
    return "?";
}

const char *epilogue_name(Epilogue e) {
    switch (e) {
    case Epilogue::STORE: return "store";
    case Epilogue::ADD: return "add";
    case Epilogue::SILU_PAIR: return "silu_pair";
    }
    return "?";
}

}  // namespace fortai_hip
