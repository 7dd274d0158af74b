// The launches that api.cpp makes, as text: linked with it in place of the kernels, on the CPU (test_launch_order.py).  A line for each:
// the launch, then for each job of it the output, the scratch memory of its pieces (0: none) and what is done there, and the workgroups.
#include <string>

#include "kernels.h"

namespace {
std::string g_log;

bool in_pieces(const magi::AttnKernArgs& a) { return a.split_from < a.per_xcd || a.share_pieces > 1; }
// does: 'w' leaves pieces, 'r' brings them together, 'b' both in launches of its own one behind the other
void note(const char* name, unsigned long long blocks, std::initializer_list<std::pair<const magi::AttnKernArgs*, char>> jobs) {
  char line[256];
  g_log += name;
  for (auto& [a, does] : jobs) {
    snprintf(line, sizeof(line), " %p %p %c", (void*)a->out, (void*)(in_pieces(*a) ? a->partial : nullptr), in_pieces(*a) ? does : '-');
    g_log += line;
  }
  snprintf(line, sizeof(line), " %llu\n", blocks);
  g_log += line;
}
unsigned long long grid(const magi::AttnKernArgs& a) {
  return 8ull * (a.per_xcd + (unsigned long long)magi::split_items(a) * (magi::split_items(a) ? a.split_pieces - 1 : 0));
}
}  // namespace

extern "C" const char* take_log() {
  static std::string last;
  last.swap(g_log);
  g_log.clear();
  return last.c_str();
}

namespace magi {
#define ONE(fn)                                              \
  hipError_t fn(const AttnKernArgs& a, hipStream_t) {        \
    note(#fn, grid(a), {{&a, 'b'}});                         \
    return hipSuccess;                                       \
  }
ONE(launch_attn_fwd_bf16)
ONE(launch_attn_fwd_bf16_r32)
ONE(launch_attn_fwd_bf16_w64)
ONE(launch_attn_fwd_fp8)
hipError_t launch_attn_fwd_bf16_x16(const AttnKernArgs& a, hipStream_t, bool merge) {
  note("launch_attn_fwd_bf16_x16", grid(a), {{&a, merge ? 'b' : 'w'}});
  return hipSuccess;
}
hipError_t launch_attn_fwd_bf16_merge(const AttnKernArgs& a, hipStream_t) {
  note("launch_attn_fwd_bf16_merge", 32ull * split_items(a), {{&a, 'r'}});
  return hipSuccess;
}
hipError_t launch_attn_text_merge(const AttnPairArgs& p, hipStream_t) {
  note("launch_attn_text_merge", 32ull * split_items(p.job[0]) + grid(p.job[1]), {{&p.job[0], 'r'}, {&p.job[1], 'b'}});
  return hipSuccess;
}
#define PAIR(fn)                                                                                \
  hipError_t fn(const AttnPairArgs& p, hipStream_t) {                                           \
    if (p.job[1].per_xcd == 0)                                                                  \
      note(#fn, grid(p.job[0]), {{&p.job[0], 'b'}});                                            \
    else                                                                                        \
      note(#fn, grid(p.job[0]) + grid(p.job[1]), {{&p.job[0], 'b'}, {&p.job[1], 'b'}});         \
    return hipSuccess;                                                                          \
  }
PAIR(launch_attn_fwd_bf16_waves)
PAIR(launch_attn_fwd_bf16_x16_pair)
PAIR(launch_attn_fwd_fp8_text)
hipError_t launch_attn_fwd_bf16_checked(const AttnKernArgs& a, int, hipStream_t) {
  note("launch_attn_fwd_bf16_checked", grid(a), {{&a, 'b'}});
  return hipSuccess;
}
hipError_t launch_gate_init(unsigned*, hipStream_t) { return hipSuccess; }
hipError_t launch_row_norm_max(const char*, long, long, int, int, unsigned*, hipStream_t) {
  g_log += "launch_row_norm_max 0\n";
  return hipSuccess;
}
hipError_t launch_prologue(const PrologueKernArgs&, hipStream_t) { return hipErrorUnknown; }
hipError_t launch_qkv_gemm_prologue(const QkvGemmKernArgs&, hipStream_t) { return hipErrorUnknown; }
hipError_t launch_small_proj(const SmallProjKernArgs&, int, hipStream_t) { return hipErrorUnknown; }
hipError_t launch_head_norm(const char*, long, long, const float*, const float*, char*, int, int, int, float, hipStream_t) { return hipErrorUnknown; }
hipError_t launch_layer_norm(const char*, long, const void*, const void*, int, char*, long, long, int, float, hipStream_t) { return hipErrorUnknown; }
hipError_t launch_layer_norm_quant(const LnQuantKernArgs&, int, int, hipStream_t) { return hipErrorUnknown; }
hipError_t launch_div_clamp(const char*, long, const float*, int, char*, long, long, int, hipStream_t) { return hipErrorUnknown; }
hipError_t launch_rotary(const void*, const float*, const float*, void*, int, int, int, int, int, int, hipStream_t) { return hipErrorUnknown; }
hipError_t launch_quantize_fp8(const char*, long, long, char*, float*, int, int, int, float, int, int, char*, float*, bool, int, hipStream_t, int*) { return hipErrorUnknown; }
hipError_t launch_quantize_fp8_row_max(const char*, long, long, char*, float*, int, int, int, float, int, int, char*, float*, const unsigned short*, int, hipStream_t) { return hipErrorUnknown; }
}  // namespace magi
