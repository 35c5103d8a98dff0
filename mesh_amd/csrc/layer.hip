// The forward pass of transformer_moe_layer_v1 with _top_2_gating
// (mesh_tensorflow/transformer/moe.py:191-525, :1312-1513) as one library call: the
// calls that make it up, in the order and under the conditions in which the layer
// makes them one by one, on one workspace.  For small layers the host's part of those
// calls (arguments checked and tensors allocated five times) takes longer than their
// kernels: 2048 tokens of 512 in float32 100 us of host time for six launches.
#include "common.h"

using namespace mesh_moe;

namespace {

struct LayerSpace {
  size_t logits, idx, pos, gate, kept, fill, loss, gating, gating_bytes;
  size_t row_offsets, ffn, ffn_bytes, h, y, expert_in, bytes;
  bool fused_router, compact, dispatched, map_by_gating;
};

// Which calls the layer is made of (those of mesh_amd/transformer/moe.py for operands
// on 16 bytes), and where their buffers lie.
LayerSpace layer_space(int G, int S, int E, int C, int M, int H, int N, int dtype) {
  LayerSpace w = {};
  const size_t size = dtype_size(dtype), rows = (size_t)G * C;
  const size_t tokens = (size_t)G * S;
  w.fused_router = fused_router_shapes(M, E, S, dtype);
  w.compact = top2_compacts(G, C) && compact_ffn_shapes(G, S, E, C, M, H, N, dtype);
  w.dispatched = !w.compact && dispatched_ffn_shapes(G, S, E, C, M, H, dtype);
  w.map_by_gating = w.dispatched && !w.fused_router && gating_makes_map(G, S) &&
                    dispatched_few_rows(G, S, E, C, M, H);
  auto take = [&](size_t n) {
    const size_t at = w.bytes;
    w.bytes += (n + 255) & ~(size_t)255;
    return at;
  };
  if (!w.fused_router) w.logits = take(sizeof(float) * tokens * E);
  w.idx = take(sizeof(int32_t) * 2 * tokens);
  w.pos = take(sizeof(int32_t) * 2 * tokens);
  w.gate = take(sizeof(float) * 2 * tokens);
  w.kept = take(2 * tokens);
  w.fill = take(sizeof(int32_t) * G * E);
  w.loss = take(sizeof(float));
  w.gating_bytes = mesh_moe_gating_workspace_bytes(G, S, E);
  w.gating = take(w.gating_bytes);
  if (w.compact) {
    w.row_offsets = take(sizeof(int32_t) * (size_t)E * G);
    w.ffn_bytes = mesh_moe_compact_expert_ffn_workspace_bytes(G, E, C, M, H, N);
  } else if (w.dispatched) {
    w.ffn_bytes = mesh_moe_dispatched_expert_ffn_workspace_bytes(G, E, C, M);
  }
  w.ffn = take(w.ffn_bytes);
  w.h = take(size * E * rows * H);
  w.y = take(size * E * rows * N);
  if (!w.compact && !w.dispatched) w.expert_in = take(size * E * rows * M);
  w.bytes += 256;
  return w;
}

bool layer_sizes_ok(int G, int S, int E, int C, int M, int H, int N) {
  return G >= 1 && S >= 1 && E >= 1 && C >= 1 && M >= 1 && H >= 1 && N >= 1 &&
         (int64_t)G * C <= 0x7fffffffLL && (int64_t)G * S <= 0x7fffffffLL;
}

}  // namespace

extern "C" size_t mesh_moe_top2_layer_workspace_bytes(int G, int S, int E, int C,
                                                      int M, int H, int N,
                                                      int dtype) {
  if (!layer_sizes_ok(G, S, E, C, M, H, N) || !valid_dtype(dtype)) return 0;
  return layer_space(G, S, E, C, M, H, N, dtype).bytes;
}

extern "C" int mesh_moe_top2_layer(
    const void* x, const void* w_gate, const void* w_gate_packed,
    const void* wi_packed, const void* wo_packed, const void* importance,
    int importance_dtype, void* out, void* loss_out, void* workspace,
    size_t workspace_bytes, int G, int S, int E, int C, int M, int H, int N,
    int activation, int dtype, int policy, double threshold,
    int use_second_place_loss, int num_microbatches, double loss_coef,
    void* stream) {
  MOE_REQUIRE(x && w_gate && w_gate_packed && wi_packed && wo_packed && out &&
                  loss_out && workspace, MESH_MOE_E_ARG, "top2_layer: null pointer");
  MOE_REQUIRE(valid_dtype(dtype), MESH_MOE_E_ARG, "top2_layer: bad dtype %d", dtype);
  MOE_REQUIRE(layer_sizes_ok(G, S, E, C, M, H, N), MESH_MOE_E_ARG,
              "top2_layer: bad sizes");
  MOE_REQUIRE(policy != MESH_MOE_SECOND_RANDOM, MESH_MOE_E_UNSUPPORTED,
              "top2_layer: policy RANDOM");
  MOE_REQUIRE(((uintptr_t)x | (uintptr_t)w_gate_packed | (uintptr_t)wi_packed |
               (uintptr_t)wo_packed) % 16 == 0,
              MESH_MOE_E_UNSUPPORTED, "top2_layer: operands off 16 bytes");
  const LayerSpace w = layer_space(G, S, E, C, M, H, N, dtype);
  MOE_REQUIRE(workspace_bytes >= w.bytes, MESH_MOE_E_ARG,
              "top2_layer: workspace too small");
  char* at = (char*)(((uintptr_t)workspace + 255) & ~(uintptr_t)255);
  int32_t *idx = (int32_t*)(at + w.idx), *pos = (int32_t*)(at + w.pos);
  float *gate = (float*)(at + w.gate), *loss = (float*)(at + w.loss);
  uint8_t* kept = (uint8_t*)(at + w.kept);
  int32_t* fill = (int32_t*)(at + w.fill);
  const int64_t tokens = (int64_t)G * S;
  int rc;
  if (w.fused_router) {
    rc = mesh_moe_router_top2_gating(
        x, w_gate_packed, nullptr, nullptr, 1, tokens, M, dtype, importance,
        importance_dtype, 0, nullptr, G, S, E, C, policy, threshold,
        use_second_place_loss, num_microbatches, idx, pos, gate, kept, fill, loss,
        at + w.gating, w.gating_bytes, stream);
  } else {
    float* logits = (float*)(at + w.logits);
    rc = mesh_moe_router_logits(x, w_gate, w_gate_packed, nullptr, logits, 1, tokens,
                                M, E, dtype, stream);
    if (rc == 0)
      rc = top2_gating(logits, importance, importance_dtype, 0, nullptr, G, S, E, C,
                       policy, threshold, use_second_place_loss, num_microbatches, idx,
                       pos, gate, kept, fill, loss, at + w.gating, w.gating_bytes,
                       stream, w.map_by_gating ? slot_map_in(at + w.ffn, G, E, C, M)
                                               : SlotMap());
  }
  if (rc != 0) return rc;
  void *h = at + w.h, *y = at + w.y;
  int32_t* row_offsets = nullptr;
  if (w.compact) {
    row_offsets = (int32_t*)(at + w.row_offsets);
    rc = mesh_moe_compact_expert_ffn(x, idx, pos, gate, kept, fill, wi_packed,
                                     wo_packed, h, y, row_offsets, nullptr, 1.0f,
                                     nullptr, at + w.ffn, w.ffn_bytes, G, S, E, C, M,
                                     H, N, activation, dtype, stream);
  } else if (w.dispatched) {
    rc = dispatched_ffn(x, idx, pos, gate, kept, fill, w.map_by_gating, wi_packed,
                        wo_packed, h, y, at + w.ffn, w.ffn_bytes, G, S, E, C, M, H, N,
                        activation, dtype, stream);
  } else {
    void* expert_in = at + w.expert_in;
    rc = mesh_moe_dispatch(x, idx, pos, gate, kept, fill, expert_in, nullptr, G, S, E,
                           C, M, dtype, stream);
    if (rc == 0)
      rc = mesh_moe_expert_ffn(expert_in, wi_packed, wo_packed, h, y, E, G * C, M, H,
                               N, activation, dtype, stream);
  }
  if (rc != 0) return rc;
  return mesh_moe_combine_loss(y, idx, pos, gate, kept, row_offsets, loss, loss_coef,
                               out, loss_out, G, S, E, C, N, dtype, stream);
}
