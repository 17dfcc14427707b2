// The launches of a run of like layers, made by one call: norm, q/k/v, its preparation, the attention of prompt portions,
// the projection out, norm, gate/up and down of one layer after the other, through the entry points that the parts
// call one by one, with the arguments that they would give.  (Host code only.)
//
// A step of few prompt tokens waits for the host: a launch through the parts costs it 12 us (a tensor's allocation,
// its checks, the conversion of some fifteen arguments, the launch itself about 3), a hundred of them are longer than
// the device takes.  Here the operands of some layers come as one array of addresses and the intermediate results as
// one set that every layer uses again: a prompt of 21 tokens through 12 layers of 4B sizes 1,321 -> 861 us.
#include "common.h"

extern "C" {
int pylon_add_rmsnorm(void*, int, float*, const void*, int, int, long long, const float*, const int*, int, int, float, float,
                      hipStream_t);
int pylon_gemm_rows(void*, int, const void*, const void*, int, int, int, long long, long long, long long, int, long long, int,
                    int, int, int, float, float, float, hipStream_t);
int pylon_gemm_wide(void*, const void*, const void*, int, int, int, long long, long long, long long, int, float, float, float,
                    int, hipStream_t);
int pylon_gemm_wide_parts(float*, const void*, const void*, int, int, int, long long, long long, int, int, hipStream_t);
int pylon_qkv_prepare(void*, void*, void*, const void*, int, long long, const float*, const float*, float, const float*, int,
                      const int*, const int*, int, int, int, int, int, hipStream_t);
int pylon_attention_prefill(void*, const void*, const void*, const void*, const int*, int, const int*, int, int, int, int, int,
                            int, float, int, hipStream_t);
}

// Of every layer, in this order; the Python side (engine/layer_run.py) fills them.
enum {
  LR_NORM1, LR_QKV, LR_LD_QKV, LR_Q_NORM, LR_K_NORM, LR_INV_FREQ, LR_K_CACHE, LR_V_CACHE, LR_SLOT_MAP, LR_TABLE,
  LR_TABLE_WIDTH, LR_OUT, LR_LD_OUT, LR_NORM2, LR_GATE_UP, LR_LD_GATE_UP, LR_DOWN, LR_LD_DOWN, LR_LAYER_FIELDS
};
// Of the step.  A product is two numbers: 0 for gemm_wide, else the ranges that K is cut into and gemm_rows' col_tiles, or,
// for gemm_wide_parts, -1 less its tile.
enum {
  LR_TOKENS, LR_WIDTH, LR_HEADS, LR_KV_HEADS, LR_HEAD_DIM, LR_ROT_DIM, LR_PAGE, LR_FF, LR_GELU, LR_MASK, LR_POSITIONS,
  LR_TILES, LR_N_TILES, LR_TILE_ROWS, LR_RESID, LR_NORMED, LR_PROJECTED, LR_Q, LR_CONTEXT, LR_OUT_SUM, LR_HIDDEN,
  LR_DOWN_SUM, LR_QKV_PARTS, LR_QKV_TILES, LR_OUT_PARTS, LR_OUT_TILES, LR_GATE_PARTS, LR_GATE_TILES, LR_DOWN_PARTS,
  LR_DOWN_TILES, LR_STEP_FIELDS
};
enum { LR_EPS1, LR_EPS2, LR_QK_EPS, LR_SCALE, LR_REALS };

extern "C" int pylon_layer_run_fields(int* fields) {
  PYLON_REQUIRE(fields != nullptr, "layer_run_fields: nowhere to put them");
  fields[0] = LR_LAYER_FIELDS, fields[1] = LR_STEP_FIELDS, fields[2] = LR_REALS;
  return 0;
}

// layers: [n_layers][LR_LAYER_FIELDS]; step: [LR_STEP_FIELDS]; reals: [LR_REALS].  The residual stream is that in front of
// the first layer of these; `pending`: what the layer before them left to be added is in LR_DOWN_SUM (else there is
// nothing), as is then what the last of these leaves.
extern "C" int pylon_layer_run(const long long* layers, int n_layers, int pending, const long long* step, const double* reals,
                               hipStream_t stream) {
  PYLON_REQUIRE(layers && step && reals && n_layers >= 1, "layer_run: no layers");
  const int tokens = static_cast<int>(step[LR_TOKENS]), width = static_cast<int>(step[LR_WIDTH]);
  const int heads = static_cast<int>(step[LR_HEADS]), kv_heads = static_cast<int>(step[LR_KV_HEADS]);
  const int dim = static_cast<int>(step[LR_HEAD_DIM]), ff = static_cast<int>(step[LR_FF]);
  const int q_size = heads * dim, qkv_size = (heads + 2 * kv_heads) * dim;
  const long long sum_stride = static_cast<long long>(tokens) * width;
  auto at = [](long long address) { return reinterpret_cast<void*>(address); };
  auto floats = [](long long address) { return reinterpret_cast<const float*>(address); };
  auto ints = [](long long address) { return reinterpret_cast<const int*>(address); };
  auto real = [&](int i) { return static_cast<float>(reals[i]); };
  // out = x w^T, a sum for the residual stream in float parts or one bfloat16 result, gated or neither
  auto product = [&](long long out, long long x, long long w, long long ldw, int n, int k, long long parts, long long col_tiles,
                     bool sums, bool gated) {
    if (parts == 0)
      return pylon_gemm_wide(at(out), at(x), at(w), tokens, n, k, k, ldw, n, gated ? (step[LR_GELU] ? 3 : 1) : 0, 0.f, 0.f, 0.f,
                             -1, stream);
    if (col_tiles < 0)
      return pylon_gemm_wide_parts(static_cast<float*>(at(out)), at(x), at(w), tokens, n, k, k, ldw, static_cast<int>(parts),
                                   static_cast<int>(-1 - col_tiles), stream);
    return pylon_gemm_rows(at(out), sums ? PYLON_F32 : PYLON_BF16, at(x), at(w), tokens, n, k, k, ldw, n, static_cast<int>(parts),
                           static_cast<long long>(tokens) * n, static_cast<int>(col_tiles),
                           gated ? (step[LR_GELU] ? 3 : 1) : 0, 0, 0, 0.f, 0.f, 0.f, stream);
  };
  auto norm = [&](long long delta, long long parts, long long gain, float eps) {
    return pylon_add_rmsnorm(at(step[LR_NORMED]), PYLON_BF16, static_cast<float*>(at(step[LR_RESID])), at(delta),
                             delta && parts == 0 ? PYLON_BF16 : PYLON_F32, parts > 1 ? static_cast<int>(parts) : 1,
                             parts > 1 ? sum_stride : 0, floats(gain), nullptr, tokens, width, eps, 1.0f, stream);
  };
  for (int i = 0; i < n_layers; ++i) {
    const long long* const l = layers + static_cast<size_t>(i) * LR_LAYER_FIELDS;
    int rc = norm(i == 0 && !pending ? 0 : step[LR_DOWN_SUM], step[LR_DOWN_PARTS], l[LR_NORM1], real(LR_EPS1));
    if (!rc) rc = product(step[LR_PROJECTED], step[LR_NORMED], l[LR_QKV], l[LR_LD_QKV], qkv_size, width, step[LR_QKV_PARTS],
                          step[LR_QKV_TILES], false, false);
    if (!rc) rc = pylon_qkv_prepare(at(step[LR_Q]), at(l[LR_K_CACHE]), at(l[LR_V_CACHE]), at(step[LR_PROJECTED]), PYLON_BF16,
                                    qkv_size, floats(l[LR_Q_NORM]), floats(l[LR_K_NORM]), real(LR_QK_EPS),
                                    floats(l[LR_INV_FREQ]), static_cast<int>(step[LR_ROT_DIM]), ints(step[LR_POSITIONS]),
                                    ints(l[LR_SLOT_MAP]), tokens, heads, kv_heads, dim, 1, stream);
    if (!rc) rc = pylon_attention_prefill(at(step[LR_CONTEXT]), at(step[LR_Q]), at(l[LR_K_CACHE]), at(l[LR_V_CACHE]),
                                          ints(l[LR_TABLE]), static_cast<int>(l[LR_TABLE_WIDTH]), ints(step[LR_TILES]),
                                          static_cast<int>(step[LR_N_TILES]), heads, kv_heads, dim,
                                          static_cast<int>(step[LR_PAGE]), static_cast<int>(step[LR_MASK]), real(LR_SCALE),
                                          static_cast<int>(step[LR_TILE_ROWS]), stream);
    if (!rc) rc = product(step[LR_OUT_SUM], step[LR_CONTEXT], l[LR_OUT], l[LR_LD_OUT], width, q_size, step[LR_OUT_PARTS],
                          step[LR_OUT_TILES], true, false);
    if (!rc) rc = norm(step[LR_OUT_SUM], step[LR_OUT_PARTS], l[LR_NORM2], real(LR_EPS2));
    if (!rc) rc = product(step[LR_HIDDEN], step[LR_NORMED], l[LR_GATE_UP], l[LR_LD_GATE_UP], ff, width, step[LR_GATE_PARTS],
                          step[LR_GATE_TILES], false, true);
    if (!rc) rc = product(step[LR_DOWN_SUM], step[LR_HIDDEN], l[LR_DOWN], l[LR_LD_DOWN], width, ff, step[LR_DOWN_PARTS],
                          step[LR_DOWN_TILES], true, false);
    if (rc) return rc;
  }
  return 0;
}
