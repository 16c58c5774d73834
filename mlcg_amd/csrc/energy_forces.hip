// Energies and forces of the fused SchNet from one call -- the node sweep (node
// linears, gathers, output network) and its reverse, issued back to back on the
// caller's stream from the blocks' filter values -- and, from a second one, the
// tangent and second reverse sweep of the force-matching gradient.
//
// The sweep is about eight launches per block of 2-10 us each on small systems,
// so what bounds a small call is the host.  Issued one entry point at a time
// from Python, a launch costs 10-20 us (allocation, checks, argument
// conversion); from here it costs the launch alone: energies and forces of one
// 35-bead chain 541 -> 280 us in all, the training step on 24 x 57 beads 1074 with
// the first sweep here and 851 with both, from 989-1296.  The launches, their
// order and their results are those of the separate entry points.
#include "common.h"

namespace {

constexpr int kF = 128;
constexpr int64_t kImageBytes = 65536;  // one split weight image

// [N, 128] arrays of the sweep within one buffer.  keep: everything the second
// reverse sweep reads has its own array; otherwise arrays are taken again as
// soon as they are read, which also keeps the sweep's footprint small enough to
// stay in the memory-side cache for longer.
struct Layout {
  int blocks;
  bool keep, want_z;
  int x(int k) const { return keep ? k : k & 1; }
  int y0() const { return keep ? blocks + 1 : 2; }
  int y(int k) const { return y0() + k; }
  int s(int k) const { return y0() + blocks + k; }
  int z(int k) const { return y0() + 2 * blocks + k; }
  int r0() const { return y0() + (want_z ? 3 : 2) * blocks; }
  int agg(int k) const { return r0() + (keep ? k : 0); }
  int gagg(int k) const { return keep ? r0() + blocks + k : r0() + 1; }
  int xbar(int k) const { return keep ? r0() + 2 * blocks + k : r0() + 2 + (k & 1); }
  int ybar(int k) const { return keep ? r0() + 3 * blocks + k : r0() + 4; }
  int sbar(int k) const { return r0() + 4 * blocks + k; }
  int zbar(int k) const { return r0() + 5 * blocks + k; }
  int count() const { return keep ? r0() + 6 * blocks : r0() + 5; }
};

// ... and of the tangent and second reverse sweep, which also reads a kept Layout.
struct Layout2 {
  int blocks;
  // input tangent of block k >= 1; k = blocks: of the last block's output
  int xdot(int k) const { return k - 1; }
  int ydot(int k) const { return blocks + k; }  // k >= 1
  int aggdot(int k) const { return 2 * blocks + k; }
  int zdot(int k) const { return 3 * blocks + k; }
  int sdot(int k) const { return 4 * blocks + k; }
  int gagg2(int k) const { return 5 * blocks + k; }
  int xbar2(int k) const { return 6 * blocks + (k & 1); }
  int zbar2() const { return 6 * blocks + 2; }
  int ybar2() const { return 6 * blocks + 3; }
  int count() const { return 6 * blocks + 4; }
};

}  // namespace

extern "C" int64_t mlcg_energy_forces_arrays(int num_blocks, int block_act, int keep) {
  return Layout{num_blocks, keep != 0, block_act != MLCG_ACT_TANH}.count();
}

extern "C" int mlcg_energy_forces(const float* pos, const float* dist, const int64_t* types,
                                  int64_t n_nodes, const int64_t* frame_ptr, int64_t n_frames,
                                  const int32_t* rowptr, const int32_t* col,
                                  const int32_t* eid2pair, const void* const* filters,
                                  int w_f16, const void* const* weights, int num_blocks,
                                  int num_types, int out_hidden, int block_act, int out_act,
                                  int keep, const float* seed, float* arrays,
                                  int64_t num_arrays, void* images, float* out_rows,
                                  float* dbar, float* energies, float* forces, void* stream) {
  MLCG_REQUIRE(filters && weights && num_blocks >= 1 && n_nodes >= 1 && n_frames >= 1);
  MLCG_REQUIRE(arrays && images && out_rows && dbar && energies && forces && seed);
  const Layout at{num_blocks, keep != 0, block_act != MLCG_ACT_TANH};
  MLCG_REQUIRE(num_arrays >= at.count());
  const auto arr = [&](int i) { return arrays + (int64_t)i * n_nodes * kF; };
  // weights: the embedding table, A1 A2 c2 A3 c3 of each block, W0 b0 w1 b1
  const auto wt = [&](int i) { return static_cast<const float*>(weights[i]); };
  const auto bw = [&](int k, int i) { return wt(1 + 5 * k + i); };
  const float* const* ow = reinterpret_cast<const float* const*>(weights) + 1 + 5 * num_blocks;
  enum { A1, A2, C2, A3, C3 };
  // images of A1 A2 A3, each as it is and transposed
  const auto img = [&](int k, int w, int t) {
    return static_cast<const char*>(images) + ((k * 3 + w) * 2 + t) * kImageBytes;
  };
  int st = mlcg_embedding_gather(wt(0), num_types, kF, types, n_nodes, arr(at.x(0)), stream);
  if (st != MLCG_OK) return st;
  for (int first = 0; first < 6 * num_blocks; first += 30) {
    const int n = 6 * num_blocks - first < 30 ? 6 * num_blocks - first : 30;
    const float* ws[30];
    int ts[30];
    for (int i = 0; i < n; ++i) {
      const int k = (first + i) / 6, w = (first + i) % 6 / 2;
      ws[i] = bw(k, w == 0 ? A1 : w == 1 ? A2 : A3);
      ts[i] = (first + i) & 1;
    }
    st = mlcg_node_weight_images(ws, ts, n, static_cast<char*>(images) + first * kImageBytes,
                                 stream);
    if (st != MLCG_OK) return st;
  }
  for (int k = 0; k < num_blocks; ++k) {
    float *x = arr(at.x(k)), *y = arr(at.y(k)), *agg = arr(at.agg(k));
    st = mlcg_node_gemm(x, n_nodes, kF, bw(k, A1), 0, nullptr, nullptr, 0, 0, nullptr, nullptr,
                        nullptr, nullptr, y, nullptr, img(k, 0, 0), stream);
    if (st == MLCG_OK)
      st = mlcg_cfconv_gather(y, filters[2 * k], w_f16, rowptr, col, eid2pair, n_nodes, kF, agg,
                              stream);
    if (st == MLCG_OK)
      st = mlcg_node_gemm2(agg, n_nodes, kF, bw(k, A2), 0, bw(k, C2), nullptr, 1, block_act,
                           nullptr, nullptr, nullptr, nullptr,
                           at.want_z ? arr(at.z(k)) : nullptr, arr(at.s(k)), bw(k, A3),
                           bw(k, C3), x, arr(at.x(k + 1)), img(k, 1, 0), img(k, 2, 0), stream);
    if (st != MLCG_OK) return st;
  }
  // out_rows: with keep os [N, HH] and, but for tanh, oz [N, HH]; then o [N]
  // (the wide rows first, where they stay aligned)
  float *os = nullptr, *oz = nullptr, *o = out_rows;
  if (keep) {
    os = o;
    o += n_nodes * out_hidden;
    if (out_act != MLCG_ACT_TANH) {
      oz = o;
      o += n_nodes * out_hidden;
    }
  }
  st = mlcg_out_forward(arr(at.x(num_blocks)), n_nodes, kF, out_hidden, ow[0], ow[1], ow[2],
                        ow[3], out_act, 1, seed, o, oz, os, arr(at.xbar(num_blocks - 1)),
                        stream);
  if (st == MLCG_OK)
    st = mlcg_segment_sum(o, 1, frame_ptr, n_frames, energies, stream);
  for (int k = num_blocks - 1; k >= 0 && st == MLCG_OK; --k) {
    float *xbar = arr(at.xbar(k)), *gagg = arr(at.gagg(k)), *ybar = arr(at.ybar(k));
    st = mlcg_node_gemm2(xbar, n_nodes, kF, bw(k, A3), 1, nullptr, nullptr, 2, block_act,
                         at.want_z ? arr(at.z(k)) : nullptr, arr(at.s(k)), nullptr, nullptr,
                         at.keep ? arr(at.sbar(k)) : nullptr,
                         at.keep ? arr(at.zbar(k)) : nullptr, bw(k, A2), nullptr, nullptr, gagg,
                         img(k, 2, 1), img(k, 1, 1), stream);
    // the first block's input depends on no position: only its distance adjoints
    if (st == MLCG_OK)
      st = mlcg_cfconv_gather_bwd(gagg, arr(at.y(k)), filters[2 * k], filters[2 * k + 1], w_f16,
                                  rowptr, col, eid2pair, n_nodes, kF, k ? ybar : nullptr, dbar,
                                  k != num_blocks - 1, stream);
    if (st == MLCG_OK && k)
      st = mlcg_node_gemm(ybar, n_nodes, kF, bw(k, A1), 1, nullptr, xbar, 0, 0, nullptr, nullptr,
                          nullptr, nullptr, arr(at.xbar(k - 1)), nullptr, img(k, 0, 1), stream);
  }
  if (st != MLCG_OK) return st;
  return mlcg_pair_forces(pos, dist, dbar, rowptr, col, eid2pair, n_nodes, 0, forces, stream);
}

extern "C" int64_t mlcg_energy_forces_grad_arrays(int num_blocks) {
  return Layout2{num_blocks}.count();
}

extern "C" int64_t mlcg_energy_forces_grad_workspace_floats(int64_t n_nodes, int num_types,
                                                            int out_hidden) {
  int64_t m = mlcg_node_tmm_batch_workspace_floats(n_nodes, 3);
  const int64_t o = mlcg_out_rev2_workspace_floats(n_nodes, out_hidden);
  const int64_t t = mlcg_type_sum_workspace_floats(n_nodes, num_types);
  if (o > m) m = o;
  return t > m ? t : m;
}

extern "C" int mlcg_energy_forces_grad(
    const float* pos, const float* dist, const int64_t* types, int64_t n_nodes,
    const int32_t* rowptr, const int32_t* col, const int32_t* eid2pair, const int32_t* pair_ij,
    int64_t pair_capacity, const int32_t* n_pairs_dev, const void* const* filters,
    const void* const* weights, int num_blocks, int num_types, int out_hidden, int block_act,
    int out_act, const float* u, float scale, const float* tw, const float* pw,
    const float* arrays, const void* images, const float* out_rows, float* ddot, float* arrays2,
    int64_t num_arrays2, float* workspace, int64_t workspace_floats, void* const* grads,
    void* stream) {
  MLCG_REQUIRE(filters && weights && grads && num_blocks >= 1 && n_nodes >= 1);
  MLCG_REQUIRE(u && tw && arrays && images && out_rows && ddot && arrays2 && workspace);
  MLCG_REQUIRE(workspace_floats >=
               mlcg_energy_forces_grad_workspace_floats(n_nodes, num_types, out_hidden));
  const Layout at{num_blocks, true, block_act != MLCG_ACT_TANH};
  const Layout2 at2{num_blocks};
  MLCG_REQUIRE(num_arrays2 >= at2.count());
  const auto arr = [&](int i) { return arrays + (int64_t)i * n_nodes * kF; };
  const auto arr2 = [&](int i) { return arrays2 + (int64_t)i * n_nodes * kF; };
  const auto wt = [&](int i) { return static_cast<const float*>(weights[i]); };
  const auto bw = [&](int k, int i) { return wt(1 + 5 * k + i); };
  const auto zz = [&](int k) { return at.want_z ? arr(at.z(k)) : nullptr; };
  const auto fw = [&](int k) { return static_cast<const float*>(filters[k]); };
  // gradients in the order of the weights
  const auto gr = [&](int i) { return static_cast<float*>(grads[i]); };
  const int out0 = 1 + 5 * num_blocks;
  enum { A1, A2, C2, A3, C3 };
  const auto img = [&](int k, int w, int t) {
    return static_cast<const char*>(images) + ((k * 3 + w) * 2 + t) * kImageBytes;
  };
  int st = mlcg_pair_ddot(pos, dist, pair_ij, pair_capacity, n_pairs_dev, pair_capacity, u, scale,
                          ddot, stream);
  for (int k = 0; k < num_blocks && st == MLCG_OK; ++k) {
    const float* xdot = k ? arr2(at2.xdot(k)) : nullptr;
    float* ydot = k ? arr2(at2.ydot(k)) : nullptr;
    if (k)
      st = mlcg_node_gemm(xdot, n_nodes, kF, bw(k, A1), 0, nullptr, nullptr, 0, 0, nullptr,
                          nullptr, nullptr, nullptr, ydot, nullptr, img(k, 0, 0), stream);
    if (st == MLCG_OK)
      st = mlcg_cfconv_gather_tangent(ydot, arr(at.y(k)), fw(2 * k), fw(2 * k + 1), ddot, rowptr,
                                      col, eid2pair, n_nodes, kF, arr2(at2.aggdot(k)), stream);
    if (st == MLCG_OK)
      st = mlcg_node_gemm2(arr2(at2.aggdot(k)), n_nodes, kF, bw(k, A2), 0, nullptr, nullptr, 2,
                           block_act, zz(k), arr(at.s(k)), nullptr, nullptr, arr2(at2.zdot(k)),
                           arr2(at2.sdot(k)), bw(k, A3), nullptr, xdot,
                           arr2(at2.xdot(k + 1)), img(k, 1, 0), img(k, 2, 0), stream);
  }
  if (st != MLCG_OK) return st;
  const float* os = out_rows;
  const float* oz = out_act != MLCG_ACT_TANH ? os + n_nodes * out_hidden : nullptr;
  st = mlcg_out_rev2(arr(at.x(num_blocks)), arr2(at2.xdot(num_blocks)), n_nodes, kF, out_hidden,
                     wt(out0), wt(out0 + 2), oz, os, out_act, tw, pw, nullptr,
                     arr2(at2.xbar2(num_blocks)), gr(out0), gr(out0 + 1), gr(out0 + 2),
                     gr(out0 + 3), workspace, workspace_floats, stream);
  for (int k = num_blocks - 1; k >= 0 && st == MLCG_OK; --k) {
    const float *xbar2 = arr2(at2.xbar2(k + 1)), *xdot = k ? arr2(at2.xdot(k)) : nullptr;
    float *gagg2 = arr2(at2.gagg2(k)), *ybar2 = arr2(at2.ybar2()), *zbar2 = arr2(at2.zbar2());
    st = mlcg_node_gemm2(xbar2, n_nodes, kF, bw(k, A3), 1, nullptr, nullptr, 3, block_act, zz(k),
                         arr(at.s(k)), arr(at.sbar(k)), arr2(at2.zdot(k)), zbar2, nullptr,
                         bw(k, A2), nullptr, nullptr, gagg2, img(k, 2, 1), img(k, 1, 1), stream);
    if (st == MLCG_OK)
      st = mlcg_cfconv_gather_rev2(gagg2, arr(at.gagg(k)), arr(at.y(k)),
                                   k ? arr2(at2.ydot(k)) : nullptr, fw(2 * k), fw(2 * k + 1),
                                   ddot, rowptr, col, eid2pair, n_nodes, kF, ybar2, nullptr,
                                   nullptr, stream);
    if (st != MLCG_OK) break;
    const int g = 1 + 5 * k;
    const void* problems[18] = {
        xbar2, arr(at.s(k)), arr(at.xbar(k)), arr2(at2.sdot(k)), gr(g + A3), gr(g + C3),
        zbar2, arr(at.agg(k)), arr(at.zbar(k)), arr2(at2.aggdot(k)), gr(g + A2), gr(g + C2),
        ybar2, arr(at.x(k)), k ? arr(at.ybar(k)) : nullptr, xdot, gr(g + A1), nullptr};
    st = mlcg_node_tmm_batch(problems, 3, n_nodes, kF, 0, workspace, workspace_floats, stream);
    if (st == MLCG_OK)
      st = mlcg_node_gemm(ybar2, n_nodes, kF, bw(k, A1), 1, nullptr, xbar2, 0, 0, nullptr,
                          nullptr, nullptr, nullptr, arr2(at2.xbar2(k)), nullptr, img(k, 0, 1),
                          stream);
  }
  if (st != MLCG_OK) return st;
  return mlcg_type_sum(arr2(at2.xbar2(0)), types, n_nodes, kF, num_types, gr(0), nullptr,
                       workspace, workspace_floats, stream);
}
