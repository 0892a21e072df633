// The force-loop handle: device state and the per-iteration sequence of
// SeismicMesh/generation/mesh_generator.py:460-527 (re-triangulate, filter
// cells, forces, update, project), for 2D and 3D domains.
#include <algorithm>
#include <chrono>
#include <cstring>
#include <vector>

#include "common.h"
#include "edges.h"
#include "mesher.h"

using namespace smk;

namespace {

template <typename T>
int dalloc(T **p, int64_t n) {
  *p = nullptr;
  if (n <= 0) n = 1;
  SM_HIP(hipMalloc((void **)p, (size_t)n * sizeof(T)));
  return SM_OK;
}

template <typename T>
void dfree(T *&p) {
  if (p) (void)hipFree((void *)p);
  p = nullptr;
}

void free_point_state(sm_mesher *m) {
  dfree(m->d_p);
  dfree(m->d_tri);
  dfree(m->d_adj);
  dfree(m->d_ori);
  dfree(m->d_claim);
  dfree(m->d_cand);
  dfree(m->d_partner);
  dfree(m->d_mark);
  dfree(m->d_queue);
  dfree(m->d_keep);
  dfree(m->d_edges);
  dfree(m->d_ews);
  dfree(m->d_sptr);
  dfree(m->d_scur);
  dfree(m->d_slist);
  dfree(m->d_scan_ws);
  dfree(m->d_L);
  dfree(m->d_h);
  dfree(m->d_F);
  dfree(m->d_Lp);
  dfree(m->d_hp);
  dfree(m->d_part);
  dfree(m->d_mid);
  dfree(m->d_hext);
  dfree(m->d_psnap);
  dfree(m->d_tri_s);
  dfree(m->d_adj_s);
  dfree(m->d_pvalid);
  dfree(m->d_pstage);
  dfree(m->d_vdom);
  dfree(m->d_tdom);
  dfree(m->d_dnn);
  m->dnn_cap = 0;
  m->h_tbase.clear();
  dfree(m->d_sl_rank);
  dfree(m->d_sl_win);
  dfree(m->d_sl_total);
  if (m->d_sl_ws) (void)hipFree(m->d_sl_ws);
  m->d_sl_ws = nullptr;
  m->sl_capT = m->sl_capN = 0;
  m->nsl = -1;
  m->have_snap = false;
  // a captured iteration refers to these buffers
  if (m->gexec) (void)hipGraphExecDestroy(m->gexec);
  if (m->graph) (void)hipGraphDestroy(m->graph);
  m->gexec = nullptr;
  m->graph = nullptr;
  m->graph_T = -1;
}

int alloc_point_state(sm_mesher *m, int64_t N) {
  free_point_state(m);
  const int dim = m->dim;
  m->capN = N;
  m->nfar = dim == 2 && m->prm.far_square ? 4 * std::max(m->ndom, 1) : 0;
  const int64_t NA = N + m->nfar;
  // 2D: real + ghost triangles of the triangulated sphere, 2 NA - 2 (a
  // batch domain owns 2 (n_d + 4) slots, far square or not); 3D:
  // tetrahedra of a Delaunay tetrahedralisation, ~6.5N for well-spaced
  // points, bounded here generously
  m->capT = dim == 2 ? 2 * (N + 4 * (int64_t)std::max(m->ndom, 1)) + 16 : 10 * N + 64;
  const int64_t T = m->capT;
  const int64_t npairs = T * (dim == 2 ? 3 : 6);
  m->capE = npairs;
  int rc;
  if ((rc = dalloc(&m->d_p, NA * dim))) return rc;
  if ((rc = dalloc(&m->d_tri, T * (dim + 1)))) return rc;
  if ((rc = dalloc(&m->d_adj, T * (dim + 1)))) return rc;
  if ((rc = dalloc(&m->d_ori, T))) return rc;
  if ((rc = dalloc(&m->d_claim, T))) return rc;
  if ((rc = dalloc(&m->d_cand, T * (dim + 1)))) return rc;
  if ((rc = dalloc(&m->d_partner, T))) return rc;
  if ((rc = dalloc(&m->d_mark, T))) return rc;
  if ((rc = dalloc(&m->d_queue, 4 * T))) return rc;
  if ((rc = dalloc(&m->d_keep, T))) return rc;
  if ((rc = dalloc(&m->d_edges, 2 * m->capE))) return rc;
  m->ews_bytes = unique_edges_workspace(npairs, N);
  SM_HIP(hipMalloc(&m->d_ews, m->ews_bytes));
  if ((rc = dalloc(&m->d_sptr, N + 1))) return rc;
  if ((rc = dalloc(&m->d_scur, N + 1))) return rc;
  if ((rc = dalloc(&m->d_slist, m->capE))) return rc;
  SM_HIP(hipMalloc(&m->d_scan_ws, scan_workspace(N + 1)));
  const size_t tsz = m->prm.precision == 64 ? 8 : 4;
  SM_HIP(hipMalloc(&m->d_L, (size_t)m->capE * tsz));
  SM_HIP(hipMalloc(&m->d_h, (size_t)m->capE * tsz));
  SM_HIP(hipMalloc(&m->d_F, (size_t)m->capE * dim * tsz));
  if ((rc = dalloc(&m->d_Lp, m->capE))) return rc;
  if ((rc = dalloc(&m->d_hp, m->capE))) return rc;
  if ((rc = dalloc(&m->d_part, 2 * (m->capE / 256 + 2) + 16))) return rc;
  if (m->host_sizing) {
    if ((rc = dalloc(&m->d_mid, m->capE * dim))) return rc;
    if ((rc = dalloc(&m->d_hext, m->capE))) return rc;
  }
  if ((rc = dalloc(&m->d_psnap, NA * dim))) return rc;
  if ((rc = dalloc(&m->d_pvalid, NA * dim))) return rc;
  if ((rc = dalloc(&m->d_pstage, NA * dim))) return rc;
  if ((rc = dalloc(&m->d_tri_s, T * (dim + 1)))) return rc;
  if ((rc = dalloc(&m->d_adj_s, T * (dim + 1)))) return rc;
  if ((rc = fill<int32_t>(m->d_mark, T, 0, m->stream))) return rc;
  if (m->ndom > 0 && (rc = dalloc(&m->d_vdom, NA))) return rc;
  if (m->ndom > 0 && (rc = dalloc(&m->d_tdom, T))) return rc;
  if (m->surrogate) {
    m->dnn_cap = std::max(T, NA);
    if ((rc = dalloc(&m->d_dnn, m->dnn_cap))) return rc;
  }
  return SM_OK;
}

// domain of each vertex from the batch's vertex offsets
__global__ void k_vertex_domains(int ndom, const int32_t *voff, int32_t *vdom) {
  const int d = blockIdx.y;
  const int32_t b = voff[d], e = voff[d + 1];
  for (int32_t v = b + (int32_t)(blockIdx.x * blockDim.x + threadIdx.x); v < e;
       v += (int32_t)(gridDim.x * blockDim.x))
    vdom[v] = d;
}

__global__ void k_midpoints(int64_t E, int dim, const int32_t *edges, const double *p,
                            double *mid) {
  int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= E) return;
  int64_t a = edges[2 * e], b = edges[2 * e + 1];
  for (int d = 0; d < dim; ++d) mid[dim * e + d] = (p[dim * a + d] + p[dim * b + d]) / 2.0;
}

int host_sizing_pass(sm_mesher *m) {
  // midpoints -> host -> user function -> device h
  const int64_t E = m->E;
  const int dim = m->dim;
  if (E == 0) return SM_OK;
  hipLaunchKernelGGL(k_midpoints, dim3(blocks_for(E, 256)), dim3(256), 0, m->stream, E, dim,
                     m->d_edges, m->d_p, m->d_mid);
  SM_LAUNCH_CHECK();
  std::vector<double> mid((size_t)E * dim), h((size_t)E);
  SM_HIP(hipMemcpyAsync(mid.data(), m->d_mid, E * dim * sizeof(double), hipMemcpyDeviceToHost,
                        m->stream));
  SM_HIP(hipStreamSynchronize(m->stream));
  int rc = m->host_sizing(m->host_sizing_ctx, mid.data(), E, h.data());
  SM_CHECK(rc == 0, SM_ERR_ARG, "host sizing callback failed (%d)", rc);
  SM_HIP(hipMemcpyAsync(m->d_hext, h.data(), E * sizeof(double), hipMemcpyHostToDevice,
                        m->stream));
  SM_HIP(hipStreamSynchronize(m->stream));
  return SM_OK;
}

// 3D: the tetrahedralisation is rebuilt from the current points every
// iteration (as the reference does with CGAL), on the device (stars3d.hip).
// *done is false when the device leaves it to host_rebuild3d.
int device_rebuild3d(sm_mesher *m, bool *done) {
  const auto t0 = std::chrono::steady_clock::now();
  int64_t count = 0;
  int rc = device_delaunay3d(&m->stars, m->d_p, m->N, m->prm.h0, m->sl_threads, m->d_tri, m->capT,
                             &count, done, m->stream);
  m->stats[15] = m->stars.left;
  if (rc || !*done) return rc;
  m->T = count;
  m->stats[11] = count;
  m->stats[13] += 1;
  m->have_tri = true;
  m->stats[14] += (int64_t)std::chrono::duration_cast<std::chrono::microseconds>(
                      std::chrono::steady_clock::now() - t0)
                      .count();
  return SM_OK;
}

// 3D on the host, where the device build declines: on sl_threads threads
// inserting the points of sl_n slabs into one shared tetrahedralisation.
// Its cells are sorted straight into pinned staging and handed out in
// pieces, each copied to the device asynchronously as it comes; the
// centroid filter then runs once over all of them (one launch keeps the
// GPU full: the SDF program is long per cell, and a piece's launch of a
// few tens of thousands of cells leaves most SIMDs idle).  *filtered tells
// whether the filter ran that way (device programs) or is still to run
// (host callbacks).
int host_rebuild3d(sm_mesher *m, bool *filtered) {
  const auto t0 = std::chrono::steady_clock::now();
  const int64_t N = m->N;
  if (m->h_pts_cap < N) {
    if (m->h_pts) (void)hipHostFree(m->h_pts);
    m->h_pts = nullptr;
    m->h_pts_cap = 0;
    SM_HIP(hipHostMalloc((void **)&m->h_pts, (size_t)N * 3 * sizeof(double),
                         hipHostMallocDefault));
    m->h_pts_cap = N;
  }
  if (m->h_tet_cap < m->capT) {
    if (m->h_tet) (void)hipHostFree(m->h_tet);
    m->h_tet = nullptr;
    m->h_tet_cap = 0;
    SM_HIP(hipHostMalloc((void **)&m->h_tet, (size_t)m->capT * 4 * sizeof(int32_t),
                         hipHostMallocDefault));
    m->h_tet_cap = m->capT;
  }
  SM_HIP(hipMemcpyAsync(m->h_pts, m->d_p, N * 3 * sizeof(double), hipMemcpyDeviceToHost,
                        m->stream));
  SM_HIP(hipStreamSynchronize(m->stream));
  int64_t off = 0;
  int err = SM_OK;
  bool over = false, all_filtered = true;
  auto emit = [&](int piece, const int32_t *v, int64_t count) {
    if (err || over) return;
    if (piece < 0) {
      // all pieces are on their way: the points do not move before the
      // filter, so it may run now
      bool done = false;
      int b = prof_begin(m);
      err = centroid_keep_range(m, 0, off, &done);
      prof_end(m, 1, b);
      all_filtered = done;
      return;
    }
    if (count == 0) return;
    if (off + count > m->capT) {
      over = true;
      return;
    }
    if (v != m->h_tet + 4 * off)
      std::memcpy(m->h_tet + 4 * off, v, (size_t)count * 4 * sizeof(int32_t));
    if (hipMemcpyAsync(m->d_tri + 4 * off, m->h_tet + 4 * off,
                       (size_t)count * 4 * sizeof(int32_t), hipMemcpyHostToDevice,
                       m->stream) != hipSuccess) {
      err = sm_set_error(SM_ERR_HIP, "host_rebuild3d: copy of piece %d failed", piece);
      return;
    }
    off += count;
  };
  // the cells are sorted straight into the pinned staging buffer
  int rc = m->dt3.run(m->h_pts, N, m->sl_axis, m->sl_n, m->sl_threads, emit, m->h_tet, m->capT);
  if (rc) return rc;
  if (err) return err;
  SM_CHECK(!over, SM_ERR_CAPACITY, "host 3D Delaunay: more than %lld tetrahedra",
           (long long)m->capT);
  m->T = off;
  m->stats[3] += 1;
  m->stats[11] = off;
  m->stats[9] += m->dt3.stats.parallel;
  m->stats[10] += m->dt3.stats.retried;
  m->have_tri = true;
  *filtered = all_filtered;
  m->stats[12] += (int64_t)std::chrono::duration_cast<std::chrono::microseconds>(
                      std::chrono::steady_clock::now() - t0)
                      .count();
  return SM_OK;
}

int triangulate(sm_mesher *m) {
  m->nsl = -1;  // a sliver selection refers to the previous cells
  if (m->dim == 3) {
    bool built = false, filtered = false;
    int rc = device_rebuild3d(m, &built);
    if (rc) return rc;
    if (!built && (rc = host_rebuild3d(m, &filtered))) return rc;
    if (!filtered) {
      int b = prof_begin(m);
      rc = centroid_keep(m);
      prof_end(m, 1, b);
      if (rc) return rc;
    }
    return SM_OK;
  }
  bool rebuild = !m->have_tri;
  if (!rebuild) {
    int rc = flip_repair2d(m, 64, &rebuild);
    if (rc) return rc;
  }
  if (rebuild) {
    int rc = host_rebuild2d(m);
    if (rc) return rc;
  }
  int b = prof_begin(m);
  int rc = centroid_keep(m);
  prof_end(m, 1, b);
  return rc;
}

}  // namespace

namespace smk {

int prof_begin(sm_mesher *m) {
  if (!m->prof) return -1;
  // event pairs are handed out in order (phases may nest)
  int idx = m->ev_next;
  m->ev_next += 2;
  while ((int)m->ev_pool.size() < idx + 2) {
    hipEvent_t e;
    if (hipEventCreate(&e) != hipSuccess) return -1;
    m->ev_pool.push_back(e);
  }
  (void)hipEventRecord(m->ev_pool[idx], m->stream);
  return idx;
}

void prof_end(sm_mesher *m, int phase, int begin_idx) {
  if (!m->prof || begin_idx < 0) return;
  (void)hipEventRecord(m->ev_pool[begin_idx + 1], m->stream);
  m->recs.push_back({phase, begin_idx, begin_idx + 1});
}

int prof_drain(sm_mesher *m) {
  if (!m->prof || m->recs.empty()) return SM_OK;
  SM_HIP(hipStreamSynchronize(m->stream));
  for (const auto &r : m->recs) {
    float ms = 0.f;
    SM_HIP(hipEventElapsedTime(&ms, m->ev_pool[r.a], m->ev_pool[r.b]));
    m->prof_ms[r.phase] += ms;
    m->prof_n[r.phase] += 1;
  }
  m->recs.clear();
  m->ev_next = 0;
  return SM_OK;
}

}  // namespace smk

extern "C" int sm_mesher_profile(sm_mesher *m, int enable) {
  SM_CHECK(m, SM_ERR_ARG, "mesher_profile: null handle");
  int rc = prof_drain(m);
  if (rc) return rc;
  m->prof = enable != 0;
  for (int i = 0; i < SM_NPHASES; ++i) {
    m->prof_ms[i] = 0.0;
    m->prof_n[i] = 0;
  }
  return SM_OK;
}

extern "C" int sm_mesher_profile_read(sm_mesher *m, double *ms, int64_t *launches, int n) {
  SM_CHECK(m && ms && launches, SM_ERR_ARG, "mesher_profile_read: null argument");
  int rc = prof_drain(m);
  if (rc) return rc;
  for (int i = 0; i < n && i < SM_NPHASES; ++i) {
    ms[i] = m->prof_ms[i];
    launches[i] = m->prof_n[i];
  }
  return SM_OK;
}

extern "C" int sm_mesher_create(const sm_mesher_params *prm, const sm_node *const *tapes,
                                const int *tape_lens, const sm_grid *sizing,
                                sm_host_sizing_fn host_sizing, void *host_sizing_ctx,
                                int device, sm_mesher **out) {
  SM_CHECK(prm && tapes && tape_lens && sizing && out, SM_ERR_ARG, "mesher_create: null argument");
  SM_CHECK(prm->dim == 2 || prm->dim == 3, SM_ERR_ARG, "mesher_create: dim must be 2 or 3 (got %d)",
           prm->dim);
  SM_CHECK(prm->precision == 32 || prm->precision == 64, SM_ERR_ARG,
           "mesher_create: precision must be 32 or 64");
  SM_CHECK(prm->nlevels >= 1 && prm->nlevels <= 64, SM_ERR_ARG, "mesher_create: bad nlevels");
  SM_HIP(hipSetDevice(device));
  sm_mesher *m = new sm_mesher();
  m->prm = *prm;
  m->dim = prm->dim;
  m->device = device;
  m->host_sizing = host_sizing;
  m->host_sizing_ctx = host_sizing_ctx;
  SM_HIP(hipStreamCreateWithFlags(&m->stream, hipStreamNonBlocking));
  // SDF programs
  int total = 0;
  for (int l = 0; l < prm->nlevels; ++l) {
    SM_CHECK(tapes[l] && tape_lens[l] > 0, SM_ERR_ARG, "mesher_create: empty SDF program");
    m->tape_off.push_back(total);
    m->tape_len.push_back(tape_lens[l]);
    total += tape_lens[l];
    if (tapes[l][0].pad[0] != 0.0) m->deep_sdf = true;
  }
  SM_HIP(hipMalloc(&m->d_tape_all, total * sizeof(sm_node)));
  for (int l = 0; l < prm->nlevels; ++l) {
    SM_HIP(hipMemcpy(m->d_tape_all + m->tape_off[l], tapes[l], tape_lens[l] * sizeof(sm_node),
                     hipMemcpyHostToDevice));
    m->d_tapes.push_back(m->d_tape_all + m->tape_off[l]);
  }
  SM_HIP(hipMalloc(&m->d_tape_off_dev, prm->nlevels * sizeof(int)));
  SM_HIP(hipMalloc(&m->d_tape_len_dev, prm->nlevels * sizeof(int)));
  SM_HIP(hipMemcpy(m->d_tape_off_dev, m->tape_off.data(), prm->nlevels * sizeof(int),
                   hipMemcpyHostToDevice));
  SM_HIP(hipMemcpy(m->d_tape_len_dev, m->tape_len.data(), prm->nlevels * sizeof(int),
                   hipMemcpyHostToDevice));
  // sizing grid
  m->grid.dim = m->dim;
  m->grid.values = nullptr;
  m->grid.hconst = sizing->hconst;
  if (sizing->values) {
    int64_t nv = 1;
    for (int k = 0; k < m->dim; ++k) {
      SM_CHECK(sizing->n[k] >= 2, SM_ERR_ARG, "mesher_create: grid axis %d has < 2 points", k);
      m->grid.n[k] = sizing->n[k];
      nv *= sizing->n[k];
      SM_HIP(hipMalloc(&m->d_axis[k], sizing->n[k] * sizeof(double)));
      SM_HIP(hipMemcpy(m->d_axis[k], sizing->axis[k], sizing->n[k] * sizeof(double),
                       hipMemcpyHostToDevice));
      m->grid.axis[k] = m->d_axis[k];
    }
    SM_HIP(hipMalloc(&m->d_values, nv * sizeof(float)));
    SM_HIP(hipMemcpy(m->d_values, sizing->values, nv * sizeof(float), hipMemcpyHostToDevice));
    m->grid.values = m->d_values;
  }
  SM_HIP(hipMalloc(&m->d_ctr, kCtrTotal * sizeof(int32_t)));
  {
    int rc0 = fill<int32_t>(m->d_ctr, kCtrTotal, 0, m->stream);
    if (rc0) return rc0;
  }
  SM_HIP(hipHostMalloc((void **)&m->h_status, 16 * sizeof(int32_t), hipHostMallocDefault));
  SM_HIP(hipMalloc(&m->d_sums, 4 * sizeof(double)));
  m->d_maxF = reinterpret_cast<uint64_t *>(m->d_ctr + kCtrMaxF);  // inside d_ctr
  SM_HIP(hipHostMalloc((void **)&m->h_ctr, kCtrTotal * sizeof(int32_t), hipHostMallocDefault));
  SM_HIP(hipHostMalloc((void **)&m->h_sums, 4 * sizeof(double), hipHostMallocDefault));
  SM_HIP(hipHostMalloc((void **)&m->h_maxF, sizeof(uint64_t), hipHostMallocDefault));
  *out = m;
  return SM_OK;
}

extern "C" int sm_mesher_create_batch(const sm_mesher_params *prm, int ndom,
                                      const sm_node *const *tapes, const int *tape_lens,
                                      const double *h, const int32_t *nfix,
                                      const int64_t *voff, int device, sm_mesher **out) {
  SM_CHECK(prm && tapes && tape_lens && h && nfix && voff && out, SM_ERR_ARG,
           "mesher_create_batch: null argument");
  SM_CHECK(prm->dim == 2, SM_ERR_ARG, "mesher_create_batch: batches are 2D");
  SM_CHECK(prm->precision == 32, SM_ERR_ARG, "mesher_create_batch: batches use FP32 forces");
  SM_CHECK(ndom >= 1 && ndom <= 65535, SM_ERR_ARG, "mesher_create_batch: bad domain count %d",
           ndom);
  SM_CHECK(voff[0] == 0, SM_ERR_ARG, "mesher_create_batch: voff[0] must be 0");
  for (int d = 0; d < ndom; ++d) {
    SM_CHECK(voff[d + 1] - voff[d] >= 3, SM_ERR_ARG,
             "mesher_create_batch: domain %d has fewer than 3 points", d);
    SM_CHECK(h[d] > 0.0, SM_ERR_ARG, "mesher_create_batch: h of domain %d must be > 0", d);
    SM_CHECK(nfix[d] >= 0 && nfix[d] <= voff[d + 1] - voff[d], SM_ERR_ARG,
             "mesher_create_batch: bad nfix of domain %d", d);
    SM_CHECK(tapes[d] && tape_lens[d] > 0, SM_ERR_ARG, "mesher_create_batch: empty program");
  }
  SM_CHECK(voff[ndom] < (int64_t)1 << 30, SM_ERR_ARG, "mesher_create_batch: too many points");
  // one program per domain takes the place of the levels; sizes are the
  // domains' own
  sm_mesher_params p1 = *prm;
  p1.nlevels = 1;
  p1.nfix = 0;
  sm_grid g{};
  g.dim = 2;
  g.hconst = 1.0;
  int rc = sm_mesher_create(&p1, tapes, tape_lens, &g, nullptr, nullptr, device, out);
  if (rc) return rc;
  sm_mesher *m = *out;
  // replace the level table by the per-domain table
  dfree(m->d_tape_all);
  dfree(m->d_tape_off_dev);
  dfree(m->d_tape_len_dev);
  m->d_tapes.clear();
  m->tape_off.clear();
  m->tape_len.clear();
  m->deep_sdf = false;
  int total = 0;
  for (int d = 0; d < ndom; ++d) {
    m->tape_off.push_back(total);
    m->tape_len.push_back(tape_lens[d]);
    total += tape_lens[d];
    if (tapes[d][0].pad[0] != 0.0) m->deep_sdf = true;
  }
  SM_HIP(hipMalloc(&m->d_tape_all, total * sizeof(sm_node)));
  for (int d = 0; d < ndom; ++d) {
    SM_HIP(hipMemcpy(m->d_tape_all + m->tape_off[d], tapes[d], tape_lens[d] * sizeof(sm_node),
                     hipMemcpyHostToDevice));
    m->d_tapes.push_back(m->d_tape_all + m->tape_off[d]);
  }
  SM_HIP(hipMalloc(&m->d_tape_off_dev, ndom * sizeof(int)));
  SM_HIP(hipMalloc(&m->d_tape_len_dev, ndom * sizeof(int)));
  SM_HIP(hipMemcpy(m->d_tape_off_dev, m->tape_off.data(), ndom * sizeof(int),
                   hipMemcpyHostToDevice));
  SM_HIP(hipMemcpy(m->d_tape_len_dev, m->tape_len.data(), ndom * sizeof(int),
                   hipMemcpyHostToDevice));
  m->ndom = ndom;
  m->h_voff.assign(voff, voff + ndom + 1);
  m->h_dh.assign(h, h + ndom);
  std::vector<int32_t> v32(ndom + 1);
  for (int d = 0; d <= ndom; ++d) v32[d] = (int32_t)voff[d];
  SM_HIP(hipMalloc(&m->d_voff, (ndom + 1) * sizeof(int32_t)));
  SM_HIP(hipMalloc(&m->d_dnfix, ndom * sizeof(int32_t)));
  SM_HIP(hipMalloc(&m->d_dh, ndom * sizeof(double)));
  SM_HIP(hipMalloc(&m->d_dscale, ndom * sizeof(double)));
  SM_HIP(hipMalloc(&m->d_act, 4 * (size_t)ndom * sizeof(int32_t)));
  SM_HIP(hipMemcpy(m->d_voff, v32.data(), (ndom + 1) * sizeof(int32_t), hipMemcpyHostToDevice));
  SM_HIP(hipMemcpy(m->d_dnfix, nfix, ndom * sizeof(int32_t), hipMemcpyHostToDevice));
  SM_HIP(hipMemcpy(m->d_dh, h, ndom * sizeof(double), hipMemcpyHostToDevice));
  return SM_OK;
}

extern "C" int sm_mesher_destroy(sm_mesher *m) {
  if (!m) return SM_OK;
  (void)hipSetDevice(m->device);
  if (m->stream) (void)hipStreamSynchronize(m->stream);
  free_point_state(m);
  dfree(m->d_tape_all);
  dfree(m->d_tape_off_dev);
  dfree(m->d_tape_len_dev);
  dfree(m->d_voff);
  dfree(m->d_dnfix);
  dfree(m->d_dh);
  dfree(m->d_dscale);
  dfree(m->d_act);
  dfree(m->d_dfail);
  for (int k = 0; k < 3; ++k) dfree(m->d_axis[k]);
  dfree(m->d_values);
  dfree(m->d_ctr);
  dfree(m->d_sums);
  dfree(m->d_sg);
  dfree(m->d_tctr);
  if (m->h_ctr) (void)hipHostFree(m->h_ctr);
  if (m->h_status) (void)hipHostFree(m->h_status);
  if (m->h_sums) (void)hipHostFree(m->h_sums);
  if (m->h_maxF) (void)hipHostFree(m->h_maxF);
  dfree(m->d_bands);
  if (m->h_pts) (void)hipHostFree(m->h_pts);
  if (m->h_tet) (void)hipHostFree(m->h_tet);
  stars_free(&m->stars);
  for (hipEvent_t e : m->ev_pool) (void)hipEventDestroy(e);
  if (m->stream) (void)hipStreamDestroy(m->stream);
  delete m;
  return SM_OK;
}

extern "C" int sm_mesher_set_points(sm_mesher *m, const double *p, int64_t n) {
  SM_CHECK(m && p && n > 0, SM_ERR_ARG, "mesher_set_points: bad argument");
  SM_HIP(hipSetDevice(m->device));
  if (n != m->capN) {
    int rc = alloc_point_state(m, n);
    if (rc) return rc;
  }
  if (m->ndom > 0)
    SM_CHECK(n == m->h_voff[m->ndom], SM_ERR_ARG,
             "mesher_set_points: a batch of %d domains holds %lld points (got %lld)", m->ndom,
             (long long)m->h_voff[m->ndom], (long long)n);
  m->N = n;
  m->NA = n + m->nfar;
  m->stars.skip = 0;  // what failed on other points says nothing about these
  SM_HIP(hipMemcpyAsync(m->d_p, p, n * m->dim * sizeof(double), hipMemcpyHostToDevice,
                        m->stream));
  m->have_tri = false;
  if (m->nfar > 0) {
    // far square of each domain (of the whole point set for one domain)
    const int nd = std::max(m->ndom, 1);
    std::vector<double> far((size_t)m->nfar * 2);
    std::vector<int32_t> fdom((size_t)m->nfar);
    for (int d = 0; d < nd; ++d) {
      const int64_t b = m->ndom > 0 ? m->h_voff[d] : 0, e = m->ndom > 0 ? m->h_voff[d + 1] : n;
      double lo[2] = {p[2 * b], p[2 * b + 1]}, hi[2] = {lo[0], lo[1]};
      for (int64_t i = b; i < e; ++i)
        for (int k = 0; k < 2; ++k) {
          lo[k] = std::min(lo[k], p[2 * i + k]);
          hi[k] = std::max(hi[k], p[2 * i + k]);
        }
      const double ext = std::max(std::max(hi[0] - lo[0], hi[1] - lo[1]), 1e-300);
      const double c[2] = {(lo[0] + hi[0]) / 2, (lo[1] + hi[1]) / 2};
      const double K = kFarSquare * ext;
      const double sx[4] = {-1, 1, 1, -1}, sy[4] = {-1, -1, 1, 1};
      for (int k = 0; k < 4; ++k) {
        far[2 * (4 * d + k)] = c[0] + K * sx[k];
        far[2 * (4 * d + k) + 1] = c[1] + K * sy[k];
        fdom[4 * d + k] = d;
      }
    }
    SM_HIP(hipMemcpy(m->d_p + 2 * n, far.data(), far.size() * sizeof(double),
                     hipMemcpyHostToDevice));
    if (m->ndom > 0)
      SM_HIP(hipMemcpy(m->d_vdom + n, fdom.data(), fdom.size() * sizeof(int32_t),
                       hipMemcpyHostToDevice));
  }
  if (m->ndom > 0) {
    hipLaunchKernelGGL(k_vertex_domains, dim3(64, m->ndom), dim3(256), 0, m->stream, m->ndom,
                       m->d_voff, m->d_vdom);
    SM_LAUNCH_CHECK();
  }
  // 3D rebuilds its tetrahedralisation at every triangulate()
  int rc = m->dim == 2 ? host_rebuild2d(m) : SM_OK;
  if (rc) return rc;
  return SM_OK;
}

extern "C" int sm_mesher_triangulate(sm_mesher *m) {
  SM_CHECK(m && m->N > 0, SM_ERR_STATE, "mesher_triangulate: no points");
  SM_HIP(hipSetDevice(m->device));
  int rc = triangulate(m);
  if (rc) return rc;
  // the edge list then describes the current triangulation too
  if ((rc = build_edges(m, true))) return rc;
  SM_HIP(hipStreamSynchronize(m->stream));
  return SM_OK;
}

namespace {

// mesh_generator.py:513-521: max movement and the divergence assertion
int check_movement(sm_mesher *m) {
  double mf;
  std::memcpy(&mf, m->h_maxF, sizeof(double));
  m->last_maxdp = m->prm.delta_t * mf;
  // batches record the movement in units of each domain's h0
  const double h0 = m->ndom > 0 ? 1.0 : m->prm.h0;
  if (!(m->last_maxdp < 1000.0 * h0))
    return sm_set_error(SM_ERR_NUMERIC,
                        "max movement indicates there's a convergence problem (%g)",
                        m->last_maxdp);
  return SM_OK;
}

// The second half of an iteration on a valid triangulation.
int edges_forces_update(sm_mesher *m) {
  int rc;
  const bool sync = m->prm.precision == 64 || m->host_sizing != nullptr || m->dim == 3;
  int pb = prof_begin(m);
  if ((rc = build_edges(m, sync))) return rc;
  prof_end(m, 2, pb);
  if (m->host_sizing && (rc = host_sizing_pass(m))) return rc;
  if ((rc = forces_and_update(m))) return rc;
  SM_HIP(hipMemcpyAsync(m->h_maxF, m->d_maxF, sizeof(uint64_t), hipMemcpyDeviceToHost,
                        m->stream));
  return SM_OK;
}

// One iteration with host decisions between the stages.
int iterate_plain(sm_mesher *m) {
  int rc;
  if ((rc = triangulate(m))) return rc;
  if ((rc = edges_forces_update(m))) return rc;
  SM_HIP(hipStreamSynchronize(m->stream));
  m->stats[0] += 1;
  return check_movement(m);
}

constexpr int kGraphRounds = 5;

// Captures one whole FP32 iteration: snapshot of the points, a batch of flip
// rounds (later rounds skip themselves once a round flips nothing),
// centroid filter, edges, forces, update and projection, then copies of the
// flip status and the max movement to pinned host memory.
int capture_iteration(sm_mesher *m) {
  if (m->gexec) {
    (void)hipGraphExecDestroy(m->gexec);
    m->gexec = nullptr;
  }
  if (m->graph) {
    (void)hipGraphDestroy(m->graph);
    m->graph = nullptr;
  }
  hipStream_t s = m->stream;
  const bool prof = m->prof;
  m->prof = false;
  SM_HIP(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
  int rc = SM_OK;
  do {
    if ((rc = enqueue_flip_rounds(m, kGraphRounds, m->d_ctr + kCtrStatus, m->d_p, false)))
      break;
    // the points do not move before the update: the snapshot kernel also
    // keeps them for a rollback (d_psnap, NA x 2 doubles: graphs are 2D)
    if ((rc = enqueue_snapshot(m, m->d_ctr + kCtrStatus, m->d_psnap))) break;
    if ((rc = centroid_keep(m))) break;
    if ((rc = build_edges(m, false))) break;
    if ((rc = forces_and_update(m))) break;
    // h_status[0..1]: the movement maximum, h_status[2..9]: the status
    if (hipMemcpyAsync(m->h_status, m->d_ctr + kCtrMaxF, 10 * sizeof(int32_t),
                       hipMemcpyDeviceToHost, s) != hipSuccess) {
      rc = sm_set_error(SM_ERR_HIP, "capture: status copy failed");
      break;
    }
  } while (false);
  hipGraph_t g = nullptr;
  hipError_t e = hipStreamEndCapture(s, &g);
  m->prof = prof;
  if (rc) {
    if (g) (void)hipGraphDestroy(g);
    return rc;
  }
  if (e != hipSuccess) return sm_set_error(SM_ERR_HIP, "capture failed: %s", hipGetErrorString(e));
  m->graph = g;
  SM_HIP(hipGraphInstantiate(&m->gexec, g, nullptr, nullptr, 0));
  m->graph_T = m->T;
  return SM_OK;
}

// One iteration as a single graph launch and one synchronisation.  The
// iteration runs speculatively on whatever triangulation the captured flip
// rounds reach; when they did not reach a valid Delaunay triangulation the
// points are restored from the snapshot and the iteration is redone with
// host decisions (more flip rounds, or an exact rebuild).
int iterate_graph(sm_mesher *m) {
  int rc;
  if (!m->gexec || m->graph_T != m->T) {
    if ((rc = capture_iteration(m))) return rc;
  }
  SM_HIP(hipGraphLaunch(m->gexec, m->stream));
  SM_HIP(hipStreamSynchronize(m->stream));
  const int32_t *st = m->h_status + 2;
  std::memcpy(m->h_maxF, m->h_status, sizeof(uint64_t));
  account_flips(m, st);
  const bool valid = st[2] && st[3] == 0 && st[4] == 0;
  if (valid) {
    m->stats[0] += 1;
    return check_movement(m);
  }
  m->stats[5] += 1;  // speculative iteration rolled back
  SM_HIP(hipMemcpyAsync(m->d_p, m->d_psnap, m->NA * m->dim * sizeof(double),
                        hipMemcpyDeviceToDevice, m->stream));
  // more flip rounds (settling uncertain predicates exactly, which the
  // captured rounds leave to this path) or a kinetic repair from the last
  // valid state; the host rebuilds when those fail
  bool rebuild = false;
  if ((rc = flip_repair2d(m, 64, &rebuild))) return rc;
  if (rebuild && (rc = host_rebuild2d(m))) return rc;
  if ((rc = centroid_keep(m))) return rc;
  if ((rc = edges_forces_update(m))) return rc;
  SM_HIP(hipStreamSynchronize(m->stream));
  m->stats[0] += 1;
  return check_movement(m);
}

}  // namespace

extern "C" int sm_mesher_run(sm_mesher *m, int iters, double *maxdp_out) {
  SM_CHECK(m && m->N > 0, SM_ERR_STATE, "mesher_run: no points");
  SM_CHECK(iters >= 0, SM_ERR_ARG, "mesher_run: negative iteration count");
  SM_HIP(hipSetDevice(m->device));
  // the graph path needs a device-only iteration: FP32 forces, sizing on
  // the device, and no per-kernel event timing
  const bool graph = m->dim == 2 && m->prm.precision == 32 && !m->host_sizing &&
                     !m->host_sdf && !m->prof && m->have_tri && m->use_graph;
  for (int it = 0; it < iters; ++it) {
    int rc = graph ? iterate_graph(m) : iterate_plain(m);
    if (rc) return rc;
  }
  if (maxdp_out) *maxdp_out = m->last_maxdp;
  return prof_drain(m);
}

extern "C" int sm_mesher_set_host_sdf(sm_mesher *m, sm_host_sdf_fn fn, void *ctx) {
  SM_CHECK(m, SM_ERR_ARG, "mesher_set_host_sdf: null handle");
  SM_CHECK(m->ndom == 0, SM_ERR_STATE, "mesher_set_host_sdf: not for batch handles");
  SM_CHECK(!fn || !m->surrogate, SM_ERR_STATE,
           "mesher_set_host_sdf: a surrogate is set (it needs the device programs)");
  m->host_sdf = fn;
  m->host_sdf_ctx = fn ? ctx : nullptr;
  return SM_OK;
}

extern "C" int sm_mesher_set_graph(sm_mesher *m, int enable) {
  SM_CHECK(m, SM_ERR_ARG, "mesher_set_graph: null handle");
  m->use_graph = enable != 0;
  return SM_OK;
}

extern "C" int sm_mesher_sizes(sm_mesher *m, int64_t *npoints, int64_t *ncells,
                               int64_t *nedges) {
  SM_CHECK(m, SM_ERR_ARG, "mesher_sizes: null handle");
  SM_HIP(hipSetDevice(m->device));
  SM_HIP(hipStreamSynchronize(m->stream));
  if (m->d_ctr) {
    // the edge count lives on the device (the graph path never reads it back)
    int32_t e = 0;
    SM_HIP(hipMemcpy(&e, m->d_ctr + kCtrE, sizeof(int32_t), hipMemcpyDeviceToHost));
    m->E = e;
  }
  if (npoints) *npoints = m->N;
  if (nedges) *nedges = m->E;
  if (ncells) {
    std::vector<uint8_t> keep((size_t)std::max<int64_t>(m->T, 1));
    SM_HIP(hipMemcpy(keep.data(), m->d_keep, m->T, hipMemcpyDeviceToHost));
    int64_t c = 0;
    for (int64_t t = 0; t < m->T; ++t) c += keep[t] != 0;
    *ncells = c;
  }
  return SM_OK;
}

extern "C" int sm_mesher_get_points(sm_mesher *m, double *p, int64_t cap) {
  SM_CHECK(m && p && cap >= m->N, SM_ERR_CAPACITY, "mesher_get_points: buffer too small");
  SM_HIP(hipSetDevice(m->device));
  SM_HIP(hipStreamSynchronize(m->stream));
  SM_HIP(hipMemcpy(p, m->d_p, m->N * m->dim * sizeof(double), hipMemcpyDeviceToHost));
  return SM_OK;
}

extern "C" int sm_mesher_get_cells(sm_mesher *m, int32_t *cells, int64_t cap) {
  SM_CHECK(m && cells, SM_ERR_ARG, "mesher_get_cells: null argument");
  SM_HIP(hipSetDevice(m->device));
  SM_HIP(hipStreamSynchronize(m->stream));
  const int k = m->dim + 1;
  std::vector<uint8_t> keep((size_t)std::max<int64_t>(m->T, 1));
  std::vector<int32_t> tri((size_t)std::max<int64_t>(m->T, 1) * k);
  SM_HIP(hipMemcpy(keep.data(), m->d_keep, m->T, hipMemcpyDeviceToHost));
  SM_HIP(hipMemcpy(tri.data(), m->d_tri, m->T * k * sizeof(int32_t), hipMemcpyDeviceToHost));
  int64_t c = 0;
  for (int64_t t = 0; t < m->T; ++t) {
    if (!keep[t]) continue;
    SM_CHECK(c < cap, SM_ERR_CAPACITY, "mesher_get_cells: buffer too small");
    for (int j = 0; j < k; ++j) cells[c * k + j] = tri[t * k + j];
    ++c;
  }
  return SM_OK;
}

extern "C" int64_t sm_mesher_get_triangulation(sm_mesher *m, int32_t *tri, int32_t *adj,
                                               int64_t cap) {
  SM_CHECK(m && tri && adj, SM_ERR_ARG, "mesher_get_triangulation: null argument");
  SM_CHECK(m->dim == 2 && m->have_tri, SM_ERR_STATE,
           "mesher_get_triangulation: needs a 2D handle with a triangulation");
  SM_CHECK(cap >= m->T, SM_ERR_CAPACITY, "mesher_get_triangulation: buffer too small");
  SM_HIP(hipSetDevice(m->device));
  SM_HIP(hipStreamSynchronize(m->stream));
  SM_HIP(hipMemcpy(tri, m->d_tri, m->T * 3 * sizeof(int32_t), hipMemcpyDeviceToHost));
  SM_HIP(hipMemcpy(adj, m->d_adj, m->T * 3 * sizeof(int32_t), hipMemcpyDeviceToHost));
  return m->T;
}

extern "C" int sm_mesher_get_edges(sm_mesher *m, int32_t *edges, int64_t cap) {
  SM_CHECK(m && edges && cap >= m->E, SM_ERR_CAPACITY, "mesher_get_edges: buffer too small");
  SM_HIP(hipSetDevice(m->device));
  SM_HIP(hipStreamSynchronize(m->stream));
  SM_HIP(hipMemcpy(edges, m->d_edges, m->E * 2 * sizeof(int32_t), hipMemcpyDeviceToHost));
  return SM_OK;
}

extern "C" int sm_mesher_stats(sm_mesher *m, int64_t *stats, int nstats) {
  SM_CHECK(m && stats, SM_ERR_ARG, "mesher_stats: null argument");
  for (int i = 0; i < nstats && i < kNumStats; ++i) stats[i] = m->stats[i];
  return SM_OK;
}

extern "C" int sm_mesher_set_scratch_limit(sm_mesher *m, int64_t bytes) {
  SM_CHECK(m && bytes >= 0, SM_ERR_ARG, "mesher_set_scratch_limit: bad argument");
  SM_CHECK(m->dim == 3, SM_ERR_ARG, "mesher_set_scratch_limit: 3D handles only");
  m->stars.max_bytes = bytes == 0 ? SIZE_MAX : (size_t)bytes;
  m->stars.skip = 0;
  return SM_OK;
}

extern "C" int sm_mesher_set_slabs(sm_mesher *m, int axis, int nslabs, int nthreads) {
  SM_CHECK(m, SM_ERR_ARG, "mesher_set_slabs: null handle");
  SM_CHECK(m->dim == 3, SM_ERR_ARG, "mesher_set_slabs: slabs split the 3D tetrahedralisation");
  SM_CHECK(axis >= 0 && axis < 3, SM_ERR_ARG, "mesher_set_slabs: axis must be 0, 1 or 2");
  SM_CHECK(nslabs >= 1 && nslabs <= 4096, SM_ERR_ARG, "mesher_set_slabs: bad slab count %d",
           nslabs);
  SM_CHECK(nthreads >= 1 && nthreads <= 1024, SM_ERR_ARG, "mesher_set_slabs: bad thread count");
  m->sl_axis = axis;
  m->sl_n = nslabs;
  m->sl_threads = nthreads;
  return SM_OK;
}

extern "C" int sm_mesher_set_surrogate_bands(sm_mesher *m, int res, const double *lo,
                                             const double *hi, const float *bands) {
  SM_CHECK(m, SM_ERR_ARG, "mesher_set_surrogate_bands: null handle");
  SM_HIP(hipSetDevice(m->device));
  SM_HIP(hipStreamSynchronize(m->stream));
  dfree(m->d_bands);
  m->band_res = 0;
  m->band_max = 0.0;
  if (!bands) return SM_OK;
  SM_CHECK(lo && hi && res >= 1 && res <= 512, SM_ERR_ARG,
           "mesher_set_surrogate_bands: bad grid (res %d)", res);
  int64_t cells = 1;
  for (int k = 0; k < m->dim; ++k) {
    SM_CHECK(hi[k] > lo[k], SM_ERR_ARG, "mesher_set_surrogate_bands: empty box on axis %d", k);
    m->band_lo[k] = lo[k];
    m->band_inv[k] = res / (hi[k] - lo[k]);
    cells *= res;
  }
  double vmax = 0.0;
  for (int64_t i = 0; i < cells; ++i) {
    SM_CHECK(bands[i] >= 0.0f, SM_ERR_ARG, "mesher_set_surrogate_bands: negative band");
    vmax = std::max(vmax, (double)bands[i]);
  }
  int rc = dalloc(&m->d_bands, cells);
  if (rc) return rc;
  SM_HIP(hipMemcpy(m->d_bands, bands, cells * sizeof(float), hipMemcpyHostToDevice));
  m->band_res = res;
  m->band_max = vmax;
  return SM_OK;
}

extern "C" int sm_mesher_set_surrogate(sm_mesher *m, const sm_mlp *net, double band) {
  SM_CHECK(m, SM_ERR_ARG, "mesher_set_surrogate: null handle");
  SM_HIP(hipSetDevice(m->device));
  if (!net) {
    m->surrogate = false;
  } else {
    int rc = mlp_check(net);
    if (rc) return rc;
    SM_CHECK(net->in_dim == m->dim, SM_ERR_ARG, "mesher_set_surrogate: network takes %dD points",
             net->in_dim);
    SM_CHECK(band > 0.0, SM_ERR_ARG, "mesher_set_surrogate: band must be positive");
    SM_CHECK(!m->host_sdf, SM_ERR_STATE,
             "mesher_set_surrogate: the handle's SDF is a host function");
    SM_CHECK(m->ndom == 0 && m->prm.nlevels == 1 && !m->host_sizing, SM_ERR_STATE,
             "mesher_set_surrogate: single-domain handles without subdomains only");
    m->net = *net;
    m->band = band;
    m->surrogate = true;
    if (!m->d_sg) {
      int rc2 = dalloc(&m->d_sg, 4);
      if (rc2) return rc2;
    }
    int rc3 = fill<uint64_t>(m->d_sg, 4, 0ull, m->stream);
    if (rc3) return rc3;
    const int64_t need = std::max(m->capT, m->NA);
    if (m->capN > 0 && m->dnn_cap < need) {
      dfree(m->d_dnn);
      m->dnn_cap = need;
      int rc4 = dalloc(&m->d_dnn, need);
      if (rc4) return rc4;
    }
  }
  // the captured iteration no longer matches the kernels to run
  if (m->gexec) (void)hipGraphExecDestroy(m->gexec);
  if (m->graph) (void)hipGraphDestroy(m->graph);
  m->gexec = nullptr;
  m->graph = nullptr;
  m->graph_T = -1;
  return SM_OK;
}

extern "C" int sm_mesher_time_kernel(sm_mesher *m, int phase, int reps, double *ms) {
  SM_CHECK(m && ms, SM_ERR_ARG, "mesher_time_kernel: null argument");
  SM_CHECK(phase == 7, SM_ERR_ARG, "mesher_time_kernel: only phase 7 (flip marking) is timed");
  SM_HIP(hipSetDevice(m->device));
  SM_HIP(hipStreamSynchronize(m->stream));
  return time_flip_mark(m, reps, ms);
}

extern "C" int sm_mesher_autotune(sm_mesher *m, int reps, int32_t *chosen, double *ms,
                                  int nk) {
  SM_CHECK(m && reps >= 1, SM_ERR_ARG, "mesher_autotune: bad argument");
  SM_CHECK(m->have_tri && m->stats[0] > 0, SM_ERR_STATE,
           "mesher_autotune: run at least one iteration first (edges and forces are timed "
           "on the current state)");
  SM_CHECK(!m->host_sdf, SM_ERR_STATE,
           "mesher_autotune: the centroid filter of a host-function domain runs on the host");
  SM_HIP(hipSetDevice(m->device));
  SM_HIP(hipStreamSynchronize(m->stream));
  static const int cand[] = {64, 128, 256, 512, 1024};
  for (int k = 0; k < kNumBlk; ++k) {
    const bool flip = k == kBlkOrient || k == kBlkMark || k == kBlkApply;
    if (flip && m->dim != 2) continue;
    int best_b = 256;
    double best = 0.0, t256 = 0.0;
    int rc = flip ? time_flip_tunable(m, k, 256, reps, &t256)
                  : time_force_tunable(m, k, 256, reps, &t256);
    if (rc) return rc;
    best = t256;
    for (int b : cand) {
      if (b == 256) continue;
      double t = 0.0;
      rc = flip ? time_flip_tunable(m, k, b, reps, &t) : time_force_tunable(m, k, b, reps, &t);
      if (rc) return rc;
      // another size must beat the default by 3 % (timing noise)
      if (t < best && t < 0.97 * t256) {
        best = t;
        best_b = b;
      }
    }
    m->blk[k] = best_b;
    if (ms && k < nk) ms[k] = best;
  }
  if (chosen)
    for (int k = 0; k < kNumBlk && k < nk; ++k) chosen[k] = m->blk[k];
  // the captured iteration used the old sizes
  if (m->gexec) (void)hipGraphExecDestroy(m->gexec);
  if (m->graph) (void)hipGraphDestroy(m->graph);
  m->gexec = nullptr;
  m->graph = nullptr;
  m->graph_T = -1;
  return SM_OK;
}

extern "C" int sm_mesher_set_workgroups(sm_mesher *m, const int32_t *sizes, int nk) {
  SM_CHECK(m && sizes && nk == kNumBlk, SM_ERR_ARG,
           "mesher_set_workgroups: need %d sizes", kNumBlk);
  for (int k = 0; k < kNumBlk; ++k)
    SM_CHECK(sizes[k] >= 64 && sizes[k] <= 1024 && sizes[k] % 64 == 0, SM_ERR_ARG,
             "mesher_set_workgroups: size %d of kernel %d is not a multiple of 64 in "
             "[64, 1024]", sizes[k], k);
  for (int k = 0; k < kNumBlk; ++k) m->blk[k] = sizes[k];
  if (m->gexec) (void)hipGraphExecDestroy(m->gexec);
  if (m->graph) (void)hipGraphDestroy(m->graph);
  m->gexec = nullptr;
  m->graph = nullptr;
  m->graph_T = -1;
  return SM_OK;
}

extern "C" int sm_mesher_surrogate_stats(sm_mesher *m, int64_t *skipped, int64_t *exact,
                                         double *max_err) {
  SM_CHECK(m && skipped && exact && max_err, SM_ERR_ARG, "mesher_surrogate_stats: null argument");
  SM_CHECK(m->d_sg, SM_ERR_STATE, "mesher_surrogate_stats: no surrogate was set");
  uint64_t v[4];
  SM_HIP(hipMemcpyAsync(v, m->d_sg, sizeof(v), hipMemcpyDeviceToHost, m->stream));
  SM_HIP(hipStreamSynchronize(m->stream));
  *skipped = (int64_t)v[0];
  *exact = (int64_t)v[1];
  std::memcpy(max_err, &v[2], sizeof(double));
  return SM_OK;
}

extern "C" int sm_mesher_device_points(sm_mesher *m, double **p) {
  SM_CHECK(m && p, SM_ERR_ARG, "mesher_device_points: null argument");
  *p = m->d_p;
  return SM_OK;
}

extern "C" int sm_mesher_stream(sm_mesher *m, void **stream) {
  SM_CHECK(m && stream, SM_ERR_ARG, "mesher_stream: null argument");
  *stream = (void *)m->stream;
  return SM_OK;
}
