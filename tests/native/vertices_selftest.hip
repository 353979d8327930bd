// Self-test entry point of the vertex finder (csrc/kern_vertex.hip) on tracks the caller
// makes up, for tests/test_gpu_vertices.py.  Test support only; the reconstruction library
// does not load it.
#include <vector>

#include "../../pixeltrack-standalone_amd/csrc/kern_vertex.hip"

// One event of nt tracks (host arrays), each a loose tuple of four hits; the outputs are
// host arrays of nt (idv, ndof) and 1024 entries.  Returns the number of vertices.
extern "C" int pxs_vertices(uint32_t nt, const float* z, const float* ez2, const float* pt, int algo, int16_t* idv,
                            int32_t* ndof, float* zv, float* wv, float* chi2, float* ptv2, uint16_t* sortInd) {
  using namespace pxg;
  const uint32_t M = (nt + 63) / 64 * 64 + 64;
  std::vector<void*> owned;
  bool ok = true;
  auto alloc = [&](auto*& p, size_t n) {
    void* q = nullptr;
    ok = ok && hipMalloc(&q, n * sizeof(*p)) == hipSuccess && hipMemset(q, 0, n * sizeof(*p)) == hipSuccess;
    owned.push_back(q);
    p = static_cast<std::remove_reference_t<decltype(p)>>(q);
  };
  auto up = [&](auto* d, const auto* s, size_t n) {
    ok = ok && hipMemcpy(d, s, n * sizeof(*s), hipMemcpyHostToDevice) == hipSuccess;
  };
  auto down = [&](auto* d, const auto* s, size_t n) {
    ok = ok && hipMemcpy(d, s, n * sizeof(*s), hipMemcpyDeviceToHost) == hipSuccess;
  };
  CAPool ca{};
  ca.caps = {M, M, M, M, M, 128};
  alloc(ca.cnt, 1);
  alloc(ca.tupleOff, M + 64);
  alloc(ca.quality, M);
  alloc(ca.state, 5 * size_t(M));
  alloc(ca.cov, 15 * size_t(M));
  alloc(ca.pt, M);
  alloc(ca.idv, M);
  alloc(ca.ndof, M);
  alloc(ca.zv, kMaxVertices);
  alloc(ca.wv, kMaxVertices);
  alloc(ca.vchi2, kMaxVertices);
  alloc(ca.ptv2, kMaxVertices);
  alloc(ca.sortInd, kMaxVertices);
  alloc(ca.vItrk, M);
  alloc(ca.vZt, M);
  alloc(ca.vEzt2, M);
  alloc(ca.vPtt2, M);
  alloc(ca.vIv, M);
  alloc(ca.vTmp, M);
  alloc(ca.vZE, M);
  alloc(ca.vNnS, M);
  alloc(ca.vMask, M / 64);
  alloc(ca.vTrk, M);
  alloc(ca.vPerm, M);
  alloc(ca.vTerm, M);
  alloc(ca.vOff, kMaxVertices + 64);
  CACounts c{};
  if (ok) {
    c.nTuples = nt;
    std::vector<uint32_t> off(M + 64);
    for (uint32_t t = 0; t < M + 64; ++t)
      off[t] = 4 * (t < nt ? t : nt);
    const std::vector<uint8_t> loose(nt, uint8_t(kQualityLoose));
    up(ca.cnt, &c, 1);
    up(ca.tupleOff, off.data(), off.size());
    up(ca.quality, loose.data(), nt);
    up(ca.state + 4 * size_t(M), z, nt);
    up(ca.cov + 14 * size_t(M), ez2, nt);
    up(ca.pt, pt, nt);
    CALaunch l{};
    Timer timer;
    l.ca = &ca;
    l.nEvents = 1;
    l.blocks = 8;
    l.t = &timer;
    l.vertexAlgo = algo;
    l.vertexPtMin = 0.f;
    launchVertices(l);
    ok = hipDeviceSynchronize() == hipSuccess && hipGetLastError() == hipSuccess;
    down(&c, ca.cnt, 1);
    down(idv, ca.idv, nt);
    down(ndof, ca.ndof, nt);
    down(zv, ca.zv, kMaxVertices);
    down(wv, ca.wv, kMaxVertices);
    down(chi2, ca.vchi2, kMaxVertices);
    down(ptv2, ca.ptv2, kMaxVertices);
    down(sortInd, ca.sortInd, kMaxVertices);
  }
  for (void* p : owned)
    (void)hipFree(p);
  return ok ? int(c.nVertices) : -1;
}
