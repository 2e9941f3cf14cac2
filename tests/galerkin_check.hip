// The AMG set-up's Galerkin kernel on arrays of a test: one call per launch,
// with the lanes per pair given.  Built into a library of its own beside the
// product's; test_gpu_galerkin.py drives it.
#include "../lowlevelfem.jl_amd/csrc/amg.hip"

using namespace llfem;

extern "C" __attribute__((visibility("default"))) int galerkin_check(
    int lanes, int64_t npairs, int64_t nfine, int64_t nadjf, int64_t nadjc, int64_t ncontrib, const int64_t* gptr,
    const int32_t* gblk, const int32_t* gcol, const int32_t* adjf, const float* Qf, const float* valf,
    const int32_t* pair_o, float* valc) {
  // every index the kernel follows stays inside its array
  if ((lanes != 16 && lanes != 64) || npairs < 1 || gptr[0] != 0 || gptr[npairs] != ncontrib) return 1;
  for (int64_t p = 0; p < npairs; ++p)
    if (gptr[p + 1] < gptr[p] || pair_o[2 * p] < 0 || pair_o[2 * p] + 1 >= nadjc || pair_o[2 * p + 1] < 0 ||
        pair_o[2 * p + 1] + 1 >= nadjc)
      return 1;
  for (int64_t c = 0; c < ncontrib; ++c)
    if (gblk[c] < 0 || gblk[c] >= nadjf || gcol[c] < 0 || gcol[c] >= nfine) return 1;
  for (int64_t g = 0; g < nadjf; ++g)
    if (adjf[g] < 0 || adjf[g] >= nfine) return 1;
  std::vector<void*> mem;
  hipError_t e = hipSuccess;
  auto up = [&](const void* src, size_t bytes) -> void* {
    void* p = nullptr;
    if (e == hipSuccess) e = hipMalloc(&p, bytes + 16);
    if (e == hipSuccess) mem.push_back(p);
    if (e == hipSuccess) e = hipMemcpy(p, src, bytes, hipMemcpyHostToDevice);
    return p;
  };
  const auto* d_gptr = (const int64_t*)up(gptr, 8 * (npairs + 1));
  const auto* d_gblk = (const int32_t*)up(gblk, 4 * ncontrib);
  const auto* d_gcol = (const int32_t*)up(gcol, 4 * ncontrib);
  const auto* d_adjf = (const int32_t*)up(adjf, 4 * nadjf);
  const auto* d_Qf = (const float*)up(Qf, 4 * 18 * nfine);
  const auto* d_valf = (const float*)up(valf, 4 * 9 * nadjf);
  const auto* d_pair_o = (const int32_t*)up(pair_o, 8 * npairs);
  float* d_valc = (float*)up(valc, 4 * 9 * nadjc);
  if (e == hipSuccess) {
    if (lanes == 64)
      k_galerkin<64><<<nblk(64 * npairs), kMB>>>(npairs, nadjf, nadjc, d_gptr, d_gblk, d_gcol, d_adjf, d_Qf, d_valf,
                                                 d_pair_o, d_valc);
    else
      k_galerkin<16><<<nblk(16 * npairs), kMB>>>(npairs, nadjf, nadjc, d_gptr, d_gblk, d_gcol, d_adjf, d_Qf, d_valf,
                                                 d_pair_o, d_valc);
    e = hipGetLastError();
    if (e == hipSuccess) e = hipMemcpy(valc, d_valc, 4 * 9 * nadjc, hipMemcpyDeviceToHost);
  }
  for (void* p : mem) (void)hipFree(p);
  return e == hipSuccess ? 0 : 2;
}
