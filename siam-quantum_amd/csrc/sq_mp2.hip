// sq_mp2.hip - MP2 energy (closed and open shell) from the dense AO pair
// matrix, by four quarter transforms.
//
// Input: V[P][Q] = (pq|rs) for the packed pairs P = pair(p,q), Q = pair(r,s)
// (n(n+1)/2 on a side, symmetric, written by the integral-store kernels), the
// correlated occupied orbitals Co (n x nc) and the virtual orbitals Cv
// (n x nv), column-major with leading dimension n (the reference's
// orbital-major C[k*n + i]), and their orbital energies.
//
// Every quarter transform is one DGEMM whose long dimension is the index
// that it leaves alone, so that its operands are dense column-major blocks:
//
// First half, per block of ket pairs j (bc of them): gather the columns j of
// V into Vf[q][p][j] (rows of V, contiguous in j), then
//   T[q][a][j] = sum_p Vf[q][p][j] Co[p,a]     batched over q
//   X[r][a][j] = sum_q T[q][a][j] Cv[q,r]      one DGEMM, rows (j, a)
// so a block of X holds (ar|j) with j fastest.  Second half, per block of bra
// virtual orbitals r (rows x = (a,r), B of them): turn X over to
// Xf[m][l][x] (pairs j = (l,m) unpacked, x fastest), then
//   U[m][b][x] = sum_l Xf[m][l][x] Co[l,b]     batched over m
//   Y[s][b][x] = sum_m U[m][b][x] Cv[m,s]      one DGEMM, rows (x, b)
// and sum the energy from Y = (ar|bs).  Operations: n^2/2 (ov) n o for the
// third quarter and n (ov) o v / 2 for the fourth, where contracting both ket
// indices in one product costs n^2/2 (ov)^2 / 2 (30 times as many at
// (H2O)16/6-31G*: 170 ms of DGEMM at 63 TFLOP/s, now 9 ms).
//
// The energy
//   E2 = sum_{a,b,r,s} (ar|bs) [2 (ar|bs) - (as|br)] / (e_a + e_b - e_r - e_s)
// has the same (r,s) and (s,r) terms (swap a<->b, r<->s), so a block of r
// needs s <= r only, and (as|br) = (br|as) is Y[s][a][(b,r)], in the same
// block.
#include <hip/hip_runtime.h>
#include <rocblas/rocblas.h>

#include <algorithm>
#include <cmath>
#include <string>
#include <vector>

#include "sq_internal.h"

namespace {

// Vf[q][p][t] = Vf[p][q][t] = V[pair(p,q)][j0 + t], t < bc: one workgroup per
// pair, its row read once and written twice, both contiguous in t.  Bound by
// memory (17 GB read, 34 GB written at (H2O)16/6-31G*).
__global__ void __launch_bounds__(256) k_gather(const double* __restrict__ V, size_t npr, size_t j0, int bc, int n,
                                                const int2* __restrict__ lm, double* __restrict__ Vf) {
  const size_t P = blockIdx.x;
  const int2 t = lm[P];
  const double* row = V + P * npr + j0;
  double* a = Vf + ((size_t)t.y * n + t.x) * bc;
  double* b = Vf + ((size_t)t.x * n + t.y) * bc;
  for (int i = threadIdx.x; i < bc; i += 256) {
    const double v = row[i];
    a[i] = v;
    b[i] = v;
  }
}

// Xf[m][l][x] = Xf[l][m][x] = X[x][t] for the pairs j0 + t = (l,m) of one
// block of X (ld bc, t < bc) and the rows x < nx: 32 x 32 tiles turned over
// in LDS, read along t and written along x.
constexpr int kTile = 32;
__global__ void __launch_bounds__(256) k_turn(const double* __restrict__ X, int bc, size_t j0, size_t nx, int n,
                                              const int2* __restrict__ lm, double* __restrict__ Xf) {
  __shared__ double t[kTile][kTile + 1];
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  const size_t x0 = (size_t)blockIdx.x * kTile;
  const int t0 = blockIdx.y * kTile;
  for (int i = ty; i < kTile; i += 8)
    if (x0 + i < nx && t0 + tx < bc) t[i][tx] = X[(x0 + i) * bc + t0 + tx];
  __syncthreads();
  for (int i = ty; i < kTile; i += 8) {
    if (t0 + i >= bc || x0 + tx >= nx) continue;
    const int2 p = lm[j0 + t0 + i];
    const double v = t[tx][i];
    Xf[((size_t)p.y * n + p.x) * nx + x0 + tx] = v;
    if (p.x != p.y) Xf[((size_t)p.x * n + p.y) * nx + x0 + tx] = v;
  }
}

// part[block] += sum over Y[s][b][x] = (ar|bs), x = (a, r), of one block of
// bra virtual orbitals r in [r0, r0 + nr), s < ns:
//   MODE 0 (closed shell):  w (ar|bs)[2(ar|bs) - (as|br)] / D, s <= r,
//          w = 2 for s < r, 1 for s = r (the (s,r) terms equal the (r,s) ones)
//   MODE 1 (one spin):      [(ar|bs) - (as|br)]^2 / (2 D), s < r
//   MODE 2 (two spins):     (ar|bs)^2 / D
// with D = e_a + e_b - e_r - e_s.  An item is a 32 x 32 tile (a, b) of one
// (r, s); modes 0 and 1 read the mirrored tile (b, a) through LDS, so that
// both are read along a.
constexpr int kEnergyBlock = 256;
template <int MODE>
__global__ void __launch_bounds__(kEnergyBlock) k_energy(const double* __restrict__ Y, int nca, int ncb, int r0, int nr,
                                                        int ns, const double* __restrict__ eca,
                                                        const double* __restrict__ eva, const double* __restrict__ ecb,
                                                        const double* __restrict__ evb, double* __restrict__ part) {
  __shared__ double tile[kTile][kTile + 1];
  __shared__ double red[kEnergyBlock];
  const int ta = (nca + kTile - 1) / kTile, tb = (ncb + kTile - 1) / kTile;
  const size_t B = (size_t)nca * nr, items = (size_t)ta * tb * nr * ns;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  double acc = 0.0;
  for (size_t it = blockIdx.x; it < items; it += gridDim.x) {
    const int A0 = (int)(it % ta) * kTile, B0 = (int)(it / ta % tb) * kTile;
    const int rl = (int)(it / ((size_t)ta * tb) % nr), s = (int)(it / ((size_t)ta * tb * nr));
    const int r = r0 + rl;
    if (MODE == 0 && s > r) continue;
    if (MODE == 1 && s >= r) continue;
    const double* Yrs = Y + (size_t)rl * nca + B * ncb * (size_t)s;  // [b][a], a contiguous
    const double ers = eva[r] + evb[s];
    if constexpr (MODE != 2) {
      for (int i = ty; i < kTile; i += 8)  // (b as first index, a as second): rows a, contiguous in b
        if (A0 + i < nca && B0 + tx < ncb) tile[i][tx] = Yrs[(size_t)(A0 + i) * B + B0 + tx];
      __syncthreads();
    }
    for (int i = ty; i < kTile; i += 8) {
      const int a = A0 + tx, b = B0 + i;
      if (a >= nca || b >= ncb) continue;
      const double v = Yrs[(size_t)b * B + a];
      const double d = eca[a] + ecb[b] - ers;
      if constexpr (MODE == 2) {
        acc += v * v / d;
      } else {
        const double x = tile[tx][i];
        if constexpr (MODE == 0)
          acc += (s == r ? 1.0 : 2.0) * v * (2.0 * v - x) / d;
        else
          acc += 0.5 * (v - x) * (v - x) / d;
      }
    }
    if constexpr (MODE != 2) __syncthreads();
  }
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int w = kEnergyBlock / 2; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] += red[0];
}

__global__ void k_zero(double* p, size_t n) {
  for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += (size_t)gridDim.x * blockDim.x) p[e] = 0.0;
}

// Work buffers from the library's block cache, given back once the stream
// has finished with them.
struct Bufs {
  hipStream_t st;
  std::vector<void*> p;
  explicit Bufs(hipStream_t s) : st(s) {}
  ~Bufs() {
    (void)hipStreamSynchronize(st);
    for (void* q : p) sq_device_release(q);
  }
  template <class T>
  bool get(T** d, size_t count) {
    void* v = sq_device_block(std::max<size_t>(count * sizeof(T), 8));
    if (!v) return false;
    p.push_back(v);
    *d = (T*)v;
    return true;
  }
};

}  // namespace

size_t sq_mp2_bytes(int n, size_t ncv_sum) {
  const size_t npr = (size_t)n * (n + 1) / 2;
  return npr * npr * 8 + npr * ncv_sum * 8;
}

namespace {

constexpr int kParts = 1024;  // energy partial sums (one per workgroup)

struct Ctx {
  hipStream_t st;
  rocblas_handle h;
  int n;
  size_t npr;
  const int2* lm;
  double* part;
  std::string* err;
  int bad(const std::string& m) {
    *err = m;
    return -1;
  }
};

// Ket pairs of a block of the half-transformed integrals, for bytes_per_pair
// of work buffers: at most 2 GiB of them, a multiple of 64 that cuts the
// pairs evenly (long DGEMM rows: 2 GiB holds 2304 pairs at n = 304).
size_t pair_block(size_t npr, size_t bytes_per_pair, size_t freeb) {
  const size_t most = std::max<size_t>(1, std::min<size_t>(freeb / 4, (size_t)2 << 30) / bytes_per_pair);
  if (most >= npr) return npr;
  const size_t nblk = (npr + most - 1) / most, even = (npr + nblk - 1) / nblk;
  return most >= 64 ? std::min(most / 64 * 64, (even + 63) / 64 * 64) : most;
}

// Half-transformed integrals of one spin: blocks of `blk` pairs from j0 =
// 0, blk, ... at X + j0 * nc * nv, each [r][a][bc] (bc = its pairs).
struct Half {
  double* X = nullptr;
  size_t blk = 0;
};

int first_half(Ctx& c, const double* dV, const SqMp2Spin& sp, Half& H) {
  const int n = c.n, nc = sp.nc, nv = sp.nv;
  const size_t npr = c.npr, ncv = (size_t)nc * nv;
  const double one = 1.0, zero = 0.0;
  size_t freeb = 0, totb = 0;
  if (hipMemGetInfo(&freeb, &totb) != hipSuccess) return c.bad("hipMemGetInfo failed");
  freeb += sq_device_cached();
  const size_t blk = H.blk = std::min<size_t>(pair_block(npr, (size_t)n * n * 8 + (size_t)nc * n * 8, freeb),
                                              (size_t)INT32_MAX / std::max(nc, nv));
  double *dVf = nullptr, *dT = nullptr;
  Bufs work(c.st);
  if (!work.get(&dVf, blk * n * n) || !work.get(&dT, blk * nc * n))
    return c.bad("device allocation of the first half's blocks failed");
  for (size_t j0 = 0; j0 < npr; j0 += blk) {
    const int bc = (int)std::min(blk, npr - j0);
    hipLaunchKernelGGL(k_gather, dim3((unsigned)npr), dim3(256), 0, c.st, dV, npr, j0, bc, n, c.lm, dVf);
    if (rocblas_dgemm_strided_batched(c.h, rocblas_operation_none, rocblas_operation_none, bc, nc, n, &one, dVf, bc,
                                      (rocblas_stride)n * bc, sp.dCo, n, 0, &zero, dT, bc, (rocblas_stride)nc * bc,
                                      n) != rocblas_status_success)
      return c.bad("rocblas_dgemm_strided_batched (first quarter) failed");
    if (rocblas_dgemm(c.h, rocblas_operation_none, rocblas_operation_none, bc * nc, nv, n, &one, dT, bc * nc, sp.dCv, n,
                      &zero, H.X + j0 * ncv, bc * nc) != rocblas_status_success)
      return c.bad("rocblas_dgemm (second quarter) failed");
  }
  if (hipStreamSynchronize(c.st) != hipSuccess)
    return c.bad(std::string("first half-transform failed: ") + hipGetErrorString(hipGetLastError()));
  return 0;
}

// Y block by block over the bra virtual orbitals, summed into c.part by
// k_energy<MODE> (MODE 0/1: bra and ket the same spin, s <= r only)
template <int MODE>
int second_half(Ctx& c, const Half& H, const SqMp2Spin& bra, const SqMp2Spin& ket, double* flop) {
  const int n = c.n;
  const size_t npr = c.npr, ncv = (size_t)bra.nc * bra.nv;
  const double one = 1.0, zero = 0.0;
  size_t freeb = 0, totb = 0;
  if (hipMemGetInfo(&freeb, &totb) != hipSuccess) return c.bad("hipMemGetInfo failed");
  freeb += sq_device_cached();
  const size_t per_x = ((size_t)n * n + (size_t)n * ket.nc + (size_t)ket.nc * ket.nv) * 8;
  const size_t most = std::min<size_t>(std::min<size_t>(freeb / 2, (size_t)2 << 30) / per_x,
                                       (size_t)INT32_MAX / std::max(ket.nc, 1));
  // evenly cut, and at least four blocks where only s <= r is wanted
  const int nr_most = (int)std::max<size_t>(1, std::min<size_t>(most / bra.nc, bra.nv));
  int nblk = (bra.nv + nr_most - 1) / nr_most;
  if (MODE != 2) nblk = std::max(nblk, std::min(4, bra.nv));
  const int nr = (bra.nv + nblk - 1) / nblk;
  double *dXf = nullptr, *dU = nullptr, *dY = nullptr;
  Bufs work(c.st);
  const size_t Bm = (size_t)nr * bra.nc;
  if (!work.get(&dXf, Bm * n * n) || !work.get(&dU, Bm * ket.nc * n) || !work.get(&dY, Bm * ket.nc * ket.nv))
    return c.bad("device allocation of the second half's blocks failed");
  for (int r0 = 0; r0 < bra.nv; r0 += nr) {
    const int rc = std::min(nr, bra.nv - r0);
    const int ns = MODE == 2 ? ket.nv : r0 + rc;
    const size_t B = (size_t)rc * bra.nc;
    for (size_t j0 = 0; j0 < npr; j0 += H.blk) {
      const int bc = (int)std::min(H.blk, npr - j0);
      hipLaunchKernelGGL(k_turn, dim3((unsigned)((B + kTile - 1) / kTile), (bc + kTile - 1) / kTile), dim3(256), 0,
                         c.st, H.X + j0 * ncv + (size_t)r0 * bra.nc * bc, bc, j0, B, n, c.lm, dXf);
    }
    if (rocblas_dgemm_strided_batched(c.h, rocblas_operation_none, rocblas_operation_none, (rocblas_int)B, ket.nc, n,
                                      &one, dXf, (rocblas_int)B, (rocblas_stride)n * B, ket.dCo, n, 0, &zero, dU,
                                      (rocblas_int)B, (rocblas_stride)ket.nc * B, n) != rocblas_status_success)
      return c.bad("rocblas_dgemm_strided_batched (third quarter) failed");
    const rocblas_int rows = (rocblas_int)(B * ket.nc);
    if (rocblas_dgemm(c.h, rocblas_operation_none, rocblas_operation_none, rows, ns, n, &one, dU, rows, ket.dCv, n,
                      &zero, dY, rows) != rocblas_status_success)
      return c.bad("rocblas_dgemm (fourth quarter) failed");
    *flop += 2.0 * (double)B * ket.nc * n * ((double)n + ns);
    hipLaunchKernelGGL(k_energy<MODE>, dim3(kParts), dim3(kEnergyBlock), 0, c.st, dY, bra.nc, ket.nc, r0, rc, ns,
                       bra.dec, bra.dev, ket.dec, ket.dev, c.part);
  }
  if (hipStreamSynchronize(c.st) != hipSuccess)
    return c.bad(std::string("second half-transform failed: ") + hipGetErrorString(hipGetLastError()));
  return 0;
}

}  // namespace

void sq_mp2_release(void* handle) {
  if (handle) (void)rocblas_destroy_handle(static_cast<rocblas_handle>(handle));
}

int sq_mp2_from_pairs(hipStream_t st, void** handle, int n, int nspin, const SqMp2Spin* sp, double** dV,
                      SqMp2Result* out, std::string* err) {
  *out = SqMp2Result{};
  const size_t npr = (size_t)n * (n + 1) / 2;
  auto fail = [&](const std::string& m) {
    *err = m;
    return -1;
  };
  bool any = false;
  for (int k = 0; k < nspin; ++k) any = any || (sp[k].nc > 0 && sp[k].nv > 0);
  if (!any) {  // nothing to correlate
    sq_device_release(*dV);
    *dV = nullptr;
    return 0;
  }
  rocblas_handle h = static_cast<rocblas_handle>(*handle);
  if (!h) {
    if (rocblas_create_handle(&h) != rocblas_status_success) return fail("rocblas_create_handle failed");
    *handle = h;
  }
  if (rocblas_set_stream(h, st) != rocblas_status_success) return fail("rocblas_set_stream failed");
  hipEvent_t e0, e1, e2;
  if (hipEventCreate(&e0) != hipSuccess || hipEventCreate(&e1) != hipSuccess || hipEventCreate(&e2) != hipSuccess)
    return fail("hipEventCreate failed");
  struct EventGuard {
    hipEvent_t a, b, c;
    ~EventGuard() { (void)hipEventDestroy(a); (void)hipEventDestroy(b); (void)hipEventDestroy(c); }
  } eg{e0, e1, e2};

  Bufs keep(st);  // buffers of the whole call
  Half X[2];
  double* dPart = nullptr;
  int2* dLM = nullptr;
  if (!keep.get(&dPart, kParts) || !keep.get(&dLM, npr)) return fail("device allocation failed");
  for (int k = 0; k < nspin; ++k)
    if (!keep.get(&X[k].X, npr * (size_t)sp[k].nc * sp[k].nv))
      return fail("device allocation of the half-transformed integrals failed (" +
                  std::to_string(npr * (size_t)sp[k].nc * sp[k].nv * 8 / 1048576) + " MiB)");
  {
    std::vector<int2> lm(npr);
    for (int l = 0, j = 0; l < n; ++l)
      for (int m = 0; m <= l; ++m, ++j) lm[j] = make_int2(l, m);
    if (hipMemcpyAsync(dLM, lm.data(), npr * sizeof(int2), hipMemcpyHostToDevice, st) != hipSuccess ||
        hipStreamSynchronize(st) != hipSuccess)
      return fail("pair table upload failed");
  }
  hipLaunchKernelGGL(k_zero, dim3(4), dim3(256), 0, st, dPart, (size_t)kParts);
  Ctx c{st, h, n, npr, dLM, dPart, err};

  if (hipEventRecord(e0, st) != hipSuccess) return fail("hipEventRecord failed");
  for (int k = 0; k < nspin; ++k)
    if (sp[k].nc > 0 && sp[k].nv > 0)
      if (int rc = first_half(c, *dV, sp[k], X[k])) return rc;
  if (hipEventRecord(e1, st) != hipSuccess) return fail("hipEventRecord failed");
  sq_device_release(*dV);  // V is no longer needed (first_half has waited)
  *dV = nullptr;

  double flop2 = 0.0;
  if (nspin == 1) {
    if (int rc = second_half<0>(c, X[0], sp[0], sp[0], &flop2)) return rc;
  } else {
    for (int k = 0; k < 2; ++k)
      if (sp[k].nc > 1 && sp[k].nv > 1)
        if (int rc = second_half<1>(c, X[k], sp[k], sp[k], &flop2)) return rc;
    if (sp[0].nc > 0 && sp[0].nv > 0 && sp[1].nc > 0 && sp[1].nv > 0)
      if (int rc = second_half<2>(c, X[0], sp[0], sp[1], &flop2)) return rc;
  }
  if (hipEventRecord(e2, st) != hipSuccess) return fail("hipEventRecord failed");
  std::vector<double> part(kParts);
  if (hipMemcpyAsync(part.data(), dPart, kParts * 8, hipMemcpyDeviceToHost, st) != hipSuccess ||
      hipStreamSynchronize(st) != hipSuccess)
    return fail(std::string("energy sum failed: ") + hipGetErrorString(hipGetLastError()));
  double e2sum = 0.0;
  for (double v : part) e2sum += v;
  float ms1 = 0.0f, ms2 = 0.0f;
  (void)hipEventElapsedTime(&ms1, e0, e1);
  (void)hipEventElapsedTime(&ms2, e1, e2);
  out->e2 = e2sum;
  out->half1_ms = ms1;
  out->half2_ms = ms2;
  double f1 = 0.0;
  for (int k = 0; k < nspin; ++k)
    f1 += 2.0 * sp[k].nc * (double)n * n * npr + 2.0 * sp[k].nc * (double)sp[k].nv * n * npr;
  out->half1_flop = f1;
  out->half2_flop = flop2;
  return 0;
}
