// Smooth PME reciprocal space: order-5 B-spline charge spread, a real-to-
// complex 3D FFT done in LDS, the convolution with the Ewald influence
// function (energy read off it in FP64), the inverse transform and the force
// gather.
//
// Replaces encodePme (webgpu/kernels/pme.js:137-463) and encodeFft3d
// (webgpu/kernels/pme-fft.js:42-197). Conventions are the reference's
// (cpu/forces/pme.js:11-15): the forward transform carries exp(+2 pi i m k/K),
// the B-spline moduli divide the convolution, grid index for weight k is
// (floor(u) + k - order + 1) mod K, and the inverse is unnormalised.
//
// MI355X shape. The default "plane" pipeline is three launches:
//   1. one workgroup per x plane gathers the charges that land on its plane
//      into an int64 fixed-point plane in LDS (exact and order independent,
//      no global atomics), then runs the z (real-to-complex, two real lines
//      per complex transform) and y transforms of that plane in LDS;
//   2. x lines: forward transform, convolution with the influence function
//      (and the energy), inverse transform;
//   3. one workgroup per x plane runs the inverse y and z transforms into a
//      real potential plane in LDS and adds each atom's share of the force
//      from that plane.
// Grids whose plane does not fit in LDS use the "slab" pipeline: the plane
// split into slabs of rows, one launch per axis pass.
// Grid sizes may carry a factor 7 (2^a 3^b 5^c 7^d).
#include <type_traits>

#include "pme_plane.h"

namespace rmd {

// The atoms by the base index of their x support, rebuilt each evaluation by
// one workgroup per system (at most BIN_MAX_ATOMS atoms): each charged atom
// takes its rank in its bin by an LDS atomic count, the counts become
// offsets, and each atom is written at its offset plus rank. The order inside
// a bin varies from run to run; nothing depends on it (the spread
// accumulates in fixed point, the gather is per atom), so the binned planes
// give the scanned planes' results bit for bit.
constexpr int BIN_THREADS = 1024;
constexpr int BIN_MAX_K = 1024;  // grid sizes are at most 1024

__device__ __forceinline__ void pmeBinBuild(const Dev &d, const PmeDev &p) {
  __shared__ int start[BIN_MAX_K];
  __shared__ int waveTotal[BIN_THREADS / 64];
  const int K0 = p.K[0], t = threadIdx.x, nt = blockDim.x;
  for (int b = t; b < K0; b += nt) start[b] = 0;
  __syncthreads();
  const double *recip = d.box->recip64;
  for (int a = t; a < d.n; a += nt) {
    const float4 pos = d.pos[a];
    int2 e = make_int2(-1, 0);
    if (pos.w != 0.f) {
      int bx;
      float ox;
      gridCoordinate(p, recip, 0, pos, bx, ox);
      e = make_int2(bx, atomicAdd(&start[bx], 1));
    }
    p.atomBin[a] = e;
  }
  __syncthreads();
  // exclusive prefix over the counts, in place: a few bins per thread, then
  // the waves in order
  const int per = (K0 + nt - 1) / nt;
  const int lo = t * per, hi = min(K0, lo + per);
  int sum = 0;
  for (int b = lo; b < hi; ++b) sum += start[b];
  const int lane = t & 63, wave = t >> 6;
  int inclusive = sum;
  for (int offset = 1; offset < 64; offset <<= 1) {
    const int v = __shfl_up(inclusive, offset, 64);
    if (lane >= offset) inclusive += v;
  }
  if (lane == 63) waveTotal[wave] = inclusive;
  __syncthreads();
  int before = 0;
  for (int w = 0; w < wave; ++w) before += waveTotal[w];
  int offset = before + inclusive - sum;
  for (int b = lo; b < hi; ++b) {
    const int c = start[b];
    start[b] = offset;
    p.binStart[b] = offset;
    offset += c;
  }
  if (t == nt - 1) p.binStart[K0] = before + inclusive;
  __syncthreads();
  for (int a = t; a < d.n; a += nt) {
    const int2 e = p.atomBin[a];
    if (e.x >= 0) p.binAtoms[start[e.x] + e.y] = a;
  }
}

// A batch member stepped alone.
__global__ void __launch_bounds__(BIN_THREADS) pmeBinKernel(Dev d, PmeDev p) { pmeBinBuild(d, p); }
__global__ void __launch_bounds__(BIN_THREADS) pmeBinBatchKernel(const BatchView *__restrict__ v,
                                                                 const int2 *__restrict__ task) {
  const int2 t = task[blockIdx.x];
  if (t.x < 0 || v[t.x].p.atoms != PME_ATOMS_BINS) return;
  pmeBinBuild(v[t.x].d, v[t.x].p);
}

bool pmeBinsFit(const PmeDev &p, int atoms) {
  return p.planes && p.K[0] >= ORDER && p.K[0] <= BIN_MAX_K && atoms <= BIN_MAX_ATOMS;
}

__global__ void __launch_bounds__(PLANE_THREADS) pmePlaneForwardKernel(Dev d, PmeDev p, const float *real) {
  extern __shared__ float2 lds[];
  pmePlaneForward(d, p, real, blockIdx.x, lds);
}

__global__ void __launch_bounds__(PLANE_THREADS) pmePlaneForwardBatchKernel(const BatchView *__restrict__ v,
                                                                          const int2 *__restrict__ task) {
  extern __shared__ float2 lds[];
  const int2 t = task[blockIdx.x];
  if (t.x < 0) return;
  pmePlaneForward<SCAN_BATCHED>(v[t.x].d, v[t.x].p, nullptr, t.y, lds);
}

__global__ void __launch_bounds__(XLINE_THREADS) pmeXLinesKernel(Dev d, PmeDev p, int convolve, int energies) {
  extern __shared__ float2 lds[];
  pmeXLines(d, p, convolve, energies, blockIdx.x, lds);
}

__global__ void __launch_bounds__(XLINE_THREADS) pmeXLinesBatchKernel(const BatchView *__restrict__ v,
                                                                    const int2 *__restrict__ task, int energies) {
  extern __shared__ float2 lds[];
  const int2 t = task[blockIdx.x];
  if (t.x < 0) return;
  pmeXLines(v[t.x].d, v[t.x].p, 1, energies, t.y, lds);
}

// A large system's planes in workgroups of WIDE_PLANE_THREADS: its
// plane's LDS (153 KB at 112^3) leaves room for one workgroup per CU, and K0
// planes occupy fewer CUs than the chip has, so each plane's spread,
// transforms and gather get the CU's four SIMDs at four waves each. (SCAN 3
// keeps a round of the scan list within its LDS at this width.) Every single
// system gathers in such workgroups - K0 planes leave most CUs idle whatever
// the system's size, and a plane's atoms are gathered twice as wide (2854
// atoms, 30^3: 18.3 -> 17.1 us per chain). The results are the 512-thread
// kernels' bit for bit: the plane is an integer sum, each transform output
// and each atom's share of a plane has one formula, and forces are integer
// sums.
constexpr int WIDE_PLANE_THREADS = 1024;

__global__ void __launch_bounds__(WIDE_PLANE_THREADS) pmePlaneForwardWideKernel(Dev d, PmeDev p) {
  extern __shared__ float2 lds[];
  pmePlaneForward<PLANE_LIST / WIDE_PLANE_THREADS>(d, p, nullptr, blockIdx.x, lds);
}

__global__ void __launch_bounds__(WIDE_PLANE_THREADS) pmePlaneGatherKernel(Dev d, PmeDev p, int folded) {
  extern __shared__ float2 lds[];
  pmePlaneGather<PLANE_LIST / WIDE_PLANE_THREADS>(d, p, blockIdx.x, lds, folded);
}

static void launchPlaneForward(const Dev &d, const PmeDev &p, size_t lds, hipStream_t s) {
  if (p.atoms != PME_ATOMS_SCAN)
    pmePlaneForwardWideKernel<<<p.K[0], WIDE_PLANE_THREADS, lds, s>>>(d, p);
  else
    pmePlaneForwardKernel<<<p.K[0], PLANE_THREADS, lds, s>>>(d, p, nullptr);
}

static void launchPlaneGather(const Dev &d, const PmeDev &p, size_t lds, hipStream_t s, int folded = 0) {
  pmePlaneGatherKernel<<<p.K[0], WIDE_PLANE_THREADS, lds, s>>>(d, p, folded);
}

// (Six waves per SIMD: three workgroups per CU, the register count the body
// needs without spills.)
__global__ void __launch_bounds__(PLANE_THREADS) __attribute__((amdgpu_waves_per_eu(6)))
pmePlaneGatherBatchKernel(const BatchView *__restrict__ v, const int2 *__restrict__ task) {
  extern __shared__ float2 lds[];
  const int2 t = task[blockIdx.x];
  if (t.x < 0) return;
  pmePlaneGather<SCAN_BATCHED>(v[t.x].d, v[t.x].p, t.y, lds);
}

// The gather from the potential grid, one thread per charged atom, in cell
// order (a batch member: bin order, where a wave's atoms share an x slab of
// the grid and nothing waits for the cell list): each of the atom's ORDER
// planes' shares is computed with the plane gather's own arithmetic and
// rounded to fixed point as it would be there, and the shares are summed in
// integers - one set of force atomics per atom instead of one per plane, and
// the same force bit for bit where the grid has at least ORDER planes, so
// that each weight lands on a plane of its own.
__device__ __forceinline__ void pmeAtomGather(const Dev &d, const PmeDev &p, int k) {
  if (k >= (p.atoms == PME_ATOMS_BINS ? p.binStart[p.K[0]] : d.n)) return;
  const int a = p.atoms == PME_ATOMS_BINS ? p.binAtoms[k] : d.cellAtoms[k];
  const float4 pos = p.atoms == PME_ATOMS_BINS ? d.pos[a] : d.slotPos[k];
  if (pos.w == 0.f) return;
  const int K0 = p.K[0], K1 = p.K[1], K2 = p.K[2];
  const double *recip = d.box->recip64;
  int bx, by, bz;
  float ox, oy, oz;
  gridCoordinate(p, recip, 0, pos, bx, ox);
  float w[ORDER], dw[ORDER], wy[ORDER], dwy[ORDER], wz[ORDER], dwz[ORDER];
  bspline5(ox, w, dw);
  gridCoordinate(p, recip, 1, pos, by, oy);
  gridCoordinate(p, recip, 2, pos, bz, oz);
  bspline5(oy, wy, dwy);
  bspline5(oz, wz, dwz);
  int iz[ORDER], iy[ORDER];
  for (int c = 0; c < ORDER; ++c) {
    iz[c] = gridIndex(bz, c, K2);
    iy[c] = gridIndex(by, c, K1);
  }
  const GlobalPtr<float> grid = globalPtr(p.rgrid);
  long long total[3] = {0, 0, 0};
  for (int r = 0; r < ORDER; ++r) {
    const size_t plane = (size_t)gridIndex(bx, r, K0) * K1;
    const float wx = 0.f + w[r], dwx = 0.f + dw[r];
    float s0 = 0.f, s1 = 0.f, s2 = 0.f;
    for (int b = 0; b < ORDER; ++b) {
      const GlobalPtr<float> row = grid + (plane + iy[b]) * K2;
      float r0 = 0.f, r2 = 0.f;
      for (int c = 0; c < ORDER; ++c) {
        const float v = row[iz[c]];
        r0 += wz[c] * v;
        r2 += dwz[c] * v;
      }
      s0 += wy[b] * r0;
      s1 += dwy[b] * r0;
      s2 += wy[b] * r2;
    }
    long long f[3];
    gridForceFixed(d, p, pos.w, dwx * s0, wx * s1, wx * s2, f);
    for (int k = 0; k < 3; ++k) total[k] += f[k];
  }
  atomicAddFixed(&d.force[a], total[0]);
  atomicAddFixed(&d.force[d.nPad + a], total[1]);
  atomicAddFixed(&d.force[2 * d.nPad + a], total[2]);
}

__global__ void __launch_bounds__(256) pmeAtomGatherKernel(Dev d, PmeDev p) {
  pmeAtomGather(d, p, blockIdx.x * blockDim.x + threadIdx.x);
}

__global__ void __launch_bounds__(256) pmeAtomGatherBatchKernel(const BatchView *__restrict__ v,
                                                                const int2 *__restrict__ task) {
  const int2 t = task[blockIdx.x];
  if (t.x < 0 || v[t.x].p.atoms == PME_ATOMS_SCAN) return;
  pmeAtomGather(v[t.x].d, v[t.x].p, t.y * blockDim.x + threadIdx.x);
}

// ============================================================================
// Slab pipeline (grids whose plane does not fit in LDS)
// ============================================================================
//
// Six launches, each a pass over the grid in tiles of LN lines by a whole
// axis (LN = 16 unless the axis is too long for LDS):
//   1. one workgroup per slab of 2 LN rows spreads the charges that land on
//      its rows into an int64 slab in LDS, as the plane pipeline does for a
//      whole plane, and transforms the rows along z (two real rows per complex
//      line);
//   2. y lines; 3. x lines with the convolution; 4. y lines back: LN columns
//      that are neighbours in memory, so every access is a run of 128 bytes;
//   5. z lines back into the real potential; 6. one thread per atom gathers.
// Bound by the passes over the half spectrum (24 MB at 180^3, held by the
// last-level cache) and the spread's LDS atomics. At 180^3 and 100,222 atoms
// the chain took 797 us when the spread went through 64-bit atomics on a
// grid in global memory (531 us of it) and lines four at a time (32-byte
// runs); it takes 190 us now.

constexpr int SLAB_THREADS = 512;

// LDS tiles hold LN lines side by side, position-major: point k of line l at
// k * (LN + 1) + l, so the index arithmetic of a pass is shifts and masks and
// neither the columns' nor the rows' accesses pile onto one bank.
template <int LN>
__device__ __forceinline__ int tileAt(int k, int l) {
  return k * (LN + 1) + l;
}

// One radix-R pass of a Stockham autosort transform over a tile's LN lines of
// length K; Ns is the product of the radices done.
template <int R, int LN>
__device__ __forceinline__ void tileStage(const float2 *src, float2 *dst, int K, int Ns, const float2 *tw,
                                          int sign) {
  const int L = K / R;
  const Div byNs(Ns);
  const int twStride = byNs(L);
  for (int idx = threadIdx.x; idx < L * LN; idx += blockDim.x) {
    const int line = idx & (LN - 1), j = idx / LN;
    const int q0 = byNs(j), k = j - q0 * Ns;
    float2 v[8];
    v[0] = src[tileAt<LN>(j, line)];
#pragma unroll
    for (int q = 1; q < R; ++q) {
      float2 w = tw[k * q * twStride];
      if (sign < 0) w.y = -w.y;
      v[q] = cmul(src[tileAt<LN>(j + q * L, line)], w);
    }
    smallDft(v, R, sign);
    const int base = q0 * Ns * R + k;
#pragma unroll
    for (int q = 0; q < R; ++q) dst[tileAt<LN>(base + q * Ns, line)] = v[q];
  }
}

// The whole transform; every stage ends with a barrier. Returns the buffer
// with the result.
template <int LN>
__device__ __forceinline__ float2 *tileFft(float2 *src, float2 *dst, int K, const int *rad, const float2 *tw,
                                           int sign) {
  int Ns = 1;
  for (int s = 0; s < 8 && rad[s] > 0; ++s) {
    switch (rad[s]) {
      case 2: tileStage<2, LN>(src, dst, K, Ns, tw, sign); break;
      case 3: tileStage<3, LN>(src, dst, K, Ns, tw, sign); break;
      case 4: tileStage<4, LN>(src, dst, K, Ns, tw, sign); break;
      case 5: tileStage<5, LN>(src, dst, K, Ns, tw, sign); break;
      default: tileStage<7, LN>(src, dst, K, Ns, tw, sign); break;
    }
    __syncthreads();
    float2 *swap = src;
    src = dst;
    dst = swap;
    Ns *= rad[s];
  }
  return src;
}

// The slots whose atoms can reach rows [y0, y0 + rows) of plane i, as runs of
// the cell order (slabRuns), in LDS.
constexpr int SLAB_RUNS = 64;
struct SlabRuns {
  int begin[SLAB_RUNS];
  int start[SLAB_RUNS + 1];  // prefix of the runs' lengths
  int count;
};

constexpr int SLAB_QUEUE = SLAB_THREADS / 64 * QUEUE_ENTRIES;

// By the first wave: the cells (by x, and by y within each x; all of z) that
// the support can come from, one contiguous run of slots per (x, y segment).
// With more runs than SLAB_RUNS every slot is a candidate.
__device__ __forceinline__ void slabRuns(const Dev &d, const PmeDev &p, int i, int y0, int rows, SlabRuns &out) {
  const int lane = threadIdx.x;
  const int cx = d.sc->builtCells[0], cy = d.sc->builtCells[1], cz = d.sc->builtCells[2];
  int x0, nx, yFirst, ny;
  supportCells(d, 0, i, 1, p.K[0], x0, nx);
  supportCells(d, 1, y0, rows, p.K[1], yFirst, ny);
  const int segs = yFirst + ny > cy ? 2 : 1;
  int runs = nx * segs, begin = 0, len = 0;
  if (runs > SLAB_RUNS) {
    runs = 1;
    len = lane == 0 ? d.n : 0;
  } else if (lane < runs) {
    const int q = lane / segs, seg = lane - q * segs;
    int x = x0 + q;
    x -= x >= cx ? cx : 0;
    const int ya = seg ? 0 : yFirst, yb = seg ? yFirst + ny - cy : min(cy, yFirst + ny);
    begin = d.cellStart[(x * cy + ya) * cz];
    len = d.cellStart[(x * cy + yb) * cz] - begin;
  }
  int inclusive = len;
  for (int offset = 1; offset < 64; offset <<= 1) {
    const int v = __shfl_up(inclusive, offset, 64);
    if (lane >= offset) inclusive += v;
  }
  if (lane < runs) {
    out.begin[lane] = begin;
    out.start[lane] = inclusive - len;
  }
  if (lane == runs - 1) out.start[runs] = inclusive;
  if (lane == 0) out.count = runs;
}

template <int LN>
static size_t slabLds(int K) {
  return (size_t)K * sizeof(float2) * (1 + (LN + 1)) + (size_t)K * 2 * LN * sizeof(long long) +
         SLAB_QUEUE * sizeof(int) + sizeof(SlabRuns);
}
template <int LN>
static size_t tileLds(int K) {
  return (size_t)K * sizeof(float2) * (1 + 2 * (LN + 1));
}

// 1. Spread onto 2 LN rows and their forward z transforms: rows [first,
// first + 2 LN) of all K0 K1 in plane order, so a slab may end in the next
// plane (or span several short ones) and two rows share a complex line
// whatever K1's parity. With `real` set the rows come from a real K0*K1*K2
// grid (the FFT verification entry).
template <int LN>
__global__ void __launch_bounds__(SLAB_THREADS) pmeSlabForwardKernel(Dev d, PmeDev p, const float *real) {
  extern __shared__ float2 lds[];
  const int K0 = p.K[0], K1 = p.K[1], K2 = p.K[2], K2h = p.K2h;
  const int firstRow = blockIdx.x * 2 * LN, rows = min(2 * LN, K0 * K1 - firstRow);
  const int t = threadIdx.x, nt = blockDim.x, lane = t & 63, wave = t >> 6, waves = nt >> 6;
  float2 *tw = lds, *A = tw + K2;
  long long *slab = reinterpret_cast<long long *>(A + (size_t)K2 * (LN + 1));
  float2 *B = reinterpret_cast<float2 *>(slab);  // (the charges are read out before B is written)
  int *list = reinterpret_cast<int *>(slab + (size_t)2 * LN * K2);
  SlabRuns &runs = *reinterpret_cast<SlabRuns *>(list + SLAB_QUEUE);
  loadTwiddles(tw, p.twiddle[2], K2);
  if (real) {
    for (int pr = wave; pr < LN; pr += waves) {
      const float *r0 = real + (size_t)(firstRow + 2 * pr) * K2;
      for (int k = lane; k < K2; k += 64)
        A[tileAt<LN>(k, pr)] = make_float2(2 * pr < rows ? r0[k] : 0.f, 2 * pr + 1 < rows ? r0[K2 + k] : 0.f);
    }
  } else {
    for (int idx = t; idx < 2 * LN * K2; idx += nt) slab[idx] = 0;
    const double *recip = d.box->recip64;
    const float rx32[3] = {(float)recip[0], (float)recip[3], (float)recip[6]};
    const float ry32[3] = {(float)recip[1], (float)recip[4], (float)recip[7]};
    // the slab's rows plane by plane: `here` rows from y0 of plane i
    for (int done = 0; done < rows;) {
      const int i = (firstRow + done) / K1, y0 = firstRow + done - i * K1, here = min(rows - done, K1 - y0);
      if (wave == 0) slabRuns(d, p, i, y0, here, runs);
      __syncthreads();
      int cur = 0;  // the run of this lane's latest candidate
      waveQueue(
          runs.start[runs.count], list,
          [&](int g) {
            while (runs.start[cur + 1] <= g) ++cur;
            return runs.begin[cur] + (g - runs.start[cur]);
          },
          [&](int slot) { return d.slotPos[slot]; },
          [&](float4 pos) {
            return pos.w != 0.f && mayReach(rx32, K0, i, 1, pos) && mayReach(ry32, K1, y0, here, pos);
          },
          [&](float4 pos) {
            int bx, by, bz;
            float ox, oy, oz;
            gridCoordinate(p, recip, 0, pos, bx, ox);
            const int rx = planeWeight(bx, i, K0);
            if (rx >= ORDER) return;  // it only came near
            float w[ORDER], wy[ORDER], wz[ORDER], dw[ORDER];
            bspline5(ox, w, dw);
            float wx = 0.f;  // (K0 >= ORDER: one weight lands on the plane)
#pragma unroll
            for (int q = 0; q < ORDER; ++q) wx = q == rx ? w[q] : wx;
            gridCoordinate(p, recip, 1, pos, by, oy);
            gridCoordinate(p, recip, 2, pos, bz, oz);
            bspline5(oy, wy, dw);
            bspline5(oz, wz, dw);
            int iz[ORDER];
            for (int c = 0; c < ORDER; ++c) iz[c] = gridIndex(bz, c, K2);
            for (int b = 0; b < ORDER; ++b) {
              const int r = gridIndex(by, b, K1) - y0;
              if (r < 0 || r >= here) continue;
              unsigned long long *row = reinterpret_cast<unsigned long long *>(slab + (size_t)(done + r) * K2);
              for (int c = 0; c < ORDER; ++c)
                atomicAdd(row + iz[c], (unsigned long long)chargeToFixed(pos.w, wx, wy[b], wz[c]));
            }
          });
      __syncthreads();  // runs is written again for the next plane
      done += here;
    }
    // Two real rows per complex line.
    for (int pr = wave; pr < LN; pr += waves) {
      const long long *r0 = slab + (size_t)2 * pr * K2;
      for (int k = lane; k < K2; k += 64)
        A[tileAt<LN>(k, pr)] = make_float2((float)((double)r0[k] * GRID_UNSCALE),
                                           (float)((double)r0[K2 + k] * GRID_UNSCALE));
    }
  }
  __syncthreads();
  const float2 *Z = tileFft<LN>(A, B, K2, p.radices[2], tw, +1);
  // Split the packed spectra: row 2p = (Z[m] + conj Z[-m]) / 2, row 2p+1 =
  // (Z[m] - conj Z[-m]) / (2i).
  for (int r = wave; r < rows; r += waves) {
    float2 *out = p.cgrid + (size_t)(firstRow + r) * K2h;
    for (int m = lane; m < K2h; m += 64) {
      const float2 z = Z[tileAt<LN>(m, r >> 1)], zc = Z[tileAt<LN>(m == 0 ? 0 : K2 - m, r >> 1)];
      out[m] = (r & 1) == 0 ? make_float2(0.5f * (z.x + zc.x), 0.5f * (z.y - zc.y))
                            : make_float2(0.5f * (z.y + zc.y), -0.5f * (z.x - zc.x));
    }
  }
}

// A tile of LN columns m0 .. of one line family: point k of column l at
// grid[k * stride + l]. Columns past the spectrum are zero and not stored.
template <int LN>
__device__ __forceinline__ void tileLoad(const float2 *grid, size_t stride, int lines, int K, float2 *A) {
  for (int idx = threadIdx.x; idx < K * LN; idx += blockDim.x) {
    const int l = idx & (LN - 1), k = idx / LN;
    A[tileAt<LN>(k, l)] = l < lines ? grid[k * stride + l] : make_float2(0.f, 0.f);
  }
}
template <int LN>
__device__ __forceinline__ void tileStore(float2 *grid, size_t stride, int lines, int K, const float2 *A) {
  for (int idx = threadIdx.x; idx < K * LN; idx += blockDim.x) {
    const int l = idx & (LN - 1), k = idx / LN;
    if (l < lines) grid[k * stride + l] = A[tileAt<LN>(k, l)];
  }
}

// y lines, either direction, in place: block b is column chunk b % chunks of
// plane b / chunks.
template <int LN>
__global__ void __launch_bounds__(SLAB_THREADS) pmeTileYKernel(PmeDev p, int sign, int chunks) {
  extern __shared__ float2 lds[];
  const int K = p.K[1], x = blockIdx.x / chunks, m0 = (blockIdx.x - x * chunks) * LN;
  float2 *tw = lds, *A = tw + K, *B = A + (size_t)K * (LN + 1);
  float2 *grid = p.cgrid + (size_t)x * K * p.K2h + m0;
  const int lines = min(LN, p.K2h - m0);
  loadTwiddles(tw, p.twiddle[1], K);
  tileLoad<LN>(grid, p.K2h, lines, K, A);
  __syncthreads();
  const float2 *r = tileFft<LN>(A, B, K, p.radices[1], tw, sign);
  tileStore<LN>(grid, p.K2h, lines, K, r);
}

// x lines: forward transform, then, with `convolve`, the influence function
// (energy in FP64, each half-spectrum column weighted by its multiplicity in
// the full spectrum) and the inverse transform. Tile b is column chunk
// b % chunks of row b / chunks; each workgroup takes every gridDim-th tile
// (one, unless there are more tiles than energy slots).
template <int LN>
__global__ void __launch_bounds__(SLAB_THREADS) pmeTileXKernel(Dev d, PmeDev p, int convolve, int energies,
                                                              int chunks) {
  extern __shared__ float2 lds[];
  const int K = p.K[0];
  const size_t stride = (size_t)p.K[1] * p.K2h;
  float2 *tw = lds, *A = tw + K, *B = A + (size_t)K * (LN + 1);
  loadTwiddles(tw, p.twiddle[0], K);
  const double *recip = d.box->recip64;
  double energy = 0.0, dscale = 0.0;
  for (int tile = blockIdx.x; tile < p.K[1] * chunks; tile += gridDim.x) {
    const int j = tile / chunks, m0 = (tile - j * chunks) * LN;
    const size_t at = (size_t)j * p.K2h + m0;
    const int lines = min(LN, p.K2h - m0);
    tileLoad<LN>(p.cgrid + at, stride, lines, K, A);
    __syncthreads();
    float2 *r = tileFft<LN>(A, B, K, p.radices[0], tw, +1);
    if (convolve) {
      for (int idx = threadIdx.x; idx < K * LN; idx += blockDim.x) {
        const int l = idx & (LN - 1), k = idx / LN, m = m0 + l;
        if (l >= lines) continue;
        const float g = p.influence[at + k * stride + l];
        float2 &f = r[tileAt<LN>(k, l)];
        if (energies) {
          const double weight = (m == 0 || (p.K[2] % 2 == 0 && m == p.K[2] / 2)) ? 1.0 : 2.0;
          const double e = weight * (double)g * ((double)f.x * f.x + (double)f.y * f.y);
          energy += e;
          dscale += e * (2.0 * p.piOverAlpha2 * waveVector2(p, recip, k, j, m) - 1.0);
        }
        f = make_float2(2.f * g * f.x, 2.f * g * f.y);
      }
      __syncthreads();
      r = tileFft<LN>(r, r == A ? B : A, K, p.radices[0], tw, -1);
    }
    tileStore<LN>(p.cgrid + at, stride, lines, K, r);
    __syncthreads();  // the next tile reuses A and B
  }
  if (convolve && energies) storeReciprocal(d, energy, dscale, blockIdx.x);
}

// z lines back: Hermitian extension of two half spectra into one complex
// line, transform, real and imaginary parts are the two real rows.
template <int LN>
__global__ void __launch_bounds__(SLAB_THREADS) pmeSlabInverseKernel(PmeDev p) {
  extern __shared__ float2 lds[];
  const int K2 = p.K[2], K2h = p.K2h;
  const int firstRow = blockIdx.x * 2 * LN, rows = min(2 * LN, p.K[0] * p.K[1] - firstRow);
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6, waves = blockDim.x >> 6;
  float2 *tw = lds, *A = tw + K2, *B = A + (size_t)K2 * (LN + 1);
  loadTwiddles(tw, p.twiddle[2], K2);
  for (int pr = wave; pr < LN; pr += waves) {
    const float2 *r0 = p.cgrid + (size_t)(firstRow + 2 * pr) * K2h;
    const bool live0 = 2 * pr < rows, live1 = 2 * pr + 1 < rows;
    for (int m = lane; m < K2h; m += 64) {
      const float2 a = live0 ? r0[m] : make_float2(0.f, 0.f), b = live1 ? r0[K2h + m] : make_float2(0.f, 0.f);
      A[tileAt<LN>(m, pr)] = make_float2(a.x - b.y, a.y + b.x);
      if (m > 0 && K2 - m >= K2h) A[tileAt<LN>(K2 - m, pr)] = make_float2(a.x + b.y, b.x - a.y);
    }
  }
  __syncthreads();
  const float2 *Z = tileFft<LN>(A, B, K2, p.radices[2], tw, -1);
  for (int r = wave; r < rows; r += waves) {
    float *out = p.rgrid + (size_t)(firstRow + r) * K2;
    for (int k = lane; k < K2; k += 64) {
      const float2 z = Z[tileAt<LN>(k, r >> 1)];
      out[k] = (r & 1) ? z.y : z.x;
    }
  }
}

// The gather, one thread per atom in cell order (a wave's atoms read nearby
// parts of the grid): the gradient summed over the support in FP32 and
// rounded to fixed point once.
__global__ void __launch_bounds__(256) pmeSlabGatherKernel(Dev d, PmeDev p) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= d.n) return;
  const float4 pos = d.slotPos[k];
  if (pos.w == 0.f) return;
  int base[3];
  float w[3][ORDER], dw[3][ORDER];
  for (int a = 0; a < 3; ++a) {
    float off;
    gridCoordinate(p, d.box->recip64, a, pos, base[a], off);
    bspline5(off, w[a], dw[a]);
  }
  int ix[ORDER], iy[ORDER], iz[ORDER];
  for (int q = 0; q < ORDER; ++q) {
    ix[q] = gridIndex(base[0], q, p.K[0]);
    iy[q] = gridIndex(base[1], q, p.K[1]);
    iz[q] = gridIndex(base[2], q, p.K[2]);
  }
  const GlobalPtr<float> grid = globalPtr(p.rgrid);
  float gu = 0.f, gv = 0.f, gw = 0.f;
  for (int a = 0; a < ORDER; ++a) {
    for (int b = 0; b < ORDER; ++b) {
      const GlobalPtr<float> row = grid + ((size_t)ix[a] * p.K[1] + iy[b]) * p.K[2];
      const float wxy = w[0][a] * w[1][b], dxy = dw[0][a] * w[1][b], xdy = w[0][a] * dw[1][b];
      for (int c = 0; c < ORDER; ++c) {
        const float v = row[iz[c]];
        gu += dxy * w[2][c] * v;
        gv += xdy * w[2][c] * v;
        gw += wxy * dw[2][c] * v;
      }
    }
  }
  addGridForce(d, p, d.cellAtoms[k], pos.w, gu, gv, gw);
}

// The lines per tile of an axis: 16 while two workgroups share a CU's LDS
// (axes up to 284, or 182 with the charges), then 8 while one fits, then 4
// (1024 with the charges: 122 KB).
static int tileLines(int K, bool charges, size_t maxLds) {
  constexpr size_t TWO_PER_CU = 80 * 1024;
  if ((charges ? slabLds<16>(K) : tileLds<16>(K)) <= TWO_PER_CU) return 16;
  if ((charges ? slabLds<8>(K) : tileLds<8>(K)) <= maxLds) return 8;
  return 4;
}

template <typename F>
static void withLines(int lines, F f) {
  if (lines == 16)
    f(std::integral_constant<int, 16>());
  else if (lines == 8)
    f(std::integral_constant<int, 8>());
  else
    f(std::integral_constant<int, 4>());
}

static int slabsOf(const PmeDev &p) {
  return (p.K[0] * p.K[1] + 2 * p.slabLines[2] - 1) / (2 * p.slabLines[2]);
}
static int chunksOf(const PmeDev &p, int axis) { return (p.K2h + p.slabLines[axis] - 1) / p.slabLines[axis]; }

static void launchSlabForward(const Dev &d, const PmeDev &p, const float *real, hipStream_t s) {
  withLines(p.slabLines[2], [&](auto n) {
    constexpr int LN = decltype(n)::value;
    pmeSlabForwardKernel<LN><<<slabsOf(p), SLAB_THREADS, slabLds<LN>(p.K[2]), s>>>(d, p, real);
  });
}
static void launchTileY(const PmeDev &p, int sign, hipStream_t s) {
  withLines(p.slabLines[1], [&](auto n) {
    constexpr int LN = decltype(n)::value;
    const int chunks = chunksOf(p, 1);
    pmeTileYKernel<LN><<<p.K[0] * chunks, SLAB_THREADS, tileLds<LN>(p.K[1]), s>>>(p, sign, chunks);
  });
}
// Returns the energy slots written.
static int launchTileX(const Dev &d, const PmeDev &p, int convolve, int energies, hipStream_t s) {
  const int chunks = chunksOf(p, 0), blocks = std::min(p.K[1] * chunks, MAX_SLOTS);
  withLines(p.slabLines[0], [&](auto n) {
    constexpr int LN = decltype(n)::value;
    pmeTileXKernel<LN><<<blocks, SLAB_THREADS, tileLds<LN>(p.K[0]), s>>>(d, p, convolve, energies, chunks);
  });
  return blocks;
}
static void launchSlabInverse(const PmeDev &p, hipStream_t s) {
  withLines(p.slabLines[2], [&](auto n) {
    constexpr int LN = decltype(n)::value;
    pmeSlabInverseKernel<LN><<<slabsOf(p), SLAB_THREADS, tileLds<LN>(p.K[2]), s>>>(p);
  });
}

// The influence function over the half spectrum, in FP64, stored as f32:
// pref * exp(-pi^2 m^2 / alpha^2) / (m^2 * B(m)) with the reference's row
// convention for the wave vector (cpu/forces/pme.js:176-209).
__device__ __forceinline__ void pmeInfluence(const PmeDev &p, const BoxF *box, const double *mod0, const double *mod1,
                                             const double *mod2, double alpha, size_t idx) {
  const double *recip = box->recip64;
  const double *bx = box->box64;
  const double volume = bx[0] * bx[4] * bx[8];
  const size_t total = (size_t)p.K[0] * p.K[1] * p.K2h;
  if (idx >= total) return;
  const int m = idx % p.K2h;
  const int y = (idx / p.K2h) % p.K[1];
  const int x = idx / ((size_t)p.K2h * p.K[1]);
  const int kx = x <= p.K[0] / 2 ? x : x - p.K[0];
  const int ky = y <= p.K[1] / 2 ? y : y - p.K[1];
  const int kz = m;
  if (kx == 0 && ky == 0 && kz == 0) {
    p.influence[idx] = 0.f;
    return;
  }
  const double mx = kx * recip[0] + ky * recip[1] + kz * recip[2];
  const double my = kx * recip[3] + ky * recip[4] + kz * recip[5];
  const double mz = kx * recip[6] + ky * recip[7] + kz * recip[8];
  const double m2 = mx * mx + my * my + mz * mz;
  const double factor = M_PI * M_PI / (alpha * alpha);
  const double pref = 138.935456 / (2.0 * M_PI * volume);
  const double modulus = mod0[x] * mod1[y] * mod2[m];
  p.influence[idx] = (float)(pref * exp(-factor * m2) / (m2 * modulus));
}

// Batched: the replicas whose box changed.
__global__ void __launch_bounds__(256) pmeInfluenceBatchKernel(const BatchView *__restrict__ v,
                                                               const int2 *__restrict__ task) {
  const int2 t = task[blockIdx.x];
  if (t.x < 0 || !v[t.x].boxChanged) return;
  const BatchView &b = v[t.x];
  pmeInfluence(b.p, b.d.box, b.moduli[0], b.moduli[1], b.moduli[2], b.alpha,
               (size_t)t.y * blockDim.x + threadIdx.x);
}

// The folded gathers' kernel X(l, c) = sum_k 2 g(k, c) exp(-2 pi i k l / K0)
// (PmeDev::xFolded), one thread per (l, c), summed in FP64 over ascending k,
// the roots from the x axis' twiddle table (exp(+2 pi i r / K0) at the
// numerator r = k l reduced modulo K0); for a rectangular box g is even in k
// and X real (the sine terms cancel), stored as its real part.
__global__ void pmeXKernelKernel(PmeDev p) {
  const int K0 = p.K[0], PK = p.K[1] * p.K2h;
  const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (size_t)K0 * PK) return;
  const int l = (int)(idx / PK), c = (int)(idx - (size_t)l * PK);
  // the column's influence values loaded together (K0 <= X_FOLD_MAX_K), not
  // one dependent round trip per term
  float g[X_FOLD_MAX_K];
#pragma unroll
  for (int k = 0; k < X_FOLD_MAX_K; ++k) g[k] = k < K0 ? p.influence[(size_t)k * PK + c] : 0.f;
  double re = 0.0, im = 0.0;
  int r = 0;  // k l mod K0
#pragma unroll
  for (int k = 0; k < X_FOLD_MAX_K; ++k) {
    if (k >= K0) break;
    const float2 w = p.twiddle[0][r];
    re += 2.0 * (double)g[k] * (double)w.x;
    im -= 2.0 * (double)g[k] * (double)w.y;
    r += l;
    r -= r >= K0 ? K0 : 0;
  }
  if (p.xReal)
    p.xKernel[idx] = (float)re;
  else
    reinterpret_cast<float2 *>(p.xKernel)[idx] = make_float2((float)re, (float)im);
}

// A single system's box change in one launch: the box by value, stored to
// the device box by the first thread, and the influence function from it.
__global__ void pmeSetBoxAndInfluenceKernel(PmeDev p, BoxF box, BoxF *dst, const double *mod0, const double *mod1,
                                            const double *mod2, double alpha) {
  const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx == 0) *dst = box;
  pmeInfluence(p, &box, mod0, mod1, mod2, alpha, idx);
}

__global__ void pmeSetBoxAndInfluenceFromKernel(PmeDev p, const BoxF *box, BoxF *dst, const double *mod0,
                                                const double *mod1, const double *mod2, double alpha) {
  const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx == 0) *dst = *box;
  pmeInfluence(p, box, mod0, mod1, mod2, alpha, idx);
}

void pmeSetBoxAndInfluenceFrom(const PmeDev &p, const BoxF *box, BoxF *dst, const double *moduli[3], double alpha,
                               hipStream_t s) {
  const size_t total = (size_t)p.K[0] * p.K[1] * p.K2h;
  pmeSetBoxAndInfluenceFromKernel<<<(unsigned)((total + 255) / 256), 256, 0, s>>>(p, box, dst, moduli[0], moduli[1],
                                                                                  moduli[2], alpha);
  if (p.xKernel) pmeXKernelKernel<<<(unsigned)((total + 255) / 256), 256, 0, s>>>(p);
}

void pmeSetBoxAndInfluence(const PmeDev &p, const BoxF &box, BoxF *dst, const double *moduli[3], double alpha,
                           hipStream_t s) {
  const size_t total = (size_t)p.K[0] * p.K[1] * p.K2h;
  pmeSetBoxAndInfluenceKernel<<<(unsigned)((total + 255) / 256), 256, 0, s>>>(p, box, dst, moduli[0], moduli[1],
                                                                              moduli[2], alpha);
  if (p.xKernel) pmeXKernelKernel<<<(unsigned)((total + 255) / 256), 256, 0, s>>>(p);
}

// ---- configuration and launchers --------------------------------------------

// LDS: twiddles, two complex work buffers (the second also holds the int64
// charge plane), then the compacted atom list and its count.
// (or the waves' queues of the wide kernel's cell scan)
static size_t listBytes() {
  return std::max((size_t)PLANE_LIST * sizeof(PlaneEntry) + 4 * sizeof(int),
                  (size_t)WIDE_PLANE_THREADS / 64 * QUEUE_ENTRIES * sizeof(PlaneEntry));
}
size_t planeForwardLds(const PmeDev &p) {
  return (size_t)(p.K[1] + p.K[2] + p.planeSpan + p.planeRegion) * sizeof(float2) + listBytes();
}
size_t planeGatherLds(const PmeDev &p) {
  return (size_t)(p.K[1] + p.K[2]) * sizeof(float2) + 2 * (size_t)p.planeSpan * sizeof(float2) + listBytes();
}
size_t xLinesLds(const PmeDev &p) { return (size_t)p.K[0] * sizeof(float2) * (1 + 2 * XLINES); }

bool pmeConfigure(PmeDev &p, int mode, size_t maxLds) {
  const int P = (p.K[1] + 1) / 2;
  const int a = P * p.K[2], b = p.K2h * p.K[1];
  p.planeSpan = a > b ? a : b;
  const int planeWords = (p.K[1] * p.K[2] * (int)sizeof(long long) + (int)sizeof(float2) - 1) / (int)sizeof(float2);
  p.planeRegion = p.planeSpan > planeWords ? p.planeSpan : planeWords;
  const size_t need = std::max(planeForwardLds(p), planeGatherLds(p));
  const bool fits = need <= maxLds && xLinesLds(p) <= maxLds;
  p.planes = (mode == PME_PLANES || mode == PME_AUTO) && fits ? 1 : 0;
  if (p.planes) {
    (void)hipFuncSetAttribute((const void *)pmePlaneForwardKernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                              (int)planeForwardLds(p));
    (void)hipFuncSetAttribute((const void *)pmePlaneGatherKernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                              (int)planeGatherLds(p));
    (void)hipFuncSetAttribute((const void *)pmePlaneForwardWideKernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                              (int)planeForwardLds(p));
  }
  p.slabLines[0] = tileLines(p.K[0], false, maxLds);
  p.slabLines[1] = tileLines(p.K[1], false, maxLds);
  p.slabLines[2] = tileLines(p.K[2], true, maxLds);
  if (!p.planes) {
    auto allow = [](const void *kernel, size_t lds) {
      (void)hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    };
    withLines(p.slabLines[0], [&](auto n) {
      constexpr int LN = decltype(n)::value;
      allow((const void *)pmeTileXKernel<LN>, tileLds<LN>(p.K[0]));
    });
    withLines(p.slabLines[1], [&](auto n) {
      constexpr int LN = decltype(n)::value;
      allow((const void *)pmeTileYKernel<LN>, tileLds<LN>(p.K[1]));
    });
    withLines(p.slabLines[2], [&](auto n) {
      constexpr int LN = decltype(n)::value;
      allow((const void *)pmeSlabForwardKernel<LN>, slabLds<LN>(p.K[2]));
      allow((const void *)pmeSlabInverseKernel<LN>, tileLds<LN>(p.K[2]));
    });
  }
  return mode != PME_PLANES || fits;
}

static int xLineBlocks(const PmeDev &p) { return p.K[1] * ((p.K2h + XLINES - 1) / XLINES); }
int pmeXLineBlocks(const PmeDev &p) { return xLineBlocks(p); }
// For a PLANE_THREADS-thread workgroup. (A batch member's planes never use the
// scan list: its LDS is left out; by cells only the waves' queues are used.)
size_t pmePlaneForwardLds(const PmeDev &p) {
  const size_t queues = (size_t)PLANE_THREADS / 64 * QUEUE_ENTRIES * sizeof(PlaneEntry);
  return planeForwardLds(p) - (p.atoms == PME_ATOMS_SCAN ? 0 : listBytes()) +
         (p.atoms == PME_ATOMS_CELLS ? queues : 0);
}
size_t pmeXLinesLds(const PmeDev &p) { return xLinesLds(p); }
size_t pmePlaneGatherLds(const PmeDev &p) {
  return planeGatherLds(p) - (p.atoms == PME_ATOMS_BINS ? listBytes() : 0);
}

// Batched plane pipeline; the LDS sizes are the largest over the replicas and
// the kernels' LDS limits were raised to them at batch creation.
void launchPmeBatch(const BatchView *v, const TaskTable &planes, const TaskTable &xlines, const TaskTable &replicas,
                    const TaskTable &atoms256, int energies, size_t forwardLds, size_t xlinesLds, size_t gatherLds,
                    hipStream_t s) {
  pmeBinBatchKernel<<<replicas.blocks, BIN_THREADS, 0, s>>>(v, replicas.task);
  pmePlaneForwardBatchKernel<<<planes.blocks, PLANE_THREADS, forwardLds, s>>>(v, planes.task);
  pmeXLinesBatchKernel<<<xlines.blocks, XLINE_THREADS, xlinesLds, s>>>(v, xlines.task, energies);
  pmePlaneGatherBatchKernel<<<planes.blocks, PLANE_THREADS, gatherLds, s>>>(v, planes.task);
  pmeAtomGatherBatchKernel<<<atoms256.blocks, 256, 0, s>>>(v, atoms256.task);
}

void launchInfluenceBatch(const BatchView *v, const TaskTable &t, hipStream_t s) {
  pmeInfluenceBatchKernel<<<t.blocks, 256, 0, s>>>(v, t.task);
}

void pmeBatchLdsLimits(size_t forwardLds, size_t xlinesLds, size_t gatherLds) {
  (void)hipFuncSetAttribute((const void *)pmePlaneForwardBatchKernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                            (int)forwardLds);
  (void)hipFuncSetAttribute((const void *)pmeXLinesBatchKernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                            (int)xlinesLds);
  (void)hipFuncSetAttribute((const void *)pmePlaneGatherBatchKernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                            (int)gatherLds);
}

// Stages 0 (the spread with the forward transforms it carries), 1 (the
// remaining transforms with the convolution; nothing where a force-only plane
// chain folds the x lines into the gathers) and 2 (the inverse transforms with
// the gather); returns stage 1's energy slots.
static int launchStage(const Dev &d, const PmeDev &p, int energies, hipStream_t s, int stage) {
  if (!p.planes) {
    if (stage == 0) {
      launchSlabForward(d, p, nullptr, s);
    } else if (stage == 1) {
      launchTileY(p, +1, s);
      const int slots = launchTileX(d, p, 1, energies, s);
      launchTileY(p, -1, s);
      return slots;
    } else {
      launchSlabInverse(p, s);
      pmeSlabGatherKernel<<<(d.n + 255) / 256, 256, 0, s>>>(d, p);
    }
    return 0;
  }
  const int folded = p.xFolded && !energies && p.atoms == PME_ATOMS_SCAN;
  if (stage == 0) {
    if (p.atoms == PME_ATOMS_BINS) pmeBinKernel<<<1, BIN_THREADS, 0, s>>>(d, p);
    launchPlaneForward(d, p, planeForwardLds(p), s);
  } else if (stage == 1) {
    if (!folded) pmeXLinesKernel<<<xLineBlocks(p), XLINE_THREADS, xLinesLds(p), s>>>(d, p, 1, energies);
    return xLineBlocks(p);
  } else {
    launchPlaneGather(d, p, planeGatherLds(p), s, folded);
    if (p.atoms != PME_ATOMS_SCAN) pmeAtomGatherKernel<<<(d.n + 255) / 256, 256, 0, s>>>(d, p);
  }
  return 0;
}

int launchPmeAfterForward(const Dev &d, const PmeDev &p, int energies, hipStream_t s) {
  const int slots = launchStage(d, p, energies, s, 1);
  launchStage(d, p, energies, s, 2);
  return slots;
}

int launchPme(const Dev &d, const PmeDev &p, int energies, hipStream_t s, int *slotsUsed) {
  launchStage(d, p, energies, s, 0);
  const int slots = launchPmeAfterForward(d, p, energies, s);
  if (slotsUsed) *slotsUsed = slots;
  return slots;
}

// One stage of launchPme's chain (no energies), for per-stage timing.
void launchPmeStage(const Dev &d, const PmeDev &p, hipStream_t s, int stage) { launchStage(d, p, 0, s, stage); }

bool pmeTransformsFolded(const PmeDev &p) { return p.planes && p.xFolded && p.atoms == PME_ATOMS_SCAN; }

// Verification entry: the forward R2C 3D transform of a real grid, through
// the same kernels as the active pipeline.
__global__ void copyComplexKernel(PmeDev p, float2 *out) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (size_t)p.K[0] * p.K[1] * p.K2h) return;
  out[i] = p.cgrid[i];
}

void launchFftForward(const Dev &d, const PmeDev &p, const float *real, float2 *out, hipStream_t s) {
  if (p.planes) {
    pmePlaneForwardKernel<<<p.K[0], PLANE_THREADS, planeForwardLds(p), s>>>(d, p, real);
    pmeXLinesKernel<<<xLineBlocks(p), XLINE_THREADS, xLinesLds(p), s>>>(d, p, 0, 0);
  } else {
    launchSlabForward(d, p, real, s);
    launchTileY(p, +1, s);
    launchTileX(d, p, 0, 0, s);
  }
  const size_t nc = (size_t)p.K[0] * p.K[1] * p.K2h;
  copyComplexKernel<<<(unsigned)((nc + 255) / 256), 256, 0, s>>>(p, out);
}

}  // namespace rmd
