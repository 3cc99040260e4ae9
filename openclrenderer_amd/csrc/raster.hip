// raster.hip — prearrange (transform, near clip, cull, sample count), the
// depth pass (u32 atomicMin) and the id pass (u64 atomicMax on a packed key),
// for camera views and for cube shadow maps.
//
// Reference: prearrange cl2.cl:4271-4409, kernel1 cl2.cl:4985-5127,
// kernel2 cl2.cl:5390-5546, prearrange_realtime_shadowing cl2.cl:4419-4636,
// kernel1_realtime_shadowing cl2.cl:5129-5246.
//
// Work decomposition.  The reference cuts every triangle's bounding box into
// fragments of op_size pixels and runs one work item per fragment; a fragment
// walks the samples q = pa .. pa + op_size (pa = op_size * chunk) with a
// running cursor and stops at the first row >= max_y.  Fragments hold from 1
// to op_size + 1 samples, so one work item per fragment leaves most lanes of
// a wavefront idle.  Here prearrange computes each cut triangle's exact
// sample count over all of its fragments and appends the triangle with its
// range in a sample space: one packed 64-bit atomicAdd per block returns both
// the record index and the sample offset, so each partition of the cut list
// is sorted by sample offset and its ranges tile [0, total).  The raster
// passes split the sample spaces into equal chunks: a wavefront finds the
// chunk's first triangle with a 64-ary search, stages 64 triangles, one per
// lane, and draws their rows with all lanes.  No per-fragment records exist.
#pragma clang fp contract(off)

#include <stdlib.h>
#include <string.h>

#include <algorithm>

#include "ocr_internal.h"
#include "setup.h"
#include "tiles.h"
#include "walk.h"

namespace ocr {

// Prearrange blocks: one triangle per work item, kPreThreads (256) of them.
// Cut records and sample ranges are allocated once per block (one 64-bit
// atomicAdd on the packed counter (cuts << 32 | samples) of the block's
// partition).  The next render's prearrange runs beside the current render's
// shading, whose wavefronts fill most of a SIMD's registers (five of 88 when this
// was measured, six of 80 now): a block of four wavefronts with at most 72
// finds room on a CU at once or as soon as one of them ends, where a block of
// eight with 90 waited until the CU had drained (prearrange 36 us alone,
// 200-260 us beside shading).  With the counters zeroed by the clear
// and pieces that cover nothing left out: 1280x719, 120,000 triangles
// 88.8 -> 81.0 us, 1080p, 1 M triangles 194.8 -> 188.2, the 16-light 4K frame
// 5.00 -> 4.88 ms.
// Lists of one partition (reserved or tiled) use blocks of 512, which append
// half as often to the one counter.
constexpr int kPreThreadsOne = 512;
constexpr int kShadowPreThreads = 256;   // independent wavefronts: 113 VGPRs and 8.5 KB of LDS each, 16 on a CU

template <int kWaves>
struct BlockAllocLds {
  uint32_t cuts[kWaves], smps[kWaves], frags[kWaves], more[kWaves];
  unsigned long long base;
  uint32_t ok, any_more;
};

// Appends ncut (0 or 1) records holding nsmp samples per work item to the
// block's partition; `seen` pieces of nfrag fragments count in the
// statistics.  Returns false (for the whole block) when the block's records
// do not fit the partition or its sample space; the overflow word then says
// which.  The block's sample total is checked before its atomic, and each
// atomic adds less than kMaxSamples, so the low half reaches the threshold
// and sets the flag before it could carry into the record count.  more: in,
// whether the work item has another piece; out, whether any of the block has.
template <int kWaves>
__device__ __forceinline__ bool block_alloc(const Lists& L, BlockAllocLds<kWaves>& sh, uint32_t ncut, uint32_t nsmp,
                                            uint32_t seen, uint32_t nfrag, bool& more, uint32_t& cut0, uint32_t& smp0) {
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  const unsigned long long cut_lanes = __ballot(ncut != 0u);
  const uint32_t is = wave_incl_scan(nsmp), ifr = wave_incl_scan(nfrag);
  const uint32_t nseen = (uint32_t)__popcll(__ballot(seen != 0u));
  const unsigned long long more_lanes = __ballot(more);
  if (lane == kWave - 1) {
    sh.cuts[wave] = (uint32_t)__popcll(cut_lanes) | nseen << 16;
    sh.smps[wave] = is;
    sh.frags[wave] = ifr;
    sh.more[wave] = more_lanes != 0ull;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t tc = 0, tn = 0, tf = 0, tm = 0;
    unsigned long long ts = 0;
    for (int w = 0; w < kWaves; w++) {
      const uint32_t c = sh.cuts[w], sm = sh.smps[w];
      sh.cuts[w] = tc;
      sh.smps[w] = (uint32_t)ts;
      tc += c & 0xFFFFu;
      tn += c >> 16;
      ts += sm;
      tf += sh.frags[w];
      tm |= sh.more[w];
    }
    const uint32_t part = blockIdx.x & (L.parts - 1u), cap = L.cap_cut / L.parts;
    uint32_t bad = ts > kMaxSamples ? kOverflowSamples : 0u;
    unsigned long long base = 0;
    if (!bad && tc) {
      base = atomicAdd(reinterpret_cast<unsigned long long*>(L.counters + kPartWord(part)),
                       ((unsigned long long)tc << 32) + ts);
      const unsigned long long end = base + ((unsigned long long)tc << 32) + ts;
      if ((end >> 32) > cap) bad |= kOverflowCuts;
      if ((uint32_t)end > kMaxSamples) bad |= kOverflowSamples;
    }
    // Pieces and fragments in one add.  A block has at most two appends: those
    // with fragments below 2^31 / gridDim.x cannot together carry into the
    // pieces; the others (no ordinary frame's) add theirs apart.
    if (tn) {
      const bool apart = ((unsigned long long)tf * gridDim.x >> 31) != 0ull;
      atomicAdd(reinterpret_cast<unsigned long long*>(L.counters + kFragCount),
                ((unsigned long long)tn << 32) + (apart ? 0u : tf));
      if (apart) atomicAdd(&L.counters[kFragMore], tf);
    }
    if (bad) atomicOr(&L.counters[kOverflow], bad);
    sh.base = base + ((unsigned long long)(part * cap) << 32);
    sh.ok = bad == 0;
    sh.any_more = tm;
  }
  __syncthreads();
  const unsigned long long base = sh.base;
  cut0 = (uint32_t)(base >> 32) + sh.cuts[wave] + lanes_below(cut_lanes);
  smp0 = (uint32_t)base + sh.smps[wave] + is - nsmp;
  const bool ok = sh.ok != 0;
  more = sh.any_more != 0;
  __syncthreads();   // the LDS record is reused by the block's next allocation
  return ok;
}

__device__ __forceinline__ void store_cut(CutTri* dst, const f3 p[3], float rconst, uint32_t oid, uint32_t view) {
  CutTri c;
  c.oid = oid | (front_facing(p[0], p[1], p[2]) ? kCutFront : 0u);
  c.view = view;
  c._pad[0] = c._pad[1] = c._pad[2] = 0u;
  // the plane kernel3's get_vtdiff builds per pixel (cl2.cl:5691-5760)
  const f3 xpv = mk3(roundf(p[0].x), roundf(p[1].x), roundf(p[2].x));
  const f3 ypv = mk3(roundf(p[0].y), roundf(p[1].y), roundf(p[2].y));
  const f3 depths = mk3(rcp_rn(p[0].z), rcp_rn(p[1].z), rcp_rn(p[2].z));   // z in [20, 350000]
  plane_const(depths, xpv, ypv, rconst, c.da, c.db, c.dc);
  *dst = c;
}

// The 144-byte triangle into the 40-byte position record read by every raster
// pass and the 112-byte record read only by shading.  Bound by the 296 bytes a
// triangle it moves.
__global__ void __launch_bounds__(256) k_split(const uint4* __restrict__ tris, uint32_t n, TriPos* __restrict__ pos,
                                               TriAttr* __restrict__ attr) {
  const uint32_t id = blockIdx.x * 256u + threadIdx.x;
  if (id >= n) return;
  TriPos P;
  TriAttr A;
#pragma unroll
  for (int v = 0; v < 3; v++) {
    // pos (4 words), normal (4), vt (2), object id, colour
    const uint4 p = tris[9 * (size_t)id + 3 * v], nm = tris[9 * (size_t)id + 3 * v + 1], r = tris[9 * (size_t)id + 3 * v + 2];
    A.p[3 * v] = P.p[3 * v] = __uint_as_float(p.x);
    A.p[3 * v + 1] = P.p[3 * v + 1] = __uint_as_float(p.y);
    A.p[3 * v + 2] = P.p[3 * v + 2] = __uint_as_float(p.z);
    A.n[3 * v] = __uint_as_float(nm.x);
    A.n[3 * v + 1] = __uint_as_float(nm.y);
    A.n[3 * v + 2] = __uint_as_float(nm.z);
    A.vt[2 * v] = __uint_as_float(r.x);
    A.vt[2 * v + 1] = __uint_as_float(r.y);
    A.col[v] = r.w;
    if (v == 0) P.oid = r.z;
  }
  A._pad = 0u;
  pos[id] = P;
  attr[id] = A;
}

hipError_t launch_split(const ocr_triangle* tris, uint32_t n, TriPos* pos, TriAttr* attr, hipStream_t s) {
  static_assert(sizeof(ocr_triangle) == 144 && sizeof(ocr_vertex) == 48, "record layout");
  if (n)
    hipLaunchKernelGGL(k_split, dim3((n + 255) / 256), dim3(256), 0, s, reinterpret_cast<const uint4*>(tris), n, pos, attr);
  return hipGetLastError();
}

// full_rotate_quat's object-to-world step (cl2.cl:700-729): the same for the
// camera and every light, so it is applied once per object update into the
// scene's world-space copy of its triangles.
__global__ void __launch_bounds__(256) k_world(const TriPos* __restrict__ tris, uint32_t ntri,
                                               const ObjDesc* __restrict__ objs, uint32_t nobj,
                                               TriPos* __restrict__ world) {
  const uint32_t id = blockIdx.x * blockDim.x + threadIdx.x;
  if (id >= ntri) return;
  const TriPos T = tris[id];
  TriPos W;
  W.oid = T.oid;
  if (T.oid < nobj) {
    const ObjDesc G = objs[T.oid];
    const f3 wp = mk3(G.wp[0], G.wp[1], G.wp[2]);
    // rot_quat's normalised quaternion, formed once per descriptor
    const f4 qn = f4{G.qn[0], G.qn[1], G.qn[2], G.qn[3]};
#pragma unroll
    for (int i = 0; i < 3; i++) {
      const f3 r = rot_quat_n(mk3(T.p[3 * i], T.p[3 * i + 1], T.p[3 * i + 2]) * G.scale, qn) + wp;
      W.p[3 * i] = r.x;
      W.p[3 * i + 1] = r.y;
      W.p[3 * i + 2] = r.z;
    }
  } else {
#pragma unroll
    for (int i = 0; i < 9; i++) W.p[i] = 0.f;
  }
  world[id] = W;
}

hipError_t launch_world(Scene* sc, hipStream_t s) {
  if (sc->ntri)
    hipLaunchKernelGGL(k_world, dim3((sc->ntri + 255) / 256), dim3(256), 0, s, sc->tri_pos, sc->ntri, sc->objs,
                       sc->nobj, sc->world);
  return hipGetLastError();
}

// Appends the work items' cut pieces that hold samples with their sample
// ranges; called by every work item of the block.  A block that would pass
// the list capacity or the sample limit writes nothing and sets the overflow
// word, which every later pass of the render checks before reading the list.
// For a tiled render (L.tb.bin set) also the records' tile boxes and their
// tiles' entry counts.  more: see block_alloc.
template <int kWaves>
__device__ __forceinline__ void append_cut(const Lists& L, BlockAllocLds<kWaves>& sh, Piece& P, uint32_t key,
                                           uint32_t oid, uint32_t view, uint32_t bin_begin, uint32_t tiles_x,
                                           bool& more) {
  const bool have = P.ns > 0u;
  uint32_t c, smp;
  if (!block_alloc(L, sh, have ? 1u : 0u, P.ns, P.seen, P.seen ? P.nf : 0u, more, c, smp)) return;
  uint4 box{};
  if (have) {
    store_cut(&L.cuts[c], P.p, P.rc, oid, view);
    P.rt.key = key | (P.rt.key & kKeyBoxForm);
    P.rt.sample_begin = smp;
    L.rast[c] = P.rt;
    if (L.tb.bin) {
      box = tile_box(P.rt, P.my, L.tb, bin_begin, tiles_x);
      L.tb.box[c] = box;
    }
  }
  if (L.tb.bin) {
    uint32_t* cnt = L.tb.cnt;
    const uint32_t ntiles = L.tb.ntiles;
    expand_tile_pairs(
        box, have, box, false,
        [cnt, ntiles](uint32_t t, uint32_t len) {
          if (t < ntiles) atomicAdd(&cnt[t], len);
          return 0u;
        },
        [](uint32_t, int, uint32_t, uint32_t) {});
  }
}

// ------------------------------------------------------------------ views
__device__ __forceinline__ const DevView& view_at(const PassArgs& a, uint32_t i) {
  return a.views ? a.views[i] : a.view0;
}
__device__ __forceinline__ const DevScene& scene_at(const PassArgs& a, uint32_t i) {
  return a.scenes ? a.scenes[i] : a.scene0;
}

// The view owning a 256-slot block: the last view whose range starts at or
// before `slot` (ranges are 256-aligned, so the answer is block-uniform).
enum class Range { Tri, Pix };
template <Range kR>
__device__ __forceinline__ uint32_t view_of(const PassArgs& a, uint32_t slot) {
  if (!a.views) return 0;
  uint32_t lo = 0, hi = a.nviews;
  while (hi - lo > 1) {
    uint32_t mid = (lo + hi) >> 1;
    const DevView& m = a.views[mid];
    uint32_t b = kR == Range::Tri ? m.tri_begin : m.pix_begin;
    if (b <= slot) lo = mid; else hi = mid;
  }
  return (uint32_t)__builtin_amdgcn_readfirstlane((int)lo);
}

// ------------------------------------------------------------------ clear
// Depth and ids of kClearSlots pixel slots, by one block of the prearrange
// launch (bound by the 12 bytes a pixel it writes).  The clear and prearrange
// touch nothing in common, and a launch of its own costs small frames 2 us and
// the gap before the next one 5 (thumbnail alone 70 -> 53 us with the counters
// zeroed on the side); together they take 59 us on a 12-view, 10 Mpixel batch
// that took 51 + 36.  2048 to 16384 slots a block measure alike.
constexpr uint32_t kClearSlots = 8192;
template <int kThreads>
__device__ __forceinline__ void clear_block(const PassArgs& a, uint32_t block) {
  uint32_t at = block * kClearSlots;
  const uint32_t end = min(at + kClearSlots, a.pix_slots);
  // the views of the block's slots (ranges start at multiples of 256)
  for (uint32_t vi = view_of<Range::Pix>(a, at); at < end; vi++) {
    const DevView& V = view_at(a, vi);
    const uint32_t first = V.pix_begin, npix = V.v.width * V.v.height;
    const uint32_t stop = a.views && vi + 1 < a.nviews ? min(end, a.views[vi + 1].pix_begin) : end;
    uint32_t* const depth = V.depth;
    unsigned long long* const ids = V.idkey;
    const uint32_t i0 = at - first, i1 = min(stop - first, npix);
    if ((((uintptr_t)depth | (uintptr_t)ids) & 15u) == 0u) {
      // four pixels per work item: one 16-byte and two 16-byte stores
      uint4* const d4 = reinterpret_cast<uint4*>(depth);
      uint4* const k4 = reinterpret_cast<uint4*>(ids);
      const uint4 ones = make_uint4(0xFFFFFFFFu, 0xFFFFFFFFu, 0xFFFFFFFFu, 0xFFFFFFFFu), zero = make_uint4(0, 0, 0, 0);
      for (uint32_t i = i0 / 4 + threadIdx.x; i < i1 / 4; i += kThreads) d4[i] = ones;
      for (uint32_t i = i0 / 2 + threadIdx.x; i < i1 / 2; i += kThreads) k4[i] = zero;
      const uint32_t rest = (i1 & ~3u) + threadIdx.x;
      if (rest >= i0 && rest < i1) {
        depth[rest] = 0xFFFFFFFFu;
        ids[rest] = 0ull;
      }
    } else {
      for (uint32_t i = i0 + threadIdx.x; i < i1; i += kThreads) {
        depth[i] = 0xFFFFFFFFu;
        ids[i] = 0ull;
      }
    }
    at = stop;
  }
}

__global__ void __launch_bounds__(256) k_zero_work(uint32_t* __restrict__ c) {
  for (uint32_t i = threadIdx.x; i < (uint32_t)kListCounterWords; i += 256u) c[i] = 0u;
}

hipError_t launch_zero_work(uint32_t* counters, hipStream_t s) {
  hipLaunchKernelGGL(k_zero_work, dim3(1), dim3(256), 0, s, counters + kListCounterWords);
  return hipGetLastError();
}

__global__ void __launch_bounds__(256) k_fill_u32(uint32_t* __restrict__ p, uint32_t v, size_t n) {
  size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  size_t stride = (size_t)gridDim.x * blockDim.x;
  for (; i < n; i += stride) p[i] = v;
}

static unsigned grid_for(size_t n, unsigned block, unsigned max_blocks) {
  size_t b = (n + block - 1) / block;
  if (b < 1) b = 1;
  if (b > max_blocks) b = max_blocks;
  return (unsigned)b;
}

hipError_t launch_fill_u32(uint32_t* p, uint32_t value, size_t n, hipStream_t s) {
  hipLaunchKernelGGL(k_fill_u32, dim3(grid_for(n, 256, 8192)), dim3(256), 0, s, p, value, n);
  return hipGetLastError();
}

// ------------------------------------------------------------- prearrange
template <int kThreads>
__global__ void __launch_bounds__(kThreads) k_prearrange(PassArgs a) {
  __shared__ BlockAllocLds<kThreads / kWave> sh;
  const uint32_t tri_blocks = (a.tri_slots + (uint32_t)kThreads - 1u) / (uint32_t)kThreads;
  if (blockIdx.x >= tri_blocks) {
    clear_block<kThreads>(a, blockIdx.x - tri_blocks);
    return;
  }
  // per-view triangle ranges are 256-aligned: each wavefront has one view
  const uint32_t slot = blockIdx.x * (uint32_t)kThreads + (threadIdx.x & ~(uint32_t)(kWave - 1));
  const uint32_t vi = view_of<Range::Tri>(a, slot);
  const DevView& V = view_at(a, vi);
  const DevScene& S = scene_at(a, V.scene);
  const ViewParams& v = V.v;
  const uint32_t id = slot - V.tri_begin + (threadIdx.x & (kWave - 1));
  const float ew = (float)v.width, eh = (float)v.height;
  f3 tris[2][3];
  int num = 0;
  uint32_t oid = 0;
  bool two_sided = false;
  if (id < S.ntri) {
    const TriPos T = S.world[id];
    oid = T.oid;
    if (oid < S.nobj) {
      const ObjDesc& G = S.objs[oid];
      const f3 cpos = mk3(v.cpos[0], v.cpos[1], v.cpos[2]);
      two_sided = (G.flags & OCR_FEATURE_TWO_SIDED) > 0;
      const f3 to_obj = mk3(G.wp[0], G.wp[1], G.wp[2]) - cpos;
      if (!(dot(to_obj, to_obj) > kDepthFarSq)) {
        const f3 w[3] = {mk3(T.p[0], T.p[1], T.p[2]), mk3(T.p[3], T.p[4], T.p[5]), mk3(T.p[6], T.p[7], T.p[8])};
        num = face_clip(w, cpos, v.cam, tris);
      }
    }
  }
  // the second piece of a triangle cut by the near plane follows in an
  // append of its own, which a block without any skips
  Piece P;
  P.nf = P.seen = P.ns = 0u;
  if (num > 0) cut_piece(tris[0], v.fov, ew, eh, two_sided, kOpSize, P);
  bool more = num > 1;
  append_cut(a.lists, sh, P, 2u * id, oid, vi, V.bin_begin, V.bin_tiles_x, more);
  if (!more) return;
  P.nf = P.seen = P.ns = 0u;
  if (num > 1) cut_piece(tris[1], v.fov, ew, eh, two_sided, kOpSize, P);
  more = false;
  append_cut(a.lists, sh, P, 2u * id + 1u, oid, vi, V.bin_begin, V.bin_tiles_x, more);
}

template <int kThreads>
static void launch_prearrange_as(const PassArgs& a, hipStream_t s) {
  const uint32_t tri = (a.tri_slots + kThreads - 1) / kThreads;
  // a tiled render's tiles write every pixel
  const uint32_t clear = a.lists.tb.bin ? 0u : (a.pix_slots + kClearSlots - 1) / kClearSlots;
  if (tri + clear) hipLaunchKernelGGL(k_prearrange<kThreads>, dim3(tri + clear), dim3(kThreads), 0, s, a);
}

hipError_t launch_prearrange(const PassArgs& a, hipStream_t s) {
  if (a.lists.parts == 1 && a.tri_slots > 64 * kPreThreads)
    launch_prearrange_as<kPreThreadsOne>(a, s);
  else
    launch_prearrange_as<(int)kPreThreads>(a, s);
  return hipGetLastError();
}

// ------------------------------------------------- sample-chunk raster passes
//
// Sample s of a cut triangle (0 <= s < nsamples) is sample o = s % (op + 1)
// of fragment a = s / (op + 1), i.e. q = op*a + o with pa = op*a.  Its cursor
// position is the closed form of the reference's running (x, y):
//   y(q) = floor(fma(q, 1/width, min_y))
//   x(q) = (r % width) + min_x + (q - r)
// where r is the later of pa and the first index of q's row run (the cursor
// is reset to running_width_mod + min_x exactly when y changes, and starts at
// pa % width + min_x).  Row-run starts come from the nominal
// (Y - min_y) * width by stepping while y disagrees, so rows whose fma
// rounding lags or leads by a sample are reproduced exactly.


enum class RasterMode { Depth, Id, Shadow };

struct ShadowTarget {
  uint32_t* map;   // the group's first map: 6 faces of L x L per light, at most 2^31 texels in all
  uint32_t L;
};

// Raster work of one wavefront.  A stage is up to 64 set-up triangles, one
// per lane, each with a range of its samples.  Triangles whose samples are
// their box's pixels (box form) and whose edge functions are exact integers
// over the box (span_exact) are drawn by rows: each (triangle, row) pair of
// the stage goes to a lane, which solves the three edge inequalities for the
// row's run of covered columns; the runs' pixels are then spread over the
// lanes, 64 a step, and every one of them is a hit.  Testing each box pixel
// instead costs a step of ~80 instructions per 64 box pixels, of which a
// triangle covers a third: 1080p, 1 M triangles: 17.0 M box pixels, 2.05 M
// rows, 5.4 M covered pixels.  The other triangles (walk samples, edges too
// long for exact integers) are swept one after the other, sample by sample.
// That frame's depth pass issues 14.0 M vector instructions instead of 22.0 M;
// its time alone (78 us) is the memory side's: 0.75 M atomic and 1.7 M read
// requests.
// The stage takes 5 KB of LDS per wavefront, so that eight blocks of four fit
// on a CU (batches: six, their targets differ per triangle).
template <RasterMode kMode, bool kBatch>
struct TriLds {
  // staged triangles drawn by rows, compacted
  uint4 qa[kWave];       // min_x | w << 16, first row of the range | rows << 16, first row's index | lane << 24,
                         // first row's first column | last row's last column << 16
  float4 qb[kWave];      // e0, e1, e2, ceil(e6) - 1
  float4 qc[kWave];      // e3, e4, e5, A
  float2 qd[kWave];      // B, C
  // runs of covered columns, compacted
  uint4 run[kWave];      // pixel - index (shadow passes: the row's offset), x - index, B*y + C, A
  uint32_t ent[kMode == RasterMode::Shadow ? 0 : kWave];   // y << 16 | lane
  uint32_t start[kWave];                                   // start[p] == tick: an item begins at index base + p
  // per lane: its triangle's target
  uint32_t face[kMode == RasterMode::Shadow ? kWave : 0];  // the cube face's first texel
  uint32_t* dst[kBatch ? kWave : 0];
  uint32_t pitch[kBatch ? kWave : 0];
  unsigned long long* ids[kBatch && kMode == RasterMode::Id ? kWave : 0];
};

__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Which item owns index base + lane, for items that tile [0, n) in lane
// order (begin: the lane's item's first index, valid: whether it has one,
// each at least one long): the items beginning at or before `base` are a
// prefix of the valid lanes (one ballot), those beginning in (base, base +
// lane] are flagged in start[] by their lanes and counted.  tick: a value no
// earlier call of this wavefront left in start[].
template <typename Lds>
__device__ __forceinline__ int owner_of(Lds& L, bool valid, uint32_t begin, uint32_t base, uint32_t tick) {
  const int lane = threadIdx.x & (kWave - 1);
  const unsigned long long before = __ballot(valid && begin <= base);
  const uint32_t off = begin - base;
  if (valid && begin > base && off < (uint32_t)kWave) L.start[off] = tick;
  wave_lds_sync();
  const bool here = L.start[lane] == tick;
  return __popcll(before) - 1 + (int)lanes_below(__ballot(here)) + (here ? 1 : 0);
}

// Where a pass's samples go: one view's buffers or a group's shadow maps
// (batches: the staged triangles' own).  ent: the chunk's covered-sample
// entries (see CoverEntries), nent of them so far.  rast: the list (id pass).
struct RasterTarget {
  uint32_t pitch;
  uint32_t* depth;
  unsigned long long* ids;
  uint2* ent;
  uint32_t ent_cap, nent;
  const RasterTri* rast;
  MapLayout lay;   // shadow passes
};

// A pointer to device memory.  A batch's targets come from tables and LDS, where
// the compiler cannot tell; through generic pointers their loads and atomics
// count as LDS operations too, so that every later wait for LDS also waits for
// memory (12-view batch: depth pass 117.7 -> 115.9 us, ids 91.4 ->
// 89.6, 453 -> 451 in all).
template <typename T>
__device__ __forceinline__ __attribute__((address_space(1))) T* dev_ptr(T* p) {
  return (__attribute__((address_space(1))) T*)(uintptr_t)p;
}

// One covered sample per lane (hit lanes): depth d at pixel pix of dst.
// Called wave-uniformly.
template <RasterMode kMode, bool kBatch>
__device__ __forceinline__ void put_sample(RasterTarget& T, bool hit, uint32_t d, uint32_t pix, uint32_t xy,
                                           uint32_t rec, uint32_t* dst, unsigned long long* ids) {
  bool keep = false;
  if (hit) {
    if constexpr (kMode == RasterMode::Id) {
      const uint32_t val = dev_ptr(dst)[pix];
      if (d > val - kBufError && d < val + kBufError)
        __hip_atomic_fetch_max(dev_ptr(ids) + pix, ((unsigned long long)((T.rast[rec].key & ~kKeyBoxForm) + 1u) << 32) | rec,
                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    } else {
      // The L2 performs atomics at ~26.6 G cache-line operations/s; a plain
      // load first drops the samples that cannot win (the stored depth only
      // decreases, so d >= any value a load returns loses).  A single view's
      // buffer is addressed from its (uniform) base with a 32-bit offset.
      uint32_t val;
      if constexpr (kMode == RasterMode::Depth && !kBatch) {
        typedef __attribute__((address_space(1))) char gchar;
        typedef __attribute__((address_space(1))) uint32_t gu32;
        gu32* g = (gu32*)((gchar*)(uintptr_t)dst + pix * 4u);   // 32-bit byte offset: frames < 2^30 px
        val = *g;
        if (d < val) __hip_atomic_fetch_min(g, d, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      } else {
        val = dev_ptr(dst)[pix];
        if (d < val) __hip_atomic_fetch_min(dev_ptr(dst) + pix, d, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      // a sample at or beyond val + BUF_ERROR stays outside the id pass's
      // window of the final depth (<= val) unless val + BUF_ERROR wraps
      keep = val > 0xFFFFFFFFu - kBufError || d < val + kBufError;
    }
  }
  if constexpr (kMode == RasterMode::Depth) {
    if (T.ent) {
      const unsigned long long m = __ballot(keep);
      if (keep) {
        const uint32_t slot = T.nent + lanes_below(m);
        if (slot < T.ent_cap) T.ent[slot] = uint2{xy, rec};
      }
      T.nent += (uint32_t)__popcll(m);
    }
  }
}

// Draws a stage: the lane's triangle t, record rec (consecutive over the
// lanes), samples [b, e) of it (indices from its first; b >= e: none); face:
// its cube face's first texel (shadow passes); dst, pitch, ids: its target
// (batches).  tick: see owner_of, kept by the caller.  Called wave-uniformly.
template <RasterMode kMode, int kOp, bool kBatch>
__device__ __forceinline__ void raster_stage(TriLds<kMode, kBatch>& L, RasterTarget& T, const RasterTri& t,
                                             uint32_t rec, uint32_t b, uint32_t e, uint32_t face, uint32_t* dst,
                                             uint32_t pitch, unsigned long long* ids, uint32_t& tick) {
  constexpr bool kShadow = kMode == RasterMode::Shadow;
  const int lane = threadIdx.x & (kWave - 1);
  const bool active = b < e, box = (t.key & kKeyBoxForm) != 0u;
  // ---- the lane's rows
  const float i0 = (float)b, i1 = (float)(e - 1u);   // below 2^24
  const float r0 = floor_div(i0, t.w, t.iw), r1 = floor_div(i1, t.w, t.iw);
  const bool span = active && box && span_exact(t.ek, t.min_x + t.w, t.min_y + r1);
  const uint32_t nrows = span ? (uint32_t)(r1 - r0) + 1u : 0u;
  const uint32_t rows_incl = wave_incl_scan(nrows), row_begin = rows_incl - nrows;   // below 2^21
  const uint32_t rows = wave_total(rows_incl);
  const unsigned long long spans = __ballot(span);
  if (span) {
    const uint32_t p = lanes_below(spans);
    L.qa[p] = make_uint4((uint32_t)t.min_x | (uint32_t)t.w << 16, (uint32_t)(t.min_y + r0) | nrows << 16,
                         row_begin | (uint32_t)lane << 24,
                         (uint32_t)fmaf(-r0, t.w, i0) | (uint32_t)fmaf(-r1, t.w, i1) << 16);
    L.qb[p] = make_float4(t.ek[0], t.ek[1], t.ek[2], ceilf(t.ek[6]) - 1.f);
    L.qc[p] = make_float4(t.ek[3], t.ek[4], t.ek[5], t.A);
    L.qd[p] = make_float2(t.B, t.C);
  }
  if constexpr (kShadow) L.face[lane] = face;
  if constexpr (kBatch) {
    L.dst[lane] = dst;
    L.pitch[lane] = pitch;
    if constexpr (kMode == RasterMode::Id) L.ids[lane] = ids;
  }
  const uint32_t rec0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)(rec - (uint32_t)lane));
  for (uint32_t rb = 0; rb < rows; rb += kWave) {
    // ---- one row per lane
    const int k = owner_of(L, span, row_begin, rb, ++tick);
    uint32_t n = 0, y = 0, xs = 0, who = 0;
    float rowc = 0.f, pa = 0.f;
    if (rb + (uint32_t)lane < rows) {
      const uint4 qa = L.qa[k];
      const float4 qb = L.qb[k], qc = L.qc[k];
      const float2 qd = L.qd[k];
      const uint32_t r = rb + (uint32_t)lane - (qa.z & 0xFFFFFFu);
      y = (qa.y & 0xFFFFu) + r;
      const uint32_t min_x = qa.x & 0xFFFFu;
      const float fy = (float)y, fx = (float)min_x;
      float lo = r == 0u ? (float)(qa.w & 0xFFFFu) : 0.f;
      float hi = (float)(r + 1u == qa.y >> 16 ? qa.w >> 16 : (qa.x >> 16) - 1u);
      row_span(qb.x, qb.y, qb.z, qc.x, qc.y, qc.z, qb.w, fx, fy, lo, hi);
      n = hi >= lo ? (uint32_t)(hi - lo) + 1u : 0u;
      xs = min_x + (uint32_t)lo;
      pa = qc.w;
      rowc = fmaf(qd.x, fy, qd.y);
      who = qa.z >> 24;
    }
    const uint32_t incl = wave_incl_scan(n), begin = incl - n;
    const uint32_t total = wave_total(incl);
    const unsigned long long runs = __ballot(n > 0u);
    if (n) {
      const uint32_t p = lanes_below(runs);
      const uint32_t rp = kBatch ? L.pitch[kBatch ? who : 0] : T.pitch;
      // y and the pitch are below 2^16: the 24-bit multiply is exact
      const uint32_t row = kShadow ? map_row(T.lay, y) + L.face[kShadow ? who : 0] : __umul24(y, rp) + xs - begin;
      L.run[p] = make_uint4(row, xs - begin, __float_as_uint(rowc), __float_as_uint(pa));
      if constexpr (!kShadow) L.ent[p] = y << 16 | who;
    }
    // ---- the runs' pixels, one per lane per step
    if constexpr (kShadow) {
      // The depths of two steps are asked for before the first is used: a
      // shadow pass has nothing beside it that would fill its waits (4 M
      // triangles, 16 lights: 2.94 -> 2.86 ms the pass; three or four steps
      // give no more, and the camera passes, which run beside other renders,
      // gain nothing).
      constexpr int kSteps = 2;
      for (uint32_t base = 0; base < total; base += kSteps * kWave) {
        uint32_t d[kSteps], val[kSteps], pix[kSteps];
#pragma unroll
        for (int i = 0; i < kSteps; i++) {
          const uint32_t at = base + (uint32_t)(i * kWave), j = at + (uint32_t)lane;
          d[i] = val[i] = pix[i] = 0u;
          if (at >= total) continue;
          const int m = owner_of(L, n > 0u, begin, at, ++tick);
          if (j < total) {
            const uint4 R = L.run[m];
            const uint32_t x = j + R.y;
            d[i] = depth_quant(fmaf(__uint_as_float(R.w), (float)x, __uint_as_float(R.z)));
            pix[i] = R.x + map_col(T.lay, x);
            val[i] = T.depth[pix[i]];
          }
        }
#pragma unroll
        for (int i = 0; i < kSteps; i++)
          if (d[i] < val[i]) atomicMin(&T.depth[pix[i]], d[i]);
      }
      wave_lds_sync();   // the runs are rewritten by the next 64 rows
      continue;
    }
    for (uint32_t base = 0; base < total; base += kWave) {
      const int m = owner_of(L, n > 0u, begin, base, ++tick);
      const uint32_t j = base + (uint32_t)lane;
      const bool hit = j < total;
      uint32_t d = 0, pix = 0, xy = 0, rr = 0;
      uint32_t* to = T.depth;
      unsigned long long* ti = T.ids;
      if (hit) {
        const uint4 R = L.run[m];
        const uint32_t x = j + R.y;
        d = depth_quant(fmaf(__uint_as_float(R.w), (float)x, __uint_as_float(R.z)));
        pix = j + R.x;
        if constexpr (!kShadow) {
          const uint32_t E = L.ent[m];
          xy = x | (E & 0xFFFF0000u);
          rr = rec0 + (E & 63u);
          if constexpr (kBatch) {
            to = L.dst[E & 63u];
            if constexpr (kMode == RasterMode::Id) ti = L.ids[E & 63u];
          }
        }
      }
      put_sample<kMode, kBatch>(T, hit, d, pix, xy, rr, to, ti);
    }
    // the runs are rewritten by the next 64 rows
    wave_lds_sync();
  }
  // ---- the other triangles, one by one, their samples over the lanes
  unsigned long long left = __ballot(active && !span);
  while (left) {
    const int k = __ffsll((long long)left) - 1;
    left &= left - 1ull;
    auto f = [k](float v) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), k)); };
    auto u = [k](uint32_t v) { return (uint32_t)__builtin_amdgcn_readlane((int)v, k); };
    const uint32_t ub = u(b), ue = u(e), uk = u(t.key), uf = kShadow ? u(face) : 0u;
    const float min_x = f(t.min_x), min_y = f(t.min_y), w = f(t.w), iw = f(t.iw);
    const float A = f(t.A), B = f(t.B), C = f(t.C);
    const float e0 = f(t.ek[0]), e1 = f(t.ek[1]), e2 = f(t.ek[2]), e3 = f(t.ek[3]), e4 = f(t.ek[4]), e5 = f(t.ek[5]),
                e6 = f(t.ek[6]);
    uint32_t* to = T.depth;
    unsigned long long* ti = T.ids;
    uint32_t up = T.pitch;
    if constexpr (kBatch) {
      const uint64_t v = (uint64_t)(uintptr_t)dst;
      to = (uint32_t*)(uintptr_t)((uint64_t)u((uint32_t)(v >> 32)) << 32 | u((uint32_t)v));
      up = u(pitch);
    }
    if constexpr (kBatch && kMode == RasterMode::Id) {
      const uint64_t v = (uint64_t)(uintptr_t)ids;
      ti = (unsigned long long*)(uintptr_t)((uint64_t)u((uint32_t)(v >> 32)) << 32 | u((uint32_t)v));
    }
    for (uint32_t base = ub; base < ue; base += kWave) {
      const uint32_t j = base + (uint32_t)lane;
      bool hit = false;
      uint32_t d = 0, pix = 0, xy = 0;
      if (j < ue) {
        const float slf = (float)j;
        float x, y;
        if (uk & kKeyBoxForm) {
          y = row_of(slf, iw, min_y);
          const float xo = slf - (y - min_y) * w;
          x = min_x + xo;
          hit = !(xo >= w) && inside_tri(x, y, e0, e1, e2, e3, e4, e5, e6);
        } else {
          hit = sample_xy<kOp>(slf, min_x, min_y, w, iw, e0, e1, e2, e3, e4, e5, e6, x, y);
        }
        if (hit) {
          d = depth_quant(fmaf(A, x, fmaf(B, y, C)));
          const uint32_t xi = (uint32_t)(int)x, yi = (uint32_t)(int)y;
          xy = xi | yi << 16;
          pix = kShadow ? map_row(T.lay, yi) + map_col(T.lay, xi) + uf : __umul24(yi, up) + xi;
        }
      }
      put_sample<kMode, kBatch>(T, hit, d, pix, xy, rec0 + (uint32_t)k, to, ti);
    }
  }
}

// The id pass over the covered-sample entries the depth pass kept: the
// wavefront's chunks (wave0, wave0 + nwaves, ...) two at a time, their
// entries as one list (at most cap per chunk; a chunk with more is swept
// by the caller), four of the lane's entries at a time: the entries, then
// their records' depth planes and keys, then the depths there, then the
// window tests.  Each entry's depth is formed again as the depth pass formed
// it.  Two chunks per round halve the rounds of dependent loads a wavefront
// waits through.
template <bool kBatch>
__device__ __forceinline__ void id_from_entries(const PassArgs& a, const Lists& Ls, uint32_t wave0, uint32_t nwaves,
                                                uint32_t nchunks, uint32_t cap) {
  const int lane = threadIdx.x & (kWave - 1);
  constexpr int kPer = 4;
  const uint4* R = reinterpret_cast<const uint4*>(Ls.rast);   // 4 x uint4 per record
  for (uint32_t ca = wave0; ca < nchunks; ca += 2 * nwaves) {
    const uint32_t cb = ca + nwaves;
    const uint32_t na0 = Ls.ent.cnt[ca], nb0 = cb < nchunks ? Ls.ent.cnt[cb] : 0u;
    const uint32_t na = na0 <= cap ? na0 : 0u, nb = nb0 <= cap ? nb0 : 0u;
    const uint32_t n = na + nb;
    const uint2* Ea = Ls.ent.ent + (size_t)ca * cap;
    // entry e >= na of the list is entry e - na of chunk cb
    const uint2* Eb = Ls.ent.ent + (size_t)(cb < nchunks ? cb : ca) * cap;
    for (uint32_t e0 = 0; e0 < n; e0 += kPer * kWave) {
      uint2 v[kPer];
      uint32_t d[kPer], key[kPer], pix[kPer], val[kPer];
      uint32_t* dep[kPer];
      unsigned long long* ids[kPer];
#pragma unroll
      for (int i = 0; i < kPer; i++) {
        const uint32_t e = e0 + (uint32_t)lane + (uint32_t)(i * kWave);
        if (e < n) v[i] = e < na ? Ea[e] : Eb[e - na];
      }
#pragma unroll
      for (int i = 0; i < kPer; i++) {
        const uint32_t e = e0 + (uint32_t)lane + (uint32_t)(i * kWave);
        dep[i] = a.view0.depth;
        ids[i] = a.view0.idkey;
        uint32_t pitch = a.view0.v.width;
        if (e < n) {
          // RasterTri words 1 (key) and 5-7 (the 1/z plane A, B, C)
          const uint4 w0 = R[4 * (size_t)v[i].y], w1 = R[4 * (size_t)v[i].y + 1];
          if constexpr (kBatch) {
            // a batch's entries hold pixels of their record's view
            const DevView& V = a.views[Ls.cuts[v[i].y].view];
            dep[i] = V.depth;
            ids[i] = V.idkey;
            pitch = V.v.width;
          }
          const float x = (float)(v[i].x & 0xFFFFu), y = (float)(v[i].x >> 16);
          d[i] = depth_quant(fmaf(__uint_as_float(w1.y), x, fmaf(__uint_as_float(w1.z), y, __uint_as_float(w1.w))));
          key[i] = w0.y & ~kKeyBoxForm;
          pix[i] = (v[i].x >> 16) * pitch + (v[i].x & 0xFFFFu);
        }
      }
#pragma unroll
      for (int i = 0; i < kPer; i++) {
        const uint32_t e = e0 + (uint32_t)lane + (uint32_t)(i * kWave);
        if (e < n) val[i] = dev_ptr(dep[i])[pix[i]];
      }
#pragma unroll
      for (int i = 0; i < kPer; i++) {
        const uint32_t e = e0 + (uint32_t)lane + (uint32_t)(i * kWave);
        if (e < n && d[i] > val[i] - kBufError && d[i] < val[i] + kBufError)
          __hip_atomic_fetch_max(dev_ptr(ids[i]) + pix[i], ((unsigned long long)(key[i] + 1u) << 32) | v[i].y,
                                 __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
  }
}

// Samples per chunk (log2) of a pass, from its sample count: the smallest power
// of two from 2^kChunkMinLog2 that leaves about kChunkTarget chunks, one or
// two per resident wavefront, up to kChunk.  A chunk is one wavefront's serial
// work: with 2048-sample chunks whatever the total, frames of a few hundred
// thousand samples occupied a few hundred of the chip's 8192 wavefronts for
// 30 us; above 16.8 M samples (1080p, 1 M triangles) chunks stay at kChunk.
// Depth / id pass alone with this rule and the row form: 800x600, 2,500
// triangles 31 -> 7.6 / 26 -> 6.2 us; 1080p, 50,000 triangles seen close
// 29 -> 6.2 / 14 -> 6.1 us; the 1280x719, 120,000-triangle frame 130 -> 109
// us in all.
constexpr int kChunkMinLog2 = 7;
constexpr uint32_t kChunkTarget = 8192;
// Shadow passes have no other render's raster beside them and up to 2^36
// samples; finding a chunk's first record reads ~150 lines of the list.  Up to
// 8192 samples a chunk (16 lights, 4 M triangles: 90 M samples): 866 -> 815 us
// alone, the whole pass 3.03 -> 2.94 ms; 4096: 805 us, 2.98 ms.
// They begin to grow at twice the camera's chunks, two to four per resident
// wavefront: large triangles' chunks differ in what they cover, and with one or
// less per wavefront the longest set the pass's time (a two-sided room of
// 12,288 triangles around 4 lights 249 -> 236 us a pass, of 768 355 -> 341;
// passes of more samples have kShadowChunkLog2 either way).
constexpr int kShadowChunkLog2 = 13;
constexpr uint32_t kShadowChunkTarget = 16384;
template <RasterMode kMode>
__device__ __forceinline__ int chunk_log2(uint32_t units) {   // units of 2^kChunkMinLog2 samples
  constexpr uint32_t kTarget = kMode == RasterMode::Shadow ? kShadowChunkTarget : kChunkTarget;
  constexpr int kMost = kMode == RasterMode::Shadow ? kShadowChunkLog2 : kChunkLog2;
  return min(kChunkMinLog2 + (units > kTarget ? 32 - __clz((int)((units - 1u) / kTarget)) : 0), kMost);
}

template <RasterMode kMode, int kOp, bool kBatch>
__global__ void __launch_bounds__(256) k_raster(PassArgs a, ShadowTarget sh) {
  __shared__ TriLds<kMode, kBatch> lds_all[256 / kWave];
  const Lists& Ls = a.lists;
  if constexpr (kMode == RasterMode::Id) {
    // prearrange and the depth pass are through with them
    if (blockIdx.x == 0 && threadIdx.x < (uint32_t)kPartWord(1)) Ls.pub[threadIdx.x] = Ls.counters[threadIdx.x];
  }
  if (Ls.counters[kOverflow]) return;
  const int lane = threadIdx.x & (kWave - 1);
  // lane p holds partition p's records, samples and inclusive chunk count
  uint32_t part_ncut = 0, part_total = 0;
  if constexpr (kMode == RasterMode::Shadow) {
    // (records << 40 | samples), up to the valid prefix
    const unsigned long long* pc = reinterpret_cast<const unsigned long long*>(Ls.counters + kPartWord(lane));
    const unsigned long long packed = min(pc[0], pc[1]);
    part_ncut = (uint32_t)(packed >> kShadowSampleBits);
    part_total = (uint32_t)(packed & kShadowSampleMask);   // at most 2^30
  } else if ((uint32_t)lane < Ls.parts) {
    const unsigned long long packed = *reinterpret_cast<const unsigned long long*>(Ls.counters + kPartWord(lane));
    part_ncut = (uint32_t)(packed >> 32);
    part_total = (uint32_t)packed;   // at most kMaxSamples
  }
  // the pass's samples in units of 2^kChunkMinLog2 (at most 2^30)
  constexpr uint32_t kUnit = 1u << kChunkMinLog2;
  const uint32_t units = wave_total(wave_incl_scan((part_total + kUnit - 1) >> kChunkMinLog2));
  if constexpr (kMode != RasterMode::Shadow) {
    // the partitions together hold at most kMaxSamples, like one list
    if (units > kMaxSamples / kUnit) {
      const unsigned long long all = ((unsigned long long)wave_total(wave_incl_scan(part_total >> 16)) << 16) +
                                     wave_total(wave_incl_scan(part_total & 0xFFFFu));
      if (all > kMaxSamples) {
        if (lane == 0) atomicOr(&Ls.counters[kOverflow], kOverflowSamples);
        return;
      }
    }
  }
  const int clog = chunk_log2<kMode>(units);
  const uint32_t part_chunks = wave_incl_scan((part_total >> clog) + ((part_total & ((1u << clog) - 1u)) ? 1u : 0u));
  const uint32_t nchunks = wave_total(part_chunks);
  const uint32_t csize = 1u << clog;
  const uint32_t ent_cap = csize / 2u, ent_chunks = kMode == RasterMode::Shadow ? 0u : Ls.ent.chunks << (kChunkLog2 - clog);
  TriLds<kMode, kBatch>& L = lds_all[threadIdx.x / kWave];
  const uint32_t wave0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)((blockIdx.x * blockDim.x + threadIdx.x) / kWave));
  const uint32_t nwaves = gridDim.x * blockDim.x / kWave;
  L.start[lane] = 0u;
  uint32_t tick = 0;
  if constexpr (kMode == RasterMode::Id) {
    if (Ls.ent.cnt) id_from_entries<kBatch>(a, Ls, wave0, nwaves, min(ent_chunks, nchunks), ent_cap);
  }
  RasterTarget T{kMode == RasterMode::Shadow ? sh.L : a.view0.v.width,
                 kMode == RasterMode::Shadow ? sh.map : a.view0.depth, a.view0.idkey, nullptr, ent_cap, 0u, Ls.rast,
                 map_layout(sh.L)};
  for (uint32_t chunk = wave0; chunk < nchunks; chunk += nwaves) {
    // the chunk's partition: the first whose inclusive chunk count passes it
    const uint32_t part = (uint32_t)__popcll(__ballot(part_chunks <= chunk));
    const uint32_t before = part ? (uint32_t)__builtin_amdgcn_readlane((int)part_chunks, (int)part - 1) : 0u;
    const uint32_t ncut = (uint32_t)__builtin_amdgcn_readlane((int)part_ncut, (int)part);
    const uint32_t total = (uint32_t)__builtin_amdgcn_readlane((int)part_total, (int)part);
    const uint32_t first = part * (Ls.cap_cut / (kMode == RasterMode::Shadow ? kListParts : Ls.parts));
    const RasterTri* rast = Ls.rast + first;
    const uint32_t s0 = (chunk - before) << clog;
    const uint32_t s1 = min(s0 + csize, total);
    // covered-sample entries of the chunk: written by the depth pass, read
    // by the id pass instead of a second sweep
    T.ent = nullptr;
    T.nent = 0;
    if constexpr (kMode != RasterMode::Shadow) {
      if (Ls.ent.cnt && chunk < ent_chunks) {
        if constexpr (kMode == RasterMode::Id) {
          // chunks whose entries the depth pass kept were done above
          if (Ls.ent.cnt[chunk] <= ent_cap) continue;
        } else {
          T.ent = Ls.ent.ent + (size_t)chunk * ent_cap;
        }
      }
    }
    // ---- the chunk's first triangle: last record with sample_begin <= s0
    // (record 0 begins at sample 0; 64-ary search, one probe per lane)
    uint32_t lo = 0, hi = ncut;
    while (hi - lo > 1) {
      const uint32_t p = lo + (uint32_t)(((unsigned long long)(hi - lo) * (uint32_t)lane) / kWave);
      const unsigned long long m = __ballot(rast[p].sample_begin <= s0);
      const int t = 63 - __clzll((long long)m);
      const uint32_t plo = __shfl(p, t, kWave);
      const uint32_t phi = __shfl(p, t < kWave - 1 ? t + 1 : t, kWave);
      lo = plo;
      hi = t < kWave - 1 ? phi : hi;
    }
    uint32_t c0 = lo;
    uint32_t s = s0;
    while (s < s1) {
      // ---- stage triangles c0 .. c0 + 63, one per lane
      const uint32_t ci = c0 + (uint32_t)lane;
      RasterTri t{};
      uint32_t begin = total, after = total;   // first sample of the lane's triangle and of the next
      uint32_t* dst = nullptr;
      unsigned long long* ids = nullptr;
      uint32_t pitch = 0, face = 0;
      if (ci < ncut) {
        t = rast[ci];
        begin = t.sample_begin;
        if constexpr (kMode == RasterMode::Shadow) face = (t.key & ~kKeyBoxForm) * sh.L * sh.L;
        if constexpr (kBatch) {
          const DevView& V = a.views[Ls.cuts[first + ci].view];
          dst = V.depth;
          ids = V.idkey;
          pitch = V.v.width;
        }
        if (ci + 1 < ncut) after = rast[ci + 1].sample_begin;
      }
      const uint32_t stage_end = min(s1, (uint32_t)__builtin_amdgcn_readlane((int)after, kWave - 1));
      const uint32_t b = max(s, begin), e = min(stage_end, after);
      raster_stage<kMode, kOp, kBatch>(L, T, t, first + ci, b < e ? b - begin : 1u, b < e ? e - begin : 0u, face, dst, pitch,
                                       ids, tick);
      s = stage_end;
      c0 += kWave;
    }
    if constexpr (kMode == RasterMode::Depth) {
      if (T.ent && lane == 0) Ls.ent.cnt[chunk] = T.nent;
    }
  }
}

int device_cu_count();

template <RasterMode kMode>
static hipError_t launch_camera_raster(const PassArgs& a, int blocks_per_cu, hipStream_t s) {
  const dim3 grid(device_cu_count() * blocks_per_cu), block(256);
  if (a.views)
    hipLaunchKernelGGL((k_raster<kMode, kOpSize, true>), grid, block, 0, s, a, ShadowTarget{nullptr, 0});
  else
    hipLaunchKernelGGL((k_raster<kMode, kOpSize, false>), grid, block, 0, s, a, ShadowTarget{nullptr, 0});
  return hipGetLastError();
}

hipError_t launch_depth(const PassArgs& a, int blocks_per_cu, hipStream_t s) {
  return launch_camera_raster<RasterMode::Depth>(a, blocks_per_cu, s);
}

// kernel2's "last writer wins" is made deterministic: among fragments inside
// the BUF_ERROR window the pixel keeps the largest (2*tri + sub) key, which
// is the fragment a sequential in-order execution writes last.
hipError_t launch_id(const PassArgs& a, int blocks_per_cu, hipStream_t s) {
  return launch_camera_raster<RasterMode::Id>(a, blocks_per_cu, s);
}

// ---------------------------------------------------------------- shadows
struct FaceTable { SinCos f[6]; };

// prearrange_realtime_shadowing (cl2.cl:4419-4636) and kernel1's shadow
// raster (cl2.cl:4638-4700) for a group of lights in one launch, each
// wavefront on its own with 64 triangles, read from HBM once for the whole
// group.  For each light: the faces a triangle's vertices fall in
// (ret_cubeface), one to three of the six, each (triangle, face) pair an item
// in the wavefront's list.  Whenever 64 items wait, of whatever lights, they
// are clipped, projected and culled, one per lane; the pieces that are left (on
// small faces half of them round to nothing) wait in registers until 64 of them
// are together, are set up, and become records, key = slot * 6 + face with slot
// the light's cube map in the group's maps, for one raster launch over the
// whole group; pieces of at most local_max samples, and any that no longer fit
// the list, are rasterised at once by the wavefront.
// Half of a light's items face away, so a block that gathered the items of one
// light at a time left half of its wavefronts waiting at each light's barrier,
// and every second piece of a draw was an empty one: 500 M -> 407 M vector
// instructions, 1.26 -> 0.85 ms (16 lights, 4 M triangles), where issuing the
// instructions takes 0.73 ms.
constexpr int kMaxShadowGroup = 16;
struct ShadowGroup {
  float pos[kMaxShadowGroup][3];
  uint32_t slot[kMaxShadowGroup];
  uint32_t n;
};

// Shadow-pass allocation for the lanes with `take` set, per wavefront: one
// atomicAdd on the packed counter of the block's partition (records
// [part * cap, part * cap + cap) of the list, cap = cap_cut / kListParts,
// and a sample space of its own).  An allocation that passes the
// partition's capacity or kShadowMaxSamples is not written: the wavefront
// rasterises those pieces itself and lowers the partition's valid-prefix
// word to its start, and every later allocation in the partition fails too
// (the counter only grows), so the raster launch reads each partition up to
// min(counter, valid prefix).
__device__ __forceinline__ bool wave_alloc_fit(const Lists& L, uint32_t ncut, uint32_t nsmp, uint32_t& cut0,
                                               uint32_t& smp0) {
  const int lane = threadIdx.x & (kWave - 1);
  // ncut is 0 or 1
  const unsigned long long m = __ballot(ncut != 0u);
  const uint32_t is = wave_incl_scan(nsmp);
  const uint32_t tc = (uint32_t)__popcll(m), ts = wave_total(is);
  cut0 = smp0 = 0;
  if (tc == 0) return true;
  const uint32_t part = blockIdx.x % kListParts, cap = L.cap_cut / kListParts;
  uint32_t base_lo = 0, base_hi = 0, ok = 0;
  if (lane == 0) {
    unsigned long long* p = reinterpret_cast<unsigned long long*>(L.counters + kPartWord(part));
    const unsigned long long seen = __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if ((seen >> kShadowSampleBits) < cap && (seen & kShadowSampleMask) < kShadowMaxSamples) {
      const unsigned long long old = atomicAdd(p, ((unsigned long long)tc << kShadowSampleBits) + ts);
      ok = (old >> kShadowSampleBits) + tc <= cap && (old & kShadowSampleMask) + ts <= kShadowMaxSamples;
      if (!ok) atomicMin(p + 1, old);   // the valid-prefix word, same line
      base_lo = (uint32_t)(old & kShadowSampleMask);   // below 2^30 when ok
      base_hi = (uint32_t)(old >> kShadowSampleBits);
    }
  }
  ok = (uint32_t)__builtin_amdgcn_readfirstlane((int)ok);
  cut0 = part * cap + (uint32_t)__builtin_amdgcn_readfirstlane((int)base_hi) + lanes_below(m);
  smp0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)base_lo) + is - nsmp;
  return ok != 0;
}

using ShadowStage = TriLds<RasterMode::Shadow, false>;
struct PieceSwap {
  float4 a[kWave], b[kWave];   // p[0], p[1].x; p[1].yz, p[2].xy
  float2 c[kWave];             // p[2].z, the map's key
  __device__ __forceinline__ void put(uint32_t s, const f3 p[3], uint32_t key) {
    a[s] = make_float4(p[0].x, p[0].y, p[0].z, p[1].x);
    b[s] = make_float4(p[1].y, p[1].z, p[2].x, p[2].y);
    c[s] = make_float2(p[2].z, __uint_as_float(key));
  }
  __device__ __forceinline__ void get(uint32_t s, f3 p[3], uint32_t& key) const {
    const float4 u = a[s], v = b[s];
    const float2 w = c[s];
    p[0] = mk3(u.x, u.y, u.z);
    p[1] = mk3(u.w, v.x, v.y);
    p[2] = mk3(v.z, v.w, w.x);
    key = __float_as_uint(w.y);
  }
};
static_assert(sizeof(PieceSwap) <= offsetof(ShadowStage, start), "the stage's start[] keeps its marks");

struct ShadowLds {
  float lpos[kMaxShadowGroup][3];
  uint32_t key[kMaxShadowGroup];   // of the light's first face
  SinCos face[6];
  struct Wave {
    float wpos[kWave][9];
    // light << 16 | lane << 4 | two_sided << 3 | face: fewer than 64 left over
    // and up to three of each lane
    uint32_t items[4 * kWave];
    // pieces on their way between lanes share the stage's place
    union {
      ShadowStage stage;
      PieceSwap swap;
    };
  } wave[kShadowPreThreads / kWave];
};

__global__ void __launch_bounds__(kShadowPreThreads) k_prearrange_shadow(const TriPos* __restrict__ world, uint32_t ntri,
                                                           const ObjDesc* __restrict__ objs, uint32_t nobj,
                                                           ShadowGroup group, ShadowTarget target,
                                                           int only_static, uint32_t local_max, FaceTable ft,
                                                           Lists lists) {
  __shared__ ShadowLds S;
  const uint32_t t = threadIdx.x;
  const int lane = t & (kWave - 1);
  ShadowLds::Wave& M = S.wave[t / kWave];
  ShadowStage& W = M.stage;
  PieceSwap& Q = M.swap;
  const uint32_t id = blockIdx.x * blockDim.x + t;
  if (t < 3u * kMaxShadowGroup) (&S.lpos[0][0])[t] = (&group.pos[0][0])[t];
  if (t < (uint32_t)kMaxShadowGroup) S.key[t] = group.slot[t] * 6u;
  if (t < 6u) S.face[t] = ft.f[t];
  __syncthreads();   // the only one: the wavefronts are independent from here
  const uint32_t L = target.L;
  const float ew = (float)L, eh = (float)L, efov = (float)L / 2.0f;
  // ---- the triangle, once for every light of the group
  bool live = false;
  uint32_t two_sided = 0;
  f3 wp = mk3(0.f, 0.f, 0.f);
  f3 wv[3] = {wp, wp, wp};
  if (id < ntri) {
    const TriPos T = world[id];
    if (T.oid < nobj) {
      const ObjDesc G = objs[T.oid];
      const bool is_static = (G.flags & OCR_FEATURE_IS_STATIC) > 0;
      live = only_static ? is_static : !is_static;
      wp = mk3(G.wp[0], G.wp[1], G.wp[2]);
      if (live) {
#pragma unroll
        for (int k = 0; k < 3; k++) {
          wv[k] = mk3(T.p[3 * k], T.p[3 * k + 1], T.p[3 * k + 2]);
          M.wpos[lane][3 * k] = wv[k].x;
          M.wpos[lane][3 * k + 1] = wv[k].y;
          M.wpos[lane][3 * k + 2] = wv[k].z;
        }
        two_sided = (G.flags & OCR_FEATURE_TWO_SIDED) > 0 ? 1u : 0u;
      }
    }
  }
  // the triangle's normal and longest edge component, for every light
  const f3 a = wv[1] - wv[0], b = wv[2] - wv[0], c = b - a;
  const f3 nrm = cross(a, b);
  const float edge = max3f(max3f(fabsf(a.x), fabsf(a.y), fabsf(a.z)), max3f(fabsf(b.x), fabsf(b.y), fabsf(b.z)),
                           max3f(fabsf(c.x), fabsf(c.y), fabsf(c.z)));
  W.start[lane] = 0u;
  uint32_t tick = 0;
  RasterTarget T{L, target.map, nullptr, nullptr, 0u, 0u, nullptr, map_layout(L)};
  // projected pieces that wait for a full wavefront: one in each lane below nq
  f3 qp[3] = {wp, wp, wp};
  uint32_t qkey = 0, nq = 0;
  auto draw = [&](bool have) {
    Piece P;
    P.nf = P.seen = P.ns = 0u;
    if (have) {
#pragma unroll
      for (int k = 0; k < 3; k++) P.p[k] = qp[k];
      setup_piece(ew, eh, kOpSizeLight, P);
    }
    // pieces above local_max samples to the list, in allocations of at
    // most kShadowWaveSamples samples (each takes the lanes whose running
    // sum fits, at least the first waiting lane); pieces of the list's
    // failed allocations and the small ones rasterised here
    const uint32_t mine = P.ns > local_max ? P.ns : 0u;   // < 2^24
    bool waiting = mine > 0, listed = false;
    while (__ballot(waiting)) {
      const uint32_t upto = wave_incl_scan(waiting ? mine : 0u);
      const bool take = waiting && upto <= kShadowWaveSamples;
      uint32_t c, smp;
      const bool ok = wave_alloc_fit(lists, take ? 1u : 0u, take ? mine : 0u, c, smp);
      if (take) {
        waiting = false;
        listed = ok;
        if (ok) {
          P.rt.key = qkey | (P.rt.key & kKeyBoxForm);
          P.rt.sample_begin = smp;
          lists.rast[c] = P.rt;
        }
      }
    }
    // The rest, straight into the maps: a map keeps the minimum depth of
    // its samples, so the order in which they arrive does not matter.
    const uint32_t n = listed ? 0u : P.ns;
    if (__any(n != 0u))
      raster_stage<RasterMode::Shadow, kOpSizeLight, false>(W, T, P.rt, (uint32_t)lane, n ? 0u : 1u, n, qkey * L * L,
                                                            nullptr, 0u, nullptr, tick);
  };
  uint32_t nit = 0;
  for (uint32_t li = 0; li <= group.n; li++) {   // and a last turn for what is left
    if (li < group.n) {
      // ---- the faces that the lane's triangle may fall on
      const f3 lpos = mk3(group.pos[li][0], group.pos[li][1], group.pos[li][2]);
      uint32_t touched = 0;
      const f3 to_obj = wp - lpos;
      if (live && !(dot(to_obj, to_obj) > kDepthFarSq)) {
        float near = 3.0e38f, far = 0.f;
        f3 rel0 = mk3(0.f, 0.f, 0.f);
#pragma unroll
        for (int k = 0; k < 3; k++) {
          const f3 rel = wv[k] - lpos;
          if (k == 0) rel0 = rel;
          const float ax = fabsf(rel.x), ay = fabsf(rel.y), az = fabsf(rel.z);
          const float z = max3f(ax, ay, az);
          near = fminf(near, z);
          far = fmaxf(far, z);
          // the bit of ret_cubeface's answer (cl2.cl:1745-1790), by selects
          const bool cx = (ax >= ay) & (ax >= az), cy = (ay > ax) & (ay >= az);
          const bool cz = (az > ax) & (az > ay) & (rel.z < 0.f);
          const uint32_t bz = cz ? 1u << 2 : 1u, by = rel.y < 0.f ? 1u << 1 : 1u << 3, bx = rel.x < 0.f ? 1u << 4 : 1u << 5;
          touched |= cx ? bx : (cy ? by : bz);
        }
        // certainly facing away: no piece of it would pass the culling
        if (!two_sided && (touched & (touched - 1u)) == 0u && faces_away(nrm, edge, rel0, near, far)) touched = 0u;
      }
      const uint32_t mine = (uint32_t)__popc(touched);
      const uint32_t incl = wave_incl_scan(mine);
      uint32_t slot = nit + incl - mine;
      nit += wave_total(incl);
      // one to three faces, nearly always one
      while (touched) {
        const uint32_t f = (uint32_t)__ffs((int)touched) - 1u;
        touched &= touched - 1u;
        M.items[slot++] = li << 16 | (uint32_t)lane << 4 | two_sided << 3 | f;
      }
      wave_lds_sync();
    }
    // ---- 64 items at a time, the last ones first
    while (nit >= (uint32_t)kWave || (li == group.n && nit)) {
      const uint32_t cnt = min(nit, (uint32_t)kWave);
      nit -= cnt;
      f3 tris[2][3];
      int num = 0;
      uint32_t key = 0;
      bool both = false;
      if ((uint32_t)lane < cnt) {
        const uint32_t it = M.items[nit + (uint32_t)lane];
        const uint32_t lt = (it >> 4) & 63u, face = it & 7u, l = it >> 16;
        both = ((it >> 3) & 1u) != 0u;
        f3 w[3];
#pragma unroll
        for (int k = 0; k < 3; k++) w[k] = mk3(M.wpos[lt][3 * k], M.wpos[lt][3 * k + 1], M.wpos[lt][3 * k + 2]);
        key = S.key[l] + face;
        num = face_clip(w, mk3(S.lpos[l][0], S.lpos[l][1], S.lpos[l][2]), S.face[face], tris);
      }
      // the second piece exists only where the near plane cuts
#pragma unroll 1
      for (int i = 0; i < 2; i++) {
        if (!__any(num > i)) break;
        f3 p[3] = {wp, wp, wp};
        bool keep = num > i;
        if (keep) {
#pragma unroll
          for (int k = 0; k < 3; k++) p[k] = depth_project_clipped(i == 0 ? tris[0][k] : tris[1][k], ew, eh, efov);
          keep = piece_kept(p, ew, eh, both) && !piece_empty(p);
        }
        // the kept pieces, compacted: those that the waiting ones leave room
        // for join them, and a full wavefront is drawn before the rest do
        const unsigned long long kept = __ballot(keep);
        const uint32_t n = (uint32_t)__popcll(kept);
        if (keep) Q.put(lanes_below(kept), p, key);
        wave_lds_sync();
        const uint32_t from = (uint32_t)lane - nq;
        if (from < n) Q.get(from, qp, qkey);
        nq += n;
        if (nq >= (uint32_t)kWave) {
          f3 rp[3] = {wp, wp, wp};
          uint32_t rkey = 0;
          nq -= kWave;
          const bool rest = (uint32_t)lane < nq;
          if (rest) Q.get(n - nq + (uint32_t)lane, rp, rkey);
          wave_lds_sync();
          draw(true);
          if (rest) {
#pragma unroll
            for (int k = 0; k < 3; k++) qp[k] = rp[k];
            qkey = rkey;
          }
        }
        wave_lds_sync();
      }
      wave_lds_sync();   // items[] is rewritten
    }
  }
  if (nq) draw((uint32_t)lane < nq);
}

// A shadow pass's counters: the render words and every partition's packed
// counter (0) and valid prefix (all ones).
__global__ void __launch_bounds__(256) k_zero_shadow_counters(uint32_t* c) {
  for (uint32_t i = threadIdx.x; i < (uint32_t)kListCounterWords; i += blockDim.x) {
    const uint32_t w = i < (uint32_t)kCounterWords ? 0u : (i - kCounterWords) % kPartLineWords;
    c[i] = i >= (uint32_t)kCounterWords && (w == 2u || w == 3u) ? 0xFFFFFFFFu : 0u;
  }
}

// Tuning of the shadow launches, read at every pass: pieces of at most
// OCR_SHADOW_LOCAL_SAMPLES samples (default 16) are rasterised by the
// prearrange launch itself, larger ones go to the list for the chip-wide
// raster launch; OCR_SHADOW_LIST_RECORDS lowers the list's capacity (the
// pieces that do not fit are rasterised by the prearrange launch too).
// Neither changes the maps, only where their samples are rasterised.
static uint32_t env_u32(const char* name, uint32_t dflt) {
  const char* e = getenv(name);
  if (!e || !*e) return dflt;
  char* end = nullptr;
  const unsigned long v = strtoul(e, &end, 10);
  return end && *end == 0 && v <= 0xFFFFFFFFul ? (uint32_t)v : dflt;
}
constexpr uint32_t kShadowLocalSamples = 16;

hipError_t launch_shadow_group(Scene* sc, const float (*lpos)[3], const uint32_t* slots, uint32_t n,
                               int only_static, uint32_t* maps, hipStream_t s) {
  if (n == 0 || n > (uint32_t)kMaxShadowGroup) return hipErrorInvalidValue;
  FaceTable ft;
  for (int i = 0; i < 6; i++) ft.f[i] = sc->ctx->face_sc[i];
  ShadowGroup g;
  memset(&g, 0, sizeof(g));
  for (uint32_t i = 0; i < n; i++) {
    for (int k = 0; k < 3; k++) g.pos[i][k] = lpos[i][k];
    g.slot[i] = slots[i] - slots[0];
  }
  g.n = n;
  // raster setups only: shadow records have no CutTri
  Lists lists{nullptr, sc->sh_rast, sc->sh_counters, sc->sh_counters,
              std::min(sc->sh_cap_cut, env_u32("OCR_SHADOW_LIST_RECORDS", sc->sh_cap_cut)), kListParts};
  // texels of the group's maps (consecutive slots) are counted from its first
  const ShadowTarget target{maps + (size_t)slots[0] * 6 * sc->lbuf_dim * sc->lbuf_dim, sc->lbuf_dim};
  hipLaunchKernelGGL(k_zero_shadow_counters, dim3(1), dim3(256), 0, s, sc->sh_counters);
  if (sc->ntri)
    hipLaunchKernelGGL(k_prearrange_shadow, dim3((sc->ntri + kShadowPreThreads - 1) / kShadowPreThreads),
                       dim3(kShadowPreThreads), 0, s, sc->world, sc->ntri, sc->objs, sc->nobj, g, target,
                       only_static, env_u32("OCR_SHADOW_LOCAL_SAMPLES", kShadowLocalSamples), ft, lists);
  PassArgs a;
  memset(&a, 0, sizeof(a));
  a.lists = lists;
  hipLaunchKernelGGL((k_raster<RasterMode::Shadow, kOpSizeLight, false>), dim3(device_cu_count() * 8), dim3(256), 0, s,
                     a, target);
  return hipGetLastError();
}

// Strips of four map rows from blocks of 4 x 4 texels to row order, four
// texels a work item.
__global__ void __launch_bounds__(256) k_map_rows(const uint4* __restrict__ map, uint32_t L, uint32_t n,
                                                  uint4* __restrict__ rows) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;   // below 2^22
  if (i >= n) return;
  const uint32_t strip = i / L, q = i % L, across = L / 4u;
  rows[i] = map[strip * L + (q % across) * 4u + q / across];
}

hipError_t launch_map_rows(const uint32_t* map, uint32_t L, uint32_t strips, uint32_t* rows, hipStream_t s) {
  const uint32_t n = strips * L;
  if (n)
    hipLaunchKernelGGL(k_map_rows, dim3((n + 255) / 256), dim3(256), 0, s, reinterpret_cast<const uint4*>(map), L, n,
                       reinterpret_cast<uint4*>(rows));
  return hipGetLastError();
}

}  // namespace ocr
