// pair_kernel.hpp -- two time steps in one pass over the populations (gfx950).
//
// A step of a large domain is bound by the traffic of 19 population planes in
// and 19 out: on MI355X that pattern alone, without any arithmetic, runs at
// 5.1-5.5 TB/s, which is what step_kernel reaches, while its FP64 BGK
// arithmetic takes a fifth of that time.  So this kernel does two steps per
// read and write of the lattice.
//
// A workgroup owns TX x TY columns and walks a segment of planes upwards.  Per
// plane s every thread gathers its node from HBM and collides it (step one), on
// the tile and on a ring of one node around it; the post-collision populations
// then meet in LDS, and the tile's threads pull, collide and store plane s - 1
// (step two).  Populations are pulled one plane up, level or one plane down:
//   c_z = -1 of plane s       written before the first barrier,
//   c_z =  0 of plane s - 1   written in the iteration before,
//   c_z = +1 of plane s - 2   kept in registers for an iteration, then written,
// so each of the 16 directions that leave the column needs one buffer only, and
// the three that stay in it (rest, +z, -z) need none.  Below FP64 there is room
// for more: two sets of buffers, used in turn, which leaves one barrier per plane, and
// registers for the next plane's loads, issued before step two.  (In FP64 those
// loads spill: 512^3 4.4 ms per step without them, 8.9 ms with.)
//
// A node whose upstream neighbour is outside a non-periodic face pushes its own
// opposite population into the slot it will pull from; that slot belongs to a
// node outside the domain, which nobody else writes.  Populations travel as they
// are stored (16-bit storage: rounded with the first step's random words), and
// the arithmetic per node and step is the single step's own code, so the result
// is the same bit for bit.
//
// Taken by domains without walls, boundary programs and start_iteration boxes, MRT
// only in FP64 and FP32.  Single / two steps per pass, ms per step: 512^3 BGK FP64
// 7.3 / 4.4, 512 x 256 x 256 FP32 0.94 / 0.58 (5.1 TB/s of actual traffic: the
// memory's limit for this pattern), 512^3 FP16 2.12 / 1.91, BF16 2.14 / 1.79.  A
// plane of a 16-bit tile takes 5.6 us, 2.8 of them vector issue: half the bytes
// leave the chain load, collide, LDS, collide in view, MRT (FP16 2.08 / 2.10)
// lengthens it, and rows that end inside a cache line (500 x 400 x 200 586 / 664
// us) meet stores of partial lines.
#pragma once

#include "pair_grid.hpp"
#include "step_kernel.hpp"

namespace hlbm {

// FP64: from this size of the two lattices together the new populations are
// stored with the non-temporal hint, so that the planes neighbouring tiles still
// share stay in L2.  Up to it the Infinity Cache (256 MiB) holds much of what was
// stored until the next pass reads it.  Without / with the hint, us per step, BGK:
// 80^3 29.9 / 30.8   96^3 (257 MiB) 38.0 / 40.6   104^3 (326) 52.8 / 51.6
// 112^3 66 / 59   200^3 374 / 325   512^3 4500-4890 / 4290-4700.
// (FP32 without the hint: no difference at any size.)
constexpr int64_t PAIR_STREAM_BYTES = 320ll << 20;

// What Rounder reads of a step's parameters.
struct PairRounding {
  int32_t sr;
  uint32_t seed;
};

// LDS slot of a direction that leaves its column, in the order c_z = 0, +1, -1.
HLBM_HD constexpr int pair_slot(int i) {
  constexpr int s[Q] = {-1, 0, 1, 2, 3, -1, -1, 4, 5, 6, 7, 8, 12, 13, 9, 10, 14, 15, 11};
  return s[i];
}

// Barrier for the LDS buffers alone: loads and stores of populations stay in flight.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

template <class S, int COLL, bool STREAM>
__global__ void __launch_bounds__((PAIR_TY + 3) * 64) pair_kernel(const StepParams p, const PairGrid g) {
  using O = StoreOps<S>;
  using C = typename O::C;
  constexpr int TY = PAIR_TY, R = TY + 2, W = PAIR_TX + 2;
  constexpr bool AHEAD = sizeof(S) <= 4;  // the next plane's loads before step two
  constexpr int BUFS = sizeof(S) <= 4 ? 2 : 1;
  using Raw = std::conditional_t<sizeof(S) == 2, uint16_t, C>;
  constexpr bool RAW = raw_store<S, COLL, MODE_FUSED>();
  __shared__ S buf[BUFS][16][R][W];

  // Tiles next to each other in x run on the same XCD at the same time: a ring's
  // column is 15 cache lines per direction, of which the neighbour reads all
  // (512^3 FP64: 198 M reads of 128 bytes leave L2 per pass, 250 M with tiles in y
  // order, 159 M populations; 4.4 ms per step, 5.1 in y order.  FP32 0.58, 0.62)
  const uint32_t nt = (uint32_t)(g.tx * g.ty * g.segs);
  uint32_t t = blockIdx.x;
  {
    const uint32_t per = nt / 8u;
    if (t < per * 8u) t = (t % 8u) * per + t / 8u;
  }
  const int tx = (int)(t % (uint32_t)g.tx);
  const uint32_t t2 = t / (uint32_t)g.tx;
  const int ty = (int)(t2 % (uint32_t)g.ty), seg = (int)(t2 / (uint32_t)g.ty);

  const int nx = p.nx, ny = p.ny, nz = p.nz;
  const bool px = p.per[0] != 0, py = p.per[1] != 0, pz = p.per[2] != 0;
  const int wx = min(PAIR_TX, nx - tx * PAIR_TX), hy = min(TY, ny - ty * TY);  // this tile's columns and rows
  const int zs = seg * g.planes, ze = min(zs + g.planes, nz);

  // rows 0 .. TY + 1 are a wave each (0 and hy + 1 the ring's); the last wave
  // holds the ring's columns left and right of every row
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = (int)(threadIdx.x & 63u);
  const bool side = wave == R;
  const int r = side ? lane >> 1 : wave;
  const int c = side ? ((lane & 1) ? wx + 1 : 0) : lane + 1;
  int x = tx * PAIR_TX + c - 1, y = ty * TY + r - 1;
  bool act = r <= hy + 1 && c <= wx + 1 && (side || c <= wx);
  if (x < 0 || x >= nx) {
    act = act && px;
    x = x < 0 ? nx - 1 : 0;
  }
  if (y < 0 || y >= ny) {
    act = act && py;
    y = y < 0 ? ny - 1 : 0;
  }
  const bool mine = !side && r >= 1 && r <= hy && c <= wx;  // the tile's own columns

  // the node's neighbours outside a non-periodic face
  const bool fxm = !px && x == 0, fxp = !px && x == nx - 1, fym = !py && y == 0, fyp = !py && y == ny - 1;
  const bool wave_face = __any(act && (fxm || fxp || fym || fyp));
  // direction i's upstream node is outside (zout: outside a z face)
  auto outside = [&](auto ic, bool zout) {
    constexpr int i = decltype(ic)::value;
    bool o = zout;
    if constexpr (CX(i) != 0) o = o || (CX(i) == 1 ? fxm : fxp);
    if constexpr (CY(i) != 0) o = o || (CY(i) == 1 ? fym : fyp);
    return o;
  };

  // byte offsets inside a plane: of the rows and columns populations come from,
  // added where they are used (nine sums kept across the loop would spill)
  const uint32_t nxy = (uint32_t)nx * (uint32_t)ny;
  const uint32_t unit = (uint32_t)sizeof(S), row = (uint32_t)nx * unit;
  const uint32_t xo[3] = {(uint32_t)(x > 0 ? x - 1 : (px ? nx - 1 : 0)) * unit, (uint32_t)x * unit,
                          (uint32_t)(x < nx - 1 ? x + 1 : (px ? 0 : x)) * unit};
  const uint32_t yo[3] = {(uint32_t)(y > 0 ? y - 1 : (py ? ny - 1 : 0)) * row, (uint32_t)y * row,
                          (uint32_t)(y < ny - 1 ? y + 1 : (py ? 0 : y)) * row};
  auto off = [&](int b, int a) { return yo[b] + lane_offset(xo[a]); };

  const S* __restrict__ fin = (const S*)p.fin;
  auto plane_valid = [&](int s) { return pz || (s >= 0 && s < nz); };
  auto wrapped = [&](int s) { return s < 0 ? s + nz : (s >= nz ? s - nz : s); };

  // step one's populations arriving at the node in plane s, as stored
  auto gather = [&](int s, S* f) {
    const int z = wrapped(s);
    const bool zlo = !pz && z == 0, zhi = !pz && z == nz - 1;
    if (wave_face || zlo || zhi) {
      // as gather_select: a lane whose upstream node is outside takes its own
      // opposite population, both addressed from the first plane of the pair
      const uint32_t stb = (uint32_t)(p.stride * sizeof(S)), pb = nxy * unit;
      const uint32_t zo[3] = {(uint32_t)wrapped(z - 1) * pb, (uint32_t)z * pb, (uint32_t)wrapped(z + 1) * pb};
      f[0] = *at_bytes(scalar_ptr(fin), lane_offset(off(1, 1) + zo[1]));
      const S* b = fin;
      static_for<1, Q>([&](auto ic) {
        constexpr int i = decltype(ic)::value;
        constexpr int lo = (i & 1) ? i : i - 1;
        if constexpr (i & 1) b = scalar_ptr(b + (size_t)(i == 1 ? 1 : 2) * p.stride);
        const uint32_t pull = off(1 - CY(i), 1 - CX(i)) + ((uint32_t)(i - lo) * stb + zo[1 - CZ(i)]);
        const uint32_t own = off(1, 1) + ((uint32_t)(OPP(i) - lo) * stb + zo[1]);
        f[i] = *at_bytes(b, outside(ic, CZ(i) == 1 ? zlo : (CZ(i) == -1 ? zhi : false)) ? own : pull);
      });
    } else {
      const size_t zo[3] = {(size_t)wrapped(z - 1) * nxy, (size_t)z * nxy, (size_t)wrapped(z + 1) * nxy};
      const S* b = fin;
      static_for([&](auto ic) {
        constexpr int i = decltype(ic)::value;
        b = scalar_ptr(i ? b + p.stride : b);
        const S* q = scalar_ptr(b + zo[1 - CZ(i)]);
        f[i] = *at_bytes(q, lane_offset(off(1 - CY(i), 1 - CX(i))));
      });
    }
  };
  // the moving-wall terms of the populations that bounced off a z face
  auto add_wall = [&](int z, C* f) {
    if (pz || !p.cav_gather) return;
    static_for<0, 2>([&](auto sc) {
      constexpr int sd = decltype(sc)::value;
      if (p.cav_on[sd] && z == (sd ? nz - 1 : 0))
        static_for<1, Q>([&](auto ic) {
          constexpr int i = decltype(ic)::value;
          if constexpr (CZ(i) == (sd ? -1 : 1)) f[i] += cav_coef<C>(p, sd, cavity_slot(i));
        });
    });
  };
  // populations as a step stores them (16-bit: rounded with that step's words)
  auto stored = [&](uint32_t seed, int z, const C* f, S* h) {
    const PairRounding rp{p.sr, seed};
    const Rounder<S> rw(rp, (uint32_t)z * nxy + (uint32_t)y * (uint32_t)nx + (uint32_t)x);
    static_for([&](auto ic) {
      constexpr int i = decltype(ic)::value;
      if constexpr (RAW)
        h[i] = O::pack_sr_scaled(f[i], rw.word(i));
      else
        h[i] = O::pack_sr(f[i], rw.word(i));
    });
  };

  S gn[Q];  // arriving in plane s
  // kept, as stored: c_z = +1 diagonals and rest of plane s - 1; +z of planes s - 1 and s - 2
  S up[4] = {}, h0 = {}, h5 = {}, u5 = {};
  if (AHEAD && act && plane_valid(zs - 1)) gather(zs - 1, gn);
  for (int s = zs - 1; s <= ze; s++) {
    const bool valid = plane_valid(s), before = plane_valid(s - 1);
    auto& lds = buf[BUFS == 2 ? s & 1 : 0];
    auto& next = buf[BUFS == 2 ? ~s & 1 : 0];  // read by the next iteration
    S h[Q];  // step one's populations of plane s
    if (act && valid) {
      if constexpr (!AHEAD) gather(s, gn);
      C f[Q];
#pragma unroll
      for (int i = 0; i < Q; i++) f[i] = O::unpack(gn[i]);
      add_wall(wrapped(s), f);
      collide_node<S, COLL, MODE_FUSED, RAW, false>(p, 0u, false, f);
      stored(p.seed, wrapped(s), f, h);
      // these reach step two in registers, rounded as the others are by LDS
      if constexpr (!O::narrow16) {
        h[0] = rounded(h[0]);
        h[5] = rounded(h[5]);
        h[6] = rounded(h[6]);
      }
    }
    if (AHEAD && s < ze && act && plane_valid(s + 1)) gather(s + 1, gn);

    // c_z = -1 of plane s; on a face, of plane s - 1's own bounce-back
    if (act && valid) {
      static_for<1, Q>([&](auto ic) {
        constexpr int i = decltype(ic)::value;
        if constexpr (CZ(i) == -1 && pair_slot(i) >= 0) lds[pair_slot(i)][r][c] = h[i];
      });
    }
    const bool top = !pz && s == nz;  // plane s - 1 lies on the high z face
    if (mine && before && (wave_face || top)) {
      static_for<1, Q>([&](auto ic) {
        constexpr int i = decltype(ic)::value;
        if constexpr (CZ(i) == -1 && pair_slot(i) >= 0) {
          if (outside(ic, top)) lds[pair_slot(i)][r - CY(i)][c - CX(i)] = up[pair_slot(OPP(i)) - 8];
        }
      });
    }
    lds_barrier();

    // step two: plane s - 1
    if (s > zs && mine) {
      const int z = s - 1;
      C f[Q];
      f[0] = O::unpack(h0);
      f[5] = O::unpack(u5);
      f[6] = O::unpack(top ? h5 : h[6]);
      static_for<1, Q>([&](auto ic) {
        constexpr int i = decltype(ic)::value;
        if constexpr (pair_slot(i) >= 0) f[i] = O::unpack(lds[pair_slot(i)][r - CY(i)][c - CX(i)]);
      });
      add_wall(z, f);
      collide_node<S, COLL, MODE_FUSED, RAW>(p, (uint32_t)z * nxy + off(1, 1) / unit, false, f);
      S o[Q];
      stored(g.seed2, z, f, o);
      S* b = (S*)p.fout + (size_t)z * nxy;
      const uint32_t bo = lane_offset(off(1, 1));
      static_for([&](auto ic) {
        constexpr int i = decltype(ic)::value;
        b = scalar_ptr(i ? b + p.stride : b);
        if constexpr (STREAM)
          __builtin_nontemporal_store(__builtin_bit_cast(Raw, o[i]), (Raw*)at_bytes(b, bo));
        else
          *at_bytes(b, bo) = o[i];
      });
    }
    if constexpr (BUFS == 1) lds_barrier();

    // c_z = 0 of plane s, c_z = +1 of plane s - 1; on a face, of plane s's own bounce-back
    const bool bottom = !pz && s == 0;
    if (act) {
      static_for<1, Q>([&](auto ic) {
        constexpr int i = decltype(ic)::value;
        if constexpr (pair_slot(i) >= 0) {
          if (CZ(i) == 0 && valid) next[pair_slot(i)][r][c] = h[i];
          if (CZ(i) == 1 && before) next[pair_slot(i)][r][c] = up[pair_slot(i) - 8];
        }
      });
    }
    if (mine && valid && (wave_face || bottom)) {
      static_for<1, Q>([&](auto ic) {
        constexpr int i = decltype(ic)::value;
        if constexpr (pair_slot(i) >= 0 && CZ(i) >= 0) {
          if (outside(ic, CZ(i) == 1 && bottom)) next[pair_slot(i)][r - CY(i)][c - CX(i)] = h[OPP(i)];
        }
      });
    }
    u5 = bottom ? h[6] : h5;
    h5 = h[5];
    h0 = h[0];
    static_for<1, Q>([&](auto ic) {
      constexpr int i = decltype(ic)::value;
      if constexpr (CZ(i) == 1 && pair_slot(i) >= 0) up[pair_slot(i) - 8] = h[i];
    });
  }
}

}  // namespace hlbm
