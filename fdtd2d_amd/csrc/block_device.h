// block_device.h - the block form of the step kernels: a work-group keeps a
// whole tile of the grid in registers for all steps of a launch. HIP-only.
//
// The streaming form (step_device.h) walks a band row by row, all levels of a
// launch in one dependency chain: 40 and more row iterations of 2 us each
// whatever the grid, so small and middle grids take as long as a 2048^2 one.
// Here a tile of 64 columns (one per lane) and W*R rows lives in the registers
// of W waves, R rows each, and a step updates all of it at once: R independent
// cells per lane, nothing reloaded between steps. Rows meet at the waves'
// edges through LDS:
//  * after each step a wave publishes Ez of its first and last row (two
//    buffers in turn, one barrier per step);
//  * it keeps a copy of the Hx row above its first one and steps it itself
//    (four operations per column) instead of waiting for its neighbour's Hx.
// Columns at the tile's left and right edge, and rows at its top and bottom,
// turn stale by one per step and are not stored: as many columns and rows as
// the launch has steps, on each side that is not the grid's own edge.
// The arithmetic per cell, its order and the index ranges are those of the
// streaming form (step_device.h), so both give the same bits.
//
// A wave runs the code its own rows need (BlockTile): plain interior, x
// strips and column ranges (kX), y strips and row ranges (kY), both, or those
// with events (kE). A work-group runs most of its code once per launch, so
// what small grids wait for, next to the steps, is instruction fetch (about
// 0.65 us per KB of straight-line code: one form with everything, its row
// constants spilled from the scalar registers, took 11 us before its first
// step, this one 5); hence compact code before clever code here.
#ifndef FDTD2D_BLOCK_DEVICE_H
#define FDTD2D_BLOCK_DEVICE_H

#include "step_device.h"

#pragma clang fp contract(off)

namespace fdtd2d {
namespace {

typedef const rec_v4i __attribute__((address_space(1))) *grec_ptr;

__device__ __forceinline__ float lane_value(float v, int lane) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

// The step loop's barrier. The wait for the wave's own LDS writes is spelled
// out: the compiler (ROCm 7.2) dropped the one that the barrier's release
// fence stands for from loops whose header holds the barrier, and a wave then
// read a neighbour's row before it had arrived (a pool of eight small table
// shots: one run of 75 launches in ten had a wrong row).
__device__ __forceinline__ void step_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __syncthreads();
}

// One wave's part of a tile. JZ as in the streaming form (0: no plasma and no
// Jz in the wave's rows, 2: all of it plasma); with K != 0, where JZ is 1,
// `jz_on` says whether there is any (uniform). Every readlane below is reached
// by all lanes: a value copied or reloaded while a lane is masked off is not
// there for a readlane of that lane.
template <int R, int W, int K, int MED, int JZ>
__device__ __forceinline__ void block_wave(const StepArgs &a, const float4 *lut_s, float *sh, int src, int n0, int T,
                                           const BlockTile &t, int wave, bool jz_on) {
  constexpr bool KX = (K & kX) != 0, KY = (K & kY) != 0, KE = (K & kE) != 0;
  const int lane = threadIdx.x & 63;
  // Everything the step loop reads is copied out of `a` first: the barriers
  // would make it read the arguments again at every step.
  const int nx = a.nx, ny = a.ny, pitch = a.pitch;
  const float db = a.db, ca0 = a.ca0, cb0 = a.cb0, cj = a.cj, decay = a.jz_decay;
  const float uden_hx = a.uden_hx, uden_ex = a.uden_ex, uden_hy = a.uden_hy, uden_ey = a.uden_ey;
  const double jz_dt = a.jz_dt, rdx = a.rdx, rdy = a.rdy;
  const int col = t.cs + lane;
  const int rb = t.rs + wave * R;
  const bool own = col >= t.own0 && col < t.own1;
  if constexpr (K == 0) jz_on = JZ != 0;
  // ---- the state of step n0. Loads are unconditional, so that they all go
  // out together: columns past the row and rows past the grid read the
  // nearest one inside (no cell that is updated depends on them).
  const unsigned cl = KX ? min(col, pitch - 1) : col;
  auto offset = [&](int row) {
    return (static_cast<unsigned>(KY ? max(0, min(row, ny - 1)) : row) * static_cast<unsigned>(pitch) + cl) * 4u;
  };
  auto load = [](const void *base, unsigned off) { return *(const gfloat *)((const gchar *)base + off); };
  float ez[R], hx[R], hy[R], jz[R], gh;
  float ca[MED == kTable ? R : 1], cb[MED == kTable ? R : 1], ne[R];
  unsigned pec = 0;  // bit r: a PEC cell
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const unsigned off = offset(rb + r);
    ez[r] = load(a.ez[src], off);
    hx[r] = load(a.hx[src], off);
    hy[r] = load(a.hy[src], off);
    if constexpr (JZ != 0 || MED == kTable)
      ne[r] = load(MED == kTable ? static_cast<const void *>(a.med_id) : a.med_ne, off);
    if constexpr (JZ != 0) jz[r] = load(a.jz[src], off);
  }
  gh = load(a.hx[src], offset(rb - 1));
  // ---- column constants, and whether the lane's column is updated
  float den_ex = uden_ex, den_hx = uden_hx, hyx_b = 0.f, hyx_c = 0.f, ezx_b = 0.f, ezx_c = 0.f;
  float phyx[KX ? R : 1], pezx[KX ? R : 1];
  int hyx_s = -1, ezx_s = -1;
  bool upd_h = true, upd_e = true;
  if constexpr (KX) {
    den_ex = gp(a.den_ex)[cl];
    den_hx = gp(a.den_hx)[cl];
    hyx_s = gp(a.hyx_slot)[cl];
    ezx_s = gp(a.ezx_slot)[cl];
    hyx_b = gp(a.hyx_b)[cl];
    hyx_c = gp(a.hyx_c)[cl];
    ezx_b = gp(a.ezx_b)[cl];
    ezx_c = gp(a.ezx_c)[cl];
    upd_h = col <= nx - 2;
    upd_e = col >= 1 && col <= nx - 2;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int rowx = (KY ? max(0, min(rb + r, ny - 1)) : rb + r) * a.xs;
      phyx[r] = gp(a.psi_hyx[src])[rowx + max(hyx_s, 0)];
      pezx[r] = gp(a.psi_ezx[src])[rowx + max(ezx_s, 0)];
    }
    if (!upd_h) hyx_s = -1;
    if (!upd_e) ezx_s = -1;
  }
  // ---- row constants: lane q holds those of row rb - 1 + q, and bit q of the
  // masks says whether H / E of that row is updated and lies in a y strip
  float row_hy = 0.f, row_ey = 0.f, row_hb = 0.f, row_hc = 0.f, row_eb = 0.f, row_ec = 0.f;
  int row_hs = -1, row_es = -1;
  unsigned upd_hr = 0, upd_er = 0, strip_hr = 0, strip_er = 0;
  float phxy[KY ? R : 1], pezy[KY ? R : 1], gphxy = 0.f;
  if constexpr (KY) {
    const int row = rb - 1 + min(lane, R);
    const grec_ptr rec = (grec_ptr)a.rowinfo + (kRowRec / 4) * max(0, min(row, ny - 1));
    const rec_v4i w0 = rec[0], w1 = rec[1], w2 = rec[2];
    row_hy = __int_as_float(w0.x);
    row_ey = __int_as_float(w0.y);
    row_hb = __int_as_float(w1.z);
    row_hc = __int_as_float(w1.w);
    row_eb = __int_as_float(w2.x);
    row_ec = __int_as_float(w2.y);
    const bool h = lane <= R && row >= 0 && row <= ny - 2, e = lane <= R && row >= 1 && row <= ny - 2;
    row_hs = h ? w1.x : -1;
    row_es = e ? w1.y : -1;
    upd_hr = static_cast<unsigned>(__builtin_amdgcn_ballot_w64(h));
    upd_er = static_cast<unsigned>(__builtin_amdgcn_ballot_w64(e));
    strip_hr = static_cast<unsigned>(__builtin_amdgcn_ballot_w64(row_hs >= 0));
    strip_er = static_cast<unsigned>(__builtin_amdgcn_ballot_w64(row_es >= 0));
    if (strip_hr | strip_er) {
#pragma unroll
      for (int r = -1; r < R; ++r) {
        const float v = load(a.psi_hxy[src],
                             (static_cast<unsigned>(max(0, __builtin_amdgcn_readlane(row_hs, r + 1))) * pitch + cl) * 4u);
        if (r < 0) {
          gphxy = v;
          continue;
        }
        phxy[r < 0 ? 0 : r] = v;
        pezy[r < 0 ? 0 : r] =
            load(a.psi_ezy[src],
                 (static_cast<unsigned>(max(0, __builtin_amdgcn_readlane(row_es, r + 1))) * pitch + cl) * 4u);
      }
    }
  }
  if constexpr (MED == kTable) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int id = __float_as_int(ne[r]);
      const float4 m = lut_s[id];
      ca[r] = m.x;
      cb[r] = m.y;
      ne[r] = m.z;
      pec |= id == a.pec ? 1u << r : 0u;
    }
  }
  // ---- the wave's events: those of its rows whose column the tile loads, in
  // row, kind and index order, one per lane (the host keeps the streaming form
  // where a wave would have more than 64). They stay in registers, a source's
  // next value is loaded one step ahead, and a detector's lane fetches its
  // sample from the lane that holds the cell: a step waits for no memory.
  int ev_lane = 0, ev_row = -1, ev_idx = 0;  // the cell: its lane, its row of the wave
  float ev_src = 0.f;
  bool ev_is_src = false, ev_det = false, ev_comp = false;
  unsigned src_rows = 0, det_rows = 0, comp_rows = 0;  // rows with a source, with a sample to take
  // RC probes: the lane's place in a step's capture (-1: none); processing
  // line: the wave's row that is the line's (-1: none)
  int cap_at = -1, line_r = -1;
  bool has_cap = false;
  if constexpr (KE) {
    const int e0 = cld(a.ev_off, max(0, min(rb, ny))), e1 = cld(a.ev_off, max(0, min(rb + R, ny)));
    if (e0 < e1) {
      // gathered through the 128 words of LDS that the wave publishes to
      float *box = sh + wave * 2 * 64;
      int n = 0;
      for (int eb = e0; eb < e1; eb += 64) {
        rec_v4i v = {-1, 0, 0, 0};
        if (eb + lane < e1) v = ((grec_ptr)a.events)[eb + lane];
        const bool in = v.x >= t.cs && v.x < t.cs + 64;
        const unsigned long long m = __builtin_amdgcn_ballot_w64(in);
        const int at = n + __builtin_amdgcn_mbcnt_hi(m >> 32, __builtin_amdgcn_mbcnt_lo(m, 0));
        if (in && at < 64) {
          box[2 * at] = __int_as_float((v.x - t.cs) | v.y << 8 | (v.w - rb) << 16);
          box[2 * at + 1] = __int_as_float(v.z);
        }
        n += __builtin_popcountll(m);
      }
      if (lane < n) {
        const int w = __float_as_int(box[2 * lane]), kind = (w >> 8) & 255;
        ev_lane = w & 255;
        ev_row = w >> 16;
        ev_idx = __float_as_int(box[2 * lane + 1]);
        ev_is_src = kind == EV_SRC;
        const bool mine = rb + ev_row >= t.r0 && rb + ev_row < t.r1 && t.cs + ev_lane >= t.own0 && t.cs + ev_lane < t.own1;
        ev_det = mine && kind == EV_DET;
        ev_comp = mine && kind == EV_COMP;
      }
      if (ev_is_src) ev_src = gp(a.src_table)[static_cast<long long>(n0 + 1) * a.nsrc + ev_idx];
#pragma unroll
      for (int r = 0; r < R; ++r) {
        src_rows |= __builtin_amdgcn_ballot_w64(ev_is_src && ev_row == r) ? 1u << r : 0u;
        det_rows |= __builtin_amdgcn_ballot_w64((ev_det || ev_comp) && ev_row == r) ? 1u << r : 0u;
        comp_rows |= __builtin_amdgcn_ballot_w64(ev_comp && ev_row == r) ? 1u << r : 0u;
      }
    }
    if (a.nprobe > 0) {
      const int pr = gp(a.probe_col)[cl];
      cap_at = pr >= 0 && own ? pr * ny + rb : -1;
      has_cap = __builtin_amdgcn_ballot_w64(cap_at >= 0) != 0;
    }
    if (a.line_j >= max(rb, t.r0) && a.line_j < min(rb + R, t.r1)) line_r = a.line_j - rb;
  }

  float *mine = sh + wave * 2 * 64 + lane;  // [buffer][wave][first, last row][lane]
  const float *above = sh + (max(wave - 1, 0) * 2 + 1) * 64 + lane, *below = sh + min(wave + 1, W - 1) * 2 * 64 + lane;
  mine[0] = ez[0];
  mine[64] = ez[R - 1];

  // Ez of row r with its sources
  auto e_row = [&](int r, float hy_w) {
    if (!KY || (upd_er >> (r + 1) & 1)) {
      const float dey = KY ? lane_value(row_ey, r + 1) : uden_ey;
      const float eb = KY ? lane_value(row_eb, r + 1) : 0.f, ec = KY ? lane_value(row_ec, r + 1) : 0.f;
      const float cb_ = MED == kTable ? cb[MED == kTable ? r : 0] : cb0;
      if (upd_e) {
        const float dHy = hy[r] - hy_w;
        const float dHx = (r == 0 ? gh : hx[r == 0 ? 0 : r - 1]) - hx[r];
        float e = dHy * den_ex + dHx * dey;
        if (JZ != 0 && jz_on) {
          const float jn = jz_update(jz[r], decay, cj, ez[r], ne[r], jz_dt);
          jz[r] = JZ == 2 || ne[r] > 0.f ? jn : jz[r];
          e = e - jz[r];
        }
        e = (MED == kTable ? ca[MED == kTable ? r : 0] : ca0) * ez[r] + cb_ * e;
        if constexpr (MED == kTable) e = pec >> r & 1u ? 0.f : e;
        if constexpr (KX) {
          if (ezx_s >= 0) {
            pezx[r] = ezx_b * pezx[r] + div_by(ezx_c * dHy, rdx);
            e = e + cb_ * pezx[r];
          }
        }
        if constexpr (KY) {
          if (strip_er >> (r + 1) & 1) {
            pezy[r] = eb * pezy[r] + div_by(ec * dHx, rdy);
            e = e + cb_ * pezy[r];
          }
        }
        ez[r] = e;
      }
    }
    if constexpr (KE) {
      if (src_rows >> r & 1)
        for (unsigned long long m = __builtin_amdgcn_ballot_w64(ev_is_src && ev_row == r); m; m &= m - 1) {
          const int l = __builtin_ctzll(m);
          const float v = lane_value(ev_src, l);
          ez[r] = lane == __builtin_amdgcn_readlane(ev_lane, l) ? ez[r] - v : ez[r];
        }
    }
  };
  // the lane's own event: the value of a row at its cell
  auto fetch = [&](float v) { return __int_as_float(__builtin_amdgcn_ds_bpermute(ev_lane * 4, __float_as_int(v))); };
  // the samples and captures of a step
  auto samples = [&](int step) {
    if (det_rows) {
      float v = 0.f, vx = 0.f, vy = 0.f;
#pragma unroll
      for (int r = 0; r < R; ++r) {
        if (!(det_rows >> r & 1)) continue;
        const float u = fetch(ez[r]);
        v = ev_row == r ? u : v;
        if (comp_rows >> r & 1) {
          const float ux = fetch(hx[r]), uy = fetch(hy[r]);
          vx = ev_row == r ? ux : vx;
          vy = ev_row == r ? uy : vy;
        }
      }
      if (ev_det) gp(a.det)[static_cast<long long>(step) * a.ndet + ev_idx] = v;
      if (ev_comp) {
        gfloat *q = gp(a.comp) + static_cast<long long>(step) * a.ncomp + ev_idx;
        q[0] = v;
        q[a.comp_plane] = vx;
        q[2 * a.comp_plane] = vy;
      }
    }
    if (has_cap) {
      gfloat *q = gp(a.rc_cap) + static_cast<long long>((step - 1) & (kMaxT - 1)) * a.nprobe * ny;
      if (cap_at >= 0) {
#pragma unroll
        for (int r = 0; r < R; ++r)
          if (rb + r >= t.r0 && rb + r < t.r1) q[cap_at + r] = ez[r];
      }
    }
    if (line_r >= 0 && step > a.line_begin && step <= a.line_end) {
      gfloat *lp = gp(a.line) + static_cast<long long>(step - a.line_begin - 1) * (a.line_i1 - a.line_i0);
      float v = ez[0];
#pragma unroll
      for (int r = 1; r < R; ++r) v = line_r == r ? ez[r] : v;
      if (own && col >= a.line_i0 && col < a.line_i1) lp[col - a.line_i0] = v;
    }
  };

  for (int s = 0; s < T; ++s) {
    step_barrier();
    // rows whose state after this step the stored rows depend on; a wave with
    // none of them is done (it still takes part in the barriers)
    const int left = T - 1 - s;
    if (rb + R <= t.r0 - left || rb >= t.r1 + left || (KY && rb >= ny)) continue;
    const int buf = (s & 1) * (W * 2 * 64);
    const float up = above[buf], dn = below[buf];
    float src_next = 0.f;
    if constexpr (KE) {
      if (src_rows) {
        if (ev_is_src) src_next = gp(a.src_table)[static_cast<long long>(n0 + min(s + 2, T)) * a.nsrc + ev_idx];
      }
    }
    // ---- H of every row (-1: the copy of the row above)
    float ez_e[R];
#pragma unroll
    for (int r = 0; r < R; ++r) ez_e[r] = lane_from_next(ez[r]);
#pragma unroll
    for (int r = -1; r < R; ++r) {
      if (KY && !(upd_hr >> (r + 1) & 1)) continue;
      const int q = r < 0 ? 0 : r;
      const float dhy = KY ? lane_value(row_hy, r + 1) : uden_hy;
      const float hb = KY ? lane_value(row_hb, r + 1) : 0.f, hc = KY ? lane_value(row_hc, r + 1) : 0.f;
      if (upd_h) {
        const float dEy = (r < 0 ? up : ez[q]) - (r + 1 < R ? ez[r + 1 < R ? r + 1 : 0] : dn);
        float &x = r < 0 ? gh : hx[q];
        x = x + db * (dEy * dhy);
        if constexpr (KY) {
          if (strip_hr >> (r + 1) & 1) {
            float &psi = r < 0 ? gphxy : phxy[q];
            psi = hb * psi + div_by(hc * dEy, rdy);
            x = x + db * psi;
          }
        }
        if (r >= 0) {
          const float dEx = ez_e[q] - ez[q];
          hy[q] = hy[q] + db * (dEx * den_hx);
          if constexpr (KX) {
            if (hyx_s >= 0) {
              phyx[q] = hyx_b * phyx[q] + div_by(hyx_c * dEx, rdx);
              hy[q] = hy[q] + db * phyx[q];
            }
          }
        }
      }
    }
    // ---- E: the edge rows first, so that they are published while the rows
    // between them are computed
    float hy_w[R];
#pragma unroll
    for (int r = 0; r < R; ++r) hy_w[r] = lane_from_prev(hy[r]);
    e_row(0, hy_w[0]);
    if constexpr (R > 1) e_row(R - 1, hy_w[R - 1]);
    mine[W * 2 * 64 - buf] = ez[0];
    mine[W * 2 * 64 - buf + 64] = ez[R - 1];
#pragma unroll
    for (int r = 1; r < R - 1; ++r) e_row(r, hy_w[r]);
    if constexpr (KE) {
      samples(n0 + s + 1);
      ev_src = src_next;
    }
  }

  // ---- step n0+T of the rows and columns the tile owns
  const int dst = 1 - src;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int row = rb + r;
    if (row < t.r0 || row >= t.r1) continue;
    const unsigned off = offset(row);
    const int hs = KY ? __builtin_amdgcn_readlane(row_hs, r + 1) : -1;
    const int es = KY ? __builtin_amdgcn_readlane(row_es, r + 1) : -1;
    if (!own) continue;
    auto store = [](void *base, unsigned o, float v) { *(gfloat *)((gchar *)base + o) = v; };
    store(a.ez[dst], off, ez[r]);
    store(a.hx[dst], off, hx[r]);
    store(a.hy[dst], off, hy[r]);
    if constexpr (JZ != 0) store(a.jz[dst], off, jz[r]);
    if constexpr (KY) {
      if (hs >= 0) store(a.psi_hxy[dst], (static_cast<unsigned>(hs) * pitch + cl) * 4u, phxy[r]);
      if (es >= 0) store(a.psi_ezy[dst], (static_cast<unsigned>(es) * pitch + cl) * 4u, pezy[r]);
    }
    if constexpr (KX) {
      if (hyx_s >= 0) gp(a.psi_hyx[dst])[row * a.xs + hyx_s] = phyx[r];
      if (ezx_s >= 0) gp(a.psi_ezx[dst])[row * a.xs + ezx_s] = pezx[r];
    }
  }
}

// One wave's part of an interior tile: 64*C columns (C per lane, adjacent), R
// rows, nothing but plain cells, straight-line code. Two columns per lane
// lose 2T of 128 columns to their halo instead of 2T of 64. CAP: the tile
// holds RC probe columns or the processing line (those need no general tile:
// they only store what a step computed).
template <int C, int R, int W, int MED, int JZ, bool CAP>
__device__ __forceinline__ void block_inner(const StepArgs &a, const float4 *lut_s, float *sh, int src, int n0, int T,
                                            const BlockTile &t, int wave) {
  const int lane = threadIdx.x & 63;
  const float db = a.db, ca0 = a.ca0, cb0 = a.cb0, cj = a.cj, decay = a.jz_decay;
  const float den_hx = a.uden_hx, den_ex = a.uden_ex, den_hy = a.uden_hy, den_ey = a.uden_ey;
  const double jz_dt = a.jz_dt;
  const int col = t.cs + lane * C;
  const int rb = t.rs + wave * R;
  const unsigned pitch4 = static_cast<unsigned>(a.pitch) * 4u;
  const unsigned off0 = static_cast<unsigned>(rb) * pitch4 + static_cast<unsigned>(col) * 4u;
  float ez[R][C], hx[R][C], hy[R][C], jz[R][C], gh[C];
  float ca[MED == kTable ? R : 1][C], cb[MED == kTable ? R : 1][C], ne[R][C];
  unsigned pec = 0;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const unsigned off = off0 + r * pitch4;
    oload<C>((const gchar *)a.ez[src], off, ez[r]);
    oload<C>((const gchar *)a.hx[src], off, hx[r]);
    oload<C>((const gchar *)a.hy[src], off, hy[r]);
    if constexpr (JZ != 0 || MED == kTable)
      oload<C>(MED == kTable ? (const gchar *)a.med_id : (const gchar *)a.med_ne, off, ne[r]);
    if constexpr (JZ != 0) oload<C>((const gchar *)a.jz[src], off, jz[r]);
  }
  oload<C>((const gchar *)a.hx[src], off0 - pitch4, gh);
  if constexpr (MED == kTable) {
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int c = 0; c < C; ++c) {
        const int id = __float_as_int(ne[r][c]);
        const float4 m = lut_s[id];
        ca[r][c] = m.x;
        cb[r][c] = m.y;
        ne[r][c] = m.z;
        pec |= id == a.pec ? 1u << (r * C + c) : 0u;
      }
  }
  int cap_at[C], line_r = -1;
  if constexpr (CAP) {
#pragma unroll
    for (int c = 0; c < C; ++c) {
      const int pr = a.nprobe > 0 ? gp(a.probe_col)[col + c] : -1;
      cap_at[c] = pr >= 0 && col + c >= t.own0 && col + c < t.own1 ? pr * a.ny + rb : -1;
    }
    if (a.line_j >= max(rb, t.r0) && a.line_j < min(rb + R, t.r1)) line_r = a.line_j - rb;
  }
  // [buffer][wave][first, last row][column of the lane][lane]
  constexpr int kRow = 64 * C, kBuf = W * 2 * kRow;
  float *mine = sh + wave * 2 * kRow + lane;
  const float *above = sh + (max(wave - 1, 0) * 2 + 1) * kRow + lane, *below = sh + min(wave + 1, W - 1) * 2 * kRow + lane;
  auto publish = [&](int buf) {
#pragma unroll
    for (int c = 0; c < C; ++c) {
      mine[buf + c * 64] = ez[0][c];
      mine[buf + kRow + c * 64] = ez[R - 1][c];
    }
  };
  publish(0);
  auto e_row = [&](int r) {
    float hy_w[C];
#pragma unroll
    for (int c = 1; c < C; ++c) hy_w[c] = hy[r][c - 1];
    hy_w[0] = lane_from_prev(hy[r][C - 1]);
#pragma unroll
    for (int c = 0; c < C; ++c) {
      const float dHy = hy[r][c] - hy_w[c];
      const float dHx = (r == 0 ? gh[c] : hx[r == 0 ? 0 : r - 1][c]) - hx[r][c];
      float e = dHy * den_ex + dHx * den_ey;
      if constexpr (JZ != 0) {
        const float jn = jz_update(jz[r][c], decay, cj, ez[r][c], ne[r][c], jz_dt);
        jz[r][c] = JZ == 2 || ne[r][c] > 0.f ? jn : jz[r][c];
        e = e - jz[r][c];
      }
      if constexpr (MED == kTable) {
        e = ca[r][c] * ez[r][c] + cb[r][c] * e;
        e = pec >> (r * C + c) & 1u ? 0.f : e;
      } else {
        e = ca0 * ez[r][c] + cb0 * e;
      }
      ez[r][c] = e;
    }
  };
  for (int s = 0; s < T; ++s) {
    step_barrier();
    const int left = T - 1 - s;
    if (rb + R <= t.r0 - left || rb >= t.r1 + left) continue;
    const int buf = (s & 1) * kBuf;
    float up[C], dn[C];
#pragma unroll
    for (int c = 0; c < C; ++c) {
      up[c] = above[buf + c * 64];
      dn[c] = below[buf + c * 64];
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
      float ez_e[C];
#pragma unroll
      for (int c = 0; c < C - 1; ++c) ez_e[c] = ez[r][c + 1];
      ez_e[C - 1] = lane_from_next(ez[r][0]);
#pragma unroll
      for (int c = 0; c < C; ++c) {
        const float dEy = ez[r][c] - (r + 1 < R ? ez[r + 1 < R ? r + 1 : 0][c] : dn[c]);
        hx[r][c] = hx[r][c] + db * (dEy * den_hy);
        const float dEx = ez_e[c] - ez[r][c];
        hy[r][c] = hy[r][c] + db * (dEx * den_hx);
      }
    }
#pragma unroll
    for (int c = 0; c < C; ++c) gh[c] = gh[c] + db * ((up[c] - ez[0][c]) * den_hy);
    e_row(0);
    if constexpr (R > 1) e_row(R - 1);
    publish(kBuf - buf);
#pragma unroll
    for (int r = 1; r < R - 1; ++r) e_row(r);
    if constexpr (CAP) {
      const int step = n0 + s + 1;
      gfloat *q = gp(a.rc_cap) + static_cast<long long>((step - 1) & (kMaxT - 1)) * a.nprobe * a.ny;
#pragma unroll
      for (int c = 0; c < C; ++c)
        if (cap_at[c] >= 0) {
#pragma unroll
          for (int r = 0; r < R; ++r)
            if (rb + r >= t.r0 && rb + r < t.r1) q[cap_at[c] + r] = ez[r][c];
        }
      if (line_r >= 0 && step > a.line_begin && step <= a.line_end) {
        gfloat *lp = gp(a.line) + static_cast<long long>(step - a.line_begin - 1) * (a.line_i1 - a.line_i0);
#pragma unroll
        for (int c = 0; c < C; ++c) {
          float v = ez[0][c];
#pragma unroll
          for (int r = 1; r < R; ++r) v = line_r == r ? ez[r][c] : v;
          const int i = col + c;
          if (i >= t.own0 && i < t.own1 && i >= a.line_i0 && i < a.line_i1) lp[i - a.line_i0] = v;
        }
      }
    }
  }
  const int dst = 1 - src;
  // own0, own1 and col are multiples of C (the host's column split)
  if (col < t.own0 || col >= t.own1) return;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    if (rb + r < t.r0 || rb + r >= t.r1) continue;
    const unsigned off = off0 + r * pitch4;
    ostore<C>((const gchar *)a.ez[dst], off, ez[r]);
    ostore<C>((const gchar *)a.hx[dst], off, hx[r]);
    ostore<C>((const gchar *)a.hy[dst], off, hy[r]);
    if constexpr (JZ != 0) ostore<C>((const gchar *)a.jz[dst], off, jz[r]);
  }
}

// The work-group's tile. An interior tile has C columns per lane and R rows
// per wave; one that holds anything else (flags) one column per lane and RG
// rows per wave, each wave running what its own rows hold. (The barriers of
// the step loop are met by every wave, each in its own form's loop.)
template <int C, int R, int RG, int W, int MED>
__device__ __forceinline__ void run_block(const StepArgs &a, const float4 *lut_s, float *sh, int src, int n0, int T,
                                          const BlockTile &t) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const bool x = t.flags & kBlockX, y = t.y_waves >> wave & 1, e = t.e_waves >> wave & 1;
  const bool jz = t.jz_waves >> wave & 1, full = t.full_waves >> wave & 1;
  // The marks keep the compiler from merging the forms' common beginnings and
  // ends (their loads and stores would then hold every form's state at once:
  // 95 instead of 67 registers at C = 2, R = 4).
#define FDTD2D_WAVE(K)                                                    \
  {                                                                       \
    asm volatile("; general %0" ::"n"(K));                                \
    block_wave<RG, W, K, MED, 1>(a, lut_s, sh, src, n0, T, t, wave, jz);  \
    asm volatile("; end general %0" ::"n"(K));                            \
  }
#define FDTD2D_INNER(JZ, CAP)                                             \
  {                                                                       \
    asm volatile("; interior %0" ::"n"(2 * JZ + CAP));                    \
    block_inner<C, R, W, MED, JZ, CAP>(a, lut_s, sh, src, n0, T, t, wave); \
    asm volatile("; end interior %0" ::"n"(2 * JZ + CAP));                \
  }
  if (t.flags & kBlockGeneral) {
    if (e) FDTD2D_WAVE(kGeneral)
    else if (x && y) FDTD2D_WAVE(kX | kY)
    else if (x) FDTD2D_WAVE(kX)
    else if (y) FDTD2D_WAVE(kY)
    else FDTD2D_WAVE(0)
    return;
  }
  if (t.flags & kBlockCap) FDTD2D_INNER(1, true)
  else if (!jz) FDTD2D_INNER(0, false)
  else if (MED == kDensity && full) FDTD2D_INNER(2, false)
  else FDTD2D_INNER(1, false)
#undef FDTD2D_WAVE
#undef FDTD2D_INNER
}

__device__ __forceinline__ BlockTile load_block(const BlockTile *list, int pos) {
  BlockTile t;
  const rec_ptr q = (rec_ptr)list + static_cast<long long>(pos) * (sizeof(BlockTile) / 16);
  const rec_v4i a = q[0], b = q[1], c = q[2];
  t.cs = a.x;
  t.rs = a.y;
  t.own0 = a.z;
  t.own1 = a.w;
  t.r0 = b.x;
  t.r1 = b.y;
  t.flags = b.z;
  t.y_waves = b.w;
  t.e_waves = c.x;
  t.jz_waves = c.y;
  t.full_waves = c.z;
  t.slot = c.w;
  return t;
}

// Every tile of the grid, one work-group each (see step_kernel for the
// arguments and the XCD-aware order).
template <int C, int R, int RG, int W, int MED, int O>
__global__ void __launch_bounds__(64 * W, O) block_kernel(const StepArgs args, int src, int n0, int T) {
  const StepArgs &a = *(const StepArgs *)((cargs_ptr)__builtin_amdgcn_kernarg_segment_ptr());
  __shared__ float4 lut_s[MED == kTable ? 256 : 1];
  __shared__ float sh[2 * W * 2 * 64 * C];
  if constexpr (MED == kTable) {
    for (int q = threadIdx.x; q < a.nmat; q += blockDim.x) lut_s[q] = gload4(a.lut, q);
    __syncthreads();
  }
  const int G = gridDim.x, b = blockIdx.x;
  const int xcd = b & 7, q = G >> 3, rr = G & 7;
  run_block<C, R, RG, W, MED>(a, lut_s, sh, src, n0, T, load_block(a.block_list, xcd * q + min(xcd, rr) + (b >> 3)));
}

// The tiles of a pool's shots (list 0 of q), launch k of a chunk.
template <int C, int R, int RG, int W, int MED, int O>
__global__ void __launch_bounds__(64 * W, O)
    block_pool_kernel(const StepArgs *__restrict__ descs, const PoolQueue *__restrict__ q, int k, int tp, int T) {
  __shared__ float4 lut_s[MED == kTable ? 256 : 1];
  __shared__ float sh[2 * W * 2 * 64 * C];
  const int G = q->count[0], b = blockIdx.x;
  if (b >= G) return;
  const int xcd = b & 7, n = G >> 3, rr = G & 7;
  const BlockTile t =
      load_block(reinterpret_cast<const BlockTile *>(q->items[0]), xcd * n + min(xcd, rr) + (b >> 3));
  const StepArgs &a = *(const StepArgs *)((cargs_ptr)(descs + t.slot));
  if constexpr (MED == kTable) {
    for (int m = threadIdx.x; m < a.nmat; m += blockDim.x) lut_s[m] = gload4(a.lut, m);
    __syncthreads();
  }
  const int g = __builtin_amdgcn_readfirstlane(q->g) + k;
  const int dg = a.g_stride == 1 ? g - a.g_base : (g - a.g_base) / a.g_stride;
  run_block<C, R, RG, W, MED>(a, lut_s, sh, a.src_base ^ (dg & 1), a.n_base + dg * tp, T, t);
}

}  // namespace
}  // namespace fdtd2d

#endif
