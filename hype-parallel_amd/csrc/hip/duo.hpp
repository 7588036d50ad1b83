// duo.hpp -- the stage kernel's work on a tile, shared by the two waves of a
// workgroup (included by sweep.hip, whose helpers it uses).
//
// Both waves sweep the tile's rows together over one LDS window.  Wave X
// (wave 0) reconstructs the first half of the components and takes the x-faces
// and the volume term; wave Y reconstructs the other half and takes the y-faces,
// the assembly and stage update, and loads the rows to come.  A row has two
// barriers:
//
//   reconstruct own components -> coefficients to LDS
//   --- barrier 1 ---
//   all coefficients; values at the own faces' nodes and their admissibility;
//   X: last row's x part to LDS; Y: row r+3 into the window
//   --- barrier 2 ---
//   fallback where either wave's check failed; own faces; Y: assembly of row r-1
//
// No value is computed twice.  A row takes 0.49 (Baer-Nunziato, conservative: a
// node's flux shares the admissibility check's divisions here) to 0.585 (Euler)
// of the time one wave takes for it, against one row in two for the halves of a
// split tile, whose ring rows and middle face come on top.  So this layout is the
// fastest where tiles are a few rows high: Kapila 512x256 174 -> 157 us per step,
// 64x64 101 -> 79; order 3 256x256 444 -> 375; Baer-Nunziato 128x128 183 -> 121,
// 512x512 464 -> 423, 2048x1024 2452 -> 2411.  The host's tile-shape model
// (hype_pick_layout) decides.
#pragma once

namespace HYPE_KNS {

template <class S, bool PRIM, int N, bool IN>
struct Duo {
  static constexpr int NV = S::NV;
  using Qd = Quad<N>;
  using T1 = Tile<S, PRIM, N, false, IN>;  // face sums and weights
  static constexpr int NDOF = Qd::NDOF, NGF = Qd::NGF, NGV = Qd::NGV;
  static constexpr int WAVES = 2;
  static constexpr int NX = NV / 2;     // components wave X reconstructs
  static constexpr int NN = 2 * NGF;    // nodes per wave: the high side's face points, then the low side's
  static constexpr bool ACACHE = PRIM && S::HAS_ACACHE && N == 2;
  static constexpr bool CHECK_EACH = NV > 6;
  static constexpr bool STAGE_ROWS = NV > 6;
  static constexpr int njump() {
    int n = 0;
    for (int c = 0; c < NV; ++c) n += S::HAS_NCP && S::DNZ[c];
    return n;
  }
  static constexpr int jump_index(int c) {
    int n = 0;
    for (int k = 0; k < c; ++k) n += S::HAS_NCP && S::DNZ[k];
    return n;
  }
  // LDS, in doubles: the window; the coefficients 1.. of every component; the x
  // part and volume term of a row; the staging of the four window columns right
  // of the lanes' 64 (primitive path, 16 rows at a time); the staging of output
  // rows (long records); the two check masks and wave Y's largest wave speed
  static constexpr int WIN = NSLOT * NV * COLS;
  static constexpr int COF = NV * (NDOF - 1) * HYPE_WAVE;
  static constexpr int PART = (NV + njump()) * HYPE_WAVE;
  static constexpr int XST = PRIM ? 16 * 4 * NV : 0;
  static_assert(!(STAGE_ROWS && N == 3), "RK104's second output row is not staged: layouts() leaves this out");
  static constexpr int OST = STAGE_ROWS ? NV * HYPE_TILE_W : 0;
  static constexpr int LDS = WIN + COF + PART + XST + OST + 3;

  // values of all components at the wave's nodes
  template <bool X>
  __device__ static __forceinline__ void at_nodes(const double (&co)[NV][NDOF], double (&fv)[NN][NV]) {
    static_for<NN>([&](auto i) {
      static_for<NV>([&](auto c) {
        fv[i][c] = basis_sum<RowNode<N, (X ? 0 : 2 * NGF) + i>, NDOF, S::RANGE[PRIM][c] != NORMAL>(co[c]);
      });
    });
  }

  __device__ static __forceinline__ void run(const hype_launch& L, int tile_id, double* lds, int lane, int wave) {
    const hype_tile T = L.tiles[tile_id];
    const hype_inst* I = &L.insts[T.inst];
    hype_dstate* st = I->st;
    const int nx = I->nx, ny = I->ny;
    const int bcL = I->bc[0], bcR = I->bc[1], bcB = I->bc[2], bcT = I->bc[3];
    const double r1_h = I->r1_h;
    Eos eos{I->g1, I->g2, I->p1, I->p2, (I->quirks & HYPE_QUIRK_BN_P2_IS_PHI) != 0, 1.0, 1.0, 1.0, 1.0};
    if constexpr (PRIM) {
      double d1, d2;
      S::energy_den(eos, d1, d2);
      eos.d1 = uniform(d1);
      eos.d2 = uniform(d2);
      eos.y1 = uniform(recip_nr(d1));
      eos.y2 = uniform(recip_nr(d2));
    }
    const bool leader = (T.flags & 1) != 0 && wave == 0;
    const int mode = L.mode;
    double dt = 0.0;
    int cur = 0;
    StageDesc sd = stage_desc(N, L.stage);
    const bool last_stage = (mode == HYPE_MODE_STAGE) && (L.stage == num_stages_dev(N) - 1);
    const auto Uin = gmem<const double>((mode == HYPE_MODE_STAGE) ? I->buf[sd.in] : (L.rhs_in ? L.rhs_in : I->buf[0]));
    const auto Out = gmem((mode == HYPE_MODE_STAGE) ? I->buf[sd.out] : (L.rhs_out ? L.rhs_out : I->buf[1]));
    const auto Xb = gmem<const double>(I->buf[sd.xb]);
    const auto Zb = gmem<const double>(I->buf[sd.zb]);
    const auto Ab = gmem(I->buf[1]);

    const int x0 = T.x0, y0 = T.y0;
    const int W = T.w, H = T.h;
    const int col = x0 - 1 + lane;
    const bool owned = lane >= 1 && lane <= W;
    const bool xlane = lane >= 1 && lane <= W + 1;
    const int cw = lane + 2;
    const int r_first = y0 - 1, r_last = y0 + H;  // ring rows below and above the tile
    const int rbase = r_first - 2;
    double* win = lds;
    double* cof = win + WIN;
    double* part = cof + COF;
    double* xs = part + PART;
    double* ost = xs + XST;
    unsigned long long* mask = (unsigned long long*)(ost + OST);
    double* y_smax = ost + OST + 2;
    auto slot = [&](int r) { return (r - rbase) % NSLOT; };
    auto W_ = [&](int s, int c, int k) -> double& { return win[(s * NV + c) * COLS + k]; };
    auto C_ = [&](int c, int k) -> double& { return cof[(c * (NDOF - 1) + k - 1) * HYPE_WAVE + lane]; };
    auto P_ = [&](int k) -> double& { return part[k * HYPE_WAVE + lane]; };

    // ---- row loader (as in Tile) ---------------------------------------
    // a cell's column is the same in every row: its source offset and the sign its
    // reflection gives the x velocity are found once (lane k's window column, and
    // the one right of the lanes' 64 that lanes 0-3, or all in turn, load)
    auto column = [&](int k, unsigned& mx) -> size_t {
      bool fx = false;
      const int sc = bc_map(min(x0 - 3 + k, nx + 2), nx, bcL, bcR, fx);  // an inlet column maps as periodic; put_inlet replaces it
      mx = fx ? SIGN_BIT : 0u;
      return (size_t)sc * NV;
    };
    unsigned mxa, mxb;
    const size_t cola = column(lane, mxa), colb = column(HYPE_WAVE + (lane & 3), mxb);
    auto fetch = [&](int rr, size_t co, double* q) -> unsigned {
      bool fy = false;
      const int sr = bc_map(rr, ny, bcB, bcT, fy);
      const auto p = Uin + (size_t)sr * nx * NV + co;
#pragma unroll
      for (int c = 0; c < NV; ++c) q[c] = p[c];
      return fy ? SIGN_BIT : 0u;
    };
    auto conv = [&](double* q, unsigned mx, unsigned my, double* v) {
      q[S::REFX[0]] = flip_sign(q[S::REFX[0]], mx);
      if (S::REFX[1] >= 0) q[S::REFX[1]] = flip_sign(q[S::REFX[1]], mx);
      q[S::REFY[0]] = flip_sign(q[S::REFY[0]], my);
      if (S::REFY[1] >= 0) q[S::REFY[1]] = flip_sign(q[S::REFY[1]], my);
      if (PRIM) {
        S::cons2prim(eos, q, v);
      } else {
#pragma unroll
        for (int c = 0; c < NV; ++c) v[c] = q[c];
      }
    };
    auto put = [&](int s, int k, double* q, unsigned mx, unsigned my) {
      double v[NV];
      conv(q, mx, my, v);
#pragma unroll
      for (int c = 0; c < NV; ++c) W_(s, c, k) = v[c];
    };
    // the four window columns right of the lanes' 64: on the primitive path
    // converted 16 rows at a time, one cell per lane, and copied a row at a time
    // by lanes 0-3; on the conservative path loaded by lanes 0-3 with each row
    auto xrow = [&](int j0) { return rbase + j0 + (lane >> 2); };
    auto xput = [&](double* q, unsigned my) {
      double v[NV];
      conv(q, mxb, my, v);
#pragma unroll
      for (int c = 0; c < NV; ++c) xs[c * HYPE_WAVE + lane] = v[c];
    };
    auto xcopy = [&](int s, int j) {
      if (lane < 4) {
#pragma unroll
        for (int c = 0; c < NV; ++c) W_(s, c, HYPE_WAVE + lane) = xs[c * HYPE_WAVE + (j & 15) * 4 + lane];
      }
    };
    const bool inlet_strip = IN && bcL == HYPE_BC_INLET && x0 == 0;
    auto put_inlet = [&](int s, int rr) {
      if constexpr (IN) {
        if (inlet_strip && lane < 3) {
          bool fy = false;
          const int sr = bc_map(rr, ny, bcB, bcT, fy);
          const bool own = (rr < 0 && bcB == HYPE_BC_PERIODIC) || (rr >= ny && bcT == HYPE_BC_PERIODIC);
          const auto p = gmem(I->inlet) + (size_t)((own ? rr : sr) + 3) * NV;
          double v[NV];
#pragma unroll
          for (int c = 0; c < NV; ++c) v[c] = p[c];
          if (fy) {
            v[S::REFY[0]] = -v[S::REFY[0]];
            if (S::REFY[1] >= 0) v[S::REFY[1]] = -v[S::REFY[1]];
          }
#pragma unroll
          for (int c = 0; c < NV; ++c) W_(s, c, lane) = v[c];
        }
      }
    };

    // prologue: rows r_first-2 .. r_first+2, three by wave X and two with the
    // right-hand columns by wave Y, in flight before the time state is read
    double pq[3][NV], pqb[NV];
    unsigned pf[3] = {0, 0, 0}, pfb = 0;
    const int pr0 = wave == 0 ? 0 : 3, prn = wave == 0 ? 3 : 2;
    const bool pxl = wave == 1 && (PRIM ? xrow(0) <= r_last + 2 : lane < 20);
#pragma unroll
    for (int i = 0; i < 3; ++i)
      if (i < prn) pf[i] = fetch(rbase + pr0 + i, cola, pq[i]);
    if (pxl) pfb = fetch(xrow(0), colb, pqb);

    // ---- time state (single writer per field per launch; as in Tile) -----
    if (mode == HYPE_MODE_STAGE) {
      if (L.stage == 0) {
        const int step = st->step;
        const double t = st->t;
        if (step >= st->max_steps || !(t < st->t_end) || st->err[(step + 1) & 1] != ~0ull) {
          if (leader && lane == 0) st->done = 1;
          return;
        }
        const double sm = __longlong_as_double((long long)st->smax[step & 1]);
        dt = (I->cfl * I->h) / (2.0 * sm);
        if (st->clip && t + dt > st->t_end) dt = st->t_end - t;
        cur = step;
        if (leader && lane == 0) {
          st->dt = dt;
          st->cur = step;
          st->smax[(step + 1) & 1] = 0ull;
          if (st->dt_hist && step < st->hist_len) st->dt_hist[step] = dt;
        }
      } else {
        if (st->done) return;
        dt = st->dt;
        cur = st->cur;
      }
      if (last_stage && leader && lane == 0) {
        st->t = st->t + dt;
        st->step = cur + 1;
        st->err[(cur + 1) & 1] = ~0ull;
      }
    }
    const double cdt = dt / sd.bden;

#pragma unroll
    for (int i = 0; i < 3; ++i)
      if (i < prn) {
        put(slot(rbase + pr0 + i), lane, pq[i], mxa, pf[i]);
        put_inlet(slot(rbase + pr0 + i), rbase + pr0 + i);
      }
    if (wave == 1) {
      if constexpr (PRIM) {
        if (pxl) xput(pqb, pfb);
        wave_sync();
#pragma unroll
        for (int i = 0; i < 5; ++i) xcopy(slot(rbase + i), i);
      } else {
        if (pxl) put(slot(rbase + (lane >> 2)), HYPE_WAVE + (lane & 3), pqb, mxb, pfb);
      }
    }
    __syncthreads();

    double smax = 0.0;  // largest wave speed of the wave's faces, over all lanes (masked at the end)
    unsigned long long err = ~0ull;
    const int seq = (mode == HYPE_MODE_STAGE) ? L.stage + 1 : 0;
    auto report = [&](long key0, int q, const double* Lv, const double* Rv, bool mine, bool bad) {
      if (mine && bad) {
        const Bad b = riemann_diag<S, PRIM>(eos, Lv, Rv);
        const unsigned long long pk = pack_err(seq, key0 + q, b.kind, b.val, I->keybits);
        if (b.kind && pk < err) err = pk;
      }
    };

    // ---- output (as in Tile) --------------------------------------------
    auto put_out = [&](double val, gmem_t<double>* dst, size_t i, int c) {
      if constexpr (STAGE_ROWS) ost[(lane - 1) * NV + c] = val;
      else __builtin_nontemporal_store(val, &dst[i]);
    };
    auto flush = [&](gmem_t<double>* dst, int row) {
      wave_sync();
      const size_t first = ((size_t)row * nx + x0) * NV;
      for (int e = lane; e < W * NV; e += HYPE_WAVE) __builtin_nontemporal_store(ost[e], &dst[first + e]);
      wave_sync();
    };
    auto operand = [&](gmem_t<const double>* B, size_t i, int row, int c) -> double {
      if constexpr (!PRIM) {
        if (B == Uin) return W_(slot(row), c, lane + 2);
      }
      return B[i];
    };
    auto record = [&](int row, const double* Gt, const double* Gb, const double* Et, const double* Eb) {
      const size_t idx = ((size_t)row * nx + col) * NV;
      double rhs[NV];
      static_for<NV>([&](auto c) {
        const double t = P_(c) - T1::template face_diff<c>(r1_h, Gt[c], Gb[c], Et[c], Eb[c]);
        rhs[c] = ((S::HAS_NCP && S::DNZ[c]) ? P_(NV + jump_index(c)) : 0.0) + t;
      });
      if (mode == HYPE_MODE_RHS) {
#pragma unroll
        for (int c = 0; c < NV; ++c) put_out(rhs[c], Out, idx + c, c);
      } else if (sd.op == 0) {
        double u[NV];
#pragma unroll
        for (int c = 0; c < NV; ++c) u[c] = operand(Uin, idx + c, row, c);
#pragma unroll
        for (int c = 0; c < NV; ++c) put_out(u[c] + cdt * rhs[c], Out, idx + c, c);
      } else if (sd.op == 2) {
        if constexpr (N == 3) {  // RK104 after its fifth stage
          double u[NV], o[NV];
#pragma unroll
          for (int c = 0; c < NV; ++c) {
            u[c] = operand(Uin, idx + c, row, c);
            o[c] = Out[idx + c];
          }
#pragma unroll
          for (int c = 0; c < NV; ++c) {
            const double w0 = u[c] + cdt * rhs[c];
            const double w1 = sd.a * o[c] + sd.g * w0;
            put_out(w1, Out, idx + c, c);
            put_out(15.0 * w1 + -5.0 * w0, Ab, idx + c, c);
          }
        }
      } else {
        double x[NV], z[NV];
#pragma unroll
        for (int c = 0; c < NV; ++c) {
          x[c] = operand(Xb, idx + c, row, c);
          z[c] = operand(Zb, idx + c, row, c);
        }
#pragma unroll
        for (int c = 0; c < NV; ++c) put_out(sd.a * x[c] + cdt * rhs[c] + sd.g * z[c], Out, idx + c, c);
      }
    };
    auto assemble = [&](int row, const double* Gt, const double* Gb, const double* Et, const double* Eb) {
      if (mode == HYPE_MODE_PRIME) return;
      if (owned) record(row, Gt, Gb, Et, Eb);
      if constexpr (STAGE_ROWS) {
        flush(Out, row);
      }
    };

    // flux and jump sums of a face from the states either side.  On the
    // conservative path the sides' fluxes and speeds come with them
    struct Side {
      double F[PRIM ? 1 : NGF][NV], s[NGF];  // s: the speed, or (ACACHE) a_sq
      int bad[NGF];
    };
    auto face = [&](auto dir, const double (&Lv)[NGF][NV], const double (&Rv)[NGF][NV], const Side& Ls, const Side& Rs,
                    long key0, bool mine, double* G, double* E) {
      constexpr int DIR = decltype(dir)::value;
      bool bad[NGF], any = false;
#pragma unroll
      for (int q = 0; q < NGF; ++q) {
        double A[NV], D[NV], s;
        if constexpr (PRIM) {
          s = riemann<S, PRIM, ACACHE, DIR>(eos, Lv[q], Rv[q], A, D, bad[q], Ls.s[q], Rs.s[q]);
        } else {
          s = pmax(Ls.s[q], Rs.s[q]);
          bad[q] = (Ls.bad[q] | Rs.bad[q]) != 0;
#pragma unroll
          for (int c = 0; c < NV; ++c) {
            const double dQ = Rv[q][c] - Lv[q][c];
            A[c] = S::FZERO[c] ? -(s * dQ) : Rs.F[q][c] + Ls.F[q][c] - s * dQ;
          }
          S::template ncp_face<PRIM, DIR>(eos, Lv[q], Rv[q], D);
        }
        smax = fmax(smax, s);
        any |= bad[q];
        if constexpr (CHECK_EACH) {
          if (__builtin_expect(__ballot(bad[q]) != 0, 0)) report(key0, q, Lv[q], Rv[q], mine, bad[q]);
        }
        T1::add_point(q, A, D, G, E);
      }
      if (!CHECK_EACH && __builtin_expect(__ballot(any) != 0, 0)) {
#pragma unroll
        for (int q = 0; q < NGF; ++q) report(key0, q, Lv[q], Rv[q], mine, bad[q]);
      }
    };

    auto sweep = [&](auto isx) {
      constexpr bool X = decltype(isx)::value;
      constexpr int DIR = X ? 0 : 1;
      // carried: X the x part and volume term of the last row; Y the values, sides
      // and sums of the last row's top face
      double keep[X ? NV + njump() : 1];
      double top[X ? 1 : NGF][NV], G0[X ? 1 : NV], E0[X ? 1 : NV];
      Side tops;
      if constexpr (!X) {
#pragma unroll
        for (int c = 0; c < NV; ++c) {
          G0[c] = 0.0;
          E0[c] = 0.0;
#pragma unroll
          for (int q = 0; q < NGF; ++q) {
            top[q][c] = 0.0;
            if constexpr (!PRIM) tops.F[q][c] = 0.0;
          }
        }
#pragma unroll
        for (int q = 0; q < NGF; ++q) {
          tops.s[q] = 0.0;
          tops.bad[q] = 0;
        }
      }

      for (int r = r_first; r <= r_last; ++r) {
        const int jn = r - r_first + 5;  // window row of row r+3, from rbase
        const bool more = (r + 3 <= r_last + 2);
        const bool xb = PRIM && more && (jn & 15) == 0;
        const bool xl = xb && xrow(jn) <= r_last + 2;
        double qa[NV], qb[NV];
        unsigned fa = 0, fb = 0;
        if constexpr (!X) {
          if (more) {
            fa = fetch(r + 3, cola, qa);
            if constexpr (PRIM) {
              if (xl) fb = fetch(xrow(jn), colb, qb);
            } else {
              if (lane < 4) fb = fetch(r + 3, colb, qb);
            }
          }
        }
        const bool ownedRow = r >= y0 && r < y0 + H;
        const int sm2 = slot(r - 2), sm1 = slot(r - 1), s0 = slot(r), sp1 = slot(r + 1), sp2 = slot(r + 2);

        // ---- own components ------------------------------------------------
        double co[NV][NDOF];
        static_for<NV>([&](auto c) {
          if constexpr ((c < NX) == X) {
            double ux[5], uy[5], ud[5];
            ux[0] = W_(s0, c, cw - 2);
            ux[1] = W_(s0, c, cw - 1);
            ux[2] = W_(s0, c, cw);
            ux[3] = W_(s0, c, cw + 1);
            ux[4] = W_(s0, c, cw + 2);
            uy[0] = W_(sm2, c, cw);
            uy[1] = W_(sm1, c, cw);
            uy[2] = ux[2];
            uy[3] = W_(sp1, c, cw);
            uy[4] = W_(sp2, c, cw);
            ud[0] = ux[2];
            ud[1] = W_(sp1, c, cw + 1);
            ud[2] = W_(sm1, c, cw + 1);
            ud[3] = W_(sp1, c, cw - 1);
            ud[4] = W_(sm1, c, cw - 1);
            reconstruct<N, S::RANGE[PRIM][c]>(ux, uy, ud, co[c]);
#pragma unroll
            for (int k = 1; k < NDOF; ++k) C_(c, k) = co[c][k];
          }
        });
        __syncthreads();  // barrier 1: coefficients; rows r-2 .. r+2 have been read

        static_for<NV>([&](auto c) {
          if constexpr ((c < NX) != X) {
            co[c][0] = W_(s0, c, cw);
#pragma unroll
            for (int k = 1; k < NDOF; ++k) co[c][k] = C_(c, k);
          }
        });
        if constexpr (X) {
          if (r > y0) {
#pragma unroll
            for (int k = 0; k < NV + njump(); ++k) P_(k) = keep[k];
          }
        } else if (more) {  // row r+3 takes the slot of row r-2
          const int sn = slot(r + 3);
          put(sn, lane, qa, mxa, fa);
          if constexpr (PRIM) {
            if (xb) {
              if (xl) xput(qb, fb);
              wave_sync();
            }
            xcopy(sn, jn);
          } else {
            if (lane < 4) put(sn, lane + HYPE_WAVE, qb, mxb, fb);
          }
          put_inlet(sn, r + 3);
        }

        // ---- values at the nodes and their admissibility --------------------
        double fv[NN][NV], an[NN];
        Side hi, lo;  // of the high (right, top) and low (left, bottom) faces' nodes
        at_nodes<X>(co, fv);
        bool ok = true;
        auto sides = [&]() {  // conservative path: flux and speed at every node
          if constexpr (!PRIM) {
#pragma unroll
            for (int q = 0; q < NGF; ++q) {
              bool bh = false, bl = false;
              hi.s[q] = S::template side_cons<DIR>(eos, fv[q], hi.F[q], bh);
              lo.s[q] = S::template side_cons<DIR>(eos, fv[NGF + q], lo.F[q], bl);
              hi.bad[q] = bh;
              lo.bad[q] = bl;
            }
          }
        };
#pragma unroll
        for (int i = 0; i < NN; ++i) {
          if constexpr (ACACHE)
            ok = S::pad_prim_a(eos, fv[i], an[i]) && ok;
          else
            ok = (PRIM ? S::pad_prim(eos, fv[i]) : S::pad(eos, fv[i])) && ok;
        }
        sides();
        const unsigned long long mine = __ballot(ok);
        if (lane == 0) mask[X ? 0 : 1] = mine;
        __syncthreads();  // barrier 2: check masks, row r+3, row r-1's x part
        const bool pad = ((mine & mask[X ? 1 : 0]) >> lane) & 1;
        if (!pad) {  // rhs_function_prim.c:407-421 / rhs_function.c:409-421
#pragma unroll
          for (int c = 0; c < NV; ++c) {
            const double w0 = W_(s0, c, cw);
            co[c][0] = w0;
            if constexpr (NDOF > 1) {
              co[c][1] = PRIM ? minmod(W_(s0, c, cw + 1) - w0, w0 - W_(s0, c, cw - 1)) : 0.0;
              co[c][2] = PRIM ? minmod(W_(sp1, c, cw) - w0, w0 - W_(sm1, c, cw)) : 0.0;
            }
#pragma unroll
            for (int k = 3; k < NDOF; ++k) co[c][k] = 0.0;
          }
          at_nodes<X>(co, fv);
          if constexpr (ACACHE) {
#pragma unroll
            for (int i = 0; i < NN; ++i) an[i] = S::sound_sq_prim(eos, fv[i]);
          }
          sides();
        }
        if constexpr (ACACHE) {
#pragma unroll
          for (int q = 0; q < NGF; ++q) {
            hi.s[q] = an[q];
            lo.s[q] = an[NGF + q];
          }
        }
        double hv[NGF][NV], lv[NGF][NV];
#pragma unroll
        for (int q = 0; q < NGF; ++q)
#pragma unroll
          for (int c = 0; c < NV; ++c) {
            hv[q][c] = fv[q][c];
            lv[q][c] = fv[NGF + q][c];
          }

        if constexpr (X) {
          if (L.fallback && ownedRow && owned) gmem(L.fallback)[(size_t)r * nx + col] = (unsigned char)(!pad);
          if (ownedRow) {
            // ---- volume non-conservative product (rhs_function_prim.c:461-479)
            if constexpr (S::HAS_NCP) {
              if (mode != HYPE_MODE_PRIME) {
                double ncp[NV];
#pragma unroll
                for (int c = 0; c < NV; ++c) ncp[c] = 0.0;
                static_for<NGV>([&](auto q) {
                  double V[NV], gx[NV], gy[NV], B[NV];
                  T1::template at_vol<q>(co, r1_h, V, gx, gy);
                  S::template vol_ncp<PRIM>(eos, V, gx, gy, B);
                  T1::add_volume(B, ncp);
                });
                static_for<NV>([&](auto c) {
                  if constexpr (S::DNZ[c]) keep[NV + jump_index(c)] = ncp[c];
                });
              }
            }
            // ---- x-faces i-1/2 (rhs_function_prim.c:485-533) -----------------
            double vl[NGF][NV], Fx[NV], Dx[NV];
            Side ls;
#pragma unroll
            for (int q = 0; q < NGF; ++q) {
#pragma unroll
              for (int c = 0; c < NV; ++c) {
                vl[q][c] = lane_from_left(hv[q][c]);
                if constexpr (!PRIM) ls.F[q][c] = S::FZERO[c] ? 0.0 : lane_from_left(hi.F[q][c]);
              }
              if constexpr (ACACHE || !PRIM) ls.s[q] = lane_from_left(hi.s[q]);
              if constexpr (!PRIM) ls.bad[q] = lane_from_left_int(hi.bad[q]);
            }
            face(std::integral_constant<int, 0>{}, vl, lv, ls, lo, ((long)r * (nx + 1) + col) * NGF, xlane, Fx, Dx);
            static_for<NV>([&](auto c) {
              const double Dr = S::DNZ[c] ? lane_from_right(Dx[c]) : 0.0;
              keep[c] = -T1::template face_diff<c>(r1_h, lane_from_right(Fx[c]), Fx[c], Dr, Dx[c]);
            });
          }
        } else {
          // ---- y-face r-1/2 (rhs_function_prim.c:537-585), assembly of row r-1
          if (r >= y0) {
            double G1[NV], E1[NV];
            face(std::integral_constant<int, 1>{}, top, lv, tops, lo,
                 (long)ny * (nx + 1) * NGF + ((long)r * nx + col) * NGF, owned, G1, E1);
            if (r > y0) assemble(r - 1, G1, G0, E1, E0);
#pragma unroll
            for (int c = 0; c < NV; ++c) {
              G0[c] = G1[c];
              E0[c] = E1[c];
            }
          }
#pragma unroll
          for (int q = 0; q < NGF; ++q)
#pragma unroll
            for (int c = 0; c < NV; ++c) top[q][c] = hv[q][c];
          tops = hi;
        }
      }
    };
    if (wave == 0)
      sweep(std::true_type{});
    else
      sweep(std::false_type{});

    // ---- CFL maximum and error word ----------------------------------------
    const bool want_smax = (mode != HYPE_MODE_STAGE) || last_stage;
    if (want_smax) {
      const double m = wave_max((wave == 0 ? xlane : owned) ? smax : 0.0);
      if (wave == 1 && lane == 0) *y_smax = m;
      __syncthreads();
      if (wave == 0 && lane == 0) send_smax(L, st, cur, fmax(m, *y_smax));
    }
    const unsigned long long e = wave_min_u64(err);
    if (lane == 0) send_error(L, st, cur, e);
  }
};

}  // namespace HYPE_KNS
