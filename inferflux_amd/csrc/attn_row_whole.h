// The body of a workgroup of ``a.waves`` waves that takes row number ``ri`` of the launch and kv head ``kvh`` whole (attn_mfma.hip), for the kernels that
// do so: RowArgs a, int kvh, int ri, float* lds and the switches STREAM and KEEP are in scope.  Text and not a function: inlined as one it takes the row kernel, which
// decode steps of few rows launch once a layer, 0.1 us longer (one row of 70 keys, 14 heads of 64 on 2, 4.34 us and 4.45).
  const int tid = threadIdx.x, wid = tid / WAVE, lane = tid % WAVE, col = lane & 15, g4 = lane >> 4;
  const int W = a.waves, n_threads = W * WAVE;
  const int row = a.rows ? a.rows[ri] : ri;
  const int pos = a.positions[row];
  const int lo = first_seen(pos, a.window, a.block);
  // this wave's keys: the visible ones from the first visible run of 32 on, in W equal shares of whole runs.  With
  // kept first keys [0, keep) before the window the runs are numbered as if the window's first run followed the last
  // kept run: walk place v is key v below kr and key v + gap from there on.
  const int first = lo / 32 * 32;
  const int keep = (KEEP && lo > 0) ? min(a.keep_first, lo) : 0;
  const int keep_runs = (keep + 31) / 32 * 32;
  const int base = (KEEP && keep > 0) ? 0 : first;
  const int gap = (KEEP && keep > 0 && keep_runs < first) ? first - keep_runs : 0, kr = (KEEP && gap > 0) ? keep_runs : 0;
  const int vend = pos + 1 - gap;
  const int chunk = ((vend - base + W - 1) / W + 31) / 32 * 32;
  const int va = base + wid * chunk, vb = min(vend, base + (wid + 1) * chunk);     // this wave's places [va, vb), whole runs
  const int ka = lo, kb = pos + 1, ke = keep;                                      // what is visible at all
  auto key_at = [&](int v) { return KEEP ? (v < kr ? v : v + gap) : v; };
  const int ratio = a.nH / a.nKV;
  const int nc_max = min(16, ratio);
  const int* table = a.block_table + (size_t)a.row_req[row] * a.max_blocks;
  float* o_s = lds;                                        // [W][nc_max][OPAD]
  float* ml_s = lds + W * nc_max * OPAD;                   // [W][nc_max][2]
  constexpr int D4 = D / 4;

  for (int qt = 0; qt < ratio; qt += 16) {
    const int nc = min(16, ratio - qt);
    const int head = kvh * ratio + qt + col;
    const bool head_ok = col < nc;
    floatx4 o[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) o[dt] = floatx4{0.f, 0.f, 0.f, 0.f};
    float m = -INFINITY, l = 0.f;
    if (va < vb) {
      bf16x8 qop[KS];
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const int c = 32 * ks + 8 * g4;
        qop[ks] = (head_ok && c < D) ? *(const bf16x8*)(a.q + ((size_t)row * a.nH + head) * D + c) : zero8();
      }
      RowBlock b0, b1;
      int j0 = va;
      int page_base = 0, pages = -1;
      bool have_pages = false;
      auto table_for = [&](int j) {
        if (have_pages && (j + 31) / a.P - page_base < WAVE) return;
        have_pages = true;
        page_base = j / a.P;
        pages = page_base + lane < a.max_blocks ? table[page_base + lane] : -1;
      };
      table_for(key_at(j0));
      load_row_block<STREAM>(b0, a, pages, page_base, kvh, key_at(j0), ka, kb, col, g4, ke);
      for (; j0 < vb; j0 += 64) {
        const bool more1 = j0 + 32 < vb, more2 = j0 + 64 < vb;
        if (more1) {
          table_for(key_at(j0 + 32));
          load_row_block<STREAM>(b1, a, pages, page_base, kvh, key_at(j0 + 32), ka, kb, col, g4, ke);
        }
        use_row_block(b0, a, qop, o, m, l, key_at(j0), ka, kb, g4, ke);
        if (more1) {
          if (more2) {
            table_for(key_at(j0 + 64));
            load_row_block<STREAM>(b0, a, pages, page_base, kvh, key_at(j0 + 64), ka, kb, col, g4, ke);
          }
          use_row_block(b1, a, qop, o, m, l, key_at(j0 + 32), ka, kb, g4, ke);
        }
      }
      l = col_sum(l);
    }
    // the waves' results meet in LDS (a wave without visible keys brings weight zero)
    if (qt > 0) __syncthreads();                           // everyone is done with the last pass's LDS
    if (head_ok) {
      float* os = o_s + (wid * nc_max + col) * OPAD;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) *(floatx4*)(os + 16 * dt + 4 * g4) = o[dt];
      if (g4 == 0) { ml_s[(wid * nc_max + col) * 2] = m; ml_s[(wid * nc_max + col) * 2 + 1] = l; }
    }
    __syncthreads();
    for (int i = tid; i < nc * D4; i += n_threads) {
      const int c = i / D4, e = 4 * (i % D4);
      float M = -INFINITY;
      for (int w = 0; w < W; ++w) M = fmaxf(M, ml_s[(w * nc_max + c) * 2]);
      floatx4 acc{0.f, 0.f, 0.f, 0.f};
      float L = 0.f;
      for (int w = 0; w < W; ++w) {
        const float mw = ml_s[(w * nc_max + c) * 2];
        if (mw == -INFINITY) continue;
        const float wgt = fast_exp2(mw - M);
        L = fmaf(wgt, ml_s[(w * nc_max + c) * 2 + 1], L);
        const floatx4 v = *(const floatx4*)(o_s + (w * nc_max + c) * OPAD + e);
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[r] = fmaf(wgt, v[r], acc[r]);
      }
      const float inv = finish_factor(M, L, a.has_sink, a.sink_l2, a.gate, (size_t)row * a.nH + kvh * ratio + qt + c, a.sinks, a.nH);
      bf16x4 w4;
#pragma unroll
      for (int r = 0; r < 4; ++r) w4[r] = (__bf16)(acc[r] * inv);
      *(bf16x4*)(a.out + ((size_t)row * a.nH + kvh * ratio + qt + c) * D + e) = w4;
    }
  }
