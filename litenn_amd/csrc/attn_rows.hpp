// litenn-hip: attention of many query rows with Float32 operands on the matrix cores (attn_rows.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>

namespace litenn_hip
{
	// Query row i of head h sees keys max(0, q_at + i - window + 1) .. (causal: q_at + i), below `keys`.  Strides are
	// in elements; key and value heads are shared by `share` query heads.
	struct RowsAttn
	{
		const float* q = nullptr; // [rows, ldq]: heads of `dim`
		size_t ldq = 0;
		const void *k = nullptr, *v = nullptr; // Float16 or Float32
		size_t ldk = 0, ldv = 0, k_head = 0, v_head = 0;
		int ring = 0, ring_first = 0; // ring > 0: key row r lives at (ring_first + r) modulo ring
		int heads = 0, share = 1, dim = 0, vdim = 0, rows = 0, keys = 0;
		long long q_at = 0;
		long long window = 1ll << 62;
		bool causal = true;
		// score = dot [* scale] [softcap: tanh(.) [* softcap]] [+ mask * slope]
		bool apply_scale = false, apply_cap = false;
		float scale = 1.0f, softcap = 0.0f;
		const float* mask = nullptr; // [rows, keys]
		double max_bias = 0.0;
		const float* sinks = nullptr; // [heads]
		const float* gate = nullptr;  // [rows, ldg]: the result times its sigmoid
		size_t ldg = 0;
		float out_scale = 1.0f;
		float* out = nullptr; // [rows, ldo]
		size_t ldo = 0;
	};

	// Whether the rows are many enough, and the keys they see, for the tiles to pay (kernel's us against the row kernel's, 32 heads
	// of 128 over 8: Float16 keys, 8 rows on 96 keys 14.0 against 14.7, 12 on 100 13 against 20, 8 on 1024 31 against 110; Float32
	// keys, 16 rows on 96 keys 19 against 26, on 300 35 against 71, heads of 64 22.8 against 22.4).
	inline bool attn_rows_pays(size_t rows, size_t keys, bool f32) { return rows >= (f32 ? 16u : 8u) && keys >= 96; }

	// Returns false, launching nothing, for shapes it does not take: head sizes that are no multiple of 8 or above 128,
	// rows that are not whole 16-byte pieces.
	bool launch_attn_rows(const RowsAttn& a, bool f32, hipStream_t s);
	bool launch_attn_rows_causal(const float* q, const void* kcache, const void* vcache, int cache_dtype, size_t m,
	                             size_t past, size_t n_head, size_t n_kv_head, size_t head_dim, float* out, hipStream_t s);
} // namespace litenn_hip
