/*
 * gemm_tiles.hip — the kernel of gemm_tiles.hpp (what it is for, its bounds and figures stand there)
 */
#include "gemm_tiles.hpp"

namespace
{
	using namespace mlhip;

	template<typename T, int BLOCKS_M_, int BLOCKS_N_, int WAVES_M_, int WAVES_N_>
	struct GemmTileShape
	{
			static constexpr int BLOCKS_M = BLOCKS_M_, BLOCKS_N = BLOCKS_N_; /* 32x32 blocks of one wavefront */
			static constexpr int WAVES_M = WAVES_M_, WAVES_N = WAVES_N_, WAVES = WAVES_M * WAVES_N, THREADS = 64 * WAVES;
			static constexpr int BM = 32 * BLOCKS_M * WAVES_M, BN = 32 * BLOCKS_N * WAVES_N;
			static constexpr int SLOTS = 2, SLOT_BYTES = (BM + BN) * 128; /* 128 bytes of K of every row of A and B */
			static constexpr int LOADS = (BM + BN) / 8 / WAVES; /* direct-to-LDS loads (8 rows x 128 bytes) per wavefront and piece */
			static constexpr int SLAB_STRIDE = 32 * BLOCKS_N * static_cast<int>(sizeof(T)) + 16;
			static constexpr int LDS_BYTES = SLOTS * SLOT_BYTES;
			/* workgroups that share a compute unit: as many as the 160 KB of LDS hold, four at most */
			static constexpr int RESIDENT = (160 * 1024 / LDS_BYTES < 4) ? 160 * 1024 / LDS_BYTES : 4;
			static_assert((BM + BN) % (8 * WAVES) == 0, "the same number of loads for every wavefront");
			static_assert(WAVES * 32 * SLAB_STRIDE <= LDS_BYTES, "the slots become the slabs of the store");
	};

	/* Epilogue: PlainStore, or a functor on 4 consecutive n whose forms are fixed at compile time (epilogues.hpp) */
	template<typename T, typename Shape, typename Epilogue>
	__global__ __launch_bounds__(Shape::THREADS, Shape::RESIDENT * Shape::WAVES / 4) void kernel_gemm_tiles_nt(const T *A, const T *B, T *C, int M, int N, int k_bytes,
			size_t stride_a, size_t stride_b, size_t stride_c, unsigned int tiles_m, unsigned int tiles_n, unsigned int matrices, int by_rows, size_t a_row_bytes, int write_through, Epilogue epilogue)
	{
		typedef MfmaTraits<T> Traits;
		typedef typename Traits::acc_vec acc_vec;
		constexpr int BLOCKS_M = Shape::BLOCKS_M, BLOCKS_N = Shape::BLOCKS_N, WAVES = Shape::WAVES, LOADS = Shape::LOADS;
		constexpr bool PLAIN = std::is_same<Epilogue, PlainStore>::value;
		const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
		const int wave_m = wave / Shape::WAVES_N, wave_n = wave % Shape::WAVES_N;
		const int frag_row = lane & 31, half_sel = lane >> 5;
		const int pieces = (k_bytes + 127) / 128;

		/* the column tiles of one row tile are neighbours on one XCD; the row tile's matrix changes slowest or its rows do */
		const unsigned int id = xcd_contiguous_block_id(blockIdx.x, gridDim.x);
		const unsigned int row_tile = id / tiles_n;
		const unsigned int slow = row_tile / (by_rows ? matrices : tiles_m);
		const unsigned int fast = row_tile - slow * (by_rows ? matrices : tiles_m);
		const unsigned int matrix = by_rows ? fast : slow;
		const int m_tile = (by_rows ? slow : fast) * Shape::BM, n_tile = (id - row_tile * tiles_n) * Shape::BN;
		const int m0 = m_tile + wave_m * 32 * BLOCKS_M, n0 = n_tile + wave_n * 32 * BLOCKS_N;

		/* bias and beta * C in the accumulators' layout, requested before everything else */
		struct Nothing
		{
				struct Column
				{
				};
				struct Extra
				{
				};
		};
		typedef typename std::conditional<PLAIN, Nothing, Epilogue>::type Parts;
		Epilogue local = epilogue;
		T *out = C + matrix * stride_c;
		size_t out_stride = N;
		typename Parts::Column column[BLOCKS_N][4];
		typename Parts::Extra extra[BLOCKS_M][BLOCKS_N][4];
		if constexpr (!PLAIN)
		{
			out = local.D + matrix * stride_c;
			out_stride = local.row_stride;
			local.bias += static_cast<size_t>(matrix) * local.bias_batch_stride;
			if (local.has_extra())
				local.C += matrix * stride_c;
#pragma unroll
			for (int j = 0; j < BLOCKS_N; j++)
#pragma unroll
				for (int q = 0; q < 4; q++)
				{
					const int n = n0 + 32 * j + 16 * half_sel + 4 * q;
					column[j][q] = local.load_column(n < N ? n : 0);
					if (local.has_extra())
#pragma unroll
						for (int i = 0; i < BLOCKS_M; i++)
							extra[i][j][q] = local.load_extra(min(m0 + 32 * i + frag_row, M - 1), n < N ? n : 0);
				}
		}

		/*
		 * Operands -> LDS slot: [row of A, then of B][128 bytes], the 16-byte chunks of a row swizzled. Rows beyond the matrix repeat its last
		 * row. Row 8 q + 4 h + e of a block of 32 rows of B holds column 16 h + 4 q + e: a lane then ends with 16 consecutive columns.
		 */
		extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];
		const uint8_t *a_base = reinterpret_cast<const uint8_t*>(A + matrix * stride_a);
		const uint8_t *b_base = reinterpret_cast<const uint8_t*>(B + matrix * stride_b);
		const uint8_t *src[LOADS];
		static_assert(WAVES % 2 == 0, "the swizzle of a lane is then the same in all its loads");
		const int chunk = ((lane & 7) ^ ((4 * wave + (lane >> 4)) & 7)) * 16;
#pragma unroll
		for (int u = 0; u < LOADS; u++)
		{
			const int row = (wave + WAVES * u) * 8 + (lane >> 3);
			const int place = row - Shape::BM;
			const int column = (place & ~31) + 16 * ((place >> 2) & 1) + 4 * ((place >> 3) & 3) + (place & 3);
			src[u] = ((row < Shape::BM) ? a_base + static_cast<size_t>(min(m_tile + row, M - 1)) * a_row_bytes
					: b_base + static_cast<size_t>(min(n_tile + column, N - 1)) * k_bytes) + chunk;
		}
		/* the last piece may have 64 bytes only: the lanes beyond them repeat what lies 64 bytes before, and nobody reads it */
		const auto request = [&](int piece, auto slot) __attribute__((always_inline))
		{
			const int back = (piece * 128 + 64 == k_bytes) ? (chunk & 64) : 0;
#pragma unroll
			for (int u = 0; u < LOADS; u++)
			{
				__builtin_amdgcn_global_load_lds((global_ptr_t) (src[u] - back), (lds_ptr_t) (lds + decltype(slot)::value * Shape::SLOT_BYTES + (wave + WAVES * u) * 1024), 16, 0, 0);
				src[u] += 128;
			}
		};
		request(0, std::integral_constant<int, 0>());
		if (pieces > 1)
			request(1, std::integral_constant<int, 1>());

		acc_vec acc[BLOCKS_M][BLOCKS_N];
#pragma unroll
		for (int i = 0; i < BLOCKS_M; i++)
#pragma unroll
			for (int j = 0; j < BLOCKS_N; j++)
#pragma unroll
				for (int r = 0; r < 16; r++)
					acc[i][j][r] = 0;
		int a_first[BLOCKS_M], b_first[BLOCKS_N]; /* this lane's fragment of a slot's first k step, the others by XOR */
#pragma unroll
		for (int i = 0; i < BLOCKS_M; i++)
		{
			const int row = wave_m * 32 * BLOCKS_M + 32 * i + frag_row;
			a_first[i] = row * 128 + ((half_sel ^ ((row >> 1) & 7)) * 16);
		}
#pragma unroll
		for (int j = 0; j < BLOCKS_N; j++)
		{
			const int row = Shape::BM + wave_n * 32 * BLOCKS_N + 32 * j + frag_row;
			b_first[j] = row * 128 + ((half_sel ^ ((row >> 1) & 7)) * 16);
		}
		const auto multiply = [&](int piece, auto slot) __attribute__((always_inline))
		{
			/* loads return in order: this piece has landed once at most those of the next one are outstanding */
			if (piece + 1 < pieces)
				wait_vmcnt<LOADS>();
			else
				wait_vmcnt<0>();
			barrier_no_fence();
			const uint8_t *base = lds + decltype(slot)::value * Shape::SLOT_BYTES;
			const auto step = [&](int kk) __attribute__((always_inline))
			{
				uint4_t a[BLOCKS_M], b[BLOCKS_N];
#pragma unroll
				for (int i = 0; i < BLOCKS_M; i++)
					a[i] = *reinterpret_cast<const uint4_t*>(base + (a_first[i] ^ (kk * 32)));
#pragma unroll
				for (int j = 0; j < BLOCKS_N; j++)
					b[j] = *reinterpret_cast<const uint4_t*>(base + (b_first[j] ^ (kk * 32)));
#pragma unroll
				for (int i = 0; i < BLOCKS_M; i++)
#pragma unroll
					for (int j = 0; j < BLOCKS_N; j++)
						Traits::mma(b[j], a[i], acc[i][j]);
			};
			step(0);
			step(1);
			if (piece * 128 + 64 < k_bytes)
			{
				step(2);
				step(3);
			}
			/* everyone has read the slot before it takes the piece after the next one, or the slabs of the store */
			wait_lgkmcnt_zero();
			if (piece + 2 < pieces)
			{
				barrier_no_fence();
				request(piece + 2, slot);
			}
		};
		for (int piece = 0; piece < pieces; piece += 2)
		{
			multiply(piece, std::integral_constant<int, 0>());
			if (piece + 1 < pieces)
				multiply(piece + 1, std::integral_constant<int, 1>());
		}
		barrier_no_fence();

		/* lane l, register r of block (i, j): m = 32 i + l % 32, n = 32 j + 16 (l / 32) + r; 32 rows at a time cross the wavefront's slab and
		 * leave as whole rows of the sub-tile, 16 bytes per lane (N is a multiple of the vector, checked by the launcher) */
		constexpr int E = 16 / sizeof(T), PER_ROW = 32 * BLOCKS_N / E;
		static_assert(PER_ROW % 2 == 0, "whole passes of 64 lanes over 32 rows");
		uint8_t *slab = lds + wave * 32 * Shape::SLAB_STRIDE;
		const __amdgpu_buffer_rsrc_t through = buffer_of(out + static_cast<size_t>(m_tile) * out_stride + n_tile); /* products_write_through: a tile within 2^31 bytes */
#pragma unroll
		for (int i = 0; i < BLOCKS_M; i++)
		{
#pragma unroll
			for (int j = 0; j < BLOCKS_N; j++)
#pragma unroll
				for (int r = 0; r < 16; r += E)
				{
					Vec<T, E> v;
#pragma unroll
					for (int e = 0; e < E; e += 4)
					{
						const float vals[4] = { acc[i][j][r + e], acc[i][j][r + e + 1], acc[i][j][r + e + 2], acc[i][j][r + e + 3] };
						if constexpr (PLAIN)
#pragma unroll
							for (int t = 0; t < 4; t++)
								v.v[e + t] = vals[t];
						else
						{
							const Vec<T, 4> four = local.result(vals, column[j][(r + e) / 4], extra[i][j][(r + e) / 4]);
#pragma unroll
							for (int t = 0; t < 4; t++)
								v.v[e + t] = four.v[t];
						}
					}
					v.store(reinterpret_cast<T*>(slab + frag_row * Shape::SLAB_STRIDE) + 32 * j + 16 * half_sel + r);
				}
			wait_lgkmcnt_zero(); /* the slab is private to this wavefront */
			__builtin_amdgcn_wave_barrier();
#pragma unroll
			for (int pass = 0; pass < PER_ROW / 2; pass++)
			{
				const int row = (64 * pass + lane) / PER_ROW, col = (64 * pass + lane) % PER_ROW * E;
				const uint4_t v = *reinterpret_cast<const uint4_t*>(slab + row * Shape::SLAB_STRIDE + col * sizeof(T));
				const int m = m0 + 32 * i + row;
				if (m < M && n0 + col < N)
				{
					if (PLAIN && write_through)
						store_through_l2(through, static_cast<int>(((m - m_tile) * static_cast<int>(out_stride) + n0 - n_tile + col) * sizeof(T)), v);
					else
						*reinterpret_cast<uint4_t*>(out + m * out_stride + n0 + col) = v;
				}
			}
			wait_lgkmcnt_zero();
			__builtin_amdgcn_wave_barrier();
		}
	}

	template<typename T, int BLOCKS_M, int BLOCKS_N, int WAVES_M, int WAVES_N, typename Epilogue>
	inline bool launch_as(hipStream_t stream, const StreamGemmArgs &g, bool by_rows, const Epilogue &epilogue)
	{
		typedef GemmTileShape<T, BLOCKS_M, BLOCKS_N, WAVES_M, WAVES_N> Shape;
		const int tiles_m = ceil_div(g.M, Shape::BM), tiles_n = ceil_div(g.N, Shape::BN);
		const unsigned long long tiles = static_cast<unsigned long long>(tiles_m) * tiles_n * g.batch;
		if (tiles > 0xffffffffULL / Shape::THREADS) /* threads that a launch can have */
			return false;
		auto kernel = kernel_gemm_tiles_nt<T, Shape, Epilogue>;
		if (Shape::LDS_BYTES > 64 * 1024)
			ensure_dynamic_lds(reinterpret_cast<const void*>(kernel), Shape::LDS_BYTES);
		hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned int>(tiles)), dim3(Shape::THREADS), Shape::LDS_BYTES, stream, reinterpret_cast<const T*>(g.A),
				reinterpret_cast<const T*>(g.B), reinterpret_cast<T*>(g.C), g.M, g.N, g.k_bytes, g.stride_a, g.stride_b, g.stride_c, tiles_m, tiles_n, g.batch, by_rows,
				g.a_row_bytes != 0 ? g.a_row_bytes : static_cast<size_t>(g.k_bytes), products_write_through(g, sizeof(T)), epilogue);
		return true;
	}
	template<typename T>
	bool try_launch_plain(hipStream_t stream, const StreamGemmArgs &g)
	{
		if (!plain_gemm_tiles_apply(g, sizeof(T)))
			return false;
		const bool by_rows = products_go_by_rows(g, sizeof(T));
		if constexpr (sizeof(T) == 2)
			switch (tile_of_plain(g, sizeof(T)))
			{
				case GemmTile::T128x192:
					return launch_as<T, 1, 3, 4, 2>(stream, g, by_rows, PlainStore { });
				case GemmTile::T128x128:
					return launch_as<T, 2, 1, 2, 4>(stream, g, by_rows, PlainStore { });
				case GemmTile::T128x64:
					return launch_as<T, 2, 1, 2, 2>(stream, g, by_rows, PlainStore { });
				default:
					break;
			}
		return launch_as<T, 1, 1, 2, 2>(stream, g, by_rows, PlainStore { });
	}

	template<typename T, typename Epilogue>
	bool launch_fixed(hipStream_t stream, const StreamGemmArgs &g, const Epilogue &epilogue)
	{
		if constexpr (sizeof(T) == 2)
			switch (tile_with_epilogue(g, sizeof(T)))
			{
				case GemmTile::T128x128:
					return launch_as<T, 2, 1, 2, 4>(stream, g, false, epilogue);
				case GemmTile::T128x64:
					return launch_as<T, 2, 1, 2, 2>(stream, g, false, epilogue);
				default:
					break;
			}
		return launch_as<T, 1, 1, 2, 2>(stream, g, false, epilogue);
	}
	template<typename T>
	bool try_launch_epilogue(hipStream_t stream, const StreamGemmArgs &g, const FloatEpilogue<T> &ep)
	{
		const auto sixteen = [](size_t elements) { return (elements * sizeof(T)) % 16 == 0; };
		if (!(ep.vectorized && ep.alpha == 1.0f && ep.bias != nullptr && (ep.act == ACTIVATION_RELU || ep.act == ACTIVATION_LINEAR)
				&& gemm_tiles_apply(g, sizeof(T), ep.beta != 0.0f) && sixteen(ep.N) && sixteen(ep.row_stride) && sixteen(g.stride_c) && reinterpret_cast<uintptr_t>(ep.D) % 16 == 0))
			return false;
		bool launched = false;
		specialise_epilogue(ep, [&](const auto &fixed)
		{ /* with what was tested above only the forms that have a bias and are fixed at compile time come here */
			if constexpr (!std::is_same<typename std::decay<decltype(fixed)>::type, FloatEpilogue<T>>::value
					&& !std::is_same<typename std::decay<decltype(fixed)>::type, FloatEpilogue<T, ACTIVATION_LINEAR, 0, 0>>::value)
				launched = launch_fixed<T>(stream, g, fixed);
		});
		return launched;
	}
}

namespace mlhip
{
	bool try_launch_gemm_tiles(hipStream_t stream, mlDataType_t dtype, const StreamGemmArgs &g)
	{
		return (dtype == DTYPE_FLOAT16) ? try_launch_plain<half_t>(stream, g) : (dtype == DTYPE_FLOAT32) ? try_launch_plain<float>(stream, g) : false;
	}
	bool try_launch_gemm_tiles(hipStream_t stream, const StreamGemmArgs &g, const FloatEpilogue<half_t> &epilogue)
	{
		return try_launch_epilogue(stream, g, epilogue);
	}
	bool try_launch_gemm_tiles(hipStream_t stream, const StreamGemmArgs &g, const FloatEpilogue<float> &epilogue)
	{
		return try_launch_epilogue(stream, g, epilogue);
	}
} /* namespace mlhip */
