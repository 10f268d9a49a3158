# bash abr.sh file.json : both trees in turn
f=$1; R=$GRAFT_REPO_ROOT; [ -z "$R" ] && R=$PWD
for k in 1 2; do (cd $R && timeout -k 10 200 python -u _work/rand.py $R/_work/$f > $R/gpurun_out/rn$k.txt) || exit 1; (cd $R/_work/prev && timeout -k 10 200 python -u $R/_work/rand.py $R/_work/$f > $R/gpurun_out/ro$k.txt) || exit 1; done
